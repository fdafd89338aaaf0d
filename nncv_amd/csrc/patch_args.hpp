// What the fp16 and the fp32 kernel for 3x3 layers with the input patch in LDS share: arguments and tile capacity.
#pragma once
#include "mfma_tile.hpp"

namespace nncv_hip {

constexpr int kPitch = 144;            // fp16: LDS bytes per patch pixel, 128 payload + 16 pad
constexpr unsigned kOOBp = 0x7fff0000u;
constexpr int kXcdsP = 8;

template <int WS> struct PatchCap;     // patch capacity in pixels for 64*WS slots
template <> struct PatchCap<4> { static constexpr int pix = 384; };
template <> struct PatchCap<2> { static constexpr int pix = 256; };
template <> struct PatchCap<1> { static constexpr int pix = 192; };

struct PatchArgs {
  const void* in;        // NHWC [N][H][W][C]
  const void* wf;        // fragment-major weights (launch_weight_frag3x3)
  void* out;             // NHWC [N][H][W][F]
  const float* scale;    // [F] or null
  const float* shift;    // [F] or null
  const void* residual;  // like out, or null
  int N, H, W, C, F, relu;
  int TN, TH;            // tile: TN images x TH output rows x TW output columns
  int tiles_y;           // tiles per group of TN images: ceil(OH / TH) row bands x NTX column tiles
  int tiles;             // ceil(N / TN) * tiles_y
  int ldo, pix;          // elements between pixels of out (and residual) / of in: F and C unless they are slices of wider tensors
  int txw;               // TW | NTX << 16.  NTX = 1 (TW = the full output width) unless a row is too wide for the loader
  int rw_log;            // patch loader: 2^rw_log >= patch columns per loader row
  int rowx;              // stride 1: spare bytes behind the cells of a patch row (see the row pitch in the kernel)
  int OH, OW;            // output size (stride 2; stride 1: H, W)
  int xcd_by_filter;     // XCD <- filter block instead of XCD <- tile range
  unsigned in_bytes, wf_bytes;
  float inv_ph, inv_thw, inv_w;  // 1/(patch rows per image), 1/(TH*TW), 1/TW
  // Stride 2 only: filter blocks >= aux_fb0 (in units of the workgroup's 32*NI filters) belong to a
  // 1x1 stride-2 convolution over the same input (the shortcut of a down-sampling block), with its
  // own output tensor [N][OH][OW][aux_F], scale/shift and ReLU flag.  aux_F = 0: none.
  const void* aux_wf;    // fragment-major, one tap per slab (launch_weight_frag1x1)
  void* aux_out;
  const float* aux_scale;
  const float* aux_shift;
  int aux_F, aux_relu, aux_fb0;
  int aux_inline;  // the workgroup of filter block b also computes block b of the auxiliary filters (aux_F == F): no extra blocks
  unsigned aux_wf_bytes;
  const void* wt;  // fp32 only: the filters as rows [F][9][C] (behind the fields that the fp16 kernel loads)
};

// The fp32 kernel (conv3x3_split.hip): 64 ws pixel slots, 64 filters (half: 32) a workgroup
void launch_conv3x3_split(const PatchArgs& a, int ws, bool half, const char* tag, double flops, double bytes, hipStream_t s);
// ... and 32 consecutive pixels x 32 filters
void launch_conv3x3_split_flat(const PatchArgs& a, double flops, double bytes, hipStream_t s);

}  // namespace nncv_hip
