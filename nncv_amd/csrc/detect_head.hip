// YOLOv5 Detect in fp16: the 1x1 head convolutions of all levels and the decode of their results in one launch.
//
//  * What bounds it: the fp32 result, 85 values per box and anchor (137 MB for 16 images of 640x640), which is three quarters
//    of the bytes.  As operators of their own the three convolutions wrote their results and the decode read them again, a
//    value per lane and load: 40 us for them and 62 for the decode; this launch takes 48 (3.4 TB/s).
//  * A workgroup has 32 pixels of one image and all A * F filters, so that an anchor's part of its result is one contiguous
//    piece of the output.  Slabs of 64 halves go from memory straight into LDS (conv_ring.hip's layout); the sigmoids are put
//    into LDS in the order of the output (a row of F floats per anchor and pixel), 4 values a box are turned into coordinates
//    there, and the pieces leave as they are, 16 bytes a lane.
//  * 36 KB of LDS: four workgroups a CU, some of them writing while others compute.  With 64 pixels and two buffers of slabs
//    two workgroups fitted a CU and the launch took 54 us.  The levels with the longest K come first, the many short tiles
//    fill up behind them.
#include "mfma_tile.hpp"

namespace nncv_hip {

using namespace mt;

namespace {

constexpr unsigned kOOBd = 0x7fffff00u;
constexpr int kPix = 32, kFil = 256, kStageH = (kPix + kFil) * 128, kLanded = 0x0f70;
typedef __attribute__((address_space(3))) void* lds_ptr_t;
__device__ __forceinline__ void fetch_row(__amdgpu_buffer_rsrc_t rs, unsigned char* lds, unsigned voffset, unsigned soffset) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr_t)lds, 16, voffset, soffset, 0, 0);
}

template <bool VEC>  // every anchor's piece of the output starts on 16 bytes
__global__ __launch_bounds__(512) void detect_head_kernel(const DetectHeadArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  int l = 0;
#pragma unroll
  for (int k = 1; k < 3; ++k) l = k < a.levels && (int)blockIdx.x >= a.lv[k].first ? k : l;
  const DetectHeadLevel& v = a.lv[l];
  int tile;
  const int n = fast_div(blockIdx.x - v.first, v.tiles, v.inv_tiles, &tile), p0 = tile * kPix, npix = min(kPix, v.HW - p0);
  const __amdgpu_buffer_rsrc_t rs_in = make_rsrc(v.in, v.in_bytes), rs_wt = make_rsrc(v.wt, v.wt_bytes);

  // rows of 128 bytes, eight lanes to a row; chunk position XORed with (row / 2) % 8
  const int pos = lane & 7, sub = lane >> 3;
  auto column = [&](int group) { return pos ^ (((group & 1) << 2) + (sub >> 1)); };
  const int prow_ = wave * 8 + sub;
  const unsigned pbase = prow_ < npix ? (unsigned)((n * v.HW + p0 + prow_) * v.pix * 2 + column(wave) * 16) : kOOBd;
  unsigned wbase[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) wbase[i] = (unsigned)((wave * 4 + i) * 8 + sub) * (unsigned)v.C * 2u + column(wave * 4 + i) * 16;
  const int slabs = v.C >> 6;
  auto fetch = [&](int s) {
    unsigned char* dst = smem;
    if (wave < kPix / 8) fetch_row(rs_in, dst + wave * 1024, pbase, s * 128);
#pragma unroll
    for (int i = 0; i < 4; ++i) fetch_row(rs_wt, dst + kPix * 128 + (wave * 4 + i) * 1024, wbase[i], s * 128);
  };
  fetch(0);

  const int lrow = lane & 31, lh = lane >> 5, key = (lrow >> 1) & 7;
  floatx16 acc;
#pragma unroll
  for (int e = 0; e < 16; ++e) acc[e] = 0.0f;
  const unsigned char* prow = smem + lrow * 128;
  const unsigned char* wrow = smem + (kPix + wave * 32 + lrow) * 128;
  for (int s = 0; s < slabs; ++s) {
    __builtin_amdgcn_s_waitcnt(kLanded);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int at = ((2 * k + lh) ^ key) * 16;
      Mma<half_t>::run(*reinterpret_cast<const u32x4*>(wrow + at), *reinterpret_cast<const u32x4*>(prow + at), acc);
    }
    __syncthreads();
    if (s + 1 < slabs) fetch(s + 1);
  }

  // ---- sigmoids to [anchor][pixel][F]; a wave's 32 filters meet at most one anchor's end ----
  float* out_tile = reinterpret_cast<float*>(smem);
  const int f0 = wave * 32, used = a.A * a.F, F = a.F;
  const int an0 = __builtin_amdgcn_readfirstlane((int)((float)f0 * a.inv_f + 0.001f)), bound = (an0 + 1) * F;  // f0 / F: whole, or at least 1/256 below the next whole number
  // address of filter f of pixel p: (anchor * kPix + p) * F + f - anchor * F
  float* row0 = out_tile + (an0 * kPix + lrow) * F + f0 - an0 * F;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int d = 8 * q + 4 * lh, f = f0 + d;
    const bool in = f < v.rows;  // (rows: a multiple of 4)
    const floatx4 m = v.scale && in ? *reinterpret_cast<const floatx4*>(v.scale + f) : floatx4{1.f, 1.f, 1.f, 1.f};
    const floatx4 h = v.shift && in ? *reinterpret_cast<const floatx4*>(v.shift + f) : floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float sg = sigmoid_fast(acc[4 * q + e] * m[e] + h[e]);
      float* at = row0 + d + (f + e >= bound ? (kPix - 1) * F : 0);
      if (f + e < used) at[e] = sg;
    }
  }
  __syncthreads();
  // ---- box coordinates ----
  for (int t = threadIdx.x; t < a.A * kPix * 4; t += 512) {
    const int k = t & 3, p = (t >> 2) & (kPix - 1), an = t / (4 * kPix);
    float* at = out_tile + (an * kPix + p) * F + k;
    const float sg = *at;
    int x;
    const int y = fast_div(p0 + p, v.W, v.inv_w, &x);
    float wh = 0.0f;
#pragma unroll
    for (int q = 0; q < 8; ++q) wh = an * 2 + (k & 1) == q ? v.anchor_wh[q] : wh;
    const float s2 = sg * 2.0f;
    *at = k < 2 ? (s2 + ((float)(k == 0 ? x : y) - 0.5f)) * v.stride : (s2 * s2) * wh;
  }
  __syncthreads();
  // ---- an anchor's piece: npix * F consecutive floats ----
  for (int an = 0; an < a.A; ++an) {
    float* dst = a.out + ((long long)n * a.boxes_total + v.box0 + (long long)an * v.HW + p0) * F;
    const float* src = out_tile + an * kPix * F;
    if constexpr (VEC) {
      for (int i = threadIdx.x * 4; i < npix * F; i += 2048) *reinterpret_cast<floatx4*>(dst + i) = *reinterpret_cast<const floatx4*>(src + i);
    } else {
      for (int i = threadIdx.x; i < npix * F; i += 512) dst[i] = src[i];
    }
  }
}

}  // namespace

// Heads of up to 256 filters and at least 64 values a box, over whole slabs.
bool detect_head_applicable(int A, int F, int C, long long in_bytes) {
  return A >= 1 && A <= 4 && F >= 64 && A * F <= kFil && C >= 64 && C % 64 == 0 && in_bytes < (long long)kOOBd;
}

void launch_detect_head(const DetectHeadArgs& a_in, hipStream_t s) {
  DetectHeadArgs a = a_in;
  a.inv_f = 1.0f / (float)a.F;
  bool vec = (a.boxes_total * a.F) % 4 == 0 && reinterpret_cast<uintptr_t>(a.out) % 16 == 0;
  long long blocks = 0;
  double flops = 0, bytes = 0;
  for (int l = 0; l < a.levels; ++l) {
    DetectHeadLevel& v = a.lv[l];
    v.tiles = (v.HW + kPix - 1) / kPix;
    v.inv_tiles = 1.0f / (float)v.tiles;
    v.inv_w = 1.0f / (float)v.W;
    v.first = (int)blocks;
    v.in_bytes = (unsigned)((long long)a.N * v.HW * v.pix * 2);
    v.wt_bytes = (unsigned)v.rows * v.C * 2u;
    blocks += (long long)a.N * v.tiles;
    vec = vec && ((long long)v.HW * a.F) % 4 == 0 && (v.box0 * a.F) % 4 == 0;
    flops += 2.0 * a.N * v.HW * v.C * a.A * a.F;
    bytes += 2.0 * ((double)a.N * v.HW * v.C + (double)v.rows * v.C) + 4.0 * a.N * v.HW * a.A * a.F;
    NNCV_REQUIRE(v.HW < (1 << 24) && v.rows % 4 == 0 && v.rows <= kFil, "detect_head: level too large");
  }
  NNCV_REQUIRE(blocks < (1 << 24), "detect_head: too many boxes");
  constexpr int lds = kStageH;  // (at least kPix * kFil floats)
  ProfScope prof("detect_head", flops, bytes, s);
  if (vec) launch_kernel(detect_head_kernel<true>, dim3((unsigned)blocks), dim3(512), lds, s, a);
  else launch_kernel(detect_head_kernel<false>, dim3((unsigned)blocks), dim3(512), lds, s, a);
  NNCV_HIP_CHECK(hipGetLastError());
}

}  // namespace nncv_hip
