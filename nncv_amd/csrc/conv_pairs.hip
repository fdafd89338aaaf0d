// Convolutions whose whole K axis is a handful of 16-byte chunks (fp16), in two forms:
//  * image_pairs: the stride-2 first layer of a network whose image has at most four channels, straight from the NCHW image:
//    two horizontally adjacent pixels x 4 channels are one chunk, the horizontal walk is stride 1 over S pairs and K is R*S
//    chunks, 18 for YOLOv5s' 6x6 window, 6 for MobileNetV3's 3x3 (tests/Nets/Yolov5s.mlir, tests/Nets/MobileNetV3.mlir);
//  * conv1x1_shortk: 1x1 convolutions over at most 144 channels in multiples of 8 (MobileNetV3's expansion and
//    projection layers, 16..144 channels: none of them a multiple of the 64-byte K step of the
//    pipelined kernel), with the residual add of an inverted-residual block.
// Replaces the compiler's tiling of linalg.conv_2d_nchw_fchw for those layers
// (src/nncv/compiler/Conversion/CodeGen/LlvmCpu/ModernTile.cpp:124-286).
//
// K is so short that a pipelined K walk through LDS only adds barriers.  In the 1x1 form a wave owns 64 pixels x 32
// or 64 filters and needs no staging at all: lane (pixel l%32, chunk half l/32) of MFMA step kk reads
// chunk 2*kk + l/32 of its pixel straight from global memory, ALL steps requested back to back (one
// latency), the filters sit in registers.  The epilogue (scale/shift, residual, activation, one
// rounding) runs on the accumulators; the halves pass through a small LDS tile only to leave as
// whole pixel rows, 16 bytes per lane.  With 5-10 KB of LDS per wave tile the kernel runs at the
// occupancy its registers allow.  HBM bound: input read once (window overlap and the re-reads of
// further filter blocks are served by the caches), result written once.
#include "mfma_tile.hpp"

namespace nncv_hip {

using namespace mt;

namespace {
constexpr unsigned kOOBc = 0x7fff0000u;  // byte offset beyond any buffer this kernel accepts
}

// 1x1 window over C = 8*nch channels, nch <= 2*KST chunks (chunks past nch read as zero).
// WV waves per workgroup, 64 pixels each (1 for small launches: more, smaller workgroups).
// RES: the launch has a residual input (instances without one carry no registers or code for it).
template <int KST, int NI, int WV, bool RES>
__global__ __launch_bounds__(64 * WV) void conv_pairs_kernel(const IgemmArgs a) {
  constexpr int TP = 64 * NI + 16;  // bytes per pixel row of the output tile: 32*NI halves + pad
  __shared__ __align__(16) unsigned char smem[WV * 64 * TP];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lrow = lane & 31, lchunk = lane >> 5;
  const int P = a.N * a.OH * a.OW;
  const int f0 = blockIdx.y * (32 * NI);
  const int p0 = blockIdx.x * (64 * WV) + wave * 64;
  const int nch = a.C / 8;  // chunks per pixel = chunks per filter row
  const __amdgpu_buffer_rsrc_t rs_in = make_rsrc(a.in, a.in_bytes);
  const __amdgpu_buffer_rsrc_t rs_wt = make_rsrc(a.wt, a.wt_bytes);

  // ---- this lane's two pixels and its chunk of every step, requested back to back ----
  u32x4 b[KST][2];
  const int pix = a.pix_stride ? a.pix_stride : a.C;
#pragma unroll
  for (int kk = 0; kk < KST; ++kk) {
    const int c = 2 * kk + lchunk;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int p = p0 + j * 32 + lrow;
      const bool ok = (p < P) & (c < nch);
      b[kk][j] = __builtin_amdgcn_raw_buffer_load_b128(rs_in, ok ? (unsigned)(p * pix + c * 8) * 2u : kOOBc, 0, 0);
    }
  }
  // ---- the filters: row f is nch chunks; lane (filter l%32, chunk half l/32) of step kk holds
  //      chunk 2*kk + l/32.  Rows past the tensor read as zero. ----
  u32x4 w[KST][NI];
#pragma unroll
  for (int kk = 0; kk < KST; ++kk)
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int c = 2 * kk + lchunk;
      w[kk][i] = __builtin_amdgcn_raw_buffer_load_b128(rs_wt, c < nch ? (unsigned)(((f0 + i * 32 + lrow) * nch + c) * 16) : kOOBc, 0, 0);
    }
  // scale/shift of this lane's accumulator channels f0 + 32 i + 8 q + 4 (l/32) .. + 3, and the
  // residual values at the same places (element offsets; rows past the end read element 0)
  floatx4 sc[NI][4], sh[NI][4];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int f = f0 + i * 32 + 8 * q + 4 * lchunk;
      const bool fin = f < a.F;
      sc[i][q] = (a.scale && fin) ? *reinterpret_cast<const floatx4*>(a.scale + f) : floatx4{1.f, 1.f, 1.f, 1.f};
      sh[i][q] = (a.shift && fin) ? *reinterpret_cast<const floatx4*>(a.shift + f) : floatx4{0.f, 0.f, 0.f, 0.f};
    }
  const half_t* res = static_cast<const half_t*>(a.residual);
  half4 rv[NI][2][4];
  if constexpr (RES) {
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int p = p0 + j * 32 + lrow, f = f0 + i * 32 + 8 * q + 4 * lchunk;
          const long long off = (p < P && f < a.F) ? (long long)p * a.ldo + f : 0;
          rv[i][j][q] = *reinterpret_cast<const half4*>(res + off);
        }
  }

  floatx16 acc[NI][2];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
#pragma unroll
  for (int kk = 0; kk < KST; ++kk)
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) Mma<half_t>::run(w[kk][i], b[kk][j], acc[i][j]);

  // ---- epilogue on the accumulators, halves to this wave's tile [pixel][channel] ----
  unsigned char* tile = smem + wave * (64 * TP);
  const int act = a.relu & 0xff;
  const bool res_after = a.relu & kActResidualAfter;  // y = act(conv) + residual instead of act(conv + residual)
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        float y[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = acc[i][j][4 * q + e] * sc[i][q][e] + sh[i][q][e];
        if (RES && !res_after) {
#pragma unroll
          for (int e = 0; e < 4; ++e) y[e] += (float)rv[i][j][q][e];
        }
        act_apply_n<true>(y, act);
        if (RES && res_after) {
#pragma unroll
          for (int e = 0; e < 4; ++e) y[e] += (float)rv[i][j][q][e];
        }
        half4 h;
#pragma unroll
        for (int e = 0; e < 4; ++e) h[e] = (half_t)y[e];
        *reinterpret_cast<half4*>(tile + (j * 32 + lrow) * TP + (i * 32 + 8 * q + 4 * lchunk) * 2) = h;
      }
  __syncthreads();
  // ---- whole pixel rows out: 4*NI lanes cover the 32*NI channels of one pixel ----
  constexpr int LPR = 4 * NI, RPI = 64 / LPR;
  const int fc = (lane % LPR) * 8;
  half_t* out = static_cast<half_t*>(a.out);
#pragma unroll
  for (int it = 0; it < 64 / RPI; ++it) {
    const int row = it * RPI + lane / LPR;
    const u32x4 v = *reinterpret_cast<const u32x4*>(tile + row * TP + fc * 2);
    if (p0 + row < P && f0 + fc < a.F) *reinterpret_cast<u32x4*>(out + (long long)(p0 + row) * a.ldo + f0 + fc) = v;
  }
}

bool conv_pairs_applicable(const IgemmArgs& a, int in_dt, int out_dt) {
  static const bool off_pw = getenv("NNCV_HIP_NO_CONV_SHORTK") != nullptr;
  const int pix = a.pix_stride ? a.pix_stride : a.C;
  const long long P = (long long)a.N * a.OH * a.OW;
  const bool common = in_dt == kF16 && out_dt == kF16 && a.batch == 1 && a.aux_f0 == 0 && a.F % 8 == 0 && a.ldo % 8 == 0 && a.ldo >= a.F &&
                      P * a.ldo < (1ll << 31) && a.in_bytes > 0 && a.in_bytes < kOOBc && a.wt_bytes > 0 && a.wt_bytes < kOOBc &&
                      (a.relu & ~(0xff | kActResidualAfter)) == 0;
  if (!common) return false;
  // 1x1, stride 1, no padding: the output pixel is the input pixel.  The LDS ring (conv_ring.hip) is the better one for whole
  // multiples of 32 channels (64 -> 32 at 5880 pixels: 2.9 against 3.2 us), and from 24 channels on where its 64 x 64 tiles
  // give every CU one and more than 32 filters share a pixel's line (40 -> 240 at 6272 pixels: 3.5 against 4.7).
  const bool ring = a.C % 32 == 0 || (a.C > 16 && a.F > 32 && (P + 63) / 64 * ((a.F + 63) / 64) >= 256);
  return !off_pw && a.R == 1 && a.S == 1 && a.stride_h == 1 && a.stride_w == 1 && a.pad_h == 0 && a.pad_w == 0 && a.OH == a.H &&
         a.OW == a.W && a.C % 8 == 0 && !ring && a.C <= 144 && pix % 8 == 0 && P * pix * 2 < (long long)kOOBc;
}

template <int KST, int NI>
static void launch_pairs_cfg(const IgemmArgs& a, const char* tag, hipStream_t s) {
  const long long P = (long long)a.N * a.OH * a.OW;
  const double flops = a.alg_flops > 0 ? a.alg_flops : 2.0 * P * a.F * a.R * a.S * a.C;
  const double bytes = 2.0 * ((double)a.N * a.H * a.W * a.C + (double)a.F * a.R * a.S * a.C + (double)P * a.F * (a.residual ? 2 : 1));
  ProfScope prof(tag, flops, bytes, s);
  const unsigned gy = (unsigned)((a.F + 32 * NI - 1) / (32 * NI));
  // fewer four-wave workgroups than CUs: one wave per workgroup instead
  const bool small = (P + 255) / 256 * gy < 256;
  const dim3 grid(small ? (unsigned)((P + 63) / 64) : (unsigned)((P + 255) / 256), gy), block(small ? 64 : 256);
  if (a.residual && small) launch_kernel((conv_pairs_kernel<KST, NI, 1, true>), grid, block, 0, s, a);
  else if (a.residual) launch_kernel((conv_pairs_kernel<KST, NI, 4, true>), grid, block, 0, s, a);
  else if (small) launch_kernel((conv_pairs_kernel<KST, NI, 1, false>), grid, block, 0, s, a);
  else launch_kernel((conv_pairs_kernel<KST, NI, 4, false>), grid, block, 0, s, a);
}

void launch_conv_pairs(const IgemmArgs& a, hipStream_t s) {
  // K steps in registers: 1 (16 channels), 3 (..48), 6 (..96), 9 (..144).  64 filters per wave tile only for launches that
  // fill the chip all the same (24 -> 112 at 1440 pixels: 4.1 us with 64, 3.1 with 32)
  const int kst = (a.C / 8 + 1) / 2;
  const bool many = ((long long)a.N * a.OH * a.OW + 63) / 64 * ((a.F + 63) / 64) >= 1024;
  if (kst <= 1) {
    if (a.F > 32 && many) launch_pairs_cfg<1, 2>(a, "conv1x1_shortk<f16,16,64>", s);
    else launch_pairs_cfg<1, 1>(a, "conv1x1_shortk<f16,16,32>", s);
  } else if (kst <= 3) {
    launch_pairs_cfg<3, 1>(a, "conv1x1_shortk<f16,48,32>", s);
  } else if (kst <= 6) {
    launch_pairs_cfg<6, 1>(a, "conv1x1_shortk<f16,96,32>", s);
  } else {
    launch_pairs_cfg<9, 1>(a, "conv1x1_shortk<f16,144,32>", s);
  }
  NNCV_HIP_CHECK(hipGetLastError());
}

// ---------------------------------------------------------------------------------------------
// The image layer.  A workgroup makes 2*WV rows x 32 columns of the result: it reads the haloed rectangle of its image from
// the channel planes (a dword is two pixels of a row; lanes walk a row's pairs), packs pairs of pixels into chunks on the
// way into LDS, and a wave takes its operands for two rows from there, 32 consecutive chunks per read and half.
// It walks a run of such tiles, as many workgroups as the CUs hold: filters, scale and shift are fetched once, and a tile's pixels
// are on their way under the products and stores of the one before (a workgroup a tile: 53.5 us for 16x640x640, 39.7 now).
// What bounds it: its bytes (16x640x640: 39 MB in, 105 out) and the SiLU of 52 million results (a quarter-rate exp and rcp
// each).  Packing the image in a launch of its own wrote 52 MB that the convolution read again, every chunk nine times
// through the vector caches: 23 + 56 us for YOLOv5s (F = 32); 6.6 + 10.5 for MobileNetV3 (F = 16, 32x224x224), 10.2 now.
// ---------------------------------------------------------------------------------------------
template <int R, int S, int NI, int WV>
__global__ __launch_bounds__(64 * WV) __attribute__((amdgpu_waves_per_eu(NI == 1 && WV == 4 ? 4 : 2))) void image_pairs_kernel(const ImagePairsArgs a) {
  constexpr int KST = R * S / 2, TP = 64 * NI + 16, kRows = 2 * (2 * WV - 1) + R, kCols = 32 + S - 1, kPitch = kCols * 16;
  static_assert(R * S % 2 == 0, "an MFMA step takes two chunks");
  constexpr int kEach = (kRows * kCols + 64 * WV - 1) / (64 * WV);
  __shared__ __align__(16) unsigned char smem[kRows * kPitch];  // the packed rectangle
  __shared__ __align__(16) unsigned char outgoing[WV * 64 * TP];
  __shared__ __align__(16) float ss[64 * NI];  // scale, shift
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lrow = lane & 31, lh = lane >> 5;
  // XCD x takes a run of tiles: neighbours share halo lines in its L2
  const int tiles = a.N * a.tiles_y * a.tiles_x, per = (tiles + 7) >> 3, from = (blockIdx.x & 7) * per, end = from + per < tiles ? from + per : tiles;
  int t = from + (blockIdx.x >> 3);
  if (t >= end) return;  // (uniform; before any barrier)
  const __amdgpu_buffer_rsrc_t rs_in = make_rsrc(a.in, a.in_bytes), rs_wt = make_rsrc(a.wt, a.wt_bytes);

  unsigned d[kEach][4];
  const unsigned plane = (unsigned)(a.H * a.W) * 2u;
  int oy0, ox0, img;  // of the tile that d is for
  auto request = [&](int tile) __attribute__((always_inline)) {
    int tx, ty;
    const int rowt = fast_div(tile, a.tiles_x, a.inv_tx, &tx), n = fast_div(rowt, a.tiles_y, a.inv_ty, &ty);
    oy0 = __builtin_amdgcn_readfirstlane(ty * 2 * WV), ox0 = __builtin_amdgcn_readfirstlane(tx * 32), img = __builtin_amdgcn_readfirstlane(n);
#pragma unroll
    for (int i = 0; i < kEach; ++i) {
      const int e = i * 64 * WV + tid, row = e / kCols, col = e - row * kCols, iy = 2 * oy0 - a.pad_h + row, ip = ox0 - a.pad_w + col;
      const bool ok = (e < kRows * kCols) & ((unsigned)iy < (unsigned)a.H) & ((unsigned)ip < (unsigned)(a.W >> 1));
      const unsigned off = ok ? (unsigned)(iy * a.W + 2 * ip) * 2u : kOOBc;
#pragma unroll
      for (int c = 0; c < 3; ++c) d[i][c] = __builtin_amdgcn_raw_buffer_load_b32(rs_in, c < a.C ? off : kOOBc, (unsigned)(img * a.C + c) * plane, 0);
      d[i][3] = 0;
      if (a.C == 4) d[i][3] = __builtin_amdgcn_raw_buffer_load_b32(rs_in, off, (unsigned)(img * 4 + 3) * plane, 0);
    }
  };
  request(t);
  for (int f = tid; f < 32 * NI; f += 64 * WV) {
    ss[f] = a.scale && f < a.F ? a.scale[f] : 1.0f;
    ss[32 * NI + f] = a.shift && f < a.F ? a.shift[f] : 0.0f;
  }
  u32x4 w[KST][NI];
#pragma unroll
  for (int kk = 0; kk < KST; ++kk)
#pragma unroll
    for (int i = 0; i < NI; ++i) w[kk][i] = __builtin_amdgcn_raw_buffer_load_b128(rs_wt, (unsigned)(((i * 32 + lrow) * R * S + 2 * kk + lh) * 16), 0, 0);
  // all of it now: waited for where it is used, in the loop, every trip would wait for the next tile's pixels too
  __builtin_amdgcn_s_waitcnt(0x0f70);
  for (;;) {
#pragma unroll
    for (int i = 0; i < kEach; ++i) {
      const int e = i * 64 * WV + tid;
      if (e < kRows * kCols)
        *reinterpret_cast<u32x4*>(smem + e * 16) = u32x4{(d[i][0] & 0xffffu) | (d[i][1] << 16), (d[i][2] & 0xffffu) | (d[i][3] << 16),
                                                        (d[i][0] >> 16) | (d[i][1] & 0xffff0000u), (d[i][2] >> 16) | (d[i][3] & 0xffff0000u)};
    }
    __syncthreads();
    // the next tile's pixels are on their way under this one's products, activation and stores
    const int row0 = oy0 + 2 * wave, col0 = ox0, at = img;
    t += gridDim.x >> 3;
    const bool more = t < end;
    if (more) request(t);

    floatx16 acc[NI][2];
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
    // chunks 2 kk and 2 kk + 1 of the window: neighbours of a row, or the last of one and the first of the next
    const unsigned char* base = smem + 4 * wave * kPitch + lrow * 16;
    const unsigned char *next = base + lh * 16, *wrap = base + lh * (kPitch - (S - 1) * 16);
#pragma unroll
    for (int kk = 0; kk < KST; ++kk) {
      const int r = 2 * kk / S, c = 2 * kk - r * S;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const u32x4 b = *reinterpret_cast<const u32x4*>((c == S - 1 ? wrap : next) + (2 * j + r) * kPitch + c * 16);
#pragma unroll
        for (int i = 0; i < NI; ++i) Mma<half_t>::run(w[kk][i], b, acc[i][j]);
      }
    }
    __syncthreads();  // the rectangle has been read

    unsigned char* tile = outgoing + wave * (64 * TP);
#pragma unroll
    for (int i = 0; i < NI; ++i) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        asm volatile("" ::: "memory");  // (scale and shift are read again for every block: registers)
        float y[16];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const floatx4 m = *reinterpret_cast<const floatx4*>(ss + i * 32 + 8 * q + 4 * lh), h = *reinterpret_cast<const floatx4*>(ss + 32 * NI + i * 32 + 8 * q + 4 * lh);
#pragma unroll
          for (int e = 0; e < 4; ++e) y[4 * q + e] = acc[i][j][4 * q + e] * m[e] + h[e];
        }
        act_apply_n<true>(y, a.act);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          half4 h;
#pragma unroll
          for (int e = 0; e < 4; ++e) h[e] = (half_t)y[4 * q + e];
          *reinterpret_cast<half4*>(tile + (j * 32 + lrow) * TP + (i * 32 + 8 * q + 4 * lh) * 2) = h;
        }
      }
    }
    // whole pixel rows out: 4*NI lanes cover the 32*NI channels of one pixel (a wave's own tile: no barrier)
    constexpr int LPR = 4 * NI, RPI = 64 / LPR;
    const int fc = (lane % LPR) * 8;
#pragma unroll
    for (int j = 0; j < 2; ++j) {  // (a row's own descriptor: the tensor may be larger than a buffer)
      const __amdgpu_buffer_rsrc_t rs_out = make_rsrc(static_cast<half_t*>(a.out) + ((long long)(at * a.OH + row0 + j) * a.OW + col0) * a.ldo, kOOBc);
#pragma unroll
      for (int it = 0; it < 32 / RPI; ++it) {
        const int px = it * RPI + lane / LPR;
        const u32x4 v = *reinterpret_cast<const u32x4*>(tile + (j * 32 + px) * TP + fc * 2);
        const bool ok = (row0 + j < a.OH) & (col0 + px < a.OW) & (fc < a.F);
        __builtin_amdgcn_raw_buffer_store_b128(v, rs_out, ok ? (unsigned)(px * a.ldo + fc) * 2u : kOOBc, 0, 0);
      }
    }
    if (!more) break;
  }
}

bool image_pairs_applicable(const ImagePairsArgs& a) {
  static const bool off = getenv("NNCV_HIP_NO_CONV_PAIRS") != nullptr;
  const bool window = (a.R == 6 && a.S == 3) || (a.R == 3 && a.S == 2);
  return !off && window && a.C >= 1 && a.C <= 4 && a.W % 2 == 0 && a.F % 8 == 0 && a.F <= 64 && a.ldo % 8 == 0 &&
         (long long)a.N * a.C * a.H * a.W * 2 < (long long)kOOBc && (long long)a.N * ((a.OH + 1) / 2) * ((a.OW + 31) / 32) < (1 << 24) &&
         reinterpret_cast<uintptr_t>(a.in) % 4 == 0;
}

template <int R, int S, int NI>
static void launch_image_cfg(ImagePairsArgs a, const char* tag, hipStream_t s) {
  // tiles of 8 rows; of 2 where those would leave CUs without a workgroup
  const bool small = (long long)a.N * ((a.OH + 7) / 8) * ((a.OW + 31) / 32) < 256;
  const int th = small ? 2 : 8;
  a.tiles_y = (a.OH + th - 1) / th; a.tiles_x = (a.OW + 31) / 32;
  a.inv_tx = 1.0f / (float)a.tiles_x; a.inv_ty = 1.0f / (float)a.tiles_y;
  a.in_bytes = (unsigned)((long long)a.N * a.C * a.H * a.W * 2);
  a.wt_bytes = (unsigned)(a.F * a.R * a.S * 16);
  const double px = (double)a.N * a.OH * a.OW;
  ProfScope prof(tag, a.alg_flops, 2.0 * ((double)a.N * a.C * a.H * a.W + (double)a.F * a.R * a.S * 8 + px * a.F), s);
  // as many workgroups as the CUs hold at most, each with a run of tiles (fewer than 1024 of the small ones)
  const int tiles = a.N * a.tiles_y * a.tiles_x;
  const dim3 grid((unsigned)(tiles < 1024 ? (tiles + 7) / 8 * 8 : 1024));
  if (small) launch_kernel((image_pairs_kernel<R, S, NI, 1>), grid, dim3(64), 0, s, a);
  else launch_kernel((image_pairs_kernel<R, S, NI, 4>), grid, dim3(256), 0, s, a);
  NNCV_HIP_CHECK(hipGetLastError());
}

void launch_image_pairs(const ImagePairsArgs& a, hipStream_t s) {
  if (a.R == 6) {
    if (a.F > 32) launch_image_cfg<6, 3, 2>(a, "conv_pairs<f16,6x3,64>", s);
    else launch_image_cfg<6, 3, 1>(a, "conv_pairs<f16,6x3,32>", s);
  } else {
    if (a.F > 32) launch_image_cfg<3, 2, 2>(a, "conv_pairs<f16,3x2,64>", s);
    else launch_image_cfg<3, 2, 1>(a, "conv_pairs<f16,3x2,32>", s);
  }
}

}  // namespace nncv_hip
