// fp16 3x3 pad-1 convolution of 32 channels, stride 1 or 2, for large images: the filters stay in registers, the haloed input
// rectangle of a tile is in LDS once.
//
//  * What bounded these layers in the LDS ring (conv_ring.hip): nine-fold pixels and the filters of every tile went through LDS.
//    Here a pixel's 64 bytes are written to LDS once (plus the halo), and a wave's 32 filters, 18 K steps, are 72 registers that
//    a workgroup loads once for all its tiles.
//  * A workgroup has four waves and walks tiles of 8 rows x 32 columns (up to 32 filters) or 4 x 32 (up to 64).  A wave makes
//    two rows of 32 pixels x 32 filters; an input row that both rows need is read from LDS once.
//  * The rectangle of the next tile is on its way while a tile is scaled, activated and stored; three workgroups a CU cover the rest.
//  * A cell of LDS is one pixel, four chunks of 16 bytes; the position of a chunk is XORed with (column / 4) % 4, by picking which
//    chunk a lane fetches, so that 16 neighbouring cells touch every bank group once.  Stride 2: a row's even columns, then its odd ones.
//  * What bounds it now: bytes in and out with a trip's chain of fetch, products and stores, three workgroups a CU deep (3.4 TB/s).
//    us in the ring -> here: 16x160x160x32 -> 32 25.7 -> 15.9; 16x320x320x32 -> 64, stride 2, 37.1 -> 29.8; 16x112x112x32 -> 64
//    20.7 -> 15.8; 13x114x31x32 -> 24 6.7 -> 5.2.  Fetching in every trip, also after the last tile, made the waits of the stored
//    part exact and cost 0.7 us a launch more than that gave.
#include "mfma_tile.hpp"

namespace nncv_hip {

using namespace mt;

namespace {

constexpr unsigned kOOBn = 0x7fffff00u;  // byte offset beyond any buffer this kernel accepts
typedef __attribute__((address_space(3))) void* lds_ptr_t;

struct NarrowArgs {
  const void* in; const void* wt; void* out; const float* scale; const float* shift; const void* residual;
  unsigned in_bytes, wt_bytes, out_bytes;
  int H, W, F, OH, OW, pix, ldo, act, tiles, tiles_x, tiles_y;
  float inv_tx, inv_ty;
};

template <int ST, int FB>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3, 3))) void conv3x3_narrow_kernel(const NarrowArgs a) {
  constexpr int kTH = 8 / FB, kRows = (kTH - 1) * ST + 3, kCols = 31 * ST + 3, kCells = kRows * kCols, kEach = (kCells + 63) / 64, kPitch = 80;
  __shared__ __align__(16) unsigned char cells[kEach * 4096];
  __shared__ __align__(16) unsigned char outgoing[4 * 32 * kPitch];  // of each wave a row of 32 pixels
  __shared__ __align__(16) float ss[FB * 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lrow = lane & 31, lh = lane >> 5;
  const int wr = wave / FB, f0 = (wave % FB) * 32;
  const __amdgpu_buffer_rsrc_t rs_in = make_rsrc(a.in, a.in_bytes), rs_wt = make_rsrc(a.wt, a.wt_bytes), rs_out = make_rsrc(a.out, a.out_bytes);
  // XCD x takes a run of tiles: neighbours share halo lines in its L2
  const int per = (a.tiles + 7) >> 3, from = (blockIdx.x & 7) * per, end = from + per < a.tiles ? from + per : a.tiles, step = gridDim.x >> 3;
  int t = from + (blockIdx.x >> 3);
  if (t >= end) return;  // (uniform; before any barrier)

  u32x4 w[18];
  const unsigned wofs = f0 + lrow < a.F ? (unsigned)((f0 + lrow) * 576 + lh * 16) : kOOBn;
#pragma unroll
  for (int k = 0; k < 18; ++k) w[k] = __builtin_amdgcn_raw_buffer_load_b128(rs_wt, wofs, k * 32, 0);
  if (tid < FB * 32) {
    ss[tid] = a.scale && tid < a.F ? a.scale[tid] : 1.0f;
    ss[FB * 32 + tid] = a.shift && tid < a.F ? a.shift[tid] : 0.0f;
  }

  int n, oy0, ox0;  // of tile t
  auto locate = [&](int tile) __attribute__((always_inline)) {
    int tx, ty;
    const int row = fast_div(tile, a.tiles_x, a.inv_tx, &tx), img = fast_div(row, a.tiles_y, a.inv_ty, &ty);
    n = __builtin_amdgcn_readfirstlane(img);
    oy0 = __builtin_amdgcn_readfirstlane(ty) * kTH;
    ox0 = __builtin_amdgcn_readfirstlane(tx) * 32;
  };
  auto fetch = [&]() __attribute__((always_inline)) {  // of 16 cells a load, lane l brings cell l / 4
    int l = lane;
    asm volatile("" : "+v"(l));  // (what follows is made again for every tile: kept, it would not fit the registers)
    const int iy0 = oy0 * ST - 1, ix0 = ox0 * ST - 1, base = ((n * a.H + iy0) * a.W + ix0) * a.pix * 2;
#pragma unroll
    for (int i = 0; i < kEach; ++i) {
      const int q = (wave * kEach + i) * 16 + (l >> 2), row = q / kCols, at = q - row * kCols;
      const int idx = ST == 1 || at < 33 ? at : at - 33, col = ST == 1 ? at : at < 33 ? 2 * at : 2 * at - 65;
      const bool ok = (q < kCells) & ((unsigned)(iy0 + row) < (unsigned)a.H) & ((unsigned)(ix0 + col) < (unsigned)a.W);
      unsigned v = (unsigned)(base + (__mul24(row, a.W) + col) * (a.pix * 2) + (((l & 3) ^ ((idx >> 2) & 3)) << 4));
      asm volatile("" : "+v"(v));  // (no branch around it)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_in, (lds_ptr_t)(cells + (wave * kEach + i) * 1024), 16, ok ? v : kOOBn, 0, 0, 0);
    }
  };
  locate(t);
  fetch();
  __builtin_amdgcn_s_waitcnt(0x0f70);  // vector memory: all of it

  const unsigned char* at[3][2];  // tap column c, channels 16 k + 8 lh ..: row 0 of this wave
#pragma unroll
  for (int c = 0; c < 3; ++c)
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int idx = lrow + (ST == 1 ? c : c >> 1), cell = 2 * ST * wr * kCols + idx + (ST == 2 && c == 1 ? 33 : 0);
      at[c][k] = cells + cell * 64 + (((2 * k + lh) ^ ((idx >> 2) & 3)) << 4);
    }
  unsigned char* mine = outgoing + wave * 32 * kPitch;
  for (;;) {
    __syncthreads();
    // where this lane's part of the rows goes, and what is added to it
    const int img = n, row0 = oy0 + 2 * wr, col0 = ox0;
    auto goes_to = [&](int j, int i) __attribute__((always_inline)) {
      const int ox = col0 + i * 16 + (lane >> 2), f = f0 + (lane & 3) * 8;
      const bool ok = (row0 + j < a.OH) & (ox < a.OW) & (f < a.F);
      return ok ? (unsigned)(((img * a.OH + row0 + j) * a.OW + ox) * a.ldo + f) * 2u : kOOBn;
    };
    u32x4 rv[2][2];
    if (a.residual) {
      const __amdgpu_buffer_rsrc_t rs_res = make_rsrc(a.residual, a.out_bytes);
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int i = 0; i < 2; ++i) rv[j][i] = __builtin_amdgcn_raw_buffer_load_b128(rs_res, goes_to(j, i), 0, 0);
    }
    floatx16 acc[2];
#pragma unroll
    for (int r = 0; r < ST + 3; ++r)
#pragma unroll
      for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          const u32x4 p = *reinterpret_cast<const u32x4*>(at[c][k] + r * (kCols * 64));
          const int s = (r * 3 + c) * 2 + k, s1 = s - ST * 6;  // K step of the first row, of the second
          if (s == 0) Mma<half_t>::start(w[0], p, acc[0]);
          else if (r < 3) Mma<half_t>::run(w[s], p, acc[0]);
          if (s1 == 0) Mma<half_t>::start(w[0], p, acc[1]);
          else if (r >= ST) Mma<half_t>::run(w[s1], p, acc[1]);
        }
    __syncthreads();  // the rectangle has been read
    t += step;
    const bool more = t < end;
    if (more) {
      locate(t);
      fetch();
    }
    __builtin_amdgcn_sched_barrier(0);  // the four stores below are the last vector-memory operations of a trip
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      asm volatile("" ::: "memory");  // (scale and shift are read again for the second row: registers)
      float y[16];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const floatx4 m = *reinterpret_cast<const floatx4*>(ss + f0 + 8 * q + 4 * lh), h = *reinterpret_cast<const floatx4*>(ss + FB * 32 + f0 + 8 * q + 4 * lh);
#pragma unroll
        for (int e = 0; e < 4; ++e) y[4 * q + e] = acc[j][4 * q + e] * m[e] + h[e];
      }
      if (a.residual) {
#pragma unroll
        for (int i = 0; i < 2; ++i) *reinterpret_cast<u32x4*>(mine + (i * 16 + (lane >> 2)) * kPitch + (lane & 3) * 16) = rv[j][i];
      }
      auto add = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const half4 v = *reinterpret_cast<const half4*>(mine + lrow * kPitch + q * 16 + lh * 8);
#pragma unroll
          for (int e = 0; e < 4; ++e) y[4 * q + e] += (float)v[e];
        }
      };
      if (a.residual && !(a.act & kActResidualAfter)) add();
      act_apply_n<true>(y, a.act & 0xff);
      if (a.residual && (a.act & kActResidualAfter)) add();
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        half4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = (half_t)y[4 * q + e];
        *reinterpret_cast<half4*>(mine + lrow * kPitch + q * 16 + lh * 8) = v;
      }
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const u32x4 v = *reinterpret_cast<const u32x4*>(mine + (i * 16 + (lane >> 2)) * kPitch + (lane & 3) * 16);
        __builtin_amdgcn_raw_buffer_store_b128(v, rs_out, goes_to(j, i), 0, 0);
      }
    }
    if (!more) break;
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0x0f74);  // all but the four stores: this wave's part of the rectangle is there
  }
}

template <int ST, int FB>
void launch_cfg(NarrowArgs d, int N, hipStream_t s) {
  constexpr int kTH = 8 / FB;
  d.tiles_x = (d.OW + 31) / 32;
  d.tiles_y = (d.OH + kTH - 1) / kTH;
  d.tiles = N * d.tiles_y * d.tiles_x;
  d.inv_tx = 1.0f / (float)d.tiles_x;
  d.inv_ty = 1.0f / (float)d.tiles_y;
  launch_kernel((conv3x3_narrow_kernel<ST, FB>), dim3((unsigned)(d.tiles < 768 ? (d.tiles + 7) / 8 * 8 : 768)), dim3(256), 0, s, d);
}

}  // namespace

static long long narrow_tiles(const IgemmArgs& a) {
  const int th = a.F > 32 ? 4 : 8;
  return (long long)a.N * ((a.OH + th - 1) / th) * ((a.OW + 31) / 32);
}

// The time of a launch (60 layers of 104 .. 5664 tiles, 5 .. 31 us, within a tenth): the fixed part is a workgroup's filters and first
// rectangle; many tiles are cheaper from stride 1 with up to 64 filters on, where a rectangle is small beside what is written.
double conv3x3_narrow_us(const IgemmArgs& a) {
  const double t = (double)narrow_tiles(a);
  if (a.stride_h == 2) return 4.2 + 0.0085 * t;
  if (a.F <= 32) return 4.4 + 0.0072 * t;
  return 4.4 + 0.0066 * t - 0.0018 * (t > 1500 ? t - 1500 : 0);
}

// Taken where the fit above is below the ring's by a twentieth.  30 layers that it takes run in 0.60 to 0.96 of the ring's time; of
// 49 where it could, those that the rule leaves to the ring would mostly be slower here: 32x42x131x32 -> 64, stride 2, 7.6 against 9.6
// (tiles of 32 columns for 66), 27x51x22x32 -> 64 6.4 against 6.9.  Fewer than 128 tiles leave CUs without one.
bool conv3x3_narrow_applicable(const IgemmArgs& a, int in_dt, int out_dt) {
  static const bool off = getenv("NNCV_HIP_NO_CONV_NARROW") != nullptr;
  const int pix = a.pix_stride ? a.pix_stride : a.C, st = a.stride_h;
  const bool form = !off && in_dt == kF16 && out_dt == kF16 && a.batch == 1 && a.R == 3 && a.S == 3 && a.pad_h == 1 && a.pad_w == 1 && st == a.stride_w &&
                    a.C == 32 && a.F <= 64 && ((st == 1) | ((st == 2) & (a.F > 32)));
  if (!form || !conv_ring_applicable(a, in_dt, out_dt) || a.split_f != 0) return false;
  const long long tiles = narrow_tiles(a);
  return tiles >= 128 && tiles < (1 << 24) && pix >= 32 && conv3x3_narrow_us(a) < 0.95 * conv_ring_us(a);
}

void launch_conv3x3_narrow(const IgemmArgs& a, hipStream_t s) {
  NarrowArgs d{};
  d.in = a.in; d.wt = a.wt; d.out = a.out; d.scale = a.scale; d.shift = a.shift; d.residual = a.residual;
  d.H = a.H; d.W = a.W; d.F = a.F; d.OH = a.OH; d.OW = a.OW; d.ldo = a.ldo; d.act = a.relu;
  d.pix = a.pix_stride ? a.pix_stride : a.C;
  const double P = (double)a.N * a.OH * a.OW;
  d.in_bytes = a.in_bytes; d.wt_bytes = (unsigned)a.F * 576u; d.out_bytes = (unsigned)((long long)a.N * a.OH * a.OW * a.ldo * 2);
  const char* tag = a.stride_h == 2 ? "conv3x3_narrow<s2,64>" : a.F > 32 ? "conv3x3_narrow<s1,64>" : "conv3x3_narrow<s1,32>";
  ProfScope prof(tag, a.alg_flops > 0 ? a.alg_flops : 2.0 * P * a.F * 288,
                 2.0 * ((double)a.N * a.H * a.W * a.C + 288.0 * a.F + P * a.F * (a.residual ? 2 : 1)), s);
  if (a.stride_h == 2) launch_cfg<2, 2>(d, a.N, s);
  else if (a.F > 32) launch_cfg<1, 2>(d, a.N, s);
  else launch_cfg<1, 1>(d, a.N, s);
  NNCV_HIP_CHECK(hipGetLastError());
}

}  // namespace nncv_hip
