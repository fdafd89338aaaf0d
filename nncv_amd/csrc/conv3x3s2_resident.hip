// fp16 3x3 pad-1 stride-2 convolution of 64 channels for many pixels, with the 1x1 shortcut of a down-sampling block behind it: the filters of
// a workgroup stay in registers, the haloed input rectangle of a tile is in LDS once.
//
//  * In the LDS ring (conv_ring.hip) these layers fetch every pixel two and a quarter times and 128 filters for every tile of 128 pixels,
//    and wait for a slab nine times a tile.  Here a workgroup has a CU, loads its 128 filters once (a wave 32 of them,
//    144 registers) and walks tiles of four rows of up to 31 output pixels; the rectangle of the next tile, 9 rows of 64 cells, is on its way while a
//    tile is multiplied and stored.
//  * Eight waves: four groups of 32 filters, two pairs of output rows.  A row of outputs is an MFMA block of 32 slots.  A patch row that both
//    rows of a pair need is read from LDS once: 60 reads for 72 products.
//  * A cell is a pixel's 64 channels; a patch row keeps its even columns in cells 0 .. 31 and the odd ones in 32 .. 63, so
//    neighbouring outputs are neighbouring cells for every tap.  The position of a 16-byte chunk in its cell is XORed with (cell / 2) % 8, by picking which
//    chunk a lane fetches (buffer_load ... lds): 16 neighbouring cells touch every bank group once.
//  * The MFMA rows hold the filters permuted so that a lane ends with 16 consecutive channels of a pixel: 16-byte stores, no transposing.
//  * Auxiliary filters (AUX) walk the centre tap behind the tile's own, from the same cells.
//  * What bounds it: bytes, a turn of tiles at a time (4.0 TB/s at 256x56x56x64 -> 128 + 128, matrix pipes 40 % busy).  That layer in the ring
//    69.7 us, here 53; conv3x3s2_resident_wins has others.
#include <algorithm>
#include <type_traits>

#include "mfma_tile.hpp"

namespace nncv_hip {

using namespace mt;

namespace {

constexpr unsigned kOOBs2 = 0x7fffff00u;  // byte offset beyond any buffer this kernel accepts
constexpr int kTH = 4, kRowCells = 64, kPatchRows = 2 * kTH + 1, kRowBytes = kRowCells * 128, kPatch = kPatchRows * kRowBytes;
constexpr int kMostCols = 31;
constexpr int kAuxKept = 3;                     // of the auxiliary filters' four steps, in LDS: there are no registers for them
constexpr int kLds = 2 * kPatch + 4 * 128 * 4 + 4 * kAuxKept * 1024;  // patches; scale, shift, and the auxiliary filters'; those filters
constexpr int kEach = kPatchRows * kRowCells / 8 / 8;  // load instructions of a wave
static_assert(kEach * 64 == kPatchRows * kRowCells, "whole instructions");
typedef __attribute__((address_space(3))) void* lds_ptr_t;
__device__ __forceinline__ void fetch16(__amdgpu_buffer_rsrc_t rs, unsigned char* lds, unsigned voffset) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr_t)lds, 16, voffset, 0, 0, 0);
}

struct S2Args {
  const void* in; const void* wf; void* out; const float* scale; const float* shift;
  const void* aux_wf; void* aux_out;
  unsigned in_bytes, wf_bytes, out_bytes, aux_wf_bytes, aux_out_bytes;
  int H, W, OH, OW, pix, F, ldo, act, aux_F, aux_ldo, aux_act;
  int TW, ntx, bands, tiles, tiles_f, walks;  // columns of a tile, tiles of a row and of a column; tiles in all, blocks of 128 filters, workgroups of a block
};

template <bool AUX>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void conv3x3s2_resident_kernel(const S2Args a) {
  extern __shared__ __align__(16) unsigned char smem[];
  float* ss = reinterpret_cast<float*>(smem + 2 * kPatch);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int x = lane & 31, lh = lane >> 5, fg = wave & 3, pair = wave >> 2;
  const int fb = blockIdx.x % a.tiles_f, walk = blockIdx.x / a.tiles_f;
  const int f0 = fb * 128 + fg * 32 + 16 * lh;  // this lane's 16 channels
  int t = (int)((long long)a.tiles * walk / a.walks);
  const int end = (int)((long long)a.tiles * (walk + 1) / a.walks);
  const __amdgpu_buffer_rsrc_t rs_in = make_rsrc(a.in, a.in_bytes);
  const __amdgpu_buffer_rsrc_t rs_wf = make_rsrc(a.wf, a.wf_bytes);
  const __amdgpu_buffer_rsrc_t rs_out = make_rsrc(a.out, a.out_bytes);

  // ---- loader: instruction i of a wave brings cells 8 (9 wave + i) .. + 7, which lie in one row and one plane of it ----
  int n, oy0, ox0, tx;  // of the tile to fetch
  {
    const int row = t / a.ntx;
    tx = t - row * a.ntx;
    n = row / a.bands;
    oy0 = (row - n * a.bands) * kTH;
    ox0 = tx * a.TW;
  }
  auto next_tile = [&]() __attribute__((always_inline)) {
    ox0 += a.TW;
    if (++tx == a.ntx) {
      tx = ox0 = 0;
      oy0 += kTH;
      if (oy0 >= a.OH) oy0 = 0, ++n;
    }
  };
  const int lane_col = 2 * (lane >> 3);
  unsigned lane_at[2];  // an even and an odd instruction's chunk
#pragma unroll
  for (int v = 0; v < 2; ++v) lane_at[v] = (unsigned)(lane_col * a.pix * 2 + (((lane & 7) ^ (4 * v + (lane >> 4))) << 4));
  auto fetch = [&](int i, unsigned to, bool any) __attribute__((always_inline)) {
    const int g = wave * kEach + i, iy = 2 * oy0 - 1 + (g >> 3), ix = 2 * ox0 - 1 + 16 * (g & 3) + ((g >> 2) & 1);
    const bool ok = any & ((unsigned)iy < (unsigned)a.H) & ((unsigned)(ix + lane_col) < (unsigned)a.W);
    const unsigned at = (unsigned)(((n * a.H + iy) * a.W + ix) * a.pix * 2) + lane_at[g & 1];
    fetch16(rs_in, smem + to + g * 1024, ok ? at : kOOBs2);
  };
  if (t < end) {
#pragma unroll
    for (int i = 0; i < kEach; ++i) fetch(i, 0, true);
  }

  // ---- filters: the operand of (64-filter block, tap, 16-channel step, half of the block) is a kilobyte; its lanes permuted ----
  const int row = x, perm = 16 * ((row >> 2) & 1) + 4 * (row >> 3) + (row & 3);
  const unsigned wlane = (unsigned)(perm + 32 * lh) * 16u;
  u32x4 w[36], aw;
  unsigned char* kept = smem + 2 * kPatch + 4 * 128 * 4 + fg * kAuxKept * 1024 + lane * 16;
  {
    const int block = fb * 2 + (fg >> 1);
#pragma unroll
    for (int q = 0; q < 36; ++q) w[q] = __builtin_amdgcn_raw_buffer_load_b128(rs_wf, wlane, (unsigned)((block * 36 + q) * 2 + (fg & 1)) * 1024u, 0);
    if constexpr (AUX) {
      const __amdgpu_buffer_rsrc_t rs_aux = make_rsrc(a.aux_wf, a.aux_wf_bytes);
      auto load = [&](int q) { return __builtin_amdgcn_raw_buffer_load_b128(rs_aux, wlane, (unsigned)((block * 4 + q) * 2 + (fg & 1)) * 1024u, 0); };
      aw = load(kAuxKept);
      if (pair == 0) {
#pragma unroll
        for (int q = 0; q < kAuxKept; ++q) *reinterpret_cast<u32x4*>(kept + q * 1024) = load(q);
      }
    }
  }
  if (tid < 128) {
    const int f = fb * 128 + tid;
    ss[tid] = a.scale && f < a.F ? a.scale[f] : 1.0f;
    ss[128 + tid] = a.shift && f < a.F ? a.shift[f] : 0.0f;
    if constexpr (AUX) {
      ss[256 + tid] = a.scale && f < a.aux_F ? a.scale[a.F + f] : 1.0f;
      ss[384 + tid] = a.shift && f < a.aux_F ? a.shift[a.F + f] : 0.0f;
    }
  }
  if (t >= end) return;  // (uniform; before any barrier)

  // ---- operands: column x of the wave's rows, chunk 2 k + lh: bytes from the cell of the pair's first patch row ----
  unsigned at0[4], at2[4];  // tap columns 0 and 1 (the other plane); 2
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    at0[k] = (unsigned)(pair * 4 * kRowBytes + x * 128 + (((2 * k + lh) ^ ((x >> 1) & 7)) << 4));
    at2[k] = (unsigned)(pair * 4 * kRowBytes + (x + 1) * 128 + (((2 * k + lh) ^ (((x + 1) >> 1) & 7)) << 4));
  }
  __builtin_amdgcn_s_waitcnt(0x0f70);
  unsigned buf = 0;
  for (;;) {
    __syncthreads();  // every wave's part of this patch is there, and nobody reads the other one any more
    const int img = n, oy = oy0 + 2 * pair, ox = ox0;
    const bool more = ++t < end;
    next_tile();
    const unsigned char* patch = smem + buf;
    auto operand = [&](int s, int k, int r) __attribute__((always_inline)) {  // tap column s, row r of the pair's five
      return *reinterpret_cast<const u32x4*>(patch + (s == 2 ? at2[k] : at0[k]) + r * kRowBytes + (s == 1 ? kRowBytes / 2 : 0));
    };
    floatx16 acc[2];
    // sixty operands in the order (row, column, step), four ahead of their products
    constexpr int kAhead = 4, kReads = 60;
    u32x4 p[kReads];
    auto read = [&](auto i_c) __attribute__((always_inline)) {
      constexpr int i = decltype(i_c)::value;
      p[i] = operand((i >> 2) % 3, i & 3, i / 12);
    };
    read(std::integral_constant<int, 0>());
    read(std::integral_constant<int, 1>());
    read(std::integral_constant<int, 2>());
    read(std::integral_constant<int, 3>());
    auto steps = [&](auto self, auto i_c) __attribute__((always_inline)) -> void {
      constexpr int i = decltype(i_c)::value;
      if constexpr (i < kReads) {
        constexpr int r = i / 12, q = i % 12;  // (q: column and step of a filter row)
        if constexpr (i + kAhead < kReads) read(std::integral_constant<int, i + kAhead>());
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (r <= 2) {
          if constexpr (i == 0) Mma<half_t>::start(w[r * 12 + q], p[i], acc[0]);
          else Mma<half_t>::run(w[r * 12 + q], p[i], acc[0]);
        }
        if constexpr (r >= 2) {
          if constexpr (i == 24) Mma<half_t>::start(w[(r - 2) * 12 + q], p[i], acc[1]);
          else Mma<half_t>::run(w[(r - 2) * 12 + q], p[i], acc[1]);
        }
        __builtin_amdgcn_sched_barrier(0);
        // the next tile's requests, behind the last tile too: a fixed number of them.  (All of them ahead of the products 47 us at
        // 256x56x56x64 -> 128, on the machine that these take 38 to 41 on.)
        if constexpr (i % 2 == 0 && i / 2 < kEach) {
          fetch(i / 2, kPatch - buf, more);
          __builtin_amdgcn_sched_barrier(0);
        }
        self(self, std::integral_constant<int, i + 1>());
      }
    };
    steps(steps, std::integral_constant<int, 0>());

    auto finish = [&](const float* tab, int act, const __amdgpu_buffer_rsrc_t rs, int ldo, int F) __attribute__((always_inline)) {
      const float* mine = tab + fg * 32 + 16 * lh;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const bool in = (oy + j < a.OH) & (x < a.TW) & (ox + x < a.OW);
        const unsigned o = (unsigned)(((img * a.OH + oy + j) * a.OW + ox + x) * ldo + f0) * 2u;
        float y[16];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const floatx4 m = *reinterpret_cast<const floatx4*>(mine + 4 * q), h = *reinterpret_cast<const floatx4*>(mine + 128 + 4 * q);
#pragma unroll
          for (int e = 0; e < 4; ++e) y[4 * q + e] = acc[j][4 * q + e] * m[e] + h[e];
        }
        act_apply_n<true>(y, act);
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          half8 v;
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] = (half_t)y[8 * c + e];
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), rs, (in & (f0 + 8 * c < F)) ? o + 16u * c : kOOBs2, 0, 0);
        }
      }
    };
    finish(ss, a.act, rs_out, a.ldo, a.F);
    if constexpr (AUX) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const u32x4 f = k < kAuxKept ? *reinterpret_cast<const u32x4*>(kept + k * 1024) : aw;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const u32x4 c = operand(1, k, 1 + 2 * j);
          if (k == 0) Mma<half_t>::start(f, c, acc[j]);
          else Mma<half_t>::run(f, c, acc[j]);
        }
      }
      finish(ss + 256, a.aux_act, make_rsrc(a.aux_out, a.aux_out_bytes), a.aux_ldo, a.aux_F);
    }
    if (!more) break;
    buf = kPatch - buf;
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0x0f70 | (AUX ? 8 : 4));  // all but the stores: this wave's part of the next patch is there
  }
}

void geometry(int OW, int* TW, int* ntx) {
  *ntx = (OW + kMostCols - 1) / kMostCols;
  *TW = (OW + *ntx - 1) / *ntx;
}

}  // namespace

// Taken where a workgroup has three and a half tiles or more and four fifths of the slots hold a pixel.  us, in the ring and here: 256x56x56 -> 128
// 57 / 38-47, 128 images 31.4 / 24-28, 16x160x160 31.6 / 25-29, 128x62x62 36.8 / 27-33, 64x56x56 -> 256 24.2 / 22-24; below that many tiles 100x56x56
// 20.1 / 19.8, 64x56x56 14.7 / 15.6, 8x160x160 14.9 / 16.5; and with 20 of 32 slots 128x58x78 41.6 / 42, 64x58x78 19.0 / 23.3.
// With passes in flight too, though a workgroup has a CU to itself, ResNet-18: four of 128 images 1853 / 1842, three of 192 2067 / 2044, four of 256 3715 / 3650, three of 64 images of
// 320x320 1418 / 1423.
bool conv3x3s2_resident_wins(const IgemmArgs& a) {
  static const bool off = getenv("NNCV_HIP_NO_S2_RESIDENT") != nullptr;
  const int pix = a.pix_stride ? a.pix_stride : a.C, main_f = a.aux_f0 ? a.aux_f0 : a.F, aux_f = a.F - main_f;
  if (off || a.stride_h != 2 || a.stride_w != 2 || a.R != 3 || a.S != 3 || a.pad_h != 1 || a.pad_w != 1 || a.C != 64 || a.residual || !a.wt_frag || a.batch != 1 ||
      a.split_f || a.OH != (a.H - 1) / 2 + 1 || a.OW != (a.W - 1) / 2 + 1 || main_f % 8 != 0 || a.ldo % 8 != 0 || pix % 8 != 0 || (a.relu & ~0xff) ||
      (a.aux_f0 && (!a.aux_wt_frag || a.aux_tap != 4 || aux_f != main_f || a.aux_ldo % 8 != 0 || (a.aux_relu & ~0xff))))
    return false;
  int TW, ntx;
  geometry(a.OW, &TW, &ntx);
  const long long P = (long long)a.N * a.OH * a.OW, tiles = (long long)a.N * ((a.OH + kTH - 1) / kTH) * ntx, blocks = (main_f + 127) / 128;
  return a.in_bytes > 0 && a.in_bytes < kOOBs2 && P * std::max(a.ldo, a.aux_ldo) * 2 < (long long)kOOBs2 && tiles < 1 << 24 && blocks <= 256 &&
         tiles * blocks >= 896 && (double)P >= 0.8 * 128 * (double)tiles;
}

void launch_conv3x3s2_resident(const IgemmArgs& a, double flops, double bytes, hipStream_t s) {
  S2Args d{};
  const int main_f = a.aux_f0 ? a.aux_f0 : a.F, P = a.N * a.OH * a.OW;
  d.in = a.in; d.wf = a.wt_frag; d.out = a.out; d.scale = a.scale; d.shift = a.shift;
  d.in_bytes = a.in_bytes; d.wf_bytes = (unsigned)weight_frag3x3_bytes(kF16, main_f, 64); d.out_bytes = (unsigned)P * a.ldo * 2u;
  d.H = a.H; d.W = a.W; d.OH = a.OH; d.OW = a.OW; d.pix = a.pix_stride ? a.pix_stride : a.C; d.F = main_f; d.ldo = a.ldo; d.act = a.relu;
  geometry(a.OW, &d.TW, &d.ntx);
  d.bands = (a.OH + kTH - 1) / kTH;
  d.tiles = a.N * d.bands * d.ntx;
  d.tiles_f = (main_f + 127) / 128;
  d.walks = std::min(d.tiles, 256 / d.tiles_f);
  if (a.aux_f0) {
    d.aux_wf = a.aux_wt_frag; d.aux_out = a.aux_out; d.aux_F = a.F - main_f; d.aux_ldo = a.aux_ldo; d.aux_act = a.aux_relu;
    d.aux_wf_bytes = (unsigned)((size_t)((d.aux_F + 63) / 64) * 64 * 64 * 2); d.aux_out_bytes = (unsigned)P * a.aux_ldo * 2u;
  }
  const auto kernel = a.aux_f0 ? conv3x3s2_resident_kernel<true> : conv3x3s2_resident_kernel<false>;
  static const bool attr = [] {
    NNCV_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(conv3x3s2_resident_kernel<true>), hipFuncAttributeMaxDynamicSharedMemorySize, kLds));
    NNCV_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(conv3x3s2_resident_kernel<false>), hipFuncAttributeMaxDynamicSharedMemorySize, kLds));
    return true;
  }();
  (void)attr;
  ProfScope prof("conv_ring<s2,resident>", flops, bytes, s);
  launch_kernel(kernel, dim3((unsigned)(d.walks * d.tiles_f)), dim3(512), kLds, s, d);
  NNCV_HIP_CHECK(hipGetLastError());
}

}  // namespace nncv_hip
