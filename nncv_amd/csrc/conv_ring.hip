// fp16 implicit GEMM whose operands go from memory straight into an LDS ring: output tile of BP pixels x BF filters per
// workgroup, K in slabs of 64 halves (one 128-byte line of a pixel and of a filter row), S slabs in the ring.
//
//  * A slab is fetched by buffer loads with the LDS bit: no registers and no LDS stores in between.  With one buffer
//    (16 KB for a 64 x 64 tile) seven workgroups share a CU and hide each other's latency: that is what layers bound by memory
//    want (160x160x64 -> 32, 16 images: 23.2 -> 13.8 us, 5.7 TB/s).  With two, a slab is fetched under the one before it, for
//    launches of a few tiles per CU and a long K axis (20x20x512 -> 256: 8.5 -> 5.9).  Rings of three and four slabs measured
//    slower everywhere: they cost resident workgroups, which hide more than the extra slabs do.
//  * A load instruction moves eight rows of 128 bytes, eight lanes to a row: whole lines of memory.  The position of a 16-byte
//    chunk inside its LDS row is XORed with (row / 2) % 8, by picking which chunk a lane fetches; a wave's 16-byte operand
//    reads (one column of 16 rows at a time) then touch every bank group once.
//  * What bounds it: bytes for 1x1 layers of up to 64 channels, LDS reads for long K axes (a wave tile of 32 x 64 reads three
//    operands for two products), the latency of a slab (0.4 us) for launches of less than a tile per CU; those with a long K
//    go to conv_direct.hip.  It measured 1.2 to 2 times the register-staged kernel (igemm_fast.hip) on all 35 layers of a
//    random 300 that came from there.
//  * Filters are the rows of the product and pixels its columns, so a lane ends with four consecutive channels of a pixel:
//    scale, shift, residual and activation are applied in fp32 in registers, the fp16 result goes through a wave-private
//    LDS tile (no barrier), and leaves as whole rows.
#include "mfma_tile.hpp"

namespace nncv_hip {

using namespace mt;

namespace {

constexpr unsigned kOOBr = 0x7fffff00u;  // byte offset beyond any buffer this kernel accepts
typedef __attribute__((address_space(3))) void* lds_ptr_t;
__device__ __forceinline__ void fetch16(__amdgpu_buffer_rsrc_t rs, unsigned char* lds, unsigned voffset, unsigned soffset) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr_t)lds, 16, voffset, soffset, 0, 0);
}
constexpr int kAllLanded = 0x0f70;  // s_waitcnt: no vector-memory operation outstanding, nothing else

struct RingArgs {
  const void* in; const void* wt; void* out; const float* scale; const float* shift; const void* residual;
  unsigned in_bytes, wt_bytes, out_bytes;
  int H, W, F, OW, OHW, P, pix;                       // pix: elements between pixels
  int stride_h, stride_w, pad_h, pad_w, S;
  int act, ldo, chunks, cpt;                          // 16-byte chunks of K, and of one tap
  int tiles_f, tiles_p, pixels_first;
  int aux_tiles, aux_f0, aux_tap, aux_act, aux_ldo;              // filters from aux_f0 on walk one tap only and go to aux_out; 0: none
  void* aux_out; unsigned aux_out_bytes;
  int split_f, split_ldo; unsigned ofs, split_ofs;    // filters from split_f on (F: none) go to rows of their own; bytes from `out`
  float inv_ohw, inv_ow, inv_tiles;
};

enum { kPoint = 0, kLines = 1, kAny = 2 };  // 1x1 without padding; taps of whole slabs (C % 64 == 0); any C % 8 == 0

template <int WP, int WF, int PB, int FB, int S, int MODE>
__global__ __launch_bounds__(64 * WP * WF) void conv_ring_kernel(const RingArgs a) {
  constexpr int NW = WP * WF, BP = 32 * WP * PB, BF = 32 * WF * FB, LP = BP / 8 / NW, LF = BF / 8 / NW;
  static_assert(BP % (8 * NW) == 0 && BF % (8 * NW) == 0, "whole load instructions per wave");
  constexpr int kStage = (BP + BF) * 128;
  constexpr int kPitch = FB * 64 + 16;               // bytes of a row of the outgoing tile
  constexpr int kRing = S * kStage > NW * PB * 32 * kPitch ? S * kStage : NW * PB * 32 * kPitch;
  extern __shared__ __align__(16) unsigned char smem[];  // ring, then scale[BF] and shift[BF]
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int wp = wave % WP, wf = wave / WP;
  int tf, tp;
  bool aux = false;
  if (MODE == kLines && a.aux_f0 > 0) {
    // XCD x takes a run of pixel tiles: all filters of the convolution over them, then the auxiliary ones, whose tiles are
    // short (in between they kept the long ones waiting: 94.6 us instead of 66.5 for 256x56x56x64 -> 128 + 128)
    const int per = (a.tiles_p + 7) >> 3, x = blockIdx.x & 7;
    int i = blockIdx.x >> 3;
    aux = i >= per * a.tiles_f;
    const int nf = aux ? a.aux_tiles : a.tiles_f;
    if (aux) i -= per * a.tiles_f;
    tp = i / nf;
    tf = i - tp * nf + (aux ? a.tiles_f : 0);
    tp += x * per;
    if (tp >= a.tiles_p) return;  // (uniform; before any barrier)
  } else {  // XCD x takes a contiguous run of tiles: its L2 holds a part of the larger operand only
    const int tiles = a.tiles_f * a.tiles_p, per = (tiles + 7) >> 3, rem = tiles & 7;
    const int x = blockIdx.x & 7, i = blockIdx.x >> 3;
    const int t = rem == 0 ? x * per + i : (x < rem ? x * per : rem * per + (x - rem) * (per - 1)) + i;
    if (a.pixels_first) tf = fast_div(t, a.tiles_p, a.inv_tiles, &tp);
    else tp = fast_div(t, a.tiles_f, a.inv_tiles, &tf);
  }
  tf = __builtin_amdgcn_readfirstlane(tf);
  tp = __builtin_amdgcn_readfirstlane(tp);
  const int p0 = tp * BP, f0 = tf * BF;
  const int fend = MODE == kLines && a.aux_f0 > 0 && !aux ? a.aux_f0 : a.F;
  const int act = aux ? a.aux_act : a.act;
  const __amdgpu_buffer_rsrc_t rs_in = make_rsrc(a.in, a.in_bytes);
  const __amdgpu_buffer_rsrc_t rs_wt = make_rsrc(a.wt, a.wt_bytes);

  float* ss = reinterpret_cast<float*>(smem + kRing);
  float ssv = 0.0f;
  if ((int)threadIdx.x < BF && f0 + (int)threadIdx.x < a.F) ssv = a.scale ? a.scale[f0 + threadIdx.x] : 1.0f;
  float shv = 0.0f;
  if ((int)threadIdx.x < BF && f0 + (int)threadIdx.x < a.F && a.shift) shv = a.shift[f0 + threadIdx.x];

  // ---- what this lane fetches: of row (wave * LP + i) * 8 + lane / 8 the chunk at position lane % 8 ----
  const int pos = lane & 7, sub = lane >> 3;
  auto column = [&](int group) { return pos ^ (((group & 1) << 2) + (sub >> 1)); };
  unsigned pbase[LP], wbase[LF];
  int py[LP], px[LP];
#pragma unroll
  for (int i = 0; i < LP; ++i) {
    const int group = wave * LP + i, p = p0 + group * 8 + sub;
    if constexpr (MODE == kPoint) {
      // (strided 1x1 windows read every stride-th pixel)
      int rem, x;
      const int n = fast_div(p < a.P ? p : 0, a.OHW, a.inv_ohw, &rem), y = fast_div(rem, a.OW, a.inv_ow, &x);
      pbase[i] = p < a.P ? (unsigned)(((n * a.H + y * a.stride_h) * a.W + x * a.stride_w) * a.pix * 2 + column(group) * 16) : kOOBr;
      py[i] = px[i] = 0;
    } else {
      int rem, x;
      const int n = fast_div(p < a.P ? p : 0, a.OHW, a.inv_ohw, &rem), y = fast_div(rem, a.OW, a.inv_ow, &x);
      py[i] = p < a.P ? y * a.stride_h - a.pad_h : -(1 << 28);
      px[i] = x * a.stride_w - a.pad_w;
      pbase[i] = (unsigned)((n * a.H * a.W + (y * a.stride_h - a.pad_h) * a.W + px[i]) * a.pix * 2 + (MODE == kLines ? column(group) * 16 : 0));
    }
  }
#pragma unroll
  for (int i = 0; i < LF; ++i) {
    const int group = wave * LF + i, f = f0 + group * 8 + sub;
    wbase[i] = f < a.F ? (unsigned)(f * a.chunks * 16 + column(group) * 16) : kOOBr;
  }
  // kAny: tap row, tap column and chunk inside the tap of this lane's chunk, for even and odd row groups
  int kr[2] = {0, 0}, ks[2] = {0, 0}, kc[2];
  auto settle = [&](int v) {
    while (kc[v] >= a.cpt) {
      kc[v] -= a.cpt;
      if (++ks[v] == a.S) ks[v] = 0, ++kr[v];
    }
  };
  if constexpr (MODE == kAny) {
#pragma unroll
    for (int v = 0; v < 2; ++v) kc[v] = column(v), settle(v);
  }
  int slab = 0, skr = 0, sks = 0, skc = 0;  // the slab to fetch next, and its tap (kLines)
  int nslab = (a.chunks + 7) >> 3;
  if (aux) {
    slab = a.aux_tap * (a.cpt >> 3);
    nslab = slab + (a.cpt >> 3);
    skr = a.aux_tap / a.S;
    sks = a.aux_tap - skr * a.S;
  }
  const int first = slab;
  auto fetch = [&](int buf) {
    unsigned char* dst = smem + buf * kStage;
    const bool tail = 8 * slab + 8 > a.chunks;
    const unsigned soff = (unsigned)slab * 128u;
#pragma unroll
    for (int i = 0; i < LP; ++i) {
      const int group = wave * LP + i;
      unsigned v;
      if constexpr (MODE == kPoint) {
        v = pbase[i];
        if (tail) v = 8 * slab + column(group) < a.chunks ? v : kOOBr;
      } else if constexpr (MODE == kLines) {
        const bool ok = ((unsigned)(py[i] + skr) < (unsigned)a.H) & ((unsigned)(px[i] + sks) < (unsigned)a.W);
        v = ok ? pbase[i] + (unsigned)((skr * a.W + sks) * a.pix * 2 + skc * 128) : kOOBr;
      } else {
        const int q = (LP & 1) ? group & 1 : i & 1;
        const int r = q ? kr[1] : kr[0], s = q ? ks[1] : ks[0], c = q ? kc[1] : kc[0];
        const bool ok = (8 * slab + column(group) < a.chunks) & ((unsigned)(py[i] + r) < (unsigned)a.H) & ((unsigned)(px[i] + s) < (unsigned)a.W);
        v = ok ? pbase[i] + (unsigned)((r * a.W + s) * a.pix * 2 + c * 16) : kOOBr;
      }
      fetch16(rs_in, dst + group * 1024, v, MODE == kPoint ? soff : 0u);
    }
#pragma unroll
    for (int i = 0; i < LF; ++i) {
      const int group = wave * LF + i;
      unsigned v = wbase[i];
      if (tail) v = 8 * slab + column(group) < a.chunks ? v : kOOBr;
      fetch16(rs_wt, dst + BP * 128 + group * 1024, v, soff);
    }
    ++slab;
    if constexpr (MODE == kLines) {
      if (8 * ++skc == a.cpt) {
        skc = 0;
        if (++sks == a.S) sks = 0, ++skr;
      }
    } else if constexpr (MODE == kAny) {
#pragma unroll
      for (int v = 0; v < 2; ++v) kc[v] += 8, settle(v);
    }
  };

  // ---- rows of the outgoing tile: 4 * FB lanes to a row; the residual's rows are requested now ----
  constexpr int kLanesRow = 4 * FB, kRowsInstr = 64 / kLanesRow, kOut = PB * 32 / kRowsInstr;
  const __amdgpu_buffer_rsrc_t rs_out = aux ? make_rsrc(a.aux_out, a.aux_out_bytes) : make_rsrc(a.out, a.out_bytes);
  const bool residual = a.residual != nullptr && !aux;
  const int orow = lane / kLanesRow, ochan = (lane % kLanesRow) * 8;
  unsigned oofs[kOut];
  u32x4 rv[kOut];
#pragma unroll
  for (int o = 0; o < kOut; ++o) {
    const int p = p0 + wp * PB * 32 + o * kRowsInstr + orow, f = f0 + wf * FB * 32 + ochan;
    oofs[o] = p < a.P && f < fend ? (unsigned)(aux ? p * a.aux_ldo + f - a.aux_f0 : p * a.ldo + f) * 2u : kOOBr;
    if (MODE == kPoint && p < a.P && f < fend) oofs[o] = f < a.split_f ? oofs[o] + a.ofs : (unsigned)(p * a.split_ldo + f - a.split_f) * 2u + a.split_ofs;
  }
  if (residual) {
    const __amdgpu_buffer_rsrc_t rs_res = make_rsrc(a.residual, a.out_bytes);
#pragma unroll
    for (int o = 0; o < kOut; ++o) rv[o] = __builtin_amdgcn_raw_buffer_load_b128(rs_res, oofs[o], 0, 0);
  }
  fetch(0);
  if ((int)threadIdx.x < BF) ss[threadIdx.x] = ssv, ss[BF + threadIdx.x] = shv;

  floatx16 acc[FB][PB];
#pragma unroll
  for (int i = 0; i < FB; ++i)
#pragma unroll
    for (int j = 0; j < PB; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

  // operand reads: row lane % 32 of a block, chunk 2 k + lane / 32 at position chunk ^ (row / 2) % 8
  const int lrow = lane & 31, lh = lane >> 5, key = (lrow >> 1) & 7;
  const unsigned char* prow = smem + (wp * PB * 32 + lrow) * 128;
  const unsigned char* wrow = smem + (BP + wf * FB * 32 + lrow) * 128;
  for (int s = first; s < nslab; ++s) {
    const int buf = S == 2 ? (s - first) & 1 : 0;
    __builtin_amdgcn_s_waitcnt(kAllLanded);
    __syncthreads();
    if (S == 2 && s + 1 < nslab) fetch(buf ^ 1);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int at = buf * kStage + (((2 * k + lh) ^ key) * 16);
      u32x4 w[FB], p[PB];
#pragma unroll
      for (int i = 0; i < FB; ++i) w[i] = *reinterpret_cast<const u32x4*>(wrow + at + i * 4096);
#pragma unroll
      for (int j = 0; j < PB; ++j) p[j] = *reinterpret_cast<const u32x4*>(prow + at + j * 4096);
#pragma unroll
      for (int i = 0; i < FB; ++i)
#pragma unroll
        for (int j = 0; j < PB; ++j) Mma<half_t>::run(w[i], p[j], acc[i][j]);
    }
    if (S == 1 && s + 1 < nslab) {
      __syncthreads();
      fetch(0);
    }
  }
  __syncthreads();

  // ---- out: this wave's tile [PB * 32 pixels][FB * 32 channels] ----
  unsigned char* tile = smem + wave * (PB * 32 * kPitch);
  if (residual) {
#pragma unroll
    for (int o = 0; o < kOut; ++o) *reinterpret_cast<u32x4*>(tile + (o * kRowsInstr + orow) * kPitch + ochan * 2) = rv[o];
  }
  const float* sc = ss + wf * FB * 32;
#pragma unroll
  for (int i = 0; i < FB; ++i)
#pragma unroll
    for (int j = 0; j < PB; ++j) {
      float y[16], r[16];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const floatx4 m = *reinterpret_cast<const floatx4*>(sc + i * 32 + 8 * q + 4 * lh), h = *reinterpret_cast<const floatx4*>(sc + BF + i * 32 + 8 * q + 4 * lh);
#pragma unroll
        for (int e = 0; e < 4; ++e) y[4 * q + e] = acc[i][j][4 * q + e] * m[e] + h[e];
      }
      unsigned char* at = tile + (j * 32 + lrow) * kPitch + i * 64 + lh * 8;
      if (residual) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const half4 x = *reinterpret_cast<const half4*>(at + q * 16);
#pragma unroll
          for (int e = 0; e < 4; ++e) r[4 * q + e] = (float)x[e];
        }
        if (!(act & kActResidualAfter)) {
#pragma unroll
          for (int e = 0; e < 16; ++e) y[e] += r[e];
        }
      }
      act_apply_n<true>(y, act & 0xff);
      if (residual && (act & kActResidualAfter)) {
#pragma unroll
        for (int e = 0; e < 16; ++e) y[e] += r[e];
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        half4 x;
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = (half_t)y[4 * q + e];
        *reinterpret_cast<half4*>(at + q * 16) = x;
      }
    }
#pragma unroll
  for (int o = 0; o < kOut; ++o) {
    const u32x4 v = *reinterpret_cast<const u32x4*>(tile + (o * kRowsInstr + orow) * kPitch + ochan * 2);
    __builtin_amdgcn_raw_buffer_store_b128(v, rs_out, oofs[o], 0, 0);
  }
}

// ---- dispatch

template <int WP, int WF, int PB, int FB, int S>
void launch_cfg(RingArgs d, int mode, hipStream_t s) {
  constexpr int NW = WP * WF, BP = 32 * WP * PB, BF = 32 * WF * FB, ring = S * (BP + BF) * 128, tile = NW * PB * 32 * (FB * 64 + 16);
  constexpr int lds = (ring > tile ? ring : tile) + BF * 8;
  const int main_f = d.aux_f0 ? d.aux_f0 : d.F;
  d.tiles_f = (main_f + BF - 1) / BF;
  d.aux_tiles = (d.F - main_f + BF - 1) / BF;
  d.tiles_p = (d.P + BP - 1) / BP;
  d.inv_tiles = 1.0f / (float)(d.pixels_first ? d.tiles_p : d.tiles_f);
  auto go = [&](auto kern) {
    static const bool attr = [&] {
      if (lds > 65536) NNCV_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, lds));
      return true;
    }();
    (void)attr;
    launch_kernel(kern, dim3((unsigned)(d.aux_f0 ? (d.tiles_p + 7) / 8 * 8 * (d.tiles_f + d.aux_tiles) : d.tiles_f * d.tiles_p)), dim3(64 * NW), lds, s, d);
  };
  if (mode == kPoint) go(conv_ring_kernel<WP, WF, PB, FB, S, kPoint>);
  else if (mode == kLines) go(conv_ring_kernel<WP, WF, PB, FB, S, kLines>);
  else go(conv_ring_kernel<WP, WF, PB, FB, S, kAny>);
}

// The forms, and what a launch of each takes: us = fixed + ((busy)^3 + (chain)^3)^(1/3) with
//   busy  = tiles / 256 CUs * (slab_us * slabs + tile_us)            (LDS, matrix and memory pipes)
//   chain = ceil(tiles / (256 * resident)) * chain_us * slabs        (a slab's latency, workgroups of a CU one after the other)
// slab_us and chain_us grow by slab_any and chain_any where the taps are not whole slabs.  Fits over 300 layers of 1x1 to 7x7
// windows, 8 to 1024 channels; the form they choose is within 1.5 % of the best one on average.
struct Form {
  int bp, bf, resident;
  double fixed_us, slab_us, tile_us, chain_us, slab_any, chain_any;
  void (*launch)(RingArgs, int, hipStream_t);
  const char* tag;
};
const Form kForms[] = {
    {64, 64, 7, 2.58, 0.220, 0.287, 0.405, 0.26, 0.18, launch_cfg<2, 2, 1, 1, 1>, "conv_ring<64x64>"},
    {64, 64, 4, 2.72, 0.233, 0.353, 0.350, 0.26, 0.38, launch_cfg<2, 2, 1, 1, 2>, "conv_ring<64x64,2>"},
    {64, 32, 13, 2.71, 0.144, 0.180, 0.423, 0.24, 0.26, launch_cfg<2, 1, 1, 1, 1>, "conv_ring<64x32>"},
    {64, 128, 3, 3.04, 0.353, 0.620, 0.434, 0.11, 0.37, launch_cfg<2, 2, 1, 2, 2>, "conv_ring<64x128,2>"},
    {128, 128, 2, 2.94, 0.626, 1.086, 0.631, 0.11, 0.11, launch_cfg<4, 2, 1, 2, 1>, "conv_ring<128x128>"},
    {128, 128, 2, 3.08, 0.583, 1.142, 0.515, 0.21, 0.48, launch_cfg<4, 2, 1, 2, 2>, "conv_ring<128x128,2>"},
};

const Form* best_form(const IgemmArgs& a, double* us) {
  const double P = (double)a.N * a.OH * a.OW, slabs = std::ceil(a.R * a.S * a.C / 64.0);
  const bool any = a.R * a.S > 1 && a.C % 64 != 0;
  const Form* best = nullptr;
  for (const Form& f : kForms) {
    const double fs = a.aux_f0 ? a.aux_f0 + (double)(a.F - a.aux_f0) / (a.R * a.S) : a.F;  // auxiliary filters walk one tap
    const double x = std::ceil(P / f.bp) * std::ceil(fs / f.bf) / 256;
    const double busy = x * (f.slab_us * slabs * (any ? 1 + f.slab_any : 1) + f.tile_us);
    const double chain = std::ceil(x / f.resident) * f.chain_us * slabs * (any ? 1 + f.chain_any : 1);
    const double v = f.fixed_us + std::cbrt(busy * busy * busy + chain * chain * chain);
    if (!best || v < *us) best = &f, *us = v;
  }
  return best;
}

}  // namespace

// Windows over 8 channels stay with the generic kernel: a slab then spans eight taps, each with its own address arithmetic
// (16x16x8 -> 8 at 3x3: 3.1 us there, 5.0 here; from 16 channels on this kernel is level or ahead).
bool conv_ring_applicable(const IgemmArgs& a, int in_dt, int out_dt) {
  const int pix = a.pix_stride ? a.pix_stride : a.C;
  const long long P = (long long)a.N * a.OH * a.OW, k = (long long)a.R * a.S * a.C, lim = 1 << 24;  // fast_div's range
  const bool aux_ok = a.aux_f0 == 0 || (a.aux_f0 % 128 == 0 && a.C % 64 == 0 && a.R * a.S > 1 && a.aux_tap >= 0 && a.aux_tap < a.R * a.S && a.aux_out &&
                                        a.aux_ldo % 8 == 0 && P * a.aux_ldo * 2 < (long long)kOOBr);
  // (two results: one range of bytes that holds both)
  const long long reach = (a.split_ofs < 0 ? -a.split_ofs : a.split_ofs) + P * (a.ldo > a.split_ldo ? a.ldo : a.split_ldo) * 2;
  const bool split_ok = a.split_f == 0 || (a.split_f % 8 == 0 && a.split_ldo % 8 == 0 && a.split_ofs % 16 == 0 && reach < (long long)kOOBr && !a.residual &&
                                           a.aux_f0 == 0 && a.R * a.S == 1 && a.pad_h == 0 && a.pad_w == 0);
  return in_dt == kF16 && out_dt == kF16 && a.batch == 1 && aux_ok && split_ok && a.C % 8 == 0 && (a.R * a.S == 1 || a.C >= 16) && pix % 8 == 0 &&
         a.F % 8 == 0 && a.ldo % 8 == 0 && P < lim && k < lim && a.in_bytes > 0 && a.in_bytes < kOOBr &&
         (long long)a.N * a.H * a.W * pix * 2 < (long long)kOOBr && (long long)a.F * k * 2 < (long long)kOOBr &&
         P * a.ldo * 2 < (long long)kOOBr && ((P + 63) / 64) * ((a.F + 31) / 32) < lim && (a.relu & ~(0xff | kActResidualAfter)) == 0;
}

// Stride-2 3x3 layers leave the patch kernel where 128 x 128 tiles keep three quarters of the CUs busy.  From 200 tiles to the
// patch kernel's limit (8 GFLOP) that kernel is bound by its patch reads: 48x56x56x64 -> 128 14.3 against 13.3 us here, 64
// images 17.4 against 14.1, 32x40x40x128 -> 256 20.0 against 15.9, 16x80x80x64 -> 128 10.2 against 10.3 at 200 tiles.  Below, its
// smaller tiles and K groups mostly fill the chip better (32x28x28x128 -> 256, 98 tiles: 9.1 against 11.6; 24x40x40x128 -> 256,
// 150 tiles, is the other way round: 16.5 against 15.1).  Larger launches used to be igemm_fast's: 23 of them take 1.14 to 1.35
// times as long there (256x28x28x128 -> 256: 52.2 against 42.0).  In a ResNet-18 pass of 256 images the three such layers with
// their shortcuts went from 78.1 + 58.4 + 52.2 us there to 65.4 + 46.6 + 43.6, the pass from 1162 to 1133 us of launches.
bool conv_ring_beats_patch_s2(const IgemmArgs& a) {
  const long long P = (long long)a.N * a.OH * a.OW, main_f = a.aux_f0 ? a.aux_f0 : a.F;
  return a.stride_h == 2 && (P + 127) / 128 * ((main_f + 127) / 128) >= 200;
}

double conv_ring_us(const IgemmArgs& a) {
  double us = 0;
  best_form(a, &us);
  return us;
}

void launch_conv_ring(const IgemmArgs& a, hipStream_t s) {
  RingArgs d{};
  d.in = a.in; d.wt = a.wt; d.out = a.out; d.scale = a.scale; d.shift = a.shift; d.residual = a.residual;
  d.pix = a.pix_stride ? a.pix_stride : a.C;
  d.chunks = a.R * a.S * a.C / 8; d.cpt = a.C / 8;
  d.H = a.H; d.W = a.W; d.F = a.F; d.S = a.S; d.OW = a.OW; d.OHW = a.OH * a.OW; d.P = a.N * d.OHW;
  d.in_bytes = a.in_bytes; d.wt_bytes = (unsigned)d.F * d.chunks * 16u; d.out_bytes = (unsigned)d.P * a.ldo * 2u;
  d.stride_h = a.stride_h; d.stride_w = a.stride_w; d.pad_h = a.pad_h; d.pad_w = a.pad_w;
  d.act = a.relu; d.ldo = a.ldo;
  d.split_f = a.F;
  if (a.split_f) {
    const long long low = a.split_ofs < 0 ? a.split_ofs : 0;
    d.split_f = a.split_f; d.split_ldo = a.split_ldo; d.ofs = (unsigned)-low; d.split_ofs = (unsigned)(a.split_ofs - low);
    d.out = static_cast<char*>(a.out) + low;
    const unsigned e0 = d.ofs + (unsigned)d.P * a.ldo * 2u, e1 = d.split_ofs + (unsigned)d.P * a.split_ldo * 2u;
    d.out_bytes = e0 > e1 ? e0 : e1;
  }
  if (a.aux_f0) {
    d.aux_f0 = a.aux_f0; d.aux_tap = a.aux_tap; d.aux_act = a.aux_relu; d.aux_ldo = a.aux_ldo; d.aux_out = a.aux_out;
    d.aux_out_bytes = (unsigned)d.P * a.aux_ldo * 2u;
  }
  d.inv_ohw = 1.0f / (float)d.OHW; d.inv_ow = 1.0f / (float)d.OW;
  d.pixels_first = d.wt_bytes > d.in_bytes;
  double us = 0;
  const Form* f = best_form(a, &us);
  const double flops = a.alg_flops > 0 ? a.alg_flops : 2.0 * d.P * (double)a.F * a.R * a.S * a.C;
  ProfScope prof(f->tag, flops, 2.0 * ((double)a.N * a.H * a.W * a.C + (double)a.F * a.R * a.S * a.C + (double)d.P * a.F * (a.residual ? 2 : 1)), s);
  f->launch(d, a.R * a.S == 1 && a.pad_h == 0 && a.pad_w == 0 ? kPoint : a.C % 64 == 0 ? kLines : kAny, s);
  NNCV_HIP_CHECK(hipGetLastError());
}

}  // namespace nncv_hip
