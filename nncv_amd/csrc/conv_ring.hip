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
  const void* chain_wt; const float* chain_scale; const float* chain_shift; void* chain_out;  // the layer behind the first result (CH > 0)
  unsigned chain_bytes; int chain_act, chain_ldo, chain_only;
  const void* up_in; unsigned up_bytes; int up_slabs, up_pix;                                 // slabs that come from another tensor (UP)
  const void* wfrag; const void* aux_wfrag; int groups, aux_groups, lead;  // the resident form's filters: 32-filter groups; bytes of padding
};

enum { kPoint = 0, kLines = 1, kAny = 2 };  // 1x1 without padding; taps of whole slabs (C % 64 == 0); any C % 8 == 0

// CH > 0: of two results the first one, 16 * CH channels, is the input of a further 1x1 layer with as many filters.  Its values are in LDS on
// their way out, rounded; the workgroups that have all its channels multiply them there.
// UP: the first slabs are those of a tensor of half the size, whose up-sampled copy is never made.
template <int WP, int WF, int PB, int FB, int S, int MODE, int CH = 0, bool UP = false>
__global__ __launch_bounds__(64 * WP * WF) void conv_ring_kernel(const RingArgs a) {
  constexpr int kChain = 16 * CH, NB = CH / (2 * WF) > 0 ? CH / (2 * WF) : 1;  // blocks of 32 of those filters a wave takes
  static_assert(CH == 0 || (PB == 1 && MODE == kPoint && kChain <= 32 * WF * FB), "a tile has all channels of the first result");
  constexpr int NW = WP * WF, BP = 32 * WP * PB, BF = 32 * WF * FB, LP = BP / 8 / NW, LF = BF / 8 / NW;
  static_assert(BP % (8 * NW) == 0 && BF % (8 * NW) == 0, "whole load instructions per wave");
  constexpr int kStage = (BP + BF) * 128;
  constexpr int kPitch = FB * 64 + 16;               // bytes of a row of the outgoing tile
  constexpr int kRing = S * kStage > NW * PB * 32 * kPitch ? S * kStage : NW * PB * 32 * kPitch;
  extern __shared__ __align__(16) unsigned char smem[];  // ring, then scale[BF] and shift[BF]
  // all arguments at once: fetched where they are first used, they are one wait after the other
  asm volatile("" ::"s"(a.in), "s"(a.wt), "s"(a.scale), "s"(a.shift), "s"(a.residual), "s"(a.in_bytes), "s"(a.wt_bytes), "s"(a.H), "s"(a.W), "s"(a.F), "s"(a.OW),
               "s"(a.OHW), "s"(a.P), "s"(a.pix), "s"(a.stride_h), "s"(a.stride_w), "s"(a.chunks), "s"(a.cpt), "s"(a.tiles_f), "s"(a.tiles_p), "s"(a.aux_f0),
               "s"(a.inv_ohw), "s"(a.inv_ow), "s"(a.inv_tiles));
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

  // ---- what this lane fetches: of row (wave * LP + i) * 8 + lane / 8 the chunk at position lane % 8 ----
  const int pos = lane & 7, sub = lane >> 3;
  auto column = [&](int group) { return pos ^ (((group & 1) << 2) + (sub >> 1)); };
  unsigned wbase[LF];
#pragma unroll
  for (int i = 0; i < LF; ++i) {
    const int group = wave * LF + i, f = f0 + group * 8 + sub;
    wbase[i] = f < a.F ? (unsigned)(f * a.chunks * 16 + column(group) * 16) : kOOBr;
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
  auto fetch_filters = [&](int buf) __attribute__((always_inline)) {
    const bool tail = 8 * slab + 8 > a.chunks;
#pragma unroll
    for (int i = 0; i < LF; ++i) {
      const int group = wave * LF + i;
      unsigned v = wbase[i];
      if (tail) v = 8 * slab + column(group) < a.chunks ? v : kOOBr;
      fetch16(rs_wt, smem + buf * kStage + BP * 128 + group * 1024, v, (unsigned)slab * 128u);
    }
  };
  fetch_filters(0);  // the filters' addresses are there long before the pixels' (59 layers: 1.015x on average, 3.05 -> 2.97 us for small ones)
  __builtin_amdgcn_sched_barrier(0);
  float* ss = reinterpret_cast<float*>(smem + kRing);
  float ssv = 0.0f;
  if ((int)threadIdx.x < BF && f0 + (int)threadIdx.x < a.F) ssv = a.scale ? a.scale[f0 + threadIdx.x] : 1.0f;
  float shv = 0.0f;
  if ((int)threadIdx.x < BF && f0 + (int)threadIdx.x < a.F && a.shift) shv = a.shift[f0 + threadIdx.x];

  unsigned pbase[LP], ubase[UP ? LP : 1];
  int py[LP], px[LP];
  const __amdgpu_buffer_rsrc_t rs_up = make_rsrc(UP ? a.up_in : a.in, UP ? a.up_bytes : 0u);
#pragma unroll
  for (int i = 0; i < LP; ++i) {
    const int group = wave * LP + i, p = p0 + group * 8 + sub;
    if constexpr (UP) {
      int rem, x;
      const int n = fast_div(p < a.P ? p : 0, a.OHW, a.inv_ohw, &rem), y = fast_div(rem, a.OW, a.inv_ow, &x);
      const int from = (n * (a.H >> 1) + (y >> 1)) * (a.W >> 1) + (x >> 1);
      ubase[i] = p < a.P ? (unsigned)(from * a.up_pix * 2 + column(group) * 16) : kOOBr;
    }
    if constexpr (MODE == kPoint) {
      int at = p;  // result p reads pixel p (40 layers: 1.03x on average without the divisions, 7.1 -> 6.7 us for 64 -> 64 channels at 16x80x80)
      if ((a.stride_h | a.stride_w) != 1) {  // strided windows read every stride-th pixel
        int rem, x;
        const int n = fast_div(p < a.P ? p : 0, a.OHW, a.inv_ohw, &rem), y = fast_div(rem, a.OW, a.inv_ow, &x);
        at = (n * a.H + y * a.stride_h) * a.W + x * a.stride_w;
      }
      pbase[i] = p < a.P ? (unsigned)(at * a.pix * 2 + column(group) * 16) : kOOBr;
      py[i] = px[i] = 0;
    } else {
      int rem, x;
      const int n = fast_div(p < a.P ? p : 0, a.OHW, a.inv_ohw, &rem), y = fast_div(rem, a.OW, a.inv_ow, &x);
      py[i] = p < a.P ? y * a.stride_h - a.pad_h : -(1 << 28);
      px[i] = x * a.stride_w - a.pad_w;
      pbase[i] = (unsigned)((n * a.H * a.W + (y * a.stride_h - a.pad_h) * a.W + px[i]) * a.pix * 2 + (MODE == kLines ? column(group) * 16 : 0));
    }
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
  auto fetch_pixels = [&](int buf) __attribute__((always_inline)) {
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
      if (UP && slab < a.up_slabs) fetch16(rs_up, dst + group * 1024, ubase[UP ? i : 0], soff);
      else fetch16(rs_in, dst + group * 1024, v, MODE == kPoint ? soff : 0u);
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
    if (CH > 0 && a.chain_only && f < a.split_f) oofs[o] = kOOBr;
    else if (MODE == kPoint && p < a.P && f < fend) oofs[o] = f < a.split_f ? oofs[o] + a.ofs : (unsigned)(p * a.split_ldo + f - a.split_f) * 2u + a.split_ofs;
  }
  if (residual) {
    const __amdgpu_buffer_rsrc_t rs_res = make_rsrc(a.residual, a.out_bytes);
#pragma unroll
    for (int o = 0; o < kOut; ++o) rv[o] = __builtin_amdgcn_raw_buffer_load_b128(rs_res, oofs[o], 0, 0);
  }
  fetch_pixels(0);
  if constexpr (CH > 0) {
    if ((int)threadIdx.x < kChain) {
      ss[2 * BF + threadIdx.x] = a.chain_scale ? a.chain_scale[threadIdx.x] : 1.0f;
      ss[2 * BF + kChain + threadIdx.x] = a.chain_shift ? a.chain_shift[threadIdx.x] : 0.0f;
    }
  }
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
    if (S == 2 && s + 1 < nslab) fetch_filters(buf ^ 1), fetch_pixels(buf ^ 1);
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
      fetch_filters(0);
      fetch_pixels(0);
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
  const int cf0 = wf * NB * 32;  // this wave's filters of the chained layer
  const bool chained = CH > 0 && tf == 0 && cf0 < kChain;
  u32x4 cw[CH > 0 ? CH : 1][NB];
  if constexpr (CH > 0) {
    const __amdgpu_buffer_rsrc_t rs_c = make_rsrc(a.chain_wt, (unsigned)(kChain * kChain) * 2u);
#pragma unroll
    for (int k = 0; k < CH; ++k)
#pragma unroll
      for (int b = 0; b < NB; ++b)
        cw[k][b] = __builtin_amdgcn_raw_buffer_load_b128(rs_c, chained ? (unsigned)((cf0 + b * 32 + lrow) * kChain + k * 16 + lh * 8) * 2u : kOOBr, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll
  for (int o = 0; o < kOut; ++o) {
    const u32x4 v = *reinterpret_cast<const u32x4*>(tile + (o * kRowsInstr + orow) * kPitch + ochan * 2);
    __builtin_amdgcn_raw_buffer_store_b128(v, rs_out, oofs[o], 0, 0);
  }
  if constexpr (CH > 0) {
    if (tf != 0) return;  // (uniform)
    __syncthreads();
    floatx16 z[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int e = 0; e < 16; ++e) z[b][e] = 0.0f;
#pragma unroll
    for (int k = 0; k < CH; ++k) {  // channels 16 k + 8 lh .. of pixel lrow: in the tile of the wave whose filters they were
      const u32x4 x = *reinterpret_cast<const u32x4*>(smem + (wp + WP * (16 * k / (32 * FB))) * (32 * kPitch) + lrow * kPitch + (16 * k % (32 * FB) + 8 * lh) * 2);
#pragma unroll
      for (int b = 0; b < NB; ++b) Mma<half_t>::run(cw[k][b], x, z[b]);
    }
    __syncthreads();
    if (!chained) return;
    constexpr int kLanes = 4 * NB, kRows = 64 / kLanes, kPitchC = NB * 64 + 16;
    const float* sc = ss + 2 * BF + cf0;
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      float y[16];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const floatx4 m = *reinterpret_cast<const floatx4*>(sc + b * 32 + 8 * q + 4 * lh), h = *reinterpret_cast<const floatx4*>(sc + kChain + b * 32 + 8 * q + 4 * lh);
#pragma unroll
        for (int e = 0; e < 4; ++e) y[4 * q + e] = z[b][4 * q + e] * m[e] + h[e];
      }
      act_apply_n<true>(y, a.chain_act);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        half4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = (half_t)y[4 * q + e];
        *reinterpret_cast<half4*>(tile + lrow * kPitchC + b * 64 + q * 16 + lh * 8) = v;
      }
    }
    const __amdgpu_buffer_rsrc_t rs_co = make_rsrc(a.chain_out, a.chain_bytes);
#pragma unroll
    for (int o = 0; o < 32 / kRows; ++o) {
      const int r = o * kRows + lane / kLanes, c = (lane % kLanes) * 8, p = p0 + wp * 32 + r;
      const u32x4 v = *reinterpret_cast<const u32x4*>(tile + r * kPitchC + c * 2);
      __builtin_amdgcn_raw_buffer_store_b128(v, rs_co, p < a.P ? (unsigned)(p * a.chain_ldo + cf0 + c) * 2u : kOOBr, 0, 0);
    }
  }
}

// 3x3 windows over whole slabs of channels: the pixels go through a ring of four slabs, the filters straight from memory into
// registers (fragments in weight_frag3x3's order, eight K steps ahead).  Four waves take 32 filters each of BP x 128 outputs, so a
// K step is PB products on one fragment and PB LDS reads: per 128 x 128 x 64 products LDS takes 16 KB of pixels and gives 64 KB, where
// the ring above takes 32 and gives 96 (LDS takes 80 and gives 256 bytes a clock).  A slab is fetched three stages ahead, and one
// barrier a stage says both that it is there and that the one before it may go.
//  * Slab outer, tap inner: of nine taps three or four bring lines that the others have not.
//  * Whether a pixel has the tap is one bit per tap and row of the tile; the tap's offset is the scalar part of the address.
//  * Auxiliary filters (AUX) are a second set of sums: the centre tap's pixels are their operands.
//  * What bounds it: nothing alone.  22x49x58x512 -> 512 takes 75 us (1000 TFLOP/s; 88 in the ring above), 70 without the filters'
//    loads, 62 without the pixels', 65 without the LDS reads, 50 without the products: a wave issues all of them in turn.
// Times against the ring's 128 x 128 form or, below 200 tiles, conv3x3_patch.hip: 16x40x40x256 -> 512 27.1 -> 21.7 us, 16x160x160x64 ->
// 128 29.0 -> 25.8, 16x40x40x256 -> 256 20.2 -> 13.3, 33x25x106x64 -> 128 14.0 -> 8.6.
// POINT: 1x1 layers, one stage to a slab (point_us).
template <int PB, bool AUX, bool POINT = false>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(PB == 4 ? 2 : 3, PB == 4 ? 2 : 4))) void conv_ring_frag_kernel(const RingArgs a) {
  constexpr int BP = 32 * PB, BF = 128, kStage = BP * 128, kStages = 4, kRing = 8;
  constexpr int kPitch = 272, kLds = kStages * kStage > BP * kPitch ? kStages * kStage : BP * kPitch;
  constexpr int kWait = ((8 + 2 * PB) & 15) | (((8 + 2 * PB) >> 4) << 14) | 0x0f70;
  extern __shared__ __align__(16) unsigned char smem[];  // ring, then scale[BF] and shift[BF]
  asm volatile("" ::"s"(a.in), "s"(a.wfrag), "s"(a.aux_wfrag), "s"(a.scale), "s"(a.shift), "s"(a.H), "s"(a.W), "s"(a.OW), "s"(a.OHW), "s"(a.P), "s"(a.pix), "s"(a.F),
               "s"(a.tiles_f), "s"(a.tiles_p), "s"(a.aux_tiles), "s"(a.aux_f0), "s"(a.groups), "s"(a.inv_ohw), "s"(a.inv_ow), "s"(a.inv_tiles), "s"(a.lead));
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  int tf, tp;
  {
    const int tiles = a.tiles_f * a.tiles_p, per = (tiles + 7) >> 3, rem = tiles & 7;
    const int x = blockIdx.x & 7, i = blockIdx.x >> 3;
    const int t = rem == 0 ? x * per + i : (x < rem ? x * per : rem * per + (x - rem) * (per - 1)) + i;
    if (a.pixels_first) tf = fast_div(t, a.tiles_p, a.inv_tiles, &tp);
    else tp = fast_div(t, a.tiles_f, a.inv_tiles, &tf);
  }
  tf = __builtin_amdgcn_readfirstlane(tf);
  tp = __builtin_amdgcn_readfirstlane(tp);
  const int p0 = tp * BP, f0 = tf * BF, fend = AUX ? a.aux_f0 : a.F;

  // ---- filters: fragment (group g, stage st, sub-step kk) is the kilobyte ((g / 2 * stages + st) * 4 + kk) * 2 + g % 2 ----
  const int nslab = a.cpt >> 3, T = POINT ? nslab : nslab * 9;
  const int g = min(tf * 4 + wave, a.groups - 1);  // (filters that are not there: the last ones again)
  const __amdgpu_buffer_rsrc_t rs_w = make_rsrc(a.wfrag, (unsigned)(a.groups >> 1) * T * 8192u);
  unsigned woff = (unsigned)((g >> 1) * T * 8192 + (g & 1) * 1024 + lane * 16);
  u32x4 wring[kRing];
  auto wload = [&](int step) __attribute__((always_inline)) { return __builtin_amdgcn_raw_buffer_load_b128(rs_w, woff + step * 2048, 0, 0); };  // step: from this stage on

  // auxiliary filters: this slab's four fragments (their order is that of one-tap filters)
  const int ga = AUX ? min(tf * 4 + wave, a.aux_groups - 1) : 0;
  const __amdgpu_buffer_rsrc_t rs_a = make_rsrc(AUX ? a.aux_wfrag : a.wfrag, AUX ? (unsigned)(a.aux_groups >> 1) * nslab * 8192u : 0u);
  unsigned aoff = (unsigned)((ga >> 1) * nslab * 8192 + (ga & 1) * 1024 + lane * 16);
  u32x4 waux[4];
  auto load_aux = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < 4; ++k) waux[k] = __builtin_amdgcn_raw_buffer_load_b128(rs_a, aoff + k * 2048, 0, 0);
    aoff += 8192;
  };

  // ---- pixels: of row (wave * PB + i) * 8 + lane / 8 the chunk at position lane % 8; bit 3 r + s of `valid`: tap (r, s) is inside ----
  const int pos = lane & 7, sub = lane >> 3;
  const __amdgpu_buffer_rsrc_t rs_in = make_rsrc(static_cast<const char*>(a.in) - a.lead, a.in_bytes + a.lead);
  unsigned pbase[PB], valid[PB];
#pragma unroll
  for (int i = 0; i < PB; ++i) {
    const int group = wave * PB + i, p = p0 + group * 8 + sub;
    if constexpr (POINT) {  // result p reads pixel p
      pbase[i] = p < a.P ? (unsigned)(p * a.pix * 2 + (pos ^ (((group & 1) << 2) + (sub >> 1))) * 16) : kOOBr;
      valid[i] = 1u;
      continue;
    }
    int rem, x;
    const int n = fast_div(p < a.P ? p : 0, a.OHW, a.inv_ohw, &rem), y = fast_div(rem, a.OW, a.inv_ow, &x);
    const int yy = y * a.stride_h, xx = x * a.stride_w;
    pbase[i] = (unsigned)(((n * a.H + yy) * a.W + xx) * a.pix * 2 + (pos ^ (((group & 1) << 2) + (sub >> 1))) * 16);
    const unsigned cols = (xx >= 1 ? 1u : 0u) | 2u | (xx + 1 < a.W ? 4u : 0u);
    valid[i] = p < a.P ? (yy >= 1 ? cols : 0u) | cols << 3 | (yy + 1 < a.H ? cols << 6 : 0u) : 0u;
  }
  const int pixB = a.pix * 2, rowB = (a.W - 2) * pixB, turnB = 128 - (2 * a.W + 2) * pixB;
  int ptap = 0, pleft = T, poff = 0;  // the stage to fetch next
  auto fetch = [&](int buf) __attribute__((always_inline)) {
    if constexpr (POINT) {
#pragma unroll
      for (int i = 0; i < PB; ++i) {
        const unsigned at = pbase[i], v = pleft > 0 ? at : kOOBr;
        fetch16(rs_in, smem + buf * kStage + (wave * PB + i) * 1024, v, (unsigned)poff);
      }
      --pleft;
      poff += 128;
      return;
    }
    const unsigned bit = pleft > 0 ? 1u << ptap : 0u;
#pragma unroll
    for (int i = 0; i < PB; ++i) {
      const unsigned at = pbase[i], v = valid[i] & bit ? at : kOOBr;
      fetch16(rs_in, smem + buf * kStage + (wave * PB + i) * 1024, v, (unsigned)poff);
    }
    --pleft;
    // (locals: of captured variables hipcc 7.2 chooses the address, in scratch)
    const int next = ptap + 1, row = rowB, pix = pixB, back = turnB;
    int step = next == 3 || next == 6 ? row : pix;
    step = next == 9 ? back : step;
    poff = __builtin_amdgcn_readfirstlane(poff + step);
    ptap = __builtin_amdgcn_readfirstlane(next == 9 ? 0 : next);
  };

  __builtin_amdgcn_sched_barrier(0);
  fetch(0);
#pragma unroll
  for (int q = 0; q < 4; ++q) wring[q] = wload(q);
  fetch(1);
#pragma unroll
  for (int q = 4; q < 8; ++q) wring[q] = wload(q);
  if constexpr (AUX) load_aux();
  fetch(2);
  // threads 0 .. 127: the filters' scale and shift; 128 .. 255: the auxiliary ones'
  const bool second = (int)threadIdx.x >= BF;
  const unsigned ssf = (unsigned)((second ? a.aux_f0 - BF : 0) + f0 + (int)threadIdx.x) * 4u;
  const __amdgpu_buffer_rsrc_t rs_sc = make_rsrc(a.scale, a.scale ? (unsigned)a.F * 4u : 0u), rs_sh = make_rsrc(a.shift, a.shift ? (unsigned)a.F * 4u : 0u);
  const unsigned scv = __builtin_amdgcn_raw_buffer_load_b32(rs_sc, ssf, 0, 0), shv = __builtin_amdgcn_raw_buffer_load_b32(rs_sh, ssf, 0, 0);
  __builtin_amdgcn_sched_barrier(0);

  floatx16 acc[PB], acc2[AUX ? PB : 1];
#pragma unroll
  for (int j = 0; j < PB; ++j)
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      acc[j][e] = 0.0f;
      if constexpr (AUX) acc2[j][e] = 0.0f;
    }
  int tap = 0;
  const int lrow = lane & 31, lh = lane >> 5, key = (lrow >> 1) & 7;
  const unsigned char* prow[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) prow[k] = smem + lrow * 128 + (((2 * k + lh) ^ key) * 16);
  u32x4 pr[2][PB];
  auto stage = [&](auto u_c) __attribute__((always_inline)) {
    constexpr int u = decltype(u_c)::value;
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(kWait);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < PB; ++j) pr[0][j] = *reinterpret_cast<const u32x4*>(prow[0] + u * kStage + j * 4096);
    fetch((u + 3) & 3);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      constexpr int base = (u * 4) % kRing;
      const u32x4 wf = wring[base + k];
#pragma unroll
      for (int j = 0; j < PB; ++j) {
        Mma<half_t>::run(wf, pr[k & 1][j], acc[j]);
        __builtin_amdgcn_sched_barrier(0);
        if (k < 3) pr[(k + 1) & 1][j] = *reinterpret_cast<const u32x4*>(prow[k + 1] + u * kStage + j * 4096);
        if (j == PB - 1) wring[base + k] = wload(8 + k);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    woff += 8192;
    if constexpr (AUX) {  // the centre tap's pixels are the auxiliary filters' operands
      if (tap == 4) {
#pragma unroll
        for (int k = 0; k < 4; ++k)
#pragma unroll
          for (int j = 0; j < PB; ++j) {
            const u32x4 x = *reinterpret_cast<const u32x4*>(prow[k] + u * kStage + j * 4096);
            Mma<half_t>::run(waux[k], x, acc2[j]);
          }
        load_aux();  // (the next slab's; beyond the last one zeros)
      }
      tap = tap == 8 ? 0 : tap + 1;
    }
  };
  for (int st = 0;;) {
    stage(std::integral_constant<int, 0>());
    if (++st >= T) break;
    stage(std::integral_constant<int, 1>());
    if (++st >= T) break;
    stage(std::integral_constant<int, 2>());
    if (++st >= T) break;
    stage(std::integral_constant<int, 3>());
    if (++st >= T) break;
  }
  float* ss = reinterpret_cast<float*>(smem + kLds);
  if (AUX || !second) {
    ss[threadIdx.x] = a.scale ? __builtin_bit_cast(float, scv) : 1.0f;
    ss[(AUX ? 2 : 1) * BF + threadIdx.x] = __builtin_bit_cast(float, shv);
  }
  __builtin_amdgcn_s_waitcnt(kAllLanded);  // (also what was asked for beyond the last stage: the tile below takes its place)
  __syncthreads();

  // ---- out, through one tile [BP pixels][128 channels]: rows of 256 bytes leave as whole lines (64 bytes of a row a wave: 81
  // instead of 66 us for 256x56x56x64 -> 128 + 128, which is bound by what it writes) ----
  const int orow = wave * 4 + (lane >> 4), ochan = (lane & 15) * 8;
  auto finish = [&](floatx16 (&sum)[PB], const float* sc, int act, __amdgpu_buffer_rsrc_t rs_out, int f, int filters, int ldo, int from, unsigned ofs) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < PB; ++j) {
      float y[16];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const floatx4 m = *reinterpret_cast<const floatx4*>(sc + 8 * q + 4 * lh), h = *reinterpret_cast<const floatx4*>(sc + (AUX ? 2 : 1) * BF + 8 * q + 4 * lh);
#pragma unroll
        for (int e = 0; e < 4; ++e) y[4 * q + e] = sum[j][4 * q + e] * m[e] + h[e];
      }
      act_apply_n<true>(y, act & 0xff);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        half4 x;
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = (half_t)y[4 * q + e];
        *reinterpret_cast<half4*>(smem + (j * 32 + lrow) * kPitch + wave * 64 + q * 16 + lh * 8) = x;
      }
    }
    __syncthreads();
#pragma unroll
    for (int o = 0; o < 2 * PB; ++o) {
      const int p = p0 + o * 16 + orow;
      const u32x4 v = *reinterpret_cast<const u32x4*>(smem + (o * 16 + orow) * kPitch + ochan * 2);
      __builtin_amdgcn_raw_buffer_store_b128(v, rs_out, p < a.P && f < filters ? (unsigned)(p * ldo + f - from) * 2u + ofs : kOOBr, 0, 0);
    }
  };
  const bool other = POINT && f0 + ochan >= a.split_f;  // (of a lane's eight filters all or none)
  finish(acc, ss + wave * 32, a.act, make_rsrc(a.out, a.out_bytes), f0 + ochan, fend, other ? a.split_ldo : a.ldo, other ? a.split_f : 0, POINT ? (other ? a.split_ofs : a.ofs) : 0u);
  if constexpr (AUX) {
    __syncthreads();
    finish(acc2, ss + BF + wave * 32, a.aux_act, make_rsrc(a.aux_out, a.aux_out_bytes), f0 + ochan, a.F - a.aux_f0, a.aux_ldo, 0, 0u);
  }
}

// ---- dispatch

template <int WP, int WF, int PB, int FB, int S, int CH = 0, bool UP = false>
void launch_cfg(RingArgs d, int mode, hipStream_t s) {
  constexpr int NW = WP * WF, BP = 32 * WP * PB, BF = 32 * WF * FB, ring = S * (BP + BF) * 128, tile = NW * PB * 32 * (FB * 64 + 16);
  constexpr int lds = (ring > tile ? ring : tile) + BF * 8 + 128 * CH;
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
  if constexpr (CH > 0 || UP) return go(conv_ring_kernel<WP, WF, PB, FB, S, kPoint, CH, UP>);
  if (mode == kPoint) go(conv_ring_kernel<WP, WF, PB, FB, S, kPoint>);
  else if (mode == kLines) go(conv_ring_kernel<WP, WF, PB, FB, S, kLines>);
  else go(conv_ring_kernel<WP, WF, PB, FB, S, kAny>);
}

template <int PB>
void launch_frag(RingArgs d, int mode, hipStream_t s) {
  constexpr int BP = 32 * PB, ring = 4 * BP * 128, tile = BP * 272, lds = (ring > tile ? ring : tile) + 128 * 16;
  const int main_f = d.aux_f0 ? d.aux_f0 : d.F;
  d.tiles_f = (main_f + 127) / 128;
  d.tiles_p = (d.P + BP - 1) / BP;
  d.inv_tiles = 1.0f / (float)(d.pixels_first ? d.tiles_p : d.tiles_f);
  d.groups = (main_f + 63) / 64 * 2;
  d.aux_groups = (d.F - main_f + 63) / 64 * 2;
  d.lead = mode == kPoint ? 0 : (d.W + 1) * d.pix * 2;
  auto go = [&](auto kern) {
    static const bool attr = [&] {
      NNCV_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, lds));
      return true;
    }();
    (void)attr;
    launch_kernel(kern, dim3((unsigned)(d.tiles_f * d.tiles_p)), dim3(256), lds, s, d);
  };
  if constexpr (PB == 2)
    if (mode == kPoint) return go(conv_ring_frag_kernel<PB, false, true>);
  if (d.aux_f0) go(conv_ring_frag_kernel<PB, true>);
  else go(conv_ring_frag_kernel<PB, false>);
}

// The forms, and what a launch of each takes: us = fixed + ((busy)^3 + (chain)^3)^(1/3) with
//   busy  = tiles / 256 CUs * (slab_us * slabs + tile_us)            (LDS, matrix and memory pipes)
//   chain = ceil(tiles / (256 * resident)) * chain_us * slabs        (a slab's latency, workgroups of a CU one after the other)
// The fragment forms: us = fixed + t * (slab_us * slabs + tile_us), t halfway between tiles / 256 (at least 1) and its ceiling, or
// chain_us + t * slab_any for 64 channels (nine slabs, bound by memory); within 6 % (1 sigma) over 112 stride-2 layers of 1 to 60
// GFLOP, and in the choice between the two 0.8 % off the better one on average.  With 64 channels, 64 pixels to a tile are up to 8 %
// ahead to 16 such tiles a CU (80x56x56 -> 128 17.1 against 18.3 us), 128 from there (241x77x91 -> 72 91.7 against 101.9).  The
// ring's own forms of 128 filters are level with them at best, save for 64 channels and more than three, up to four tiles of 64 x 128 a CU:
// the two tiles of 128 x 128 that a CU has there run side by side with 16 waves, in one turn.  It is the number of tiles that does it, not
// the layer: of 31 layers in that band, 72 to 384 filters on maps of 14x14 to 224x20, 28 take 0.90 to 0.995 times as long on the ring
// and three 1.00 to 1.01 (1037x14x14 -> 72 13.3 against 14.0 us, 318x28x28 -> 96 15.1 / 16.0, 79x56x56 -> 128 15.8 / 17.6, 19x80x80 -> 256
// 15.7 / 16.3); of 38 layers on both sides of it, 2.3 to 6.5 tiles, 36 take 1.00 to 1.19 times as long there (41x80x80 -> 96, 4.004
// tiles: 19.9 against 17.1; 242x28x28 -> 128, 2.9: 14.8 / 13.2).
// slab_us and chain_us grow by slab_any and chain_any where the taps are not whole slabs.  Fits over 300 layers of 1x1 to 7x7
// windows, 8 to 1024 channels; the form they choose is within 1.5 % of the best one on average.
struct Form {
  int bp, bf, resident;
  double fixed_us, slab_us, tile_us, chain_us, slab_any, chain_any;
  void (*launch)(RingArgs, int, hipStream_t);
  const char* tag;
  bool frag = false;
};
const Form kForms[] = {
    {64, 64, 7, 2.58, 0.220, 0.287, 0.405, 0.26, 0.18, launch_cfg<2, 2, 1, 1, 1>, "conv_ring<64x64>"},
    {64, 64, 4, 2.72, 0.233, 0.353, 0.350, 0.26, 0.38, launch_cfg<2, 2, 1, 1, 2>, "conv_ring<64x64,2>"},
    {64, 32, 13, 2.71, 0.144, 0.180, 0.423, 0.24, 0.26, launch_cfg<2, 1, 1, 1, 1>, "conv_ring<64x32>"},
    {64, 128, 3, 3.04, 0.353, 0.620, 0.434, 0.11, 0.37, launch_cfg<2, 2, 1, 2, 2>, "conv_ring<64x128,2>"},
    {128, 128, 2, 2.94, 0.626, 1.086, 0.631, 0.11, 0.11, launch_cfg<4, 2, 1, 2, 1>, "conv_ring<128x128>"},
    {128, 128, 2, 3.08, 0.583, 1.142, 0.515, 0.21, 0.48, launch_cfg<4, 2, 1, 2, 2>, "conv_ring<128x128,2>"},
    {64, 128, 4, 2.64, 0.293, 0.448, 2.98, 3.06, 0, launch_frag<2>, "conv_ring<64x128,frag>", true},
    {128, 128, 2, 1.51, 0.472, 2.537, 2.41, 6.32, 0, launch_frag<4>, "conv_ring<128x128,frag>", true},
};

// 1x1 layers of 512 channels and more, one to one and a half tiles of 64 x 128 a CU: long chains of slabs that the ring fetches one ahead and the
// fragment form three, with filters from memory that may not be in L2.  us, ring / here: 4x28x28x512 -> 512 7.2 / 6.5, 2x40x40x768 -> 384 8.3 / 7.1,
// 12x20x20x1024 -> 384 13.2 / 9.2, 48x20x20x1536 -> 96 22.2 / 17.5, 32x14x14x1536 -> 512 19.1 / 17.0; of 12 such layers the least gains 1.8 %
// (32x14x14x768 -> 384, 24x10x10x640 -> 384).  With 256 and 384 channels, below 112 tiles and above 400 it is level at best (12x20x20x256 -> 96
// 4.5 / 4.9, 16x28x28x768 -> 384 15.4 / 15.7).  The model: the same layers, within 8 %.
bool point_serves(int dt, int F, int RS, int C, int stride, int pad) { return dt == kF16 && RS == 1 && stride == 1 && pad == 0 && C % 64 == 0 && C >= 512 && F > 64; }
const Form kPointForm{64, 128, 4, 0, 0, 0, 0, 0, 0, launch_frag<2>, "conv_ring<64x128,point>", true};
double point_us(const IgemmArgs& a) {  // 0: not taken
  const double tiles = std::ceil((double)a.N * a.OH * a.OW / 64) * std::ceil(a.F / 128.0), slabs = a.C / 64;
  if (!a.wt_frag || !point_serves(kF16, a.F, a.R * a.S, a.C, a.stride_h, a.pad_h) || a.stride_w != 1 || a.pad_w != 0 || a.residual || a.aux_f0 || a.chain_f || tiles < 112 || tiles > 400)
    return 0;
  return tiles <= 256 ? 3.1 + 0.36 * slabs : 4.9 + 0.51 * slabs;
}

// What the fragment forms cover.  With auxiliary filters, whose sums take the registers of a third wave, from 256 channels on
// (ResNet-18, 256 images: 44.3 -> 41.2 us; 47.2 -> 49.7 at 128 channels, 65.8 -> 67.8 at 64), and with 128 pixels to a tile (64: 77).
bool frag_ok(const IgemmArgs& a) {
  const long long pix = a.pix_stride ? a.pix_stride : a.C;
  return a.wt_frag && a.R == 3 && a.S == 3 && a.pad_h == 1 && a.pad_w == 1 && a.C % 64 == 0 && !a.residual && (a.aux_f0 == 0 || (a.C >= 256 && a.aux_wt_frag && a.aux_tap == 4 && a.F <= 2 * a.aux_f0)) &&
         (long long)a.in_bytes + (a.W + 1) * pix * 2 < (long long)kOOBr;
}

const Form* best_form(const IgemmArgs& a, double* us) {
  if ((*us = point_us(a)) > 0) return &kPointForm;
  const double P = (double)a.N * a.OH * a.OW, slabs = std::ceil(a.R * a.S * a.C / 64.0), main_f = a.aux_f0 ? a.aux_f0 : a.F;
  const bool any = a.R * a.S > 1 && a.C % 64 != 0, nine = slabs <= 9;
  auto per_cu = [&](const Form& f, double filters) { return std::ceil(P / f.bp) * std::ceil(filters / f.bf) / 256; };
  // (tiles of 64 x 128 a CU: see the forms)
  const double quarters = std::ceil(P / 64) * std::ceil(main_f / 128) / 256;
  const bool frag = frag_ok(a) && !(nine && quarters > 3 && quarters <= 4);
  const Form* best = nullptr;
  for (const Form& f : kForms) {
    double v;
    if (f.frag) {
      if (!frag || (a.aux_f0 ? f.bp == 64 : nine && (quarters < 16) != (f.bp == 64))) continue;
      const double x = per_cu(f, main_f), t = (0.5 * std::ceil(x) + 0.5 * std::max(1.0, x)) * (a.aux_f0 ? 10 / 9.0 : 1);
      v = nine ? f.chain_us + t * f.slab_any : f.fixed_us + t * (f.slab_us * slabs + f.tile_us);
    } else {
      if (frag && f.bf == 128) continue;
      const double x = per_cu(f, main_f + (a.F - main_f) / (a.R * a.S));  // auxiliary filters walk one tap
      const double busy = x * (f.slab_us * slabs * (any ? 1 + f.slab_any : 1) + f.tile_us);
      const double chain = std::ceil(x / f.resident) * f.chain_us * slabs * (any ? 1 + f.chain_any : 1);
      v = f.fixed_us + std::cbrt(busy * busy * busy + chain * chain * chain);
    }
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

bool conv_ring_point_serves(int dt, int F, int RS, int C, int stride, int pad) { return point_serves(dt, F, RS, C, stride, pad); }

// Stride-2 3x3 layers without auxiliary filters leave the patch kernel for the fragment forms from 112 tiles of 64 x 128 on: of 41
// layers between there and 400 tiles 38 take 0.5 to 0.96 times as long, the others 1.0 (24x19x16x256 -> 512, 120 tiles: 19.9 -> 12.7;
// 19x31x77x64 -> 192, 372: 9.5 -> 9.1).  Below, its smaller tiles and K groups mostly fill the chip better (6x22x86x256 -> 256, 92
// tiles: 9.1 against 12.3 us; 11x25x67x128, 73: 6.7 against 8.5), and 64 filters are half a tile (9x65x151x64 -> 64: 7.3 against 7.8).
// The rest leaves it where 128 x 128 tiles keep three quarters of the CUs busy.  From 200 tiles to the
// patch kernel's limit (8 GFLOP) that kernel is bound by its patch reads: 48x56x56x64 -> 128 14.3 against 13.3 us here, 64
// images 17.4 against 14.1, 32x40x40x128 -> 256 20.0 against 15.9, 16x80x80x64 -> 128 10.2 against 10.3 at 200 tiles.  Below, its
// smaller tiles and K groups mostly fill the chip better (32x28x28x128 -> 256, 98 tiles: 9.1 against 11.6; 24x40x40x128 -> 256,
// 150 tiles, is the other way round: 16.5 against 15.1).  Larger launches used to be igemm_fast's: 23 of them take 1.14 to 1.35
// times as long there (256x28x28x128 -> 256: 52.2 against 42.0).  In a ResNet-18 pass of 256 images the three such layers with
// their shortcuts went from 78.1 + 58.4 + 52.2 us there to 65.4 + 46.6 + 43.6, the pass from 1162 to 1133 us of launches.
bool conv_ring_beats_patch_s2(const IgemmArgs& a) {
  const long long P = (long long)a.N * a.OH * a.OW, main_f = a.aux_f0 ? a.aux_f0 : a.F;
  if (a.stride_h == 2 && frag_ok(a) && a.aux_f0 == 0 && a.F > 64 && (P + 63) / 64 * ((main_f + 127) / 128) >= 112) return true;
  return a.stride_h == 2 && (P + 127) / 128 * ((main_f + 127) / 128) >= 200;
}

// Blocks of two 1x1 layers with one bottleneck, us with its first layer in a launch of its own / here, MB of that layer's input: 16x160x160x64 ->
// 32 + 32 -> 32 158.4 / 152.6 (25 MB), 4 images 73.8 / 71.5 (6), 1 image 50.7 / 49.2 (1.6); 16x80x80x128 -> 64 + 64 -> 64 112.5 / 111.8 (12.5), 4
// images 60.2 / 59.1 (3); 2 images 50.2 / 50.3 (1.6); 4x80x80x256 -> 64 + 64 -> 64, where nothing else reads the first result, 73.3 / 70.4 (3).
// With 128 channels the chained filters take the registers of a CU's second workgroup: 16x40x40x256 21.0 us against 11.5 + 6.7.
bool conv_ring_chains(long long P, int C, int F) { return (F == 32 || F == 64) && C % 8 == 0 && P * F * 2 >= 2 << 20; }

// The forms that have it: two slabs in the ring, tiles of 128 x 128, where those run anyway.  A lane reads its pixel or its quarter as easily:
// 16x40x40x(256 + 256) -> 128 + 128 15.5 us, 15.9 behind a copy of 6.1; 16x80x80x(128 + 128) -> 64 + 64 -> 64 24.6, 25.1 behind 8.8.
bool conv_ring_upsamples(const IgemmArgs& a, int up_c, int up_pix) {
  double us = 0;
  const bool form = a.chain_f ? a.chain_f == 64 && a.C > 128 : best_form(a, &us)->launch == static_cast<void (*)(RingArgs, int, hipStream_t)>(launch_cfg<4, 2, 1, 2, 2>);
  return form && up_c % 64 == 0 && up_c > 0 && up_pix % 8 == 0 && a.H % 2 == 0 && a.W % 2 == 0 && a.OH == a.H && a.OW == a.W &&
         (long long)a.N * (a.H / 2) * (a.W / 2) * up_pix * 2 < (long long)kOOBr;
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
  d.wfrag = a.wt_frag; d.aux_wfrag = a.aux_wt_frag;
  const double flops = a.alg_flops > 0 ? a.alg_flops : 2.0 * d.P * (double)a.F * a.R * a.S * a.C;
  const double bytes = 2.0 * ((double)a.N * a.H * a.W * a.C + (double)a.F * a.R * a.S * a.C + (double)d.P * a.F * (a.residual ? 2 : 1));
  if (a.up_in) {
    d.up_in = a.up_in; d.up_slabs = a.up_c / 64; d.up_pix = a.up_pix;
    d.up_bytes = (unsigned)((long long)a.N * (a.H / 2) * (a.W / 2) * a.up_pix * 2);
  }
  if (a.chain_f) {
    d.chain_wt = a.chain_wt; d.chain_scale = a.chain_scale; d.chain_shift = a.chain_shift; d.chain_out = a.chain_out;
    d.chain_act = a.chain_act; d.chain_ldo = a.chain_ldo; d.chain_only = a.chain_only;
    d.chain_bytes = (unsigned)d.P * a.chain_ldo * 2u;
    d.pixels_first = false;
    ProfScope prof("conv_ring<chain>", flops + 2.0 * d.P * (double)a.chain_f * a.chain_f, bytes + 2.0 * d.P * (double)a.chain_f, s);
    const bool two = d.chunks > 16;  // (slabs in the ring: one up to 128 channels, as without the chained layer)
    if (a.up_in) launch_cfg<4, 2, 1, 2, 2, 4, true>(d, kPoint, s);
    else if (a.chain_f == 32) launch_cfg<2, 2, 1, 1, 1, 2>(d, kPoint, s);
    else if (two) launch_cfg<4, 2, 1, 2, 2, 4>(d, kPoint, s);
    else launch_cfg<4, 2, 1, 2, 1, 4>(d, kPoint, s);
    NNCV_HIP_CHECK(hipGetLastError());
    return;
  }
  if (a.up_in) {
    ProfScope prof("conv_ring<128x128,2,up>", flops, bytes, s);
    launch_cfg<4, 2, 1, 2, 2, 0, true>(d, kPoint, s);
    NNCV_HIP_CHECK(hipGetLastError());
    return;
  }
  if (conv3x3s2_resident_wins(a)) {
    launch_conv3x3s2_resident(a, flops, bytes, s);
    return;
  }
  ProfScope prof(f->tag, flops, bytes, s);
  f->launch(d, a.R * a.S == 1 && a.pad_h == 0 && a.pad_w == 0 ? kPoint : a.C % 64 == 0 ? kLines : kAny, s);
  NNCV_HIP_CHECK(hipGetLastError());
}

}  // namespace nncv_hip
