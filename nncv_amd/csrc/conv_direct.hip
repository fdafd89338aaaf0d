// Implicit-GEMM convolution with waves that do not wait for each other: fp32 layers of any size, and fp16 layers too small to
// fill the chip with the workgroup tiles of the other kernels.  Replaces the compiler's tiling of linalg.conv_2d_nchw_fchw
// (src/nncv/compiler/Conversion/CodeGen/LlvmCpu/ModernTile.cpp:124-286) for those.
//
// A wave owns TM x TN accumulators of BT x BT (filters x pixels).  K is the flat (r, s, c) axis in 16-byte chunks, eight of
// them (one 128-byte line of a pixel) to a round.
//  * Weights come fragment-major (launch_weight_flat): an operand of a wave is one contiguous kilobyte, straight into
//    registers a round ahead.
//  * Pixels: an operand wants 32 (16) pixels x 2 (4) chunks, and read like that every lane of the load touches a line of
//    its own, which the CU's address unit serves one lane a clock (58 cycles per load measured, against 16 for whole
//    lines).  So a wave loads whole lines, eight lanes to a pixel, a round ahead, passes them through an LDS buffer of its
//    own (chunks XORed with the row: no bank conflicts either way) and reads its operands from there.  Nothing is shared
//    between waves, so there is no barrier in the K loop.
//  * fp32 MFMAs take 64 (32) cycles on four bytes per lane, so one wave keeps its matrix pipe busy on a sixteenth of the
//    CU's load path.  fp16 would need all of it for a 2 x 2 wave: large layers stay with the other kernels; small ones are
//    bound by how many CUs stream the weights and by latency, which is what KG is for.
//  * KG "K groups": all waves of the workgroup share its tile and split the rounds; their sums meet in LDS in a fixed order.
//    With 16 x 16 tiles a 7x7x512 layer of one image is 128 workgroups of 16 waves with five rounds each.
//  * The halo is the buffer range check: a tap outside the image gets an offset beyond the descriptor and reads as zero.
//  * Auxiliary filters (IgemmArgs::aux_f0: the 1x1 shortcut of a down-sampling block) are further filter tiles that walk
//    the channels of their one tap only.
#include <algorithm>
#include <cmath>

#include "split.hpp"

namespace nncv_hip {

using namespace mt;

namespace {

constexpr unsigned kOOBd = 0x7fff0000u;  // byte offset beyond any buffer this kernel accepts

template <typename T, int BT>
struct Block;
template <>
struct Block<float, 32> {
  typedef floatx16 acc;
  static __device__ __forceinline__ void run(const u32x4& a, const u32x4& b, acc& c) {
    const floatx4 fa = __builtin_bit_cast(floatx4, a), fb = __builtin_bit_cast(floatx4, b);
#pragma unroll
    for (int e = 0; e < 4; ++e) c = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[e], fb[e], c, 0, 0, 0);
  }
};
template <>
struct Block<float, 16> {
  typedef floatx4 acc;
  static __device__ __forceinline__ void run(const u32x4& a, const u32x4& b, acc& c) {
    const floatx4 fa = __builtin_bit_cast(floatx4, a), fb = __builtin_bit_cast(floatx4, b);
#pragma unroll
    for (int e = 0; e < 4; ++e) c = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[e], fb[e], c, 0, 0, 0);
  }
};
template <>
struct Block<half_t, 32> {
  typedef floatx16 acc;
  static __device__ __forceinline__ void run(const u32x4& a, const u32x4& b, acc& c) {
    c = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8, a), __builtin_bit_cast(half8, b), c, 0, 0, 0);
  }
};
template <>
struct Block<half_t, 16> {
  typedef floatx4 acc;
  static __device__ __forceinline__ void run(const u32x4& a, const u32x4& b, acc& c) {
    c = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, a), __builtin_bit_cast(half8, b), c, 0, 0, 0);
  }
};

struct DirectArgs {
  const void* in; const void* wt; const void* aux_wt; void* out; const float* scale; const float* shift; const void* residual; void* aux_out;
  unsigned in_bytes, wt_bytes, aux_wt_bytes;
  int H, W, F, S, OW, OHW, P, pix;
  int stride_h, stride_w, pad_h, pad_w;
  int act, aux_act, ldo, aux_ldo;
  int chunks, cpt;       // 16-byte chunks of K, and of one tap
  int main_tiles, tiles_f, tiles_p, pixels_first;
  int main_f, aux_tap;   // filters of the convolution itself; the tap the others walk
  float inv_ohw, inv_ow, inv_s, inv_cpt, inv_tiles;
};
constexpr int kStoreF32 = 1 << 30;  // in `act`: the result is fp32 whatever OutT (no residual, no auxiliary filters)

// UNI: a tap is a whole number of rounds (C elements = whole 128-byte lines), so the tap of a round is the same for all lanes
// BEHIND: a workgroup takes its tile's auxiliary filters behind it, over the same pixels; there are no workgroups for them
template <typename T, typename OutT, int BT, int TM, int TN, int KG, bool UNI, int D, bool BEHIND>
__global__ __launch_bounds__(64 * KG) void conv_direct_kernel(const DirectArgs a) {
  // Three-way bf16 splits (split.hpp) where two filter blocks share a split of the pixels and there are waves to hide it:
  // 6x58x78x64 -> 128 at stride 2 15.9 -> 14.1 us, 16x28x28x128 -> 256 24.5 -> 21.2.  32 x 32 waves spend as long splitting as they
  // save (0.83 to 1.11 times), 64 x 64 ones are alone on their SIMD (0.91).
  constexpr bool kSplit = sizeof(T) == 4 && BT == 32 && TM == 2 && TN == 1;
  constexpr int kEs = sizeof(T), LG = 64 / BT, NQ = BT / 8, GL = BT * TN / 8;  // GL: pixel loads of a round
  constexpr int kBuf = BT * TN * 128, kPart = TM * TN * BT * BT * 4;
  constexpr int kWaveLds = 2 * kBuf > kPart || KG == 1 ? 2 * kBuf : kPart;
  constexpr int kQuadsPerBlock = BT * BT / 256, kQuads = TM * TN * kQuadsPerBlock, kMine = (kQuads + KG - 1) / KG;
  extern __shared__ __align__(16) unsigned char smem[];
  // all arguments at once: fetched where they are first used, they are one wait after the other
  asm volatile("" ::"s"(a.in), "s"(a.wt), "s"(a.in_bytes), "s"(a.wt_bytes), "s"(a.H), "s"(a.W), "s"(a.F), "s"(a.S), "s"(a.OW), "s"(a.OHW), "s"(a.P), "s"(a.pix),
               "s"(a.stride_h), "s"(a.stride_w), "s"(a.pad_h), "s"(a.pad_w), "s"(a.chunks), "s"(a.cpt), "s"(a.main_tiles), "s"(a.tiles_f), "s"(a.tiles_p), "s"(a.main_f),
               "s"(a.inv_ohw), "s"(a.inv_ow), "s"(a.inv_s), "s"(a.inv_cpt), "s"(a.inv_tiles));
  const int lane = threadIdx.x & 63, grp = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int lrow = lane & (BT - 1), lh = lane / BT;
  unsigned char* lds = smem + grp * kWaveLds;
  // XCD x (workgroups x, x + 8, ...) takes a contiguous run of tiles: of pixels under all filters, or (when the weights
  // are the larger operand) of filters over all pixels, so that its L2 holds a part of that operand only
  int tf, tp;
  {
    const int tiles = a.tiles_f * a.tiles_p, per = (tiles + 7) >> 3, rem = tiles & 7;
    const int x = blockIdx.x & 7, i = blockIdx.x >> 3;
    const int t = rem == 0 ? x * per + i : (x < rem ? x * per : rem * per + (x - rem) * (per - 1)) + i;
    if (a.pixels_first) tf = fast_div(t, a.tiles_p, a.inv_tiles, &tp);
    else tp = fast_div(t, a.tiles_f, a.inv_tiles, &tf);
    tf = __builtin_amdgcn_readfirstlane(tf);
    tp = __builtin_amdgcn_readfirstlane(tp);
  }
  const int p0 = tp * BT * TN;
  const __amdgpu_buffer_rsrc_t rs_in = make_rsrc(a.in, a.in_bytes);
  int base[GL], iy0[GL], ix0[GL];
  u32x4 w[D][NQ][TM], gx[D][GL];
  for (int pass = 0;; ++pass, tf += a.main_tiles) {
  const bool aux = tf >= a.main_tiles;
  const int f0 = aux ? a.main_f + (tf - a.main_tiles) * BT * TM : tf * BT * TM;
  const int f_end = aux ? a.F : a.main_f;
  const __amdgpu_buffer_rsrc_t rs_wt = aux ? make_rsrc(a.aux_wt, a.aux_wt_bytes) : make_rsrc(a.wt, a.wt_bytes);

  // rounds of this group; an auxiliary tile walks the rounds of its tap (UNI)
  const int nr = (a.chunks + 7) >> 3, rpt = a.cpt >> 3;
  const int r_lo = aux ? a.aux_tap * rpt : 0, r_n = aux ? rpt : nr;
  const int rb = r_lo + grp, re = r_lo + r_n;  // group g takes rounds g, g + KG, ...: neighbouring lines at the same time

  // weights: filter block of 32, unit of two chunks, 1 KB each; a 16-filter block reads its half of two units
  unsigned woff[TM];
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int f = f0 + BT * i - (aux ? a.main_f : 0);
    const unsigned fb = (unsigned)(f >> 5) * (unsigned)(r_n * 4);
    woff[i] = BT == 32 ? (fb * 64u + lane) * 16u : ((fb + (lh >> 1)) * 64u + (lh & 1) * 32u + (f & 16) + lrow) * 16u;
  }
  auto load_w = [&](int r, int q, u32x4 (&w)[NQ][TM]) __attribute__((always_inline)) {
    const unsigned at = (unsigned)(4 * (r - r_lo) + (BT == 32 ? q : 2 * q)) * 1024u;
#pragma unroll
    for (int i = 0; i < TM; ++i) w[q][i] = __builtin_amdgcn_raw_buffer_load_b128(rs_wt, ((f0 + BT * i < f_end) & (r < re)) ? woff[i] + at : kOOBd, 0, 0);
  };
  // the first ones are asked for now: their addresses are there long before the pixels' (those of the second pass are on their way)
  if (pass == 0) {
#pragma unroll
    for (int q = 0; q < NQ; ++q) load_w(rb, q, w[0]);
  }
  __builtin_amdgcn_sched_barrier(0);

  // pixels: this lane loads chunk lane % 8 of the rows lane / 8, + 8, ...; pixels past the end read the last one (not stored)
  // (worked out once per row, a lane each, and handed round through the LDS buffer that is still empty)
  if (pass == 0) {
    static_assert(BT * TN <= 64, "a lane per pixel row");
    int rem, ox;
    const int n = fast_div(min(p0 + lane, a.P - 1), a.OHW, a.inv_ohw, &rem);
    const int oy = fast_div(rem, a.OW, a.inv_ow, &ox);
    const int iy = oy * a.stride_h - a.pad_h, ix = ox * a.stride_w - a.pad_w;
    typedef int int4v __attribute__((ext_vector_type(4)));
    if (lane < BT * TN) reinterpret_cast<int4v*>(lds)[lane] = int4v{((n * a.H + iy) * a.W + ix) * a.pix * kEs, iy, ix, 0};
#pragma unroll
    for (int g = 0; g < GL; ++g) {
      const int4v v = reinterpret_cast<const int4v*>(lds)[8 * g + (lane >> 3)];
      base[g] = v[0] + (UNI ? (lane & 7) * 16 : 0);
      iy0[g] = v[1];
      ix0[g] = v[2];
    }
  }
  int ur, us, uc;  // UNI: filter row, filter column and chunk of the next round to load
  {
    const int tap = fast_div(8 * rb, a.cpt, a.inv_cpt, &uc);
    ur = fast_div(tap, a.S, a.inv_s, &us);
  }
  int dr, ds, dc;  // KG rounds further on
  {
    const int tap = fast_div(8 * KG, a.cpt, a.inv_cpt, &dc);
    dr = fast_div(tap, a.S, a.inv_s, &ds);
  }
  int rload = rb;
  auto step_tap = [&]() __attribute__((always_inline)) {
    uc += dc;
    us += ds;
    ur += dr;
    if (uc >= a.cpt) uc -= a.cpt, ++us;
    if (us >= a.S) us -= a.S, ++ur;
    rload += KG;
  };
  auto load_x = [&](u32x4 (&gx)[GL]) __attribute__((always_inline)) {
    int r = ur, s = us, at;
    bool in_k = rload < re;
    if constexpr (UNI) {
      at = ((ur * a.W + us) * a.pix) * kEs + uc * 16;
      step_tap();
    } else {
      const int kc = 8 * rload + (lane & 7);
      int c;
      const int tap = fast_div(kc, a.cpt, a.inv_cpt, &c);
      r = fast_div(tap, a.S, a.inv_s, &s);
      at = ((r * a.W + s) * a.pix) * kEs + c * 16;
      in_k &= kc < a.chunks;
      rload += KG;
    }
#pragma unroll
    for (int g = 0; g < GL; ++g) {
      const bool ok = in_k & ((unsigned)(iy0[g] + r) < (unsigned)a.H) & ((unsigned)(ix0[g] + s) < (unsigned)a.W);
      gx[g] = __builtin_amdgcn_raw_buffer_load_b128(rs_in, ok ? (unsigned)(base[g] + at) : kOOBd, 0, 0);
    }
  };
  const int wr_at = (lane >> 3) * 128 + (((lane & 7) ^ (lane >> 3)) * 16);
  auto park = [&](int buf, const u32x4 (&gx)[GL]) __attribute__((always_inline)) {
#pragma unroll
    for (int g = 0; g < GL; ++g) *reinterpret_cast<u32x4*>(lds + buf * kBuf + g * 1024 + wr_at) = gx[g];
  };
  auto operand = [&](int buf, int q, int j) {
    return *reinterpret_cast<const u32x4*>(lds + buf * kBuf + (BT * j + lrow) * 128 + (((LG * q + lh) ^ (lrow & 7)) * 16));
  };

  // (split: the small products in sums of their own)
  typename Block<T, BT>::acc acc[TM][TN], low[kSplit ? TM : 1][kSplit ? TN : 1];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int v = 0; v < BT * BT / 64; ++v) {
        acc[i][j][v] = 0.0f;
        if constexpr (kSplit) low[i][j][v] = 0.0f;
      }
  if (pass == 0) load_x(gx[0]);
  else step_tap();
#pragma unroll
  for (int d = 1; d < D; ++d) {
    __builtin_amdgcn_sched_barrier(0);  // (the first requests leave before the addresses of the others are there)
#pragma unroll
    for (int q = 0; q < NQ; ++q) load_w(rb + d * KG, q, w[d]);
    load_x(gx[d]);
  }

  // what this wave finishes: quads of four consecutive filters of a pixel.  Their residual and scale / shift are asked for
  // now; they arrive under the K walk.
  const OutT* res = aux ? nullptr : static_cast<const OutT*>(a.residual);
  OutT* out = static_cast<OutT*>(aux ? a.aux_out : a.out);
  const int ldo = aux ? a.aux_ldo : a.ldo, act = aux ? a.aux_act : a.act;
  typedef OutT out4_whole __attribute__((ext_vector_type(4)));
  typedef out4_whole out4 __attribute__((aligned(sizeof(OutT) == 4 ? 4 : 8)));  // (a caller's fp32 tensor may begin at any float)
  typedef floatx4 float4_any __attribute__((aligned(4)));
  struct Quad {
    floatx4 sc, sh;
    out4 rv;
    long long at;  // element of the result, -1: not stored
  };
  auto quad_of = [&](int k) {
    Quad q;
    const int blk = k / kQuadsPerBlock, g4 = k % kQuadsPerBlock, i = blk / TN, j = blk % TN;
    const int f = f0 + BT * i + (BT == 32 ? 8 * g4 : 0) + 4 * lh, p = p0 + BT * j + lrow;
    const bool ok = f < f_end && p < a.P;
    q.at = ok ? (long long)p * ldo + (aux ? f - a.main_f : f) : -1;
    q.sc = a.scale && ok ? *reinterpret_cast<const floatx4*>(a.scale + f) : floatx4{1.f, 1.f, 1.f, 1.f};
    q.sh = a.shift && ok ? *reinterpret_cast<const floatx4*>(a.shift + f) : floatx4{0.f, 0.f, 0.f, 0.f};
    q.rv = out4{};
    if (res && ok) q.rv = *reinterpret_cast<const out4*>(res + q.at);
    return q;
  };
  auto put = [&](const Quad& q, const floatx4& sum) {
    float y[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) y[e] = sum[e] * q.sc[e] + q.sh[e];
    const bool after = act & kActResidualAfter;
    if (res && !after) {
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] += (float)q.rv[e];
    }
    act_apply_n<sizeof(OutT) == 2>(y, act & 0xff);
    if (res && after) {
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] += (float)q.rv[e];
    }
    if constexpr (sizeof(OutT) == 2) {
      if (act & kStoreF32) {
        *reinterpret_cast<float4_any*>(reinterpret_cast<float*>(out) + q.at) = float4_any{y[0], y[1], y[2], y[3]};
        return;
      }
    }
    out4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = (OutT)y[e];
    *reinterpret_cast<out4*>(out + q.at) = o;
  };
  auto finish = [&](const Quad& q, const floatx4& sum) {
    if (q.at >= 0) put(q, sum);
  };
  Quad mine[KG > 1 ? kMine : 1];
  if constexpr (KG > 1) {
#pragma unroll
    for (int k = 0; k < kMine; ++k)
      if (grp + k * KG < kQuads) mine[k] = quad_of(grp + k * KG);
  }

  park(0, gx[0]);
  load_x(gx[0]);
  u32x4 x[TN];  // the pixel operand is read one step ahead of its products
#pragma unroll
  for (int j = 0; j < TN; ++j) x[j] = operand(0, 0, j);
  int buf = 0;
  if constexpr (kSplit) {
    // two units of the fp32 order make one bf16 operand: its k are the same eight channels for filters and pixels
    u32x4 y[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) y[j] = operand(0, 1, j);
    for (int r = rb; r < re; r += KG, buf ^= 1) {
#pragma unroll
      for (int q = 0; q < NQ; q += 2) {
        u32x4 wp[TM][3], xp[TN][3];
#pragma unroll
        for (int i = 0; i < TM; ++i) split_eight(w[0][q][i], w[0][q + 1][i], wp[i]);
#pragma unroll
        for (int j = 0; j < TN; ++j) split_eight(x[j], y[j], xp[j]);
        load_w(r + KG, q, w[0]);
        load_w(r + KG, q + 1, w[0]);
        if (q == 0) {
          park(buf ^ 1, gx[0]);
          load_x(gx[0]);
        }
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          x[j] = q == 0 ? operand(buf, 2, j) : operand(buf ^ 1, 0, j);
          y[j] = q == 0 ? operand(buf, 3, j) : operand(buf ^ 1, 1, j);
        }
        split_products(wp, xp, acc, low);
      }
    }
    if (__builtin_expect(split_sums(acc, low), 0)) {  // once more with the fp32 instructions: a step is a unit of the weights, two chunks
      int rem, ox;
      const int n = fast_div(min(p0 + lrow, a.P - 1), a.OHW, a.inv_ohw, &rem), oy = fast_div(rem, a.OW, a.inv_ow, &ox);
      const int iy = oy * a.stride_h - a.pad_h, ix = ox * a.stride_w - a.pad_w;
      plain_products(acc, 4 * ((r_n - grp + KG - 1) / KG), [&](int step, u32x4 (&f)[TM], u32x4 (&p)[TN]) {
        const int r = rb + (step >> 2) * KG, unit = 4 * (r - r_lo) + (step & 3), kc = 8 * r + 2 * (step & 3) + lh;
        int c, s;
        const int tap = fast_div(kc, a.cpt, a.inv_cpt, &c), row = fast_div(tap, a.S, a.inv_s, &s);
        const bool ok = (r < re) & (kc < a.chunks) & ((unsigned)(iy + row) < (unsigned)a.H) & ((unsigned)(ix + s) < (unsigned)a.W);
#pragma unroll
        for (int i = 0; i < TM; ++i)
          f[i] = __builtin_amdgcn_raw_buffer_load_b128(rs_wt, ((f0 + BT * i < f_end) & (r < re)) ? woff[i] + (unsigned)unit * 1024u : kOOBd, 0, 0);
        p[0] = __builtin_amdgcn_raw_buffer_load_b128(rs_in, ok ? (unsigned)((((n * a.H + iy + row) * a.W + ix + s) * a.pix) * 4 + c * 16) : kOOBd, 0, 0);
      });
    }
  } else {
    for (int r = rb; r < re; r += D * KG, buf ^= D & 1) {
#pragma unroll
      for (int d = 0; d < D; ++d) {
        if (d > 0 && r + d * KG >= re) break;  // (uniform)
        const int here = buf ^ (d & 1);
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
          u32x4 xn[TN];
          if (q == NQ / 2) {
            park(here ^ 1, gx[(d + 1) % D]);
            load_x(gx[(d + 1) % D]);
          }
#pragma unroll
          for (int j = 0; j < TN; ++j) xn[j] = q + 1 < NQ ? operand(here, q + 1, j) : operand(here ^ 1, 0, j);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) Block<T, BT>::run(w[d][q][i], x[j], acc[i][j]);
          __builtin_amdgcn_sched_barrier(0);
          load_w(r + (d + D) * KG, q, w[d]);
#pragma unroll
          for (int j = 0; j < TN; ++j) x[j] = xn[j];
        }
      }
    }
  }

  if constexpr (BEHIND) {
    static_assert(UNI && D == 1, "one round of the second pass is asked for here, of one tap");
    if (pass == 0) {  // under the sums and their stores
      const int ur = fast_div(a.aux_tap, a.S, a.inv_s, &us), r = grp, at = ((ur * a.W + us) * a.pix) * kEs + 8 * grp * 16;
      const __amdgpu_buffer_rsrc_t rs_aux = make_rsrc(a.aux_wt, a.aux_wt_bytes);
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const int f = tf * BT * TM + BT * i;
        const unsigned fb = (unsigned)(f >> 5) * (unsigned)(rpt * 4);
        const unsigned off = BT == 32 ? (fb * 64u + lane) * 16u : ((fb + (lh >> 1)) * 64u + (lh & 1) * 32u + (f & 16) + lrow) * 16u;
#pragma unroll
        for (int q = 0; q < NQ; ++q)
          w[0][q][i] = __builtin_amdgcn_raw_buffer_load_b128(rs_aux, ((a.main_f + f < a.F) & (r < rpt)) ? off + (unsigned)(4 * r + (BT == 32 ? q : 2 * q)) * 1024u : kOOBd, 0, 0);
      }
#pragma unroll
      for (int g = 0; g < GL; ++g) {
        const bool ok = (r < rpt) & ((unsigned)(iy0[g] + ur) < (unsigned)a.H) & ((unsigned)(ix0[g] + us) < (unsigned)a.W);
        gx[0][g] = __builtin_amdgcn_raw_buffer_load_b128(rs_in, ok ? (unsigned)(base[g] + at) : kOOBd, 0, 0);
      }
    }
  }

  auto quad_sum = [&](int k) {
    const int blk = k / kQuadsPerBlock, g4 = k % kQuadsPerBlock;
    floatx4 s;
#pragma unroll
    for (int e = 0; e < 4; ++e) s[e] = acc[blk / TN][blk % TN][4 * g4 + e];
    return s;
  };
  if constexpr (KG == 1) {
#pragma unroll
    for (int k = 0; k < kQuads; ++k) finish(quad_of(k), quad_sum(k));
  } else {
    floatx4* part = reinterpret_cast<floatx4*>(lds);  // this wave's own region: [quad][lane]
#pragma unroll
    for (int k = 0; k < kQuads; ++k) part[k * 64 + lane] = quad_sum(k);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kMine; ++k) {
      if (grp + k * KG >= kQuads) break;
      const floatx4* p = reinterpret_cast<const floatx4*>(smem) + (grp + k * KG) * 64 + lane;
      floatx4 v[KG];
#pragma unroll
      for (int g = 0; g < KG; ++g) v[g] = p[g * (kWaveLds / 16)];
#pragma unroll
      for (int d = 1; d < KG; d *= 2)  // pairwise: a chain of log2(KG) additions
#pragma unroll
        for (int g = 0; g + d < KG; g += 2 * d) v[g] += v[g + d];
      finish(mine[k], v[0]);
    }
  }
  if (!BEHIND || pass == 1) break;
  if constexpr (KG > 1) __syncthreads();  // every sum has been read: LDS holds pixels again
  }
}

// Auxiliary filters, as many as the convolution's own: behind them in the same workgroups where those alone are for most of the CUs;
// on their own they start late and their pixels come from memory again.  Six images, us: 58x78x64 -> 128 + 128 26.0 -> 21.8,
// 29x39x128 -> 256 + 256 21.8 -> 19.6, 15x20x256 -> 512 + 512 29.0 -> 19.6.  Whole ResNet-18 passes, never / from 200 tiles on / always: one image of 224x224 144 / 143 / 144,
// 8 279 / 270 / 268, 16 446 / 432 / 431, 32 760 / 752 / 751, 64 1421 / 1406 / 1405, 128 of 160x160 1445 / 1433 / 1429; between 150 and 199 tiles there is something left
// (three 214 / 214 / 210, two of 231x309 217 / 216 / 212), below that nothing.
// (fp32 only; tiles of 32 x 32 over two K groups are no down-sampling block's at any number of pixels, by the models)
constexpr bool behind_form(size_t es, int rows, int cols, int kg) { return es == 4 && !(rows == 32 && cols == 32 && kg == 2); }
bool aux_behind(int cpt, int F, int main_f, long long main_tiles) { return cpt % 8 == 0 && F == 2 * main_f && main_tiles >= 200; }

template <typename T, typename OutT, int BT, int TM, int TN, int KG>
void launch_cfg(DirectArgs d, hipStream_t s) {
  constexpr bool kBehind = behind_form(sizeof(T), BT * TM, BT * TN, KG);
  constexpr int kBuf = 2 * BT * TN * 128, kPart = TM * TN * BT * BT * 4, lds = KG * (kBuf > kPart || KG == 1 ? kBuf : kPart);
  d.main_tiles = (d.main_f + BT * TM - 1) / (BT * TM);
  d.tiles_f = d.main_tiles + (d.F - d.main_f + BT * TM - 1) / (BT * TM);
  d.tiles_p = (d.P + BT * TN - 1) / (BT * TN);
  const bool behind = kBehind && aux_behind(d.cpt, d.F, d.main_f, (long long)d.main_tiles * d.tiles_p);
  if (behind) d.tiles_f = d.main_tiles;
  d.inv_tiles = 1.0f / (float)(d.pixels_first ? d.tiles_p : d.tiles_f);
  auto go = [&](auto kern) {
    static const bool attr = [&] {
      if (lds > 65536) NNCV_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, lds));
      return true;
    }();
    (void)attr;
    launch_kernel(kern, dim3((unsigned)((long long)d.tiles_f * d.tiles_p)), dim3(64 * KG), lds, s, d);
  };
  auto depth = [&](auto dc) {
    if (d.cpt % 8 == 0) go(conv_direct_kernel<T, OutT, BT, TM, TN, KG, true, decltype(dc)::value, false>);
    else go(conv_direct_kernel<T, OutT, BT, TM, TN, KG, false, decltype(dc)::value, false>);
  };
  // Three rounds of operands in flight for fp16 walks of nine rounds a wave and more, up to two workgroups a CU: the weights of a
  // pass over one image come from beyond L2 (7x7x512 in such a pass: 8.1 -> 6.9 us, the pass 104.3 -> 101.2; alone, from L2, 6.4 either
  // way).  Shorter walks lose up to 0.7 us to the longer start, fp32 ones 0.5 (twice the requests per round of products), and 32 x 32
  // tiles the third wave of a SIMD (55x66x32x128 -> 32 at 7x7, stride 2: 34.1 -> 40.2).
  if constexpr (sizeof(T) == 2 && BT == 16) {
    if ((d.chunks + 7) / 8 >= 9 * KG && (long long)d.tiles_f * d.tiles_p <= 512) {
      depth(std::integral_constant<int, 3>());
      return;
    }
  }
  if constexpr (kBehind) {
    if (behind) {
      go(conv_direct_kernel<T, OutT, BT, TM, TN, KG, true, 1, true>);
      return;
    }
  }
  depth(std::integral_constant<int, 1>());
}

// [F][C][RS] filters -> the order a wave reads its operands in: [ceil(F / 32)][rounds * 4 units][64 lanes][16 bytes], lane l of
// unit u holding chunk 2 u + l / 32 of the flat K axis (tap, channel; Cp channels per tap) of filter l % 32; padding channels,
// filters and the rest of the last round are zero.  One workgroup per filter, its values read once and in order (they may
// lie in pinned host memory), a range of channels at a time through LDS.
template <typename T>
__global__ __launch_bounds__(256) void weight_flat_kernel(const T* __restrict__ w, T* __restrict__ dst, int F, int C, int RS, int Cp, int units, int cc,
                                                          int staged) {
  constexpr int CE = 16 / (int)sizeof(T);
  extern __shared__ __align__(16) unsigned char raw[];
  T* stage = reinterpret_cast<T*>(raw);  // [cc][RS]
  const int f = blockIdx.x;
  const T* src = w + (long long)f * C * RS;
  T* out = dst + ((long long)(f >> 5) * units * 64 + (f & 31)) * CE;
  auto put = [&](long long k, T v) {
    const long long chunk = k / CE;
    out[((chunk >> 1) * 64 + (chunk & 1) * 32) * CE + (k - chunk * CE)] = v;
  };
  for (int c0 = 0; c0 < Cp; c0 += cc) {
    const int have = f < F ? max(0, min(cc, C - c0)) : 0, width = min(cc, Cp - c0);
    if (staged)
      for (int e = threadIdx.x; e < have * RS; e += 256) stage[e] = src[(long long)c0 * RS + e];
    __syncthreads();
    for (int e = threadIdx.x; e < width * RS; e += 256) {
      const int t = e / width, c = e - t * width;
      put((long long)t * Cp + c0 + c, c >= have ? (T)0.0f : staged ? stage[c * RS + t] : src[(long long)(c0 + c) * RS + t]);
    }
    __syncthreads();
  }
  for (long long k = (long long)RS * Cp + threadIdx.x; k < (long long)units * 2 * CE; k += 256) put(k, (T)0.0f);
}

// The forms of the kernel and what a launch of each takes:
//   us = fixed + t (round_us * rounds of a wave + tile_us) + chain_us * rounds of a wave
// with t between tiles / 256 CUs and its ceiling, and a round = one 128-byte line of K.  Least-squares fits over 117 (fp32) and
// 146 (fp16) layers of 1x1 to 7x7 windows, 8 to 1000 channels, one to 48 images, within 5-12 % of the measured times.
// (fp32 64x64 tiles over four K groups are no form: 64x32 ones take less per area at every number of tiles.)
#define TAGS(x) {"conv1x1_direct<" x ">", "conv3x3_direct<" x ">", "conv_direct<" x ">"}
struct Form {
  int rows, cols, kg;
  double fixed_us, round_us, tile_us, chain_us;
  void (*launch)(DirectArgs, hipStream_t);
  const char* tags[3];  // 1x1, 3x3 and other windows
};
const Form kForms32[] = {
    {32, 32, 2, 3.1, 0.265, 0.32, 0.53, launch_cfg<float, float, 32, 1, 1, 2>, TAGS("f32,32x32,splitk2")},
    {32, 32, 4, 3.0, 0.571, 0.27, 0.25, launch_cfg<float, float, 32, 1, 1, 4>, TAGS("f32,32x32,splitk4")},
    {32, 32, 8, 2.8, 1.146, 0.60, 0.11, launch_cfg<float, float, 32, 1, 1, 8>, TAGS("f32,32x32,splitk8")},
    {16, 16, 4, 2.6, 0.157, 0.23, 0.20, launch_cfg<float, float, 16, 1, 1, 4>, TAGS("f32,16x16,splitk4")},
    {16, 16, 16, 2.1, 0.538, 1.24, 0.31, launch_cfg<float, float, 16, 1, 1, 16>, TAGS("f32,16x16,splitk16")},
    {32, 16, 8, 2.6, 0.543, 0.51, 0.12, launch_cfg<float, float, 16, 2, 1, 8>, TAGS("f32,32x16,splitk8")},
    {64, 32, 4, 3.3, 0.790, 1.30, 0.22, launch_cfg<float, float, 32, 2, 1, 4>, TAGS("f32,64x32,splitk4")},
    {64, 64, 1, 6.0, 0.297, 1.44, 1.89, launch_cfg<float, float, 32, 2, 2, 1>, TAGS("f32,64x64")},
};
const Form kForms16[] = {
    {32, 32, 4, 2.9, 0.268, 0.41, 0.21, launch_cfg<half_t, half_t, 32, 1, 1, 4>, TAGS("f16,32x32,splitk4")},
    {32, 32, 8, 2.6, 0.539, 0.87, 0.01, launch_cfg<half_t, half_t, 32, 1, 1, 8>, TAGS("f16,32x32,splitk8")},
    {16, 16, 4, 2.7, 0.113, 0.22, 0.17, launch_cfg<half_t, half_t, 16, 1, 1, 4>, TAGS("f16,16x16,splitk4")},
    {16, 16, 8, 2.5, 0.207, 0.49, 0.14, launch_cfg<half_t, half_t, 16, 1, 1, 8>, TAGS("f16,16x16,splitk8")},
    {16, 16, 16, 2.0, 0.337, 1.41, 0.22, launch_cfg<half_t, half_t, 16, 1, 1, 16>, TAGS("f16,16x16,splitk16")},
    {32, 16, 8, 2.7, 0.346, 0.47, 0.01, launch_cfg<half_t, half_t, 16, 2, 1, 8>, TAGS("f16,32x16,splitk8")},
    {64, 32, 4, 3.2, 0.399, 0.64, 0.03, launch_cfg<half_t, half_t, 32, 2, 1, 4>, TAGS("f16,64x32,splitk4")},
    {64, 64, 4, 3.0, 0.618, 1.66, 0.08, launch_cfg<half_t, half_t, 32, 2, 2, 4>, TAGS("f16,64x64,splitk4")},
    {64, 64, 1, 6.1, 0.108, 0.89, 0.55, launch_cfg<half_t, half_t, 32, 2, 2, 1>, TAGS("f16,64x64")},
};

#undef TAGS

const Form* best_form(const IgemmArgs& a, int dt, double* us) {
  const int es = (int)dtype_size(dt), rounds = (a.R * a.S * a.C * es + 127) / 128;
  const int main_f = a.aux_f0 ? a.aux_f0 : a.F;
  const long long P = (long long)a.N * a.OH * a.OW;
  const Form* best = nullptr;
  auto consider = [&](const Form& f) {
    const double tiles = (double)((main_f + f.rows - 1) / f.rows) * (double)((P + f.cols - 1) / f.cols), per_cu = tiles / 256;
    const int wave_rounds = (rounds + f.kg - 1) / f.kg;
    const double t = 0.5 * std::ceil(per_cu) + 0.5 * std::max(1.0, per_cu);
    const double v = f.fixed_us + t * (f.round_us * wave_rounds + f.tile_us) + f.chain_us * wave_rounds;
    if (!best || v < *us) best = &f, *us = v;
  };
  if (dt == kF16) for (const Form& f : kForms16) consider(f);
  else for (const Form& f : kForms32) consider(f);
  return best;
}

// The same for the kernel that would run the layer otherwise.  Implicit GEMM: fits over its 64 x 64 tiles, within 7-16 %.
// fp32 3x3 stride-1 layers (conv3x3_split.hip): a start and so much for every 32 channels and tap of a CU's turns; 75 layers of 20
// MFLOP to 20 GFLOP, within 10 %.  Half blocks of filters are the launches of up to 128 whole ones; just above, where nearly half of the
// chip is idle, the model holds too: of 75 layers of 120 to 160 whole blocks the 15 that it gives to that kernel from 129 to 144 on
// take 1.2 to 1.7 times as long here (7x15x20x256 32.1 against 19.7 us, 5x9x25x192 -> 440 21.2 against 16.2, 16x36x16x512 -> 64 55.6
// against 32.1).
double other_us(const IgemmArgs& a, int dt, DirectRival rival) {
  struct Fit { double fixed, round, tile, chain; };
  static const Fit f32[] = {{3.3, 0.642, 0.79, 0.0}, {2.7, 0.835, 0.14, 0.26}};
  static const Fit f16[] = {{2.9, 0.21, 0.74, 0.16}, {2.5, 0.197, 0.43, 0.52}};
  static const Fit f16_3x3[] = {{2.7, 0.097, 0.85, 0.0}, {1.5, 0.009, 2.43, 0.10}};
  const int rounds = (a.R * a.S * a.C * (int)dtype_size(dt) + 127) / 128, main_f = a.aux_f0 ? a.aux_f0 : a.F;
  if (rival == kRivalPatch && dt == kF32) {
    // From 257 channels at the price of tiles of 32 pixels: 4x8x10x512 -> 512 24.5 us here, 15.5 there, 2x14x14x384 18.5 and 13.4.  Up to 256 at that of
    // half blocks, more than those tiles take, which run there all the same: what goes there gains, and what stays here could (14.2 against 9.7 to 11.4 at
    // 256 channels, 11.6 against 8.9 to 10.4 at 192).
    const double flat = a.C > 256 ? conv3x3_split_flat_us(a.N, a.OH, a.OW, a.C, main_f) : 0;
    if (flat > 0) return flat;
    int p[8];
    if (!conv3x3_patch_plan(1, a.N, a.OH, a.OW, main_f, a.C / 32, p)) return 1e30;
    const double wgs = (double)((a.N + p[1] - 1) / p[1]) * ((a.OH + p[2] - 1) / p[2]) * p[4] * ((main_f + 63) / 64), turns = std::ceil(wgs / 256);
    if (p[0] == 4) return 5.0 + 1.2 * rounds * turns;
    if (p[0] == 2) return 6.0 + 0.5 * rounds * turns;
    if (wgs <= 128 && main_f % 64 == 0) return 4.9 + 0.132 * rounds;
    return 4.3 + 0.26 * rounds * turns;
  }
  if (rival == kRivalIgemmFast && dt == kF32) {
    const double split = igemm_fast_split_us(a);
    if (split > 0) return split;
  }
  const Fit& f = rival == kRivalPatch || rival == kRivalPatchS2 ? f16_3x3[rival] : (dt == kF16 ? f16 : f32)[rival - kRivalIgemmFast];
  const double tiles = (double)((main_f + 63) / 64) * (double)(((long long)a.N * a.OH * a.OW + 63) / 64);
  return f.fixed + std::max(1.0, tiles / 256) * (f.round * rounds + f.tile) + f.chain * rounds;
}

}  // namespace

size_t weight_flat_bytes(int dt, int F, int RS, int Cp) {
  const size_t k_bytes = (size_t)RS * Cp * dtype_size(dt);
  return (size_t)((F + 31) / 32) * 32 * ((k_bytes + 127) / 128 * 128);
}

void launch_weight_flat(const void* w_fcrs, void* dst, int dt, int F, int C, int RS, int Cp, hipStream_t s) {
  const int es = (int)dtype_size(dt), units = (int)(((long long)RS * Cp * es + 127) / 128) * 4;
  const int room = 32768 / es, staged = RS <= room, cc = staged ? std::min(Cp, room / RS) : Cp;
  const size_t lds = staged ? (size_t)cc * RS * es : 0;
  const dim3 grid((unsigned)((F + 31) / 32 * 32));
  if (dt == kF16)
    launch_kernel((weight_flat_kernel<half_t>), grid, dim3(256), lds, s, static_cast<const half_t*>(w_fcrs), static_cast<half_t*>(dst), F, C, RS,
                       Cp, units, cc, staged);
  else
    launch_kernel((weight_flat_kernel<float>), grid, dim3(256), lds, s, static_cast<const float*>(w_fcrs), static_cast<float*>(dst), F, C, RS, Cp,
                       units, cc, staged);
  NNCV_HIP_CHECK(hipGetLastError());
}

// K values in memory order are the flat K axis: C = K channels of one tap
void launch_weight_flat_rows(const void* w, void* dst, int dt, int F, int K, hipStream_t s) { launch_weight_flat(w, dst, dt, F, K, 1, K, s); }

// fp16 1x1 layers of up to 64 channels have one round of K at most, which conv_pairs and one slab of the LDS ring do sooner at
// every number of pixels: the models below never choose this kernel for them (88 combinations of channels and filters, one
// pixel to a million).  Filter counts those kernels do not take, and every other layer, have sizes that come here.
bool conv_direct_serves(int dt, int F, int RS, int Cp) { return dt != kF16 || RS > 1 || Cp > 64 || F % 8 != 0; }

bool conv_direct_applicable(const IgemmArgs& a, int in_dt, int out_dt) {
  const int es = (int)dtype_size(in_dt), pix = a.pix_stride ? a.pix_stride : a.C;
  const long long P = (long long)a.N * a.OH * a.OW, k = (long long)a.R * a.S * a.C, lim = 1 << 24;  // fast_div's range
  const bool aux_ok = a.aux_f0 == 0 || (a.aux_f0 % 32 == 0 && a.C * es % 128 == 0 && a.aux_wt_flat && a.aux_out && a.aux_ldo % 4 == 0);
  return a.wt_flat && in_dt == out_dt && a.batch == 1 && aux_ok && a.C * es % 16 == 0 && pix * es % 16 == 0 && a.F % 4 == 0 && a.ldo % 4 == 0 &&
         P < lim && k < lim && a.in_bytes > 0 && a.in_bytes < kOOBd && (long long)a.N * a.H * a.W * pix * es < (long long)kOOBd &&
         (long long)((a.F + 31) / 32) * 32 * ((k * es + 127) / 128 * 128) < (long long)kOOBd &&
         ((long long)(a.F + 15) / 16 + 1) * ((P + 15) / 16) < lim && (a.relu & ~(0xff | kActResidualAfter)) == 0;
}

bool conv_direct_wins(const IgemmArgs& a, int dt, DirectRival rival) {
  if (rival == kRivalShortK) return false;  // already one latency long (3.0-4.5 us either way)
  // fp32 3x3 stride-2 layers of up to 8 GFLOP: the model below flatters igemm_fast there.  Of 40 random shapes that it would
  // give to that kernel 38 are 2-60 % faster here (3x56x80x64 -> 640: 31.3 against 45.3 us, 1x154x199x64 -> 240: 26.9 against 28.1).
  const double main_flops = 2.0 * a.N * a.OH * a.OW * (a.aux_f0 ? a.aux_f0 : a.F) * a.R * a.S * (double)a.C;
  if (dt == kF32 && a.R == 3 && a.S == 3 && a.stride_h == 2 && a.stride_w == 2 && a.pad_h == 1 && a.pad_w == 1 && a.C % 32 == 0 && main_flops <= 8e9) return true;
  const bool patch = rival == kRivalPatch || rival == kRivalPatchS2;
  // fp16 3x3 layers leave the patch kernels only where those have less than a quarter of the chip to work with (blocks of 64
  // pixels x 32 filters): there the layer is bound by how many CUs stream its weights (7x7x512, one image: 8.4 -> 6.0 us).
  // (Maps of under 32 pixels stay too: the patch kernel packs many such images into a tile.)
  if (patch && dt == kF16 &&
      ((long long)((a.F + 31) / 32) * (((long long)a.N * a.OH * a.OW + 63) / 64) >= 64 || (a.N > 1 && a.OH * a.OW < 32)))
    return false;
  // fp16 implicit GEMMs stay with the LDS kernel once its 128 x 128 tiles fill the chip: the models below end there.
  if ((rival == kRivalIgemmFast || rival == kRivalRing) && dt == kF16 && (long long)((a.F + 127) / 128) * (((long long)a.N * a.OH * a.OW + 127) / 128) >= 256) return false;
  double us = 0;
  if (!best_form(a, dt, &us)) return false;
  if (rival == kRivalNarrow) return us < 0.97 * conv3x3_narrow_us(a);
  if (rival == kRivalRing) return us < 0.97 * conv_ring_us(a);
  // margins cover the fits' errors: the fp16 3x3 stride-1 kernels' times are the least well fitted
  const double margin = dt == kF32 ? (rival == kRivalPatch ? 1.0 : 0.97) : rival == kRivalPatch ? 0.85 : 0.9;
  return us < margin * other_us(a, dt, rival);
}

bool conv_direct_plan(const IgemmArgs& a, int dt, int* plan) {
  double us = 0;
  const Form* f = igemm_takes_direct(a, dt, dt) ? best_form(a, dt, &us) : nullptr;
  if (!f) return false;
  const int es = (int)dtype_size(dt), main_f = a.aux_f0 ? a.aux_f0 : a.F;
  const long long tiles = (long long)((main_f + f->rows - 1) / f->rows) * (((long long)a.N * a.OH * a.OW + f->cols - 1) / f->cols);
  plan[0] = f->rows; plan[1] = f->cols; plan[2] = f->kg; plan[3] = (int)tiles;
  plan[4] = behind_form(es, f->rows, f->cols, f->kg) && aux_behind(a.C * es / 16, a.F, main_f, tiles);
  return true;
}

void launch_conv_direct(const IgemmArgs& a, int dt, hipStream_t s, bool store_f32) {
  NNCV_REQUIRE(!store_f32 || (!a.residual && a.aux_f0 == 0), "conv_direct: fp32 results take no residual and no auxiliary filters");
  DirectArgs d{};
  const int es = (int)dtype_size(dt);
  d.in = a.in; d.wt = a.wt_flat; d.out = a.out; d.scale = a.scale; d.shift = a.shift; d.residual = a.residual; d.aux_out = a.aux_out;
  d.in_bytes = a.in_bytes;
  d.wt_bytes = (unsigned)weight_flat_bytes(dt, a.aux_f0 ? a.aux_f0 : a.F, a.R * a.S, a.C);
  if (a.aux_f0) d.aux_wt = a.aux_wt_flat, d.aux_wt_bytes = (unsigned)weight_flat_bytes(dt, a.F - a.aux_f0, 1, a.C);
  d.H = a.H; d.W = a.W; d.F = a.F; d.S = a.S; d.OW = a.OW; d.OHW = a.OH * a.OW; d.P = a.N * a.OH * a.OW; d.pix = a.pix_stride ? a.pix_stride : a.C;
  d.stride_h = a.stride_h; d.stride_w = a.stride_w; d.pad_h = a.pad_h; d.pad_w = a.pad_w;
  d.act = a.relu | (store_f32 ? kStoreF32 : 0); d.aux_act = a.aux_relu; d.ldo = a.ldo; d.aux_ldo = a.aux_ldo;
  d.chunks = a.R * a.S * a.C * es / 16; d.cpt = a.C * es / 16;
  d.main_f = a.aux_f0 ? a.aux_f0 : a.F; d.aux_tap = a.aux_tap;
  d.inv_ohw = 1.0f / (float)d.OHW; d.inv_ow = 1.0f / (float)d.OW; d.inv_s = 1.0f / (float)d.S; d.inv_cpt = 1.0f / (float)d.cpt;
  d.pixels_first = d.wt_bytes > d.in_bytes;
  double us = 0;
  const Form* f = best_form(a, dt, &us);
  const double P = (double)d.P, flops = a.alg_flops > 0 ? a.alg_flops : 2.0 * P * a.F * a.R * a.S * a.C;
  ProfScope prof(f->tags[a.R == 1 && a.S == 1 ? 0 : a.R == 3 && a.S == 3 ? 1 : 2], flops,
                 (double)es * ((double)a.N * a.H * a.W * a.C + (double)a.F * a.R * a.S * a.C + P * a.F * (a.residual ? 2 : 1)), s);
  f->launch(d, s);
  NNCV_HIP_CHECK(hipGetLastError());
}

}  // namespace nncv_hip
