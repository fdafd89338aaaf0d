// A residual block of 64 channels in one launch (gfx950, fp16): relu(bn2(conv2(relu(bn1(conv1(x))))) + x), both convolutions 3x3 stride 1 pad 1
// (tests/Nets/Res18.mlir:152-203, :205-251), for many pixels.
//
//  * As two launches the block writes and reads a tensor between its convolutions and reads x twice: five times the tensor over memory.
//    Here it is two: what lies between the convolutions stays in LDS, and x is there when it is added.  At 256x56x56 (118 GFLOP, 205 MB)
//    it takes 120.8 us, 980 TFLOP/s, where the two launches (conv3x3_f16.hip's stream form, filters resident) took 153.5.
//  * What bounds it: the matrix pipe and LDS, which the products need for the same time.  A step's 144 products of a SIMD are 4608 of its
//    6100 cycles (56 pixels: 112 of 128 slots), and with 32 filters of a wave each 1 KB fragment of pixels read feeds one product, 128 B a
//    cycle over four SIMDs.  64 filters a wave would halve the reads and need 288 registers for them: one wave a SIMD, nothing to run
//    beside its epilogues.  The rest are the second convolution's results (1900 cycles, beside the first one's products) and the first
//    one's epilogue (1300, beside the second one's products).  Wave priority for either of them made it slower (the pass lost 8 us).
//  * A workgroup has a CU and a strip of whole rows of an image.  It walks down in steps of two rows (W > 42), three (W > 32) or four, so that
//    they fill most of 128 slots: four waves make a step's rows of the first convolution, four the rows of the second one that the steps
//    before have completed; a step later the next.  Nothing but a strip's first and last row is computed twice.  With two rows a step,
//    256 images of 128x128 lost 21 us of a pass of 448 to the two launches and 160x160 gained one; with four and three it gains 15 and 32.
//  * A row of more than 64 pixels is cut into columns of up to 40 (WIDE), each with a pixel of the first convolution and two of x more on
//    either side: 42 of them three rows a step, 32 four.  64 images of 320x320, a pass: 633 us with two launches a block, 568.
//  * A wave has 32 filters of its convolution for good, 144 registers of them, and 64 of the 128 slots.  Two waves share a
//    SIMD, one of each convolution: the second one's begin a step with the results of the step before, the first one's end it with theirs,
//    so that the matrix pipe has work from one or the other.
//  * x comes by DMA (buffer_load ... lds) two steps ahead into a ring of five steps' rows; the rows between the convolutions have a ring
//    of three.  With two rows a step the x that results add is the second of two blocks and stays one step less; with three and four
//    (TALL) the results read the block whose place the next one takes, so that fetch waits for them in the middle of the step.  A cell is a pixel's 64 channels in 144 bytes, a row's pitch continues the sequence of its cells' units: reads of 16
//    neighbouring slots are free of bank conflicts, across the end of a row too (conv3x3_f16.hip).  Cells left and right of a row are zeros.
#include <algorithm>
#include <type_traits>

#include "mfma_tile.hpp"

namespace nncv_hip {

using namespace mt;

namespace {

constexpr unsigned kOOBb = 0x7fffff00u;  // byte offset beyond any buffer this kernel accepts
constexpr int kCell = 144, kInBlocks = 5, kMidBlocks = 3, kMostW = 64, kMostRow = 256;  // slots of a row; pixels of a row (in columns)
constexpr int kEach = 3;  // load instructions of a wave for a step's rows, at most
typedef __attribute__((address_space(3))) void* lds_ptr_t;
__device__ __forceinline__ void fetch16(__amdgpu_buffer_rsrc_t rs, unsigned char* lds, unsigned voffset) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr_t)lds, 16, voffset, 0, 0, 0);
}
constexpr int row_bytes(int W) { return (W + 2) * kCell + 224; }                       // = W * 144 modulo 256
constexpr int in_block(int W, int R) { return (R * row_bytes(W) + 1023) / 1024 * 1024; }  // whole load instructions
constexpr int step_rows(int W) { return W <= 32 ? 4 : W <= 42 ? 3 : 2; }
constexpr int lds_bytes(int Wi, int Wo) {  // slots of a row of the first and of the second convolution
  const int R = step_rows(Wi);
  return kInBlocks * in_block(Wi, R) + kMidBlocks * R * row_bytes(Wo) + (R == 2 ? 1024 : 0);
}
static_assert(lds_bytes(32, 32) <= 160 * 1024 && lds_bytes(42, 42) <= 160 * 1024 && lds_bytes(kMostW, kMostW) <= 160 * 1024, "LDS of a CU");
static_assert(in_block(32, 4) <= kEach * 8 * 1024 && in_block(42, 3) <= kEach * 8 * 1024 && in_block(kMostW, 2) <= kEach * 8 * 1024, "a step's rows are three instructions a wave");

// columns a row is cut into, their pixels (of the last one at most), slots of a row of the first convolution, rows of a step
struct Cut { int cols, Wo, Wi, R; };
Cut cut_of(int W) {
  if (W <= kMostW) return Cut{1, W, W, step_rows(W)};
  Cut best{0, 0, 0, 1};
  for (int c = 2; c <= 8; ++c) {
    const int Wo = (W + c - 1) / c, R = step_rows(Wo + 2);
    if (R > 2 && (c - 1) * Wo < W && (!best.cols || c * best.R < best.cols * R)) best = Cut{c, Wo, Wo + 2, R};
  }
  return best;
}

struct BlockArgs {
  const void* in; void* out; const void* wf1; const void* wf2;
  const float* scale1; const float* shift1; const float* scale2; const float* shift2;
  int H, W, Wi, Wo, R, cols, strips, rows;  // Cut; strips of an image, their rows (whole steps)
  float inv_row;           // 1 / 16-byte units of a row
};

template <bool TALL, bool WIDE>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void basic_block_kernel(const BlockArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  static_assert(TALL || !WIDE, "columns have three or four rows a step");
  const int W = a.W, H = a.H, R = TALL ? a.R : 2, Wi = WIDE ? a.Wi : W, Wo = WIDE ? a.Wo : W;
  const int rowI = (Wi + 2) * kCell + 224, rowM = WIDE ? (Wo + 2) * kCell + 224 : rowI, inB = (R * rowI + 1023) & ~1023, midB = R * rowM;
  const int mid0 = kInBlocks * inB;
  // scale and shift of both, in pieces of 32 channels: behind the rows; TALL: a piece in what is spare behind each of the first eight of them
  auto tab = [&](int piece) __attribute__((always_inline)) {
    return reinterpret_cast<float*>(smem + mid0 + (TALL ? piece * rowM + (Wo + 2) * kCell : kMidBlocks * midB + piece * 128));
  };
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lrow = lane & 31, lh = lane >> 5, second = wave >> 2, fg = wave & 1, half = (wave >> 1) & 1;
  const int part_of = WIDE ? blockIdx.x / a.cols : blockIdx.x, x0 = WIDE ? (blockIdx.x - part_of * a.cols) * Wo : 0;  // first column of the result
  const int n = part_of / a.strips, strip = part_of - n * a.strips;
  const int y0 = strip * a.rows, y1 = min(y0 + a.rows, H), K = (y1 - y0 + R - 1) / R;  // steps' rows of the result
  const long long image = (long long)n * H * W * 128;
  const __amdgpu_buffer_rsrc_t rs_in = make_rsrc(static_cast<const char*>(a.in) + image, (unsigned)(H * W) * 128u);
  const __amdgpu_buffer_rsrc_t rs_out = make_rsrc(static_cast<char*>(a.out) + image, (unsigned)(H * W) * 128u);

  // ---- loader: unit u of a step's rows is part of a cell, of the spare 16 bytes behind it or of those behind the row ----
  const int units = rowI >> 4, calls = inB >> 10;
  unsigned from[kEach];  // row << 20 | byte behind the first row's start; all ones: zeros
#pragma unroll
  for (int i = 0; i < kEach; ++i) {
    int v;
    const int u = (i * 8 + wave) * 64 + lane, r = fast_div(u, units, a.inv_row, &v), cell = (v * 7282) >> 16, part = v - cell * 9;
    const int x = x0 + cell - (WIDE ? 2 : 1);
    const bool ok = r < R && part < 8 && cell < Wi + 2 && (unsigned)x < (unsigned)W;
    from[i] = ok ? (unsigned)(r << 20 | ((r * W + x) * 128 + part * 16)) : ~0u;
  }
  auto fetch = [&](int b, int slot) __attribute__((always_inline)) {  // block b of the input: rows y0 - 2 + R b ..
    const int y = y0 - 2 + R * b;
#pragma unroll
    for (int i = 0; i < kEach; ++i)
      if (i * 8 + wave < calls) fetch16(rs_in, smem + slot * inB + (i * 8 + wave) * 1024, from[i] != ~0u && (unsigned)(y + (int)(from[i] >> 20)) < (unsigned)H ? (unsigned)(y * W * 128) + (from[i] & 0xfffffu) : kOOBb);
  };
  fetch(0, 0);
  fetch(1, 1);
  u32x4 w[36];
  {
    const __amdgpu_buffer_rsrc_t rs_w = make_rsrc(second ? a.wf2 : a.wf1, 2u * 36u * 1024u);
#pragma unroll
    for (int q = 0; q < 36; ++q) w[q] = __builtin_amdgcn_raw_buffer_load_b128(rs_w, (unsigned)lane * 16u, (unsigned)((fg * 36 + q) * 1024), 0);
  }
  for (int i = tid * 16; i < kMidBlocks * midB; i += 512 * 16) *reinterpret_cast<u32x4*>(smem + mid0 + i) = u32x4{0, 0, 0, 0};
  if constexpr (TALL) __syncthreads();
  if (tid < 64) {
    const int h = tid >> 5, f = tid & 31;
    tab(h)[f] = a.scale1[tid], tab(2 + h)[f] = a.shift1[tid];
    tab(4 + h)[f] = a.scale2[tid], tab(6 + h)[f] = a.shift2[tid];
  }

  // ---- this lane's two slots: pixel x of row i of the block; slots behind the last pixel read with one 16, 32 .. before them ----
  const int Ws = WIDE && second ? Wo : Wi;
  int xs[2], is[2];
  bool there[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    int s = (2 * half + u) * 32 + lrow;
    there[u] = s < R * Ws;
    if (s >= R * Ws) s -= (((s - R * Ws) >> 4) + 1) << 4;
    is[u] = s >= Ws ? 1 : 0;
    if constexpr (TALL) is[u] += (s >= 2 * Ws ? 1 : 0) + (s >= 3 * Ws ? 1 : 0);
    xs[u] = s - is[u] * Ws;
  }
  // byte of tap (r, 0) of a slot: block t (first convolution: of the input; second: of the rows between) and two rows of the one behind it
  const int block = second ? midB : inB, rowB = second ? rowM : rowI, ring0 = second ? mid0 : 0, ring_end = ring0 + (second ? kMidBlocks * midB : kInBlocks * inB), ring = ring_end - ring0;
  int base[3][2];
#pragma unroll
  for (int r = 0; r < 3; ++r)
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int j = is[u] + r;
      base[r][u] = ring0 + (j >= R ? block + (j - R) * rowB : j * rowB) + xs[u] * kCell + lh * 16;
    }
  // A slot's place in 3 bytes.  WIDE: opaque to the compiler, which would keep what follows from it in registers beyond the 256 (14 spilled)
  unsigned place[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) place[u] = (unsigned)(xs[u] | is[u] << 8 | (there[u] ? 1 << 16 : 0));
  auto placed = [&](int u) __attribute__((always_inline)) {
    unsigned v = place[u];
    if constexpr (WIDE) asm volatile("" : "+v"(v));
    return v;
  };
  const int f0 = fg * 32 + 16 * lh;  // this lane's 16 consecutive channels
  const float *sc = tab(second * 4 + fg) + 16 * lh, *sh = tab(second * 4 + 2 + fg) + 16 * lh;
  floatx16 acc[2];
  int slot_in = 2, slot_mid = 0, slot_res = TALL ? 0 : 1;  // of the block to fetch, to write between the convolutions, of the (first) block of x to add

  auto scaled = [&](int u, float (&y)[16]) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const floatx4 m = *reinterpret_cast<const floatx4*>(sc + 4 * q), h = *reinterpret_cast<const floatx4*>(sh + 4 * q);
#pragma unroll
      for (int e = 0; e < 4; ++e) y[4 * q + e] = acc[u][4 * q + e] * m[e] + h[e];
    }
  };
  auto halves = [](const float (&y)[16], int c) __attribute__((always_inline)) {
    half8 v;
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = (half_t)y[8 * c + e];
    return __builtin_bit_cast(u32x4, v);
  };
  // the first convolution's rows y0 - 1 + R t ..: to LDS, zeros where they lie outside the image
  auto between = [&](int t) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const unsigned v = placed(u);
      const int x = v & 255, i = v >> 8 & 255;
      float y[16];
      scaled(u, y);
      act_apply_n<true>(y, kActRelu);
      const bool inside = (unsigned)(y0 - 1 + R * t + i) < (unsigned)H && (!WIDE || (unsigned)(x0 - 1 + x) < (unsigned)W);
      unsigned char* to = smem + mid0 + slot_mid * midB + i * rowM + (x + (WIDE ? 0 : 1)) * kCell + f0 * 2;
      if (v >> 16) {
#pragma unroll
        for (int c = 0; c < 2; ++c) *reinterpret_cast<u32x4*>(to + 16 * c) = inside ? halves(y, c) : u32x4{0, 0, 0, 0};
      }
    }
    slot_mid = slot_mid == kMidBlocks - 1 ? 0 : slot_mid + 1;
  };
  // the second one's rows y0 + R k ..: x (from row 2 of block k on) added, to memory (always four stores)
  auto result = [&](int k) __attribute__((always_inline)) {
    const int next = slot_res == kInBlocks - 1 ? 0 : slot_res + 1;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const unsigned v = placed(u);
      const int xo = v & 255, i = v >> 8 & 255;
      float y[16];
      scaled(u, y);
      int xrow = slot_res * inB + i * rowI;
      if constexpr (TALL) xrow = i + 2 < R ? xrow + 2 * rowI : next * inB + (i + 2 - R) * rowI;
      const unsigned char* x = smem + xrow + (xo + (WIDE ? 2 : 1)) * kCell + f0 * 2;
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const half8 add = *reinterpret_cast<const half8*>(x + 16 * c);
#pragma unroll
        for (int e = 0; e < 8; ++e) y[8 * c + e] += (float)add[e];
      }
      act_apply_n<true>(y, kActRelu);
      const int yo = y0 + R * k + i;
      const unsigned o = v >> 16 && yo < y1 && (!WIDE || x0 + xo < W) ? (unsigned)((yo * W + x0 + xo) * 128 + f0 * 2) : kOOBb;
#pragma unroll
      for (int c = 0; c < 2; ++c) __builtin_amdgcn_raw_buffer_store_b128(halves(y, c), rs_out, o + 16u * c, 0, 0);
    }
    slot_res = next;
  };
  auto fetch_next = [&](int t) __attribute__((always_inline)) {
    if (t + 2 <= K + 1) {
      fetch(t + 2, slot_in);
      slot_in = slot_in == kInBlocks - 1 ? 0 : slot_in + 1;
    }
  };
  // TALL: results read x from the block whose place the next one takes
  auto results_read = [&](int t) __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0xc07f);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    fetch_next(t);
    __builtin_amdgcn_sched_barrier(0);
  };
  auto products = [&](int t) __attribute__((always_inline)) {
    constexpr int kAhead = 2;
    u32x4 p[36][2];
    auto read = [&](auto q_c) __attribute__((always_inline)) {
      constexpr int q = decltype(q_c)::value, tap = q >> 2;
#pragma unroll
      for (int u = 0; u < 2; ++u) p[q][u] = *reinterpret_cast<const u32x4*>(smem + base[tap / 3][u] + (tap % 3) * kCell + (q & 3) * 32);
    };
    read(std::integral_constant<int, 0>());
    read(std::integral_constant<int, 1>());
    auto steps = [&](auto self, auto q_c) __attribute__((always_inline)) -> void {
      constexpr int q = decltype(q_c)::value;
      if constexpr (q < 36) {
        if constexpr (q + kAhead < 36) read(std::integral_constant<int, q + kAhead>());
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          if constexpr (q == 0) Mma<half_t>::start(w[q], p[q][u], acc[u]);
          else Mma<half_t>::run(w[q], p[q][u], acc[u]);
        }
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (TALL && q == 24) {
          if (!second) results_read(t);
        }
        self(self, std::integral_constant<int, q + 1>());
      }
    };
    steps(steps, std::integral_constant<int, 0>());
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int v = base[r][u] + block;
        base[r][u] = v >= ring_end ? v - ring : v;
      }
  };

  __builtin_amdgcn_s_waitcnt(0x0f70);  // filters and the first two steps' rows: waited for where they are used, every step would count them
  // Step t: the first convolution's block t (t <= K), the second one's block t - 2, and the results of its block t - 3.
  for (int t = 0; t < K + 3; ++t) {
    __builtin_amdgcn_sched_barrier(0);
    if (!TALL && second && t > 3) __builtin_amdgcn_s_waitcnt(0xc07f & (0x0f70 | 4));  // x's next rows (the last step's four stores may be on their way), LDS
    else __builtin_amdgcn_s_waitcnt(0x0070);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (!TALL) fetch_next(t);
    __builtin_amdgcn_sched_barrier(0);
    if (second && t > 2) result(t - 3);
    const bool work = second ? t >= 2 && t < K + 2 : t <= K;
    if constexpr (TALL) {
      if (second || !work) results_read(t);
    }
    if (work) products(t);
    if (!second && t <= K) between(t);
  }
}

}  // namespace

long long basic_block_steps(int N, int H, int W) {
  if (W < 24 || W > kMostRow || H < 2 || (long long)H * W * 128 >= (long long)kOOBb || N >= (1 << 20)) return 0;
  const Cut c = cut_of(W);
  return (long long)N * c.cols * ((H + c.R - 1) / c.R);
}

void launch_basic_block(const BasicBlockArgs& g, hipStream_t s) {
  NNCV_REQUIRE(basic_block_steps(g.N, g.H, g.W) > 0, "basic_block: shape not covered");
  const Cut cut = cut_of(g.W);
  const int R = cut.R;
  BlockArgs d{};
  d.in = g.in; d.out = g.out; d.wf1 = g.wf1; d.wf2 = g.wf2; d.scale1 = g.scale1; d.shift1 = g.shift1; d.scale2 = g.scale2; d.shift2 = g.shift2;
  d.H = g.H; d.W = g.W; d.R = R; d.Wi = cut.Wi; d.Wo = cut.Wo; d.cols = cut.cols;
  int strips = 1;
  double best = 1e30;
  for (int c = 1; c <= (g.H + R - 1) / R; ++c) {
    const int rows = ((g.H + c - 1) / c + R - 1) / R * R;
    if ((c - 1) * rows >= g.H) continue;
    const double us = std::ceil((double)g.N * cut.cols * c / 256) * (rows / R + 5);
    if (us < best) best = us, strips = c, d.rows = rows;
  }
  d.strips = strips;
  d.inv_row = 1.0f / (float)(row_bytes(cut.Wi) / 16);
  const int lds = lds_bytes(cut.Wi, cut.Wo);
  const auto kernel = cut.cols > 1 ? basic_block_kernel<true, true> : R == 2 ? basic_block_kernel<false, false> : basic_block_kernel<true, false>;
  static const bool attr = [] {
    for (auto k : {basic_block_kernel<false, false>, basic_block_kernel<true, false>, basic_block_kernel<true, true>})
      NNCV_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
    return true;
  }();
  (void)attr;
  const double px = (double)g.N * g.H * g.W;
  ProfScope prof("basic_block<f16,64>", 4.0 * px * 9 * 64 * 64, 2.0 * (2 * px * 64 + 2 * 9 * 64 * 64), s);
  launch_kernel(kernel, dim3((unsigned)(g.N * strips * cut.cols)), dim3(512), lds, s, d);
  NNCV_HIP_CHECK(hipGetLastError());
}

}  // namespace nncv_hip
