// The ResNet stem in one launch, fp32 (gfx950): conv 7x7 stride 2 pad 3 over 3 channels + BN + ReLU (tests/Nets/Res18.mlir:118-142)
// and max-pool 3x3 stride 2 (:144-151), NCHW image in, NHWC pooled activation out, the products on the bf16 matrix pipes (split.hpp).
//
// The walk is stem_pool.hip's: a wave owns a strip of 32 convolution columns (15 pooled ones) and goes down its pooled rows, the pixels are
// the rows of the products and the filters their columns, the pool is taken between accumulators of one lane.  What differs:
//   * a wave has 32 of the 64 filters: their three pieces are 132 registers.  Two waves walk the same rows, each on its own;
//   * image rows go through registers, are split once and lie in a ring of eight rows in LDS, [channel][piece][35 pairs of pixels]: a
//     row of pixels is read by up to four convolution rows.  The two rows that the next convolution row needs are requested a row ahead and
//     split under its products, where the row's oldest pair has been read for the last time;
//   * a convolution row is 66 products of 32 cycles; its sums are finished (BN, maximum) while the SIMD's other wave multiplies;
//   * a wave with a sum that is not finite takes the row again with the fp32 instructions, from memory (split.hpp).
// Bound: matrix instructions, 66 of 32 cycles a convolution row, strip and half of the filters (49 % of the cycles of six 231x309 images, where a
// wave has two pooled rows, a few three, and the row above them).  There 29 us, where packing, implicit GEMM and pool took 47; one
// 256x256 image 11.6 us (19.7).
#include <algorithm>
#include <type_traits>

#include "split.hpp"

namespace nncv_hip {

using namespace mt;

namespace {
constexpr int kPoolCols = 15, kPairs = 35;
constexpr int kPlane = 144;                  // 35 pairs of bf16, bytes
constexpr int kPitch = 9 * kPlane;           // of a ring row: three channels of three pieces
constexpr int kRing = 8 * kPitch;
constexpr int kSteps = 11;
constexpr int kFrag = 2 * kSteps * 3 * 1024; // [32 filters][step][piece][lane][8 bf16]
constexpr int kPlain = 64 * 168 * 4;         // [filter][row][channel][8]: column 0 is zero
constexpr unsigned kOOBs = 0x7fff0000u;
typedef u32x4 u32x4_a4 __attribute__((aligned(4)));

__device__ __forceinline__ float max2(float a, float b) { return __builtin_elementwise_maximum(a, b); }
}  // namespace

struct StemSplitArgs {
  const float* in;     // [N][3][H][W]
  const void* wt;      // launch_stem_weight_strip
  const float* scale;  // [64]
  const float* shift;  // [64]
  float* out;          // [N][PH][PW][64]
  int N, H, W, OH, OW, PH, PW;
  int strips, walks;
  int share;           // walks that divide a strip between them; 0: walk w is
  int run, extra;      // run pooled rows of the list [N][strips][PH], the first `extra` ones one more
  unsigned in_bytes;
};

// 16 bytes per lane from global memory straight into LDS, lane l to lds + 16 l
typedef __attribute__((address_space(3))) void* lds_ptr_t;
__device__ __forceinline__ void fetch16(__amdgpu_buffer_rsrc_t rs, unsigned char* lds, unsigned voffset) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr_t)lds, 16, voffset, 0, 0, 0);
}

__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void stem_pool_split_kernel(const StemSplitArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63, waves = blockDim.x >> 6;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n2 = lane & 31, half = lane >> 5;
  const int grp = wave & 1, f = 32 * grp + n2;  // this lane's filter
  unsigned char* zeros = smem + kFrag;
  unsigned char* ring = smem + kFrag + 16 + wave * kRing;
  const __amdgpu_buffer_rsrc_t rs_in = make_rsrc(a.in, a.in_bytes);
  const __amdgpu_buffer_rsrc_t rs_wt = make_rsrc(a.wt, (unsigned)(kFrag + kPlain));

  // an XCD takes neighbouring workgroups of the list
  const int grid = gridDim.x, per = grid >> 3, more = grid & 7, xcd = blockIdx.x & 7;
  const int wg = xcd * per + (xcd < more ? xcd : more) + (blockIdx.x >> 3);
  const int w = wg * (waves >> 1) + (wave >> 1);
  int strip, y, left = 0;
  if (a.share > 0) {
    strip = w / a.share;
    const int part = w - strip * a.share;
    y = part * a.PH / a.share;
    if (w < a.walks) left = (part + 1) * a.PH / a.share - y;
  } else {
    const int first = w * a.run + (w < a.extra ? w : a.extra);
    strip = first / a.PH;
    y = first - strip * a.PH;
    if (w < a.walks) left = a.run + (w < a.extra);
  }

  // ---- loader: lane l takes pixel pair l of the two image rows 2c + 4, 2c + 5 that convolution row c + 1 needs beyond row c; image row r is
  //      ring row (r - 3) & 7 ----
  const unsigned plane = (unsigned)(a.H * a.W) * 4u;
  int n = 0, px0 = 0;
  struct Pixels { float v[2][3][2]; };
  auto request = [&](Pixels& p, int row) {  // rows `row`, row + 1
    const int ix = 4 * px0 - 6 + 2 * lane;
    const bool ok0 = (lane < kPairs) & ((unsigned)ix < (unsigned)a.W), ok1 = (lane < kPairs) & ((unsigned)(ix + 1) < (unsigned)a.W);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const bool row_ok = (unsigned)(row + i) < (unsigned)a.H;
      const unsigned at = (unsigned)((row + i) * a.W + ix) * 4u;
      const unsigned o0 = (row_ok & ok0) ? at : kOOBs, o1 = (row_ok & ok1) ? at + 4u : kOOBs;
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        p.v[i][c][0] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs_in, o0, (unsigned)(n * 3 + c) * plane, 0));
        p.v[i][c][1] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs_in, o1, (unsigned)(n * 3 + c) * plane, 0));
      }
    }
  };
  auto deposit = [&](const Pixels& p, auto i_c, auto c_c, int row) {
    constexpr int i = decltype(i_c)::value, c = decltype(c_c)::value;
    unsigned q[3];
    split_pair(p.v[i][c][0], p.v[i][c][1], q);
    unsigned char* d = ring + ((row + i - 3) & 7) * kPitch + c * 3 * kPlane + (lane < kPairs ? lane : kPairs) * 4;  // the others on the spare pair
#pragma unroll
    for (int k = 0; k < 3; ++k) *reinterpret_cast<unsigned*>(d + k * kPlane) = q[k];
  };
  auto deposit_rows = [&](const Pixels& p, int row) {
    deposit(p, std::integral_constant<int, 0>(), std::integral_constant<int, 0>(), row);
    deposit(p, std::integral_constant<int, 0>(), std::integral_constant<int, 1>(), row);
    deposit(p, std::integral_constant<int, 0>(), std::integral_constant<int, 2>(), row);
    deposit(p, std::integral_constant<int, 1>(), std::integral_constant<int, 0>(), row);
    deposit(p, std::integral_constant<int, 1>(), std::integral_constant<int, 1>(), row);
    deposit(p, std::integral_constant<int, 1>(), std::integral_constant<int, 2>(), row);
  };
  // the rows 2c - 4 .. 2c + 3 of the walk's first convolution row c, and the two after them
  Pixels head[4], next;
  auto begin_walk = [&]() {
    n = strip / a.strips;
    px0 = (strip - n * a.strips) * kPoolCols;
    const int c = 2 * y - 1;
#pragma unroll
    for (int k = 0; k < 4; ++k) request(head[k], 2 * c - 4 + 2 * k);
    request(next, 2 * c + 4);
  };
  auto await_walk = [&]() {
#pragma unroll
    for (int k = 0; k < 4; ++k) deposit_rows(head[k], 2 * (2 * y - 1) - 4 + 2 * k);
  };

  // ---- once per wave: the filters, through LDS so that a workgroup fetches them once ----
  for (int k = wave; k < kFrag / 1024; k += waves) fetch16(rs_wt, smem + k * 1024, (unsigned)(k * 64 + lane) * 16u);
  const float sc = a.scale ? a.scale[f] : 1.0f, sh = a.shift ? a.shift[f] : 0.0f;
  if (tid < 4) reinterpret_cast<unsigned*>(zeros)[tid] = 0u;
  if (left > 0) {
    begin_walk();
    await_walk();  // (these requests are younger than the filters')
  }
  __builtin_amdgcn_sched_barrier(0);
  if (left <= 0) __builtin_amdgcn_s_waitcnt(0x0f70);
  __syncthreads();
  if (left <= 0) return;
  u32x4 wreg[kSteps][3];
#pragma unroll
  for (int s = 0; s < kSteps; ++s)
#pragma unroll
    for (int k = 0; k < 3; ++k) wreg[s][k] = *reinterpret_cast<const u32x4*>(smem + ((grp * kSteps + s) * 3 + k) * 1024 + lane * 16);

  // ---- operands: steps 0 .. 8 take the filter rows 0 .. 5 in pairs, row 2q on lanes 0 .. 31 and 2q + 1 on lanes 32 .. 63, a
  //      channel a step; step 9 the first two channels of row 6, step 10 its last one and zeros.  Row 8q + 4h + e of a product is pixel
  //      16h + 4q + e of the strip ----
  const int col = 16 * ((n2 >> 2) & 1) + 4 * (n2 >> 3) + (n2 & 3);
  const unsigned char* base = ring + col * 4;
  auto operand = [&](auto s_c, int c, u32x4 (&o)[3]) {
    constexpr int s = decltype(s_c)::value;
    const unsigned char* p = base + half * kPitch + ((2 * c - 6 + 2 * (s / 3)) & 7) * kPitch + (s % 3) * 3 * kPlane;
    if (s == 9) p = base + half * 3 * kPlane + ((2 * c) & 7) * kPitch;
    if (s == 10) p = base + 6 * kPlane + ((2 * c) & 7) * kPitch;
#pragma unroll
    for (int k = 0; k < 3; ++k) o[k] = *reinterpret_cast<const u32x4_a4*>(s == 10 && half ? zeros : p + k * kPlane);
  };

  floatx16 big[1][1], low[1][1];
  float st[16] = {};  // of the odd row above, then its maximum with the even row
  bool row_in = false;
  int thirds = -1;                // bit i: the third column of the lane's window i is inside
  bool left_in = true;            // the strip's first column is inside
  __amdgpu_buffer_rsrc_t rs_row = make_rsrc(a.out, 0u);
  unsigned dst = 0u, dst7 = 0u;

  // The row's sums once more with the fp32 instructions: step s is (filter row, channel) = (s / 3, s % 3), four columns a lane half.
  auto again = [&](int c) __attribute__((always_inline)) {
    const int ix0 = 2 * (2 * px0 - 1 + col) - 4 + 4 * half;
    plain_products(big, 21, [&](int s, u32x4 (&x)[1], u32x4 (&b)[1]) {
      const int r = s / 3, ch = s - 3 * r, iy = 2 * c - 3 + r;
      const bool in = (s < 21) & ((unsigned)iy < (unsigned)a.H);
#pragma unroll
      for (int e = 0; e < 4; ++e) {  // (not the pixel under column 0, whose weight is the padding's zero)
        const int ix = ix0 + e;
        const bool ok = in & ((unsigned)ix < (unsigned)a.W) & (half + e > 0);
        x[0][e] = __builtin_amdgcn_raw_buffer_load_b32(rs_in, ok ? (unsigned)(iy * a.W + ix) * 4u : kOOBs, (unsigned)(n * 3 + ch) * plane, 0);
      }
      b[0] = __builtin_amdgcn_raw_buffer_load_b128(rs_wt, s < 21 ? (unsigned)(kFrag + ((f * 21 + s) * 8 + 4 * half) * 4) : kOOBs, 0, 0);
    });
  };

  u32x4 lead[3];
  // One convolution row: its products, the deposit of the rows that came for the next one, and what its sums are worth.
  auto walk_row = [&](int c) __attribute__((always_inline)) {
    u32x4 o[2][3];
#pragma unroll
    for (int k = 0; k < 3; ++k) o[0][k] = lead[k];
    const floatx16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    auto steps = [&](auto self, auto s_c) -> void {
      constexpr int s = decltype(s_c)::value;
      if constexpr (s < kSteps) {
        u32x4(&cur)[3] = o[s & 1];
        if constexpr (s + 1 < kSteps) operand(std::integral_constant<int, s + 1>(), c, o[(s + 1) & 1]);
        else operand(std::integral_constant<int, 0>(), c + 1, lead);
        __builtin_amdgcn_sched_barrier(0);
        constexpr int kX[6] = {0, 0, 1, 0, 1, 2}, kY[6] = {0, 1, 0, 2, 1, 0};
#pragma unroll
        for (int p = 0; p < 6; ++p) {
          floatx16& sum = p == 0 ? big[0][0] : low[0][0];
          sum = mma_bf16(cur[kX[p]], wreg[s][kY[p]], s == 0 && p < 2 ? zero : sum);
          if (p == 2) {
            // (the pair that these rows take the place of was read in steps 0 .. 2)
            if constexpr (s >= 4 && s < 10) deposit(next, std::integral_constant<int, (s - 4) / 3>(), std::integral_constant<int, (s - 4) % 3>(), 2 * c + 4);
            if constexpr (s == 10) request(next, 2 * c + 6);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
        self(self, std::integral_constant<int, s + 1>());
      }
    };
    steps(steps, std::integral_constant<int, 0>());
    if (__builtin_expect(split_sums(big, low), 0)) again(c);
    float hold = 0.0f, beyond = 0.0f;
    auto window = [&](int i, float two, float third) {
      third = (thirds >> i) & 1 ? third : 0.0f;
      const float v = max2(max2(two, third), 0.0f);
      __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), rs_row, i < 7 ? dst + i * 256 : dst7, 0, 0);
    };
    if (c & 1) {
#pragma unroll
      for (int p = 0; p < 16; ++p) {
        const float lo = row_in ? big[0][0][p] * sc + sh : 0.0f;
        float v = max2(st[p], lo);
        st[p] = lo;
        if (p == 0) {
          v = left_in ? v : 0.0f;
          const unsigned b = __builtin_bit_cast(unsigned, v);
          const unsigned upper = __builtin_amdgcn_permlane32_swap(b, b, false, false)[1];  // on the lower lanes the upper ones' first column
          beyond = __builtin_bit_cast(float, upper);
        }
        if (p > 0 && p % 2 == 0) window(p / 2 - 1, hold, v);
        hold = p % 2 ? max2(hold, v) : v;
        if (p == 15) window(7, hold, beyond);
      }
    } else {
#pragma unroll
      for (int p = 0; p < 16; ++p) st[p] = max2(st[p], big[0][0][p] * sc + sh);
    }
  };

  for (;;) {
    const int count = left < a.PH - y ? left : a.PH - y;
    left_in = (px0 > 0) | (half > 0);
    const int last = a.PW - 1 - px0 - 8 * half;
    thirds = (a.OW & 1) != 0 && (unsigned)last < 8u ? ~(1 << last) : -1;
    dst = (unsigned)((px0 + 8 * half) * 256 + f * 4);
    dst7 = half ? kOOBs : dst + 7 * 256;
    operand(std::integral_constant<int, 0>(), 2 * y - 1, lead);
    // from the odd row above the first window, which completes none, to the last window's odd row
    for (int c = 2 * y - 1; c < 2 * (y + count); ++c) {
      if (c & 1) {
        row_in = (unsigned)c < (unsigned)a.OH;
        const int py = c >> 1;
        rs_row = make_rsrc(a.out + ((long long)n * a.PH + max(py, 0)) * a.PW * 64, py >= y ? (unsigned)a.PW * 256u : 0u);
      }
      walk_row(c);
    }
    left -= count;
    if (left <= 0) break;
    ++strip;
    y = 0;
    begin_walk();
    await_walk();
  }
}

// The split filters, [filter group][step][piece][lane][8], and behind them the filters as they are, [filter][row][channel][8].
__global__ void stem_weight_strip_split_kernel(const float* __restrict__ w, unsigned char* __restrict__ dst) {
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx < kFrag / 3 / 16 * 4) {  // a pair of halves of a lane's eight
    const int e = (idx & 3) * 2, lane = (idx >> 2) & 63, s = (idx >> 8) % kSteps, g = (idx >> 8) / kSteps;
    const int half = lane >> 5, f = 32 * g + (lane & 31);
    const int r = s < 9 ? 2 * (s / 3) + half : 6, c = s < 9 ? s % 3 : s == 9 ? half : 2 + half;
    float v[2];
    for (int k = 0; k < 2; ++k) v[k] = (c < 3 && e + k > 0) ? w[((f * 3 + c) * 7 + r) * 7 + e + k - 1] : 0.0f;
    unsigned p[3];
    split_pair(v[0], v[1], p);
    for (int k = 0; k < 3; ++k) *reinterpret_cast<unsigned*>(dst + (((g * kSteps + s) * 3 + k) * 64 + lane) * 16 + e * 2) = p[k];
  }
  if (idx < kPlain / 4) {
    const int x = idx & 7, c = (idx >> 3) % 3, r = (idx / 24) % 7, f = idx / 168;
    reinterpret_cast<float*>(dst + kFrag)[idx] = x > 0 ? w[((f * 3 + c) * 7 + r) * 7 + x - 1] : 0.0f;
  }
}

size_t stem_weight_strip_split_bytes() { return kFrag + kPlain; }

void launch_stem_weight_strip_split(const void* w, void* dst, hipStream_t s) {
  const int threads = std::max(kFrag / 3 / 16 * 4, kPlain / 4);
  launch_kernel(stem_weight_strip_split_kernel, dim3((threads + 255) / 256), dim3(256), 0, s, static_cast<const float*>(w), static_cast<unsigned char*>(dst));
  NNCV_HIP_CHECK(hipGetLastError());
}

void launch_stem_pool_split(const void* in, const void* wt, const float* scale, const float* shift, void* out, int N, int H, int W, hipStream_t s) {
  StemSplitArgs a{};
  a.in = static_cast<const float*>(in); a.wt = wt; a.scale = scale; a.shift = shift;
  a.out = static_cast<float*>(out);
  a.N = N; a.H = H; a.W = W;
  a.OH = (H + 6 - 7) / 2 + 1; a.OW = (W + 6 - 7) / 2 + 1;
  a.PH = (a.OH + 2 - 3) / 2 + 1; a.PW = (a.OW + 2 - 3) / 2 + 1;
  a.strips = (a.PW + kPoolCols - 1) / kPoolCols;
  const long long rows = (long long)N * a.strips * a.PH;
  NNCV_REQUIRE(rows < (1ll << 30), "stem: too many rows");
  // 1024 walks of two waves each are two waves on every SIMD (see launch_stem_pool)
  a.walks = rows < 1024 ? (int)rows : 1024;
  a.run = (int)(rows / a.walks);
  a.extra = (int)(rows % a.walks);
  const int all_strips = N * a.strips, share = std::min(a.walks / all_strips, a.PH);
  if (share > 0 && (a.PH + share - 1) / share <= a.run + (a.extra > 0) + 1) {
    a.share = share;
    a.walks = all_strips * share;
  }
  a.in_bytes = (unsigned)((size_t)N * 3 * H * W * 4);
  const int waves = a.walks <= 512 ? 4 : 8;  // a CU each while there are CUs
  const int lds = kFrag + 16 + waves * kRing;
  static const bool attr = [] {
    NNCV_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(stem_pool_split_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kFrag + 16 + 8 * kRing));
    return true;
  }();
  (void)attr;
  const double flops = 2.0 * N * a.OH * a.OW * 64.0 * 147.0;
  const double bytes = 4.0 * ((double)N * 3 * H * W + (double)N * a.PH * a.PW * 64 + 64.0 * 147);
  ProfScope prof("stem_conv7x7_bn_relu_maxpool<f32,split>", flops, bytes, s);
  launch_kernel(stem_pool_split_kernel, dim3((2 * a.walks + waves - 1) / waves), dim3(64 * waves), lds, s, a);
  NNCV_HIP_CHECK(hipGetLastError());
}

}  // namespace nncv_hip
