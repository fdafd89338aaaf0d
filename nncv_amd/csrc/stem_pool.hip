// ResNet stem in one launch (gfx950, fp16): conv 7x7 stride 2 pad 3 over 3 channels + BN + ReLU
// (tests/Nets/Res18.mlir:118-142) followed by max-pool 3x3 stride 2 over a -inf halo of 1
// (tests/Nets/Res18.mlir:144-151), NCHW image in, NHWC pooled activation out.
//
// The 112x112x64 convolution output (51 MB at batch 32, four times the pooled tensor) never reaches memory, nor LDS.
// A WAVE owns a strip of 32 convolution columns (15 pooled ones) and walks down its pooled rows; waves share nothing but
// the filters they start with, there is no barrier in the walk:
//   1. the image rows of a strip lie in a ring of 16 rows in LDS, the three planes one behind the other.  Four rows, one pooled
//      row's worth, go there straight from memory (buffer_load ... lds, a pixel pair a lane) a whole pooled row ahead;
//   2. a filter row of a channel is eight pixels = 16 bytes of a plane, so K is 7 x 3 x 8 = 168, padded to 176: 11 steps of 16
//      (rows of eight pixels of four channels, aligned to 16 bytes, were 14).  An output pixel's eight start one pair behind its left
//      neighbour's: every MFMA operand is 16 bytes at an address that is a multiple of four, with no im2col anywhere (the
//      eighth pixel of a row is the image pixel left of the window under a zero weight: a non-finite pixel there turns into NaN);
//   3. all 64 filters sit in 88 registers for the life of the wave: a convolution row of 32 columns is 22 MFMAs behind 11
//      LDS reads.  The pixels are the rows of the products and the filters their columns, so a lane has ONE pair of neighbouring filters (two scales,
//      two shifts) and 16 neighbouring pixels of a row;
//   4. scale / shift in fp32, one rounding to fp16, the lane's two filters packed, then the 3x3 maximum in registers: the
//      rows of a window are accumulators of the same place (the last row stays for the next window: no row is computed twice
//      inside a walk), the columns neighbouring registers; one value comes from the other half of the wave.  v_pk_maximum3_f16 is
//      the NaN-propagating arith.maximumf of three values, so ReLU is one more maximum with +0 at the end, and +0 stands for every
//      pixel outside the convolution output;
//   5. 32 lanes store the 128 bytes of a pooled pixel, two pixels an instruction.
// The epilogue of a convolution row runs in pieces between the MFMAs of the next one, so one wave alone keeps both the matrix
// and the vector unit busy; two waves share a SIMD.  The list of all pooled rows of all strips is dealt to the waves in runs
// of equal length, so the last wave of a launch ends with the first.
//
// Bound: matrix instructions, 44 of 32 cycles a pooled row and strip, and the power they draw: on pixels and filters as
// they are this chip sustains 1.5-1.6 PFLOP/s of them (2.36 on zeros) at 1.6-1.7 GHz.  At batch 256, 224x224, the launch takes 92 us,
// 1030 TFLOP/s executed (the workgroup-tiled kernel before it, whose convolution tile went through LDS to the pool between
// two barriers: 122); batch 32 19.6 us (20.4), one image 5.8 (6.6).  The transposed product (filters as rows, 16 channels of one
// pixel a lane: tables of scale and shift in LDS, maxima over columns across lanes) took 105 us.  Odd widths, which went through a packed
// copy, an implicit GEMM and the pool, take this kernel too.
#include <algorithm>
#include <type_traits>

#include "mfma_tile.hpp"

namespace nncv_hip {

using namespace mt;

namespace {
constexpr int kPoolCols = 15;                // pooled columns of a strip: its 32 convolution columns are 2 * px0 - 1 ..
constexpr int kPairs = 35;                   // pixel pairs of an image row that the strip's windows touch
constexpr int kPlane = 256;                  // bytes of a ring row's channel: a dword a lane, the first 35 are read
constexpr int kPitch = 3 * kPlane;
constexpr int kRing = 16 * kPitch;
constexpr int kSteps = 11;
constexpr int kWtBytes = 2 * kSteps * 1024;  // fragments of a wave: [filter of a lane's pair][step][lane][8 halves]
constexpr int kLds = 4 * kRing + kWtBytes + 16;  // rings, filters, zeros
constexpr unsigned kOOBs = 0x7fff0000u;

typedef half_t half2v __attribute__((ext_vector_type(2)));
typedef u32x4 u32x4_a4 __attribute__((aligned(4)));

// waits until at most N of this wave's vector-memory requests are outstanding
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt(0x0f70 | (N & 15) | ((N >> 4) << 14));
  __builtin_amdgcn_sched_barrier(0);
}

__device__ __forceinline__ unsigned max2(unsigned a, unsigned b) {
  return __builtin_bit_cast(unsigned, __builtin_elementwise_maximum(__builtin_bit_cast(half2v, a), __builtin_bit_cast(half2v, b)));
}
}  // namespace

struct StemPoolArgs {
  const half_t* in;    // [N][3][H][W]
  const void* wt;      // launch_stem_weight_strip
  const float* scale;  // [64]
  const float* shift;  // [64]
  half_t* out;         // [N][PH][PW][64]
  int N, H, W, OH, OW, PH, PW;
  int strips;             // of an image
  int waves;
  int share;              // waves that divide a strip between them; 0: wave w walks
  int run, extra;         // run pooled rows of the list [N][strips][PH], the first `extra` waves one more
  unsigned in_bytes;
};

// 4 or 16 bytes per lane from global memory straight into LDS, lane l to lds + 4 l or 16 l
typedef __attribute__((address_space(3))) void* lds_ptr_t;
__device__ __forceinline__ void fetch16(__amdgpu_buffer_rsrc_t rs, unsigned char* lds, unsigned voffset) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr_t)lds, 16, voffset, 0, 0, 0);
}
__device__ __forceinline__ void fetch4(__amdgpu_buffer_rsrc_t rs, unsigned char* lds, unsigned voffset, unsigned soffset) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr_t)lds, 4, voffset, soffset, 0, 0);
}

// kDirect: every pixel pair is an aligned dword (W even, the image at a multiple of four bytes) and goes straight to LDS; otherwise
// pixels come one by one through registers, two rows at a time.
template <bool kDirect>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void stem_pool_kernel(const StemPoolArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  unsigned char* wlds = smem + 4 * kRing;
  unsigned char* zeros = wlds + kWtBytes;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n2 = lane & 31, half = lane >> 5;  // this lane's filters are 2 n2 and 2 n2 + 1, its pixels columns 16 half .. 16 half + 15 of the strip
  unsigned char* ring = smem + wave * kRing;
  const __amdgpu_buffer_rsrc_t rs_in = make_rsrc(a.in, a.in_bytes);
  const __amdgpu_buffer_rsrc_t rs_wt = make_rsrc(a.wt, (unsigned)kWtBytes);
  const __amdgpu_buffer_rsrc_t rs_sc = make_rsrc(a.scale ? (const void*)a.scale : (const void*)a.in, a.scale ? 256u : 0u);
  const __amdgpu_buffer_rsrc_t rs_sh = make_rsrc(a.shift ? (const void*)a.shift : (const void*)a.in, a.shift ? 256u : 0u);

  // an XCD takes neighbouring workgroups of the list: strips of one image share an L2
  const int grid = gridDim.x, per = grid >> 3, more = grid & 7, xcd = blockIdx.x & 7;
  const int wg = xcd * per + (xcd < more ? xcd : more) + (blockIdx.x >> 3);
  const int w = wg * 4 + wave;
  int strip, y, left = 0;  // the walk's strip and next pooled row, and the pooled rows to go
  if (a.share > 0) {
    strip = w / a.share;
    const int part = w - strip * a.share;
    y = part * a.PH / a.share;
    if (w < a.waves) left = (part + 1) * a.PH / a.share - y;
  } else {
    const int first = w * a.run + (w < a.extra ? w : a.extra);
    strip = first / a.PH;
    y = first - strip * a.PH;
    if (w < a.waves) left = a.run + (w < a.extra);
  }

  // ---- loader: lane l takes pixel pair l of each of a batch's four rows.  Batch y is image rows 4y + 3 .. 4y + 6, what
  //      the two convolution rows of pooled row y need beyond what pooled row y - 1 needed; image row r is ring row (r - 3) & 15 ----
  const unsigned plane = (unsigned)(a.H * a.W) * 2u;
  int n = 0, px0 = 0;  // of the strip being walked
  auto offset = [&](int y, int i, int p) -> unsigned {  // of pixel p of the lane's pair in row i of batch y, inside a plane
    const int iy = 4 * y + 3 + i, ix = 4 * px0 - 6 + 2 * lane + p;  // convolution column 2 px0 - 1 starts at pixel 4 px0 - 5; one further left for whole pairs
    const bool ok = (lane < kPairs) & ((unsigned)iy < (unsigned)a.H) & ((unsigned)ix < (unsigned)a.W);
    return ok ? (unsigned)(iy * a.W + ix) * 2u : kOOBs;
  };
  auto fetch = [&](int y) {
    int rows = ((4 * y) & 15) * kPitch;
    asm("" : "+s"(rows));  // twelve LDS addresses from here, not twelve kept for each place in the ring
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const unsigned o = offset(y, i, 0);
#pragma unroll
      for (int c = 0; c < 3; ++c) fetch4(rs_in, ring + rows + i * kPitch + c * kPlane, o, (unsigned)(n * 3 + c) * plane);
    }
  };
  struct Pixels { unsigned short v[2][3][2]; };  // [row][channel][pixel]: half a batch
  auto request = [&](Pixels& p, int y, int hb) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const unsigned o = offset(y, 2 * hb + i, k);
#pragma unroll
        for (int c = 0; c < 3; ++c) p.v[i][c][k] = (unsigned short)__builtin_amdgcn_raw_buffer_load_b16(rs_in, o, (unsigned)(n * 3 + c) * plane, 0);
      }
  };
  auto deposit = [&](const Pixels& p, int y, int hb) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int c = 0; c < 3; ++c)
        *reinterpret_cast<unsigned*>(ring + (((4 * y) & 15) + 2 * hb + i) * kPitch + c * kPlane + lane * 4) = p.v[i][c][0] | ((unsigned)p.v[i][c][1] << 16);
  };
  Pixels next;  // kDirect does without

  // the rows that the odd convolution row above the first window and that window need
  Pixels p[kDirect ? 1 : 6];
  auto begin_walk = [&]() {
    n = strip / a.strips;
    px0 = (strip - n * a.strips) * kPoolCols;
    if constexpr (kDirect) {
      fetch(y - 2);
      fetch(y - 1);
      fetch(y);
      fetch(y + 1);
    } else {
#pragma unroll
      for (int k = 0; k < 6; ++k) request(p[k], y - 2 + k / 2, k & 1);
      request(next, y + 1, 0);
    }
  };
  auto await_walk = [&]() {
    if constexpr (kDirect) {
      wait_vmcnt<12>();  // all but the last batch
    } else {
#pragma unroll
      for (int k = 0; k < 6; ++k) deposit(p[k], y - 2 + k / 2, k & 1);
    }
  };

  // ---- once per wave: the filters, through LDS so that a workgroup fetches them once, while the first rows are on their way ----
  float sc[2], sh[2];
#pragma unroll
  for (int g = 0; g < 2; ++g) {  // a missing vector is a buffer of no bytes: the load returns zeros
    sc[g] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs_sc, (unsigned)(2 * n2 + g) * 4u, 0, 0));
    sh[g] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs_sh, (unsigned)(2 * n2 + g) * 4u, 0, 0));
    if (!a.scale) sc[g] = 1.0f;
  }
  static_assert(2 * kSteps % 4 == 2, "every wave fetches five fragments, the first two one more");
#pragma unroll
  for (int k = 0; k < 5; ++k) fetch16(rs_wt, wlds + (4 * k + wave) * 1024, (unsigned)((4 * k + wave) * 64 + lane) * 16u);
  if (wave < 2) fetch16(rs_wt, wlds + (20 + wave) * 1024, (unsigned)((20 + wave) * 64 + lane) * 16u);
  if (tid < 4) reinterpret_cast<unsigned*>(zeros)[tid] = 0u;
  __builtin_amdgcn_sched_barrier(0);
  if (left > 0) {
    begin_walk();
    await_walk();
  } else {
    wait_vmcnt<0>();
  }
  __builtin_amdgcn_s_waitcnt(0xc07f);  // LDS operations; the last batch of rows stays on its way
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  if (left <= 0) return;
  u32x4 wreg[kSteps][2];
#pragma unroll
  for (int g = 0; g < 2; ++g)
#pragma unroll
    for (int s = 0; s < kSteps; ++s) wreg[s][g] = *reinterpret_cast<const u32x4*>(wlds + (g * kSteps + s) * 1024 + lane * 16);

  // ---- operands.  The K axis: steps 0 .. 8 take the filter rows 5 .. 0 in pairs, row 2q on lanes 0 .. 31 and 2q + 1 on lanes 32 .. 63,
  //      a channel a step; step 9 the first two channels of row 6, step 10 its last one and zeros.  Convolution row c
  //      starts at image row 2c - 3, an even ring row: a pair of rows does not wrap.  Row 8q + 4h + e of the product is pixel
  //      16h + 4q + e: a lane's accumulators are 16 neighbouring pixels ----
  const unsigned char* base = ring + (16 * ((n2 >> 2) & 1) + 4 * (n2 >> 3) + (n2 & 3)) * 4;
  auto operand = [&](auto s_c, int c) -> u32x4 {
    constexpr int s = decltype(s_c)::value;
    const unsigned char* p = base + half * kPitch + ((2 * c - 2 - 2 * (s / 3)) & 15) * kPitch + (s % 3) * kPlane;
    if (s == 9) p = base + half * kPlane + ((2 * c) & 15) * kPitch;
    if (s == 10) p = half ? zeros : base + 2 * kPlane + ((2 * c) & 15) * kPitch;
    return *reinterpret_cast<const u32x4_a4*>(p);
  };

  floatx16 acc[2][2];  // [row parity][filter of the lane's pair]; row 0: the even convolution row 2y, row 1: the odd one 2y + 1
  unsigned st[16] = {};  // packed pairs of the lane's pixels: of the odd row above (between the walks of an odd and an even row), then the maximum of the two
  constexpr int kAhead = 4;
  unsigned row_mask = 0u, left_mask = ~0u;  // zero where the row, the strip's first column is outside the convolution output
  int thirds = -1;                          // bit i: the third column of the lane's window i is inside
  __amdgpu_buffer_rsrc_t rs_row = make_rsrc(a.out, 0u);  // the pooled row that is written: what lies right of it is out of range
  unsigned dst = 0u, dst7 = 0u;             // of the lane's windows 0 .. 6, and of the eighth, which the upper half does not have
  unsigned hold = 0u, beyond = 0u;          // between the pieces of a row: the columns of a window so far; the column right of the lane's own

  auto window = [&](int i, unsigned two, unsigned third) {
    const unsigned o = max2(max2(two, third & (unsigned)__builtin_amdgcn_sbfe(thirds, i, 1)), 0u);
    __builtin_amdgcn_raw_buffer_store_b32(o, rs_row, i < 7 ? dst + i * 128 : dst7, 0, 0);
  };
  // Piece p of a row's epilogue: the lane's pixel p, and the window that it completes.
  auto piece = [&](auto p_c, auto odd_c) {
    constexpr int p = decltype(p_c)::value;
    constexpr bool odd = decltype(odd_c)::value;
    half2v h;
#pragma unroll
    for (int g = 0; g < 2; ++g) h[g] = (half_t)(acc[odd][g][p] * sc[g] + sh[g]);
    const unsigned u = __builtin_bit_cast(unsigned, h);
    if constexpr (odd) {
      const unsigned low = u & row_mask;
      unsigned v = max2(st[p], low);
      st[p] = low;
      if constexpr (p == 0) {
        v &= left_mask;
        beyond = __builtin_amdgcn_permlane32_swap(v, v, false, false)[1];  // on the lower lanes the upper ones' first column
      }
      if constexpr (p > 0 && p % 2 == 0) window(p / 2 - 1, hold, v);
      hold = p % 2 ? max2(hold, v) : v;
      if constexpr (p == 15) window(7, hold, beyond);
    } else {
      st[p] = max2(st[p], u);
    }
  };

  // One convolution row: 22 MFMAs into acc[odd], between them the epilogue of the row before (the other parity) and the
  // traffic of the next rows.
  u32x4 lead[kAhead];  // the first operands of the row that comes next
  auto lead_in = [&](int c) {
    lead[0] = operand(std::integral_constant<int, 0>(), c);
    lead[1] = operand(std::integral_constant<int, 1>(), c);
    lead[2] = operand(std::integral_constant<int, 2>(), c);
    lead[3] = operand(std::integral_constant<int, 3>(), c);
  };
  static_assert(kAhead == 4, "lead_in is spelled out");
  auto walk_row = [&](auto odd_c, auto pieces_c, int c, int y, bool more_rows) {
    constexpr int odd = decltype(odd_c)::value;
    constexpr bool pieces = decltype(pieces_c)::value;
    u32x4 f[kSteps + kAhead];
#pragma unroll
    for (int k = 0; k < kAhead; ++k) f[k] = lead[k];
    auto between = [&](auto k_c) {  // behind MFMA k = 0 .. 21
      constexpr int k = decltype(k_c)::value;
      if constexpr (pieces) {
        if constexpr (k >= 1 && k <= 16) piece(std::integral_constant<int, k - 1>(), std::integral_constant<bool, !odd>());
        if constexpr (kDirect && odd && k == 17) {
          // Batch y + 1, requested under the odd row above, has to be in the ring now: the eight stores of the even row are
          // the only requests younger than it.  Batch y + 2 takes the place of rows that nothing reads any more.
          wait_vmcnt<8>();
          if (more_rows) fetch(y + 2);
        }
        if constexpr (!kDirect && k == 17) {
          if (odd) {
            deposit(next, y + 1, 1);
            if (more_rows) request(next, y + 2, 0);
          } else {
            deposit(next, y + 1, 0);
            request(next, y + 1, 1);
          }
        }
      }
    };
    // The two workgroups of a CU take turns at the higher priority, row by row (the first 256 workgroups of a launch are the first on
    // their CUs, more or less): left alone the arbiter favours the older wave of a SIMD, and the younger one runs its last rows alone.
    if (((blockIdx.x >> 8) ^ odd) & 1) __builtin_amdgcn_s_setprio(1);
    else __builtin_amdgcn_s_setprio(0);
    auto steps = [&](auto self, auto s_c) -> void {
      constexpr int s = decltype(s_c)::value;
      if constexpr (s < kSteps) {
        if constexpr (s + kAhead < kSteps) f[s + kAhead] = operand(std::integral_constant<int, s + kAhead>(), c);
        else f[s + kAhead] = operand(std::integral_constant<int, s + kAhead - kSteps>(), c + 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int g = 0; g < 2; ++g) {
          if constexpr (s == 0) Mma<half_t>::start(f[s], wreg[s][g], acc[odd][g]);
          else Mma<half_t>::run(f[s], wreg[s][g], acc[odd][g]);
          __builtin_amdgcn_sched_barrier(0);
          if (g == 0) between(std::integral_constant<int, 2 * s>());
          else between(std::integral_constant<int, 2 * s + 1>());
          __builtin_amdgcn_sched_barrier(0);
        }
        self(self, std::integral_constant<int, s + 1>());
      }
    };
    steps(steps, std::integral_constant<int, 0>());
#pragma unroll
    for (int k = 0; k < kAhead; ++k) lead[k] = f[kSteps + k];
  };
  constexpr std::integral_constant<int, 0> even_row{};
  constexpr std::integral_constant<int, 1> odd_row{};

  for (;;) {
    const int count = left < a.PH - y ? left : a.PH - y;  // pooled rows y .. y + count - 1 of this strip
    left_mask = ((px0 > 0) | (half > 0)) ? ~0u : 0u;
    const int last = a.PW - 1 - px0 - 8 * half;  // the image's last window as a window of this lane
    thirds = (a.OW & 1) != 0 && (unsigned)last < 8u ? ~(1 << last) : -1;
    dst = (unsigned)((px0 + 8 * half) * 128 + n2 * 4);
    dst7 = half ? kOOBs : dst + 7 * 128;
    auto row_of = [&](int py, bool live) {
      return make_rsrc(a.out + ((long long)n * a.PH + py) * a.PW * 64, live ? (unsigned)a.PW * 128u : 0u);
    };
    lead_in(2 * y - 1);
    walk_row(odd_row, std::false_type(), 2 * y - 1, y - 1, false);
    for (int k = 0; k < count; ++k, ++y) {
      // the odd row above window y: outside the image above the first one; it completes window y - 1, which this walk owns from its second window on
      row_mask = y > 0 ? ~0u : 0u;
      rs_row = row_of(k > 0 ? y - 1 : 0, k > 0);
      walk_row(even_row, std::true_type(), 2 * y, y, false);
      walk_row(odd_row, std::true_type(), 2 * y + 1, y, k + 1 < count);
    }
    // the last window's lowest row, outside the image if the convolution's height is odd
    row_mask = 2 * y - 1 < a.OH ? ~0u : 0u;
    rs_row = row_of(y - 1, true);
    auto drain = [&](auto self, auto q_c) -> void {
      constexpr int q = decltype(q_c)::value;
      if constexpr (q < 16) {
        piece(q_c, std::true_type());
        self(self, std::integral_constant<int, q + 1>());
      }
    };
    drain(drain, std::integral_constant<int, 0>());
    left -= count;
    if (left <= 0) break;
    ++strip;
    y = 0;
    begin_walk();
    await_walk();
  }
}

bool stem_pool_applicable(int dt, int N, int H, int W, int F) {
  static const bool off = getenv("NNCV_HIP_NO_STEM_FUSION") != nullptr;
  return !off && F == 64 && H >= 7 && W >= 7 && (long long)N * 3 * H * W * (long long)dtype_size(dt) < (long long)kOOBs &&
         (long long)((W + 3) / 4) * 256 < (long long)kOOBs;  // the image and a pooled row within a buffer descriptor's range check
}

size_t stem_weight_strip_bytes() { return kWtBytes; }

// The fragments of the 64 filters, [filter of a lane's pair][step][lane][8]: see the K axis in the kernel.
__global__ void stem_weight_strip_kernel(const half_t* __restrict__ w, half_t* __restrict__ dst) {
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= kWtBytes / 2) return;
  const int e = idx & 7, lane = (idx >> 3) & 63, s = (idx >> 9) % kSteps, g = (idx >> 9) / kSteps;
  const int half = lane >> 5, f = 2 * (lane & 31) + g;
  const int r = s < 9 ? 4 - 2 * (s / 3) + half : 6, c = s < 9 ? s % 3 : s == 9 ? half : 2 + half;
  dst[idx] = (c < 3 && e > 0) ? w[((f * 3 + c) * 7 + r) * 7 + e - 1] : (half_t)0.0f;
}

void launch_stem_weight_strip(const void* w, void* dst, hipStream_t s) {
  launch_kernel(stem_weight_strip_kernel, dim3((kWtBytes / 2 + 255) / 256), dim3(256), 0, s, static_cast<const half_t*>(w), static_cast<half_t*>(dst));
  NNCV_HIP_CHECK(hipGetLastError());
}

// wt: launch_stem_weight_strip; out: [N][PH][PW][64] with PH, PW the pooled size.
void launch_stem_pool(const void* in, const void* wt, const float* scale, const float* shift, void* out, int N, int H, int W,
                      hipStream_t s) {
  StemPoolArgs a{};
  a.in = static_cast<const half_t*>(in); a.wt = wt; a.scale = scale; a.shift = shift;
  a.out = static_cast<half_t*>(out);
  a.N = N; a.H = H; a.W = W;
  a.OH = (H + 6 - 7) / 2 + 1; a.OW = (W + 6 - 7) / 2 + 1;
  a.PH = (a.OH + 2 - 3) / 2 + 1; a.PW = (a.OW + 2 - 3) / 2 + 1;
  a.strips = (a.PW + kPoolCols - 1) / kPoolCols;
  const long long rows = (long long)N * a.strips * a.PH;
  NNCV_REQUIRE(rows < (1ll << 30), "stem: too many rows");
  // 2048 waves are two on every SIMD.  Equal runs of the whole list leave no wave idle, but a run that goes on in another strip
  // starts there afresh (a trip to memory, a row above the first window: about two pooled rows); equal shares of a strip never do.
  a.waves = rows < 2048 ? (int)rows : 2048;
  a.run = (int)(rows / a.waves);
  a.extra = (int)(rows % a.waves);
  const int all_strips = N * a.strips, share = std::min(a.waves / all_strips, a.PH);
  if (share > 0 && (a.PH + share - 1) / share <= a.run + (a.extra > 0) + 2) {
    a.share = share;
    a.waves = all_strips * share;
  }
  a.in_bytes = (unsigned)((size_t)N * 3 * H * W * 2);
  const auto kernel = W % 2 == 0 && reinterpret_cast<uintptr_t>(in) % 4 == 0 ? stem_pool_kernel<true> : stem_pool_kernel<false>;
  const double flops = 2.0 * N * a.OH * a.OW * 64.0 * 147.0;
  const double bytes = 2.0 * ((double)N * 3 * H * W + (double)N * a.PH * a.PW * 64 + 64.0 * 176);
  ProfScope prof("stem_conv7x7_bn_relu_maxpool<f16>", flops, bytes, s);
  static const bool attr = [] {
    NNCV_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(stem_pool_kernel<true>), hipFuncAttributeMaxDynamicSharedMemorySize, kLds));
    NNCV_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(stem_pool_kernel<false>), hipFuncAttributeMaxDynamicSharedMemorySize, kLds));
    return true;
  }();
  (void)attr;
  launch_kernel(kernel, dim3((a.waves + 3) / 4), dim3(256), kLds, s, a);
  NNCV_HIP_CHECK(hipGetLastError());
}

}  // namespace nncv_hip
