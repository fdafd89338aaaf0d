// fp32 row-major D = C + A.B on gfx950 MFMA (D may be C) — the linalg.matmul of
// tests/MatMulOptimization/MatMulDeafult.mlir:6-9, which the reference lowers with 16/8/k8 tiles
// and 8x8x8 vector contracts (ModernTile.cpp:289-296, PrepareModernVec.cpp:43-48) and for which
// its unfinished CUDA kernel intended a 128x128x8 shared-memory tiling
// (src/libnncv/kernel/sgemm.cu:13-100).  Nothing of either is reused.
#include <algorithm>

#include "mfma_tile.hpp"

namespace nncv_hip {

using mt::bytes_left;
using mt::floatx16;
using mt::floatx4;
using mt::u32x4;

namespace {

// One wave owns TM x TN accumulators of BT x BT (BT = 32: v_mfma_f32_32x32x2_f32, 16: v_mfma_f32_16x16x4_f32, both 256
// flops a cycle and CU) and feeds them straight from memory: fp32 matrix instructions are so slow (64 / 32 cycles) that a wave
// needs only 4-5 KB of operands per 1024 cycles (a fifth of the CU's 64 B/clk), and with no LDS tile there is no
// barrier, no store pass and no wave that waits for another.
//  * A (K contiguous): lane l holds row l % BT; a 16-byte load along k is the operand of four MFMAs (lane group h = l / BT
//    takes k = QK q + 4 h + e, QK = 256 / BT).  The loads that cover a row's 128-byte line go out together, one round (32 k) ahead.
//  * B (N contiguous): the MFMA columns are dealt to lanes so that lane l holds columns TN l .. TN l + TN - 1: one 4 or 8
//    byte load of row k is the operand of TN accumulators, whole rows of 4 BT TN contiguous bytes per lane group.  C is
//    read and written the same way.
//  * Nothing asks for alignment beyond 4 bytes, so odd K and N (rows that do not start on 16 bytes) take the same loads.
//    Only the last 32 k of the matrix can hold k >= K or leave the buffers; the group that owns them walks them FIRST,
//    with A masked (B's rows past the end come back as zeros from the range check), so the main loop masks nothing.
//    Rows m >= M read row M - 1 and columns n >= N read the next row: both only reach results that are not stored.
//  * KG "K groups": waves of a workgroup that share a tile of C and split K.  Their sums meet in LDS, in a fixed order
//    (results do not change from run to run), and every wave adds its share of rows to C, requested before the loop.
template <int BT, int TM, int TN, int WM, int WN, int KG>
struct GemmCfg {
  static constexpr int kWaves = WM * WN * KG, kRows = BT * TM * WM, kCols = BT * TN * WN;
  static constexpr int kAcc = BT * BT / 64;  // accumulator registers of a BT x BT block
  static constexpr int kLds = KG > 1 ? KG * WM * WN * TM * TN * BT * BT * 4 : 0;
};

template <int TN>
struct Vec { typedef float type __attribute__((ext_vector_type(TN))); };
template <>
struct Vec<1> { typedef float type; };

template <int BT>
struct Mma32;
template <>
struct Mma32<32> {
  typedef floatx16 acc;
  static __device__ __forceinline__ acc run(float a, float b, acc c) { return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0); }
};
template <>
struct Mma32<16> {
  typedef floatx4 acc;
  static __device__ __forceinline__ acc run(float a, float b, acc c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
};

template <int TN>
__device__ __forceinline__ void load_row(__amdgpu_buffer_rsrc_t rs, unsigned voff, float (&b)[TN]) {
  if constexpr (TN == 1) {
    b[0] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, voff, 0, 0));
  } else {
    typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
    static_assert(TN == 2, "a lane holds one or two columns");
    const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(rs, voff, 0, 0);
    const typename Vec<2>::type f = __builtin_bit_cast(typename Vec<2>::type, v);
    b[0] = f[0];
    b[1] = f[1];
  }
}

// A copy that rides in front of a launch: its first `blocks` workgroups move `bytes` (a multiple of 16) and are done.
__device__ __forceinline__ void ride_along_copy(const RideCopy& r, int block, int threads) {
  const u32x4* src = static_cast<const u32x4*>(r.src);
  u32x4* dst = static_cast<u32x4*>(r.dst);
  const size_t n = r.bytes >> 4, step = (size_t)r.blocks * threads;
  size_t i = (size_t)block * threads + threadIdx.x;
  for (; i + 3 * step < n; i += 4 * step) {
    u32x4 v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = src[i + k * step];
#pragma unroll
    for (int k = 0; k < 4; ++k) dst[i + k * step] = v[k];
  }
  for (; i < n; i += step) dst[i] = src[i];
}

__global__ __launch_bounds__(256) void copy16_kernel(RideCopy r) { ride_along_copy(r, blockIdx.x, 256); }

template <int BT, int TM, int TN, int WM, int WN, int KG, bool RIDE = false>
__global__ __launch_bounds__(64 * WM * WN * KG) void gemm_nn_f32_kernel(const float* __restrict__ A, const float* __restrict__ B,
                                                                        const float* C, float* D, int M, int N, int K, int tiles_m,
                                                                        int tiles_n, RideCopy ride) {
  using Cfg = GemmCfg<BT, TM, TN, WM, WN, KG>;
  constexpr int QK = 256 / BT, NQ = 32 / QK, kAcc = Cfg::kAcc;
  int block = blockIdx.x;
  if constexpr (RIDE) {
    if (block < ride.blocks) {
      ride_along_copy(ride, block, 64 * Cfg::kWaves);
      return;
    }
    block -= ride.blocks;
  }
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int grp = wave / (WM * WN), wmn = wave % (WM * WN);
  const int lrow = lane & (BT - 1), lh = lane / BT;
  // XCD x (workgroups x, x + 8, ...) takes a contiguous run of tiles, walked in bands of eight tile rows
  int tm, tn;
  {
    const int tiles = tiles_m * tiles_n, per = (tiles + 7) >> 3, rem = tiles & 7;
    const int x = block & 7, i = block >> 3;
    const int t = rem == 0 ? x * per + i : (x < rem ? x * per : rem * per + (x - rem) * (per - 1)) + i;
    const int band = t / (8 * tiles_n), in = t - band * 8 * tiles_n, h = min(8, tiles_m - 8 * band);
    tn = in / h;
    tm = 8 * band + (in - tn * h);
  }
  const int m0 = tm * Cfg::kRows + (wmn % WM) * BT * TM, n0 = tn * Cfg::kCols + (wmn / WM) * BT * TN;
  const bool live = m0 < M && n0 < N;  // a wave of a multi-wave tile may lie outside the matrix altogether
  // accumulator register v of block row i: matrix row of this lane's result
  auto row_of = [&](int i, int v) { return BT * i + (BT == 32 ? 8 * (v >> 2) + 4 * lh + (v & 3) : 4 * lh + v); };
  typedef typename Vec<TN>::type vec;
  auto c_row = [&](int row, bool* whole) -> long long {  // element of C and D, -1 outside the matrix
    const int m = m0 + row, n = n0 + TN * lrow;
    *whole = n + TN <= N;
    return live && m < M && n < N ? (long long)m * N + n : -1;
  };
  auto fetch = [&](long long at, bool whole) {
    const float* c = at >= 0 ? C + at : nullptr;
    vec v;
    if constexpr (TN == 1) {
      v = c ? *c : 0.0f;
    } else {
#pragma unroll
      for (int j = 0; j < TN; ++j) v[j] = 0.0f;
      if (c && whole) {
        __builtin_memcpy(&v, c, sizeof(v));
      } else if (c) {
        v[0] = c[0];  // TN = 2: the last column of an odd row
      }
    }
    return v;
  };
  auto put = [&](long long at, bool whole, vec v) {
    if (at < 0) return;
    float* c = D + at;
    if constexpr (TN == 1) {
      *c = v;
    } else {
      if (whole) __builtin_memcpy(c, &v, sizeof(v));
      else c[0] = v[0];
    }
  };

  typename Mma32<BT>::acc acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int v = 0; v < kAcc; ++v) acc[i][j][v] = 0.0f;

  // row units (i, v) of the tile this wave adds to C
  constexpr int kUnits = TM * kAcc, kMine = kUnits / KG;
  static_assert(kUnits % KG == 0, "every wave of a tile takes the same number of row units");
  vec cpre[KG > 1 ? kMine : 1];

  // rounds of 32 k: group g owns [begin, end)
  const int nk = (K + 31) >> 5;
  const int begin = (int)((long long)nk * grp / KG), end = (int)((long long)nk * (grp + 1) / KG);
  if (live && begin < end) {
    unsigned aoff[TM];
#pragma unroll
    for (int i = 0; i < TM; ++i) aoff[i] = ((unsigned)min(BT * i + lrow, M - 1 - m0) * (unsigned)K + 4u * lh) * 4u;
    const unsigned boff = (4u * lh * (unsigned)N + (unsigned)(TN * lrow)) * 4u, brow = (unsigned)N * 4u;
    // A is one round ahead in a second buffer, requested in one burst per round; B's registers are refilled for the next
    // round as each quarter's products are issued (three rounds in flight measured slower: fewer waves per SIMD)
    floatx4 fa[2][TM][NQ];
    float fb[NQ][4][TN];
    auto load_a = [&](int r, floatx4 (&f)[TM][NQ]) {
      const long long at = (long long)m0 * K + 32ll * r;
      const __amdgpu_buffer_rsrc_t rs = mt::make_rsrc(A + at, bytes_left((long long)M * K, at));
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int q = 0; q < NQ; ++q)
          f[i][q] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(rs, aoff[i] + 4 * QK * q, 0, 0));
    };
    auto rsrc_b = [&](int r) {
      const long long at = 32ll * r * N + n0;
      return mt::make_rsrc(B + at, bytes_left((long long)K * N, at));
    };
    auto load_b = [&](__amdgpu_buffer_rsrc_t rs, int q) {
#pragma unroll
      for (int e = 0; e < 4; ++e) load_row<TN>(rs, boff + (unsigned)(QK * q + e) * brow, fb[q][e]);
    };
    auto mma = [&](const floatx4 (&f)[TM][NQ], int q) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) acc[i][j] = Mma32<BT>::run(f[i][q][e], fb[q][e][j], acc[i][j]);
    };
    // the group's last round first
    load_a(end - 1, fa[0]);
    {
      const __amdgpu_buffer_rsrc_t rb = rsrc_b(end - 1);
#pragma unroll
      for (int q = 0; q < NQ; ++q) load_b(rb, q);
    }
    if constexpr (KG > 1) {
#pragma unroll
      for (int u = 0; u < kMine; ++u) {
        bool whole;
        const long long c = c_row(row_of((grp * kMine + u) / kAcc, (grp * kMine + u) % kAcc), &whole);
        cpre[u] = fetch(c, whole);
      }
    }
    if (const int left = K - 32 * (end - 1); left < 32) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int q = 0; q < NQ; ++q)
#pragma unroll
          for (int e = 0; e < 4; ++e) fa[0][i][q][e] = QK * q + 4 * lh + e < left ? fa[0][i][q][e] : 0.0f;
    }
    // one round: its products, and behind each part of it the loads of the round after it
    auto round = [&](const floatx4 (&cur)[TM][NQ], floatx4 (&nxt)[TM][NQ], int next, bool more) {
      if (more) {
        load_a(next, nxt);
        const __amdgpu_buffer_rsrc_t rb = rsrc_b(next);
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
          mma(cur, q);
          __builtin_amdgcn_sched_barrier(0);
          load_b(rb, q);
          __builtin_amdgcn_sched_barrier(0);
        }
      } else {
#pragma unroll
        for (int q = 0; q < NQ; ++q) mma(cur, q);
      }
    };
    int r = begin;
    const int last = end - 1;
    for (; r + 1 < last; r += 2) {
      round(fa[0], fa[1], r, true);
      round(fa[1], fa[0], r + 1, true);
    }
    if (r < last) {
      round(fa[0], fa[1], r, true);
      round(fa[1], fa[0], 0, false);
    } else {
      round(fa[0], fa[1], 0, false);
    }
  } else if constexpr (KG > 1) {
#pragma unroll
    for (int u = 0; u < kMine; ++u) {
      bool whole;
      const long long c = c_row(row_of((grp * kMine + u) / kAcc, (grp * kMine + u) % kAcc), &whole);
      cpre[u] = fetch(c, whole);
    }
  }

  if constexpr (KG == 1) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int v = 0; v < kAcc; ++v) {
        bool whole;
        const long long c = c_row(row_of(i, v), &whole);
        vec y = fetch(c, whole);
        if constexpr (TN == 1) {
          y += acc[i][0][v];
        } else {
#pragma unroll
          for (int j = 0; j < TN; ++j) y[j] += acc[i][j][v];
        }
        put(c, whole, y);
      }
  } else {
    // [group][tile][row unit][lane][TN]: lane-linear, no bank conflicts
    extern __shared__ __align__(16) float red[];
    vec* mine = reinterpret_cast<vec*>(red) + (size_t)(grp * WM * WN + wmn) * kUnits * 64 + lane;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int v = 0; v < kAcc; ++v) {
        vec y;
        if constexpr (TN == 1) {
          y = acc[i][0][v];
        } else {
#pragma unroll
          for (int j = 0; j < TN; ++j) y[j] = acc[i][j][v];
        }
        mine[(kAcc * i + v) * 64] = y;
      }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kMine; ++u) {
      const int unit = grp * kMine + u;
      const vec* p = reinterpret_cast<const vec*>(red) + ((size_t)wmn * kUnits + unit) * 64 + lane;
      vec sum = p[0];
#pragma unroll
      for (int g = 1; g < KG; ++g) sum += p[(size_t)g * WM * WN * kUnits * 64];
      bool whole;
      const long long c = c_row(row_of(unit / kAcc, unit % kAcc), &whole);
      put(c, whole, cpre[u] + sum);
    }
  }
}

// Rows too long for 32-bit byte offsets over a tile (N or K from 2^24 up): one thread per element of C.
__global__ void gemm_nn_f32_any_kernel(const float* __restrict__ A, const float* __restrict__ B, const float* C, float* D, int M, int N, int K) {
  const long long total = (long long)M * N;
  for (long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x; t < total; t += (long long)gridDim.x * blockDim.x) {
    const long long m = t / N, n = t - m * N;
    float part[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (long long k = 0; k < K; ++k) part[k & 7] += A[m * K + k] * B[k * N + n];
    D[t] = C[t] + ((part[0] + part[1]) + (part[2] + part[3])) + ((part[4] + part[5]) + (part[6] + part[7]));
  }
}

template <int BT, int TM, int TN, int WM, int WN, int KG, bool RIDE = false>
void launch_gemm_cfg(const float* A, const float* B, const float* C, float* D, int M, int N, int K, const RideCopy& ride, hipStream_t s) {
  using Cfg = GemmCfg<BT, TM, TN, WM, WN, KG>;
  auto kern = gemm_nn_f32_kernel<BT, TM, TN, WM, WN, KG, RIDE>;
  static const bool attr = [&] {
    if (Cfg::kLds) NNCV_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, Cfg::kLds));
    return true;
  }();
  (void)attr;
  const long long tm = (M + Cfg::kRows - 1) / Cfg::kRows, tn = (N + Cfg::kCols - 1) / Cfg::kCols;
  NNCV_REQUIRE(tm * tn < (1ll << 31), "matmul: too many tiles");
  launch_kernel(kern, dim3((unsigned)(tm * tn + ride.blocks)), dim3(64 * Cfg::kWaves), Cfg::kLds, s, A, B, C, D, M, N, K, (int)tm, (int)tn, ride);
}

}  // namespace

namespace {

// The forms of the kernel, and what a launch of each takes:
//   us = fixed + rounds * (k_us * 32 x 32 blocks of a tile * K + tile_us),   rounds = ceil(tiles / 256 CUs)
// with K rounded up to whole rounds of 32.  The coefficients are least-squares fits over 24 shapes from 16x16x4096 to 4096^3
// (launches back to back, clocks warm; the fit is within 5-15 % of every time, and the form it picks is on average 3 %
// slower than the best one).  k_us at the matrix rate is 0.0033: large tiles come close, 16-wide ones are bound by the
// number of operand loads (their MFMAs take half as long on the same loads), but split a small C over more CUs.
//   20x488x536 14.6 -> 3.2 us, 64x64x4096 81 -> 11, 92x3260x2312 52 -> 22 (against the LDS-tiled kernel with 128x128 / 64x64
//   tiles that this replaces).  From 352 k on the larger products go to gemm_split.hip, by its model against this one.
struct GemmForm {
  int rows, cols;
  double fixed_us, k_us, tile_us;
  void (*launch)(const float*, const float*, const float*, float*, int, int, int, const RideCopy&, hipStream_t);
  const char* tag;
};
const GemmForm kForms[] = {
    {128, 128, 5.7, 0.00367, 9.0, launch_gemm_cfg<32, 2, 2, 2, 2, 1>, "gemm_nn_f32<128x128>"},
    {64, 128, 0.0, 0.00377, 5.3, launch_gemm_cfg<32, 1, 2, 2, 2, 2>, "gemm_nn_f32<64x128,splitk2>"},
    {32, 64, 2.3, 0.00407, 1.0, launch_gemm_cfg<32, 1, 2, 1, 1, 4>, "gemm_nn_f32<32x64,splitk4>"},
    {32, 32, 2.4, 0.00477, 0.56, launch_gemm_cfg<32, 1, 1, 1, 1, 4>, "gemm_nn_f32<32x32,splitk4>"},
    {32, 32, 2.1, 0.00440, 1.2, launch_gemm_cfg<32, 1, 1, 1, 1, 8>, "gemm_nn_f32<32x32,splitk8>"},
    {16, 32, 2.95, 0.00623, 0.13, launch_gemm_cfg<16, 1, 2, 1, 1, 4>, "gemm_nn_f32<16x32,splitk4>"},
    {16, 16, 2.95, 0.00847, 0.11, launch_gemm_cfg<16, 1, 1, 1, 1, 4>, "gemm_nn_f32<16x16,splitk4>"},
};

}  // namespace

void launch_copy16(const RideCopy& r, hipStream_t s) {
  if (r.bytes == 0) return;
  launch_kernel(copy16_kernel, dim3((unsigned)r.blocks), dim3(256), 0, s, r);
  NNCV_HIP_CHECK(hipGetLastError());
}

void launch_gemm_nn_f32(const float* A, const float* B, const float* C, float* D, int M, int N, int K, hipStream_t s, const RideCopy* ride) {
  NNCV_REQUIRE(M > 0 && N > 0 && K > 0, "matmul: empty operand");
  const double flops = 2.0 * M * N * K, bytes = 4.0 * ((double)M * K + (double)K * N + 2.0 * M * N);
  if (ride && ride->bytes) {
    if (N < 1 << 24 && K < 1 << 24) {
      // one form only: these launches are bands of a product whose operands arrive over the bus
      ProfScope prof("gemm_nn_f32<32x64,splitk4,ride>", flops, bytes, s);
      launch_gemm_cfg<32, 1, 2, 1, 1, 4, true>(A, B, C, D, M, N, K, *ride, s);
      NNCV_HIP_CHECK(hipGetLastError());
      return;
    }
    launch_copy16(*ride, s);
  }
  if (N >= 1 << 24 || K >= 1 << 24) {  // 64 rows of A or 32 of B beyond 32-bit byte offsets
    const long long blocks = ((long long)M * N + 255) / 256;
    ProfScope prof("gemm_nn_f32<any>", flops, bytes, s);
    launch_kernel(gemm_nn_f32_any_kernel, dim3((unsigned)std::min(blocks, 1ll << 20)), dim3(256), 0, s, A, B, C, D, M, N, K);
    NNCV_HIP_CHECK(hipGetLastError());
    return;
  }
  const GemmForm* best = nullptr;
  double best_us = 0;
  for (const GemmForm& f : kForms) {
    const long long tiles = (long long)((M + f.rows - 1) / f.rows) * ((N + f.cols - 1) / f.cols), rounds = (tiles + 255) / 256;
    const double us = f.fixed_us + (double)rounds * (f.k_us * (f.rows * f.cols / 1024.0) * ((K + 31) / 32 * 32) + f.tile_us);
    if (!best || us < best_us) best = &f, best_us = us;
  }
  if (gemm_split_wins(M, N, K, best_us)) {
    launch_gemm_split(A, B, C, D, M, N, K, s);
    return;
  }
  ProfScope prof(best->tag, flops, bytes, s);
  best->launch(A, B, C, D, M, N, K, RideCopy{}, s);
  NNCV_HIP_CHECK(hipGetLastError());
}

}  // namespace nncv_hip
