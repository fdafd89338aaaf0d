// fp32 row-major D = C + A.B (D may be C) on the bf16 matrix pipes, operands split in three (split.hpp).
//
// One wave owns TM x TN accumulators of 32 x 32 and walks K in rounds of 32, on its own: no barrier before the sums meet.
//  * A (K contiguous): whole 128-byte lines, eight lanes each, a round ahead, through an LDS buffer of the wave's own, because an
//    operand wants 16 bytes of 32 rows and read like that every lane of a load touches a line of its own.
//  * B (N contiguous): lane l holds columns TN l .. TN l + TN - 1, so a load of row k is whole lines again.
//  * Both are split in registers, thirteen vector instructions for two values: 208 of them (832 clocks) feed the 24 products (768 clocks)
//    of a 64 x 64 tile and 16 k, and run under the products of the SIMD's other wave.
//  * Nothing asks for alignment beyond 4 bytes.  Only the last round of the matrix can hold k >= K or leave the buffers; the
//    group that owns it walks it first, with A masked (B's rows past the end come back as zeros from the range check,
//    gemm_split_walk.hpp).
//    Rows m >= M read row M - 1 and columns n >= N the tile's first one: both only reach results that are not stored.
//  * KG "K groups": waves of a workgroup that share a tile of C and take every KG-th round.  Their sums meet in LDS, in a
//    fixed order.
#include <cmath>
#include <type_traits>

#include "gemm_split_walk.hpp"
#include "split.hpp"

namespace nncv_hip {

using namespace mt;

namespace {

template <int TM, int TN, int KG>
struct SplitCfg {
  static constexpr int kPitch = 144;  // of a row of 32 k in LDS
  static constexpr int kStage = 32 * TM * kPitch, kPart = KG > 1 ? 32 * TM * 32 * TN * 4 : 0;
  static constexpr int kWave = kStage > kPart ? kStage : kPart, kLds = KG * kWave;
};

template <int TM, int TN, int KG>
__global__ __launch_bounds__(64 * KG, TM * TN == 4 ? 2 : TM * TN == 2 ? 3 : 4) void gemm_split_kernel(const float* __restrict__ A, const float* __restrict__ B, const float* C, float* D, int M,
                                                               int N, int K, int tiles_m, int tiles_n) {
  typedef SplitCfg<TM, TN, KG> Cfg;
  static_assert(TN == 1 || TN == 2, "a lane holds one or two columns");
  extern __shared__ __align__(16) unsigned char smem[];
  const int lane = threadIdx.x & 63, grp = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int lrow = lane & 31, lh = lane >> 5;
  unsigned char* lds = smem + grp * Cfg::kWave;
  // XCD x (workgroups x, x + 8, ...) takes a contiguous run of tiles, walked in bands of eight tile rows
  int tm, tn;
  {
    const int tiles = tiles_m * tiles_n, per = (tiles + 7) >> 3, rem = tiles & 7;
    const int x = blockIdx.x & 7, i = blockIdx.x >> 3;
    const int t = rem == 0 ? x * per + i : (x < rem ? x * per : rem * per + (x - rem) * (per - 1)) + i;
    const int band = t / (8 * tiles_n), in = t - band * 8 * tiles_n, h = min(8, tiles_m - 8 * band);
    tn = in / h;
    tm = 8 * band + (in - tn * h);
  }
  const int m0 = tm * 32 * TM, n0 = tn * 32 * TN;

  constexpr int kA = 4 * TM;  // loads of a round: eight rows each
  unsigned aoff[kA];
#pragma unroll
  for (int i = 0; i < kA; ++i) aoff[i] = ((unsigned)min((lane >> 3) + 8 * i, M - 1 - m0) * (unsigned)K + 4u * (lane & 7)) * 4u;
  const unsigned boff = split_b_lane(lane, TN, n0, N);
  floatx4 ra[kA];
  float rb[2][8][TN];
  // (rounds below the first read nothing: descriptors of no bytes)
  auto left = [&](long long elems, long long at, int r) { return r >= 0 ? bytes_left(elems, at) : 0u; };
  auto load_a = [&](int r) {
    const long long at = (long long)m0 * K + 32ll * r;
    const __amdgpu_buffer_rsrc_t rs = make_rsrc(A + at, left((long long)M * K, at, r));
#pragma unroll
    for (int i = 0; i < kA; ++i) ra[i] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(rs, aoff[i], 0, 0));
  };
  auto load_b = [&](int r, int k, auto last) {
    const SplitBRows rows = split_b_rows(r, k, n0, N, K);
    const __amdgpu_buffer_rsrc_t rs = make_rsrc(B + rows.first, rows.bytes);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const unsigned vo = split_b_vector(boff, e, N, last), so = split_b_scalar(e, N, last);
      if constexpr (TN == 1) {
        rb[k][e][0] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, vo, so, 0));
      } else {
        const floatx2 v = __builtin_bit_cast(floatx2, __builtin_amdgcn_raw_buffer_load_b64(rs, vo, so, 0));
        rb[k][e][0] = v[0];
        rb[k][e][1] = v[1];
      }
    }
  };

  floatx16 big[TM][TN], low[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) big[i][j][v] = low[i][j][v] = 0.0f;

  // units of the tile: register u % 16 of block row u / 16, columns TN lrow .. ; the ones this wave adds to C are asked for now
  typedef float vec __attribute__((ext_vector_type(TN)));
  constexpr int kUnits = 16 * TM, kMine = kUnits / KG;
  auto row_of = [&](int u, int lane) { return m0 + 32 * (u >> 4) + 8 * ((u & 15) >> 2) + 4 * (lane >> 5) + (u & 3); };
  auto fetch = [&](int u, int lane) {
    const int m = row_of(u, lane), n = n0 + TN * (lane & 31);
    vec v = {};
    if (m < M && n < N) {
      const float* c = C + ((long long)m * N + n);
      if (TN == 1 || n + 1 < N) __builtin_memcpy(&v, c, sizeof(v));
      else v[0] = c[0];
    }
    return v;
  };

  const int nk = (K + 31) >> 5;
  int r = nk - 1 - grp;  // this group's rounds, from the last one down
  load_a(r);
  load_b(r, 0, std::true_type());
  load_b(r, 1, std::true_type());
  constexpr bool kEarly = KG > 1 && TM * TN < 4;  // (the 64 x 64 forms have no registers to spare)
  vec cpre[kEarly ? kMine : 1];
  if constexpr (kEarly) {
#pragma unroll
    for (int q = 0; q < kMine; ++q) cpre[q] = fetch(grp * kMine + q, lane);
  }
  if (grp == 0) {
    const int kend = K - 32 * r - 4 * (lane & 7);  // of this lane's four k
#pragma unroll
    for (int i = 0; i < kA; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) ra[i][e] = e < kend ? ra[i][e] : 0.0f;
  }
  unsigned char* put = lds + (lane >> 3) * Cfg::kPitch + (lane & 7) * 16;
  const unsigned char* get = lds + lrow * Cfg::kPitch + lh * 32;
  for (; r >= 0; r -= KG) {
#pragma unroll
    for (int i = 0; i < kA; ++i) *reinterpret_cast<floatx4*>(put + 8 * i * Cfg::kPitch) = ra[i];
    load_a(r - KG);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      u32x4 a[TM][3], b[TN][3];
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const unsigned char* at = get + i * 32 * Cfg::kPitch + k * 64;
        split_eight(*reinterpret_cast<const u32x4*>(at), *reinterpret_cast<const u32x4*>(at + 16), a[i]);
      }
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        unsigned p[4][3];
#pragma unroll
        for (int e = 0; e < 4; ++e) split_pair(rb[k][2 * e][j], rb[k][2 * e + 1][j], p[e]);
#pragma unroll
        for (int c = 0; c < 3; ++c) b[j][c] = u32x4{p[0][c], p[1][c], p[2][c], p[3][c]};
      }
      load_b(r - KG, k, std::false_type());
      split_products(a, b, big, low);
    }
  }
  // The lane's number once more: what follows from it is not kept over the loop, in registers that the loop needs.  (32-row forms only
  // behind the sums: 1500x1001x777 36.4 -> 35.2 us a call; 64 x 64 tiles spill with it.)
  const int again = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)), late = TM == 1 ? again : lane;
  if (__builtin_expect(split_sums(big, low), 0)) {  // once more with the fp32 instructions: eight k a step, four steps a round
    const int lrow = again & 31, lh = again >> 5;
    plain_products(big, 4 * ((nk - grp + KG - 1) / KG), [&](int s, u32x4 (&a)[TM], u32x4 (&b)[TN]) {
      const int round = nk - 1 - grp - (s >> 2) * KG, k0 = 32 * round + 8 * (s & 3);
      const long long at = (long long)m0 * K + k0, rows = (long long)k0 * N + n0;
      const __amdgpu_buffer_rsrc_t rs_a = make_rsrc(A + at, k0 < K ? left((long long)M * K, at, round) : 0u);
      const __amdgpu_buffer_rsrc_t rs_b = make_rsrc(B + rows, k0 < K ? left((long long)K * N, rows, round) : 0u);
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const floatx4 v = __builtin_bit_cast(
            floatx4, __builtin_amdgcn_raw_buffer_load_b128(rs_a, ((unsigned)min(32 * i + lrow, M - 1 - m0) * (unsigned)K + 4u * lh) * 4u, 0, 0));
        floatx4 in;
#pragma unroll
        for (int e = 0; e < 4; ++e) in[e] = k0 + 4 * lh + e < K ? v[e] : 0.0f;
        a[i] = __builtin_bit_cast(u32x4, in);
      }
      const unsigned col = n0 + TN * lrow < N ? (unsigned)(TN * lrow) : 0u;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const unsigned vo = ((4u * lh + e) * (unsigned)N + col) * 4u;
        if constexpr (TN == 1) {
          b[0][e] = __builtin_amdgcn_raw_buffer_load_b32(rs_b, vo, 0, 0);
        } else {
          const u32x2 v = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rs_b, vo, 0, 0));
          b[0][e] = v[0];
          b[1][e] = v[1];
        }
      }
    });
  }

  // ---- D = C + sums ----
  auto emit = [&](int unit, const vec& c, vec sum) {
    const int m = row_of(unit, late), n = n0 + TN * (late & 31);
    if (m >= M || n >= N) return;
    sum += c;
    float* d = D + ((long long)m * N + n);
    if (TN == 1 || n + 1 < N) __builtin_memcpy(d, &sum, sizeof(sum));
    else d[0] = sum[0];
  };
  if constexpr (KG == 1) {
#pragma unroll
    for (int u = 0; u < kUnits; ++u) {
      vec y;
#pragma unroll
      for (int j = 0; j < TN; ++j) y[j] = big[u >> 4][j][u & 15];
      emit(u, fetch(u, late), y);
    }
  } else {
    // [group][unit][lane][TN]
    vec* mine = reinterpret_cast<vec*>(lds) + late;
#pragma unroll
    for (int u = 0; u < kUnits; ++u) {
      vec y;
#pragma unroll
      for (int j = 0; j < TN; ++j) y[j] = big[u >> 4][j][u & 15];
      mine[u * 64] = y;
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kMine; ++q) {
      const int u = grp * kMine + q;
      const vec* p = reinterpret_cast<const vec*>(smem) + u * 64 + late;
      vec sum = p[0];
#pragma unroll
      for (int g = 1; g < KG; ++g) sum += p[g * (Cfg::kWave / sizeof(vec))];
      emit(u, kEarly ? cpre[kEarly ? q : 0] : fetch(u, late), sum);
    }
  }
}

template <int TM, int TN, int KG>
void launch_cfg(const float* A, const float* B, const float* C, float* D, int M, int N, int K, hipStream_t s) {
  typedef SplitCfg<TM, TN, KG> Cfg;
  auto kern = gemm_split_kernel<TM, TN, KG>;
  static const bool attr = [&] {
    NNCV_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, Cfg::kLds));
    return true;
  }();
  (void)attr;
  const long long tm = (M + 32 * TM - 1) / (32 * TM), tn = (N + 32 * TN - 1) / (32 * TN);
  NNCV_REQUIRE(tm * tn < (1ll << 31), "matmul: too many tiles");
  launch_kernel(kern, dim3((unsigned)(tm * tn)), dim3(64 * KG), Cfg::kLds, s, A, B, C, D, M, N, K, (int)tm, (int)tn);
}

// The forms, and what a launch of each takes:
//   us = fixed + x (round_us * rounds of a wave + tile_us) + turns (turn_round_us * rounds of a wave + turn_us)
// with x = tiles / 256 CUs and turns = ceil(x / workgroups that a CU holds): the matrix pipes' share, and a workgroup's own length.
// Least-squares fits over 115 shapes of 30 MFLOP to 137 GFLOP, within 4-8 % of the times without the scaling of the operands, which
// made the 64 x 64 forms 6 to 11 % and the others 2 to 3 % longer.  The choice between these and the fp32 instructions holds all the
// same: over 70 shapes of 60 MFLOP to 80 GFLOP it takes 0.4 % longer than the sooner one on average (4 % at most), the fp32 ones 8.7 %.
//   fp32 instructions -> these: 1024^3 20.8 -> 16.7 us (129 TFLOP/s), 1500x1001x777 27.4 -> 23.3, 4096^3 965 -> 789 (174 TFLOP/s),
//   676x1382x829 18.8 -> 16.0
struct Form {
  int rows, cols, kg, resident;
  double fixed_us, round_us, tile_us, turn_round_us, turn_us;
  void (*launch)(const float*, const float*, const float*, float*, int, int, int, hipStream_t);
  const char* tag;
};
const Form kForms[] = {
    {64, 64, 8, 1, 1.297, 0.938, 0.685, 2.075, 2.064, launch_cfg<2, 2, 8>, "gemm_split<64x64,splitk8>"},
    {64, 64, 4, 2, 1.208, 0.631, 1.424, 1.550, 2.232, launch_cfg<2, 2, 4>, "gemm_split<64x64,splitk4>"},
    {64, 64, 1, 8, 0.0, 0.115, 1.504, 1.534, 6.457, launch_cfg<2, 2, 1>, "gemm_split<64x64>"},
    {32, 64, 8, 1, 1.696, 0.492, 0.0, 1.382, 1.533, launch_cfg<1, 2, 8>, "gemm_split<32x64,splitk8>"},
    {32, 64, 4, 3, 2.922, 0.570, 0.798, 0.827, 0.0, launch_cfg<1, 2, 4>, "gemm_split<32x64,splitk4>"},
};

const Form* best_form(int M, int N, int K, double* us) {
  const Form* best = nullptr;
  for (const Form& f : kForms) {
    const double x = (double)((M + f.rows - 1) / f.rows) * ((N + f.cols - 1) / f.cols) / 256, turns = std::ceil(x / f.resident);
    const double rounds = ((K + 31) / 32 + f.kg - 1) / f.kg;
    const double v = f.fixed_us + x * (f.round_us * rounds + f.tile_us) + turns * (f.turn_round_us * rounds + f.turn_us);
    if (!best || v < *us) best = &f, *us = v;
  }
  return best;
}

}  // namespace

// `other_us`: the modelled time of the fp32 kernel, which is 10 % short of what it takes on rows that are not whole lines (hence
// the margin).  Below 352 k the first loads and the reading and writing of C are most of a launch: what is left to gain there
// is under a quarter for large M and N and nothing for the rest.
bool gemm_split_wins(int M, int N, int K, double other_us) {
  double us = 0;
  return K >= 352 && N < 1 << 24 && K < 1 << 24 && best_form(M, N, K, &us) && us < 1.06 * other_us;
}

void launch_gemm_split(const float* A, const float* B, const float* C, float* D, int M, int N, int K, hipStream_t s) {
  double us = 0;
  const Form* f = best_form(M, N, K, &us);
  ProfScope prof(f->tag, 2.0 * M * N * K, 4.0 * ((double)M * K + (double)K * N + 2.0 * M * N), s);
  f->launch(A, B, C, D, M, N, K, s);
  NNCV_HIP_CHECK(hipGetLastError());
}

}  // namespace nncv_hip
