// fp16 inverted-residual blocks (MobileNetV3.mlir:260-420) in two launches instead of four or five.
//
//  1. dw_block: 1x1 expansion + BN + activation -> depthwise 3x3 / 5x5 + BN + activation, and what the workgroup's channel sums
//     add to the squeezed vector.
//  2. se_project: the squeezed vector from those parts, the gate, gated 1x1 projection + BN, residual.
//
// The layers are far too small to be bound by anything but launches and dependent loads: 14x14x240 at batch 32 is 3 MB and
// 0.1 GFLOP and took 5.5 (expansion) + 15.5 (depthwise) + 11.4 (gate) + 5 us (projection) in a kernel each; it takes 9.3 + 6.9
// here (7x7x576: 5.5 + 11.6 + 19.0 + 5.0 -> 10.2 + 9.3).  What is kept on chip is the expanded image (its values rounded to
// fp16 as they were when they went through memory), the pooled and squeezed vectors and the gate (fp32), and the gated image
// (fp16).
//
// The squeeze is linear in the pooled vector, so every dw_block workgroup puts its 32 channel sums through their 32 rows of
// the squeeze weights (4 multiply-adds a thread at SQ = 32) and se_project adds up bands * C / 32 vectors of SQ elements.  With
// the sums handed over instead, each of se_project's workgroups went through all C x SQ weights: 166 KB at 7x7x576, and
// 9.4 + 15.0 us; 9.0 + 8.7 at 14x14x240.  (The vectors are as many bytes as the weights at 16 bands; an image has 1 to 4 where
// C is above 200.)
//
// A 7x7x576 workgroup of dw_block spends 2200 clocks on its requests (mostly instruction and argument fetches: they are asked
// for at once, and what is the same for all threads is not worked out by branches), 2200 until the operands are there, 1300 on
// the expansion, 3700 on the depthwise part and the stores, 1400 on the sums and the squeeze.
#include "mfma_tile.hpp"

namespace nncv_hip {

using namespace mt;

namespace {

constexpr unsigned kOOBm = 0x7fffff00u;  // byte offset beyond any buffer these kernels accept
constexpr int kDwThreads = 256;
typedef __attribute__((address_space(3))) void* lds_ptr_t;

__device__ __forceinline__ half8 as_half8(const u32x4& v) { return __builtin_bit_cast(half8, v); }

// LDS cells of one pixel x 32 channels: 64 bytes, 16-byte chunk c at position c ^ (cell / 2) % 4, so that neither the
// 16-byte reads of four lanes per pixel nor the 8-byte writes of one lane per pixel pile up on a few banks
__device__ __forceinline__ int cell_at(int cell, int chunk) { return cell * 64 + ((chunk ^ ((cell >> 1) & 3)) << 4); }

// Sums over lanes that each hold eight elements.  Every step hands half of the elements over to the lane that goes on with
// them, by moves within the vector unit: seven exchanges where sums of all elements in all lanes take 24 trips through LDS.
template <int CTRL>
__device__ __forceinline__ float lane_move(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}
constexpr int kQuadXor1 = 0xb1, kQuadXor2 = 0x4e, kQuadXor3 = 0x1b, kRowRor8 = 0x128, kHalfMirror = 0x141;
// over lanes l, l ^ 1, .. l ^ 7: lane l returns element l & 7
__device__ __forceinline__ float sum_of_eight(const float (&v)[8], int lane) {
  float a[4], b[2];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float lo = v[e], hi = v[e + 4];
    a[e] = (lane & 4 ? hi : lo) + lane_move<kHalfMirror>(lane & 4 ? lo : hi);
  }
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const float lo = a[e], hi = a[e + 2];
    b[e] = (lane & 2 ? hi : lo) + lane_move<kQuadXor2>(lane & 2 ? lo : hi);
  }
  const float lo = b[0], hi = b[1];
  return (lane & 1 ? hi : lo) + lane_move<kQuadXor1>(lane & 1 ? lo : hi);
}
// over the sixteen lanes with the same l & 3: lane l returns element l >> 3
__device__ __forceinline__ float sum_of_sixteen(const float (&v)[8], int lane) {
  float a[4], b[2];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, v[e]), __builtin_bit_cast(unsigned, v[e + 4]), false, false);
    const unsigned r0 = r[0], r1 = r[1];  // (a bit_cast of r[1] itself takes element 0)
    a[e] = __builtin_bit_cast(float, r0) + __builtin_bit_cast(float, r1);
  }
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, a[e]), __builtin_bit_cast(unsigned, a[e + 2]), false, false);
    const unsigned r0 = r[0], r1 = r[1];
    b[e] = __builtin_bit_cast(float, r0) + __builtin_bit_cast(float, r1);
  }
  const float lo = b[0], hi = b[1], s = (lane & 8 ? hi : lo) + lane_move<kRowRor8>(lane & 8 ? lo : hi);
  return s + lane_move<kQuadXor3>(lane_move<kHalfMirror>(s));  // l ^ 7 ^ 3
}

// BatchNorm of channels c + STEP q .. + 3, q < Q
template <int Q, int STEP>
__device__ __forceinline__ void batch_norm(const float* scale, const float* shift, int C, int c, floatx4 (&sc)[Q], floatx4 (&sh)[Q]) {
  const __amdgpu_buffer_rsrc_t rs_sc = make_rsrc(scale, scale ? (unsigned)C * 4u : 0u), rs_sh = make_rsrc(shift, shift ? (unsigned)C * 4u : 0u);
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    sc[q] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(rs_sc, (unsigned)(c + STEP * q) * 4u, 0, 0));
    sh[q] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(rs_sh, (unsigned)(c + STEP * q) * 4u, 0, 0));
  }
  if (!scale)
#pragma unroll
    for (int q = 0; q < Q; ++q) sc[q] = floatx4{1.f, 1.f, 1.f, 1.f};
}

}  // namespace

// A workgroup takes one image's band of OR output rows, for 32 channels.  KST: 16-channel K steps of the expansion (0: the
// input is taken as it is).  The expansion's operands come straight from memory (a wave reads 32 pixels x 16 channels as 32
// runs of 32 bytes), its filters stay in registers.  The depthwise part reads the LDS image OXT outputs at a time.
// Zeros around the image are cells of their own: no branch in the taps.
template <int K, int S, int OXT, int KST>
__global__ __launch_bounds__(kDwThreads) void dw_block_kernel(const DwBlockArgs a) {
  constexpr int LW = (OXT - 1) * S + K;
  extern __shared__ __align__(16) unsigned char smem[];  // cells, then the taps [K * K][32 channels]
  // all arguments at once: fetched where they are first used, they are one wait after the other
  asm volatile("" ::"s"(a.in), "s"(a.w1), "s"(a.scale1), "s"(a.shift1), "s"(a.wt), "s"(a.scale), "s"(a.shift), "s"(a.H), "s"(a.W), "s"(a.pix), "s"(a.Cin), "s"(a.C),
               "s"(a.pad), "s"(a.OH), "s"(a.rows), "s"(a.pitch), "s"(a.cells), "s"(a.parts), "s"(a.sq_w), "s"(a.SQ), "s"(a.inv_w),
               "s"(a.out), "s"(a.OW), "s"(a.act), "s"(a.act1), "s"(a.inv_strips), "s"(a.bands));
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = blockIdx.x, g = blockIdx.y, band = blockIdx.z;
  const int c0 = g * 32, oy0 = band * a.rows, rows = min(a.rows, a.OH - oy0);
  const int iy0 = oy0 * S - a.pad, in_rows = (rows - 1) * S + K;
  unsigned char* taps = smem + a.cells * 64;
  const int chunk = tid & 3, ch = c0 + chunk * 8;  // the channels of this thread's depthwise work
  const bool live = ch < a.C;

  // Squeeze weights of this group's channels, a run of 32 rows, by DMA into LDS: in registers they take the third workgroup
  // from the CU (13.8 instead of 10.2 us at 7x7x576), and requested behind the stores they wait for the stores.
  unsigned char* sqw = taps + K * K * 64;
  auto request_squeeze = [&] {
    const __amdgpu_buffer_rsrc_t rs = make_rsrc(a.sq_w, (unsigned)(a.C * a.SQ * 2));
    for (int u = wave * 64; u < 4 * a.SQ; u += kDwThreads)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr_t)(sqw + u * 16), 16, (unsigned)(c0 * a.SQ * 2 + (u + lane) * 16), 0, 0, 0);
  };

  // rows of the input that exist
  const int ya = max(iy0, 0), yb = min(iy0 + in_rows, a.H), npx = max(0, yb - ya) * a.W;
  const int cell0 = (ya - iy0) * a.pitch + a.pad;  // cell of the first of them
  const __amdgpu_buffer_rsrc_t rs_in = make_rsrc(static_cast<const half_t*>(a.in) + ((long long)n * a.H + ya) * a.W * a.pix, (unsigned)(npx * a.pix * 2));
  auto cell_of = [&](int q) {
    int x;
    const int y = fast_div(q, a.W, a.inv_w, &x);
    return cell0 + y * a.pitch + x;
  };
  // BatchNorm of this thread's depthwise channels and its share of the taps; what lies beyond channel C reads as zero
  floatx4 dsc[2], dsh[2];
  u32x4 tap;
  auto request = [&] {
    batch_norm<2, 4>(a.scale, a.shift, a.C, ch, dsc, dsh);
    const __amdgpu_buffer_rsrc_t rs = make_rsrc(a.wt, (unsigned)(K * K * a.C * 2));
    tap = __builtin_amdgcn_raw_buffer_load_b128(rs, live ? (unsigned)((tid >> 2) * a.C + ch) * 2u : kOOBm, 0, 0);
  };
  auto prepare = [&] {  // zeros around the image, and the taps
    const u32x4 zero = {0, 0, 0, 0};
    for (int u = tid; u < in_rows * a.pitch * 4; u += kDwThreads) *reinterpret_cast<u32x4*>(smem + u * 16) = zero;
    if (tid < K * K * 4) *reinterpret_cast<u32x4*>(taps + tid * 16) = tap;
    if (a.parts) request_squeeze();
    __syncthreads();
  };

  if constexpr (KST > 0) {
    const int lrow = lane & 31, lh = lane >> 5, nch = a.Cin >> 3;
    const __amdgpu_buffer_rsrc_t rs_w = make_rsrc(a.w1, (unsigned)(a.C * a.Cin * 2));
    u32x4 w[KST], x[KST];
    floatx4 sc[4], sh[4];
    auto load = [&](int blk) {  // (pixels beyond npx and filters beyond C lie beyond their buffers)
      const unsigned off = (unsigned)((blk * 32 + lrow) * a.pix + lh * 8) * 2u;
#pragma unroll
      for (int k = 0; k < KST; ++k) x[k] = __builtin_amdgcn_raw_buffer_load_b128(rs_in, 2 * k + lh < nch ? off + 32u * k : kOOBm, 0, 0);
    };
    load(wave);
    const unsigned off_w = (unsigned)((c0 + lrow) * a.Cin + lh * 8) * 2u;
#pragma unroll
    for (int k = 0; k < KST; ++k) w[k] = __builtin_amdgcn_raw_buffer_load_b128(rs_w, 2 * k + lh < nch ? off_w + 32u * k : kOOBm, 0, 0);
    batch_norm<4, 8>(a.scale1, a.shift1, a.C, c0 + 4 * lh, sc, sh);  // accumulator channels 8 q + 4 (lane / 32) .. + 3
    request();
    prepare();
    constexpr int NW = kDwThreads / 64;
    for (int blk = wave; blk * 32 < npx; blk += NW) {
      floatx16 acc;
#pragma unroll
      for (int k = 0; k < KST; ++k) {
        if (k == 0) Mma<half_t>::start(w[k], x[k], acc);
        else Mma<half_t>::run(w[k], x[k], acc);
      }
      load(blk + NW);
      const int q = blk * 32 + lrow;
      float y[16];
#pragma unroll
      for (int e = 0; e < 16; ++e) y[e] = acc[e] * sc[e >> 2][e & 3] + sh[e >> 2][e & 3];
      act_apply_n<true>(y, a.act1);
      const int cell = cell_of(min(q, npx - 1));
      if (q < npx) {
#pragma unroll
        for (int p = 0; p < 4; ++p) {
          half4 h;
#pragma unroll
          for (int e = 0; e < 4; ++e) h[e] = (half_t)y[4 * p + e];
          *reinterpret_cast<half4*>(smem + cell_at(cell, p) + lh * 8) = h;
        }
      }
    }
  } else {
    request();
    prepare();
    for (int u = tid; u < npx * 4; u += kDwThreads)
      if (live) *reinterpret_cast<u32x4*>(smem + cell_at(cell_of(u >> 2), chunk)) = __builtin_amdgcn_raw_buffer_load_b128(rs_in, (unsigned)((u >> 2) * a.pix + ch) * 2u, 0, 0);
  }
  __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): the squeeze weights
  __syncthreads();

  // ---- depthwise: (kh, kw) order, fp32 ----
  const int strips = (a.OW + OXT - 1) / OXT;
  float sum[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) sum[e] = 0.0f;
  half_t* out = static_cast<half_t*>(a.out) + (((long long)n * a.OH + oy0) * a.OW) * a.C + ch;
  for (int t = tid >> 2; live && t < rows * strips; t += kDwThreads / 4) {
    int sx;
    const int oy = fast_div(t, strips, a.inv_strips, &sx), ox0 = sx * OXT;
    float acc[OXT][8];
#pragma unroll
    for (int j = 0; j < OXT; ++j)
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[j][e] = 0.0f;
#pragma unroll 1  // (reading the next row under this one's multiply-adds, or all rows at once, measured slower: registers)
    for (int r = 0; r < K; ++r) {
      const int cell = (oy * S + r) * a.pitch + ox0 * S;
      half8 x[LW];
#pragma unroll
      for (int q = 0; q < LW; ++q) x[q] = *reinterpret_cast<const half8*>(smem + cell_at(cell + q, chunk));
#pragma unroll
      for (int s = 0; s < K; ++s) {
        const half8 w = *reinterpret_cast<const half8*>(taps + (r * K + s) * 64 + chunk * 16);
#pragma unroll
        for (int j = 0; j < OXT; ++j)
#pragma unroll
          for (int e = 0; e < 8; ++e) acc[j][e] += (float)x[j * S + s][e] * (float)w[e];
      }
    }
#pragma unroll
    for (int j = 0; j < OXT; ++j) {
      if (ox0 + j >= a.OW) break;
      float y[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) y[e] = acc[j][e] * dsc[e >> 2][e & 3] + dsh[e >> 2][e & 3];
      act_apply_n<true>(y, a.act);
      half8 h;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        h[e] = (half_t)y[e];
        sum[e] += (float)h[e];
      }
      *reinterpret_cast<half8*>(out + ((long long)oy * a.OW + ox0 + j) * a.C) = h;
    }
  }
  if (!a.parts) return;  // (uniform)
  // ---- channel sums of the band, in a fixed order, through the squeeze weights of these channels ----
  const float total = sum_of_sixteen(sum, lane);
  __syncthreads();
  float* part = reinterpret_cast<float*>(smem);
  if (!(lane & 4)) part[wave * 32 + chunk * 8 + (lane >> 3)] = total;
  __syncthreads();
  const int sq_o = tid >> 3, sq_r = tid & 7;  // rows r, r + 8, ... of outputs 8 o .. 8 o + 7
  if (8 * sq_o >= a.SQ) return;
  float v[8];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int c = sq_r + 8 * u;
    const float m = (part[c] + part[32 + c]) + (part[64 + c] + part[96 + c]);
    const half8 w = *reinterpret_cast<const half8*>(sqw + (c * a.SQ + sq_o * 8) * 2);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = u ? v[e] + m * (float)w[e] : m * (float)w[e];
  }
  const float r = sum_of_eight(v, lane);
  a.parts[(((long long)n * a.bands + band) * ((a.C + 31) >> 5) + g) * a.SQ + tid] = r;
}

namespace {

// The excitation: out[j] = act(b[j] + sum_c in[c] w[c][j]), both vectors fp32 in LDS.  Thread (g, o) takes rows c = g, g + G, ...
// of the eight outputs of chunk o, so that a wave reads the weights in one run (a row of them per output instead, two lanes to
// a row, took 22 us for 576 x 144); the G <= 8 partial sums of an output meet in LDS (`part`).  The first U rows of a thread
// are requested long before the vector is there (`request`).
template <int THREADS, int U>
struct Excitation {
  static constexpr int kGroups = 8;
  __amdgpu_buffer_rsrc_t rs;
  int n_out, n_in, groups, g, o, step;
  unsigned first;
  u32x4 x[U];
  __device__ __forceinline__ Excitation(const void* w, int outs, int ins, float inv_oc) : rs(make_rsrc(w, (unsigned)(outs * ins) * 2u)), n_out(outs), n_in(ins) {
    const int oc = outs >> 3;
    groups = min(kGroups, min(THREADS / oc, (ins + 7) >> 3));
    g = fast_div((int)threadIdx.x, oc, inv_oc, &o);
    first = (unsigned)((g * oc + o) * 16);
    step = groups * oc * 16;
  }
  // rows beyond the last read as zeros
  __device__ __forceinline__ void request(int c0 = 0) {
    unsigned off = first + (unsigned)(c0 * (n_out * 2));
#pragma unroll
    for (int u = 0; u < U; ++u, off += step) x[u] = __builtin_amdgcn_raw_buffer_load_b128(rs, off, 0, 0);
  }
  // `in` is followed by zeros up to the next multiple of U * kGroups
  __device__ __forceinline__ void run(const float* in, float* part) {
    if (g >= groups) return;
    float s[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) s[e] = 0.0f;
    for (int c0 = 0; c0 < n_in; c0 += U * groups) {
      if (c0) request(c0);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const float m = in[c0 + g + u * groups];
        const half8 w = as_half8(x[u]);
#pragma unroll
        for (int e = 0; e < 8; ++e) s[e] += m * (float)w[e];
      }
    }
    float* at = part + (g * (n_out >> 3) + o) * 8;
    *reinterpret_cast<floatx4*>(at) = floatx4{s[0], s[1], s[2], s[3]};
    *reinterpret_cast<floatx4*>(at + 4) = floatx4{s[4], s[5], s[6], s[7]};
  }
  __device__ __forceinline__ float result(const float* part, int j, float bias) const {
    float v[kGroups];
#pragma unroll
    for (int k = 0; k < kGroups; ++k) v[k] = part[min(k, groups - 1) * n_out + j];
#pragma unroll
    for (int k = 0; k < kGroups; ++k) bias += k < groups ? v[k] : 0.0f;
    return bias;
  }
};

constexpr int kSpThreads = 512, kSpMaxC = 768, kSpMaxSq = 256;

}  // namespace

// A workgroup takes PT * 16 pixels of one image (KSPLIT: eight waves share its K axis, wave w taking the 32-channel steps w,
// w + 8, ...; otherwise C <= 32 and every wave has pixels of its own) and all FT * 16 filters.  It works out the image's gate
// for itself: the weights of the two vectors come from L2, and the operands of the projection, requested before that, are
// there when the gate is.  One image per workgroup tile, so the last tile of an image is short.
template <int NS, int FT, int PT, bool KSPLIT>
__global__ __launch_bounds__(kSpThreads) void se_project_kernel(const SeProjectArgs a) {
  constexpr int NW = kSpThreads / 64;
  constexpr int U = NS == 3 ? 21 : 8;  // rows of the excitation weights that a thread holds
  __shared__ __align__(16) float gate[kSpMaxC];
  __shared__ __align__(16) float hid[kSpMaxSq + 8 * U];
  __shared__ __align__(16) float part_sum[kSpThreads * 8];
  extern __shared__ __align__(16) unsigned char smem[];  // partial sums of the K steps (KSPLIT)
  asm volatile("" ::"s"(a.x), "s"(a.parts), "s"(a.b1), "s"(a.w2t), "s"(a.b2), "s"(a.wp_flat), "s"(a.scale), "s"(a.shift), "s"(a.residual), "s"(a.out), "s"(a.HW),
               "s"(a.C), "s"(a.SQ), "s"(a.F), "s"(a.bands), "s"(a.tiles), "s"(a.inv_sq), "s"(a.inv_c));  // one wait for all, as above
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lrow = lane & 15, lq = lane >> 4;
  const int tile = blockIdx.x % a.tiles, n = blockIdx.x / a.tiles;
  const int p0 = KSPLIT ? tile * PT * 16 : (tile * NW + wave) * PT * 16;
  const int nch = a.C >> 3;
  const __amdgpu_buffer_rsrc_t rs_x = make_rsrc(static_cast<const half_t*>(a.x) + (long long)n * a.HW * a.C, (unsigned)(a.HW * a.C * 2));
  // (filters in launch_weight_flat's order: blocks of 32, units of two chunks)
  const int units = ((a.C * 2 + 127) >> 7) * 4;
  const __amdgpu_buffer_rsrc_t rs_w = make_rsrc(a.wp_flat, (unsigned)((a.F + 31) / 32 * units) * 1024u);
  // The squeezed vector's parts: thread (g, j) takes parts g, g + G, ... of element j.  Requested before everything else, and
  // what the gate needs before what the projection does: results arrive in the order of the requests.
  const int parts = a.bands * ((a.C + 31) >> 5), groups = min(8, kSpThreads / a.SQ);
  int sj;
  const int sg = fast_div(tid, a.SQ, a.inv_sq, &sj);
  const __amdgpu_buffer_rsrc_t rs_p = make_rsrc(a.parts + (long long)n * parts * a.SQ, (unsigned)(parts * a.SQ) * 4u);
  float hid_sum = 0.0f;
  for (int b = sg < groups ? sg : parts; b < parts; b += 8 * groups) {
    float v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs_p, (unsigned)((b + k * groups) * a.SQ + sj) * 4u, 0, 0));
    hid_sum += ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
  }
  const float bias1 = a.b1[min(tid, a.SQ - 1)];
  float bias2[(kSpMaxC + kSpThreads - 1) / kSpThreads];
#pragma unroll
  for (int k = 0; k < (kSpMaxC + kSpThreads - 1) / kSpThreads; ++k) bias2[k] = a.b2[min(tid + k * kSpThreads, a.C - 1)];
  Excitation<kSpThreads, U> excite(a.w2t, a.C, a.SQ, a.inv_c);
  excite.request();
  u32x4 x[NS][PT], w[NS][FT];
#pragma unroll
  for (int j = 0; j < NS; ++j) {
    const int c = 4 * ((KSPLIT ? wave : 0) + NW * j) + lq;
#pragma unroll
    for (int q = 0; q < PT; ++q) {
      const int p = p0 + q * 16 + lrow;
      x[j][q] = __builtin_amdgcn_raw_buffer_load_b128(rs_x, ((p < a.HW) & (c < nch)) ? (unsigned)(p * a.C + c * 8) * 2u : kOOBm, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < FT; ++i) {
      const int f = i * 16 + lrow;
      w[j][i] = __builtin_amdgcn_raw_buffer_load_b128(
          rs_w, ((f < a.F) & (c < nch)) ? (unsigned)(((f >> 5) * units + (c >> 1)) * 1024 + (c & 1) * 512 + (f & 31) * 16) : kOOBm, 0, 0);
    }
  }

  // what the results of this wave need at the end: the blocks it finishes are known, too
  struct Tail { floatx4 scale, shift; half4 residual; };
  constexpr int kTails = KSPLIT ? (FT * PT + NW - 1) / NW : FT * PT;
  Tail tail[kTails];
#pragma unroll
  for (int k = 0; k < kTails; ++k) {
    const int blk = KSPLIT ? k * NW + wave : k, p = min(p0 + blk % PT * 16 + lrow, a.HW - 1), f = min(blk / PT * 16 + 4 * lq, a.F - 4);
    tail[k] = Tail{{1.f, 1.f, 1.f, 1.f}, {0.f, 0.f, 0.f, 0.f}, {}};
    if (a.scale) tail[k].scale = *reinterpret_cast<const floatx4*>(a.scale + f);
    if (a.shift) tail[k].shift = *reinterpret_cast<const floatx4*>(a.shift + f);
    if (a.residual) tail[k].residual = *reinterpret_cast<const half4*>(static_cast<const half_t*>(a.residual) + ((long long)n * a.HW + p) * a.F + f);
  }

  if (sg < groups) part_sum[tid] = hid_sum;
  __syncthreads();
  if (tid < a.SQ) {
    float v[8], s = 0.0f;
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = part_sum[min(k, groups - 1) * a.SQ + tid];
#pragma unroll
    for (int k = 0; k < 8; ++k) s += k < groups ? v[k] : 0.0f;
    hid[tid] = act_apply<false>(s / (float)a.HW + bias1, a.act1);
  } else if (tid < kSpMaxSq + 8 * U) {
    hid[tid] = 0.0f;
  }
  __syncthreads();
  excite.run(hid, part_sum);
  __syncthreads();
#pragma unroll
  for (int k = 0; k < (kSpMaxC + kSpThreads - 1) / kSpThreads; ++k)
    if (tid + k * kSpThreads < a.C) gate[tid + k * kSpThreads] = act_apply<false>(excite.result(part_sum, tid + k * kSpThreads, bias2[k]), a.act2);
  __syncthreads();

  floatx4 acc[FT][PT];
#pragma unroll
  for (int i = 0; i < FT; ++i)
#pragma unroll
    for (int q = 0; q < PT; ++q) acc[i][q] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < NS; ++j) {
    const int c = 4 * ((KSPLIT ? wave : 0) + NW * j) + lq;
    if (4 * ((KSPLIT ? wave : 0) + NW * j) >= nch) continue;  // (uniform)
    floatx4 g[2] = {};
    if (c < nch) {
      g[0] = *reinterpret_cast<const floatx4*>(gate + c * 8);
      g[1] = *reinterpret_cast<const floatx4*>(gate + c * 8 + 4);
    }
#pragma unroll
    for (int q = 0; q < PT; ++q) {
      const half8 v = as_half8(x[j][q]);
      half8 s;
#pragma unroll
      for (int e = 0; e < 8; ++e) s[e] = (half_t)(g[e >> 2][e & 3] * (float)v[e]);
#pragma unroll
      for (int i = 0; i < FT; ++i) acc[i][q] = __builtin_amdgcn_mfma_f32_16x16x32_f16(as_half8(w[j][i]), s, acc[i][q], 0, 0, 0);
    }
  }

  auto finish = [&](int i, int q, floatx4 v, const Tail& t) {
    const int p = p0 + q * 16 + lrow, f = i * 16 + 4 * lq;  // a lane holds filters f .. f + 3 of one pixel
    if (p >= a.HW || f >= a.F) return;
    float y[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) y[e] = v[e] * t.scale[e] + t.shift[e];
    if (a.residual && !(a.act & kActResidualAfter)) {
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] += (float)t.residual[e];
    }
    act_apply_n<true>(y, a.act & 0xff);
    if (a.residual && (a.act & kActResidualAfter)) {
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] += (float)t.residual[e];
    }
    half4 h;
#pragma unroll
    for (int e = 0; e < 4; ++e) h[e] = (half_t)y[e];
    *reinterpret_cast<half4*>(static_cast<half_t*>(a.out) + ((long long)n * a.HW + p) * a.F + f) = h;
  };
  if constexpr (!KSPLIT) {
#pragma unroll
    for (int i = 0; i < FT; ++i)
#pragma unroll
      for (int q = 0; q < PT; ++q) finish(i, q, acc[i][q], tail[i * PT + q]);
  } else {
    floatx4* part = reinterpret_cast<floatx4*>(smem);  // [wave][block][lane]
#pragma unroll
    for (int i = 0; i < FT; ++i)
#pragma unroll
      for (int q = 0; q < PT; ++q) part[(wave * FT * PT + i * PT + q) * 64 + lane] = acc[i][q];
    __syncthreads();
#pragma unroll
    for (int b0 = 0; b0 < FT * PT; b0 += NW) {
      const int b = b0 + wave;
      if (b >= FT * PT) break;
      floatx4 v[NW];
#pragma unroll
      for (int k = 0; k < NW; ++k) v[k] = part[(k * FT * PT + b) * 64 + lane];
#pragma unroll
      for (int d = 1; d < NW; d *= 2)
#pragma unroll
        for (int k = 0; k < NW; k += 2 * d) v[k] += v[k + d];
      finish(b / PT, b % PT, v[0], tail[b0 / NW]);
    }
  }
}

namespace {

// output rows of a band: all of them, or as many as keep the LDS image at 40 KB (three workgroups a CU) and at least two
// workgroups to a CU
struct DwPlan { int rows, bands, pitch, cells; };
bool dw_plan(int N, int W, int C, int K, int S, int pad, int OH, int OW, DwPlan* p) {
  const int oxt = 4;  // pitch for the widest strip
  p->pitch = std::max(W + pad, ((OW + oxt - 1) / oxt * oxt - 1) * S + K);
  const int groups = (C + 31) / 32;
  int rows = OH;
  while (rows > 1 && (((rows - 1) * S + K) * p->pitch * 64 > (40 << 10) || (rows > 4 && (long long)N * groups * ((OH + rows - 1) / rows) < 512))) rows = (rows + 1) / 2;
  p->rows = rows;
  p->bands = (OH + rows - 1) / rows;
  p->cells = ((rows - 1) * S + K) * p->pitch;
  return p->cells * 64 <= (96 << 10);
}

}  // namespace

int dw_block_bands(int N, int H, int W, int Cin, int C, int K, int S, int pad) {
  const int OH = (H + 2 * pad - K) / S + 1, OW = (W + 2 * pad - K) / S + 1;
  DwPlan p;
  const bool ok = (K == 3 || K == 5) && (S == 1 || S == 2) && pad >= 0 && pad < K && OH >= 1 && OW >= 1 && C % 8 == 0 &&
                  (Cin == 0 || (Cin % 8 == 0 && Cin <= 96)) && (long long)H * W * std::max(C, 96) * 2 < (1ll << 30) && (long long)H * W < (1 << 24) &&
                  (long long)N * OH * ((C + 31) / 32) < (1ll << 30) && dw_plan(N, W, C, K, S, pad, OH, OW, &p) && p.bands < 65536 && C < (1 << 20);
  return ok ? p.bands : 0;
}

void launch_dw_block(const DwBlockArgs& args, hipStream_t s) {
  DwBlockArgs a = args;
  DwPlan p;
  NNCV_REQUIRE(dw_block_bands(a.N, a.H, a.W, a.Cin, a.C, a.K, a.stride, a.pad) > 0 && dw_plan(a.N, a.W, a.C, a.K, a.stride, a.pad, a.OH, a.OW, &p),
               "dw_block: shape not covered");
  a.rows = p.rows; a.bands = p.bands; a.pitch = p.pitch; a.cells = p.cells;
  a.inv_w = 1.0f / (float)a.W;
  const double px_in = (double)a.N * a.H * a.W, px_out = (double)a.N * a.OH * a.OW;
  // Outputs a thread takes at a time, by the clocks that eight waves of a CU need for a round of them: LDS reads (a row of
  // taps and of pixels per filter row, shared by all) or multiply-adds (two waves a SIMD).  More share their operands, fewer
  // leave no thread of the last round idle.
  auto clocks = [&](int oxt) {
    const int lds = 8 * a.K * ((oxt - 1) * a.stride + 2 * a.K) * 8, fma = 2 * oxt * a.K * a.K * 32;
    return (long long)((a.rows * ((a.OW + oxt - 1) / oxt) + 63) / 64) * std::max(lds, fma);
  };
  int oxt = 1;
  for (int o : {2, 4})
    if (clocks(o) < clocks(oxt)) oxt = o;
  a.inv_strips = 1.0f / (float)((a.OW + oxt - 1) / oxt);
  const int steps16 = (a.Cin + 15) / 16, kst = steps16 <= 1 ? steps16 : steps16 <= 3 ? 3 : 6;  // K steps of the expansion that are unrolled
  char tag[40];
  snprintf(tag, sizeof tag, "dw_block<%d,%d,%d,%d>", a.K, a.stride, oxt, kst);
  ProfScope prof(tag, 2.0 * px_out * a.C * a.K * a.K + 2.0 * px_in * a.C * a.Cin,
                 2.0 * (px_in * (a.Cin ? a.Cin : a.C) + px_out * a.C + a.C * (a.K * a.K + a.Cin)), s);
  // images first: where their number is a multiple of the eight chiplets, an image's groups of channels find it in one L2
  const dim3 grid((unsigned)a.N, (unsigned)((a.C + 31) / 32), (unsigned)a.bands);
  const size_t lds = (size_t)a.cells * 64 + a.K * a.K * 64 + (a.parts ? (size_t)(a.SQ + 15) / 16 * 1024 : 0);
  auto go = [&](auto kern) {
    static const bool attr = [&] {
      NNCV_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, 116 << 10));
      return true;
    }();
    (void)attr;
    launch_kernel(kern, grid, dim3(kDwThreads), lds, s, a);
  };
  auto steps = [&](auto k, auto st, auto ox) {
    constexpr int K = decltype(k)::value, S = decltype(st)::value, OXT = decltype(ox)::value;
    if (kst == 0) go(dw_block_kernel<K, S, OXT, 0>);
    else if (kst == 1) go(dw_block_kernel<K, S, OXT, 1>);
    else if (kst == 3) go(dw_block_kernel<K, S, OXT, 3>);
    else go(dw_block_kernel<K, S, OXT, 6>);
  };
  auto strips = [&](auto k, auto st) {
    if (oxt == 4) steps(k, st, std::integral_constant<int, 4>());
    else if (oxt == 2) steps(k, st, std::integral_constant<int, 2>());
    else steps(k, st, std::integral_constant<int, 1>());
  };
  typedef std::integral_constant<int, 1> I1;
  typedef std::integral_constant<int, 2> I2;
  typedef std::integral_constant<int, 3> I3;
  typedef std::integral_constant<int, 5> I5;
  if (a.K == 3 && a.stride == 1) strips(I3(), I1());
  else if (a.K == 3) strips(I3(), I2());
  else if (a.stride == 1) strips(I5(), I1());
  else strips(I5(), I2());
  NNCV_HIP_CHECK(hipGetLastError());
}

namespace {
__global__ __launch_bounds__(256) void transpose_half_kernel(const half_t* __restrict__ w, half_t* __restrict__ dst, int rows, int cols) {
  const int i = blockIdx.x * 256 + threadIdx.x;  // destination: [cols][rows]
  if (i < rows * cols) dst[i] = w[(i % rows) * cols + i / rows];
}
}  // namespace

void launch_transpose_half(const void* w, void* dst, int rows, int cols, hipStream_t s) {
  launch_kernel(transpose_half_kernel, dim3((unsigned)((rows * cols + 255) / 256)), dim3(256), 0, s, static_cast<const half_t*>(w),
                     static_cast<half_t*>(dst), rows, cols);
  NNCV_HIP_CHECK(hipGetLastError());
}

bool se_project_applicable(int HW, int C, int SQ, int F) {
  return C % 8 == 0 && SQ % 8 == 0 && F % 8 == 0 && C <= kSpMaxC && SQ <= kSpMaxSq && F <= 96 && HW >= 1 && (long long)HW * C * 2 < (long long)kOOBm;
}

void launch_se_project(const SeProjectArgs& args, hipStream_t s) {
  SeProjectArgs a = args;
  NNCV_REQUIRE(se_project_applicable(a.HW, a.C, a.SQ, a.F) && a.b1 && a.b2, "se_project: shape not covered");
  ProfScope prof("se_project", 2.0 * a.N * a.HW * (double)a.C * a.F + 4.0 * a.N * a.C * a.SQ,
                 2.0 * ((double)a.N * a.HW * (a.C + a.F * (a.residual ? 2 : 1)) + 2.0 * a.C * a.SQ + (double)a.F * a.C), s);
  const bool ksplit = a.C > 32;
  const int ns = ksplit ? (a.C / 8 + 31) / 32 : 1;
  // 32 pixels to a tile once 16 would be more than four workgroups a CU
  const int pt = !ksplit || (long long)a.N * ((a.HW + 15) / 16) > 1024 ? 2 : 1, px = pt * 16 * (ksplit ? 1 : kSpThreads / 64);
  a.tiles = (a.HW + px - 1) / px;
  a.inv_sq = 1.0f / (float)a.SQ;
  a.inv_c = 1.0f / (float)(a.C / 8);
  const dim3 grid((unsigned)(a.tiles * a.N));
  auto go = [&](auto nsc, auto ftc, auto ptc, auto kc) {
    constexpr int NS = decltype(nsc)::value, FT = decltype(ftc)::value, PT = decltype(ptc)::value;
    constexpr bool KS = decltype(kc)::value;
    auto kern = se_project_kernel<NS, FT, PT, KS>;
    constexpr int lds = KS ? kSpThreads / 64 * FT * PT * 1024 : 0;
    static const bool attr = [&] {
      if (lds > 49152) NNCV_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, lds));
      return true;
    }();
    (void)attr;
    launch_kernel(kern, grid, dim3(kSpThreads), lds, s, a);
  };
  auto filters = [&](auto nsc, auto ptc, auto kc) {
    const int ft = (a.F + 15) / 16;
    if (ft <= 1) go(nsc, std::integral_constant<int, 1>(), ptc, kc);
    else if (ft <= 3) go(nsc, std::integral_constant<int, 3>(), ptc, kc);
    else go(nsc, std::integral_constant<int, 6>(), ptc, kc);
  };
  auto pixels = [&](auto nsc) {
    if (pt == 2) filters(nsc, std::integral_constant<int, 2>(), std::true_type());
    else filters(nsc, std::integral_constant<int, 1>(), std::true_type());
  };
  if (!ksplit) filters(std::integral_constant<int, 1>(), std::integral_constant<int, 2>(), std::false_type());
  else if (ns == 1) pixels(std::integral_constant<int, 1>());
  else if (ns == 2) pixels(std::integral_constant<int, 2>());
  else pixels(std::integral_constant<int, 3>());
  NNCV_HIP_CHECK(hipGetLastError());
}

}  // namespace nncv_hip
