// fp16 pointwise convolution + BN + activation whose result is only averaged over the image (the end of MobileNetV3's features,
// tests/Nets/MobileNetV3.mlir): the means leave the launch, the map is never stored.
#include "mfma_tile.hpp"

namespace nncv_hip {

using namespace mt;

namespace {

constexpr unsigned kOOBp = 0x7fffff00u;  // byte offset beyond any buffer this kernel accepts
constexpr int kSteps = 6;                // K steps of 16 channels that are asked for together

// A workgroup = one image x 32 * (4 / PW) filters; its waves share the filters out in blocks of 32 and the pixels in tiles of 32,
// PW waves to a block.  The pixels are the rows of the products, so a lane's 16 sums belong to one filter: activation and sum over
// pixels stay in its registers, fp32, and meet across the wave's halves and the PW waves once at the end.  Operands come straight
// from memory (L2: every block of filters reads the image again), all of 96 channels at once, so a tile is one trip.
// What bounds it: the launch and that trip.  32x7x7x96 -> 576 takes 4.7 us, where the convolution and the pass over its
// map took 5.4 + 4.8 (0.17 GFLOP and 2 us of launch: the rest is one trip for arguments and one for operands).
template <int PW>
__global__ __launch_bounds__(256) void conv_pool_kernel(const ConvPoolArgs a) {
  constexpr int FB = 4 / PW, BF = 32 * FB;
  __shared__ float part[PW][BF];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), wp = wave % PW, wf = wave / PW;
  const int lrow = lane & 31, lh = lane >> 5;
  // workgroups x, x + 8, ... (one XCD's) take neighbouring tiles: the blocks of filters of an image share an L2
  int fb, n;
  {
    const int tiles = a.N * a.blocks, per = (tiles + 7) >> 3, rem = tiles & 7, x = blockIdx.x & 7, i = blockIdx.x >> 3;
    const int t = rem == 0 ? x * per + i : (x < rem ? x * per : rem * per + (x - rem) * (per - 1)) + i;
    n = fast_div(t, a.blocks, a.inv_blocks, &fb);
    n = __builtin_amdgcn_readfirstlane(n);
    fb = __builtin_amdgcn_readfirstlane(fb);
  }
  const int f = fb * BF + wf * 32 + lrow, chunks = a.C >> 3;
  const __amdgpu_buffer_rsrc_t rs_in = make_rsrc(static_cast<const half_t*>(a.in) + (long long)n * a.HW * a.pix, (unsigned)(a.HW * a.pix) * 2u);
  const __amdgpu_buffer_rsrc_t rs_w = make_rsrc(a.wt, (unsigned)(a.F * a.C) * 2u);
  const bool there = f < a.F;
  const float sc = a.scale && there ? a.scale[f] : 1.0f, sh = a.shift && there ? a.shift[f] : 0.0f;
  const unsigned wofs = there ? (unsigned)(f * a.C + lh * 8) * 2u : kOOBp;
  float sum = 0.0f;
  for (int p0 = wp * 32; p0 < a.HW; p0 += PW * 32) {
    const unsigned xofs = p0 + lrow < a.HW ? (unsigned)((p0 + lrow) * a.pix + lh * 8) * 2u : kOOBp;
    floatx16 acc = {};
    for (int c0 = 0; c0 < chunks; c0 += 2 * kSteps) {
      u32x4 x[kSteps], w[kSteps];
#pragma unroll
      for (int k = 0; k < kSteps; ++k) {
        const bool in = c0 + 2 * k + lh < chunks;
        x[k] = __builtin_amdgcn_raw_buffer_load_b128(rs_in, in ? xofs + (unsigned)(c0 + 2 * k) * 16u : kOOBp, 0, 0);
        w[k] = __builtin_amdgcn_raw_buffer_load_b128(rs_w, in ? wofs + (unsigned)(c0 + 2 * k) * 16u : kOOBp, 0, 0);
      }
#pragma unroll
      for (int k = 0; k < kSteps; ++k) Mma<half_t>::run(x[k], w[k], acc);
    }
    float y[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) y[e] = acc[e] * sc + sh;
    act_apply_n<true>(y, a.act);
#pragma unroll
    for (int e = 0; e < 16; ++e) sum += p0 + 8 * (e >> 2) + 4 * lh + (e & 3) < a.HW ? y[e] : 0.0f;
  }
  sum += __shfl_xor(sum, 32);
  if (lane < 32) part[wp][wf * 32 + lane] = sum;
  __syncthreads();
  const int o = threadIdx.x;
  if (o < BF && fb * BF + o < a.F) {
    float s = part[0][o];
#pragma unroll
    for (int q = 1; q < PW; ++q) s += part[q][o];
    static_cast<half_t*>(a.out)[(long long)n * a.F + fb * BF + o] = (half_t)(s / (float)a.HW);
  }
}

}  // namespace

// Two launches take longer up to here, us, there / here, 96 -> 576: 32x7x7 5.4 + 4.8 / 4.7, 32x10x10 7.7 + 6.3 / 7.7, 32x16x16 11.3 + 6.3 / 10.0, 256x7x7
// 14.3 + 6.7 / 12.3, 1x20x20 6.3 + 6.7 / 9.3.  Nothing is staged or asked for ahead of a tile, so beyond it the convolution's own kernels
// and a pass over the map are the faster (64x20x20x320 -> 1280: 38 + 14 against 161).
bool conv_pool_applicable(int N, int HW, int pix, int C, int F) {
  return HW <= 512 && (long long)N * HW <= 16384 && C <= 128 && C % 8 == 0 && pix % 8 == 0 && (long long)N * ((F + 31) / 32) < (1 << 24) &&
         (long long)HW * pix * 2 < (long long)kOOBp - 65536 && (long long)F * C * 2 < (long long)kOOBp - 65536;
}

void launch_conv_pool(const ConvPoolArgs& args, hipStream_t s) {
  ConvPoolArgs a = args;
  NNCV_REQUIRE(conv_pool_applicable(a.N, a.HW, a.pix, a.C, a.F), "conv_pool: shape not covered");
  ProfScope prof("conv_pool", 2.0 * a.N * a.HW * (double)a.C * a.F, 2.0 * ((double)a.N * a.HW * a.C + (double)a.F * a.C + (double)a.N * a.F), s);
  const bool wide = a.HW > 64;  // (up to two tiles an image: two waves share its pixels)
  a.blocks = (a.F + (wide ? 31 : 63)) / (wide ? 32 : 64);
  a.inv_blocks = 1.0f / (float)a.blocks;
  const dim3 grid((unsigned)(a.N * a.blocks));
  if (wide) launch_kernel(conv_pool_kernel<4>, grid, dim3(256), 0, s, a);
  else launch_kernel(conv_pool_kernel<2>, grid, dim3(256), 0, s, a);
  NNCV_HIP_CHECK(hipGetLastError());
}

}  // namespace nncv_hip
