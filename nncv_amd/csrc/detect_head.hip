// YOLOv5 Detect in fp16: the 1x1 head convolutions of all levels and the decode of their results in one launch.
//
//  * What bounds it: a sigmoid per value on the vector units (an exponential and a reciprocal, 13 us of them) and the fp32 result, 85 values per box
//    and anchor (137 MB for 16 images of 640x640, 22 us at the rate of a fill), which overlap in part: without the stores it takes 28 us, with them
//    45.6.  As operators of their own the three convolutions wrote their results and the decode read them again, a value per lane and load:
//    40 us for them and 62 for the decode.
//  * A workgroup has 32 pixels of one image and all A * F filters, so that an anchor's part of its result is one contiguous
//    piece of the output.  Pixels are the rows of the products: a lane has sixteen values of one filter, so scale, shift and the place in LDS
//    are worked out once, and its neighbours write neighbouring floats.  The results wait in LDS in the order of the output (a row of F floats
//    per anchor and pixel), 4 values a box are turned into coordinates there, and the pieces leave as they are, 16 bytes a lane.
//  * Up to 128 channels (the level of most boxes) the filters stay in registers for a run of four tiles, whose pixels arrive a tile ahead, past
//    the stores of the tile before.  Above, filters come from memory two slabs ahead, as fragments.  With filters through LDS, a slab at
//    a time and 64 KB and more for every tile, the launch took 50.9 us.
//  * The levels with the longest K come first, the many short tiles fill up behind them.
#include <algorithm>

#include "mfma_tile.hpp"

namespace nncv_hip {

using namespace mt;

namespace {

constexpr unsigned kOOBd = 0x7fffff00u;
constexpr int kPix = 32, kFil = 256, kLanded = 0x0f70;
typedef __attribute__((address_space(3))) void* lds_ptr_t;
__device__ __forceinline__ void fetch_row(__amdgpu_buffer_rsrc_t rs, unsigned char* lds, unsigned voffset, unsigned soffset) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr_t)lds, 16, voffset, soffset, 0, 0);
}

// A store's cache hint: the result is more than any cache holds and nothing here reads it again.  What it would push out are the tensors of the
// pass: with the plain hint YOLOv5s (16 images) takes 796 us instead of 784.
constexpr int kStreamed = 2;
// bytes of a workgroup's results; channels of a level whose filters stay in registers, and a tile's pixels there
constexpr int kOut = kPix * kFil * 4, kResident = 128, kPixBuf = kPix * kResident * 2, kLds = kOut + 2 * kPixBuf;

// a barrier that leaves loads and stores of memory on their way (__syncthreads waits for them)
__device__ __forceinline__ void meet() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xc07f);  // LDS
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

template <bool VEC>  // every anchor's piece of the output starts on 16 bytes
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4, 6))) void detect_head_kernel(const DetectHeadArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  int l = 0;
#pragma unroll
  for (int k = 1; k < 3; ++k) l = k < a.levels && (int)blockIdx.x >= a.lv[k].first ? k : l;
  const DetectHeadLevel v = a.lv[l];
  const int t0 = (blockIdx.x - v.first) * v.run, t1 = min(t0 + v.run, a.N * v.tiles);
  const __amdgpu_buffer_rsrc_t rs_in = make_rsrc(v.in, v.in_bytes), rs_wt = make_rsrc(v.wt, v.wt_bytes);

  // rows of 128 bytes, eight lanes to a row; chunk position XORed with (row / 2) % 8
  const int pos = lane & 7, sub = lane >> 3;
  auto column = [&](int group) { return pos ^ (((group & 1) << 2) + (sub >> 1)); };
  const int lrow = lane & 31, lh = lane >> 5, key = (lrow >> 1) & 7;
  const int f0 = wave * 32, used = a.A * a.F, F = a.F;
  floatx16 acc;
  float* out_tile = reinterpret_cast<float*>(smem);

  // ---- sigmoids to [anchor][pixel][F]: pixels are the rows of the products, a lane has one filter of sixteen of them ----
  const int f = f0 + lrow, an_ = (f >= F) + (f >= 2 * F) + (f >= 3 * F);
  const bool mine = f < used;
  const float scale = v.scale && f < v.rows ? v.scale[f] : 1.0f, shift = v.shift && f < v.rows ? v.shift[f] : 0.0f;
  auto decode = [&](int p0) __attribute__((always_inline)) {
    if (mine) {
      float* at = out_tile + an_ * (kPix - 1) * F + 4 * lh * F + f;  // (anchor * kPix + pixel) * F + f - anchor * F
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int e = 0; e < 4; ++e) at[(8 * q + e) * F] = sigmoid_fast(acc[4 * q + e] * scale + shift);
    }
    meet();
    // ---- box coordinates ----
    for (int t = threadIdx.x; t < a.A * kPix * 4; t += 512) {
      const int k = t & 3, p = (t >> 2) & (kPix - 1), an = t / (4 * kPix);
      float* at = out_tile + (an * kPix + p) * F + k;
      const float sg = *at;
      int x;
      const int y = fast_div(p0 + p, v.W, v.inv_w, &x);
      float wh = 0.0f;
#pragma unroll
      for (int q = 0; q < 8; ++q) wh = an * 2 + (k & 1) == q ? v.anchor_wh[q] : wh;
      const float s2 = sg * 2.0f;
      *at = k < 2 ? (s2 + ((float)(k == 0 ? x : y) - 0.5f)) * v.stride : (s2 * s2) * wh;
    }
    meet();
  };
  // ---- an anchor's piece: npix * F consecutive floats; of 16 bytes at a time there are at most four a thread, all of them requested ----
  auto store = [&](int n, int p0, int npix) __attribute__((always_inline)) {
    float* to = a.out + ((long long)n * a.boxes_total + v.box0 + p0) * F;
    if constexpr (VEC) {
      const __amdgpu_buffer_rsrc_t rs = make_rsrc(to, 0x7fffffffu);
      const int piece = npix * F >> 2;
      const float inv = 1.0f / (float)piece;
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int i = s * 512 + (int)threadIdx.x;
        int r;
        const int an = fast_div(i, piece, inv, &r);
        const u32x4 q = *reinterpret_cast<const u32x4*>(out_tile + (an < a.A ? an * kPix * F + 4 * r : 0));
        __builtin_amdgcn_raw_buffer_store_b128(q, rs, an < a.A ? (unsigned)(an * v.HW * F + 4 * r) * 4u : 0xfffffff0u, 0, kStreamed);
      }
    } else {
      for (int an = 0; an < a.A; ++an)
        for (int i = threadIdx.x; i < npix * F; i += 512) to[(long long)an * v.HW * F + i] = out_tile[an * kPix * F + i];
    }
  };

  // ---- operands: the kilobyte of filters (wave's 32, 16-channel step k), and chunk 2 k + lh of a pixel's slab of 64 channels ----
  const int slabs = v.C >> 6;
  const unsigned wlane = (unsigned)(((wave >> 1) * slabs * 8 + (wave & 1)) * 1024 + lane * 16);
  auto filters = [&](int k) __attribute__((always_inline)) { return __builtin_amdgcn_raw_buffer_load_b128(rs_wt, wlane + (unsigned)k * 2048u, 0, 0); };
  auto pixels = [&](const unsigned char* slab, int k) __attribute__((always_inline)) {
    return *reinterpret_cast<const u32x4*>(slab + lrow * 128 + ((2 * k + lh) ^ key) * 16);
  };
  u32x4 w[8];

  if (v.C <= kResident) {
    // Filters in registers, a run of tiles one after the other: wave w brings rows 8 (w % 4) .. of slab w / 4 of the next tile's pixels
    const int group = wave & 3, row = group * 8 + sub;
    auto fetch = [&](int t) __attribute__((always_inline)) {
      int tile;
      const int n = fast_div(t, v.tiles, v.inv_tiles, &tile), p = tile * kPix + row;
      const unsigned at = t < t1 && p < v.HW ? (unsigned)((n * v.HW + p) * v.pix * 2 + column(group) * 16) : kOOBd;
      if ((wave >> 2) < slabs) fetch_row(rs_in, smem + kOut + (t & 1) * kPixBuf + wave * 1024, at, (wave >> 2) * 128);
    };
    fetch(t0);
#pragma unroll
    for (int k = 0; k < 8; ++k) w[k] = filters(k < 4 || slabs > 1 ? k : 0);
    for (int t = t0; t < t1; ++t) {
      int tile;
      const int n = fast_div(t, v.tiles, v.inv_tiles, &tile), p0 = tile * kPix, npix = min(kPix, v.HW - p0);
      if (VEC && t > t0) __builtin_amdgcn_s_waitcnt(kLanded | 4);  // (the last tile's four stores may be on their way)
      else __builtin_amdgcn_s_waitcnt(kLanded);
      meet();  // this tile's pixels are there, the last one's results have been read
      fetch(t + 1);
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[e] = 0.0f;
      const unsigned char* at = smem + kOut + (t & 1) * kPixBuf;
#pragma unroll
      for (int k = 0; k < 4; ++k) Mma<half_t>::run(pixels(at, k), w[k], acc);
      if (slabs > 1) {
#pragma unroll
        for (int k = 0; k < 4; ++k) Mma<half_t>::run(pixels(at + kPix * 128, k), w[4 + k], acc);
      }
      decode(p0);
      store(n, p0, npix);
    }
    return;
  }

  // One tile: up to 512 channels of its pixels at a time in the place of the results, filters two slabs ahead
  int tile;
  const int n = fast_div(t0, v.tiles, v.inv_tiles, &tile), p0 = tile * kPix, npix = min(kPix, v.HW - p0);
#pragma unroll
  for (int k = 0; k < 8; ++k) w[k] = filters(k);
#pragma unroll
  for (int e = 0; e < 16; ++e) acc[e] = 0.0f;
  const int group = wave & 3, row = group * 8 + sub;
  const unsigned at0 = row < npix ? (unsigned)((n * v.HW + p0 + row) * v.pix * 2 + column(group) * 16) : kOOBd;
  for (int s0 = 0; s0 < slabs; s0 += 8) {
    const int ns = min(8, slabs - s0);
    if (s0 > 0) meet();
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if ((wave >> 2) + 2 * i < ns) fetch_row(rs_in, smem + (i * 8 + wave) * 1024, at0, (s0 + (wave >> 2) + 2 * i) * 128);
    __builtin_amdgcn_s_waitcnt(kLanded);
    meet();
    for (int s = 0; s < ns; s += 2) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if (s + h >= ns) break;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          Mma<half_t>::run(pixels(smem + (s + h) * (kPix * 128), k), w[4 * h + k], acc);
          w[4 * h + k] = filters((s0 + s + h + 2) * 4 + k);  // (behind the last: zeros, or another group's)
        }
      }
    }
  }
  meet();
  decode(p0);
  store(n, p0, npix);
}

}  // namespace

// Heads of up to 256 filters and at least 64 values a box, over whole slabs.
bool detect_head_applicable(int A, int F, int C, long long in_bytes) {
  return A >= 1 && A <= 4 && F >= 64 && A * F <= kFil && C >= 64 && C % 64 == 0 && in_bytes < (long long)kOOBd;
}

void launch_detect_head(const DetectHeadArgs& a_in, hipStream_t s) {
  DetectHeadArgs a = a_in;
  bool vec = (a.boxes_total * a.F) % 4 == 0 && reinterpret_cast<uintptr_t>(a.out) % 16 == 0;
  long long blocks = 0;
  double flops = 0, bytes = 0;
  for (int l = 0; l < a.levels; ++l) {
    DetectHeadLevel& v = a.lv[l];
    v.tiles = (v.HW + kPix - 1) / kPix;
    v.inv_tiles = 1.0f / (float)v.tiles;
    v.inv_w = 1.0f / (float)v.W;
    v.first = (int)blocks;
    v.in_bytes = (unsigned)((long long)a.N * v.HW * v.pix * 2);
    v.wt_bytes = (unsigned)weight_frag1x1_bytes(v.rows, v.C);
    // (filters in registers: four tiles to a workgroup, fewer where that would leave workgroups of the CUs idle)
    const long long tiles = (long long)a.N * v.tiles;
    v.run = v.C <= kResident ? (int)std::min(4ll, std::max(1ll, tiles / 768)) : 1;
    blocks += (tiles + v.run - 1) / v.run;
    NNCV_REQUIRE(tiles < (1 << 24), "detect_head: too many boxes");
    vec = vec && (long long)v.HW * a.F * a.A < 1ll << 29 && ((long long)v.HW * a.F) % 4 == 0 && (v.box0 * a.F) % 4 == 0;
    flops += 2.0 * a.N * v.HW * v.C * a.A * a.F;
    bytes += 2.0 * ((double)a.N * v.HW * v.C + (double)v.rows * v.C) + 4.0 * a.N * v.HW * a.A * a.F;
    NNCV_REQUIRE(v.HW < (1 << 24) && v.rows % 4 == 0 && v.rows <= kFil, "detect_head: level too large");
  }
  NNCV_REQUIRE(blocks < (1 << 24), "detect_head: too many boxes");
  constexpr int lds = kLds;
  ProfScope prof("detect_head", flops, bytes, s);
  if (vec) launch_kernel(detect_head_kernel<true>, dim3((unsigned)blocks), dim3(512), lds, s, a);
  else launch_kernel(detect_head_kernel<false>, dim3((unsigned)blocks), dim3(512), lds, s, a);
  NNCV_HIP_CHECK(hipGetLastError());
}

}  // namespace nncv_hip
