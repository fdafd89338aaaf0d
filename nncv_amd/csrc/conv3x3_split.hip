// fp32 3x3 pad-1 stride-1 convolution on the bf16 matrix pipes, operands split in three (split.hpp), with the haloed input patch
// resident in LDS.  Tiles and their plan are those of conv3x3_patch.hip: 64 * WS pixel slots x 32 * NI filters a workgroup, channel
// slabs of 32.
//
//  * The patch of a slab is loaded once, split once, and read by nine taps: splitting pixels costs a ninth of what it costs a
//    kernel that reads taps from memory.  A cell of LDS is one pixel's 32 channels as three runs of 64 bytes, one per piece.
//  * Filters are split once, when the layer is made, in fragment order (launch_weight_frag3x3): an operand of a wave is three
//    contiguous kilobytes, straight into registers, three steps ahead.
//  * Two patch buffers: a slab is multiplied while the next one is split into the other buffer, between the products, and the one
//    after that is on its way to registers.  One barrier a slab.
//  * Eight waves, or four where two workgroups share a CU (launch_ws1).  A wave's share of the tile is 64 slots x 32 filters (WS = 1,
//    NI = 1: 32 x 32), its K groups take a 16-channel half of a slab each, four of them the even or the odd taps of a half; their
//    sums meet in LDS.
//  * A wave with a sum that is not finite takes its sums again with the fp32 instructions, from memory (split.hpp).
//  * FLAT: tiles of 32 consecutive pixels for small maps (conv3x3_split_flat_us).
//  * What bounds it: the matrix pipes where tiles fill the CUs (six products, 2.7 times the fp32 instructions' rate), a slab's
//    barrier and the LDS reads behind it where they do not: two waves a SIMD cover each other there (six 224x224 images classified by an
//    fp32 ResNet-18: 373 us with one, 353 with two).
#include <type_traits>

#include "patch_args.hpp"
#include "split.hpp"

namespace nncv_hip {

using namespace mt;

namespace {

constexpr int kCell = 208;              // 3 x 64 + 16: at 13 units of 16 bytes, 16 neighbouring cells touch every bank once
constexpr int kRowSpare = 96;           // behind a patch row: its pitch is 13 TW units mod 16 then, as if a tile's rows were one

constexpr int split_units(int ws) { return ws == 1 ? 2 : 4; }  // waves that a workgroup's tile is dealt to

// FLAT: a tile is 32 consecutive pixels of the batch, whatever rows and images they lie in (images one row of zeros apart in the
// patch), and a trip of the slab loop takes two slabs: a wave a 16-channel half of one, and the even or the odd taps.
constexpr int kFlatCells[2] = {128, 160};  // (WS = 0 and -1: two and three passes of the loader)

template <int WS>
struct SplitCfg {
  static constexpr int cap = PatchCap<WS>::pix;
  static constexpr int buffers = WS == 4 ? 1 : 2;                     // (256 slots: layers of one slab)
  static constexpr int patch = cap * kCell, dump = buffers * patch, scale = dump + 640, smem = scale + 512;
};

template <int V>
struct FlatCfg {
  static constexpr int cap = kFlatCells[V], buffers = 2;
  static constexpr int patch = 2 * cap * kCell, dump = buffers * patch, scale = dump + 640, smem = scale + 512;
};
template <> struct SplitCfg<0> : FlatCfg<0> {};
template <> struct SplitCfg<-1> : FlatCfg<1> {};
constexpr int split_threads(int ws, int kg) { return 64 * kg * (ws <= 0 ? 1 : split_units(ws)); }

template <int WS, int NI, int KG>  // KG: K groups, waves that share a tile's sums
__global__ __launch_bounds__(split_threads(WS, KG)) __attribute__((amdgpu_waves_per_eu(2, 2))) void conv3x3_split_kernel(
    // (the values the patch addressing needs first: preloaded into SGPRs)
    const void* in_p, int tiles_p, int tiles_y_p, int tn_p, int th_p, int n_p, int h_p, int w_p, int c_p, int rw_log_p, int xcd_by_filter_p,
    unsigned in_bytes_p, int txw_p, const PatchArgs a_rest) {
  PatchArgs a = a_rest;
  a.txw = txw_p;
  a.in = in_p; a.tiles = tiles_p; a.tiles_y = tiles_y_p; a.TN = tn_p; a.TH = th_p; a.N = n_p; a.H = h_p; a.W = w_p; a.C = c_p;
  a.rw_log = rw_log_p; a.xcd_by_filter = xcd_by_filter_p; a.in_bytes = in_bytes_p;
  typedef SplitCfg<WS> Cfg;
  constexpr bool FLAT = WS <= 0;
  constexpr int kThreads = split_threads(WS, KG), kPass = kThreads / 8;  // loader: 8 threads a pixel
  constexpr int kCellPasses = (Cfg::cap + kPass - 1) / kPass, kSlabs = FLAT ? 2 : 1, kPasses = kCellPasses * kSlabs;  // (pass i: cells of pass i % kCellPasses)
  constexpr int JN = WS <= 1 && NI == 1 ? 1 : 2;  // slot blocks of a wave
  constexpr int kQuads = JN * 4;
  static_assert(WS != 2 || NI == 2, "128 slots: two waves to a filter half");
  static_assert(WS != 4 || NI == 1, "256 slots: every wave has its own");
  extern __shared__ __align__(16) unsigned char smem[];

  int tile, fblk;  // (as conv3x3_patch.hip)
  if (a.xcd_by_filter) {
    const int lin = blockIdx.y * gridDim.x + blockIdx.x, per = gridDim.y / kXcdsP, k = lin / kXcdsP;
    fblk = lin % kXcdsP + kXcdsP * (k % per);
    tile = k / per;
  } else {
    const int per_xcd = (a.tiles + kXcdsP - 1) / kXcdsP;
    tile = (blockIdx.x % kXcdsP) * per_xcd + blockIdx.x / kXcdsP;
    fblk = blockIdx.y;
  }
  if (tile >= a.tiles) return;
  const int TW = FLAT ? a.W : a.txw & 0xffff, ntx = a.txw >> 16;
  // FLAT: rows of the images with one row of zeros behind each, `top` the one above the tile's first pixel
  const int P = a.N * a.H * a.W;
  auto virtual_row = [&](int p, int* x) {
    int rem;
    const int n = fast_div(p, a.H * a.W, a.inv_thw, &rem);
    return n * (a.H + 1) + fast_div(rem, a.W, a.inv_w, x);
  };
  int top = 0, flat_rows = 0;
  if constexpr (FLAT) {
    int x;
    top = virtual_row(tile * 32, &x) - 1;
    flat_rows = virtual_row(min(tile * 32 + 31, P - 1), &x) + 2 - top;
  }
  const int n0 = (tile / a.tiles_y) * a.TN;
  int band = tile % a.tiles_y, x0 = 0;
  if (!FLAT && ntx > 1) {
    x0 = (band % ntx) * TW;
    band /= ntx;
  }
  const int y0 = band * a.TH, PH = a.TH + 2, PW = TW + 2, RP = PW * kCell + kRowSpare;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // K group g: channels 16 (g % 2) .. of a slab, and with four groups the taps 2 i + g / 2.  Waves w and w + 4 share a SIMD: one
  // of them has the five even taps, the other the four odd ones.
  // FLAT: one unit, group g has slab g / 4 of the trip.
  const int unit = wave / KG, kg = KG == 4 ? (wave & 3) ^ (unit << 1) : wave % KG, slab_of = KG == 8 ? kg >> 2 : 0;
  auto wave_of = [&](int g) { return unit * KG + (KG == 4 ? g ^ (unit << 1) : g); };
  const int slot0 = FLAT ? 0 : WS == 4 ? unit * 64 : WS == 2 ? (unit & 1) * 64 : NI == 1 ? unit * 32 : 0;
  const int half = NI == 1 ? fblk & 1 : WS == 2 ? unit >> 1 : unit;                  // of the 64-filter block
  const int fb64 = NI == 1 ? fblk >> 1 : fblk, f0 = fb64 * 64 + half * 32;          // this wave's first filter
  const int lrow = lane & 31, lh = lane >> 5;
  const __amdgpu_buffer_rsrc_t rs_in = make_rsrc(a.in, a.in_bytes);
  const __amdgpu_buffer_rsrc_t rs_wf = make_rsrc(a.wf, a.wf_bytes);
  const int nslab = a.C >> 5, niter = nslab * 9;

  // ---- patch loader: the patch is walked as rows of 2^rw_log pixels ----
  const int p8 = tid >> 3, c4 = tid & 7, pc = c4 * 16;
  const int prows = a.TN * PH, rwm = (1 << a.rw_log) - 1;
  const unsigned ces = (unsigned)(a.pix * 4);
  unsigned pvoff[kCellPasses];
  // four channels go where the operand of their step has them: units 4 s + h and 4 s + 2 + h of a step s are lane half h's.
  // Lanes whose pass lies outside the patch write to a dump behind it.
  unsigned pdst[kCellPasses];
  const int sub = (c4 >> 2) * 32 + (c4 & 1) * 16 + ((c4 >> 1) & 1) * 8;
#pragma unroll
  for (int i = 0; i < kCellPasses; ++i) {
    const int q = i * kPass + p8;
    bool ok, cell;
    int r, px, at;
    if constexpr (FLAT) {
      int y;
      r = fast_div(q, PW, __builtin_amdgcn_rcpf((float)PW), &px);
      const int n = fast_div(max(top + r, 0), a.H + 1, a.inv_ph, &y);
      cell = r < flat_rows;
      ok = cell & (top + r >= 0) & (n < a.N) & (y < a.H) & ((unsigned)(px - 1) < (unsigned)a.W);
      at = (n * a.H + y) * a.W + px - 1;
    } else {
      r = q >> a.rw_log, px = q & rwm;
      int n = n0, py = r;
      if (a.TN > 1) n += fast_div(r, PH, a.inv_ph, &py);
      const int iy = y0 + py - 1;
      cell = (px < PW) & (r < prows);
      ok = (r < prows) & (n < a.N) & ((unsigned)iy < (unsigned)a.H) & ((unsigned)(x0 + px - 1) < (unsigned)a.W);
      at = (n * a.H + iy) * a.W + x0 + px - 1;
    }
    pvoff[i] = ok ? __umul24((unsigned)at, ces) + pc : kOOBp;
    pdst[i] = cell ? __umul24(r, RP) + __umul24(px, kCell) + sub : Cfg::dump + lane * 8;
  }
  u32x4 pregs[kPasses];
  // (`trip`: of the slab loop)
  auto pload = [&](int i, int trip) {
    pregs[i] = __builtin_amdgcn_raw_buffer_load_b128(rs_in, pvoff[i % kCellPasses] + (kSlabs * trip + i / kCellPasses) * 128, 0, 0);
  };
  auto pstore = [&](int i, unsigned to) {  // `to`: byte offset of the buffer (the dump is shared)
    const floatx4 v = __builtin_bit_cast(floatx4, pregs[i]);
    unsigned p[2][3];
    split_pair(v[0], v[1], p[0]);
    split_pair(v[2], v[3], p[1]);
    const unsigned d = pdst[i % kCellPasses];
    unsigned char* dst = smem + (d < (unsigned)Cfg::dump ? d + to + i / kCellPasses * (Cfg::cap * kCell) : d);
#pragma unroll
    for (int c = 0; c < 3; ++c) *reinterpret_cast<u32x2*>(dst + c * 64) = u32x2{p[0][c], p[1][c]};
  };
#pragma unroll
  for (int i = 0; i < kPasses; ++i) pload(i, 0);
  __builtin_amdgcn_sched_barrier(0);

  // ---- filters: the operand of iteration (slab, tap), step k, half i, piece c is the kilobyte at
  //      (((fb64 * niter + it) * 2 + k) * 2 + i) * 3 + c ----
  const int wbase = (fb64 * niter * 4 + (kg & 1) * 2 + half) * 3072;
  const unsigned wlane = lane * 16;
  auto wload = [&](u32x4 (&r)[1][3], int it, int k) __attribute__((always_inline)) {
    const int so = it < niter ? wbase + it * 12288 + k * 6144 : 0;  // past the end: block 0 again (never used)
#pragma unroll
    for (int c = 0; c < 3; ++c) r[0][c] = __builtin_amdgcn_raw_buffer_load_b128(rs_wf, wlane, so + c * 1024, 0);
  };
  if (tid < 64) {
    const int f = fb64 * 64 + tid;
    float* ss = reinterpret_cast<float*>(smem + Cfg::scale);
    ss[tid] = a.scale && f < a.F ? a.scale[f] : 1.0f;
    ss[64 + tid] = a.shift && f < a.F ? a.shift[f] : 0.0f;
  }

  // ---- this lane's pixel slots ----
  const int nslots = a.TN * a.TH * TW;
  int sbase[JN];  // byte offset of the slot's tap-(0,0) cell
  int obase[JN];  // element offset of the slot's output pixel row, or -1
#pragma unroll
  for (int j = 0; j < JN; ++j) {
    const int sl0 = slot0 + j * 32 + lrow;
    int sl = sl0;
    if constexpr (FLAT) {
      const int p = tile * 32 + lrow;
      int x;
      const int r = virtual_row(min(p, P - 1), &x) - 1 - top;
      sbase[j] = (int)__umul24(r, RP) + (int)__umul24(x, kCell) + lh * 16 + (kg & 1) * 32 + slab_of * (Cfg::cap * kCell);
      obase[j] = p < P ? p * a.ldo : -1;
      continue;
    }
    if (sl0 >= nslots) {  // reads with the slot 16, 32 ... before it (the same banks), is not stored
      const int back = (((sl0 - nslots) >> 4) + 1) << 4;
      sl = sl0 >= back ? sl0 - back : 0;
    }
    int nl = 0, rem = sl, tx;
    if (a.TN > 1) nl = fast_div(sl, a.TH * TW, a.inv_thw, &rem);
    const int ty = fast_div(rem, TW, a.inv_w, &tx);
    const bool ok = (sl < nslots) & ((n0 + nl) < a.N) & ((y0 + ty) < a.H) & ((x0 + tx) < a.W);
    sbase[j] = (ok ? (int)__umul24(__umul24(nl, PH) + ty, RP) + (int)__umul24(tx, kCell) : 0) + lh * 16 + (kg & 1) * 32;
    obase[j] = (ok && sl0 < nslots) ? (((n0 + nl) * a.H + y0 + ty) * a.W + x0 + tx) * a.ldo : -1;
  }

  floatx16 big[1][JN], low[1][JN];
#pragma unroll
  for (int j = 0; j < JN; ++j)
#pragma unroll
    for (int v = 0; v < 16; ++v) big[0][j][v] = low[0][j][v] = 0.0f;

  // ---- tap loop: one trip = one slab = this wave's taps, unrolled.  Under the products of a step: the pixel operand of the next
  //      one is read, the filters of NSET steps further on are asked for, and a share of the next slab's patch is split into the
  //      other buffer and that of the slab after it asked for ----
  auto walk = [&](auto par_c) __attribute__((always_inline)) {
    constexpr int PAR = decltype(par_c)::value;                                 // four K groups: odd taps
    constexpr int kSteps = KG == 1 ? 18 : KG == 2 ? 9 : 5 - PAR, NSET = KG >= 4 ? kSteps : JN == 1 ? 9 : 3;  // steps whose filters are on their way
    auto tap_of = [](int st) constexpr { return KG == 1 ? st / 2 : KG == 2 ? st : 2 * st + PAR; };
    auto k_of = [](int st) constexpr { return KG == 1 ? st & 1 : 0; };
    u32x4 w[NSET][1][3];
#pragma unroll
    for (int t = 0; t < NSET; ++t) wload(w[t], slab_of * 9 + tap_of(t), k_of(t));
    u32x4 ring[2][JN][3];
    int row[3][JN];
    auto ldp = [&](auto step_c) __attribute__((always_inline)) {
      constexpr int st = decltype(step_c)::value, t = tap_of(st), k = k_of(st);
#pragma unroll
      for (int j = 0; j < JN; ++j)
#pragma unroll
        for (int c = 0; c < 3; ++c) ring[st & 1][j][c] = *reinterpret_cast<const u32x4*>(smem + row[t / 3][j] + (t % 3) * kCell + k * 32 + c * 64);
    };
#pragma unroll
    for (int i = 0; i < kPasses; ++i) {
      pstore(i, 0);
      if (Cfg::buffers == 2) pload(i, 1);
    }
    __syncthreads();
    for (int slab = 0; slab < nslab / kSlabs; ++slab) {  // (FLAT: pairs of them)
      const int at = Cfg::buffers == 2 ? (slab & 1) * Cfg::patch : 0;
      const unsigned other = Cfg::patch - at;
#pragma unroll
      for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int j = 0; j < JN; ++j) row[r][j] = sbase[j] + at + r * RP;
      ldp(std::integral_constant<int, 0>());
      __builtin_amdgcn_sched_barrier(0);
      auto steps = [&](auto self, auto step_c) __attribute__((always_inline)) -> void {
        constexpr int st = decltype(step_c)::value;
        if constexpr (st < kSteps) {
          constexpr int nx = st + NSET, p0 = st * kPasses / kSteps, p1 = Cfg::buffers == 2 ? (st + 1) * kPasses / kSteps : p0;
          if constexpr (st + 1 < kSteps) ldp(std::integral_constant<int, st + 1>());
          split_products(w[st % NSET], ring[st & 1], big, low);
          wload(w[st % NSET], (kSlabs * (slab + nx / kSteps) + slab_of) * 9 + tap_of(nx % kSteps), k_of(nx % kSteps));
#pragma unroll
          for (int i = p0; i < p1; ++i) {
            pstore(i, other);
            pload(i, slab + 2);
          }
          constexpr int kMma = 6 * JN, kValu = (30 * (p1 - p0) + kMma - 1) / kMma;
#pragma unroll
          for (int n = 0; n < kMma; ++n) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            if (kValu) __builtin_amdgcn_sched_group_barrier(0x002, kValu, 0);
            __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
          }
          __builtin_amdgcn_sched_barrier(0);
          self(self, std::integral_constant<int, st + 1>());
        }
      };
      steps(steps, std::integral_constant<int, 0>());
      __syncthreads();  // every wave has left this patch and written its share of the next
    }
  };
  if constexpr (KG < 4) {
    walk(std::integral_constant<int, 0>());
  } else {  // (as many barriers on both sides)
    if (!(kg & 2)) walk(std::integral_constant<int, 0>());
    else walk(std::integral_constant<int, 1>());
  }

  if (__builtin_expect(split_sums(big, low), 0)) {
    // a slab of this wave: 16 channels, or both halves with one K group, of its taps; two steps of eight channels each
    const int taps = KG >= 4 ? 5 - ((kg >> 1) & 1) : 9, per = KG == 1 ? 2 * taps : taps, HW = a.H * a.W;
    int py[JN], px[JN], img[JN];
#pragma unroll
    for (int j = 0; j < JN; ++j) {
      const int p = max(obase[j], 0) / a.ldo, n = p / HW, rem = p - n * HW, y = rem / a.W;
      img[j] = n * HW;
      py[j] = obase[j] >= 0 ? y : -(1 << 20);
      px[j] = rem - y * a.W;
    }
    const __amdgpu_buffer_rsrc_t rs_wt = make_rsrc(a.wt, (unsigned)a.F * 9u * (unsigned)a.C * 4u);
    plain_products(big, 2 * per * (nslab / kSlabs), [&](int step, u32x4 (&f)[1], u32x4 (&x)[JN]) {
      const int t = step >> 1, trip = t / per, slab = kSlabs * trip + slab_of, st = t - trip * per;
      const int tap = KG == 1 ? st >> 1 : KG == 2 ? st : 2 * st + ((kg >> 1) & 1), half16 = KG == 1 ? st & 1 : kg & 1;
      const int c = slab * 32 + half16 * 16 + (step & 1) * 8 + 4 * lh, dy = tap / 3 - 1, dx = tap - tap / 3 * 3 - 1;
      const bool in = slab < nslab;
      f[0] = __builtin_amdgcn_raw_buffer_load_b128(rs_wt, in ? (unsigned)((min(f0 + lrow, a.F - 1) * 9 + tap) * a.C + c) * 4u : kOOBp, 0, 0);
#pragma unroll
      for (int j = 0; j < JN; ++j) {
        const bool ok = in & ((unsigned)(py[j] + dy) < (unsigned)a.H) & ((unsigned)(px[j] + dx) < (unsigned)a.W);
        x[j] = __builtin_amdgcn_raw_buffer_load_b128(rs_in, ok ? (unsigned)((img[j] + (py[j] + dy) * a.W + px[j] + dx) * a.pix + c) * 4u : kOOBp, 0, 0);
      }
    });
  }

  // ---- out: quad (j, g): filters 8 g + 4 lh .. + 3 of slot block j.  K group g finishes quads g, g + KG ... ----
  constexpr int kMine = (kQuads + KG - 1) / KG;
  const bool finishes = kg < kQuads;  // (FLAT: four quads, eight groups)
  auto sum_of = [&](int q) {
    const int j = q / 4, g = q & 3;
    floatx4 s;
#pragma unroll
    for (int e = 0; e < 4; ++e) s[e] = big[0][j][4 * g + e];
    return s;
  };
  const float* res = static_cast<const float*>(a.residual);
  float* out = static_cast<float*>(a.out);
  const float* ss = reinterpret_cast<const float*>(smem + Cfg::scale) + half * 32 + 4 * lh;
  auto at_of = [&](int q, int* f) {  // element of the quad's first result, -1: not stored
    const int o = JN == 2 && q / 4 ? obase[JN - 1] : obase[0];
    *f = f0 + (q & 3) * 8 + 4 * lh;
    return o >= 0 && *f < a.F ? (long long)o + *f : -1ll;
  };
  floatx4 rv[kMine];
  if (res) {
#pragma unroll
    for (int m = 0; m < kMine; ++m) {
      int f;
      const long long at = finishes ? at_of(KG * m + kg, &f) : -1ll;
      rv[m] = at >= 0 ? *reinterpret_cast<const floatx4*>(res + at) : floatx4{};
    }
  }
  floatx4 sums[kMine];
  if constexpr (KG == 1) {
#pragma unroll
    for (int m = 0; m < kMine; ++m) sums[m] = sum_of(m);
  } else {
    floatx4* part = reinterpret_cast<floatx4*>(smem);  // [wave][quad][lane]
#pragma unroll
    for (int q = 0; q < kQuads; ++q) part[(wave * kQuads + q) * 64 + lane] = sum_of(q);
    __syncthreads();
    if (!finishes) return;
#pragma unroll
    for (int m = 0; m < kMine; ++m) {
      floatx4 v[KG];
#pragma unroll
      for (int g = 0; g < KG; ++g) v[g] = part[(wave_of(g) * kQuads + KG * m + kg) * 64 + lane];
#pragma unroll
      for (int d = 1; d < KG; d *= 2)
#pragma unroll
        for (int g = 0; g + d < KG; g += 2 * d) v[g] += v[g + d];
      sums[m] = v[0];
    }
  }
  auto put = [&](int q, long long at, floatx4 y, const floatx4& r) {
    const int b = (q & 3) * 8;
    y = y * *reinterpret_cast<const floatx4*>(ss + b) + *reinterpret_cast<const floatx4*>(ss + 64 + b);
    if (res) y += r;
    if (a.relu == kActRelu) {
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] = relu_ugt(y[e]);
    }
    *reinterpret_cast<floatx4*>(out + at) = y;
  };
#pragma unroll
  for (int m = 0; m < kMine; ++m) {
    const int q = KG * m + kg;
    int f;
    const long long at = at_of(q, &f);
    if (at >= 0) put(q, at, sums[m], rv[m]);
  }
}

template <int WS, int NI, int KG>
void launch_cfg(const PatchArgs& b, int fblocks, hipStream_t s) {
  auto kern = conv3x3_split_kernel<WS, NI, KG>;
  static const bool attr = [&] {
    NNCV_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, SplitCfg<WS>::smem));
    return true;
  }();
  (void)attr;
  const dim3 grid((b.tiles + kXcdsP - 1) / kXcdsP * kXcdsP, fblocks);
  launch_kernel(kern, grid, dim3(split_threads(WS, KG)), SplitCfg<WS>::smem, s, b.in, b.tiles, b.tiles_y, b.TN, b.TH, b.N, b.H, b.W, b.C,
                b.rw_log, b.xcd_by_filter && fblocks % kXcdsP == 0, b.in_bytes, b.txw, b);
}

// WS = 1: eight waves unless a CU gets a second workgroup beside its first (LDS has room for two): there are more of them than the 32
// CUs of an XCD.  Four -> eight waves, us: one a CU 15.3 -> 14.8 (128 -> 128 channels, 29x39, 6 images), 17.6 -> 16.0 (256 -> 256,
// 15x20, 6), 10.4 -> 9.0 (128 -> 128, 16x27, 6); two a CU 22.7 -> 25.2 (128 -> 64, 35x57, 9), 32.5 -> 35.6 (224 -> 152, 14x19, 17: 33
// on an XCD).  WS = 2 leaves room for one only: eight, 29.1 -> 27.8 (64 -> 64, 56x56, 16).  WS = 4 comes with many workgroups, two a
// CU: four, 36.3 -> 42.9 (32 -> 352, 53x47, 8).
template <int NI>
void launch_ws1(const PatchArgs& b, int fblocks, hipStream_t s) {
  const bool by_filter = b.xcd_by_filter && fblocks % kXcdsP == 0;
  const long long on_xcd = by_filter ? (long long)b.tiles * (fblocks / kXcdsP) : (long long)((b.tiles + kXcdsP - 1) / kXcdsP) * fblocks;
  if (on_xcd > 32) launch_cfg<1, NI, 2>(b, fblocks, s);
  else launch_cfg<1, NI, 4>(b, fblocks, s);
}

// an XCD takes the filters of its workgroups into its L2, where they are more than half of it
bool flat_by_filter(int C, int F) { return (F / 32) % kXcdsP == 0 && weight_frag3x3_bytes(kF32, F, C) > 2u << 20; }

// LDS that the patch of 32 consecutive pixels can need: the rows from its first to its last, one for every image that ends between, two of halo.
long long flat_bytes(int H, int W) { return ((W + 30) / W + (30ll + H * W) / (H * W) + 3) * ((W + 2ll) * kCell + kRowSpare); }

}  // namespace

// Tiles of 32 consecutive pixels where every workgroup has a CU to itself; us, back to back, to within 5 % on 20 layers of 128 to 512
// channels, or 0.  Half the products of a 64-slot tile a workgroup and none for slots without a pixel: 6x8x10x512 -> 512 24.5 -> 17,
// 55x3x3 25 -> 18.5, 4x15x17x256 -> 256 13 -> 11.4; with more workgroups than CUs a second turn takes as long as the first
// (3x14x14x384, 36 workgroups on an XCD, 24).  Every layer of this file that it covers takes it: 50 layers of 192 and 256 channels, which half blocks of a
// 64-slot tile take 10.5 to 13.4 us for, 8.1 to 11.1.  Layers of fewer channels are conv_direct.hip's at all of these sizes (237 000 of them, by the models).
double conv3x3_split_flat_us(int N, int H, int W, int C, int F) {
  if (C < 192 || C % 64 != 0 || F % 64 != 0 || flat_bytes(H, W) > kFlatCells[1] * kCell) return 0;
  const long long tiles = ((long long)N * H * W + 31) / 32, fblocks = F / 32;
  const bool by_filter = flat_by_filter(C, F);
  const long long on_xcd = by_filter ? tiles * (fblocks / kXcdsP) : (tiles + kXcdsP - 1) / kXcdsP * fblocks;
  if (on_xcd > 32) return 0;
  return 5.3 + 9 * C / 32 * (0.056 + 0.026 * (double)(tiles * fblocks) / 256);
}

void launch_conv3x3_split_flat(const PatchArgs& a, double flops, double bytes, hipStream_t s) {
  ProfScope prof("conv3x3_split<f32,flat>", flops, bytes, s);
  PatchArgs b = a;
  b.tiles = (a.N * a.H * a.W + 31) / 32;
  b.xcd_by_filter = flat_by_filter(a.C, a.F);
  b.inv_ph = 1.0f / (a.H + 1);
  b.inv_thw = 1.0f / (a.H * a.W);
  b.inv_w = 1.0f / a.W;
  if (flat_bytes(a.H, a.W) <= kFlatCells[0] * kCell) launch_cfg<0, 1, 8>(b, a.F / 32, s);
  else launch_cfg<-1, 1, 8>(b, a.F / 32, s);
}

void launch_conv3x3_split(const PatchArgs& a, int ws, bool half, const char* tag, double flops, double bytes, hipStream_t s) {
  ProfScope prof(tag, flops, bytes, s);
  const int halves = (a.F + 31) / 32, blocks = (a.F + 63) / 64;
  if (ws == 4) launch_cfg<4, 1, 1>(a, halves, s);
  else if (ws == 2) launch_cfg<2, 2, 2>(a, blocks, s);
  else if (half) launch_ws1<1>(a, halves, s);
  else launch_ws1<2>(a, blocks, s);
}

}  // namespace nncv_hip
