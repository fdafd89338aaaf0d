#include "model.hpp"

#include "arena_plan.hpp"

#include <cstring>

namespace nncv_hip {

static int env_algo3x3() {
  const char* e = getenv("NNCV_HIP_CONV3X3");
  if (!e) return kAlgoAuto;
  if (!strcmp(e, "winograd")) return kAlgoWinograd;
  if (!strcmp(e, "igemm")) return kAlgoIgemm;
  return kAlgoAuto;
}

static int round_up(int v, int m) { return (v + m - 1) / m * m; }

int ConvLayer::pick_algo(const Desc& d) {
  const int ce = d.dt == kF16 ? 8 : 4;
  const bool wino_ok = !d.stem && d.relu <= kActRelu && d.R == 3 && d.S == 3 && d.stride == 1 && d.C % ce == 0 && d.F % 4 == 0;
  int algo = d.algo;
  if (algo == kAlgoAuto) algo = env_algo3x3();
  // default: the direct form for both types.  In fp16 F(4,3) costs about 10x the rounding error;
  // in fp32 it is exact enough, but its three extra passes over 2.25x larger tensors cost more
  // than the 2.25x fewer multiplies save at every ResNet-18 size measured (batch 1..32).
  if (algo == kAlgoAuto) algo = kAlgoIgemm;
  if (algo == kAlgoWinograd && !wino_ok) algo = kAlgoIgemm;
  // F(4x4,3x3) with half-precision V, U and M loses about ten times the direct form's rounding error per
  // layer (2.5-3e-3 relative L2, up to 3e-2 on some shapes): outside the 1e-2 / identical-top-1 bar this
  // library holds fp16 results to.  A request for it is therefore served by the direct form, and says so
  // once.  (The four stages stay available as fp16 operators, nncv_hip_wino43_*.)
  if (algo == kAlgoWinograd && d.dt == kF16) {
    static bool told = false;
    if (!told) {
      fprintf(stderr, "[ Warn ] nncv_hip: fp16 Winograd F(4x4,3x3) does not hold the fp16 accuracy bar; 3x3 layers use the direct form\n");
      told = true;
    }
    algo = kAlgoIgemm;
  }
  return algo;
}

ConvLayer::Sizes ConvLayer::sizes(const Desc& d, int algo, bool bn) {
  const size_t es = dtype_size(d.dt);
  const int Cp = round_up(d.C, d.dt == kF16 ? 8 : 4), Fp = round_up(d.F, 4), RS = d.R * d.S;
  Sizes z{};
  if (d.stem) {
    z.wt = (size_t)d.F * 224 * es;
    if (d.F == 64) z.wstrip = d.dt == kF16 ? stem_weight_strip_bytes() : stem_weight_strip_split_bytes();
    z.wflat = weight_flat_bytes(d.dt, d.F, 7, 32);
  } else if (algo == kAlgoWinograd) {
    z.U = (size_t)36 * d.F * d.C * es;
  } else {
    z.wt = (size_t)Fp * RS * Cp * es;
    if (d.shortcut || conv_direct_serves(d.dt, Fp, RS, Cp)) z.wflat = weight_flat_bytes(d.dt, Fp, RS, Cp);
    if (d.R == 3 && d.S == 3 && (d.stride == 1 || (d.stride == 2 && d.dt == kF16)) && d.pad == 1 && d.C % (128 / (int)es) == 0) {
      z.wfrag = weight_frag3x3_bytes(d.dt, d.F, d.C);
      if (d.dt == kF16 && d.stride == 1 && d.C % 64 == 0 && d.F % 32 == 0) z.wfrag32 = weight_frag32_bytes(d.F, d.C);
    } else if (conv_ring_point_serves(d.dt, d.F, RS, d.C, d.stride, d.pad)) {
      z.wfrag = weight_frag1x1_bytes(d.F, d.C);
    }
  }
  if (bn) z.scale = (size_t)Fp * 4;
  return z;
}

size_t ConvLayer::device_bytes(const Desc& d, bool bn) {
  const Sizes z = sizes(d, pick_algo(d), bn);
  size_t total = 0;
  for (const size_t b : {z.wt, z.wflat, z.wfrag, z.wfrag32, z.U, z.wstrip, z.scale, z.scale}) total += align256(b);
  return total;
}

ConvLayer::ConvLayer(const Desc& d, const void* w, const void* gamma, const void* beta, const void* mean, const void* var,
                     hipStream_t s)
    : d_(d) {
  NNCV_REQUIRE(d.dt == kF32 || d.dt == kF16, "conv: dtype must be f32 or f16");
  NNCV_REQUIRE(d.C > 0 && d.F > 0 && d.R > 0 && d.S > 0 && d.stride > 0 && d.pad >= 0, "conv: bad geometry");
  NNCV_REQUIRE(d.relu >= kActNone && d.relu <= kActSigmoid, "conv: unknown activation");
  NNCV_REQUIRE(!d.stem || (d.C == 3 && d.R == 7 && d.S == 7 && d.stride == 2 && d.pad == 3), "stem: must be 7x7 s2 p3 over 3 channels");
  NNCV_REQUIRE(!d.stem || d.F % 4 == 0, "stem: F must be a multiple of 4");
  NNCV_REQUIRE(!gamma || (beta && mean && var), "conv: BN needs gamma, beta, mean and var");
  algo_ = pick_algo(d);
  const Sizes z = sizes(d, algo_, gamma != nullptr);
  wt_.reset(z.wt, d.pool);
  wflat_.reset(z.wflat, d.pool);
  wfrag_.reset(z.wfrag, d.pool);
  wfrag32_.reset(z.wfrag32, d.pool);
  U_.reset(z.U, d.pool);
  wstrip_.reset(z.wstrip, d.pool);
  scale_.reset(z.scale, d.pool);
  shift_.reset(z.scale, d.pool);

  const int Cp = round_up(d.C, d.dt == kF16 ? 8 : 4), Fp = round_up(d.F, 4);
  if (d.stem) {
    launch_stem_weight(w, d.dt, wt_.get(), d.dt, d.F, s);
    launch_weight_flat_rows(wt_.get(), wflat_.get(), d.dt, d.F, 224, s);
    if (z.wstrip) (d.dt == kF16 ? launch_stem_weight_strip : launch_stem_weight_strip_split)(w, wstrip_.get(), s);
  } else if (algo_ == kAlgoWinograd) {
    launch_wino43_filter(w, d.dt, U_.get(), d.dt, d.F, d.C, s);
  } else {
    if (Fp > d.F) NNCV_HIP_CHECK(hipMemsetAsync(wt_.get(), 0, wt_.bytes(), s));  // padding filters; padding channels are written
    launch_weight_frsc(w, d.dt, wt_.get(), d.dt, d.F, d.C, d.R, d.S, Cp, s);
    if (z.wflat) launch_weight_flat(w, wflat_.get(), d.dt, d.F, d.C, d.R * d.S, Cp, s);
    if (z.wfrag && d.R == 1) launch_weight_frag1x1(w, d.dt, wfrag_.get(), d.dt, d.F, d.C, s);
    else if (z.wfrag) launch_weight_frag3x3(w, d.dt, wfrag_.get(), d.dt, d.F, d.C, s);
    if (z.wfrag32) launch_weight_frag32(w, d.dt, wfrag32_.get(), d.F, d.C, s);
  }
  if (gamma) {
    launch_fill_f32(scale_.as<float>(), 0.0f, Fp, s);
    launch_fill_f32(shift_.as<float>(), 0.0f, Fp, s);
    launch_bn_fold(gamma, beta, mean, var, d.dt, scale_.as<float>(), shift_.as<float>(), d.F, s);
  }
}

size_t ConvLayer::workspace_bytes(int N, int H, int W, bool strided) const {
  const size_t es = dtype_size(d_.dt);
  const int ce = d_.dt == kF16 ? 8 : 4;
  const int OH = out_h(H), OW = out_w(W);
  size_t b = 0;
  if (d_.stem) b += align256((size_t)N * (H + 6) * ((W + 9) / 2) * 8 * es);
  if (algo_ == kAlgoWinograd) {
    const size_t tiles = (size_t)N * ((OH + 3) / 4) * ((OW + 3) / 4);
    b += align256(36 * tiles * d_.C * es) + align256(36 * tiles * d_.F * es);
  }
  // strided (operator-level) form of the igemm path stages NHWC copies of input and output
  if (strided && !d_.stem && algo_ == kAlgoIgemm)
    b += align256((size_t)N * H * W * round_up(d_.C, ce) * es) + 2 * align256((size_t)N * OH * OW * round_up(d_.F, 4) * es);
  return b;
}

void ConvLayer::forward(const void* in, int N, int H, int W, const void* residual, void* out, void* ws, hipStream_t s) const {
  const int OH = out_h(H), OW = out_w(W);
  NNCV_REQUIRE(N > 0 && OH > 0 && OW > 0, "conv: empty tensor");
  const size_t es = dtype_size(d_.dt);
  char* wsp = static_cast<char*>(ws);
  if (d_.stem) {
    const int HP = H + 6, WP = (W + 9) / 2;
    launch_stem_pack(in, d_.dt, wsp, d_.dt, N, H, W, s);
    IgemmArgs a{};
    a.in = wsp; a.wt = wt_.get(); a.wt_flat = wflat_.get(); a.out = out;
    a.scale = scale_.as<float>(); a.shift = shift_.as<float>(); a.residual = residual;
    // a filter row is 4 consecutive pixel pairs = 32 contiguous elements: one K step
    a.N = N; a.H = HP; a.W = WP; a.C = 32; a.pix_stride = 8; a.F = d_.F; a.R = 7; a.S = 1; a.OH = OH; a.OW = OW;
    a.stride_h = 2; a.stride_w = 1; a.pad_h = 0; a.pad_w = 0;
    a.relu = d_.relu; a.ldo = d_.F; a.batch = 1;
    a.alg_flops = 2.0 * N * OH * OW * d_.F * 147.0;  // the 7x7x3 filter, not its padded 7x8x4 packing
    launch_igemm(a, d_.dt, d_.dt, s);
    return;
  }
  if (algo_ == kAlgoWinograd) {
    forward_strided(in, strides_of(kNHWC, d_.C, H, W), N, H, W, residual, out, strides_of(kNHWC, d_.F, OH, OW), false, ws, s);
    return;
  }
  NNCV_REQUIRE(d_.C % (16 / (int)es) == 0 && d_.F % 4 == 0, "conv: NHWC igemm needs C %% chunk == 0 and F %% 4 == 0");
  IgemmArgs a{};
  a.in = in; a.wt = wt_.get(); a.wt_frag = wfrag_.get(); a.wt_frag32 = wfrag32_.get(); a.wt_flat = wflat_.get(); a.out = out;
  a.scale = scale_.as<float>(); a.shift = shift_.as<float>(); a.residual = residual;
  a.N = N; a.H = H; a.W = W; a.C = d_.C; a.F = d_.F; a.R = d_.R; a.S = d_.S; a.OH = OH; a.OW = OW;
  a.stride_h = a.stride_w = d_.stride; a.pad_h = a.pad_w = d_.pad;
  a.relu = d_.relu; a.ldo = d_.F; a.batch = 1;
  launch_igemm(a, d_.dt, d_.dt, s);
}

bool ConvLayer::forward_stem_pool(const void* in, int N, int H, int W, void* pooled_out, hipStream_t s) const {
  if (!d_.stem || d_.relu != kActRelu || !stem_pool_applicable(d_.dt, N, H, W, d_.F)) return false;
  (d_.dt == kF16 ? launch_stem_pool : launch_stem_pool_split)(in, wstrip_.get(), scale_.as<float>(), shift_.as<float>(), pooled_out, N, H, W, s);
  return true;
}

bool ConvLayer::forward_block(const ConvLayer& second, const void* in, int N, int H, int W, void* out, hipStream_t s) const {
  auto fits = [](const ConvLayer& c) {
    const Desc& d = c.d_;
    return !d.stem && c.algo_ == kAlgoIgemm && d.dt == kF16 && d.C == 64 && d.F == 64 && d.R == 3 && d.S == 3 && d.stride == 1 && d.pad == 1 && d.relu == kActRelu &&
           c.wfrag32_.get() && c.scale_.get();
  };
  static const bool off = getenv("NNCV_HIP_NO_BASIC_BLOCK") != nullptr;
  if (off || !fits(*this) || !fits(second)) return false;
  // Against the two launches of conv3x3_f16.hip, a whole ResNet-18 pass in microseconds, theirs first:
  //  * 256 images, rows of W: 24 319 against 313, 28 366 against 351, 32 421 against 406, 33 500 against 477, 40 592 against 559, 43 742
  //    against 707, 48 887 against 837, 56 1032 against 976, 64 1440 against 1223;
  //    64 images: 65 498 against 464, 72 542 against 487, 80 633 against 568, 90 872 against 809; 16: 160 639 against 568; 8: 256 801 against 736.
  //  * Steps for each CU (replayed graphs): a strip pays five beyond its own.  Three and four rows a step (W <= 42): 1.5 of them (64 images of
  //    96x96) 161 against 158, 2 (64 of 128x128) 187 against 185, 2.6 (48 of 160x160) 223 against 214, and few lose (2 of 128x128 108 against
  //    114); two is the line.  Two rows: W = 56 0.1 (1 image) 94 against 99, 1.8 (16) 161 against 159, 5.3 (48) 297 against 286; four is the
  //    line, and up to 36 images of 224x224 keep the launches they had, though less than all of them need to: 2.2 (20) 195 against 187, 2.6 (24) 199 against 190,
  //    3.5 (32) 207 against 200, 3.9 (36) 225 against 218.  W > 56, where two rows are nearly the 128 slots and the stream
  //    form's tile of a row is two thirds full: 4 images of 256x256 (0.5) 129 against 129, 8 (1) 151 against 141, 16 200 against 179, 8
  //    of 240x240 (0.9) 139 against 138; one is the line, for rows in columns too: 2 images of 320x320 (0.4) 126 against 128, 4 (0.8) 139 against 139, 8 (1.7)
  //    181 against 172.
  //  * Three and more passes in flight, each workgroup of this kernel with a CU to itself: 64 images of 160x160 (3.5) 670 against 683 for
  //    four passes, 48 of 224x224 (5.3) 642 against 653 for three, 32 (3.5) 448 against 455, for four 585 against 581, 128 of 160x160 (7) 1153 against 1131, 64 of 224x224 (7) 1075 against
  //    1044, 64 of 256x256 (8) 1313 against 1176; 8 of 320x320 (1.7) 411 against 418, 32 (6.8) 1144 against 1088; six is the line.
  const long long steps = basic_block_steps(N, H, W);
  if (!steps || steps < 256 * (overlap_hint() >= 3 ? 6 : W <= 42 ? 2 : W <= 56 ? 4 : 1)) return false;
  launch_basic_block(BasicBlockArgs{in, out, wfrag32_.get(), second.wfrag32_.get(), scale_.as<float>(), shift_.as<float>(), second.scale_.as<float>(), second.shift_.as<float>(), N, H, W}, s);
  return true;
}

bool ConvLayer::fuse_shortcut(const ConvLayer& ds, hipStream_t s) {
  const Desc& q = ds.d_;
  const size_t es = dtype_size(d_.dt);
  const int ce = d_.dt == kF16 ? 8 : 4;
  if (d_.stem || algo_ != kAlgoIgemm || ds.algo_ != kAlgoIgemm || q.dt != d_.dt || q.C != d_.C || q.stride != d_.stride ||
      d_.R != 3 || d_.S != 3 || d_.pad != 1 || q.R != 1 || q.S != 1 || q.pad != 0 || d_.F % 128 != 0 || q.F % 8 != 0 ||
      d_.C % ce != 0 || !scale_.get() || !ds.scale_.get())
    return false;
  const size_t row = (size_t)9 * d_.C * es;
  wt_cat_.reset((size_t)(d_.F + q.F) * row, d_.pool);
  NNCV_HIP_CHECK(hipMemsetAsync(wt_cat_.get(), 0, wt_cat_.bytes(), s));
  NNCV_HIP_CHECK(hipMemcpyAsync(wt_cat_.get(), wt_.get(), (size_t)d_.F * row, hipMemcpyDeviceToDevice, s));
  // the shortcut's [F][C] rows become the centre tap (r = s = 1) of otherwise zero 3x3 filters
  NNCV_HIP_CHECK(hipMemcpy2DAsync(wt_cat_.as<char>() + (size_t)d_.F * row + (size_t)4 * d_.C * es, row, ds.wt_.get(),
                                  (size_t)d_.C * es, (size_t)d_.C * es, q.F, hipMemcpyDeviceToDevice, s));
  scale_cat_.reset((size_t)(d_.F + q.F) * 4, d_.pool);
  shift_cat_.reset((size_t)(d_.F + q.F) * 4, d_.pool);
  NNCV_HIP_CHECK(hipMemcpyAsync(scale_cat_.get(), scale_.get(), (size_t)d_.F * 4, hipMemcpyDeviceToDevice, s));
  NNCV_HIP_CHECK(hipMemcpyAsync(shift_cat_.get(), shift_.get(), (size_t)d_.F * 4, hipMemcpyDeviceToDevice, s));
  NNCV_HIP_CHECK(hipMemcpyAsync(scale_cat_.as<float>() + d_.F, ds.scale_.get(), (size_t)q.F * 4, hipMemcpyDeviceToDevice, s));
  NNCV_HIP_CHECK(hipMemcpyAsync(shift_cat_.as<float>() + d_.F, ds.shift_.get(), (size_t)q.F * 4, hipMemcpyDeviceToDevice, s));
  if (wfrag_.get() && d_.C % (128 / (int)es) == 0) {
    aux_wfrag_.reset((size_t)((q.F + 63) / 64) * 64 * d_.C * es, d_.pool);
    launch_weight_frag1x1(ds.wt_.get(), d_.dt, aux_wfrag_.get(), d_.dt, q.F, d_.C, s);  // [F][1][1][C] rows
  }
  aux_wflat_ = ds.wflat_.get();
  aux_F_ = q.F;
  aux_relu_ = q.relu;
  aux_flops_per_pixel_ = 2.0 * q.F * q.C;
  return true;
}

void ConvLayer::forward_with_shortcut(const void* in, int N, int H, int W, void* out, void* shortcut_out, void* ws,
                                      hipStream_t s) const {
  NNCV_REQUIRE(aux_F_ > 0, "conv: no fused shortcut");
  const int OH = out_h(H), OW = out_w(W);
  NNCV_REQUIRE(N > 0 && OH > 0 && OW > 0, "conv: empty tensor");
  IgemmArgs a{};
  a.in = in; a.wt = wt_cat_.get(); a.wt_frag = wfrag_.get(); a.aux_wt_frag = aux_wfrag_.get(); a.out = out;
  a.wt_flat = wflat_.get(); a.aux_wt_flat = aux_wflat_;
  a.scale = scale_cat_.as<float>(); a.shift = shift_cat_.as<float>();
  a.N = N; a.H = H; a.W = W; a.C = d_.C; a.F = d_.F + aux_F_; a.R = 3; a.S = 3; a.OH = OH; a.OW = OW;
  a.stride_h = a.stride_w = d_.stride; a.pad_h = a.pad_w = 1;
  a.relu = d_.relu; a.ldo = d_.F; a.batch = 1;
  a.aux_f0 = d_.F; a.aux_tap = 4; a.aux_relu = aux_relu_; a.aux_ldo = aux_F_; a.aux_out = shortcut_out;
  a.alg_flops = (2.0 * d_.F * 9.0 * d_.C + aux_flops_per_pixel_) * N * OH * OW;
  launch_igemm(a, d_.dt, d_.dt, s);
}

void ConvLayer::forward_strided(const void* in, Strides4 in_st, int N, int H, int W, const void* residual, void* out,
                                Strides4 out_st, bool accumulate, void* ws, hipStream_t s) const {
  NNCV_REQUIRE(!d_.stem, "conv: the stem has no strided form");
  const int OH = out_h(H), OW = out_w(W);
  NNCV_REQUIRE(N > 0 && OH > 0 && OW > 0, "conv: empty tensor");
  const size_t es = dtype_size(d_.dt);
  const int ce = d_.dt == kF16 ? 8 : 4;
  char* wsp = static_cast<char*>(ws);
  if (algo_ == kAlgoWinograd) {
    const int TH = (OH + 3) / 4, TW = (OW + 3) / 4;
    const long long tiles = (long long)N * TH * TW;
    void* V = wsp;
    void* M = wsp + align256((size_t)36 * tiles * d_.C * es);
    launch_wino43_input(in, d_.dt, in_st, V, d_.dt, N, d_.C, H, W, d_.pad, s);
    IgemmArgs a{};
    a.in = V; a.wt = U_.get(); a.out = M;
    NNCV_REQUIRE(tiles < (1ll << 31), "conv: too many Winograd tiles");
    a.N = (int)tiles; a.H = 1; a.W = 1; a.C = d_.C; a.F = d_.F; a.R = 1; a.S = 1; a.OH = 1; a.OW = 1;
    a.stride_h = a.stride_w = 1; a.ldo = d_.F; a.batch = 36;
    a.in_bs = tiles * d_.C; a.wt_bs = (long long)d_.F * d_.C; a.out_bs = tiles * d_.F;
    launch_igemm(a, d_.dt, d_.dt, s);
    WinoOutArgs o{};
    o.M = M; o.out = out; o.residual = residual; o.scale = scale_.as<float>(); o.shift = shift_.as<float>();
    o.st = out_st; o.N = N; o.F = d_.F; o.OH = OH; o.OW = OW; o.relu = d_.relu; o.accumulate = accumulate;
    launch_wino43_output(o, d_.dt, d_.dt, s);
    return;
  }
  // implicit GEMM through NHWC staging copies (operator-level forms only; the network itself is
  // NHWC end to end and never comes here)
  const int Cp = round_up(d_.C, ce), Fp = round_up(d_.F, 4);
  const size_t in_b = align256((size_t)N * H * W * Cp * es), out_b = align256((size_t)N * OH * OW * Fp * es);
  void* xin = wsp;
  void* yout = wsp + in_b;
  void* rin = residual ? wsp + in_b + out_b : nullptr;
  launch_relayout(in, d_.dt, in_st, xin, d_.dt, strides_of(kNHWC, Cp, H, W), N, d_.C, Cp, H, W, false, s);
  if (residual)
    launch_relayout(residual, d_.dt, out_st, rin, d_.dt, strides_of(kNHWC, Fp, OH, OW), N, d_.F, Fp, OH, OW, false, s);
  IgemmArgs a{};
  a.in = xin; a.wt = wt_.get(); a.wt_flat = wflat_.get(); a.out = yout; a.residual = rin;
  if (Cp == d_.C && Fp == d_.F) { a.wt_frag = wfrag_.get(); a.wt_frag32 = wfrag32_.get(); }  // the staged tensors are the layer's own
  a.scale = scale_.as<float>(); a.shift = shift_.as<float>();
  a.N = N; a.H = H; a.W = W; a.C = Cp; a.F = Fp; a.R = d_.R; a.S = d_.S; a.OH = OH; a.OW = OW;
  a.stride_h = a.stride_w = d_.stride; a.pad_h = a.pad_w = d_.pad;
  a.relu = d_.relu; a.ldo = Fp; a.batch = 1;
  NNCV_REQUIRE(!(accumulate && (d_.relu || residual)), "conv: accumulate form has no epilogue");
  launch_igemm(a, d_.dt, d_.dt, s);
  // out (+)= y : y is NHWC with Fp channels; only the first F are copied
  launch_relayout(yout, d_.dt, strides_of(kNHWC, Fp, OH, OW), out, d_.dt, out_st, N, d_.F, d_.F, OH, OW, accumulate, s);
}

// ---------------------------------------------------------------------------------------------

ResNet18::ResNet18(const void* params, long long n_elems, int dt, int algo3x3, hipStream_t s, DevicePool pool)
    : dt_(dt), pool_(std::move(pool)) {
  pool_.rewind();
  NNCV_REQUIRE(n_elems == kResNet18Elems,
               "ResNet-18 params: expected 11699112 elements in the canonical model.bin order, got " + std::to_string(n_elems));
  const size_t es = dtype_size(dt);
  const char* p = static_cast<const char*>(params);
  auto take = [&](long long n) { const void* r = p; p += n * es; return r; };
  auto make = [&](int C, int F, int R, int stride, int pad, bool relu, bool stem) {
    ConvLayer::Desc d;
    d.dt = dt; d.C = C; d.F = F; d.R = d.S = R; d.stride = stride; d.pad = pad; d.relu = relu; d.stem = stem;
    d.algo = (R == 3 && stride == 1) ? algo3x3 : kAlgoIgemm;
    d.shortcut = R == 1;
    d.pool = &pool_;
    const void* w = take((long long)F * C * R * R);
    const void* g = take(F); const void* b = take(F); const void* m = take(F); const void* v = take(F);
    return std::make_unique<ConvLayer>(d, w, g, b, m, v, s);
  };
  stem_ = make(3, 64, 7, 2, 3, true, true);
  int cin = 64;
  const int widths[4] = {64, 128, 256, 512};
  for (int L = 0; L < 4; ++L)
    for (int blk = 0; blk < 2; ++blk) {
      const int F = widths[L], stride = (L > 0 && blk == 0) ? 2 : 1;
      Block b;
      b.c1 = make(cin, F, 3, stride, 1, true, false);
      b.c2 = make(F, F, 3, 1, 1, true, false);  // ReLU after the residual add
      if (stride != 1 || cin != F) {
        b.ds = make(cin, F, 1, stride, 0, false, false);
        static const bool no_fuse = getenv("NNCV_HIP_NO_SHORTCUT_FUSION") != nullptr;
        if (!no_fuse) b.c1->fuse_shortcut(*b.ds, s);
      }
      blocks_.push_back(std::move(b));
      cin = F;
    }
  const void* fw = take(1000 * 512);
  const void* fb = take(1000);
  fc_w_.reset((size_t)1000 * 512 * es, &pool_);
  NNCV_HIP_CHECK(hipMemcpyAsync(fc_w_.get(), fw, fc_w_.bytes(), hipMemcpyDeviceToDevice, s));
  fc_b_.reset(1000 * 4, &pool_);
  launch_cast(fb, dt, fc_b_.get(), kF32, 1000, s);
  NNCV_REQUIRE((p - static_cast<const char*>(params)) == (long long)(kResNet18Elems * es), "ResNet-18 params: table walk mismatch");
}

const ResNet18::Plan& ResNet18::plan_of(int N, int H, int W) const {
  const int linger = (overlap_hint() >= 3 && N >= 16 && !arena_linger_forced()) ? 0 : arena_linger();  // see overlap_hint
  for (const Plan& p : plans_)
    if (p.N == N && p.H == H && p.W == W && p.linger == linger) return p;
  NNCV_REQUIRE(blocks_.size() == 8, "ResNet-18 has eight BasicBlocks");
  const ConvLayer& stem = *stem_;
  Plan p{};
  p.N = N; p.H = H; p.W = W; p.linger = linger;
  const size_t es = dtype_size(dt_);
  p.h1 = stem.out_h(H); p.w1 = stem.out_w(W);
  p.h2 = (p.h1 + 2 - 3) / 2 + 1; p.w2 = (p.w1 + 2 - 3) / 2 + 1;
  std::vector<TensorLife> t;
  auto add = [&](int first, int last, size_t bytes) { t.push_back(TensorLife{first, last, bytes, 0}); return (int)t.size() - 1; };
  // the fused stem kernel writes the pooled tensor directly: no stem output, no packed image
  const bool fused_stem = stem.desc().relu == kActRelu && stem_pool_applicable(dt_, N, H, W, stem.desc().F);
  const int i_stem = add(0, 1, fused_stem ? 0 : (size_t)N * p.h1 * p.w1 * 64 * es);
  size_t cws = fused_stem ? 0 : stem.workspace_bytes(N, H, W);
  int h = p.h2, w = p.w2, ch = 64;
  int ix[9], iy1[8], iidn[8];
  ix[0] = add(1, 0, 0);  // last use filled in below
  const int nb = (int)blocks_.size();
  for (int k = 0; k < nb; ++k) {
    const ConvLayer &c1 = *blocks_[k].c1, &c2 = *blocks_[k].c2;
    const ConvLayer* ds = blocks_[k].ds.get();
    const int o = 2 + 3 * k;
    const int oh = c1.out_h(h), ow = c1.out_w(w), f = c2.desc().F;
    cws = std::max(cws, c1.workspace_bytes(N, h, w));
    cws = std::max(cws, c2.workspace_bytes(N, oh, ow));
    if (ds) cws = std::max(cws, ds->workspace_bytes(N, h, w));
    t[ix[k]].bytes = (size_t)N * h * w * ch * es;
    t[ix[k]].last_op = ds ? o + 1 : o + 2;  // identity shortcuts are read by conv2
    iy1[k] = add(o, o + 2, (size_t)N * oh * ow * f * es);
    iidn[k] = ds ? add(o, o + 2, (size_t)N * oh * ow * f * es) : -1;
    ix[k + 1] = add(o + 2, o + 3, 0);
    h = oh; w = ow; ch = f;
  }
  p.h_out = h; p.w_out = w;
  t[ix[nb]].bytes = (size_t)N * h * w * ch * es;
  t[ix[nb]].last_op = 26;
  const int i_pooled = add(26, 27, (size_t)N * 512 * es);
  const int i_cws = add(0, 27, cws);
  for (auto& e : t) e.last_op = std::min(27, e.last_op + linger);
  p.total = plan_offsets(t, 256) + 4096;
  p.stem_out = t[i_stem].offset; p.pooled = t[i_pooled].offset; p.cws = t[i_cws].offset;
  for (int k = 0; k <= nb; ++k) p.x[k] = t[ix[k]].offset;
  for (int k = 0; k < nb; ++k) { p.y1[k] = t[iy1[k]].offset; p.idn[k] = iidn[k] >= 0 ? t[iidn[k]].offset : 0; }
  if (plans_.size() >= 8) plans_.erase(plans_.begin());
  plans_.push_back(p);
  return plans_.back();
}

size_t ResNet18::workspace_bytes(int N, int H, int W) const { return plan_of(N, H, W).total; }

void ResNet18::forward_body(const void* src, int N, int H, int W, void* ws, hipStream_t s, int tap_stage, void* tap) const {
  NNCV_REQUIRE(N > 0 && H >= 32 && W >= 32, "ResNet-18: input must be at least 32x32");
  const Plan& p = plan_of(N, H, W);
  char* base = static_cast<char*>(ws);
  char* stem_out = base + p.stem_out;
  char* cws = base + p.cws;
  char* x0 = base + p.x[0];

  // stem: conv7x7 s2 + BN + ReLU (Res18.mlir:118-142), then maxpool 3x3 s2 (:144-151)
  if (!stem_->forward_stem_pool(src, N, H, W, x0, s)) {
    stem_->forward(src, N, H, W, nullptr, stem_out, cws, s);
    launch_maxpool3x3s2_nhwc(stem_out, x0, dt_, N, p.h1, p.w1, 64, s);
  }
  int h = p.h2, w = p.w2, nblk = 0, ch = 64;
  const size_t es = dtype_size(dt_);
  if (tap_stage == 0) NNCV_HIP_CHECK(hipMemcpyAsync(tap, x0, (size_t)N * h * w * 64 * es, hipMemcpyDeviceToDevice, s));
  for (const Block& b : blocks_) {
    // BasicBlock (Res18.mlir:152-203, :255-320): y = relu(bn2(conv2(relu(bn1(conv1(x))))) + shortcut(x))
    char* x = base + p.x[nblk];
    char* y1 = base + p.y1[nblk];
    char* idn = base + p.idn[nblk];
    char* y2 = base + p.x[nblk + 1];
    const int oh = b.c1->out_h(h), ow = b.c1->out_w(w);
    const void* shortcut = x;
    const bool whole = !b.ds && b.c1->forward_block(*b.c2, x, N, h, w, y2, s);
    if (whole) {
      // y1 is never stored
    } else if (b.ds && b.c1->has_shortcut()) {
      b.c1->forward_with_shortcut(x, N, h, w, y1, idn, cws, s);
      shortcut = idn;
    } else {
      b.c1->forward(x, N, h, w, nullptr, y1, cws, s);
      if (b.ds) {
        b.ds->forward(x, N, h, w, nullptr, idn, cws, s);
        shortcut = idn;
      }
    }
    if (!whole) b.c2->forward(y1, N, oh, ow, shortcut, y2, cws, s);
    h = oh; w = ow;
    ch = b.c2->desc().F;
    ++nblk;
    if (nblk % 2 == 0 && tap_stage == nblk / 2)
      NNCV_HIP_CHECK(hipMemcpyAsync(tap, y2, (size_t)N * h * w * ch * es, hipMemcpyDeviceToDevice, s));
  }
}

void ResNet18::forward_head(int N, int H, int W, void* logits, void* ws, hipStream_t s) const {
  const Plan& p = plan_of(N, H, W);
  char* body_out = static_cast<char*>(ws) + p.x[8];
  char* pooled = static_cast<char*>(ws) + p.pooled;
  const int h = p.h_out, w = p.w_out;
  // head: global average pool (sum, one divide), FC with bias (Res18.mlir:609-628)
  static const bool never_fused = getenv("NNCV_HIP_NO_HEAD_FUSION") != nullptr;
  // see overlap_hint (arena_plan.hpp); at small batches the fused head is a few dozen workgroups and one launch less
  const bool split_head = never_fused || (overlap_hint() >= 3 && N >= 16);
  if (!split_head) {
    launch_avgpool_fc(body_out, fc_w_.get(), fc_b_.as<float>(), static_cast<float*>(logits), dt_, N, h * w, 512, 1000, s);
    return;
  }
  launch_global_avgpool_nhwc(body_out, pooled, dt_, N, h * w, 512, s);
  IgemmArgs a{};
  a.in = pooled; a.wt = fc_w_.get(); a.out = logits; a.shift = fc_b_.as<float>();
  a.N = N; a.H = 1; a.W = 1; a.C = 512; a.F = 1000; a.R = 1; a.S = 1; a.OH = 1; a.OW = 1;
  a.stride_h = a.stride_w = 1; a.ldo = 1000; a.batch = 1;
  launch_igemm(a, dt_, kF32, s);
}

}  // namespace nncv_hip
