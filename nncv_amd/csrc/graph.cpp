#include "graph.hpp"

#include <algorithm>

#include "arena_plan.hpp"

namespace nncv_hip {

namespace {

int round_up(int v, int m) { return (v + m - 1) / m * m; }

// shift[c] = (shift ? shift[c] : 0) + (scale ? scale[c] : 1) * bias[c]:  BN(conv + bias) folded
// into one scale/shift pair, or a plain bias turned into the epilogue's fp32 shift.
template <typename T>
__global__ void fold_bias_kernel(const T* __restrict__ bias, const float* __restrict__ scale, float* __restrict__ shift, int has_shift,
                                 int F) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= F) return;
  const float b = (float)bias[c];
  shift[c] = (has_shift ? shift[c] : 0.0f) + (scale ? scale[c] : 1.0f) * b;
}

const char* kind_name(int k) {
  switch (k) {
    case NNCV_HIP_OP_CONV: return "conv";
    case NNCV_HIP_OP_DWCONV: return "dwconv";
    case NNCV_HIP_OP_MAXPOOL: return "maxpool";
    case NNCV_HIP_OP_GAVGPOOL: return "gavgpool";
    case NNCV_HIP_OP_SCALE: return "scale";
    case NNCV_HIP_OP_ADD: return "add";
    case NNCV_HIP_OP_ACT: return "act";
    case NNCV_HIP_OP_CONCAT: return "concat";
    case NNCV_HIP_OP_UPSAMPLE2X: return "upsample2x";
    case NNCV_HIP_OP_YOLO_DETECT: return "yolo_detect";
    default: return "?";
  }
}

int n_inputs(int kind) {
  switch (kind) {
    case NNCV_HIP_OP_SCALE:
    case NNCV_HIP_OP_ADD: return 2;
    case NNCV_HIP_OP_CONCAT: return 4;
    case NNCV_HIP_OP_YOLO_DETECT: return 3;
    case NNCV_HIP_OP_CONV: return 2;  // second one (residual) optional
    default: return 1;
  }
}

}  // namespace

Graph::Graph(const GraphOp* ops, int n, int in_channels, const void* params, long long n_elems, int dt, hipStream_t s)
    : dt_(dt), c_in_(in_channels), dry_(params == nullptr) {
  NNCV_REQUIRE(dt == kF32 || dt == kF16, "graph: dtype must be 1 (fp32) or 2 (fp16)");
  NNCV_REQUIRE(ops && n > 0 && in_channels > 0, "graph: empty operator list");
  const int vn = dt == kF16 ? 8 : 4;
  const size_t es = dtype_size(dt);
  const char* blob = static_cast<const char*>(params);

  int max_id = 0;
  for (int i = 0; i < n; ++i) max_id = std::max(max_id, ops[i].out);
  NNCV_REQUIRE(max_id >= 1 && max_id <= 4 * n + 4, "graph: tensor ids out of range");
  n_tensors_ = max_id + 1;
  channels_.assign(n_tensors_, 0);
  logical_.assign(n_tensors_, 0);
  last_use_.assign(n_tensors_, -1);
  channels_[0] = round_up(in_channels, vn);
  logical_[0] = in_channels;
  nodes_.resize(n);

  // Two 1x1 convolutions of one tensor, equal but for their filters (cv1 and cv2 of a YOLOv5 C3 block): the second one's
  // parameters lie behind the first one's, so that one launch can compute both where the shape is the LDS ring's (plan_of).
  for (int i = 0; i < n && dt == kF16; ++i) {
    auto point = [&](const GraphOp& o) {
      return o.kind == NNCV_HIP_OP_CONV && o.K == 1 && o.stride == 1 && o.pad == 0 && o.in[0] > 0 && o.in[1] < 0 && o.F > 0 && o.F % vn == 0;
    };
    if (!point(ops[i]) || nodes_[i].joined) continue;
    for (int j = i + 1; j < n; ++j)
      if (point(ops[j]) && ops[j].in[0] == ops[i].in[0] && ops[j].F == ops[i].F && ops[j].act == ops[i].act &&
          (ops[j].gamma < 0) == (ops[i].gamma < 0) && (ops[j].bias < 0) == (ops[i].bias < 0) && !nodes_[j].joined) {
        nodes_[i].joins = j;
        nodes_[j].joined = true;
        break;
      }
  }
  auto joined_by = [&](int i) -> Node* {
    for (int k = 0; nodes_[i].joined && k < i; ++k)
      if (nodes_[k].joins == i) return &nodes_[k];
    return nullptr;
  };
  // an array of filters; without parameters a placeholder, so that the plan is made for the kernels that a graph with them has
  static char nothing;
  auto keep = [&](DeviceBuffer& b, size_t bytes) {
    if (dry_) b.borrow(&nothing, bytes);
    else b.reset(bytes, &pool_);
  };
  // a buffer of node i, with room behind it for the node it joins, or the second half of its joiner's
  auto take = [&](int i, DeviceBuffer Node::*b, size_t bytes) {
    if (const Node* first = dry_ ? nullptr : joined_by(i)) (nodes_[i].*b).borrow((first->*b).as<char>() + bytes, bytes);
    else keep(nodes_[i].*b, bytes * (nodes_[i].joins >= 0 ? 2 : 1));
  };

  auto param = [&](long long off, long long count, const std::string& what) -> const void* {
    NNCV_REQUIRE(off >= 0 && (dry_ || off + count <= n_elems), "graph: " + what + " lies outside the parameter blob");
    return blob + (size_t)off * es;
  };

  std::vector<char> pixel(n_tensors_, 0);  // tensors of one pixel an image
  for (int i = 0; i < n; ++i) {
    const GraphOp& op = ops[i];
    const std::string where = "graph: operator " + std::to_string(i) + " (" + kind_name(op.kind) + "): ";
    Node& nd = nodes_[i];
    nd.op = op;
    NNCV_REQUIRE(op.kind >= NNCV_HIP_OP_CONV && op.kind <= NNCV_HIP_OP_YOLO_DETECT, where + "unknown kind");
    NNCV_REQUIRE(op.kind != NNCV_HIP_OP_YOLO_DETECT || i == n - 1, where + "must be the last operator");
    NNCV_REQUIRE(op.out >= 1 && op.out < n_tensors_ && channels_[op.out] == 0, where + "`out` must be a new tensor id");
    NNCV_REQUIRE(op.act >= kActNone && op.act <= kActSigmoid, where + "unknown activation");
    const int ni = n_inputs(op.kind);
    for (int k = 0; k < 4; ++k) {
      const int t = op.in[k];
      if (k >= ni) {
        NNCV_REQUIRE(t < 0, where + "too many inputs");
        continue;
      }
      const bool optional =
          k > 0 && (op.kind == NNCV_HIP_OP_CONV || op.kind == NNCV_HIP_OP_CONCAT || op.kind == NNCV_HIP_OP_YOLO_DETECT);
      if (t < 0 && optional) continue;
      NNCV_REQUIRE(t >= 0 && t < n_tensors_ && channels_[t] > 0, where + "input is not a tensor defined earlier");
      last_use_[t] = i;
    }
    const int C = channels_[op.in[0]];
    nd.C = C;
    int Cout = C;       // logical channels of the result
    int Cstored = -1;   // stored channels when they differ
    // Only convolutions (which know the real count from their filters), the Detect decode and the
    // network output may read a tensor that is stored with padding channels.
    if (op.kind != NNCV_HIP_OP_CONV && op.kind != NNCV_HIP_OP_YOLO_DETECT)
      for (int k = 0; k < ni; ++k)
        if (op.in[k] >= 0)
          NNCV_REQUIRE(logical_[op.in[k]] == channels_[op.in[k]],
                       where + "channel count of an input must be a multiple of the 16-byte vector");
    switch (op.kind) {
      case NNCV_HIP_OP_CONV: {
        NNCV_REQUIRE(op.F > 0, where + "F must be positive");
        NNCV_REQUIRE(op.K >= 1 && op.K <= 11 && op.stride >= 1 && op.pad >= 0, where + "bad geometry");
        NNCV_REQUIRE(op.in[1] < 0 || logical_[op.in[1]] == op.F, where + "residual has another channel count");
        Cout = op.F;
        Cstored = round_up(op.F, vn);
        const int Cl = logical_[op.in[0]];  // channels the filters really have
        const void* w = param(op.w, (long long)op.F * Cl * op.K * op.K, where + "w");
        take(i, &Node::wt, (size_t)Cstored * op.K * op.K * C * es);
        if (!dry_) {
          if (Cstored > op.F) NNCV_HIP_CHECK(hipMemsetAsync(nd.wt.get(), 0, (size_t)Cstored * op.K * op.K * C * es, s));
          launch_weight_frsc(w, dt, nd.wt.get(), dt, op.F, Cl, op.K, op.K, C, s);
        }
        pixel[op.out] = pixel[op.in[0]];
        // (1x1: not for single pixels, which are never enough; with the filters of both where two are joined, whole blocks of 64 of the first)
        if (!pixel[op.in[0]] && Cl == C && Cstored == op.F && ((nd.joins < 0 && !nd.joined) || op.F % 64 == 0) && conv_ring_point_serves(dt, nd.joins >= 0 || nd.joined ? 2 * op.F : op.F, op.K * op.K, C, op.stride, op.pad)) {
          take(i, &Node::wfrag, weight_frag1x1_bytes(op.F, C));
          if (!dry_) launch_weight_frag1x1(w, dt, nd.wfrag.get(), dt, op.F, C, s);
        }
        if (op.K == 3 && (op.stride == 1 || (op.stride == 2 && dt == kF16)) && op.pad == 1 && Cl == C && Cstored == op.F && C % (128 / (int)es) == 0) {
          keep(nd.wfrag, weight_frag3x3_bytes(dt, op.F, C));
          if (!dry_) launch_weight_frag3x3(w, dt, nd.wfrag.get(), dt, op.F, C, s);
          if (dt == kF16 && op.stride == 1 && C % 64 == 0 && op.F % 32 == 0) {
            keep(nd.wfrag32, weight_frag32_bytes(op.F, C));
            if (!dry_) launch_weight_frag32(w, dt, nd.wfrag32.get(), op.F, C, s);
          }
        }
        break;
      }
      case NNCV_HIP_OP_DWCONV: {
        NNCV_REQUIRE(op.K == 3 || op.K == 5, where + "K must be 3 or 5");
        NNCV_REQUIRE(op.stride >= 1 && op.pad >= 0, where + "bad geometry");
        const void* w = param(op.w, (long long)C * op.K * op.K, where + "w");
        keep(nd.wt, (size_t)C * op.K * op.K * es);
        if (!dry_) launch_weight_dw(w, dt, nd.wt.get(), dt, C, op.K, s);
        break;
      }
      case NNCV_HIP_OP_MAXPOOL:
        NNCV_REQUIRE(op.K >= 1 && op.stride >= 1 && op.pad >= 0 && 2 * op.pad <= op.K, where + "bad geometry");
        break;
      case NNCV_HIP_OP_GAVGPOOL: pixel[op.out] = 1; break;
      case NNCV_HIP_OP_SCALE:
      case NNCV_HIP_OP_ADD:
        NNCV_REQUIRE(channels_[op.in[1]] == C, where + "operands have different channel counts");
        break;
      case NNCV_HIP_OP_CONCAT:
        for (int k = 1; k < 4; ++k)
          if (op.in[k] >= 0) Cout += channels_[op.in[k]];
        break;
      case NNCV_HIP_OP_YOLO_DETECT: {
        NNCV_REQUIRE(op.K >= 1 && op.K <= 4 && op.F >= 5, where + "K anchors (1..4) of F >= 5 values each");
        int levels = 0;
        for (int k = 0; k < 3; ++k)
          if (op.in[k] >= 0) {
            NNCV_REQUIRE(k == levels, where + "levels must be in[0], in[1], ... without gaps");
            NNCV_REQUIRE(logical_[op.in[k]] == op.K * op.F, where + "a head must have K * F channels");
            ++levels;
          }
        // anchors and strides are tiny and needed as kernel arguments: read them back once
        const void* an = param(op.w, (long long)levels * op.K * 2, where + "anchors");
        const void* st = param(op.bias, levels, where + "strides");
        std::vector<float> anchors((size_t)levels * op.K * 2), strides(levels);
        Cout = op.F;
        Cstored = op.F;
        if (dry_) break;
        DeviceBuffer tmp((anchors.size() + strides.size()) * 4);
        launch_cast(an, dt, tmp.get(), kF32, (long long)anchors.size(), s);
        launch_cast(st, dt, tmp.as<float>() + anchors.size(), kF32, levels, s);
        NNCV_HIP_CHECK(hipMemcpyAsync(anchors.data(), tmp.get(), anchors.size() * 4, hipMemcpyDeviceToHost, s));
        NNCV_HIP_CHECK(hipMemcpyAsync(strides.data(), tmp.as<float>() + anchors.size(), strides.size() * 4, hipMemcpyDeviceToHost, s));
        NNCV_HIP_CHECK(hipStreamSynchronize(s));
        detect_stride_ = strides;
        detect_anchor_wh_.resize(anchors.size());
        for (int l = 0; l < levels; ++l)
          for (int q = 0; q < op.K * 2; ++q) detect_anchor_wh_[l * op.K * 2 + q] = anchors[l * op.K * 2 + q] * strides[l];
        break;
      }
      default: break;
    }
    if (!dry_ && (op.kind == NNCV_HIP_OP_CONV || op.kind == NNCV_HIP_OP_DWCONV)) {
      const int F = Cout, Fs = Cstored > 0 ? Cstored : Cout;
      if (op.gamma >= 0) {
        NNCV_REQUIRE(op.beta >= 0 && op.mean >= 0 && op.var >= 0, where + "BatchNorm needs gamma, beta, mean and var");
        take(i, &Node::scale, (size_t)Fs * 4);
        take(i, &Node::shift, (size_t)Fs * 4);
        launch_fill_f32(nd.scale.as<float>(), 0.0f, Fs, s);
        launch_fill_f32(nd.shift.as<float>(), 0.0f, Fs, s);
        launch_bn_fold(param(op.gamma, F, where + "gamma"), param(op.beta, F, where + "beta"), param(op.mean, F, where + "mean"),
                       param(op.var, F, where + "var"), dt, nd.scale.as<float>(), nd.shift.as<float>(), F, s, op.eps);
      }
      if (op.bias >= 0) {
        const void* b = param(op.bias, F, where + "bias");
        const bool had = nd.shift.get() != nullptr;
        if (!had) {
          take(i, &Node::shift, (size_t)Fs * 4);
          launch_fill_f32(nd.shift.as<float>(), 0.0f, Fs, s);
        }
        const unsigned grid = (unsigned)((F + 255) / 256);
        if (dt == kF16)
          launch_kernel((fold_bias_kernel<half_t>), dim3(grid), dim3(256), 0, s, (const half_t*)b, nd.scale.as<float>(),
                             nd.shift.as<float>(), had ? 1 : 0, F);
        else
          launch_kernel((fold_bias_kernel<float>), dim3(grid), dim3(256), 0, s, (const float*)b, nd.scale.as<float>(),
                             nd.shift.as<float>(), had ? 1 : 0, F);
        NNCV_HIP_CHECK(hipGetLastError());
      }
    }
    if (Cstored < 0) Cstored = Cout;
    NNCV_REQUIRE(Cstored % vn == 0 || op.kind == NNCV_HIP_OP_YOLO_DETECT,
                 where + "channel count must be a multiple of the 16-byte vector");
    channels_[op.out] = Cstored;
    logical_[op.out] = Cout;
  }
  for (int t = 1; t < n_tensors_; ++t) NNCV_REQUIRE(channels_[t] > 0, "graph: tensor " + std::to_string(t) + " is never produced");

  // squeeze-excitation blocks
  static const bool no_se = getenv("NNCV_HIP_NO_SE_FUSION") != nullptr;
  std::vector<int> readers(n_tensors_, 0);
  for (int i = 0; i < n; ++i)
    for (int k = 0; k < 4; ++k)
      if (ops[i].in[k] >= 0) ++readers[ops[i].in[k]];
  auto plain_fc = [&](const GraphOp& o, int in) {
    return o.kind == NNCV_HIP_OP_CONV && o.K == 1 && o.stride == 1 && o.pad == 0 && o.in[0] == in && o.in[1] < 0 && o.bias >= 0 &&
           o.gamma < 0 && readers[in] == 1;
  };
  for (int i = 0; !no_se && i + 3 < n; ++i) {
    const GraphOp &p0 = ops[i], &f1 = ops[i + 1], &f2 = ops[i + 2], &sc = ops[i + 3];
    if (p0.kind != NNCV_HIP_OP_GAVGPOOL || p0.in[0] == 0 || !plain_fc(f1, p0.out) || !plain_fc(f2, f1.out)) continue;
    if (sc.kind != NNCV_HIP_OP_SCALE || sc.in[0] != p0.in[0] || sc.in[1] != f2.out || readers[f2.out] != 1) continue;
    if (f2.F != channels_[p0.in[0]] || !se_block_applicable(dt, 1, f2.F, f1.F)) continue;
    nodes_[i].se_head = true;
    nodes_[i + 1].skip = nodes_[i + 2].skip = nodes_[i + 3].skip = true;
    i += 3;
  }

  // an image convolution (fp16, <= 4 channels, stride 2) that is the only reader of the input
  static const bool no_pairs = getenv("NNCV_HIP_NO_PAIR_STEM") != nullptr;
  if (!no_pairs && dt == kF16 && c_in_ <= 4 && readers[0] == 1)
    for (int i = 0; i < n; ++i)
      if (ops[i].kind == NNCV_HIP_OP_CONV && ops[i].in[0] == 0 && ops[i].stride == 2 && ops[i].in[1] < 0) {
        const GraphOp& o = ops[i];
        const int Fp = channels_[o.out], S2 = (o.K + (o.pad & 1) + 1) / 2;
        pair_stem_ = i;
        keep(nodes_[i].wt_pairs, (size_t)Fp * o.K * S2 * 8 * es);
        if (dry_) continue;
        launch_weight_pairs(param(o.w, (long long)o.F * c_in_ * o.K * o.K, "pair stem w"), dt, nodes_[i].wt_pairs.get(), o.F, Fp, c_in_,
                            o.K, o.pad, s);
      }

  // x + act(conv(.)): the ADD rides in the convolution's epilogue
  static const bool no_add = getenv("NNCV_HIP_NO_ADD_FUSION") != nullptr;
  for (int i = 0; !no_add && i + 1 < n; ++i) {
    const GraphOp &cv = ops[i], &ad = ops[i + 1];
    if (cv.kind != NNCV_HIP_OP_CONV || cv.in[1] >= 0 || ad.kind != NNCV_HIP_OP_ADD || ad.act != kActNone) continue;
    if (readers[cv.out] != 1 || logical_[cv.out] != channels_[cv.out]) continue;
    const int other = ad.in[0] == cv.out ? ad.in[1] : (ad.in[1] == cv.out ? ad.in[0] : -1);
    if (other < 0 || other == cv.out) continue;
    nodes_[i].add_res = other;
    nodes_[i].add_out = ad.out;
    nodes_[i + 1].skip = true;
  }

  // inverted-residual blocks
  if (dt == kF16) {
    std::vector<int> uses(n_tensors_, 0);
    for (int i = 0; i < n; ++i)
      for (int k = 0; k < 4; ++k)
        if (ops[i].in[k] >= 0) ++uses[ops[i].in[k]];
    for (int i = 0; i < n; ++i) {
      const GraphOp& d = ops[i];
      if (d.kind == NNCV_HIP_OP_DWCONV && i > 0) {
        const GraphOp& e = ops[i - 1];
        if (e.kind == NNCV_HIP_OP_CONV && e.out == d.in[0] && e.K == 1 && e.stride == 1 && e.pad == 0 && e.in[1] < 0 && e.in[0] != 0 && uses[e.out] == 1 &&
            nodes_[i - 1].add_out < 0 && logical_[e.out] == channels_[e.out])
          nodes_[i].expands = i - 1;
      }
      // (the pooled tensor must be the depthwise convolution right before it, read by the pool and the gate alone)
      if (nodes_[i].se_head && i > 0 && i + 4 < n && ops[i - 1].kind == NNCV_HIP_OP_DWCONV && ops[i - 1].out == d.in[0] && uses[d.in[0]] == 2) {
        const GraphOp &g = ops[i + 3], &pr = ops[i + 4];
        if (pr.kind == NNCV_HIP_OP_CONV && pr.in[0] == g.out && pr.in[1] != g.out && uses[g.out] == 1 && pr.K == 1 && pr.stride == 1 && pr.pad == 0 &&
            nodes_[i + 4].add_out < 0 && logical_[pr.out] == channels_[pr.out] && se_project_applicable(1, g.in[0] >= 0 ? channels_[g.in[0]] : 0, ops[i + 1].F, pr.F))
        {
          nodes_[i].projects = i + 4;
          for (int k = 1; k <= 2; ++k) {
            Node& f = nodes_[i + k];
            keep(f.wt_t, (size_t)f.op.F * f.C * es);
            if (!dry_) launch_transpose_half(f.wt.get(), f.wt_t.get(), f.op.F, f.C, s);
          }
        }
      }
    }
  }

  // The filters in conv_direct.hip's order, for the layers that may run there, and for projections (mobile_block.hip).  The two
  // vectors of a squeeze-excitation block are never convolutions of their own.
  for (int i = 0; i < n; ++i) {
    const GraphOp& o = ops[i];
    const bool projection = i >= 4 && nodes_[i - 4].projects == i;
    if (o.kind != NNCV_HIP_OP_CONV || nodes_[i].skip) continue;
    const int C = nodes_[i].C, Fs = channels_[o.out];
    if (!projection && !conv_direct_serves(dt, Fs, o.K * o.K, C)) continue;
    keep(nodes_[i].wflat, weight_flat_bytes(dt, Fs, o.K * o.K, C));
    if (!dry_) launch_weight_flat(blob + (size_t)o.w * es, nodes_[i].wflat.get(), dt, o.F, logical_[o.in[0]], o.K * o.K, C, s);
  }

  // a pointwise convolution that is only averaged: its result need not be stored
  static const bool no_pool = getenv("NNCV_HIP_NO_POOL_FUSION") != nullptr;
  for (int i = 0; !no_pool && dt == kF16 && i + 1 < n; ++i) {
    const GraphOp &c = ops[i], &q = ops[i + 1];
    nodes_[i].pools = c.kind == NNCV_HIP_OP_CONV && c.K == 1 && c.stride == 1 && c.pad == 0 && c.in[0] > 0 && c.in[1] < 0 && q.kind == NNCV_HIP_OP_GAVGPOOL &&
                      q.in[0] == c.out && readers[c.out] == 1 && !nodes_[i].skip && !nodes_[i + 1].skip && !nodes_[i + 1].se_head &&
                      logical_[c.in[0]] == channels_[c.in[0]] && !(i >= 4 && nodes_[i - 4].projects == i);
  }

  for (int i = 0; i < n; ++i) {  // what rides in another launch, or carries one, does not join
    auto single = [&](int k) {
      return !nodes_[k].pools && !nodes_[k].skip && nodes_[k].add_out < 0 && !(k >= 4 && nodes_[k - 4].projects == k) && !(k + 1 < n && nodes_[k + 1].expands == k);
    };
    if (nodes_[i].joins >= 0 && !(single(i) && single(nodes_[i].joins))) nodes_[nodes_[i].joins].joined = false, nodes_[i].joins = -1;
  }
  // the first pointwise layer of the bottleneck behind the first of two joined ones
  static const bool no_chain = getenv("NNCV_HIP_NO_CHAIN") != nullptr;
  for (int i = 0; !no_chain && i + 1 < n; ++i) {
    if (nodes_[i].joins < 0) continue;
    for (int k = i + 1; k < n && nodes_[i].chain < 0; ++k) {
      const GraphOp& o = ops[k];
      const Node& nk = nodes_[k];
      if (o.kind == NNCV_HIP_OP_CONV && o.K == 1 && o.stride == 1 && o.pad == 0 && o.in[0] == ops[i].out && o.in[1] < 0 && o.F == ops[i].F && !nk.skip &&
          nk.add_out < 0 && nk.joins < 0 && !nk.joined && !nk.pools && !nk.head && !(k >= 4 && nodes_[k - 4].projects == k) &&
          !(k + 1 < n && nodes_[k + 1].expands == k) && k != n - 1)
        nodes_[i].chain = k, nodes_[i].chain_only = readers[ops[i].out] == 1, nodes_[k].chained_by = i;
    }
  }

  // detection heads
  if (dt == kF16 && ops[n - 1].kind == NNCV_HIP_OP_YOLO_DETECT) {
    const GraphOp& d = ops[n - 1];
    std::vector<int> made;
    bool ok = true;
    for (int k = 0; k < 3 && d.in[k] >= 0; ++k) {
      int h = -1;
      for (int i = 0; i < n; ++i)
        if (ops[i].out == d.in[k]) h = i;
      const GraphOp& c = ops[std::max(h, 0)];
      ok = ok && h >= 0 && c.kind == NNCV_HIP_OP_CONV && c.K == 1 && c.stride == 1 && c.pad == 0 && c.in[0] > 0 && c.in[1] < 0 && c.act == kActNone &&
           readers[d.in[k]] == 1 && !nodes_[h].skip && nodes_[h].chained_by < 0 && !nodes_[h].joined && nodes_[h].joins < 0 && logical_[c.in[0]] == channels_[c.in[0]] &&
           detect_head_applicable(d.K, d.F, channels_[c.in[0]], 0);
      made.push_back(h);
    }
    for (int h : made) {
      Node& c = nodes_[std::max(h, 0)];
      c.head = ok;
      if (!ok) continue;
      keep(c.wfrag, weight_frag1x1_bytes(c.op.F, c.C));
      if (!dry_) launch_weight_frag1x1(blob + (size_t)c.op.w * es, dt, c.wfrag.get(), dt, c.op.F, c.C, s);
    }
  }

  // concatenation views
  row_ = channels_;
  view_of_.assign(n_tensors_, -1);
  view_c0_.assign(n_tensors_, 0);
  static const bool no_views = getenv("NNCV_HIP_NO_CONCAT_VIEWS") != nullptr;
  if (!no_views) {
    std::vector<int> producer(n_tensors_, -1), cat_uses(n_tensors_, 0);
    for (int i = 0; i < n; ++i) {
      if (i == 0 || nodes_[i - 1].add_out != ops[i].out) producer[nodes_[i].add_out >= 0 ? nodes_[i].add_out : ops[i].out] = i;
      if (ops[i].kind == NNCV_HIP_OP_CONCAT)
        for (int k = 0; k < 4; ++k)
          if (ops[i].in[k] >= 0) ++cat_uses[ops[i].in[k]];
    }
    // may operator i read tensor t at a pitch / write its result at a pitch?
    auto reads_pitched = [&](int i, int t) {
      const GraphOp& o = ops[i];
      if (nodes_[i].skip)  // merged into its predecessor: the residual of a conv + ADD pair shares the result's pitch
        return i > 0 && nodes_[i - 1].add_out >= 0 && nodes_[i - 1].add_res != t;
      switch (o.kind) {
        case NNCV_HIP_OP_CONV:  // not as the residual, nor as the input of a projection
          return o.in[1] != t && !(i >= 4 && nodes_[i - 4].projects == i);
        case NNCV_HIP_OP_MAXPOOL:
        case NNCV_HIP_OP_UPSAMPLE2X:
        case NNCV_HIP_OP_ADD:
        case NNCV_HIP_OP_ACT:
        case NNCV_HIP_OP_CONCAT:
        case NNCV_HIP_OP_YOLO_DETECT: return true;
        default: return false;
      }
    };
    auto writes_pitched = [&](int i) {
      const GraphOp& o = ops[i];
      if (nodes_[i].se_head || nodes_[i].skip) return false;
      switch (o.kind) {
        case NNCV_HIP_OP_CONV:  // residual and result share one pitch; so do the results of the merged blocks
          return o.in[1] < 0 && nodes_[i].add_res < 0 && !(i >= 4 && nodes_[i - 4].projects == i) && !(i + 1 < n && nodes_[i + 1].expands == i);
        case NNCV_HIP_OP_MAXPOOL:
        case NNCV_HIP_OP_UPSAMPLE2X:
        case NNCV_HIP_OP_ADD:
        case NNCV_HIP_OP_ACT:
        case NNCV_HIP_OP_CONCAT: return true;
        default: return false;
      }
    };
    // The result of conv + ADD shares its pitch with the residual.  To put it into a concatenated tensor, the residual (and
    // what was added to that, and so on) is given rows of the same width, the rest of them unused: that costs memory but no
    // traffic, where copying the result into its slice cost a read and a write of it (10 us for 16x160x160x32).
    auto widen = [&](int t, int to, int reader, auto& self) -> bool {
      const int pr = t > 0 ? producer[t] : -1;
      if (pr < 0 || view_of_[t] >= 0 || cat_uses[t] > 0 || logical_[t] != channels_[t] || row_[t] != channels_[t] || row_[t] > to) return false;
      const int res = nodes_[pr].add_res;
      if (ops[pr].kind != NNCV_HIP_OP_CONV || (res < 0 && !writes_pitched(pr))) return false;
      for (int j = 0; j < n; ++j)
        for (int q = 0; q < 4; ++q)
          if (ops[j].in[q] == t && !(j == reader + 1 && nodes_[j].skip) && !reads_pitched(j, t)) return false;
      if (res >= 0 && !self(res, to, pr, self)) return false;
      row_[t] = to;
      return true;
    };
    for (int i = 0; i < n; ++i) {
      if (ops[i].kind != NNCV_HIP_OP_CONCAT) continue;
      int c0 = 0;
      for (int k = 0; k < 4; ++k) {
        const int t = ops[i].in[k];
        if (t < 0) continue;
        const int res = producer[t] >= 0 ? nodes_[producer[t]].add_res : -1;
        bool ok = t != 0 && cat_uses[t] == 1 && producer[t] >= 0 && (res >= 0 || writes_pitched(producer[t])) && logical_[t] == channels_[t];
        for (int j = 0; ok && j < n; ++j)
          for (int q = 0; q < 4; ++q)
            if (ops[j].in[q] == t && !reads_pitched(j, t)) ok = false;
        if (ok && res >= 0) ok = cat_uses[ops[i].out] == 0 && widen(res, channels_[ops[i].out], producer[t], widen);
        if (ok) {
          view_of_[t] = ops[i].out;
          view_c0_[t] = c0;
        }
        c0 += channels_[t];
      }
    }
  }
  // an up-sampled tensor that is the beginning of a concatenated one, which two joined convolutions read and nothing else
  static const bool no_up = getenv("NNCV_HIP_NO_UP_FUSION") != nullptr;
  for (int u = 0; !no_up && u < n; ++u) {
    const int t = ops[u].out, cat = view_of_[t];
    if (ops[u].kind != NNCV_HIP_OP_UPSAMPLE2X || ops[u].in[0] == 0 || cat < 0 || view_c0_[t] != 0 || readers[t] != 1 || readers[cat] != 2 || view_of_[cat] >= 0) continue;
    for (int i = u + 1; i < n; ++i)
      if (ops[i].in[0] == cat && nodes_[i].joins >= 0 && ops[nodes_[i].joins].in[0] == cat) nodes_[i].ups = u, nodes_[u].upped_by = i;
  }
}

void Graph::root_of(int t, int* root, int* c0) const {
  int off = 0;
  while (view_of_[t] >= 0) {
    off += view_c0_[t];
    t = view_of_[t];
  }
  *root = t;
  *c0 = off;
}

const Graph::Plan& Graph::plan_of(int N, int H, int W) const {
  for (const Plan& p : plans_)
    if (p.N == N && p.H == H && p.W == W) return p;
  NNCV_REQUIRE(N >= 1 && H >= 1 && W >= 1, "graph: empty input");
  Plan p;
  p.N = N; p.H = H; p.W = W;
  p.dims.assign(n_tensors_, Dims{0, 0, 0});
  p.dims[0] = Dims{channels_[0], H, W};
  const int n = (int)nodes_.size();
  for (int i = 0; i < n; ++i) {
    const GraphOp& op = nodes_[i].op;
    const std::string where = "graph: operator " + std::to_string(i) + " (" + kind_name(op.kind) + "): ";
    const Dims a = p.dims[op.in[0]];
    Dims o{channels_[op.out], a.H, a.W};
    switch (op.kind) {
      case NNCV_HIP_OP_CONV:
      case NNCV_HIP_OP_DWCONV:
      case NNCV_HIP_OP_MAXPOOL:
        NNCV_REQUIRE(a.H + 2 * op.pad >= op.K && a.W + 2 * op.pad >= op.K, where + "image smaller than the window");
        o.H = (a.H + 2 * op.pad - op.K) / op.stride + 1;
        o.W = (a.W + 2 * op.pad - op.K) / op.stride + 1;
        if (op.kind == NNCV_HIP_OP_CONV && op.in[1] >= 0)
          NNCV_REQUIRE(p.dims[op.in[1]].H == o.H && p.dims[op.in[1]].W == o.W, where + "residual has another size");
        break;
      case NNCV_HIP_OP_GAVGPOOL: o.H = o.W = 1; break;
      case NNCV_HIP_OP_SCALE:
        NNCV_REQUIRE(p.dims[op.in[1]].H == 1 && p.dims[op.in[1]].W == 1, where + "the gate must be [N,C,1,1]");
        break;
      case NNCV_HIP_OP_ADD:
        NNCV_REQUIRE(p.dims[op.in[1]].H == a.H && p.dims[op.in[1]].W == a.W, where + "operands have different sizes");
        break;
      case NNCV_HIP_OP_CONCAT:
        for (int k = 1; k < 4; ++k)
          if (op.in[k] >= 0)
            NNCV_REQUIRE(p.dims[op.in[k]].H == a.H && p.dims[op.in[k]].W == a.W, where + "operands have different sizes");
        break;
      case NNCV_HIP_OP_UPSAMPLE2X: o.H = 2 * a.H; o.W = 2 * a.W; break;
      case NNCV_HIP_OP_YOLO_DETECT: {  // [N, boxes, F]: reported as channels = boxes, height = F, width = 1
        long long boxes = 0;
        for (int k = 0; k < 3; ++k)
          if (op.in[k] >= 0) boxes += (long long)op.K * p.dims[op.in[k]].H * p.dims[op.in[k]].W;
        NNCV_REQUIRE(boxes * op.F * N < (1ll << 31), where + "tensor too large");
        o.C = (int)boxes; o.H = op.F; o.W = 1;
        break;
      }
      default: break;
    }
    NNCV_REQUIRE((long long)N * o.H * o.W * o.C < (1ll << 31), where + "tensor too large");
    p.dims[op.out] = o;
  }
  p.dw.assign(n, 0);
  p.se.assign(n, 0);
  if (dt_ == kF16)
    for (int i = 0; i < n; ++i) {
      const GraphOp& op = nodes_[i].op;
      if (op.kind != NNCV_HIP_OP_DWCONV) continue;
      const bool expands = nodes_[i].expands >= 0, projects = i + 1 < n && nodes_[i + 1].projects >= 0;
      if (!expands && !projects) continue;
      const Dims a = p.dims[op.in[0]], o = p.dims[op.out];
      const int Cin = expands ? p.dims[nodes_[i - 1].op.in[0]].C : 0;
      p.dw[i] = dw_block_bands(N, a.H, a.W, Cin, a.C, op.K, op.stride, op.pad);
      if (p.dw[i] && projects)
        p.se[i + 1] = se_project_applicable(o.H * o.W, a.C, nodes_[i + 2].op.F, nodes_[i + 5].op.F);
      if (!expands && !p.se[i + 1]) p.dw[i] = 0;
    }
  // Lifetimes in operator steps: step 0 lays the input out as NHWC, step i + 1 is operator i,
  // step n + 1 converts the output.  A tensor is live from the step that writes it to the last
  // step that reads it, so an operator's output never shares memory with any of its inputs.
  std::vector<TensorLife> life(n_tensors_);
  const size_t es = dtype_size(dt_);
  life[0] = TensorLife{0, std::max(0, last_use_[0] + 1), (size_t)N * H * W * channels_[0] * es, 0};
  for (int i = 0; i < n; ++i) {
    const int t = nodes_[i].op.out;
    const Dims d = p.dims[t];
    life[t] = TensorLife{i + 1, std::max(i + 1, last_use_[t] + 1), (size_t)N * d.H * d.W * (nodes_[i].op.kind == NNCV_HIP_OP_YOLO_DETECT ? d.C : row_[t]) * es, 0};
    if (nodes_[i].op.kind == NNCV_HIP_OP_YOLO_DETECT) life[t].bytes = 256;  // written straight to the caller's buffer
  }
  // Operators that were merged into an earlier launch write their result at that launch's step, so the
  // result is live from there: the tail of a squeeze-excitation block (written by the block's one launch
  // at the pooling operator's step), the ADD of a convolution + ADD pair (written by the convolution),
  // the later two of three chained 5x5 stride-1 pad-2 max-pools (one launch writes all three results).
  // Without this the planner sees the merged result and an input of the earlier launch as disjoint in
  // time and may lay one over the other.
  for (int i = 0; i < n; ++i) {
    if (nodes_[i].se_head && i + 3 < n) life[nodes_[i + 3].op.out].first_op = i + 1;
    if (p.dw[i] && nodes_[i].expands >= 0) {  // one launch, at the expansion's step; the expanded tensor is never stored
      life[nodes_[i].op.out].first_op = i;
      life[nodes_[i - 1].op.out] = TensorLife{i, i, 0, 0};
    }
    if (p.se[i]) {  // parts of the squeezed vector, from the depthwise launch on; the gated tensor is never stored
      const size_t parts = (size_t)N * p.dw[i - 1] * ((p.dims[nodes_[i].op.in[0]].C + 31) / 32);
      life[nodes_[i].op.out] = TensorLife{nodes_[i - 1].expands >= 0 ? i - 1 : i, i + 1, parts * nodes_[i + 1].op.F * 4, 0};
      life[nodes_[i + 3].op.out] = TensorLife{i + 1, i + 1, 0, 0};
      life[nodes_[i + 4].op.out].first_op = i + 1;
    }
    if (nodes_[i].add_out >= 0) life[nodes_[i].add_out].first_op = std::min(life[nodes_[i].add_out].first_op, i + 1);
    if (nodes_[i].joins >= 0) life[nodes_[nodes_[i].joins].op.out].first_op = i + 1;  // (also where the shape is not joined)
    if (nodes_[i].ups >= 0) life[nodes_[nodes_[i].ups].op.in[0]].last_op = std::max(life[nodes_[nodes_[i].ups].op.in[0]].last_op, i + 1);
    if (nodes_[i].chain >= 0) life[nodes_[nodes_[i].chain].op.out].first_op = i + 1;  // (likewise)
  }
  {
    auto pool5 = [&](int k, int in) {
      return k < n && !nodes_[k].skip && nodes_[k].op.kind == NNCV_HIP_OP_MAXPOOL && nodes_[k].op.K == 5 && nodes_[k].op.stride == 1 &&
             nodes_[k].op.pad == 2 && (in < 0 || nodes_[k].op.in[0] == in);
    };
    for (int i = 0; i + 2 < n; ++i)
      if (pool5(i, -1) && pool5(i + 1, nodes_[i].op.out) && pool5(i + 2, nodes_[i + 1].op.out)) {
        life[nodes_[i + 1].op.out].first_op = i + 1;
        life[nodes_[i + 2].op.out].first_op = i + 1;
      }
  }
  p.pooled.assign(n, 0);
  for (int i = 0; i + 1 < n; ++i) {
    const int in = nodes_[i].op.in[0], t = nodes_[i].op.out;
    const Dims a = p.dims[in];
    if (!nodes_[i].pools || !conv_pool_applicable(N, a.H * a.W, pitch(in), a.C, channels_[t])) continue;
    p.pooled[i] = 1;
    life[t] = TensorLife{i + 1, i + 1, 0, 0};
    life[nodes_[i + 1].op.out].first_op = i + 1;
  }
  // A last convolution to one pixel, where its kernel can store fp32: in the order of the caller's tensor already (32x1x1x1024 -> 1000: 5.9 us
  // behind the pass; 4.2 and as much again for the conversion before).
  if (const Node& nd = nodes_[n - 1]; nd.op.kind == NNCV_HIP_OP_CONV && !nd.skip && !nd.joined && nd.op.in[1] < 0 && nd.op.in[0] > 0 && nd.wflat.get() &&
                                      nd.op.F % 4 == 0 && p.dims[nd.op.out].H * p.dims[nd.op.out].W == 1 && pair_stem_ != n - 1 &&
                                      !(n >= 5 && nodes_[n - 5].projects == n - 1))
    p.last_f32 = igemm_takes_direct(last_args(p, nullptr, nullptr), dt_, dt_);
  if (p.last_f32) {
    life[nodes_[n - 1].op.out].bytes = 0;
    life[nodes_[n - 1].op.in[0]].last_op = n + 1;
  }
  p.head = nodes_[n - 1].op.kind == NNCV_HIP_OP_YOLO_DETECT;
  for (int k = 0; p.head && k < 3 && nodes_[n - 1].op.in[k] >= 0; ++k) {
    const Node* c = maker(nodes_[n - 1].op.in[k]);
    const int t = c ? c->op.in[0] : 0;
    p.head = c && c->head && detect_head_applicable(nodes_[n - 1].op.K, nodes_[n - 1].op.F, channels_[t], (long long)N * p.dims[t].H * p.dims[t].W * pitch(t) * (long long)es);
  }
  for (int k = 0; p.head && k < 3 && nodes_[n - 1].op.in[k] >= 0; ++k) {  // the heads are never stored, what they read lives on
    const int h = nodes_[n - 1].op.in[k], t = maker(h)->op.in[0];
    life[t].last_op = std::max(life[t].last_op, n);
    life[h] = TensorLife{n, n, 0, 0};
  }
  life[nodes_[n - 1].op.out].last_op = n + 1;
  // a tensor that lives inside a concatenated one has no memory of its own; the concatenated
  // tensor is live from its first such input to the last reader of any of them
  for (int t = 1; t < n_tensors_; ++t) {
    if (view_of_[t] < 0) continue;
    int root, c0;
    root_of(t, &root, &c0);
    life[root].first_op = std::min(life[root].first_op, life[t].first_op);
    life[root].last_op = std::max(life[root].last_op, life[t].last_op);
  }
  for (int t = 1; t < n_tensors_; ++t)
    if (view_of_[t] >= 0) life[t] = TensorLife{life[t].first_op, life[t].first_op, 0, 0};
  for (int i = 0; i < n; ++i)  // the output of a convolution that was merged with its ADD is never stored
    if (nodes_[i].add_out >= 0) life[nodes_[i].op.out] = TensorLife{i + 1, i + 1, 0, 0};
  // memory is handed on a few launches after its last reader, not at once (arena_plan.hpp)
  for (int t = 0; t < n_tensors_; ++t)
    if (life[t].bytes > 0) life[t].last_op = std::min(n + 1, life[t].last_op + arena_linger());
  p.total = plan_offsets(life, 256);
  p.offset.resize(n_tensors_);
  p.root_bytes.resize(n_tensors_);
  for (int t = 0; t < n_tensors_; ++t) {
    int root, c0;
    root_of(t, &root, &c0);
    p.offset[t] = life[root].offset + (size_t)c0 * es;
    p.root_bytes[t] = life[root].bytes;
  }
  // Joined convolutions: one launch where the LDS ring takes the doubled filters and both results lie within its reach.
  p.joint.assign(n, 0);
  p.chained.assign(n, 0);
  p.upped.assign(n, 0);
  for (int i = 0; i < n; ++i) {
    if (nodes_[i].joins < 0) continue;
    const IgemmArgs g = joint_args(p, i, nullptr);
    p.joint[i] = g.in_bytes < 0x7fffff00u && !igemm_takes_direct(g, dt_, dt_) && conv_ring_applicable(g, dt_, dt_);
    const long long P = (long long)N * g.OH * g.OW;
    p.chained[i] = p.joint[i] && nodes_[i].chain >= 0 && conv_ring_chains(P, g.C, nodes_[i].op.F) && P * pitch(nodes_[nodes_[i].chain].op.out) * 2 < 0x7fffff00ll;
    if (const int u = nodes_[i].ups; p.joint[i] && u >= 0)
      p.upped[i] = conv_ring_upsamples(joint_args(p, i, nullptr), channels_[nodes_[u].op.out], pitch(nodes_[u].op.in[0]));
  }
  check_plan(p);
  if (plans_.size() >= 8) plans_.erase(plans_.begin());
  plans_.push_back(std::move(p));
  return plans_.back();
}

const Graph::Node* Graph::maker(int t) const {
  for (const Node& nd : nodes_)
    if (nd.op.out == t) return &nd;
  return nullptr;
}

bool Graph::chained_third(const Plan& p, int i) const { return nodes_[i].chained_by >= 0 && p.chained[nodes_[i].chained_by]; }

bool Graph::joint_second(const Plan& p, int i) const {
  for (int k = 0; k < i; ++k)
    if (nodes_[k].joins == i) return p.joint[k];
  return false;
}

int Graph::pitch(int t) const {
  int root, c0;
  root_of(t, &root, &c0);
  return row_[root];
}

// The last convolution, to one pixel of `out`.
IgemmArgs Graph::last_args(const Plan& p, const char* base, float* out) const {
  const Node& nd = nodes_.back();
  const GraphOp& op = nd.op;
  const Dims a = p.dims[op.in[0]];
  IgemmArgs g{};
  g.in = base ? base + p.offset[op.in[0]] : nullptr; g.wt = nd.wt.get(); g.wt_flat = nd.wflat.get(); g.out = out;
  g.scale = nd.scale.as<float>(); g.shift = nd.shift.as<float>();
  g.N = p.N; g.H = a.H; g.W = a.W; g.C = a.C; g.F = g.ldo = op.F; g.R = g.S = op.K; g.OH = g.OW = 1;
  g.stride_h = g.stride_w = op.stride; g.pad_h = g.pad_w = op.pad; g.relu = op.act; g.batch = 1;
  g.pix_stride = pitch(op.in[0]);
  const unsigned long long span = (unsigned long long)p.N * a.H * a.W * g.pix_stride * dtype_size(dt_);
  g.in_bytes = span < 0xffffffffull ? (unsigned)span : 0xffffffffu;
  g.alg_flops = 2.0 * p.N * op.F * (double)op.K * op.K * logical_[op.in[0]];
  return g;
}

// The launch that computes operator i and the one it joins: filters of both, results to two tensors.
IgemmArgs Graph::joint_args(const Plan& p, int i, char* base) const {
  const Node &nd = nodes_[i], &nj = nodes_[nd.joins];
  const Dims a = p.dims[nd.op.in[0]];
  const int F = nd.op.F, t = nd.op.out, u = nj.op.out, ldi = pitch(nd.op.in[0]);
  IgemmArgs g{};
  g.in = base + p.offset[nd.op.in[0]]; g.wt = nd.wt.get(); g.wt_flat = nd.wflat.get(); g.wt_frag = nd.wfrag.get();
  g.scale = nd.scale.as<float>(); g.shift = nd.shift.as<float>();
  g.N = p.N; g.H = g.OH = a.H; g.W = g.OW = a.W; g.C = a.C; g.F = 2 * F; g.R = g.S = 1;
  g.stride_h = g.stride_w = 1; g.relu = nd.op.act; g.batch = 1;
  g.pix_stride = ldi;
  const unsigned long long span = (unsigned long long)p.N * a.H * a.W * ldi * dtype_size(dt_);
  g.in_bytes = span < 0xffffffffull ? (unsigned)span : 0xffffffffu;
  g.out = base + p.offset[t]; g.ldo = pitch(t);
  if (p.upped[i]) {
    const GraphOp& u = nodes_[nd.ups].op;
    g.up_in = base + p.offset[u.in[0]]; g.up_c = channels_[u.out]; g.up_pix = pitch(u.in[0]);
  }
  if (p.chained[i]) {
    const Node& nk = nodes_[nd.chain];
    g.chain_wt = nk.wt.get(); g.chain_scale = nk.scale.as<float>(); g.chain_shift = nk.shift.as<float>();
    g.chain_out = base + p.offset[nk.op.out]; g.chain_f = F; g.chain_act = nk.op.act; g.chain_ldo = pitch(nk.op.out); g.chain_only = nd.chain_only;
  }
  g.split_f = F; g.split_ldo = pitch(u); g.split_ofs = (long long)p.offset[u] - (long long)p.offset[t];
  g.alg_flops = 2.0 * p.N * a.H * a.W * 2 * F * (double)logical_[nd.op.in[0]];
  return g;
}

// The tensors one launch of forward() touches: what it writes and what it reads.
void Graph::launch_io(const Plan& p, int i, std::vector<int>* writes, std::vector<int>* reads) const {
  writes->clear();
  reads->clear();
  const int n = (int)nodes_.size();
  const Node& nd = nodes_[i];
  const GraphOp& op = nd.op;
  if (nd.skip || (nd.head && p.head)) return;
  if (op.kind == NNCV_HIP_OP_YOLO_DETECT && p.head) {
    for (int k = 0; k < 3; ++k)
      if (op.in[k] >= 0) reads->push_back(maker(op.in[k])->op.in[0]);
    return;
  }
  if ((nd.joined && joint_second(p, i)) || chained_third(p, i) || (nd.upped_by >= 0 && p.upped[nd.upped_by])) return;
  if (i > 0 && p.pooled[i - 1]) return;
  if (p.pooled[i] || (i == n - 1 && p.last_f32)) {
    reads->push_back(op.in[0]);
    if (p.pooled[i]) writes->push_back(nodes_[i + 1].op.out);
    return;
  }
  if (nd.joins >= 0 && p.joint[i]) {
    reads->push_back(op.in[0]);
    if (p.upped[i]) reads->push_back(nodes_[nd.ups].op.in[0]);
    if (!(p.chained[i] && nd.chain_only)) writes->push_back(op.out);
    writes->push_back(nodes_[nd.joins].op.out);
    if (p.chained[i]) writes->push_back(nodes_[nd.chain].op.out);
    return;
  }
  if (op.kind == NNCV_HIP_OP_CONV && i + 1 < n && nodes_[i + 1].expands == i && p.dw[i + 1]) {
    reads->push_back(op.in[0]);
    writes->push_back(nodes_[i + 1].op.out);
    if (i + 2 < n && p.se[i + 2]) writes->push_back(nodes_[i + 2].op.out);
    return;
  }
  if (op.kind == NNCV_HIP_OP_DWCONV && p.dw[i]) {
    if (nd.expands >= 0) return;
    reads->push_back(op.in[0]);
    writes->push_back(op.out);
    writes->push_back(nodes_[i + 1].op.out);
    return;
  }
  if (p.se[i]) {
    const GraphOp& pr = nodes_[i + 4].op;
    reads->push_back(op.in[0]);
    reads->push_back(op.out);
    if (pr.in[1] >= 0) reads->push_back(pr.in[1]);
    writes->push_back(pr.out);
    return;
  }
  if (op.kind == NNCV_HIP_OP_CONV && i >= 4 && p.se[i - 4]) return;
  if (nd.se_head) {
    reads->push_back(op.in[0]);
    writes->push_back(nodes_[i + 3].op.out);
    return;
  }
  for (int k = 0; k < 4; ++k)  // inputs of a CONCAT that already live in its result are not copied
    if (op.in[k] >= 0 && !(op.kind == NNCV_HIP_OP_CONCAT && view_of_[op.in[k]] == op.out)) reads->push_back(op.in[k]);
  if (nd.add_res >= 0) reads->push_back(nd.add_res);
  if (op.kind == NNCV_HIP_OP_YOLO_DETECT) return;  // writes the caller's buffer
  writes->push_back(nd.add_out >= 0 ? nd.add_out : op.out);
  auto pool5 = [&](int k, int in) {
    return k < n && !nodes_[k].skip && nodes_[k].op.kind == NNCV_HIP_OP_MAXPOOL && nodes_[k].op.K == 5 && nodes_[k].op.stride == 1 &&
           nodes_[k].op.pad == 2 && (in < 0 || nodes_[k].op.in[0] == in);
  };
  if (pool5(i, -1) && pool5(i + 1, op.out) && pool5(i + 2, nodes_[i + 1].op.out)) {
    writes->push_back(nodes_[i + 1].op.out);
    writes->push_back(nodes_[i + 2].op.out);
  }
}

// No launch may write memory that it also reads (a 3x3 convolution in place is a race between
// workgroups on the halo rows) or that another tensor it writes occupies.  Two tensors inside the same
// concatenated tensor are channel slices of the same rows and must not share channels; everything
// else is compared as whole byte ranges.
void Graph::check_plan(const Plan& p) const {
  const size_t es = dtype_size(dt_);
  auto clash = [&](int a, int b) {
    int ra, ca, rb, cb;
    root_of(a, &ra, &ca);
    root_of(b, &rb, &cb);
    if (ra == rb) return a == b || (ca < cb + channels_[b] && cb < ca + channels_[a]);
    const size_t a0 = p.offset[a] - (size_t)ca * es, b0 = p.offset[b] - (size_t)cb * es;
    return p.root_bytes[a] > 0 && p.root_bytes[b] > 0 && a0 < b0 + p.root_bytes[b] && b0 < a0 + p.root_bytes[a];
  };
  std::vector<int> w, r;
  for (int i = 0; i < (int)nodes_.size(); ++i) {
    launch_io(p, i, &w, &r);
    for (size_t x = 0; x < w.size(); ++x) {
      for (int t : r)
        NNCV_REQUIRE(!clash(w[x], t), "graph: workspace plan lays the result of operator " + std::to_string(i) + " (tensor " +
                                          std::to_string(w[x]) + ") over its input tensor " + std::to_string(t));
      for (size_t y = x + 1; y < w.size(); ++y)
        NNCV_REQUIRE(!clash(w[x], w[y]), "graph: workspace plan lays two results of operator " + std::to_string(i) + " over each other");
    }
  }
}

size_t Graph::describe_plan(int N, int H, int W, long long* tensor_info, int* launch_dst) const {
  const Plan& p = plan_of(N, H, W);
  for (int t = 0; t < n_tensors_; ++t) {
    int root, c0;
    root_of(t, &root, &c0);
    tensor_info[4 * t + 0] = root;
    tensor_info[4 * t + 1] = (long long)p.offset[t];
    tensor_info[4 * t + 2] = (long long)p.root_bytes[t];
    tensor_info[4 * t + 3] = c0;
  }
  std::vector<int> w, r;
  for (int i = 0; i < (int)nodes_.size(); ++i) {
    launch_io(p, i, &w, &r);
    launch_dst[i] = w.empty() ? -1 : w[0];
  }
  return p.total;
}

void Graph::output_shape(int H, int W, int* C, int* OH, int* OW) const {
  const Plan& p = plan_of(1, H, W);
  const int t = nodes_.back().op.out;
  const Dims d = p.dims[t];
  *C = nodes_.back().op.kind == NNCV_HIP_OP_YOLO_DETECT ? d.C : logical_[t];
  *OH = d.H; *OW = d.W;
}

size_t Graph::workspace_bytes(int N, int H, int W) const { return plan_of(N, H, W).total; }

void Graph::forward_body(const void* src, int N, int H, int W, void* ws, hipStream_t s) const {
  const Plan& p = plan_of(N, H, W);
  char* base = static_cast<char*>(ws);
  auto at = [&](int t) -> void* { return base + p.offset[t]; };
  const bool pairs = pair_stem_ >= 0 && W % 2 == 0;
  ImagePairsArgs image{};
  if (pairs) {
    const Node& nd = nodes_[pair_stem_];
    const Dims o = p.dims[nd.op.out];
    image.in = src; image.wt = nd.wt_pairs.get(); image.scale = nd.scale.as<float>(); image.shift = nd.shift.as<float>(); image.out = at(nd.op.out);
    image.N = N; image.C = c_in_; image.H = H; image.W = W; image.F = o.C; image.OH = o.H; image.OW = o.W;
    image.R = nd.op.K; image.S = (nd.op.K + (nd.op.pad & 1) + 1) / 2; image.pad_h = nd.op.pad; image.pad_w = (nd.op.pad + 1) / 2;
    image.ldo = pitch(nd.op.out); image.act = nd.op.act;
    image.alg_flops = 2.0 * N * o.H * o.W * nd.op.F * (double)nd.op.K * nd.op.K * c_in_;
  }
  const bool direct = pairs && nodes_[pair_stem_].add_out < 0 && image_pairs_applicable(image);
  if (direct) {
    // its one reader takes the image as it is
  } else if (pairs)
    launch_image_to_nhwc(src, at(0), dt_, N, c_in_, H, W, s, 4);
  else if (image_to_nhwc_applicable(dt_, c_in_))
    launch_image_to_nhwc(src, at(0), dt_, N, c_in_, H, W, s);
  else
    launch_relayout(src, dt_, strides_of(kNCHW, c_in_, H, W), at(0), dt_, strides_of(kNHWC, channels_[0], H, W), N, c_in_,
                    channels_[0], H, W, false, s);
  for (size_t i = 0; i < nodes_.size(); ++i) {
    const Node& nd = nodes_[i];
    const GraphOp& op = nd.op;
    const Dims a = p.dims[op.in[0]], o = p.dims[op.out];
    if (direct && (int)i == pair_stem_) {
      launch_image_pairs(image, s);
      continue;
    }
    if (nd.skip || (nd.head && p.head) || (nd.joined && joint_second(p, (int)i)) || chained_third(p, (int)i) || (nd.upped_by >= 0 && p.upped[nd.upped_by])) continue;
    if ((i > 0 && p.pooled[i - 1]) || (i + 1 == nodes_.size() && p.last_f32)) continue;
    if (p.pooled[i]) {
      ConvPoolArgs c{};
      c.in = at(op.in[0]); c.wt = nd.wt.get(); c.scale = nd.scale.as<float>(); c.shift = nd.shift.as<float>(); c.out = at(nodes_[i + 1].op.out);
      c.N = N; c.HW = a.H * a.W; c.pix = pitch(op.in[0]); c.C = a.C; c.F = o.C; c.act = op.act;
      launch_conv_pool(c, s);
      continue;
    }
    if (nd.joins >= 0 && p.joint[i]) {
      launch_conv_ring(joint_args(p, (int)i, base), s);
      continue;
    }
    if (op.kind == NNCV_HIP_OP_CONV && i + 1 < nodes_.size() && nodes_[i + 1].expands == (int)i && p.dw[i + 1]) continue;  // rides below
    if (op.kind == NNCV_HIP_OP_DWCONV && p.dw[i]) {
      DwBlockArgs d{};
      const Node* e = nd.expands >= 0 ? &nodes_[i - 1] : nullptr;
      const int src = e ? e->op.in[0] : op.in[0];
      d.in = at(src); d.pix = pitch(src); d.wt = nd.wt.get(); d.scale = nd.scale.as<float>(); d.shift = nd.shift.as<float>(); d.out = at(op.out);
      if (e) {
        d.w1 = e->wt.get(); d.scale1 = e->scale.as<float>(); d.shift1 = e->shift.as<float>();
        d.Cin = p.dims[src].C; d.act1 = e->op.act;
      }
      if (i + 1 < nodes_.size() && p.se[i + 1]) {
        d.parts = static_cast<float*>(at(nodes_[i + 1].op.out));
        d.sq_w = nodes_[i + 2].wt_t.get(); d.SQ = nodes_[i + 2].op.F;
      }
      d.N = N; d.H = a.H; d.W = a.W; d.C = a.C; d.K = op.K; d.stride = op.stride; d.pad = op.pad; d.OH = o.H; d.OW = o.W; d.act = op.act;
      launch_dw_block(d, s);
      continue;
    }
    if (p.se[i]) {
      const Node &f1 = nodes_[i + 1], &f2 = nodes_[i + 2], &pr = nodes_[i + 4];
      SeProjectArgs e{};
      e.x = at(op.in[0]); e.parts = static_cast<const float*>(at(op.out)); e.bands = p.dw[i - 1];
      e.b1 = f1.shift.as<float>(); e.w2t = f2.wt_t.get(); e.b2 = f2.shift.as<float>(); e.act1 = f1.op.act; e.act2 = f2.op.act;
      e.wp_flat = pr.wflat.get(); e.scale = pr.scale.as<float>(); e.shift = pr.shift.as<float>(); e.out = at(pr.op.out);
      e.residual = pr.op.in[1] >= 0 ? at(pr.op.in[1]) : nullptr;
      e.N = N; e.HW = a.H * a.W; e.C = a.C; e.SQ = f1.op.F; e.F = pr.op.F; e.act = pr.op.act;
      launch_se_project(e, s);
      i += 4;
      continue;
    }
    if (nd.se_head) {
      const Node &f1 = nodes_[i + 1], &f2 = nodes_[i + 2];
      SeArgs e{};
      e.x = at(op.in[0]); e.w1 = f1.wt.get(); e.b1 = f1.shift.as<float>(); e.w2 = f2.wt.get(); e.b2 = f2.shift.as<float>();
      e.out = at(nodes_[i + 3].op.out);
      e.N = N; e.HW = a.H * a.W; e.C = a.C; e.SQ = f1.op.F; e.act1 = f1.op.act; e.act2 = f2.op.act;
      launch_se_block(e, dt_, s);
      continue;
    }
    switch (op.kind) {
      case NNCV_HIP_OP_CONV: {
        IgemmArgs g{};
        const int dst = nd.add_out >= 0 ? nd.add_out : op.out;
        g.in = at(op.in[0]); g.wt = nd.wt.get(); g.wt_frag = nd.wfrag.get(); g.wt_frag32 = nd.wfrag32.get(); g.wt_flat = nd.wflat.get(); g.out = at(dst);
        g.scale = nd.scale.as<float>(); g.shift = nd.shift.as<float>();
        g.residual = nd.add_res >= 0 ? at(nd.add_res) : (op.in[1] >= 0 ? at(op.in[1]) : nullptr);
        // padding filters (zero rows, zero scale/shift) are computed like any other: o.C >= op.F
        g.N = N; g.H = a.H; g.W = a.W; g.C = a.C; g.F = o.C; g.R = g.S = op.K; g.OH = o.H; g.OW = o.W;
        g.stride_h = g.stride_w = op.stride; g.pad_h = g.pad_w = op.pad;
        g.relu = nd.add_res >= 0 ? (op.act | kActResidualAfter) : op.act;
        g.ldo = pitch(dst); g.batch = 1;
        if (pairs && (int)i == pair_stem_) {  // the image as [N][H][W/2][2 pixels x 4 channels]
          g.wt = nd.wt_pairs.get();
          g.wt_flat = nullptr;
          g.W = a.W / 2; g.C = 8; g.S = (op.K + (op.pad & 1) + 1) / 2;
          g.stride_w = 1; g.pad_w = (op.pad + 1) / 2;
        }
        if (pitch(op.in[0]) != a.C) {  // the input is a slice of a wider tensor
          g.pix_stride = pitch(op.in[0]);
          const unsigned long long span = (unsigned long long)N * a.H * a.W * g.pix_stride * dtype_size(dt_);
          g.in_bytes = span < 0xffffffffull ? (unsigned)span : 0xffffffffu;
        }
        g.alg_flops = 2.0 * N * o.H * o.W * op.F * (double)op.K * op.K * logical_[op.in[0]];
        launch_igemm(g, dt_, dt_, s);
        break;
      }
      case NNCV_HIP_OP_DWCONV: {
        DwConvArgs d{};
        d.in = at(op.in[0]); d.wt = nd.wt.get(); d.out = at(op.out);
        d.scale = nd.scale.as<float>(); d.shift = nd.shift.as<float>();
        d.N = N; d.H = a.H; d.W = a.W; d.C = a.C; d.K = op.K; d.stride = op.stride; d.pad = op.pad; d.OH = o.H; d.OW = o.W;
        d.act = op.act;
        launch_dwconv(d, dt_, s);
        break;
      }
      case NNCV_HIP_OP_MAXPOOL: {
        // three 5x5 stride-1 pad-2 pools in a row (SPPF): one launch that keeps all three results
        auto pool5 = [&](size_t k, int in) {
          return k < nodes_.size() && !nodes_[k].skip && nodes_[k].op.kind == NNCV_HIP_OP_MAXPOOL && nodes_[k].op.K == 5 &&
                 nodes_[k].op.stride == 1 && nodes_[k].op.pad == 2 && (in < 0 || nodes_[k].op.in[0] == in);
        };
        if (pool5(i, -1) && pool5(i + 1, op.out) && pool5(i + 2, nodes_[i + 1].op.out) && maxpool5_chain3_applicable(dt_, a.H, a.W, a.C)) {
          const int t2 = nodes_[i + 1].op.out, t3 = nodes_[i + 2].op.out;
          launch_maxpool5_chain3(at(op.in[0]), at(op.out), at(t2), at(t3), dt_, N, a.H, a.W, a.C, pitch(op.in[0]), pitch(op.out),
                                 pitch(t2), pitch(t3), s);
          i += 2;
          break;
        }
        launch_maxpool_nhwc(at(op.in[0]), at(op.out), dt_, N, a.H, a.W, a.C, op.K, op.stride, op.pad, s, pitch(op.in[0]),
                            pitch(op.out));
        break;
      }
      case NNCV_HIP_OP_GAVGPOOL:
        launch_global_avgpool_nhwc(at(op.in[0]), at(op.out), dt_, N, a.H * a.W, a.C, s);
        break;
      case NNCV_HIP_OP_SCALE:
        launch_scale_channels(at(op.in[0]), at(op.in[1]), at(op.out), dt_, N, a.H * a.W, a.C, s);
        break;
      case NNCV_HIP_OP_ADD:
        launch_eltwise_pitched(at(op.in[0]), pitch(op.in[0]), at(op.in[1]), pitch(op.in[1]), at(op.out), pitch(op.out), dt_,
                               (long long)N * a.H * a.W, a.C, op.act, s);
        break;
      case NNCV_HIP_OP_ACT:
        launch_eltwise_pitched(at(op.in[0]), pitch(op.in[0]), nullptr, pitch(op.in[0]), at(op.out), pitch(op.out), dt_,
                               (long long)N * a.H * a.W, a.C, op.act, s);
        break;
      case NNCV_HIP_OP_CONCAT: {
        int c0 = 0;
        for (int k = 0; k < 4; ++k) {
          if (op.in[k] < 0) continue;
          const int Ck = p.dims[op.in[k]].C;
          // inputs that live in this tensor already are in place; the others are copied into their slice
          if (view_of_[op.in[k]] != op.out)
            launch_concat_slice(at(op.in[k]), static_cast<char*>(at(op.out)) + (size_t)c0 * dtype_size(dt_), dt_,
                                (long long)N * o.H * o.W, Ck, pitch(op.out), 0, s, pitch(op.in[k]));
          c0 += Ck;
        }
        break;
      }
      case NNCV_HIP_OP_UPSAMPLE2X:
        launch_upsample2x(at(op.in[0]), at(op.out), dt_, N, a.H, a.W, a.C, pitch(op.out), 0, s, pitch(op.in[0]));
        break;
      case NNCV_HIP_OP_YOLO_DETECT: break;  // the last operator: forward_tail
      default: fail("graph: unknown operator kind");
    }
  }
}

void Graph::forward_tail(int N, int H, int W, float* out, void* ws, hipStream_t s) const {
  const Plan& p = plan_of(N, H, W);
  char* base = static_cast<char*>(ws);
  auto at = [&](int t) -> void* { return base + p.offset[t]; };
  const GraphOp& op = nodes_.back().op;
  const Dims o = p.dims[op.out];
  if (op.kind == NNCV_HIP_OP_YOLO_DETECT) {  // decoded straight into the caller's buffer, fp32
    long long box0 = 0;
    if (p.head) {
      DetectHeadArgs d{};
      d.out = out; d.N = N; d.A = op.K; d.F = op.F; d.boxes_total = o.C;
      while (d.levels < 3 && op.in[d.levels] >= 0) ++d.levels;
      for (int k = 0; k < d.levels; ++k) {
        const Node& c = *maker(op.in[k]);
        const int t = c.op.in[0];
        const Dims h = p.dims[t];
        DetectHeadLevel& v = d.lv[d.levels - 1 - k];  // (the later levels are the ones with more channels)
        v.in = at(t); v.wt = c.wfrag.get(); v.scale = c.scale.as<float>(); v.shift = c.shift.as<float>();
        v.HW = h.H * h.W; v.W = h.W; v.pix = pitch(t); v.C = h.C; v.rows = channels_[c.op.out]; v.box0 = box0; v.stride = detect_stride_[k];
        for (int q = 0; q < op.K * 2; ++q) v.anchor_wh[q] = detect_anchor_wh_[k * op.K * 2 + q];
        box0 += (long long)op.K * h.H * h.W;
      }
      launch_detect_head(d, s);
      return;
    }
    for (int k = 0; k < 3 && op.in[k] >= 0; ++k) {
      const Dims h = p.dims[op.in[k]];
      DetectArgs d{};
      d.head = at(op.in[k]); d.out = out; d.N = N; d.H = h.H; d.W = h.W; d.A = op.K; d.F = op.F; d.ldc = pitch(op.in[k]);
      d.box0 = box0; d.boxes_total = o.C; d.stride = detect_stride_[k];
      for (int q = 0; q < op.K * 2; ++q) d.anchor_wh[q] = detect_anchor_wh_[k * op.K * 2 + q];
      launch_yolo_detect(d, dt_, s);
      box0 += (long long)op.K * h.H * h.W;
    }
    return;
  }
  if (p.last_f32) {
    launch_conv_direct(last_args(p, base, out), dt_, s, dt_ == kF16);
    return;
  }
  const int Cl = logical_[op.out];
  launch_relayout(at(op.out), dt_, strides_of(kNHWC, o.C, o.H, o.W), out, kF32, strides_of(kNCHW, Cl, o.H, o.W), N, Cl, Cl, o.H, o.W,
                  false, s);
}

// ---------------------------------------------------------------------------------------------
// MobileNetV3-small, the network of tests/Nets/MobileNetV3.mlir (torchvision's mobilenet_v3_small:
// 52 convolutions of which 11 depthwise, 9 squeeze-excitation blocks, BatchNorm epsilon 1e-3,
// two Linear layers).  Parameter order = state_dict order without num_batches_tracked:
//   conv weight, then BN weight / bias / running_mean / running_var; SE fc1 weight, bias, fc2
//   weight, bias; classifier weight, bias.
// ---------------------------------------------------------------------------------------------
std::vector<GraphOp> mobilenetv3_small_ops(long long* n_elems) {
  std::vector<GraphOp> ops;
  long long off = 0;
  int next = 1;
  const float eps = 1e-3f;
  auto blank = [](int kind) {
    GraphOp o{};
    o.kind = kind;
    o.in[0] = o.in[1] = o.in[2] = o.in[3] = -1;
    o.w = o.bias = o.gamma = o.beta = o.mean = o.var = -1;
    return o;
  };
  // conv / dwconv followed by BatchNorm
  auto conv_bn = [&](int in, int C, int F, int K, int stride, bool depthwise, int act, int residual) {
    GraphOp o = blank(depthwise ? NNCV_HIP_OP_DWCONV : NNCV_HIP_OP_CONV);
    o.in[0] = in; o.in[1] = residual; o.out = next++;
    o.F = F; o.K = K; o.stride = stride; o.pad = (K - 1) / 2; o.act = act; o.eps = eps;
    o.w = off; off += (long long)F * (depthwise ? 1 : C) * K * K;
    o.gamma = off; off += F;
    o.beta = off; off += F;
    o.mean = off; off += F;
    o.var = off; off += F;
    ops.push_back(o);
    return o.out;
  };
  // 1x1 convolution / Linear with bias
  auto fc = [&](int in, int C, int F, int act) {
    GraphOp o = blank(NNCV_HIP_OP_CONV);
    o.in[0] = in; o.out = next++;
    o.F = F; o.K = 1; o.stride = 1; o.pad = 0; o.act = act;
    o.w = off; off += (long long)F * C;
    o.bias = off; off += F;
    ops.push_back(o);
    return o.out;
  };
  auto simple = [&](int kind, int a, int b) {
    GraphOp o = blank(kind);
    o.in[0] = a; o.in[1] = b; o.out = next++;
    ops.push_back(o);
    return o.out;
  };
  auto make_divisible8 = [](int v) {  // torchvision _make_divisible(v, 8)
    int nv = std::max(8, (v + 4) / 8 * 8);
    if (nv * 10 < 9 * v) nv += 8;
    return nv;
  };

  int x = conv_bn(0, 3, 16, 3, 2, false, kActHardSwish, -1);
  struct Cfg { int cin, k, exp, cout, se, hs, stride; };
  const Cfg cfgs[11] = {{16, 3, 16, 16, 1, 0, 2},  {16, 3, 72, 24, 0, 0, 2},  {24, 3, 88, 24, 0, 0, 1},  {24, 5, 96, 40, 1, 1, 2},
                        {40, 5, 240, 40, 1, 1, 1}, {40, 5, 240, 40, 1, 1, 1}, {40, 5, 120, 48, 1, 1, 1}, {48, 5, 144, 48, 1, 1, 1},
                        {48, 5, 288, 96, 1, 1, 2}, {96, 5, 576, 96, 1, 1, 1}, {96, 5, 576, 96, 1, 1, 1}};
  for (const Cfg& c : cfgs) {
    const int act = c.hs ? kActHardSwish : kActRelu;
    const int block_in = x;
    int y = x;
    if (c.exp != c.cin) y = conv_bn(y, c.cin, c.exp, 1, 1, false, act, -1);
    y = conv_bn(y, c.exp, c.exp, c.k, c.stride, true, act, -1);
    if (c.se) {
      const int sq = make_divisible8(c.exp / 4);
      int g = simple(NNCV_HIP_OP_GAVGPOOL, y, -1);
      g = fc(g, c.exp, sq, kActRelu);
      g = fc(g, sq, c.exp, kActHardSigmoid);
      y = simple(NNCV_HIP_OP_SCALE, y, g);
    }
    const bool res = c.stride == 1 && c.cin == c.cout;
    x = conv_bn(y, c.exp, c.cout, 1, 1, false, kActNone, res ? block_in : -1);
  }
  x = conv_bn(x, 96, 576, 1, 1, false, kActHardSwish, -1);
  x = simple(NNCV_HIP_OP_GAVGPOOL, x, -1);
  x = fc(x, 576, 1024, kActHardSwish);
  x = fc(x, 1024, 1000, kActNone);
  if (n_elems) *n_elems = off;
  return ops;
}

}  // namespace nncv_hip
