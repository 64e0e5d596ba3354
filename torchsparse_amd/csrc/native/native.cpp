// Native host path: stages of convolutions - what a network applies between two places where Python
// has something to decide - carried out by one call each.
//
// A convolution called through its module costs the host several times its launch (module calls, cache look-ups,
// argument conversion; in training six autograd nodes and a dozen launches made from Python).  Host time of the
// 42-layer U-Net on an 80k-voxel scan, through modules and through stages: inference 1.23 -> 0.76 ms, a training
// step 11.6 -> 4.8 ms (11.3 -> 7.1 ms with the device, which then is what bounds it).
// Here a stage is compiled once into a list of operations over numbered buffers; a call gets the
// stage's input and its kernel maps, allocates from torch's allocator, and launches through the library's
// C ABI without the interpreter.  In training the stage is ONE autograd node, whose backward walks the
// list the other way.
#include <ATen/ATen.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <pybind11/pybind11.h>
#include <pybind11/stl.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/autograd/variable.h>
#include <torch/csrc/utils/pybind.h>

#include <map>
#include <memory>
#include <mutex>
#include <string>
#include <tuple>
#include <vector>

#include "../../../include/tsmi.h"

namespace py = pybind11;
using at::Tensor;

namespace {

void check(int status) {
  if (status == TSMI_OK) return;
  const char *msg = tsmi_last_error();
  if (status == TSMI_ERR_INVALID_ARGUMENT) throw py::value_error(msg);
  throw std::runtime_error(msg);
}

tsmi_stream_t stream_of(const Tensor &t) {
  return (tsmi_stream_t)c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream();
}

int dtype_code(const Tensor &t) {
  switch (t.scalar_type()) {
    case at::kFloat: return TSMI_F32;
    case at::kHalf: return TSMI_F16;
    case at::kBFloat16: return TSMI_BF16;
    default: throw py::value_error("unsupported feature dtype");
  }
}

int64_t ceil128(int64_t n) { return (n + 127) / 128 * 128; }

// Rows of x in whole 16-byte pieces (what the fast kernels load): with zero columns appended where they are not.
Tensor whole_pieces(const Tensor &x) {
  const int64_t per = 16 / x.element_size(), c = x.size(1);
  if (c % per == 0) return x;
  Tensor y = at::empty({x.size(0), (c + per - 1) / per * per}, x.options());
  check(tsmi_pad_columns(stream_of(x), x.data_ptr(), x.size(0), (int)c, dtype_code(x), y.data_ptr()));
  return y;
}

Tensor ints(int64_t n, const Tensor &like) { return at::empty({n}, like.options().dtype(at::kInt)); }
Tensor floats(int64_t n, const Tensor &like) { return at::empty({n}, like.options().dtype(at::kFloat)); }

// What the calls queued on one stream share: scratch for partial sums and products - every launch writes
// before it reads, and a stream runs its launches one after the other - and counters that every launch
// leaves zero.  The lock is held while a call that uses them queues its launches.
struct Scratch {
  Tensor bytes, counters;
  void *need(int64_t n, const Tensor &like) {
    if (!bytes.defined() || bytes.numel() < n)
      bytes = at::empty({std::max<int64_t>(n, 1 << 20)}, like.options().dtype(at::kByte));
    return bytes.data_ptr();
  }
};
constexpr int64_t kPadNarrowRows = 131072;
constexpr int64_t kCounters = 4096;
std::mutex g_scratch_lock;
std::map<std::tuple<int, void *, bool>, Scratch> g_scratch;

// (g_scratch_lock held.  Calls that go to the launch thread have scratch of their own: another host thread's
// launches may fall between the launches of one of them.)
Scratch &scratch_of(const Tensor &like, tsmi_stream_t s, bool handed_over = false) {
  Scratch &sc = g_scratch[{like.device().index(), s, handed_over}];
  if (!sc.counters.defined()) sc.counters = at::zeros({kCounters}, like.options().dtype(at::kInt));
  return sc;
}

void release_scratch() {
  std::lock_guard<std::mutex> hold(g_scratch_lock);
  g_scratch.clear();
}

// ------------------------------------------------------------------------------ kernel maps

// A kernel map and what has been derived from it, in both directions: rows of `map` (or of `map_t`) to the
// input rows they gather from.  No map and a kernel volume of one: the identity of a 1x1x1 layer.
struct KernelMap {
  int kvol = 1;
  int64_t n_in = 0, n_out = 0;
  bool symmetric = false;  // a submanifold map over distinct rows: its own transposed map, offsets mirrored
  Tensor map, map_t;
  // pair segments of `map` (tsmi_pair_segments), where its layers are to run over them
  Tensor segments;
  int64_t seg_in = 0, seg_counts = 0, seg_pos = 0, seg_rows = 0;
  double density = 0;  // pairs per entry as far as it is known
  // grouped copy of `map` (tsmi_map_group_rows)
  Tensor grouped;
  std::vector<int64_t> grouped_at;
  int64_t grouped_rows = 0;
  // pair lists of the gather-scatter ([nnz, 2]) and fetch-on-demand ([2, nnz]) dataflows, each offset's first
  // pair, the same in whole tiles, and per row and offset its product (of outputs, and of inputs for a transposed layer)
  Tensor lists, list_at, list_tiles, list_of_out, list_of_in;
  int64_t list_tiled = 0;
  bool list_planar = false, centered = false;
  // pair lists of the weight gradient
  Tensor pairs, seg_steps;
  int64_t pair_cap = 0;
  std::mutex lock;

  const Tensor &transposed(tsmi_stream_t s) {
    std::lock_guard<std::mutex> hold(lock);
    if (!map_t.defined()) {
      map_t = at::empty({ceil128(n_in), kvol}, map.options());
      check(tsmi_transpose_map(s, map.data_ptr<int32_t>(), n_out, kvol, map_t.data_ptr<int32_t>(), map_t.size(0)));
    }
    return map_t;
  }
  void need_pairs(tsmi_stream_t s) {
    std::lock_guard<std::mutex> hold(lock);
    if (pairs.defined()) return;
    pair_cap = tsmi_wgrad_pairs_capacity(n_out, kvol);
    pairs = ints(2 * std::max<int64_t>(pair_cap, 1), map);
    Tensor work = ints(kvol * std::max<int64_t>((n_out + 255) / 256, 1) + kvol, map);
    seg_steps = ints(kvol + 1, map);
    check(tsmi_wgrad_pairs_build(s, map.data_ptr<int32_t>(), n_out, kvol, work.data_ptr<int32_t>() + kvol,
                                 work.data_ptr<int32_t>(), pairs.data_ptr<int32_t>(), seg_steps.data_ptr<int32_t>()));
  }
};
using Map = std::shared_ptr<KernelMap>;

// ------------------------------------------------------------------------------ one convolution

struct Place {  // columns [first, first + cout) of a wider contiguous buffer
  Tensor buffer;
  int64_t first = 0;
};

struct Rules {  // the module-wide switches the Python layer would have looked at
  bool segments = false;     // pair segments where the map has them
  bool lists = false;        // the forward in the dataflow of the map's pair lists
  int64_t group_min_rows = 0;
};

// Calls handed to the library's launch thread (tsmi_launch_thread_submit) instead of made, and what they read and
// write, which has to stay until the last of them has been carried out.
struct Pending {
  int64_t ticket = 0;
  std::vector<Tensor> tensors;
  std::vector<Map> maps;
  std::shared_ptr<void> stage;
  ~Pending() {  // (a call that ended in an exception: what it had handed over still runs)
    const int64_t *done = tsmi_launch_thread_completed();
    while (__atomic_load_n(done, __ATOMIC_ACQUIRE) < ticket) __builtin_ia32_pause();
  }
};

void make(const tsmi_conv_call &c, Pending *pending) {
  if (pending) {
    const int64_t ticket = tsmi_launch_thread_submit(3, reinterpret_cast<const int64_t *>(&c), sizeof(c) / 8);
    if (ticket > 0) {
      pending->ticket = ticket;
      return;
    }
    check(tsmi_launch_thread_flush());  // (no region any more)
  }
  check(tsmi_conv(&c));
}

// y (rows of `map`, or with `backward` of its transposed direction) = act(conv(x) + bias + residual).
// `w`: packed weights, the reduction axis contiguous.
Tensor convolve(KernelMap &m, bool transposed, bool backward, const Tensor &x0, const void *w, int cin, int cout,
                const Tensor &bias, const Tensor &residual, bool relu, const Rules &rules, const Place *out,
                const Place *also, Pending *pending = nullptr) {
  tsmi_conv_call c{};
  Tensor x = x0;
  cin = (int)x.size(1);  // (a gradient may come in whole pieces)
  // (16-bit layers of up to 8 channels have a kernel that takes any number, but over many rows the one for whole
  // pieces is ahead by more than the copy: 4 -> 32 over 320k rows 52 us, 4 + 23.  Packed weights are padded already.)
  if (cin * x.element_size() % 16 != 0 &&
      (x.element_size() != 2 || cin > 8 || (x.size(0) >= kPadNarrowRows && tsmi_conv_streams(m.kvol, 8, cout, dtype_code(x))))) {
    if (pending) check(tsmi_launch_thread_flush());
    x = whole_pieces(x0);
    cin = (int)x.size(1);
    if (pending) pending->tensors.push_back(x);
  }
  c.stream = stream_of(x);
  c.x = x.data_ptr();
  c.w_packed = w;
  c.bias = bias.defined() ? bias.data_ptr() : nullptr;
  c.residual = residual.defined() ? residual.data_ptr() : nullptr;
  c.relu = relu;
  c.dtype = dtype_code(x);
  c.n_in = x.size(0);
  c.kvol = m.kvol;
  c.cin = cin;
  c.cout = cout;
  // direction of the walk: a transposed layer goes from the map's outputs to its inputs, a gradient back
  const bool to_inputs = transposed != backward;
  c.n_out = to_inputs ? m.n_in : m.n_out;
  const bool mirrored = to_inputs && m.symmetric;
  c.mirrored = mirrored;
  const int64_t es = x.element_size();
  Tensor y;
  if (out && out->buffer.defined()) {
    y = out->buffer;
    c.y = (char *)y.data_ptr() + out->first * es;
    c.ldy = y.size(1);
  } else {
    y = at::empty({c.n_out, cout}, x.options());
    c.y = y.data_ptr();
  }
  if (also && also->buffer.defined()) {
    c.y2 = (char *)also->buffer.data_ptr() + also->first * es;
    c.ldy2 = also->buffer.size(1);
  }
  if (c.n_out == 0) return y;
  if (x.size(0) == 0) {  // (no inputs: every sum is empty; the kernels take no null features)
    TORCH_CHECK(!(out && out->buffer.defined()), "a placed result of an empty input");
    if (pending) check(tsmi_launch_thread_flush());
    y.zero_();
    if (bias.defined()) y.add_(bias);
    if (residual.defined()) y.add_(residual);
    if (relu) y.relu_();
    return y;
  }
  const bool own_map = !to_inputs || mirrored;
  if (own_map && rules.segments && m.segments.defined() &&
      tsmi_conv_segments_pay(c.n_out, m.kvol, cin, cout, c.dtype, m.density)) {
    c.in_rows = (const int32_t *)m.seg_in;
    c.counts = (const int32_t *)m.seg_counts;
    c.pos = (const int32_t *)m.seg_pos;
    c.seg_rows = m.seg_rows;
    std::lock_guard<std::mutex> hold(g_scratch_lock);
    Scratch &sc = scratch_of(x, c.stream, pending);
    c.products = sc.need(m.kvol * m.seg_rows * cout * es, x);
    if (pending) pending->tensors.push_back(sc.bytes);
    make(c, pending);
    return y;
  }
  if (own_map && m.grouped.defined() && m.kvol == 27 && c.n_out >= rules.group_min_rows && cin > 8 &&
      !tsmi_conv_streams(m.kvol, cin, cout, c.dtype) &&
      cin * es % 16 == 0 && (cout < 128 || c.n_out >= 65536)) {
    c.grouped = (const int32_t *)m.grouped_at[0];
    c.row_of = (const int32_t *)m.grouped_at[1];
    c.order64 = (const int32_t *)m.grouped_at[3];
    c.order128 = (const int32_t *)m.grouped_at[4];
    c.n_grouped = m.grouped_rows;
    make(c, pending);
    return y;
  }
  if (m.kvol == 1 && !m.map.defined()) {
    c.n_map_rows = c.n_out;
  } else {
    const Tensor &map = own_map ? m.map : m.transposed(c.stream);
    c.map = map.data_ptr<int32_t>();
    c.n_map_rows = map.size(0);
  }
  if (c.n_out < 65536) {  // (only maps with few row tiles use the offset split)
    const int64_t ws = tsmi_conv_workspace_elems(c.n_out, c.n_out, m.kvol, 1, cin, cout, c.dtype, 0);
    if (ws > 0) {
      std::lock_guard<std::mutex> hold(g_scratch_lock);
      Scratch &sc = scratch_of(x, c.stream, pending);
      c.workspace = (float *)sc.need(4 * ws, x);
      c.workspace_elems = ws;
      c.tile_counters = sc.counters.data_ptr<int32_t>();
      c.n_tile_counters = kCounters;
      if (pending) pending->tensors.push_back(sc.bytes);
      make(c, pending);
      return y;
    }
  }
  make(c, pending);
  return y;
}

// y = conv(x) in the dataflow of the map's pair lists.  Small training layers are bound by the host: 13 -> 64
// channels, 5.3k rows, fp16, forward and backward 177 us from Python, 90 as a stage (32 -> 32, 16k rows, fp32: 135, 70).
Tensor convolve_lists(KernelMap &m, bool transposed, const Tensor &x0, const void *w, int cout) {
  const Tensor x = whole_pieces(x0);
  const int64_t n_out = transposed ? m.n_in : m.n_out, nnz = m.lists.numel() / 2;
  Tensor y = at::empty({n_out, cout}, x.options());
  const Tensor products = at::empty({std::max<int64_t>(nnz, 1), cout}, x.options());
  // (the masks of an odd submanifold map leave its identity offset out)
  const int center = m.centered ? m.kvol / 2 : -1;
  const auto forward = m.list_planar ? tsmi_conv_fetch_on_demand : tsmi_gs_forward;
  check(forward(stream_of(x), x.data_ptr(), w, m.lists.data_ptr<int32_t>(), nnz, m.list_at.data_ptr<int32_t>(),
                m.list_tiles.data_ptr<int32_t>(), m.list_tiled,
                (transposed ? m.list_of_in : m.list_of_out).data_ptr<int32_t>(), n_out, m.kvol, (int)x.size(1), cout,
                dtype_code(x), transposed, center, nullptr, nullptr, 0, products.data_ptr(), y.data_ptr()));
  return y;
}

// ------------------------------------------------------------------------------ stages

struct Norm {
  int gamma = -1, beta = -1;  // parameters (-1: not affine)
  Tensor running_mean, running_var, batches;
  double momentum = 0.1, eps = 1e-5;
};

// dst = act(norm(conv(src)) + residual); buffer 0 is the stage's input.
struct Op {
  int src = 0, dst = 0, residual = -1;
  int map = 0;
  bool transposed = false, relu = false, has_norm = false;
  int weight = 0, bias = -1;  // parameters
  int kvol = 1, cin = 0, cout = 0;
  Norm norm;
};

struct Packed {
  Tensor data;
  uint32_t version = 0;
  const void *at = nullptr;  // of the weight it was made from
};

struct Stage {
  std::vector<Op> ops;
  std::vector<Tensor> params;
  std::vector<Packed> packed;  // per operation
  int buffers = 1;

  // Whether the backward reads the last result (the caller may write over it otherwise): a residual layer's mask.
  bool needs_output() const { return ops.back().has_norm && ops.back().relu && ops.back().residual >= 0; }

  void fits(const Tensor &x, const std::vector<Map> &maps) const {
    TORCH_CHECK(!ops.empty() && x.dim() == 2 && x.is_contiguous() && x.size(1) == ops[0].cin, "stage: another input");
    for (const Op &op : ops) {
      TORCH_CHECK(op.map < (int)maps.size() && maps[op.map] && maps[op.map]->kvol == op.kvol, "stage: another map");
      if (op.src == 0)
        TORCH_CHECK(x.size(0) == (op.transposed ? maps[op.map]->n_out : maps[op.map]->n_in),
                    "stage: a map over another number of rows");
    }
  }

  // Packed weights of every operation whose weight has changed since, in one launch.
  void pack(tsmi_stream_t s) {
    std::vector<const void *> from;
    std::vector<void *> to;
    std::vector<int32_t> shapes;
    std::vector<size_t> stale;
    std::vector<int64_t> sizes;
    int64_t total = 0;
    packed.resize(ops.size());
    for (size_t i = 0; i < ops.size(); ++i) {
      const Tensor &w = params[ops[i].weight];
      const uint32_t version = w._version();
      if (packed[i].data.defined() && packed[i].version == version && packed[i].at == w.data_ptr() &&
          packed[i].data.scalar_type() == w.scalar_type())
        continue;
      packed[i].version = version;
      packed[i].at = w.data_ptr();
      stale.push_back(i);
      sizes.push_back((tsmi_packed_weight_elems(ops[i].kvol, ops[i].cin, ops[i].cout) + 63) / 64 * 64);
      total += sizes.back();
    }
    if (stale.empty()) return;
    const Tensor all = at::empty({total}, params[ops[0].weight].options().requires_grad(false));
    int64_t first = 0;
    for (size_t j = 0; j < stale.size(); ++j) {
      const Op &op = ops[stale[j]];
      packed[stale[j]].data = all.narrow(0, first, sizes[j]);
      first += sizes[j];
      from.push_back(packed[stale[j]].at);
      to.push_back(packed[stale[j]].data.data_ptr());
      shapes.insert(shapes.end(), {op.kvol, op.cin, op.cout});
    }
    check(tsmi_pack_weights_many(s, from.data(), to.data(), shapes.data(), (int)stale.size(), dtype_code(all)));
  }

  // Inference: the output of the last operation.  `placed` / `place`: operation whose result is written into
  // columns of a wider buffer, which is its destination from there on; `also`: a second place for the last one's.
  Tensor run(const Tensor &x, const std::vector<Map> &maps, const Rules &rules, int placed, const Place &place,
             const Place &also, Pending *pending) {
    fits(x, maps);
    at::AutoDispatchBelowADInplaceOrView below;  // (nothing here is recorded)
    pack(stream_of(x));
    std::vector<Tensor> buf(buffers);
    buf[0] = x;
    Tensor y;
    for (size_t i = 0; i < ops.size(); ++i) {
      const Op &op = ops[i];
      const Tensor none;
      y = convolve(*maps[op.map], op.transposed, false, buf[op.src], packed[i].data.data_ptr(), op.cin, op.cout,
                   op.bias >= 0 ? params[op.bias] : none, op.residual >= 0 ? buf[op.residual] : none, op.relu, rules,
                   (int)i == placed ? &place : nullptr, i + 1 == ops.size() ? &also : nullptr, pending);
      buf[op.dst] = y;
    }
    if (pending) {
      for (const Packed &w : packed) buf.push_back(w.data);
      for (const Tensor &t : {place.buffer, also.buffer})
        if (t.defined()) buf.push_back(t);
      pending->tensors.insert(pending->tensors.end(), buf.begin(), buf.end());
      pending->maps = maps;
    }
    return y;
  }
};

// dW [kvol, cin, cout] of a convolution from its input and its output's gradient.
Tensor weight_grad(KernelMap &m, bool transposed, const Tensor &x0, const Tensor &dy0, int cin, int cout) {
  const Tensor x = whole_pieces(x0), dy = whole_pieces(dy0);
  const int ci = (int)x.size(1), co = (int)dy.size(1), code = dtype_code(x);
  const tsmi_stream_t s = stream_of(x);
  Tensor dw = at::empty({m.kvol, ci, co}, x.options());
  const bool pointwise = m.kvol == 1 && !m.map.defined();
  if (!pointwise) m.need_pairs(s);
  const int64_t cap = pointwise ? x.size(0) : m.pair_cap;
  const int64_t elems = tsmi_conv_wgrad_pairs_workspace_elems(cap, m.kvol, ci, co, code);
  {
    std::lock_guard<std::mutex> hold(g_scratch_lock);
    float *ws = (float *)scratch_of(x, s).need(4 * std::max<int64_t>(elems, 1), x);
    if (pointwise)
      check(tsmi_conv_wgrad_pointwise(s, x.data_ptr(), dy.data_ptr(), x.size(0), ci, co, code, ws, elems,
                                      dw.data_ptr()));
    else
      check(tsmi_conv_wgrad_pairs(s, x.data_ptr(), dy.data_ptr(), m.pairs.data_ptr<int32_t>(),
                                  m.seg_steps.data_ptr<int32_t>(), cap, transposed ? 1 : 0, m.kvol, ci, co, code, ws,
                                  elems, dw.data_ptr()));
  }
  if (ci == cin && co == cout) return dw;
  return dw.narrow(1, 0, cin).narrow(2, 0, cout).contiguous();
}

// dX = sum_k dY W[k]^T (+ more).
Tensor input_grad(KernelMap &m, bool transposed, const Tensor &dy, const Tensor &weight, int cin, int cout,
                  const Tensor &more, const Rules &rules) {
  // the packed layout of W[k]^T is W[k] itself when neither channel count needs padding
  const void *w = weight.data_ptr();
  Tensor packed;
  if (tsmi_packed_weight_elems(m.kvol, cout, cin) != weight.numel()) {
    packed = at::empty({tsmi_packed_weight_elems(m.kvol, cout, cin)}, weight.options().requires_grad(false));
    check(tsmi_pack_weights_turned(stream_of(dy), weight.data_ptr(), packed.data_ptr(), m.kvol, cout, cin,
                                   dtype_code(dy)));
    w = packed.data_ptr();
  }
  return convolve(m, transposed, true, dy, w, cout, cin, Tensor(), more, false, rules, nullptr, nullptr);
}

// ------------------------------------------------------------------------------ training

struct StageNode : public torch::autograd::Node {
  std::shared_ptr<Stage> stage;
  std::vector<Map> maps;
  Rules rules;
  std::vector<torch::autograd::SavedVariable> params;
  torch::autograd::SavedVariable input, output;
  std::vector<Tensor> buf;        // results of the operations but the last (buffer 0 and it are saved above)
  std::vector<Tensor> conv_out;   // what the norms were applied to
  std::vector<Tensor> stats;
  std::mutex once;
  bool released = false;

  std::string name() const override { return "SparseStageBackward"; }
  void release_variables() override {
    std::lock_guard<std::mutex> hold(once);
    for (auto &p : params) p.reset_data();
    input.reset_data();
    output.reset_data();
    buf.clear();
    conv_out.clear();
    stats.clear();
    released = true;
  }
  torch::autograd::variable_list apply(torch::autograd::variable_list &&grads) override;
};

torch::autograd::variable_list StageNode::apply(torch::autograd::variable_list &&grads) {
  std::lock_guard<std::mutex> hold(once);
  TORCH_CHECK(!released, "Trying to backward through the graph a second time (or directly access saved tensors "
                         "after they have already been freed).");
  const auto &ops = stage->ops;
  const size_t n_params = stage->params.size();
  torch::autograd::variable_list result(1 + n_params);
  if (!grads[0].defined()) return result;
  at::AutoDispatchBelowADInplaceOrView below;
  std::vector<Tensor> value = buf, weights(n_params);
  value[0] = input.unpack();
  if (stage->needs_output()) value[ops.back().dst] = output.unpack(shared_from_this());
  for (size_t i = 0; i < n_params; ++i) weights[i] = params[i].unpack();
  std::vector<Tensor> grad(stage->buffers);
  Tensor top = grads[0].contiguous();
  if (top.scalar_type() != value[0].scalar_type()) top = top.to(value[0].scalar_type());
  grad[ops.back().dst] = top;
  const Tensor &x = value[0];
  const tsmi_stream_t s = stream_of(x);
  const int code = dtype_code(x);
  for (int i = (int)ops.size() - 1; i >= 0; --i) {
    const Op &op = ops[i];
    Tensor g = grad[op.dst];
    grad[op.dst] = Tensor();
    if (!g.defined()) continue;
    KernelMap &m = *maps[op.map];
    const int64_t n = g.size(0);
    if (op.has_norm) {
      const Tensor &c = conv_out[i];
      const int ch = op.cout;
      const Tensor &w = op.norm.gamma >= 0 ? weights[op.norm.gamma] : c;
      const Tensor work = floats(tsmi_bn_partial_elems(ch) + 2 * ch, x);
      float *partial = work.data_ptr<float>(), *sums = partial + tsmi_bn_partial_elems(ch);
      Tensor pg;
      if (op.norm.gamma >= 0) pg = at::empty({2 * ch}, w.options().requires_grad(false));
      Tensor dz, dconv = at::empty_like(c);
      if (op.residual >= 0 && op.relu) dz = at::empty_like(c);
      check(tsmi_bn_backward(s, g.data_ptr(), c.data_ptr(),
                             op.relu && op.residual >= 0 ? value[op.dst].data_ptr() : nullptr, n, ch, code, op.relu,
                             op.norm.gamma >= 0 ? w.data_ptr() : nullptr, dtype_code(w), stats[i].data_ptr<float>(),
                             partial, sums, pg.defined() ? pg.data_ptr() : nullptr,
                             dz.defined() ? dz.data_ptr() : nullptr, dconv.data_ptr()));
      if (op.norm.gamma >= 0) result[1 + op.norm.gamma] = pg.narrow(0, ch, ch);
      if (op.norm.beta >= 0) result[1 + op.norm.beta] = pg.narrow(0, 0, ch);
      if (op.residual >= 0) {
        Tensor &r = grad[op.residual];
        const Tensor &add = dz.defined() ? dz : g;
        r = r.defined() ? at::add(r, add) : add;
      }
      g = dconv;
    }
    if (g.size(1) * g.element_size() % 16 != 0) g = whole_pieces(g);  // (once for both gradients)
    if (task_should_compute_output(1 + op.weight)) {
      Tensor dw = weight_grad(m, op.transposed, value[op.src], g, op.cin, op.cout);
      result[1 + op.weight] = dw.view(weights[op.weight].sizes());
    }
    if (op.src != 0 || task_should_compute_output(0))
      grad[op.src] = input_grad(m, op.transposed, g, weights[op.weight], op.cin, op.cout, grad[op.src], rules);
  }
  if (task_should_compute_output(0)) result[0] = grad[0];
  return result;
}

// Forward in training mode: every convolution followed by its norm (batch statistics), activation and shortcut.
Tensor train_stage(const std::shared_ptr<Stage> &stage, const Tensor &x, const std::vector<Map> &maps,
                   const Rules &rules) {
  stage->fits(x, maps);
  auto node = std::shared_ptr<StageNode>(new StageNode(), torch::autograd::deleteNode);
  torch::autograd::variable_list inputs{x};
  inputs.insert(inputs.end(), stage->params.begin(), stage->params.end());
  const bool record = torch::autograd::compute_requires_grad(inputs);
  Tensor y;
  {
    at::AutoDispatchBelowADInplaceOrView below;
    const tsmi_stream_t s = stream_of(x);
    const int code = dtype_code(x);
    stage->pack(s);
    const auto &ops = stage->ops;
    node->buf.resize(stage->buffers);
    node->conv_out.resize(ops.size());
    node->stats.resize(ops.size());
    std::vector<Tensor> buf(stage->buffers);
    buf[0] = x;
    for (size_t i = 0; i < ops.size(); ++i) {
      const Op &op = ops[i];
      const Tensor none;
      KernelMap &m = *maps[op.map];
      const void *w = stage->packed[i].data.data_ptr();
      Tensor c = rules.lists && m.map.defined()
                     ? convolve_lists(m, op.transposed, buf[op.src], w, op.cout)
                     : convolve(m, op.transposed, false, buf[op.src], w, op.cin, op.cout, none, none, false, rules,
                                nullptr, nullptr);
      y = c;
      if (op.has_norm) {
        const Norm &nm = op.norm;
        const int ch = op.cout;
        y = at::empty_like(c);
        const Tensor work = floats(tsmi_bn_partial_elems(ch), x);
        node->stats[i] = floats(4 * ch, x);
        const Tensor &kind = nm.gamma >= 0 ? stage->params[nm.gamma] : nm.running_mean.defined() ? nm.running_mean : c;
        check(tsmi_bn_forward_train(
            s, c.data_ptr(), c.size(0), ch, code, nm.gamma >= 0 ? stage->params[nm.gamma].data_ptr() : nullptr,
            nm.beta >= 0 ? stage->params[nm.beta].data_ptr() : nullptr, dtype_code(kind),
            nm.running_mean.defined() ? nm.running_mean.data_ptr() : nullptr,
            nm.running_var.defined() ? nm.running_var.data_ptr() : nullptr,
            nm.batches.defined() ? nm.batches.data_ptr<int64_t>() : nullptr, (float)nm.momentum, (float)nm.eps,
            op.residual >= 0 ? buf[op.residual].data_ptr() : nullptr, op.relu, work.data_ptr<float>(),
            node->stats[i].data_ptr<float>(), y.data_ptr()));
      }
      buf[op.dst] = y;
      if (record) node->conv_out[i] = op.has_norm ? c : Tensor();
      if (record && i + 1 < ops.size()) node->buf[op.dst] = y;
    }
  }
  if (record) {
    node->stage = stage;
    node->maps = maps;
    node->rules = rules;
    node->set_next_edges(torch::autograd::collect_next_edges(inputs));
    node->input = torch::autograd::SavedVariable(x, false);
    for (const Tensor &p : stage->params) node->params.emplace_back(p, false);
    torch::autograd::set_history(y, node);
    if (stage->needs_output()) node->output = torch::autograd::SavedVariable(y, true);
  }
  return y;
}

// ------------------------------------------------------------------------------ binding

Place place_of(const py::object &slice) {  // None or (buffer, first column)
  if (slice.is_none()) return {};
  const auto t = slice.cast<std::pair<Tensor, int64_t>>();
  return {t.first, t.second};
}

}  // namespace

PYBIND11_MODULE(_native, mod) {
  mod.def("release_scratch", &release_scratch);
  py::class_<KernelMap, Map>(mod, "KernelMap")
      .def(py::init([](int kvol, int64_t n_in, int64_t n_out, bool symmetric, std::optional<Tensor> map,
                       std::optional<Tensor> map_t) {
        auto m = std::make_shared<KernelMap>();
        m->kvol = kvol, m->n_in = n_in, m->n_out = n_out, m->symmetric = symmetric;
        if (map) m->map = *map;
        if (map_t) m->map_t = *map_t;
        TORCH_CHECK(map || kvol == 1, "a kernel map needs its table");
        TORCH_CHECK(!map || (map->is_contiguous() && map->scalar_type() == at::kInt && map->size(0) >= n_out &&
                             map->size(1) == kvol), "kernel map of another shape");
        TORCH_CHECK(!map_t || (map_t->is_contiguous() && map_t->scalar_type() == at::kInt && map_t->size(0) >= n_in &&
                               map_t->size(1) == kvol), "transposed kernel map of another shape");
        return m;
      }))
      .def("set_transposed", [](KernelMap &m, Tensor map_t) { m.map_t = std::move(map_t); })
      .def_property_readonly("has_transposed", [](const KernelMap &m) { return m.map_t.defined(); })
      .def_property_readonly("has_segments", [](const KernelMap &m) { return m.segments.defined(); })
      .def_property_readonly("has_grouped", [](const KernelMap &m) { return m.grouped.defined(); })
      .def("set_segments",
           [](KernelMap &m, Tensor buffer, int64_t in, int64_t counts, int64_t pos, int64_t rows, double density) {
             m.density = density;
             m.segments = std::move(buffer);
             m.seg_in = in, m.seg_counts = counts, m.seg_pos = pos, m.seg_rows = rows;
           })
      .def("set_lists",
           [](KernelMap &m, bool planar, Tensor lists, Tensor at, Tensor tiles, int64_t tiled, Tensor of_out,
              Tensor of_in, bool centered) {
             for (const Tensor &t : {lists, at, tiles, of_out, of_in})
               TORCH_CHECK(t.is_contiguous() && t.scalar_type() == at::kInt && t.device() == m.map.device(),
                           "pair lists are int32 on the map's device");
             TORCH_CHECK(lists.dim() == 2 && lists.size(planar ? 0 : 1) == 2 && at.numel() == m.kvol + 1 &&
                         tiles.numel() == m.kvol + 1 && of_out.numel() >= m.n_out * m.kvol &&
                         of_in.numel() >= m.n_in * m.kvol, "pair lists of another map");
             m.list_planar = planar, m.centered = centered, m.list_tiled = tiled;
             m.lists = std::move(lists), m.list_at = std::move(at), m.list_tiles = std::move(tiles);
             m.list_of_out = std::move(of_out), m.list_of_in = std::move(of_in);
           })
      .def_property_readonly("lists", [](const KernelMap &m) { return !m.lists.defined() ? 0 : m.list_planar ? 2 : 1; })
      .def("set_grouped", [](KernelMap &m, Tensor buffer, std::vector<int64_t> at, int64_t rows) {
        TORCH_CHECK(at.size() == 5, "a grouped map has five parts");
        m.grouped = std::move(buffer);
        m.grouped_at = std::move(at);
        m.grouped_rows = rows;
      });
  py::class_<Pending>(mod, "Pending").def(py::init<>()).def_readonly("ticket", &Pending::ticket);
  py::class_<Stage, std::shared_ptr<Stage>>(mod, "Stage")
      .def(py::init([](std::vector<Tensor> params, int buffers) {
        auto st = std::make_shared<Stage>();
        st->params = std::move(params);
        st->buffers = buffers;
        return st;
      }))
      .def_readonly("params", &Stage::params)
      // (src, dst, residual, map, transposed, relu, weight, bias, kvol, cin, cout)
      .def("add", [](Stage &st, int src, int dst, int residual, int map, bool transposed, bool relu, int weight,
                     int bias, int kvol, int cin, int cout) {
        Op op;
        op.src = src, op.dst = dst, op.residual = residual, op.map = map, op.transposed = transposed;
        op.relu = relu, op.weight = weight, op.bias = bias, op.kvol = kvol, op.cin = cin, op.cout = cout;
        const int n = (int)st.params.size();
        TORCH_CHECK(src >= 0 && src < st.buffers && dst > 0 && dst < st.buffers && residual < st.buffers && map >= 0 &&
                    weight >= 0 && weight < n && bias < n, "stage: an operation outside its stage");
        TORCH_CHECK(st.params[weight].numel() == (int64_t)kvol * cin * cout && st.params[weight].is_contiguous() &&
                    (bias < 0 || st.params[bias].numel() == cout), "stage: parameters of another shape");
        st.ops.push_back(std::move(op));
      })
      .def("norm", [](Stage &st, int gamma, int beta, std::optional<Tensor> mean, std::optional<Tensor> var,
                      std::optional<Tensor> batches, double momentum, double eps) {
        TORCH_CHECK(!st.ops.empty() && gamma < (int)st.params.size() && beta < (int)st.params.size(),
                    "stage: a norm outside its stage");
        const int64_t ch = st.ops.back().cout;
        TORCH_CHECK((gamma < 0 || st.params[gamma].numel() == ch) && (beta < 0 || st.params[beta].numel() == ch) &&
                    (!mean || mean->numel() == ch) && (!var || var->numel() == ch), "stage: a norm of another width");
        Norm &nm = st.ops.back().norm;
        st.ops.back().has_norm = true;
        nm.gamma = gamma, nm.beta = beta, nm.momentum = momentum, nm.eps = eps;
        if (mean) nm.running_mean = *mean;
        if (var) nm.running_var = *var;
        if (batches) nm.batches = *batches;
      })
      .def("run",
           [](const std::shared_ptr<Stage> &st, const Tensor &x, const std::vector<Map> &maps, bool segments,
              int64_t group_min_rows, int placed, const py::object &place, const py::object &also, Pending *pending) {
             const Place p = place_of(place), a = place_of(also);
             if (pending) pending->stage = st;
             py::gil_scoped_release free;
             return st->run(x, maps, Rules{segments, false, group_min_rows}, placed, p, a, pending);
           })
      .def("train", [](const std::shared_ptr<Stage> &st, const Tensor &x, const std::vector<Map> &maps, bool segments,
                       bool lists, int64_t group_min_rows) {
        for (const Map &m : maps)
          TORCH_CHECK(!lists || !m->map.defined() || m->lists.defined(), "a kernel map without pair lists");
        py::gil_scoped_release free;
        return train_stage(st, x, maps, Rules{segments, lists, group_min_rows});
      });
}
