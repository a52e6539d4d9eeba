// PyTorch-ROCm binding: module `grouped_gemm_backend`, one function
// gmm(a, b, c, batch_sizes, trans_a, trans_b) -> None, the same entry point the
// reference's extension exports (csrc/ops.cu:7-9, csrc/grouped_gemm.h:5-9).
//
// All tensor validation lives here, in the order of the reference's checks
// (csrc/grouped_gemm.cu:470-540, :437-460, :120-124), and runs before anything touches
// the device; the compute is one call into the C ABI of libgrouped_gemm_hip.so on
// torch's current HIP stream.
#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/hip/HIPCachingAllocator.h>
#include <torch/extension.h>

#include <map>
#include <mutex>
#include <tuple>
#include <utility>

#include "../../include/grouped_gemm_hip.h"

namespace grouped_gemm {

namespace {

bool IsFloat8(torch::ScalarType t) { return t == torch::kFloat8_e4m3fn || t == torch::kFloat8_e5m2; }

// Element type of c for operands of type `t`: the same for the two-byte types, bf16 for fp8.
torch::ScalarType OutputType(torch::ScalarType t) { return IsFloat8(t) ? torch::kBFloat16 : t; }

int DtypeCode(torch::ScalarType t) {
  switch (t) {
    case torch::kFloat16: return GG_DTYPE_F16;
    case torch::kFloat8_e4m3fn: return GG_DTYPE_F8E4M3;
    case torch::kFloat8_e5m2: return GG_DTYPE_F8E5M2;
    default: return GG_DTYPE_BF16;
  }
}

// Row indices of the fused gather / scatter forms (see gg_gmm): undefined tensors mean "rows in place".
struct RowIndices {
  torch::Tensor a, b, c;
  bool any() const { return a.defined() || b.defined() || c.defined(); }
};

// `on_device` false skips the checks that a tensor lives on the GPU, so that the shape,
// rank and dtype rules can be exercised with CPU tensors on a machine without one.
// With row indices, `tokens` (the rows of the product) is the length of the index instead of the
// row count of the tensor it redirects.
// With `gate_up`, b holds two matrices per expert side by side and c is half as wide as b.
void Validate(const torch::Tensor& a, const torch::Tensor& b, const torch::Tensor& c,
              const torch::Tensor& batch_sizes, bool trans_a, bool trans_b, bool on_device,
              const RowIndices& rows = RowIndices(), bool gate_up = false) {
  // Only one of the operands may be transposed (csrc/grouped_gemm.cu:476).
  TORCH_CHECK(!(trans_a && trans_b), "grouped_gemm: trans_a and trans_b cannot both be set");

  // batch_sizes may live on the host or on the device (csrc/grouped_gemm.cu:478-486).
  TORCH_CHECK(batch_sizes.is_cuda() || batch_sizes.is_cpu(),
              "grouped_gemm: batch_sizes must be a CPU or GPU tensor");
  TORCH_CHECK(batch_sizes.ndimension() == 1, "grouped_gemm: batch_sizes must be 1-d");
  TORCH_CHECK(batch_sizes.scalar_type() == torch::kInt64, "grouped_gemm: batch_sizes must be int64");

  // a: (tokens, hidden_in) bf16 on the GPU (csrc/grouped_gemm.cu:490-492).  float16 is accepted
  // as well, for all three tensors alike; the reference takes bfloat16 only.
  if (on_device) TORCH_CHECK(a.is_cuda(), "grouped_gemm: a must be a GPU tensor");
  TORCH_CHECK(a.ndimension() == 2, "grouped_gemm: a must be 2-d");
  TORCH_CHECK(a.scalar_type() == torch::kBFloat16 || a.scalar_type() == torch::kFloat16 || IsFloat8(a.scalar_type()),
              "grouped_gemm: a must be bfloat16 (or float16, float8_e4m3fn, float8_e5m2)");

  // b, c: bf16 on the GPU (csrc/grouped_gemm.cu:503-506).
  if (on_device) {
    TORCH_CHECK(b.is_cuda(), "grouped_gemm: b must be a GPU tensor");
    TORCH_CHECK(c.is_cuda(), "grouped_gemm: c must be a GPU tensor");
  }
  TORCH_CHECK(b.scalar_type() == a.scalar_type(), "grouped_gemm: b must be bfloat16 (the element type of a)");
  TORCH_CHECK(c.scalar_type() == OutputType(a.scalar_type()),
              "grouped_gemm: c must be bfloat16 (the element type of a; bfloat16 for float8 operands)");
  for (const torch::Tensor* idx : {&rows.a, &rows.b, &rows.c}) {
    if (!idx->defined()) continue;
    TORCH_CHECK(idx->ndimension() == 1 && idx->scalar_type() == torch::kInt32 && idx->is_contiguous(),
                "grouped_gemm: a row index must be a contiguous 1-d int32 tensor");
    if (on_device) TORCH_CHECK(idx->is_cuda() && idx->device() == a.device(), "grouped_gemm: a row index must be on a's GPU");
  }
  TORCH_CHECK(!(trans_a && rows.c.defined()), "grouped_gemm: the trans_a output has no row per token to scatter");
  TORCH_CHECK(!(trans_a && gate_up), "grouped_gemm: the SwiGLU epilogue is not for the trans_a layout");
  TORCH_CHECK(trans_a || !rows.b.defined(), "grouped_gemm: only the trans_a layout has a row per token in b");
  const int64_t tokens = rows.a.defined() ? rows.a.size(0) : a.size(0);

  if (trans_a) {
    // b (tokens, hidden_out), c (num_experts, hidden_in, hidden_out)
    // (csrc/grouped_gemm.cu:513-522).
    TORCH_CHECK(b.ndimension() == 2, "grouped_gemm: with trans_a, b must be 2-d");
    TORCH_CHECK(c.ndimension() == 3, "grouped_gemm: with trans_a, c must be 3-d");
    TORCH_CHECK((rows.b.defined() ? rows.b.size(0) : b.size(0)) == tokens,
                "grouped_gemm: a and b must have the same number of rows");
    TORCH_CHECK(c.size(0) == batch_sizes.size(0), "grouped_gemm: c.size(0) must equal the number of experts");
    TORCH_CHECK(c.size(1) == a.size(1), "grouped_gemm: c.size(1) must equal a.size(1)");
    TORCH_CHECK(c.size(2) == b.size(1), "grouped_gemm: c.size(2) must equal b.size(1)");
  } else {
    // b (num_experts, hidden_in, hidden_out) or transposed, c (tokens, hidden_out)
    // (csrc/grouped_gemm.cu:524-534).
    TORCH_CHECK(b.ndimension() == 3, "grouped_gemm: b must be 3-d");
    TORCH_CHECK(c.ndimension() == 2, "grouped_gemm: c must be 2-d");
    const int64_t hidden_in = trans_b ? b.size(2) : b.size(1);
    TORCH_CHECK(hidden_in == a.size(1), "grouped_gemm: contraction dimensions of a and b differ");
    TORCH_CHECK(batch_sizes.size(0) == b.size(0), "grouped_gemm: need one batch size per expert");
    // The reference leaves the shape of c unchecked here; a wrong one would make the
    // kernel write outside c, so it is rejected.
    TORCH_CHECK(!gate_up || (trans_b ? b.size(1) : b.size(2)) % 2 == 0,
                "grouped_gemm: with gate | up columns, b must hold an even number of them");
    const int64_t hidden_out = (trans_b ? b.size(1) : b.size(2)) / (gate_up ? 2 : 1);
    if (rows.c.defined()) {
      TORCH_CHECK(rows.c.size(0) == tokens, "grouped_gemm: c_rows needs one entry per row of the product");
      TORCH_CHECK(c.size(1) == hidden_out, "grouped_gemm: c must have hidden_out columns");
    } else {
      TORCH_CHECK(c.size(0) == tokens && c.size(1) == hidden_out,
                  "grouped_gemm: c must have shape (tokens, hidden_out)");
    }
  }

  // Transposition goes through the flags only (csrc/grouped_gemm.cu:538-540).
  TORCH_CHECK(a.is_contiguous(), "grouped_gemm: a must be contiguous");
  TORCH_CHECK(b.is_contiguous(), "grouped_gemm: b must be contiguous");
  TORCH_CHECK(c.is_contiguous(), "grouped_gemm: c must be contiguous");

  // Device-resident sizes: any number of experts (the reference stops at 512,
  // csrc/grouped_gemm.cu:120-124; here further experts go to further launches).
  if (batch_sizes.is_cuda()) {
    TORCH_CHECK(batch_sizes.is_contiguous(), "grouped_gemm: batch_sizes must be contiguous");
    if (on_device)
      TORCH_CHECK(batch_sizes.device() == a.device(), "grouped_gemm: batch_sizes is on another GPU");
  }
  if (on_device) {
    TORCH_CHECK(b.device() == a.device() && c.device() == a.device(),
                "grouped_gemm: a, b and c must be on the same GPU");
  }
}

// Number of the capture that `stream` is in, 0: in none.
unsigned long long CaptureNumber(hipStream_t stream) {
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  unsigned long long number = 0;
  if (hipStreamGetCaptureInfo(stream, &status, &number) != hipSuccess) {
    (void)hipGetLastError();
    return 0;
  }
  return status == hipStreamCaptureStatusNone ? 0 : number;
}

// Whether a tensor made during a capture belongs to the graph that is captured, i.e. lies in a pool that the
// allocator keeps for it.  It does in torch's own captures (torch.cuda.graph), not in one that was begun past
// torch: there the allocator would give the memory to others while the graph still uses it.
bool BelongsToGraph(const torch::Tensor& t) {
  namespace allocator = c10::hip::HIPCachingAllocator;
  if (allocator::get()->name() != "native") return true;   // (the stream-ordered one makes it a node of the graph)
  const size_t at = reinterpret_cast<size_t>(t.data_ptr());
  for (const auto& segment : allocator::snapshot().segments)
    if (at >= segment.address && at - segment.address < segment.total_size)
      return segment.owner_private_pool_id.first != 0 || segment.owner_private_pool_id.second != 0;
  return false;
}

// Workspace for the depth pieces of a call's last round (see gg_gmm).
//
// Outside a graph capture: one per device and stream, allocated and zeroed at the first call there that can
// use one (gg_workspace_bytes_for) and kept for the life of the process.  Calls on one stream run one after
// the other, so they can share it; the kernels leave its counters zero.  Two calls in one launch (gg_gmm_pair) run
// at the same time: the second one's is another, `which` = 1, made at the first pair whose both halves can use one.
//
// A captured call runs at every replay, on whatever stream and beside whatever other graphs the program
// chooses, and what it allocates is the graph's pool's, which graphs may share.  It takes a workspace for
// itself alone, which its graph's later calls and no others can get again, and clears the counters as a
// part of the graph (a fill of 4 KiB ahead of the launch).  Where the graph cannot own one (BelongsToGraph; asked
// once per capture and thread) there is none, an undefined tensor: the call keeps its tiles whole.
torch::Tensor Workspace(const torch::Device& device, hipStream_t stream, int which = 0) {
  constexpr int64_t kCounterBytes = 4096;   // the arrival counters at its beginning, see gg_gmm_args.workspace
  const auto bytes = torch::dtype(torch::kUInt8).device(device);
  if (const unsigned long long capture = CaptureNumber(stream)) {
    thread_local unsigned long long asked = 0;
    thread_local bool owned = false;
    if (asked == capture && !owned) return torch::Tensor();
    torch::Tensor ws = torch::empty({(int64_t)GG_WORKSPACE_BYTES}, bytes);
    if (asked != capture) {
      owned = BelongsToGraph(ws);
      asked = capture;
      if (!owned) return torch::Tensor();
    }
    ws.narrow(0, 0, kCounterBytes).zero_();
    return ws;
  }
  static std::mutex mu;
  static std::map<std::tuple<int, hipStream_t, int>, torch::Tensor> cache;
  const auto key = std::make_tuple((int)device.index(), stream, which);
  {
    std::lock_guard<std::mutex> lock(mu);
    const auto it = cache.find(key);
    if (it != cache.end()) return it->second;
  }
  // (allocated with the lock released: the allocation may have to wait for another thread)
  torch::Tensor ws = torch::zeros({(int64_t)GG_WORKSPACE_BYTES}, bytes);
  std::lock_guard<std::mutex> lock(mu);
  return cache.emplace(key, ws).first->second;
}

// The library's int32 word of the current device that the kernels OR GG_STATUS_* bits into when
// device-resident batch_sizes had to be clamped (negative, or summing past the rows of a): what a
// host-resident size vector would have been rejected for.  Read (and cleared) through size_status().
// (No tensor: one made during a graph capture would lie in that graph's pool, under other graphs' temporaries,
// and be cleared by its replays.)
int32_t* SizeStatusWord() {
  int32_t* word = gg_size_status_word();
  TORCH_CHECK(word != nullptr, "grouped_gemm: ", gg_last_error());
  return word;
}

// The C ABI's arguments for a validated call on the current device and `stream`, without a workspace.  `sizes`:
// contiguous batch_sizes, which have to live until the call is enqueued.
gg_gmm_args Arguments(const torch::Tensor& a, const torch::Tensor& b, const torch::Tensor& c, const torch::Tensor& sizes,
                      bool trans_a, bool trans_b, bool accumulate_f32, int64_t flags, const RowIndices& rows, bool gate_up,
                      hipStream_t stream) {
  gg_gmm_args g = {};
  g.struct_bytes = sizeof(g);
  g.dtype = DtypeCode(a.scalar_type());
  g.a = a.data_ptr();
  g.b = b.data_ptr();
  g.c = c.data_ptr();
  g.batch_sizes = sizes.data_ptr<int64_t>();
  g.batch_sizes_on_device = sizes.is_cuda() ? 1 : 0;
  g.trans_a = trans_a ? 1 : 0;
  g.trans_b = trans_b ? 1 : 0;
  g.accumulate_f32 = accumulate_f32 ? 1 : 0;
  g.num_groups = sizes.size(0);
  g.tokens = rows.a.defined() ? rows.a.size(0) : a.size(0);
  g.a_row_index = rows.a.defined() ? rows.a.data_ptr<int32_t>() : nullptr;
  g.b_row_index = rows.b.defined() ? rows.b.data_ptr<int32_t>() : nullptr;
  g.c_row_index = rows.c.defined() ? rows.c.data_ptr<int32_t>() : nullptr;
  g.hidden_in = a.size(1);
  g.hidden_out = (trans_a ? b.size(1) : (trans_b ? b.size(1) : b.size(2))) / (gate_up ? 2 : 1);
  g.epilogue = gate_up ? GG_EPILOGUE_SWIGLU : GG_EPILOGUE_NONE;
  g.a_num_rows = a.size(0);
  g.c_num_rows = trans_a ? 0 : c.size(0);
  g.b_num_rows = trans_a ? (int32_t)b.size(0) : 0;
  g.flags = (int32_t)flags | GG_FLAG_FEW_TILES | GG_FLAG_EVEN_PIECES;
  g.stream = static_cast<void*>(stream);
  if (sizes.is_cuda()) g.size_status = SizeStatusWord();
  return g;
}

// A workspace for calls that can make use of one (`bytes` of gg_workspace_bytes_for: deep products, weight gradients)
// and only for them; the tensor has to live until the call is enqueued.
torch::Tensor AttachWorkspace(gg_gmm_args* g, uint64_t bytes, const torch::Device& device, hipStream_t stream, int which = 0) {
  torch::Tensor workspace;
  if (bytes > 0) {
    workspace = Workspace(device, stream, which);
    if (workspace.defined()) {
      g->workspace = workspace.data_ptr();
      g->workspace_bytes = (uint64_t)workspace.numel();
    }
  }
  return workspace;
}

void Run(const torch::Tensor& a, const torch::Tensor& b, const torch::Tensor& c, const torch::Tensor& batch_sizes,
         bool trans_a, bool trans_b, bool accumulate_f32, int64_t flags, const RowIndices& rows = RowIndices(),
         bool gate_up = false) {
  torch::Tensor sizes = batch_sizes.is_cpu() ? batch_sizes.contiguous() : batch_sizes;
  c10::hip::HIPGuardMasqueradingAsCUDA guard(a.device());
  hipStream_t stream = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(a.device().index()).stream();
  TORCH_CHECK(gg_init() == GG_OK, "grouped_gemm: ", gg_last_error());
  gg_gmm_args g = Arguments(a, b, c, sizes, trans_a, trans_b, accumulate_f32, flags, rows, gate_up, stream);
  const torch::Tensor workspace = AttachWorkspace(&g, gg_workspace_bytes_for(&g), a.device(), stream);
  const int rc = gg_gmm(&g);
  TORCH_CHECK(rc == GG_OK, "grouped_gemm: ", gg_last_error());
}

// Both gradients of a product, agrad = grad @ b (or b^T) and bgrad = lhs^T @ rhs, all validated.
void RunGradients(const torch::Tensor& grad, const torch::Tensor& b, const torch::Tensor& agrad, bool trans_b,
                  const torch::Tensor& lhs, const torch::Tensor& rhs, const torch::Tensor& bgrad,
                  const torch::Tensor& batch_sizes) {
  torch::Tensor sizes = batch_sizes.is_cpu() ? batch_sizes.contiguous() : batch_sizes;
  c10::hip::HIPGuardMasqueradingAsCUDA guard(grad.device());
  hipStream_t stream = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(grad.device().index()).stream();
  TORCH_CHECK(gg_init() == GG_OK, "grouped_gemm: ", gg_last_error());
  gg_gmm_args g1 = Arguments(grad, b, agrad, sizes, false, trans_b, false, 0, RowIndices(), false, stream);
  gg_gmm_args g2 = Arguments(lhs, rhs, bgrad, sizes, true, false, false, 0, RowIndices(), false, stream);
  const torch::Tensor workspace1 = AttachWorkspace(&g1, gg_workspace_bytes_for(&g1), grad.device(), stream);
  const torch::Tensor workspace2 =
      AttachWorkspace(&g2, gg_workspace_bytes_for(&g2), grad.device(), stream, workspace1.defined() ? 1 : 0);
  const int rc = gg_gmm_pair(&g1, &g2);
  TORCH_CHECK(rc == GG_OK, "grouped_gemm: ", gg_last_error());
}

}  // namespace

void GroupedGemm(torch::Tensor a, torch::Tensor b, torch::Tensor c, torch::Tensor batch_sizes,
                 bool trans_a, bool trans_b) {
  Validate(a, b, c, batch_sizes, trans_a, trans_b, /*on_device=*/true);
  Run(a, b, c, batch_sizes, trans_a, trans_b, /*accumulate_f32=*/false, /*flags=*/0);
}

// Whether a call runs on the streaming kernels as it is: well-formed contiguous operands whose sizes
// and addresses need no padded copies (of a well-formed call, what _needs_padding in backend.py says no to).
// Everything else is left to the Python side, whose checks and error messages then apply.
bool IsDirect(const torch::Tensor& a, const torch::Tensor& b, const torch::Tensor& batch_sizes, bool trans_a,
              bool trans_b, const torch::Tensor* c) {
  if ((trans_a && trans_b) || batch_sizes.dim() != 1 || a.dim() != 2 || b.dim() != (trans_a ? 2 : 3)) return false;
  if (!a.is_cuda() || !b.is_cuda() || a.scalar_type() != b.scalar_type()) return false;
  const torch::ScalarType t = a.scalar_type();
  if (t != torch::kBFloat16 && t != torch::kFloat16 && !IsFloat8(t)) return false;
  if (!a.is_contiguous() || !b.is_contiguous() || (c != nullptr && !c->is_contiguous())) return false;
  const int64_t hin = a.size(1), hout = trans_a || trans_b ? b.size(1) : b.size(2);
  if (a.size(0) == 0 || hin == 0 || hout == 0) return false;
  const uintptr_t addresses = reinterpret_cast<uintptr_t>(a.data_ptr()) | reinterpret_cast<uintptr_t>(b.data_ptr()) |
                              (c != nullptr ? reinterpret_cast<uintptr_t>(c->data_ptr()) : 0);
  const int64_t mult = IsFloat8(t) ? 16 : 8;
  if (hin % mult == 0 && hout % mult == 0 && (addresses & 15) == 0) return true;
  return !IsFloat8(t) && hin % 2 == 0 && hout % 2 == 0 && (addresses & 3) == 0;
}

torch::Tensor AllocateOutput(const torch::Tensor& a, const torch::Tensor& b, const torch::Tensor& batch_sizes,
                             bool trans_a, bool trans_b) {
  const auto options = a.options().dtype(OutputType(a.scalar_type()));
  if (trans_a) return torch::empty({batch_sizes.size(0), a.size(1), b.size(1)}, options);
  return torch::empty({a.size(0), trans_b ? b.size(1) : b.size(2)}, options);
}

// backend.gmm in one step for direct calls; nothing is returned (and nothing done) for others.
c10::optional<torch::Tensor> GroupedGemmDirect(const torch::Tensor& a, const torch::Tensor& b,
                                               const torch::Tensor& batch_sizes, bool trans_a, bool trans_b,
                                               const c10::optional<torch::Tensor>& c) {
  if (!IsDirect(a, b, batch_sizes, trans_a, trans_b, c.has_value() ? &*c : nullptr)) return c10::nullopt;
  torch::Tensor out = c.has_value() ? *c : AllocateOutput(a, b, batch_sizes, trans_a, trans_b);
  GroupedGemm(a, b, out, batch_sizes, trans_a, trans_b);
  return out;
}

// Both gradients of gmm(a, b, batch_sizes, trans_b=trans_b); the launches of both are one where the library has
// a kernel for the two (gg_gmm_pair).
std::pair<torch::Tensor, torch::Tensor> BothGradients(const torch::Tensor& grad, const torch::Tensor& a, const torch::Tensor& b,
                                                      const torch::Tensor& batch_sizes, bool trans_b) {
  const torch::Tensor &lhs = trans_b ? grad : a, &rhs = trans_b ? a : grad;
  torch::Tensor agrad = AllocateOutput(grad, b, batch_sizes, false, !trans_b);
  Validate(grad, b, agrad, batch_sizes, false, !trans_b, /*on_device=*/true);
  torch::Tensor bgrad = AllocateOutput(lhs, rhs, batch_sizes, true, false);
  Validate(lhs, rhs, bgrad, batch_sizes, true, false, /*on_device=*/true);
  RunGradients(grad, b, agrad, !trans_b, lhs, rhs, bgrad, batch_sizes);
  return {agrad, bgrad};
}

// ... for operands that the streaming kernels take as they are; nothing is returned (and nothing done) for others.
c10::optional<std::pair<torch::Tensor, torch::Tensor>> GroupedGemmGradients(const torch::Tensor& grad, const torch::Tensor& a,
                                                                            const torch::Tensor& b,
                                                                            const torch::Tensor& batch_sizes, bool trans_b) {
  const torch::Tensor &lhs = trans_b ? grad : a, &rhs = trans_b ? a : grad;
  if (!IsDirect(grad, b, batch_sizes, false, !trans_b, nullptr) || !IsDirect(lhs, rhs, batch_sizes, true, false, nullptr))
    return c10::nullopt;
  return BothGradients(grad, a, b, batch_sizes, trans_b);
}

// ops.GroupedGemm (the reference's grouped_gemm/ops.py:8-29) as a native autograd node: a training
// step of a small layer is bound by what the host does between the three launches, and the
// interpreter was most of it.
class GroupedGemmNode : public torch::autograd::Function<GroupedGemmNode> {
 public:
  static torch::Tensor forward(torch::autograd::AutogradContext* ctx, const torch::Tensor& a, const torch::Tensor& b,
                               const torch::Tensor& batch_sizes, bool trans_b) {
    ctx->save_for_backward({a, b, batch_sizes});
    ctx->saved_data["trans_b"] = trans_b;
    torch::Tensor out = AllocateOutput(a, b, batch_sizes, false, trans_b);
    GroupedGemm(a, b, out, batch_sizes, false, trans_b);
    return out;
  }

  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                 torch::autograd::variable_list grads) {
    torch::Tensor grad = grads[0].contiguous();
    if (reinterpret_cast<uintptr_t>(grad.data_ptr()) & 15) grad = grad.clone();
    const auto saved = ctx->get_saved_variables();
    const torch::Tensor &a = saved[0], &b = saved[1], &batch_sizes = saved[2];
    const bool trans_b = ctx->saved_data["trans_b"].toBool();
    torch::Tensor agrad, bgrad;
    if (ctx->needs_input_grad(0) && ctx->needs_input_grad(1)) {
      std::tie(agrad, bgrad) = BothGradients(grad, a, b, batch_sizes, trans_b);
    } else if (ctx->needs_input_grad(0)) {
      agrad = AllocateOutput(grad, b, batch_sizes, false, !trans_b);
      GroupedGemm(grad, b, agrad, batch_sizes, false, !trans_b);
    } else if (ctx->needs_input_grad(1)) {
      const torch::Tensor &lhs = trans_b ? grad : a, &rhs = trans_b ? a : grad;
      bgrad = AllocateOutput(lhs, rhs, batch_sizes, true, false);
      GroupedGemm(lhs, rhs, bgrad, batch_sizes, true, false);
    }
    return {agrad, bgrad, torch::Tensor(), torch::Tensor()};
  }
};

c10::optional<torch::Tensor> GroupedGemmAutograd(const torch::Tensor& a, const torch::Tensor& b,
                                                 const torch::Tensor& batch_sizes, bool trans_b) {
  if (!IsDirect(a, b, batch_sizes, false, trans_b, nullptr)) return c10::nullopt;
  return GroupedGemmNode::apply(a, b, batch_sizes, trans_b);
}

// Operands whose rows are further apart than they are long (gg_gmm_strided): a (tokens, a row), b (experts, rows,
// a row), or (tokens, a row) with trans_a; c as for gmm with the given hidden sizes.
void CheckStrided(const torch::Tensor& a, const torch::Tensor& b, const torch::Tensor& c, const torch::Tensor& batch_sizes,
                  bool trans_a, bool trans_b, int64_t hin, int64_t hout) {
  TORCH_CHECK(a.is_cuda() && b.is_cuda() && c.is_cuda() && a.device() == b.device() && a.device() == c.device() &&
                  a.is_contiguous() && b.is_contiguous() && c.is_contiguous(),
              "grouped_gemm: a, b and c must be contiguous tensors on the same GPU");
  TORCH_CHECK((a.scalar_type() == torch::kBFloat16 || a.scalar_type() == torch::kFloat16) && b.scalar_type() == a.scalar_type() &&
                  c.scalar_type() == a.scalar_type(),
              "grouped_gemm: a, b and c must all be bfloat16 or float16");
  TORCH_CHECK(batch_sizes.dim() == 1 && batch_sizes.scalar_type() == torch::kInt64 &&
                  (batch_sizes.is_cpu() || (batch_sizes.device() == a.device() && batch_sizes.is_contiguous())),
              "grouped_gemm: batch_sizes must be 1-d int64 on the host or on a's GPU");
  TORCH_CHECK(!(trans_a && trans_b), "grouped_gemm: trans_a and trans_b cannot both be set");
  const int64_t experts = batch_sizes.size(0), tokens = a.dim() == 2 ? a.size(0) : -1;
  const int64_t b_rows = trans_a ? tokens : (trans_b ? hout : hin), b_row = trans_b ? hin : hout;
  TORCH_CHECK(tokens >= 0 && a.size(1) >= hin && b.dim() == (trans_a ? 2 : 3) && (trans_a || b.size(0) == experts) &&
                  b.size(-2) == b_rows && b.size(-1) >= b_row,
              "grouped_gemm: a or b does not hold operands of these hidden sizes");
  TORCH_CHECK(trans_a ? c.dim() == 3 && c.size(0) == experts && c.size(1) == hin && c.size(2) == hout
                      : c.dim() == 2 && c.size(0) == tokens && c.size(1) == hout,
              "grouped_gemm: c does not have the shape of the product");
}

// Arguments of such a call, with a workspace where it can make use of one.
gg_gmm_args StridedArguments(const torch::Tensor& a, const torch::Tensor& b, const torch::Tensor& c, const torch::Tensor& sizes,
                             bool trans_a, bool trans_b, int64_t hin, int64_t hout, hipStream_t stream, int which,
                             torch::Tensor* workspace) {
  gg_gmm_args g = Arguments(a, b, c, sizes, trans_a, trans_b, false, 0, RowIndices(), false, stream);
  g.hidden_in = hin;
  g.hidden_out = hout;
  *workspace = AttachWorkspace(&g, gg_workspace_bytes_for_strided(&g, a.size(-1), b.size(-1)), a.device(), stream, which);
  return g;
}

void GroupedGemmStrided(torch::Tensor a, torch::Tensor b, torch::Tensor c, torch::Tensor batch_sizes, bool trans_a,
                        bool trans_b, int64_t hin, int64_t hout) {
  CheckStrided(a, b, c, batch_sizes, trans_a, trans_b, hin, hout);
  torch::Tensor sizes = batch_sizes.is_cpu() ? batch_sizes.contiguous() : batch_sizes;
  c10::hip::HIPGuardMasqueradingAsCUDA guard(a.device());
  hipStream_t stream = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(a.device().index()).stream();
  TORCH_CHECK(gg_init() == GG_OK, "grouped_gemm: ", gg_last_error());
  torch::Tensor workspace;
  const gg_gmm_args g = StridedArguments(a, b, c, sizes, trans_a, trans_b, hin, hout, stream, 0, &workspace);
  const int rc = gg_gmm_strided(&g, a.size(-1), b.size(-1));
  TORCH_CHECK(rc == GG_OK, "grouped_gemm: ", gg_last_error());
}

// Both gradients of gmm with hidden sizes hin and hout, from such operands.
std::pair<torch::Tensor, torch::Tensor> GradientsStrided(torch::Tensor grad, torch::Tensor a, torch::Tensor b,
                                                         torch::Tensor batch_sizes, bool trans_b, int64_t hin, int64_t hout) {
  const torch::Tensor &lhs = trans_b ? grad : a, &rhs = trans_b ? a : grad;
  const int64_t lhs_cols = trans_b ? hout : hin, rhs_cols = trans_b ? hin : hout;
  c10::hip::HIPGuardMasqueradingAsCUDA guard(grad.device());
  torch::Tensor agrad = torch::empty({grad.size(0), hin}, grad.options());
  torch::Tensor bgrad = torch::empty({batch_sizes.size(0), lhs_cols, rhs_cols}, grad.options());
  CheckStrided(grad, b, agrad, batch_sizes, false, !trans_b, hout, hin);
  CheckStrided(lhs, rhs, bgrad, batch_sizes, true, false, lhs_cols, rhs_cols);
  torch::Tensor sizes = batch_sizes.is_cpu() ? batch_sizes.contiguous() : batch_sizes;
  hipStream_t stream = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(grad.device().index()).stream();
  TORCH_CHECK(gg_init() == GG_OK, "grouped_gemm: ", gg_last_error());
  torch::Tensor workspace1, workspace2;
  const gg_gmm_args g1 = StridedArguments(grad, b, agrad, sizes, false, !trans_b, hout, hin, stream, 0, &workspace1);
  const gg_gmm_args g2 = StridedArguments(lhs, rhs, bgrad, sizes, true, false, lhs_cols, rhs_cols, stream,
                                          workspace1.defined() ? 1 : 0, &workspace2);
  const int rc = gg_gmm_pair_strided(&g1, grad.size(-1), b.size(-1), &g2, lhs.size(-1), rhs.size(-1));
  TORCH_CHECK(rc == GG_OK, "grouped_gemm: ", gg_last_error());
  return {agrad, bgrad};
}

// gmm with GG_FLAG_* bits, for tests that compare the ways a call can be scheduled.
void GroupedGemmWithFlags(torch::Tensor a, torch::Tensor b, torch::Tensor c, torch::Tensor batch_sizes,
                          bool trans_a, bool trans_b, int64_t flags) {
  Validate(a, b, c, batch_sizes, trans_a, trans_b, /*on_device=*/true);
  Run(a, b, c, batch_sizes, trans_a, trans_b, /*accumulate_f32=*/false, flags);
}

// gmm with row indices: a gather fused into the loads of a (and of b with trans_a), a scatter
// fused into the stores of c.  An undefined (None) index leaves those rows in place.
void GroupedGemmIndexed(torch::Tensor a, torch::Tensor b, torch::Tensor c, torch::Tensor batch_sizes,
                        bool trans_a, bool trans_b, c10::optional<torch::Tensor> a_rows,
                        c10::optional<torch::Tensor> b_rows, c10::optional<torch::Tensor> c_rows) {
  RowIndices rows;
  if (a_rows.has_value()) rows.a = *a_rows;
  if (b_rows.has_value()) rows.b = *b_rows;
  if (c_rows.has_value()) rows.c = *c_rows;
  Validate(a, b, c, batch_sizes, trans_a, trans_b, /*on_device=*/true, rows);
  Run(a, b, c, batch_sizes, trans_a, trans_b, /*accumulate_f32=*/false, /*flags=*/0, rows);
}

// c = silu(a @ gate) * (a @ up) with b = [gate | up] per expert, optionally with row indices.
void GroupedGemmSwiGLU(torch::Tensor a, torch::Tensor b, torch::Tensor c, torch::Tensor batch_sizes, bool trans_b,
                       c10::optional<torch::Tensor> a_rows, c10::optional<torch::Tensor> c_rows) {
  RowIndices rows;
  if (a_rows.has_value()) rows.a = *a_rows;
  if (c_rows.has_value()) rows.c = *c_rows;
  Validate(a, b, c, batch_sizes, /*trans_a=*/false, trans_b, /*on_device=*/true, rows, /*gate_up=*/true);
  Run(a, b, c, batch_sizes, /*trans_a=*/false, trans_b, /*accumulate_f32=*/false, /*flags=*/0, rows, /*gate_up=*/true);
}

// The same for a gradient to come: c, and gate | up (tokens, 2 * hidden_out) as gmm(a, b) would give them; nothing (and
// nothing done) for calls whose kernels do not keep them.
c10::optional<std::pair<torch::Tensor, torch::Tensor>> GroupedGemmSwiGLUKeep(const torch::Tensor& a, const torch::Tensor& b,
                                                                             const torch::Tensor& batch_sizes, bool trans_b) {
  if (!IsDirect(a, b, batch_sizes, false, trans_b, nullptr) || IsFloat8(a.scalar_type())) return c10::nullopt;
  const int64_t cols = trans_b ? b.size(1) : b.size(2);
  if (cols % 16 != 0) return c10::nullopt;   // (odd numbers of columns are rejected, others run on the general kernels)
  torch::Tensor c = torch::empty({a.size(0), cols / 2}, a.options());
  Validate(a, b, c, batch_sizes, false, trans_b, /*on_device=*/true, RowIndices(), /*gate_up=*/true);
  torch::Tensor sizes = batch_sizes.is_cpu() ? batch_sizes.contiguous() : batch_sizes;
  c10::hip::HIPGuardMasqueradingAsCUDA guard(a.device());
  hipStream_t stream = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(a.device().index()).stream();
  TORCH_CHECK(gg_init() == GG_OK, "grouped_gemm: ", gg_last_error());
  gg_gmm_args g = Arguments(a, b, c, sizes, false, trans_b, false, 0, RowIndices(), true, stream);
  if (!gg_keeps_gate_up(&g)) return c10::nullopt;
  torch::Tensor gate_up = torch::empty({a.size(0), cols}, a.options());
  const torch::Tensor workspace = AttachWorkspace(&g, gg_workspace_bytes_for(&g), a.device(), stream);
  const int rc = gg_gmm_keep_gate_up(&g, gate_up.data_ptr());
  TORCH_CHECK(rc == GG_OK, "grouped_gemm: ", gg_last_error());
  return std::make_pair(c, gate_up);
}

// Gradients of gate | up (rows, 2 * cols) from the gradient of silu(gate) * up (rows, cols); see
// gg_swiglu_backward.
torch::Tensor SwiGLUBackward(torch::Tensor gate_up, torch::Tensor grad) {
  TORCH_CHECK(gate_up.is_cuda() && grad.is_cuda() && gate_up.device() == grad.device(),
              "grouped_gemm: gate_up and grad must be on the same GPU");
  TORCH_CHECK(gate_up.scalar_type() == torch::kBFloat16 || gate_up.scalar_type() == torch::kFloat16,
              "grouped_gemm: gate_up must be bfloat16 or float16");
  TORCH_CHECK(grad.scalar_type() == gate_up.scalar_type(), "grouped_gemm: grad must have the element type of gate_up");
  TORCH_CHECK(gate_up.dim() == 2 && grad.dim() == 2 && gate_up.size(0) == grad.size(0) &&
                  gate_up.size(1) == 2 * grad.size(1),
              "grouped_gemm: gate_up must be (rows, 2 * cols) and grad (rows, cols)");
  TORCH_CHECK(gate_up.is_contiguous() && grad.is_contiguous(), "grouped_gemm: gate_up and grad must be contiguous");
  c10::hip::HIPGuardMasqueradingAsCUDA guard(gate_up.device());
  torch::Tensor out = torch::empty_like(gate_up);
  hipStream_t stream = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(gate_up.device().index()).stream();
  const int rc = gg_swiglu_backward(gate_up.data_ptr(), grad.data_ptr(), out.data_ptr(), grad.size(0), grad.size(1),
                                    DtypeCode(gate_up.scalar_type()), static_cast<void*>(stream));
  TORCH_CHECK(rc == GG_OK, "grouped_gemm: ", gg_last_error());
  return out;
}

// out (num_dst, cols): row d is the sum of the rows of src that row_index sends there; see gg_sum_rows.
torch::Tensor SumRows(torch::Tensor src, torch::Tensor row_index, int64_t num_dst) {
  TORCH_CHECK(src.is_cuda() && src.dim() == 2 && src.is_contiguous(), "grouped_gemm: src must be a contiguous 2-d GPU tensor");
  TORCH_CHECK(src.scalar_type() == torch::kBFloat16 || src.scalar_type() == torch::kFloat16,
              "grouped_gemm: src must be bfloat16 or float16");
  TORCH_CHECK(row_index.dim() == 1 && row_index.scalar_type() == torch::kInt32 && row_index.is_contiguous() &&
                  row_index.device() == src.device() && row_index.size(0) == src.size(0),
              "grouped_gemm: row_index must be a contiguous int32 tensor with one entry per row, on src's GPU");
  TORCH_CHECK(num_dst >= 0, "grouped_gemm: negative row count");
  c10::hip::HIPGuardMasqueradingAsCUDA guard(src.device());
  torch::Tensor out = torch::empty({num_dst, src.size(1)}, src.options());
  torch::Tensor scratch = torch::empty({(int64_t)gg_sum_rows_scratch_bytes(src.size(0), num_dst)},
                                       src.options().dtype(torch::kUInt8));
  hipStream_t stream = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(src.device().index()).stream();
  const int rc = gg_sum_rows(src.data_ptr(), row_index.data_ptr<int32_t>(), out.data_ptr(), src.size(0), num_dst,
                             src.size(1), DtypeCode(src.scalar_type()), scratch.data_ptr(), static_cast<void*>(stream));
  TORCH_CHECK(rc == GG_OK, "grouped_gemm: ", gg_last_error());
  return out;
}

// t (batch, rows, cols) or (rows, cols), zero-padded to `rows` x `cols` per batch; see gg_pad_rows.
torch::Tensor PadRows(torch::Tensor t, int64_t rows, int64_t cols) {
  TORCH_CHECK(t.is_cuda() && t.is_contiguous() && (t.dim() == 2 || t.dim() == 3) && t.element_size() <= 2,
              "grouped_gemm: pad_rows needs a contiguous 2-d or 3-d GPU tensor of 1 or 2 byte elements");
  c10::hip::HIPGuardMasqueradingAsCUDA guard(t.device());
  const int64_t batches = t.dim() == 3 ? t.size(0) : 1;
  torch::Tensor out = t.dim() == 3 ? torch::empty({batches, rows, cols}, t.options()) : torch::empty({rows, cols}, t.options());
  if (out.numel() == 0) return out;
  hipStream_t stream = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream();
  const int rc = gg_pad_rows(t.data_ptr(), out.data_ptr(), batches, t.size(-2), t.size(-1), rows, cols, (int)t.element_size(),
                             static_cast<void*>(stream));
  TORCH_CHECK(rc == GG_OK, "grouped_gemm: ", gg_last_error());
  return out;
}

// c = the upper left corner of every batch of t; see gg_unpad_rows.
void UnpadRows(torch::Tensor t, torch::Tensor c) {
  TORCH_CHECK(t.is_cuda() && c.is_cuda() && t.device() == c.device() && t.is_contiguous() && c.is_contiguous() &&
                  t.dim() == c.dim() && (t.dim() == 2 || (t.dim() == 3 && t.size(0) == c.size(0))) &&
                  t.scalar_type() == c.scalar_type() && t.element_size() == 2,
              "grouped_gemm: unpad_rows needs two contiguous GPU tensors of the same two-byte type, 2-d or of as many batches");
  c10::hip::HIPGuardMasqueradingAsCUDA guard(t.device());
  if (c.numel() == 0) return;
  hipStream_t stream = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream();
  const int rc = gg_unpad_rows(t.data_ptr(), c.data_ptr(), t.dim() == 3 ? t.size(0) : 1, t.size(-2), t.size(-1), c.size(-2),
                               c.size(-1), static_cast<void*>(stream));
  TORCH_CHECK(rc == GG_OK, "grouped_gemm: ", gg_last_error());
}

// c (num_experts, hidden_in, hidden_out) fp32 += per expert a_e^T @ b_e; see gg_gmm_bf16_acc_f32.
void AccumulateWeightGradient(torch::Tensor a, torch::Tensor b, torch::Tensor c, torch::Tensor batch_sizes) {
  TORCH_CHECK(c.scalar_type() == torch::kFloat32, "grouped_gemm: the accumulated gradient must be float32");
  // every other check is the one of the bf16 weight-gradient call
  torch::Tensor shape_of_c = torch::empty(c.sizes(), torch::dtype(OutputType(a.scalar_type())).device(torch::kMeta));
  Validate(a, b, shape_of_c, batch_sizes, /*trans_a=*/true, /*trans_b=*/false, /*on_device=*/false);
  TORCH_CHECK(a.is_cuda() && b.is_cuda() && c.is_cuda(), "grouped_gemm: a, b and c must be GPU tensors");
  TORCH_CHECK(b.device() == a.device() && c.device() == a.device(),
              "grouped_gemm: a, b and c must be on the same GPU");
  TORCH_CHECK(c.is_contiguous(), "grouped_gemm: c must be contiguous");
  if (batch_sizes.is_cuda())
    TORCH_CHECK(batch_sizes.device() == a.device(), "grouped_gemm: batch_sizes is on another GPU");
  Run(a, b, c, batch_sizes, /*trans_a=*/true, /*trans_b=*/false, /*accumulate_f32=*/true, /*flags=*/0);
}

// GG_STATUS_* bits collected on `device` since the last call of this function (waits for the
// device): 0 unless device-resident batch_sizes had to be clamped.
int64_t SizeStatus(torch::Device device) {
  TORCH_CHECK(device.is_cuda(), "grouped_gemm: size_status is kept per GPU");
  c10::hip::HIPGuardMasqueradingAsCUDA guard(device);
  if (!device.has_index()) device = torch::Device(device.type(), c10::hip::current_device());
  torch::Tensor word = torch::from_blob(SizeStatusWord(), {1}, torch::dtype(torch::kInt32).device(device));
  const int64_t bits = word.item<int32_t>();
  if (bits != 0) word.zero_();
  return bits;
}

// The on-device scheduler's view of the groups, as an int64 tensor
// (num_experts, GG_SCHED_COLS) on `device`; see gg_debug_schedule.
torch::Tensor DebugSchedule(torch::Tensor batch_sizes, int64_t tokens, int64_t hidden_in,
                            int64_t hidden_out, bool trans_a, bool trans_b, torch::Device device) {
  TORCH_CHECK(batch_sizes.ndimension() == 1 && batch_sizes.scalar_type() == torch::kInt64);
  TORCH_CHECK(device.is_cuda(), "grouped_gemm: the schedule is computed on a GPU");
  torch::Tensor sizes = batch_sizes.contiguous();
  if (sizes.is_cuda()) TORCH_CHECK(sizes.device() == device);
  c10::hip::HIPGuardMasqueradingAsCUDA guard(device);
  torch::Tensor out = torch::zeros({sizes.size(0), GG_SCHED_COLS},
                                   torch::dtype(torch::kInt64).device(device));
  hipStream_t stream = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(device.index()).stream();
  const int rc = gg_debug_schedule(sizes.data_ptr<int64_t>(), sizes.is_cuda() ? 1 : 0, sizes.size(0),
                                   tokens, hidden_in, hidden_out, trans_a ? 1 : 0, trans_b ? 1 : 0,
                                   out.data_ptr<int64_t>(), static_cast<void*>(stream));
  TORCH_CHECK(rc == GG_OK, "grouped_gemm: ", gg_last_error());
  return out;
}

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("gmm", &GroupedGemm, "Grouped GEMM.");
  m.def("gmm_direct", &GroupedGemmDirect,
        "gmm with the output allocated where c is None, for calls the streaming kernels take as they are; None for others.");
  m.def("gmm_autograd", &GroupedGemmAutograd, "The differentiable form of gmm_direct without trans_a.");
  m.def("gmm_gradients", &GroupedGemmGradients,
        "Both gradients of gmm, for operands the streaming kernels take as they are; None for others.");
  m.def("gmm_strided", &GroupedGemmStrided, "gmm on operands whose rows are further apart than they are long.");
  m.def("gmm_gradients_strided", &GradientsStrided, "Both gradients of gmm from such operands.");
  m.def("validate",
        [](torch::Tensor a, torch::Tensor b, torch::Tensor c, torch::Tensor batch_sizes, bool trans_a,
           bool trans_b) { Validate(a, b, c, batch_sizes, trans_a, trans_b, /*on_device=*/false); },
        "Shape, rank and dtype checks of gmm without the device checks.");
  m.def("gmm_indexed", &GroupedGemmIndexed, "gmm with fused row gather / scatter.", py::arg("a"), py::arg("b"),
        py::arg("c"), py::arg("batch_sizes"), py::arg("trans_a"), py::arg("trans_b"), py::arg("a_rows") = py::none(),
        py::arg("b_rows") = py::none(), py::arg("c_rows") = py::none());
  m.def("gmm_swiglu", &GroupedGemmSwiGLU, "silu(a @ gate) * (a @ up) with b = [gate | up].", py::arg("a"),
        py::arg("b"), py::arg("c"), py::arg("batch_sizes"), py::arg("trans_b"), py::arg("a_rows") = py::none(),
        py::arg("c_rows") = py::none());
  m.def("gmm_swiglu_keep", &GroupedGemmSwiGLUKeep, "gmm_swiglu, and gate | up for its gradient; None where they are not kept.");
  m.def("swiglu_backward", &SwiGLUBackward, "Gradients of gate | up from the gradient of silu(gate) * up.");
  m.def("sum_rows", &SumRows, "Row d of the result is the sum of the rows of src that row_index sends there.");
  m.def("pad_rows", &PadRows, "A zero-padded copy with `rows` rows of `cols` elements per batch.");
  m.def("unpad_rows", &UnpadRows, "The second tensor = the upper left corner of every batch of the first.");
  m.def("size_status", &SizeStatus,
        "Bits collected since the last call: 1 a device-resident batch size was negative, 2 they summed past the "
        "rows of a (both clamped by the kernel).");
  m.attr("status_negative_size") = GG_STATUS_NEGATIVE_SIZE;
  m.attr("status_rows_past_end") = GG_STATUS_ROWS_PAST_END;
  m.def("gmm_with_flags", &GroupedGemmWithFlags, "gmm with GG_FLAG_* bits (testing).");
  m.attr("flag_whole_tiles") = GG_FLAG_WHOLE_TILES;
  m.attr("flag_group_order") = GG_FLAG_GROUP_ORDER;
  m.def("accumulate_weight_gradient", &AccumulateWeightGradient,
        "c (fp32) += per expert a_e^T @ b_e.");
  m.def("debug_schedule", &DebugSchedule, "Per-group table derived by the on-device scheduler.");
  m.attr("max_groups_per_launch") = GG_MAX_GROUPS_PER_LAUNCH;
  m.attr("sched_cols") = GG_SCHED_COLS;
}

}  // namespace grouped_gemm
