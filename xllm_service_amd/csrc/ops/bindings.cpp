// PyTorch bindings for the MI355X (gfx950) HIP kernels.
//
// All tensor-shape/dtype validation lives here so the kernels stay lean.
#include "linear.h"
#include <hip/hip_runtime.h>
#include <ATen/autocast_mode.h>
#include <ATen/hip/tunable/Tunable.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

#include <vector>
#include <cstring>

namespace xllm {
void launch_rmsnorm(unsigned short*, const unsigned short*,
                    const unsigned short*, float, int, int, hipStream_t);
void launch_fused_add_rmsnorm(unsigned short*, unsigned short*,
                              const unsigned short*, float, int, int,
                              hipStream_t);
void launch_rope(unsigned short*, unsigned short*, const long*, const float*,
                 int, int, int, int, int, long, long, hipStream_t);
void launch_fused_rope_cache(unsigned short*, const unsigned short*,
                             const unsigned short*, unsigned short*,
                             unsigned short*, const long*, const long*,
                             const float*, int, int, int, int, int, long,
                             long, int, int, int, hipStream_t);
void launch_silu_and_mul(unsigned short*, const unsigned short*, int, int,
                         hipStream_t);
void launch_gelu_and_mul(unsigned short*, const unsigned short*, int, int,
                         hipStream_t);
void launch_reshape_and_cache(unsigned short*, unsigned short*,
                              const unsigned short*, const unsigned short*,
                              const long*, int, int, int, int, long,
                              hipStream_t);
void launch_copy_blocks(unsigned short*, unsigned short*, const long*, int,
                        long, hipStream_t);
void launch_gather_blocks(unsigned short*, unsigned short*, const long*, int,
                          long, bool, hipStream_t);
void launch_paged_attn_decode(unsigned short*, const unsigned short*,
                              const unsigned short*, const unsigned short*,
                              const int*, const int*, float*, float*, float,
                              int, int, int, int, int, long, long, bool,
                              hipStream_t);
int paged_attn_decode_parts(int, int, int, int);
long paged_attn_prefill_scratch(long, int, int, int, int, int);
void launch_paged_attn_prefill(unsigned short*, float*, const unsigned short*,
                               const unsigned short*, const unsigned short*,
                               const int*, const int*, const int*, long, int,
                               float, int, int, int, int, long, long,
                               const void* const*, const long*, long, hipStream_t);
void launch_greedy_sample(long*, const unsigned short*, int, int, hipStream_t);
void launch_mfma_gemm(unsigned short*, const unsigned short*,
                      const unsigned short*, const unsigned short*, int, int,
                      int, hipStream_t);
int skinny_gemm_splitk(int M, int N, int K);
int skinny_gemm_rows(int M);
void launch_skinny_gemm(unsigned short*, const unsigned short*,
                        const unsigned short*, const unsigned short*, float*,
                        int, int, int, hipStream_t);
int linear_takes(long M, long N, long K, bool bias, bool ends);
int linear_tiles(int M, int N, int K, int kind);
void launch_linear(unsigned short*, const unsigned short*,
                   const unsigned short*, const unsigned short*, int, int, int,
                   long, int, int, const LinearEnds&, hipStream_t);
int packed_gemm_splitk(int M, int N, int K, int S);
void launch_packed_gemm(unsigned short*, const unsigned short*,
                        unsigned short*, const unsigned short*,
                        const unsigned short*, float*, int, int, int, int,
                        hipStream_t);
int packed_gemm_pick_s(int N);
void launch_packed_gemm_probe(unsigned short*, const unsigned short*,
                              const unsigned short*, float*, int, int, int,
                              hipStream_t);
void launch_mfma_probe(float*, const unsigned short*, const unsigned short*,
                       hipStream_t);
}  // namespace xllm

namespace {

#define CHECK_BF16_CUDA(t)                                      \
  TORCH_CHECK((t).is_cuda(), #t " must be on GPU");             \
  TORCH_CHECK((t).dtype() == torch::kBFloat16, #t " must be bf16"); \
  TORCH_CHECK((t).is_contiguous(), #t " must be contiguous")

// bf16 [T, H, D] (or [T, H*D]) view: innermost contiguous, heads packed;
// rows may be strided (views into a fused qkv output)
#define CHECK_BF16_ROWVIEW(t)                                              \
  TORCH_CHECK((t).is_cuda() && (t).dtype() == torch::kBFloat16,            \
              #t " must be bf16 on GPU");                                  \
  TORCH_CHECK((t).stride(-1) == 1, #t " innermost dim must be contiguous");\
  TORCH_CHECK((t).dim() < 3 || (t).stride(1) == (t).size(2),               \
              #t " heads must be packed")

inline unsigned short* u16(torch::Tensor& t) {
  return reinterpret_cast<unsigned short*>(t.data_ptr());
}
inline const unsigned short* u16c(const torch::Tensor& t) {
  return reinterpret_cast<const unsigned short*>(t.data_ptr());
}
// every row starts at a multiple of n bytes
inline bool on_bytes(const torch::Tensor& t, int n) {
  return reinterpret_cast<uintptr_t>(t.data_ptr()) % n == 0 &&
         (t.size(0) <= 1 || t.stride(0) * 2 % n == 0);
}
inline hipStream_t cur_stream() {
  return at::hip::getCurrentHIPStream().stream();
}

void rmsnorm(torch::Tensor out, torch::Tensor x, torch::Tensor w, double eps) {
  CHECK_BF16_CUDA(out); CHECK_BF16_CUDA(x); CHECK_BF16_CUDA(w);
  const int H = x.size(-1);
  const int T = x.numel() / H;
  TORCH_CHECK(H % 8 == 0, "hidden size must be a multiple of 8");
  xllm::launch_rmsnorm(u16(out), u16c(x), u16c(w), (float)eps, T, H,
                       cur_stream());
}

void fused_add_rmsnorm(torch::Tensor x, torch::Tensor residual,
                       torch::Tensor w, double eps) {
  CHECK_BF16_CUDA(x); CHECK_BF16_CUDA(residual); CHECK_BF16_CUDA(w);
  const int H = x.size(-1);
  const int T = x.numel() / H;
  TORCH_CHECK(H % 8 == 0, "hidden size must be a multiple of 8");
  xllm::launch_fused_add_rmsnorm(u16(x), u16(residual), u16c(w), (float)eps, T,
                                 H, cur_stream());
}

void rope(torch::Tensor positions, torch::Tensor q, torch::Tensor k,
          torch::Tensor cos_sin, long head_dim, long rot_dim) {
  CHECK_BF16_ROWVIEW(q); CHECK_BF16_ROWVIEW(k);
  TORCH_CHECK(positions.dtype() == torch::kLong && positions.is_cuda());
  TORCH_CHECK(cos_sin.dtype() == torch::kFloat && cos_sin.is_cuda());
  const int T = positions.size(0);
  const int n_q = q.numel() / T / head_dim;
  const int n_k = k.numel() / T / head_dim;
  xllm::launch_rope(u16(q), u16(k), positions.data_ptr<long>(),
                    cos_sin.data_ptr<float>(), T, n_q, n_k, (int)head_dim,
                    (int)rot_dim, q.stride(0), k.stride(0), cur_stream());
}

void fused_rope_cache(torch::Tensor positions, torch::Tensor q,
                      torch::Tensor k, torch::Tensor v,
                      torch::Tensor k_cache, torch::Tensor v_cache,
                      torch::Tensor slot_mapping, torch::Tensor cos_sin,
                      long rot_dim, long ms0, long ms1) {
  // ms0/ms1: cumulative M-RoPE frequency-section bounds; 0 = 1-D rope.
  // With ms0 > 0, positions is [3, T] (temporal / height / width rows).
  CHECK_BF16_ROWVIEW(q); CHECK_BF16_ROWVIEW(k); CHECK_BF16_ROWVIEW(v);
  CHECK_BF16_CUDA(k_cache); CHECK_BF16_CUDA(v_cache);
  TORCH_CHECK(positions.dtype() == torch::kLong && positions.is_cuda() &&
              positions.is_contiguous());
  TORCH_CHECK(ms0 == 0 ? positions.dim() == 1
                       : (positions.dim() == 2 && positions.size(0) == 3));
  TORCH_CHECK(slot_mapping.dtype() == torch::kLong && slot_mapping.is_cuda());
  TORCH_CHECK(cos_sin.dtype() == torch::kFloat && cos_sin.is_cuda());
  TORCH_CHECK(k.stride(0) == v.stride(0));
  const int T = positions.size(positions.dim() - 1);
  const int n_kv = k_cache.size(1);
  const int bs = k_cache.size(2);
  const int D = k_cache.size(3);
  const int n_q = q.numel() / T / D;
  xllm::launch_fused_rope_cache(
      u16(q), u16c(k), u16c(v), u16(k_cache), u16(v_cache),
      positions.data_ptr<long>(), slot_mapping.data_ptr<long>(),
      cos_sin.data_ptr<float>(), T, n_q, n_kv, D, (int)rot_dim, q.stride(0),
      k.stride(0), bs, (int)ms0, (int)ms1, cur_stream());
}

void silu_and_mul(torch::Tensor out, torch::Tensor x) {
  CHECK_BF16_CUDA(out); CHECK_BF16_CUDA(x);
  const int I = out.size(-1);
  const int T = out.numel() / I;
  TORCH_CHECK(x.size(-1) == 2 * I && I % 8 == 0);
  xllm::launch_silu_and_mul(u16(out), u16c(x), T, I, cur_stream());
}

void gelu_and_mul(torch::Tensor out, torch::Tensor x) {
  CHECK_BF16_CUDA(out); CHECK_BF16_CUDA(x);
  const int I = out.size(-1);
  const int T = out.numel() / I;
  TORCH_CHECK(x.size(-1) == 2 * I && I % 8 == 0);
  xllm::launch_gelu_and_mul(u16(out), u16c(x), T, I, cur_stream());
}

void reshape_and_cache(torch::Tensor k, torch::Tensor v,
                       torch::Tensor k_cache, torch::Tensor v_cache,
                       torch::Tensor slot_mapping) {
  CHECK_BF16_ROWVIEW(k); CHECK_BF16_ROWVIEW(v);
  CHECK_BF16_CUDA(k_cache); CHECK_BF16_CUDA(v_cache);
  TORCH_CHECK(slot_mapping.dtype() == torch::kLong && slot_mapping.is_cuda());
  TORCH_CHECK(k.stride(0) == v.stride(0), "k/v must share row stride");
  const int T = k.size(0);
  const int n_kv = k_cache.size(1);
  const int bs = k_cache.size(2);
  const int D = k_cache.size(3);
  TORCH_CHECK(D % 8 == 0);
  xllm::launch_reshape_and_cache(u16(k_cache), u16(v_cache), u16c(k), u16c(v),
                                 slot_mapping.data_ptr<long>(), T, n_kv, D, bs,
                                 k.stride(0), cur_stream());
}

void copy_blocks(torch::Tensor k_cache, torch::Tensor v_cache,
                 torch::Tensor pairs) {
  CHECK_BF16_CUDA(k_cache); CHECK_BF16_CUDA(v_cache);
  TORCH_CHECK(pairs.dtype() == torch::kLong && pairs.is_cuda() &&
              pairs.is_contiguous());
  const long numel = (long)k_cache.size(1) * k_cache.size(2) * k_cache.size(3);
  xllm::launch_copy_blocks(u16(k_cache), u16(v_cache), pairs.data_ptr<long>(),
                           pairs.size(0), numel, cur_stream());
}

void gather_blocks(torch::Tensor staging, torch::Tensor cache,
                   torch::Tensor block_ids, bool gather) {
  CHECK_BF16_CUDA(staging); CHECK_BF16_CUDA(cache);
  TORCH_CHECK(block_ids.dtype() == torch::kLong && block_ids.is_cuda());
  const long numel = (long)cache.size(1) * cache.size(2) * cache.size(3);
  xllm::launch_gather_blocks(u16(staging), u16(cache),
                             block_ids.data_ptr<long>(), block_ids.size(0),
                             numel, gather, cur_stream());
}

void paged_attn_decode(torch::Tensor out, torch::Tensor q,
                       torch::Tensor k_cache, torch::Tensor v_cache,
                       torch::Tensor block_tables, torch::Tensor seq_lens,
                       double scale) {
  CHECK_BF16_ROWVIEW(out); CHECK_BF16_ROWVIEW(q);
  CHECK_BF16_CUDA(k_cache); CHECK_BF16_CUDA(v_cache);
  TORCH_CHECK(block_tables.dtype() == torch::kInt && block_tables.is_cuda());
  TORCH_CHECK(seq_lens.dtype() == torch::kInt && seq_lens.is_cuda());
  const int num_seqs = q.size(0);
  const int n_qheads = q.size(1);
  const int D = q.size(2);
  const int n_kv = k_cache.size(1);
  TORCH_CHECK(k_cache.size(2) == 16, "block_size must be 16");
  TORCH_CHECK(D <= 128 && D % 8 == 0, "head_dim must be <=128, mult of 8");
  TORCH_CHECK(n_qheads % n_kv == 0 && n_qheads / n_kv <= 8,
              "GQA group must be <= 8");
  int parts = 1;
  torch::Tensor ws;            // [seqs * heads][parts][D + 2], fp32, and counters
  float *ws_o = nullptr, *ws_ml = nullptr;
  const bool stream = (D == 128 || D == 64) && on_bytes(k_cache, 16) &&
                      on_bytes(v_cache, 16) && on_bytes(q, 16) &&
                      on_bytes(out, 8);
  if (stream) {
    parts = xllm::paged_attn_decode_parts(num_seqs, n_kv, D,
                                          block_tables.size(1));
    if (parts > 1) {
      const long n = (long)num_seqs * n_qheads * parts;
      ws = torch::empty({n * (D + 2) + 2L * num_seqs * n_kv}, q.options().dtype(torch::kFloat));
      ws_o = ws.data_ptr<float>();
      ws_ml = ws_o + n * D;
    }
  }
  xllm::launch_paged_attn_decode(
      u16(out), u16c(q), u16c(k_cache), u16c(v_cache),
      block_tables.data_ptr<int>(), seq_lens.data_ptr<int>(), ws_ml, ws_o,
      (float)scale, num_seqs, n_qheads, n_kv, D, block_tables.size(1),
      q.stride(0), out.stride(0), stream, cur_stream());
}

// Weights that are read after an attention, in their order: PagedAhead
struct Ahead {
  const void* at[4] = {};
  long bytes[4] = {};
  long streamed = 0;             // of the caches of decoded rows, before them
  void add(int i, const torch::Tensor& w) {
    // read by 16 bytes
    if (!w.is_contiguous() || reinterpret_cast<uintptr_t>(w.data_ptr()) % 16 != 0)
      return;
    at[i] = w.data_ptr();
    bytes[i] = w.numel() * w.element_size();
  }
};

static void prefill_attn(torch::Tensor out, torch::Tensor q,
                         torch::Tensor k_cache, torch::Tensor v_cache,
                         torch::Tensor block_tables, torch::Tensor cu_q,
                         torch::Tensor seq_lens, double scale,
                         const Ahead* ahead) {
  CHECK_BF16_ROWVIEW(out); CHECK_BF16_ROWVIEW(q);
  CHECK_BF16_CUDA(k_cache); CHECK_BF16_CUDA(v_cache);
  for (auto* t : {&block_tables, &cu_q, &seq_lens}) {
    TORCH_CHECK(t->dtype() == torch::kInt && t->is_cuda() && t->is_contiguous());
  }
  const long tokens = q.size(0);
  const int n_qheads = q.size(1);
  const int D = q.size(2);
  const int n_kv = k_cache.size(1);
  const int n_seqs = cu_q.size(0) - 1;
  TORCH_CHECK(D == 128 || D == 64, "prefill kernel: head_dim 64 or 128");
  TORCH_CHECK(k_cache.size(2) == 16, "block_size must be 16");
  // out: [tokens, heads, D] or [tokens, heads * D]; q and out may have rows
  // beyond the last prompt's, either cache pages that no table names
  const long row = (long)n_qheads * D;
  TORCH_CHECK(k_cache.size(3) == D &&
              v_cache.sizes().slice(1) == k_cache.sizes().slice(1) &&
              n_qheads % n_kv == 0 &&
              (out.dim() == 3 ? out.size(1) * out.size(2)
                              : out.size(1)) == row &&
              seq_lens.size(0) >= n_seqs && block_tables.size(0) >= n_seqs,
              "prefill kernel: shapes do not match");
  // the kernel moves caches and queries by 16 B and results by 8 B: copies of
  // what lies at other addresses
  if (!on_bytes(out, 8)) {
    auto rows = out.clone(at::MemoryFormat::Contiguous);
    prefill_attn(rows, q, k_cache, v_cache, block_tables, cu_q, seq_lens, scale,
                 ahead);
    out.copy_(rows);
    return;
  }
  for (auto* t : {&q, &k_cache, &v_cache})
    if (!on_bytes(*t, 16)) *t = t->clone(at::MemoryFormat::Contiguous);
  const long need = xllm::paged_attn_prefill_scratch(
      tokens, n_seqs, n_qheads / n_kv, n_kv, D, block_tables.size(1));
  torch::Tensor ws;
  if (need > 0) ws = torch::empty({need}, q.options().dtype(torch::kFloat));
  xllm::launch_paged_attn_prefill(
      u16(out), need > 0 ? ws.data_ptr<float>() : nullptr, u16c(q),
      u16c(k_cache), u16c(v_cache), block_tables.data_ptr<int>(),
      cu_q.data_ptr<int>(), seq_lens.data_ptr<int>(), tokens, n_seqs,
      (float)scale, n_qheads, n_kv, D, block_tables.size(1), q.stride(0),
      out.stride(0), ahead ? ahead->at : nullptr,
      ahead ? ahead->bytes : nullptr, ahead ? ahead->streamed : 0, cur_stream());
}
void paged_attn_prefill(torch::Tensor out, torch::Tensor q,
                        torch::Tensor k_cache, torch::Tensor v_cache,
                        torch::Tensor block_tables, torch::Tensor cu_q,
                        torch::Tensor seq_lens, double scale) {
  prefill_attn(out, q, k_cache, v_cache, block_tables, cu_q, seq_lens, scale,
               nullptr);
}

torch::Tensor greedy_sample(torch::Tensor logits) {
  CHECK_BF16_CUDA(logits);
  const int B = logits.size(0);
  const int V = logits.size(1);
  auto out = torch::empty({B}, logits.options().dtype(torch::kLong));
  xllm::launch_greedy_sample(out.data_ptr<long>(), u16c(logits), B, V,
                             cur_stream());
  return out;
}

torch::Tensor mfma_gemm(torch::Tensor a, torch::Tensor b,
                        c10::optional<torch::Tensor> bias) {
  // a: [M, K]; b: [N, K] (torch weight layout); returns [M, N]
  CHECK_BF16_CUDA(a); CHECK_BF16_CUDA(b);
  TORCH_CHECK(a.size(1) == b.size(1), "K mismatch");
  TORCH_CHECK(a.size(1) % 8 == 0, "K must be a multiple of 8");
  const int M = a.size(0), K = a.size(1), N = b.size(0);
  auto c = torch::empty({M, N}, a.options());
  const unsigned short* bp = nullptr;
  if (bias.has_value()) {
    CHECK_BF16_CUDA(bias.value());
    bp = u16c(bias.value());
  }
  xllm::launch_mfma_gemm(u16(c), u16c(a), u16c(b), bp, M, N, K,
                         cur_stream());
  return c;
}

torch::Tensor skinny_gemm(torch::Tensor a, torch::Tensor b,
                          c10::optional<torch::Tensor> bias) {
  // a: [M, K]; b: [N, K]; returns [M, N]
  CHECK_BF16_CUDA(a); CHECK_BF16_CUDA(b);
  const int M = a.size(0), K = a.size(1), N = b.size(0);
  TORCH_CHECK(a.size(1) == b.size(1) && M <= 256);
  TORCH_CHECK(K % 64 == 0 && N % 4 == 0);
  auto c = torch::empty({M, N}, a.options());
  const int SK = xllm::skinny_gemm_splitk(M, N, K);
  const long mpad = xllm::skinny_gemm_rows(M);   // rows of a partial result
  torch::Tensor ws;
  if (SK > 1)
    ws = torch::empty({(long)SK * mpad * N}, a.options().dtype(torch::kFloat));
  else
    ws = torch::empty({1}, a.options().dtype(torch::kFloat));
  const unsigned short* bp = nullptr;
  if (bias.has_value()) bp = u16c(bias.value());
  xllm::launch_skinny_gemm(u16(c), u16c(a), u16c(b), bp,
                           ws.data_ptr<float>(), M, N, K, cur_stream());
  return c;
}

// plain memory without a transform or a tangent
static bool plain(const torch::Tensor& t) {
  return t.layout() == torch::kStrided && !t.is_nested() &&
         !t.key_set().has_any(c10::DispatchKeySet(
             {c10::DispatchKey::FuncTorchBatched,
              c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Python,
              c10::DispatchKey::Functionalize, c10::DispatchKey::ZeroTensor,
              c10::DispatchKey::Conjugate, c10::DispatchKey::Negative})) &&
         !t._fw_grad(0).defined();
}

// Whether a call may go past torch's dispatcher: no gradient is wanted, and no
// transform, mode, trace or autocast has to see it
bool direct(const std::vector<torch::Tensor>& tensors) {
  if (c10::impl::TorchDispatchModeTLS::any_modes_set() ||
      torch::jit::tracer::isTracing() ||
      at::autocast::is_autocast_enabled(at::kCUDA))
    return false;
  const bool grad = at::GradMode::is_enabled();
  for (const auto& t : tensors)
    if (!plain(t) || (grad && t.requires_grad())) return false;
  return true;
}

// Whether torch's table of tuned products, if it is in use, names a kernel of the
// library for y [M, N] = x [M, K] w [N, K]^T
static bool tuned(long M, long N, long K, long x_stride) {
  auto* ctx = at::cuda::tunable::getTuningContext();
  if (!ctx->IsTunableOpEnabled()) return false;
  char shape[160];
  snprintf(shape, sizeof shape, "tn_%ld_%ld_%ld_ld_%ld_%ld_%ld", N, M, K, K,
           x_stride, N);
  const auto entry = ctx->GetTuningResultsManager().Lookup(
      "GemmTunableOp_BFloat16_TN", shape);
  return entry != at::cuda::tunable::ResultEntry::Null() &&
         entry != at::cuda::tunable::ResultEntry::Default();
}

// Which kernels of linear.hip take x @ w^T (+ bias), with LinearEnds' options or
// without: linear_takes, 0 for none
static int linear_kind(const torch::Tensor& x, const torch::Tensor& w,
                       const c10::optional<torch::Tensor>& bias, bool ends) {
  auto rows16 = [](const torch::Tensor& t) {
    return t.dim() == 2 && t.is_cuda() && t.dtype() == torch::kBFloat16 &&
           t.stride(1) == 1 &&
           reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
  };
  if (!((bias.has_value() ? direct({x, w, *bias}) : direct({x, w})) &&
        rows16(x) && rows16(w) && x.size(1) == w.size(1) &&
        x.stride(0) % 8 == 0 && x.stride(0) >= x.size(1) &&
        x.stride(0) < (1L << 24) && w.is_contiguous() &&
        x.device() == w.device() &&
        (!bias.has_value() ||
         (bias->dim() == 1 && bias->is_contiguous() &&
          bias->dtype() == torch::kBFloat16 && bias->size(0) == w.size(0) &&
          bias->device() == w.device()))))
    return 0;
  const long M = x.size(0), N = w.size(0), K = w.size(1);
  const int kind = xllm::linear_takes(M, N, K, bias.has_value(), ends);
  return kind != 0 && M > (N > 8192 ? 32 : 48) && !bias.has_value() &&
                 tuned(M, N, K, x.stride(0))
             ? 0
             : kind;
}

// x [..., K] @ w [N, K]^T (+ bias): the kernels of linear.hip where they take the
// call, the library elsewhere (and wherever a gradient is wanted)
torch::Tensor linear(torch::Tensor x, torch::Tensor w,
                     c10::optional<torch::Tensor> bias) {
  if (const int kind = linear_kind(x, w, bias, false)) {
    const long M = x.size(0), N = w.size(0), K = w.size(1);
    c10::OptionalDeviceGuard guard(x.device());
    auto y = torch::empty({M, N}, x.options());
    xllm::launch_linear(u16(y), u16c(x), u16c(w),
                        bias.has_value() ? u16c(*bias) : nullptr, (int)M,
                        (int)N, (int)K, x.stride(0), kind, 0, {}, cur_stream());
    return y;
  }
  return at::linear(x, w, bias.has_value() ? *bias : torch::Tensor());
}

// silu(x gates^T) (x ups^T), w = [gates | ups] by rows: one kernel where linear.hip
// takes the product (a launch, and twice the result written and read again: 24 rows,
// 2 x 4096 x 4096 18.5 us as two kernels), the same two calls as always elsewhere
torch::Tensor linear_gated(torch::Tensor x, torch::Tensor w,
                           c10::optional<torch::Tensor> bias) {
  if (!bias.has_value() && w.dim() == 2 && w.size(0) % 16 == 0) {
    if (const int kind = linear_kind(x, w, bias, true)) {
      const long M = x.size(0), N = w.size(0), K = w.size(1);
      c10::OptionalDeviceGuard guard(x.device());
      auto y = torch::empty({M, N / 2}, x.options());
      xllm::launch_linear(u16(y), u16c(x), u16c(w), nullptr, (int)M, (int)N,
                          (int)K, x.stride(0), kind, xllm::LN_GATE, {},
                          cur_stream());
      return y;
    }
  }
  const auto h = ::linear(x, w, bias);
  auto shape = h.sizes().vec();
  shape.back() /= 2;
  auto y = torch::empty(shape, h.options());
  silu_and_mul(y, h);
  return y;
}

// Rows between two products of a layer: as an RMS norm leaves them, or without their
// factors, with the sums of their squares' parts [rows][tiles] and the kernels that
// take the product which they were made for (linear_kind, asked once: torch's table
// of tuned products may change meanwhile)
struct Rows { torch::Tensor x, squares; int kind = 0; };

static xllm::LinearEnds scale_of(const Rows& in, double eps) {
  xllm::LinearEnds e;
  e.squares = in.squares.data_ptr<float>();
  e.n_squares = in.squares.size(1);
  e.eps = (float)eps;
  return e;
}

// in W^T (+ bias), or of W = [gates | ups] silu(in gates^T) (in ups^T)
static torch::Tensor product(const Rows& in, const torch::Tensor& w,
                             const c10::optional<torch::Tensor>& bias, bool gate,
                             double eps) {
  if (!in.squares.defined())
    return gate ? linear_gated(in.x, w, bias) : ::linear(in.x, w, bias);
  const long M = in.x.size(0), N = w.size(0), K = w.size(1);
  auto y = torch::empty({M, gate ? N / 2 : N}, in.x.options());
  xllm::launch_linear(u16(y), u16c(in.x), u16c(w),
                      bias.has_value() ? u16c(*bias) : nullptr, (int)M, (int)N,
                      (int)K, in.x.stride(0), in.kind,
                      xllm::LN_SCALE | (gate ? xllm::LN_GATE : 0),
                      scale_of(in, eps), cur_stream());
  return y;
}

// The rows of the next product: res += x w^T, normed. One kernel where linear.hip
// takes this product and the next one (next_w), else product and norm.
static Rows product_normed(const torch::Tensor& x, const torch::Tensor& w,
                           const torch::Tensor& res, const torch::Tensor& norm,
                           const torch::Tensor& next_w,
                           const c10::optional<torch::Tensor>& next_bias,
                           bool next_gate, double eps) {
  const c10::optional<torch::Tensor> none;
  const int kind = linear_kind(x, w, none, true);
  const long M = x.size(0), N = w.size(0), K = w.size(1);
  if (kind != 0 && res.dim() == 2 && res.is_contiguous() && res.size(0) == M &&
      res.size(1) == N && res.dtype() == torch::kBFloat16 && on_bytes(res, 16) &&
      norm.dim() == 1 && norm.size(0) == N && norm.is_contiguous() &&
      norm.dtype() == torch::kBFloat16 &&
      reinterpret_cast<uintptr_t>(norm.data_ptr()) % 16 == 0 &&
      res.is_cuda() && norm.is_cuda() &&
      !(next_gate && (next_bias.has_value() || next_w.size(0) % 16 != 0))) {
    Rows out{torch::empty({M, N}, x.options())};
    const int next = linear_kind(out.x, next_w, next_bias, true);
    const int tiles = xllm::linear_tiles((int)M, (int)N, (int)K, kind);
    out.kind = next;
    if (next != 0 && tiles % 4 == 0 && tiles <= (next == 1 ? 256 : 64)) {
      out.squares = torch::empty({M, tiles}, x.options().dtype(torch::kFloat));
      xllm::LinearEnds e;
      e.residual = reinterpret_cast<unsigned short*>(res.data_ptr());
      e.norm = u16c(norm);
      e.sums = out.squares.data_ptr<float>();
      xllm::launch_linear(u16(out.x), u16c(x), u16c(w), nullptr, (int)M, (int)N,
                          (int)K, x.stride(0), kind, xllm::LN_ADD, e,
                          cur_stream());
      return out;
    }
  }
  auto h = ::linear(x, w, none);
  fused_add_rmsnorm(h, res, norm, eps);
  return {h};
}

struct DecoderLayer {
  torch::Tensor input_norm, qkv_w;
  c10::optional<torch::Tensor> qkv_b;
  torch::Tensor o_w, post_norm, gate_up_w;
  c10::optional<torch::Tensor> gate_up_b;
  torch::Tensor down_w, k_cache, v_cache;
};

// Whether the first product of a layer rotates its heads and fills the caches itself:
// rows of a product before it, one position to a row, heads of 128 without a bias
static bool rotates(const Rows& in, const DecoderLayer& p, long heads,
                    const torch::Tensor& positions, const torch::Tensor& slots,
                    const torch::Tensor& cos_sin) {
  const long T = in.x.size(0);
  auto cache = [&](const torch::Tensor& t) {
    return t.is_cuda() && t.dim() == 4 && t.dtype() == torch::kBFloat16 &&
           t.is_contiguous() && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
  };
  auto rows = [&](const torch::Tensor& t) {
    return t.is_cuda() && t.dtype() == torch::kLong && t.dim() == 1 &&
           t.is_contiguous() && t.size(0) == T;
  };
  return in.squares.defined() && !p.qkv_b.has_value() && cache(p.k_cache) &&
         cache(p.v_cache) && p.k_cache.sizes() == p.v_cache.sizes() &&
         p.k_cache.size(3) == xllm::LN_HEAD &&
         p.qkv_w.size(0) == (heads + 2 * p.k_cache.size(1)) * xllm::LN_HEAD &&
         rows(positions) && rows(slots) && cos_sin.is_cuda() &&
         cos_sin.dtype() == torch::kFloat && cos_sin.is_contiguous() &&
         cos_sin.dim() == 2 && cos_sin.size(1) == xllm::LN_HEAD &&
         reinterpret_cast<uintptr_t>(cos_sin.data_ptr()) % 16 == 0;
}

// Layers of the dense decoders (models/llama.py) over prompt rows and decode rows:
// what their modules call, in their order, without the interpreter between two
// launches (75 us of host time a layer, 25 here, where the kernels of 300 rows of 2048
// take 70), and without launches for the norms between two products and for the rotation
// and the cache rows of what comes out of one (LN_ROPE). Nothing, with
// nothing done, where torch has to see the calls.
c10::optional<std::tuple<torch::Tensor, torch::Tensor>> decoder_layers(
    torch::Tensor x, c10::optional<torch::Tensor> residual,
    std::vector<std::vector<c10::optional<torch::Tensor>>> weights, double eps,
    long heads, double scale, torch::Tensor positions,
    torch::Tensor slot_mapping, torch::Tensor cos_sin, long ms0, long ms1,
    long n_prefill, long n_decode, c10::optional<torch::Tensor> prefill_tables,
    c10::optional<torch::Tensor> cu_q,
    c10::optional<torch::Tensor> prefill_lens,
    c10::optional<torch::Tensor> decode_tables,
    c10::optional<torch::Tensor> decode_lens) {
  std::vector<DecoderLayer> layers;
  for (const auto& w : weights) {
    TORCH_CHECK(w.size() == 10, "decoder layer: ten tensors");
    layers.push_back({w[0].value(), w[1].value(), w[2], w[3].value(),
                      w[4].value(), w[5].value(), w[6], w[7].value(),
                      w[8].value(), w[9].value()});
  }
  TORCH_CHECK(!layers.empty(), "decoder layers: none");
  for (const auto& p : layers)
    if (!direct({x, p.input_norm, p.qkv_w, p.o_w, p.post_norm, p.gate_up_w,
                 p.down_w, p.k_cache, p.v_cache}))
      return c10::nullopt;
  c10::OptionalDeviceGuard guard(x.device());
  torch::Tensor res;
  Rows in;
  if (residual.has_value()) {
    res = *residual;
    in.x = x;
    fused_add_rmsnorm(in.x, res, layers[0].input_norm, eps);
  } else {
    res = x;
    in.x = torch::empty_like(x);
    rmsnorm(in.x, x, layers[0].input_norm, eps);
  }
  for (size_t i = 0; i < layers.size(); i++) {
    const auto& p = layers[i];
    const long T = in.x.size(0), D = p.k_cache.size(3), n_kv = p.k_cache.size(1);
    torch::Tensor q;
    if (ms0 == 0 && rotates(in, p, heads, positions, slot_mapping, cos_sin)) {
      q = torch::empty({T, heads, D}, in.x.options());
      auto e = scale_of(in, eps);
      e.positions = positions.data_ptr<long>();
      e.slots = slot_mapping.data_ptr<long>();
      e.cos_sin = cos_sin.data_ptr<float>();
      e.k_cache = reinterpret_cast<unsigned short*>(p.k_cache.data_ptr());
      e.v_cache = reinterpret_cast<unsigned short*>(p.v_cache.data_ptr());
      e.n_q = (int)heads;
      e.n_kv = (int)n_kv;
      e.block = (int)p.k_cache.size(2);
      xllm::launch_linear(u16(q), u16c(in.x), u16c(p.qkv_w), nullptr, (int)T,
                          (int)p.qkv_w.size(0), (int)p.qkv_w.size(1),
                          in.x.stride(0), in.kind,
                          xllm::LN_SCALE | xllm::LN_ROPE, e, cur_stream());
    } else {
      const auto qkv = product(in, p.qkv_w, p.qkv_b, false, eps);
      const long row = qkv.stride(0), at = qkv.storage_offset();
      TORCH_CHECK(qkv.dim() == 2 && qkv.size(1) == (heads + 2 * n_kv) * D &&
                  qkv.stride(1) == 1, "decoder layer: shapes do not match");
      q = qkv.as_strided({T, heads, D}, {row, D, 1}, at);
      const auto k = qkv.as_strided({T, n_kv, D}, {row, D, 1}, at + heads * D);
      const auto v =
          qkv.as_strided({T, n_kv, D}, {row, D, 1}, at + (heads + n_kv) * D);
      fused_rope_cache(positions, q, k, v, p.k_cache, p.v_cache, slot_mapping,
                       cos_sin, D, ms0, ms1);
    }
    auto out = torch::empty({T, heads * D}, q.options());
    const auto out3 = out.view({T, heads, D});
    if (n_prefill > 0) {
      Ahead ahead;
      ahead.add(0, p.o_w);
      ahead.add(1, p.gate_up_w);
      ahead.add(2, p.down_w);
      if (i + 1 < layers.size()) ahead.add(3, layers[i + 1].qkv_w);
      if (n_decode > 0)
        ahead.streamed = decode_tables.value().numel() * 4 *
                         p.k_cache.size(1) * p.k_cache.size(2) * D;
      prefill_attn(out3.slice(0, 0, n_prefill), q.slice(0, 0, n_prefill),
                   p.k_cache, p.v_cache, prefill_tables.value(), cu_q.value(),
                   prefill_lens.value(), scale, &ahead);
    }
    if (n_decode > 0)
      paged_attn_decode(out3.slice(0, n_prefill), q.slice(0, n_prefill),
                        p.k_cache, p.v_cache, decode_tables.value(),
                        decode_lens.value(), scale);
    in = product_normed(out, p.o_w, res, p.post_norm, p.gate_up_w, p.gate_up_b,
                        true, eps);
    const auto act = product(in, p.gate_up_w, p.gate_up_b, true, eps);
    if (i + 1 == layers.size())
      return std::make_tuple(::linear(act, p.down_w, c10::nullopt), res);
    const auto& next = layers[i + 1];
    in = product_normed(act, p.down_w, res, next.input_norm, next.qkv_w,
                        next.qkv_b, false, eps);
  }
  return c10::nullopt;
}

torch::Tensor packed_gemm(torch::Tensor a, torch::Tensor wp, int64_t N,
                          c10::optional<torch::Tensor> bias,
                          int64_t s_override) {
  // a: [M, K]; wp: W[N,K] pre-packed by ops.pack_gemm_weight; returns [M, N]
  CHECK_BF16_CUDA(a); CHECK_BF16_CUDA(wp);
  const int M = a.size(0), K = a.size(1);
  TORCH_CHECK(wp.numel() == (long)N * K, "packed weight size mismatch");
  TORCH_CHECK(K % 256 == 0 && N % 64 == 0 && M <= 128);
  auto c = torch::empty({M, (long)N}, a.options());
  const int S = s_override > 0 ? (int)s_override
                               : xllm::packed_gemm_pick_s((int)N);
  TORCH_CHECK(N % (64 * S) == 0, "N not divisible for S");
  const int SK = xllm::packed_gemm_splitk(M, (int)N, K, S);
  const long mpad = M <= 16 ? 16 : M <= 32 ? 32 : M <= 64 ? 64 : 128;
  torch::Tensor ws;
  if (SK > 1)
    ws = torch::empty({(long)SK * mpad * N}, a.options().dtype(torch::kFloat));
  else
    ws = torch::empty({1}, a.options().dtype(torch::kFloat));
  const unsigned short* bp = nullptr;
  if (bias.has_value()) bp = u16c(bias.value());
  const long mt = mpad / 16;
  auto ap = torch::empty({(long)(K / 32) * mt * 512}, a.options());
  xllm::launch_packed_gemm(u16(c), u16c(a), u16(ap), u16c(wp), bp,
                           ws.data_ptr<float>(), M, (int)N, K, S,
                           cur_stream());
  return c;
}

torch::Tensor packed_gemm_probe(torch::Tensor a, torch::Tensor wp,
                                int64_t N) {
  // W-stream timing probe: output is garbage (A loads compiled out)
  CHECK_BF16_CUDA(a); CHECK_BF16_CUDA(wp);
  const int M = a.size(0), K = a.size(1);
  auto c = torch::empty({M, (long)N}, a.options());
  const int SK = xllm::packed_gemm_splitk(M, (int)N, K, 1);
  torch::Tensor ws;
  if (SK > 1)
    ws = torch::empty({(long)SK * 64 * N}, a.options().dtype(torch::kFloat));
  else
    ws = torch::empty({1}, a.options().dtype(torch::kFloat));
  xllm::launch_packed_gemm_probe(u16(c), u16c(a), u16c(wp),
                                 ws.data_ptr<float>(), M, (int)N, K,
                                 cur_stream());
  return c;
}

torch::Tensor mfma_probe_16x16x32(torch::Tensor a, torch::Tensor b) {
  CHECK_BF16_CUDA(a); CHECK_BF16_CUDA(b);
  TORCH_CHECK(a.size(0) == 16 && a.size(1) == 32);
  TORCH_CHECK(b.size(0) == 32 && b.size(1) == 16);
  auto c = torch::empty({16, 16}, a.options().dtype(torch::kFloat));
  xllm::launch_mfma_probe(c.data_ptr<float>(), u16c(a), u16c(b), cur_stream());
  return c;
}

// ------ cross-GPU KV-block migration over xGMI ----------------------------------
// Direct peer copy of whole blocks: both caches must have identical geometry.
// Contiguous runs of (src,dst) pairs collapse into single hipMemcpyPeerAsync
// calls on the CURRENT stream (callers use a dedicated side stream to overlap
// with decode; see engine/kv_migration.py).
void migrate_blocks_peer(torch::Tensor dst_cache, long dst_device,
                         torch::Tensor src_cache, long src_device,
                         std::vector<long> src_blocks,
                         std::vector<long> dst_blocks) {
  TORCH_CHECK(src_blocks.size() == dst_blocks.size());
  const long numel =
      (long)src_cache.size(1) * src_cache.size(2) * src_cache.size(3);
  const long bytes = numel * 2;  // bf16
  char* dst = reinterpret_cast<char*>(dst_cache.data_ptr());
  const char* src = reinterpret_cast<const char*>(src_cache.data_ptr());
  hipStream_t stream = cur_stream();
  size_t i = 0;
  while (i < src_blocks.size()) {
    // collapse contiguous runs
    size_t j = i + 1;
    while (j < src_blocks.size() && src_blocks[j] == src_blocks[j - 1] + 1 &&
           dst_blocks[j] == dst_blocks[j - 1] + 1)
      j++;
    const long n = (long)(j - i);
    hipError_t err = hipMemcpyPeerAsync(
        dst + dst_blocks[i] * bytes, (int)dst_device,
        src + src_blocks[i] * bytes, (int)src_device, (size_t)(n * bytes),
        stream);
    TORCH_CHECK(err == hipSuccess, "hipMemcpyPeerAsync failed: ",
                hipGetErrorString(err));
    i = j;
  }
}

// ---- HIP IPC: cross-process cache sharing for same-node KV migration ----
// A decode worker opens the prefill worker's cache once at LinkInstance
// time, then pulls blocks with device-to-device copies over xGMI.
std::vector<char> ipc_get_handle(torch::Tensor t) {
  TORCH_CHECK(t.is_cuda());
  hipIpcMemHandle_t h;
  hipError_t err = hipIpcGetMemHandle(&h, t.data_ptr());
  TORCH_CHECK(err == hipSuccess, "hipIpcGetMemHandle: ",
              hipGetErrorString(err));
  return std::vector<char>(reinterpret_cast<char*>(&h),
                           reinterpret_cast<char*>(&h) + sizeof(h));
}

int64_t ipc_open_handle(std::vector<char> handle_bytes, long device) {
  TORCH_CHECK(handle_bytes.size() == sizeof(hipIpcMemHandle_t));
  hipIpcMemHandle_t h;
  memcpy(&h, handle_bytes.data(), sizeof(h));
  hipSetDevice((int)device);
  void* ptr = nullptr;
  hipError_t err =
      hipIpcOpenMemHandle(&ptr, h, hipIpcMemLazyEnablePeerAccess);
  TORCH_CHECK(err == hipSuccess, "hipIpcOpenMemHandle: ",
              hipGetErrorString(err));
  return reinterpret_cast<int64_t>(ptr);
}

void ipc_close_handle(int64_t ptr) {
  hipIpcCloseMemHandle(reinterpret_cast<void*>(ptr));
}

// Pull blocks from a peer cache (opened via IPC) into the local cache.
// Both caches share geometry; contiguous runs collapse into single copies.
void migrate_blocks_from_ptr(torch::Tensor dst_cache, int64_t src_ptr,
                             long src_device, long dst_device,
                             std::vector<long> src_blocks,
                             std::vector<long> dst_blocks) {
  TORCH_CHECK(src_blocks.size() == dst_blocks.size());
  const long numel =
      (long)dst_cache.size(1) * dst_cache.size(2) * dst_cache.size(3);
  const long bytes = numel * dst_cache.element_size();
  char* dst = reinterpret_cast<char*>(dst_cache.data_ptr());
  const char* src = reinterpret_cast<const char*>(src_ptr);
  hipStream_t stream = cur_stream();
  size_t i = 0;
  while (i < src_blocks.size()) {
    size_t j = i + 1;
    while (j < src_blocks.size() && src_blocks[j] == src_blocks[j - 1] + 1 &&
           dst_blocks[j] == dst_blocks[j - 1] + 1)
      j++;
    const long n = (long)(j - i);
    hipError_t err;
    if (src_device == dst_device) {
      err = hipMemcpyAsync(dst + dst_blocks[i] * bytes,
                           src + src_blocks[i] * bytes, (size_t)(n * bytes),
                           hipMemcpyDeviceToDevice, stream);
    } else {
      err = hipMemcpyPeerAsync(dst + dst_blocks[i] * bytes, (int)dst_device,
                               src + src_blocks[i] * bytes, (int)src_device,
                               (size_t)(n * bytes), stream);
    }
    TORCH_CHECK(err == hipSuccess, "block migration copy failed: ",
                hipGetErrorString(err));
    i = j;
  }
}

// ---- KV block swap GPU<->CPU (the "dram" cache tier) ---------------------
// Contiguous (src,dst) runs collapse into single async copies on the
// current stream; callers use a side stream + synchronize.
void swap_blocks(torch::Tensor dst_cache, torch::Tensor src_cache,
                 std::vector<long> src_blocks, std::vector<long> dst_blocks) {
  TORCH_CHECK(src_blocks.size() == dst_blocks.size());
  TORCH_CHECK(src_cache.element_size() == dst_cache.element_size());
  const long numel =
      (long)src_cache.size(1) * src_cache.size(2) * src_cache.size(3);
  const long bytes = numel * src_cache.element_size();
  char* dst = reinterpret_cast<char*>(dst_cache.data_ptr());
  const char* src = reinterpret_cast<const char*>(src_cache.data_ptr());
  hipMemcpyKind kind =
      src_cache.is_cuda()
          ? (dst_cache.is_cuda() ? hipMemcpyDeviceToDevice
                                 : hipMemcpyDeviceToHost)
          : hipMemcpyHostToDevice;
  hipStream_t stream = cur_stream();
  size_t i = 0;
  while (i < src_blocks.size()) {
    size_t j = i + 1;
    while (j < src_blocks.size() && src_blocks[j] == src_blocks[j - 1] + 1 &&
           dst_blocks[j] == dst_blocks[j - 1] + 1)
      j++;
    const long n = (long)(j - i);
    hipError_t err = hipMemcpyAsync(dst + dst_blocks[i] * bytes,
                                    src + src_blocks[i] * bytes,
                                    (size_t)(n * bytes), kind, stream);
    TORCH_CHECK(err == hipSuccess, "swap_blocks copy failed: ",
                hipGetErrorString(err));
    i = j;
  }
}

void enable_peer_access(long device, long peer) {
  int can = 0;
  hipError_t err = hipDeviceCanAccessPeer(&can, (int)device, (int)peer);
  TORCH_CHECK(err == hipSuccess && can, "no P2P path between GPUs ", device,
              " and ", peer);
  hipSetDevice((int)device);
  err = hipDeviceEnablePeerAccess((int)peer, 0);
  TORCH_CHECK(err == hipSuccess || err == hipErrorPeerAccessAlreadyEnabled,
              "hipDeviceEnablePeerAccess failed: ", hipGetErrorString(err));
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("rmsnorm", &rmsnorm);
  m.def("fused_add_rmsnorm", &fused_add_rmsnorm);
  m.def("rope", &rope);
  m.def("fused_rope_cache", &fused_rope_cache);
  m.def("silu_and_mul", &silu_and_mul);
  m.def("gelu_and_mul", &gelu_and_mul);
  m.def("reshape_and_cache", &reshape_and_cache);
  m.def("copy_blocks", &copy_blocks);
  m.def("gather_blocks", &gather_blocks);
  m.def("paged_attn_decode", &paged_attn_decode);
  m.def("paged_attn_prefill", &paged_attn_prefill);
  m.def("greedy_sample", &greedy_sample);
  m.def("mfma_probe_16x16x32", &mfma_probe_16x16x32);
  m.def("mfma_gemm", &mfma_gemm);
  m.def("skinny_gemm", &skinny_gemm);
  m.def("linear", &linear);
  m.def("linear_gated", &linear_gated);
  m.def("direct", &direct);
  m.def("decoder_layers", &decoder_layers);
  m.def("packed_gemm", &packed_gemm);
  m.def("packed_gemm_probe", &packed_gemm_probe);
  m.def("migrate_blocks_peer", &migrate_blocks_peer);
  m.def("ipc_get_handle", &ipc_get_handle);
  m.def("ipc_open_handle", &ipc_open_handle);
  m.def("ipc_close_handle", &ipc_close_handle);
  m.def("migrate_blocks_from_ptr", &migrate_blocks_from_ptr);
  m.def("swap_blocks", &swap_blocks);
  m.def("enable_peer_access", &enable_peer_access);
}
