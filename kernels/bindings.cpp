// Torch extension bindings for the CDNA4 kernels.
// Built in-tree as vllm_tgis_adapter_amd/_C.so by kernels/build.py
// (hipcc --offload-arch=gfx950).

#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>

// launchers (defined in the .hip translation units)
template <typename T>
void launch_rms_norm(T*, const T*, const T*, float, int, int, hipStream_t);
template <typename T>
void launch_fused_add_rms_norm(T*, T*, const T*, float, int, int, hipStream_t);
template <typename T>
void launch_silu_and_mul(T*, const T*, int, int, hipStream_t);
template <typename T>
void launch_rotary_embedding(const long*, T*, const T*, T*, const float*, int, int,
                             int, int, long, long, hipStream_t);
template <typename T>
void launch_reshape_and_cache(const T*, const T*, T*, T*, const long*, int,
                              int, long, long, hipStream_t);
void launch_mfma_probe_32(const unsigned short*, const unsigned short*, float*,
                          hipStream_t);
void launch_mfma_probe_16(const unsigned short*, const unsigned short*, float*,
                          hipStream_t);
int gemm_skinny_num_ksplit(int N, int K, int M);
void launch_logsoftmax_topk(float*, int*, float*, int*,
                            const __hip_bfloat16*, const long*, int, int,
                            int, hipStream_t);
void launch_gemm_tile(__hip_bfloat16*, const __hip_bfloat16*,
                      const __hip_bfloat16*, int, int, int, hipStream_t);
void launch_xgmi_allreduce(const unsigned long long*, __hip_bfloat16*,
                           const __hip_bfloat16*, long, long, int, int,
                           hipStream_t);
void launch_reshape_and_cache_fp8(const __hip_bfloat16*,
                                  const __hip_bfloat16*, unsigned char*,
                                  unsigned char*, const long*, int, int, long,
                                  long, hipStream_t);
int gemm_stream_parts(int qbits, int M, int N, int K, bool gated);
void launch_rotary_cache(const long*, __hip_bfloat16*, const __hip_bfloat16*,
                         const __hip_bfloat16*, const __hip_bfloat16*, const float*, void*, void*,
                         const long*, int, int, int, int, long, long, long, bool, hipStream_t);
void launch_decode_inputs(const long*, long*, long*, long*, int*, int*, int*, int, int, int, int,
                          hipStream_t);
int gemm_ring_plan(int M, int N, int K, bool gated);
void launch_gemm_ring_parts(__hip_bfloat16*, float*, const __hip_bfloat16*,
                            const __hip_bfloat16*, int, int, int, int, hipStream_t);
bool gemm_ring_takes(int N, int K, int plan, bool gated);
bool gemm_ring_reads_once(int M, int N, int K, int plan, bool gated);
int gemm_ring_lora_cuts(int M, int K, int L, int PR, int plan);
bool gemm_ring_lora_wins(long M, long N, long K, int rank);
void launch_gemm_ring_lora(__hip_bfloat16*, float*, const __hip_bfloat16*, const __hip_bfloat16*,
                           int, int, int, int, float*, const __hip_bfloat16*, const int*, int, int,
                           int, hipStream_t);
bool gemm_ring_wins(long M, long N, long K, bool gated);
bool gemm_block_takes(long M, long N, long K);
int gemm_tiles_route(long M, long N, long K);
int moe_tile(int mean, int experts, long columns, int K, bool gated);
void launch_gemm_ring(__hip_bfloat16*, float*, const __hip_bfloat16*, const __hip_bfloat16*, int,
                      int, int, int, bool, hipStream_t);
void launch_gemm_stream(__hip_bfloat16*, float*, const __hip_bfloat16*, const __hip_bfloat16*,
                        int, int, int, int, hipStream_t);
bool gemm_row_fits(int K);
int gemm_row_form(int qbits, int mode, int N, int K);
void launch_gemm_row_norm_gated(__hip_bfloat16*, __hip_bfloat16*, const __hip_bfloat16*,
                                const __hip_bfloat16*, const __hip_bfloat16*, float, const void*,
                                const float*, int, int, int, hipStream_t);
void launch_gemm_row_norm_turn(__hip_bfloat16*, __hip_bfloat16*, const __hip_bfloat16*,
                               const __hip_bfloat16*, const __hip_bfloat16*, float, const void*,
                               const float*, int, int, const long*, const long*, const float*,
                               void*, void*, int, int, int, bool, hipStream_t);
void launch_gemm_stream_gated(__hip_bfloat16*, float*, const __hip_bfloat16*,
                              const __hip_bfloat16*, int, int, int, int, hipStream_t);
void launch_gemm_stream_q(__hip_bfloat16*, float*, const __hip_bfloat16*, const unsigned char*,
                          const float*, int, int, int, int, int, hipStream_t);
void launch_gemm_skinny(__hip_bfloat16*, float*, const __hip_bfloat16*,
                        const __hip_bfloat16*, int, int, int, int,
                        hipStream_t);
void launch_gemm_skinny_gated(__hip_bfloat16*, float*, const __hip_bfloat16*,
                              const __hip_bfloat16*, int, int, int, int,
                              hipStream_t);
int gemm_panel_plan(int M, int N, int K, int qbits);
int gemm_panel_gated_plan(int M, int N, int K, int qbits);
int gemm_panel_few_plan(int M, int N, int K, int qbits);
void launch_gemm_panel_gated(__hip_bfloat16*, const __hip_bfloat16*, const unsigned char*,
                             const float*, int, int, int, int, int, hipStream_t);
void launch_gemm_block_q(__hip_bfloat16*, float*, const __hip_bfloat16*, const unsigned char*,
                         const float*, int, int, int, int, int, hipStream_t);
void launch_widen_weight(__hip_bfloat16*, const unsigned char*, const float*, int, long, int,
                         hipStream_t);
struct LoraCols {
  int end[3], shift[3];
};
int lora_shrink_cuts(int T, int K);
bool lora_tiles_win(int T, int L, int R, int W);
void launch_lora_shrink_tiles(float*, const __hip_bfloat16*, const __hip_bfloat16*, const int*,
                              int, int, int, int, int, hipStream_t);
void launch_lora_finish(__hip_bfloat16*, const __hip_bfloat16*, const float*, const float*,
                        const __hip_bfloat16*, const int*, const float*, const LoraCols&, int, int, int,
                        int, int, int, int, int, bool, hipStream_t);
void launch_lora_tiles(__hip_bfloat16*, float*, const __hip_bfloat16*, const __hip_bfloat16*,
                       const __hip_bfloat16*, const int*, const float*, const LoraCols&, int,
                       int, int, int, int, int, int, int, hipStream_t);
void launch_lora_slots(int*, const int*, const int*, int, int, hipStream_t);
template <typename T>
void launch_lora_shrink(float*, const T*, const T*, const int*, int, int, int,
                        hipStream_t);
template <typename T>
void launch_lora_expand(T*, const float*, const T*, const int*, const float*,
                        int, int, int, int, int, hipStream_t);
template <typename T>
void launch_sample_argmax(long*, const T*, const float*, const float*, int,
                          int, hipStream_t);
void launch_moe_gemm(__hip_bfloat16*, const __hip_bfloat16*, const __hip_bfloat16*, const int*,
                     const int*, int, int, int, int, int, float*, hipStream_t);
long moe_gemm_scratch(int E, int N, int K, int T, int mode);
int moe_topk_max_experts();
int moe_topk_max_top();
void launch_moe_topk(int*, float*, const __hip_bfloat16*, const __hip_bfloat16*, int, int, int,
                     int, hipStream_t);
void launch_moe_group(int*, int*, int*, const int*, int, int, int, hipStream_t);
void launch_moe_sum(__hip_bfloat16*, const __hip_bfloat16*, const int*, const float*, int, int,
                    int, hipStream_t);

// paged attention (bindings_attn.cpp, shared with the `_C_attn` extension)
void register_attention_ops(pybind11::module& m);

namespace {

hipStream_t current_stream() {
  return at::hip::getCurrentHIPStream().stream();
}

template <typename T>
T* ptr(torch::Tensor& t) {
  return reinterpret_cast<T*>(t.data_ptr());
}
template <typename T>
const T* cptr(const torch::Tensor& t) {
  return reinterpret_cast<const T*>(t.data_ptr());
}

#define DISPATCH_FLOATING(DTYPE, BODY)                                   \
  switch (DTYPE) {                                                       \
    case at::ScalarType::BFloat16: {                                     \
      using scalar_t = __hip_bfloat16;                                   \
      BODY;                                                              \
      break;                                                             \
    }                                                                    \
    case at::ScalarType::Half: {                                         \
      using scalar_t = __half;                                           \
      BODY;                                                              \
      break;                                                             \
    }                                                                    \
    case at::ScalarType::Float: {                                        \
      using scalar_t = float;                                            \
      BODY;                                                              \
      break;                                                             \
    }                                                                    \
    default:                                                             \
      TORCH_CHECK(false, "unsupported dtype");                           \
  }

void rms_norm(torch::Tensor out, torch::Tensor input, torch::Tensor weight,
              double eps) {
  const int hidden = input.size(-1);
  const int rows = input.numel() / hidden;
  TORCH_CHECK(input.is_contiguous() && out.is_contiguous());
  TORCH_CHECK(hidden % 8 == 0, "hidden must be a multiple of 8");
  DISPATCH_FLOATING(input.scalar_type(), {
    launch_rms_norm<scalar_t>(ptr<scalar_t>(out), cptr<scalar_t>(input),
                              cptr<scalar_t>(weight), (float)eps, rows, hidden,
                              current_stream());
  });
}

void fused_add_rms_norm(torch::Tensor x, torch::Tensor residual,
                        torch::Tensor weight, double eps) {
  const int hidden = x.size(-1);
  const int rows = x.numel() / hidden;
  TORCH_CHECK(x.is_contiguous() && residual.is_contiguous());
  DISPATCH_FLOATING(x.scalar_type(), {
    launch_fused_add_rms_norm<scalar_t>(
        ptr<scalar_t>(x), ptr<scalar_t>(residual), cptr<scalar_t>(weight),
        (float)eps, rows, hidden, current_stream());
  });
}

void silu_and_mul(torch::Tensor out, torch::Tensor x) {
  const int d = out.size(-1);
  const int rows = out.numel() / d;
  TORCH_CHECK(x.size(-1) == 2 * d);
  TORCH_CHECK(d % 8 == 0, "intermediate size must be a multiple of 8");
  DISPATCH_FLOATING(x.scalar_type(), {
    launch_silu_and_mul<scalar_t>(ptr<scalar_t>(out), cptr<scalar_t>(x), rows,
                                  d, current_stream());
  });
}

// Elements between the starts of a [rows, ...] tensor's rows, whose own elements
// are dense.
int64_t row_stride(const torch::Tensor& t, const char* name) {
  if (t.is_contiguous() && t.size(0) > 0) return t.numel() / t.size(0);
  int64_t want = 1;
  for (int64_t d = t.dim() - 1; d > 0; --d) {
    TORCH_CHECK(t.size(d) == 1 || t.stride(d) == want, name, ": rows must be dense");
    want *= t.size(d);
  }
  return t.size(0) > 1 ? t.stride(0) : want;
}

void rotary_embedding(torch::Tensor positions, torch::Tensor q_out, torch::Tensor q,
                      torch::Tensor k, int64_t head_dim,
                      torch::Tensor cos_sin_cache) {
  const int tokens = positions.size(0);
  const int nq = q.size(-1) / head_dim;
  const int nk = k.size(-1) / head_dim;
  TORCH_CHECK(positions.scalar_type() == at::ScalarType::Long);
  TORCH_CHECK(cos_sin_cache.scalar_type() == at::ScalarType::Float);
  TORCH_CHECK(q.dim() == 2 && k.dim() == 2 && q.size(0) == tokens && k.size(0) == tokens,
              "q and k must be [tokens, heads * head_dim]");
  TORCH_CHECK(q_out.is_contiguous() && q_out.sizes() == q.sizes() &&
              q_out.scalar_type() == q.scalar_type() && k.scalar_type() == q.scalar_type());
  DISPATCH_FLOATING(q.scalar_type(), {
    launch_rotary_embedding<scalar_t>(
        positions.data_ptr<long>(), ptr<scalar_t>(q_out), cptr<scalar_t>(q),
        ptr<scalar_t>(k), cos_sin_cache.data_ptr<float>(), tokens, nq, nk, (int)head_dim,
        row_stride(q, "q"), row_stride(k, "k"), current_stream());
  });
}

void reshape_and_cache(torch::Tensor k, torch::Tensor v, torch::Tensor k_cache,
                       torch::Tensor v_cache, torch::Tensor slot_mapping) {
  const int tokens = k.size(0);
  const int row_elems = k_cache.size(2) * k_cache.size(3);
  TORCH_CHECK(slot_mapping.scalar_type() == at::ScalarType::Long);
  // the copies are 16 bytes wide
  const int64_t wide = 16 / k.element_size();
  auto lined_up = [&](const torch::Tensor& t) {
    return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0 &&
           (t.is_contiguous() || t.size(0) <= 1 || t.stride(0) % wide == 0);
  };
  if (!lined_up(k)) k = k.contiguous();
  if (!lined_up(v)) v = v.contiguous();
  const int64_t ks = row_stride(k, "k"), vs = row_stride(v, "v");
  if (k_cache.scalar_type() == at::ScalarType::Byte) {
    TORCH_CHECK(k.scalar_type() == at::ScalarType::BFloat16,
                "fp8 KV cache takes bf16 K/V inputs");
    TORCH_CHECK(row_elems % 8 == 0);
    launch_reshape_and_cache_fp8(
        reinterpret_cast<const __hip_bfloat16*>(k.data_ptr()),
        reinterpret_cast<const __hip_bfloat16*>(v.data_ptr()),
        reinterpret_cast<unsigned char*>(k_cache.data_ptr()),
        reinterpret_cast<unsigned char*>(v_cache.data_ptr()),
        slot_mapping.data_ptr<long>(), tokens, row_elems, ks, vs, current_stream());
    return;
  }
  DISPATCH_FLOATING(k.scalar_type(), {
    launch_reshape_and_cache<scalar_t>(
        cptr<scalar_t>(k), cptr<scalar_t>(v), ptr<scalar_t>(k_cache),
        ptr<scalar_t>(v_cache), slot_mapping.data_ptr<long>(), tokens,
        row_elems, ks, vs, current_stream());
  });
}

// q turned into q_out, k turned and v into the cache, in one launch (bf16)
void rotary_cache(torch::Tensor positions, torch::Tensor q_out, torch::Tensor q, torch::Tensor k,
                  torch::Tensor v, int64_t head_dim, torch::Tensor cos_sin_cache,
                  torch::Tensor k_cache, torch::Tensor v_cache, torch::Tensor slot_mapping) {
  const int64_t tokens = positions.size(0), nq = q.size(-1) / head_dim, nk = k.size(-1) / head_dim;
  for (const auto& t : {q_out, q, k, v})
    TORCH_CHECK(t.is_cuda() && t.scalar_type() == at::ScalarType::BFloat16 && t.dim() == 2 &&
                t.size(0) == tokens && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0);
  TORCH_CHECK(head_dim % 16 == 0 && nq * head_dim == q.size(1) && nk * head_dim == k.size(1) &&
              v.size(1) == k.size(1) && q_out.size(1) == q.size(1) && q_out.is_contiguous());
  const int64_t qs = row_stride(q, "q"), ks = row_stride(k, "k"), vs = row_stride(v, "v");
  TORCH_CHECK(qs % 8 == 0 && ks % 8 == 0 && vs % 8 == 0, "rows start at 16 bytes");
  TORCH_CHECK(positions.scalar_type() == at::ScalarType::Long && positions.is_contiguous() &&
              slot_mapping.scalar_type() == at::ScalarType::Long && slot_mapping.is_contiguous() &&
              slot_mapping.numel() >= tokens);
  TORCH_CHECK(cos_sin_cache.scalar_type() == at::ScalarType::Float &&
              cos_sin_cache.is_contiguous() && cos_sin_cache.size(-1) == head_dim);
  const bool fp8 = k_cache.scalar_type() == at::ScalarType::Byte;
  TORCH_CHECK(k_cache.scalar_type() == v_cache.scalar_type() &&
              (fp8 || k_cache.scalar_type() == at::ScalarType::BFloat16));
  TORCH_CHECK(k_cache.is_contiguous() && v_cache.is_contiguous() && k_cache.size(2) == nk &&
              k_cache.size(3) == head_dim);
  if (tokens == 0) return;
  launch_rotary_cache(positions.data_ptr<long>(), ptr<__hip_bfloat16>(q_out),
                      cptr<__hip_bfloat16>(q), cptr<__hip_bfloat16>(k), cptr<__hip_bfloat16>(v),
                      cos_sin_cache.data_ptr<float>(), k_cache.data_ptr(), v_cache.data_ptr(),
                      slot_mapping.data_ptr<long>(), (int)tokens, (int)nq, (int)nk, (int)head_dim,
                      qs, ks, vs, fp8, current_stream());
}

// ---- direct-xGMI all-reduce plumbing (E15) --------------------------------
// Raw hipMalloc (NOT the torch caching allocator: hipIpcGetMemHandle needs
// the allocation base).  Returns (device_ptr, ipc_handle_bytes).
std::tuple<int64_t, py::bytes> xar_alloc(int64_t nbytes) {
  void* p = nullptr;
  TORCH_CHECK(hipMalloc(&p, nbytes) == hipSuccess, "xar_alloc failed");
  TORCH_CHECK(hipMemset(p, 0, nbytes) == hipSuccess);
  TORCH_CHECK(hipDeviceSynchronize() == hipSuccess);
  hipIpcMemHandle_t h;
  TORCH_CHECK(hipIpcGetMemHandle(&h, p) == hipSuccess,
              "hipIpcGetMemHandle failed");
  return {reinterpret_cast<int64_t>(p),
          py::bytes(reinterpret_cast<const char*>(&h), sizeof(h))};
}

int64_t xar_open(const std::string& handle_bytes) {
  TORCH_CHECK(handle_bytes.size() == sizeof(hipIpcMemHandle_t));
  hipIpcMemHandle_t h;
  memcpy(&h, handle_bytes.data(), sizeof(h));
  void* p = nullptr;
  TORCH_CHECK(hipIpcOpenMemHandle(&p, h, hipIpcMemLazyEnablePeerAccess) ==
                  hipSuccess,
              "hipIpcOpenMemHandle failed");
  return reinterpret_cast<int64_t>(p);
}

void xgmi_allreduce(torch::Tensor tensor, torch::Tensor bufs, int64_t cap,
                    int64_t rank, int64_t world) {
  TORCH_CHECK(tensor.scalar_type() == at::ScalarType::BFloat16);
  TORCH_CHECK(tensor.is_contiguous() && tensor.is_cuda());
  TORCH_CHECK(bufs.scalar_type() == at::ScalarType::Long && bufs.is_cuda());
  TORCH_CHECK(tensor.numel() * 2 <= cap, "tensor exceeds staging capacity");
  launch_xgmi_allreduce(
      reinterpret_cast<const unsigned long long*>(bufs.data_ptr()),
      reinterpret_cast<__hip_bfloat16*>(tensor.data_ptr()),
      reinterpret_cast<const __hip_bfloat16*>(tensor.data_ptr()),
      tensor.numel(), cap, (int)rank, (int)world, current_stream());
}

void gemm_tile(torch::Tensor y, torch::Tensor x, torch::Tensor w) {
  const int M = x.size(0);
  const int K = x.size(1);
  const int N = w.size(0);
  TORCH_CHECK(x.scalar_type() == at::ScalarType::BFloat16 &&
              w.scalar_type() == at::ScalarType::BFloat16);
  TORCH_CHECK(x.is_contiguous() && w.is_contiguous() && y.is_contiguous());
  TORCH_CHECK(M >= 1 && N % 128 == 0 && K % 64 == 0);
  TORCH_CHECK(w.size(1) == K && y.size(0) == M && y.size(1) == N);
  launch_gemm_tile(reinterpret_cast<__hip_bfloat16*>(y.data_ptr()),
                   reinterpret_cast<const __hip_bfloat16*>(x.data_ptr()),
                   reinterpret_cast<const __hip_bfloat16*>(w.data_ptr()), M, N,
                   K, current_stream());
}

// f32 space for the parts of a result that the streaming products leave for a merge
float* stream_parts(torch::Tensor& space, const torch::Tensor& x, int parts, int64_t elems) {
  if (parts <= 1) return nullptr;
  space = at::empty({parts, elems}, x.options().dtype(at::ScalarType::Float));
  return space.data_ptr<float>();
}

bool on16(const torch::Tensor& t);
void run_ring(torch::Tensor& y, const torch::Tensor& x, const torch::Tensor& w, int64_t M,
              int64_t N, int64_t K, bool gated, int plan);

void gemm_skinny(torch::Tensor y, torch::Tensor x, torch::Tensor w) {
  const int M = x.size(0);
  const int K = x.size(1);
  const int N = w.size(0);
  TORCH_CHECK(x.scalar_type() == at::ScalarType::BFloat16 &&
              w.scalar_type() == at::ScalarType::BFloat16);
  TORCH_CHECK(x.is_contiguous() && w.is_contiguous() && y.is_contiguous());
  TORCH_CHECK(M >= 1 && N % 128 == 0 && K % 64 == 0);
  TORCH_CHECK(w.size(1) == K && y.size(0) == M && y.size(1) == N);
  torch::Tensor part;
  if (M <= 64) {
    if (gemm_ring_wins(M, N, K, false) && on16(x) && on16(w) && on16(y)) {
      run_ring(y, x, w, M, N, K, false, gemm_ring_plan(M, N, K, false));
      return;
    }
    const int parts = gemm_stream_parts(16, M, N, K, false);
    launch_gemm_stream(ptr<__hip_bfloat16>(y), stream_parts(part, x, parts, (int64_t)M * N),
                       cptr<__hip_bfloat16>(x), cptr<__hip_bfloat16>(w), M, N, K, parts,
                       current_stream());
    return;
  }
  const int KS = gemm_skinny_num_ksplit(N, K, M);
  float* pp = nullptr;
  if (KS > 1) {
    part = at::empty({KS, M, N}, x.options().dtype(at::ScalarType::Float));
    pp = part.data_ptr<float>();
  }
  launch_gemm_skinny(reinterpret_cast<__hip_bfloat16*>(y.data_ptr()), pp,
                     reinterpret_cast<const __hip_bfloat16*>(x.data_ptr()),
                     reinterpret_cast<const __hip_bfloat16*>(w.data_ptr()), M,
                     N, K, KS, current_stream());
}

void check_rounded(const torch::Tensor& wq, const torch::Tensor& wscale, int64_t qbits,
                   int64_t N, int64_t K) {
  TORCH_CHECK(qbits == 8 || qbits == 4);
  TORCH_CHECK(wq.scalar_type() == at::ScalarType::Byte ||
              wq.scalar_type() == at::ScalarType::Char);
  TORCH_CHECK(wscale.scalar_type() == at::ScalarType::Float);
  TORCH_CHECK(wq.is_cuda() && wq.is_contiguous() && wscale.is_contiguous());
  TORCH_CHECK(N % 128 == 0 && K % 128 == 0);
  TORCH_CHECK(wq.size(0) == N && wq.size(1) == (qbits == 8 ? K : K / 2));
  TORCH_CHECK(wscale.numel() == (qbits == 8 ? N : N * (K / 128)));
}

// y = x W^T for rounded weights, any number of rows
void gemm_q(torch::Tensor y, torch::Tensor x, torch::Tensor wq, torch::Tensor wscale,
            int64_t qbits) {
  const int M = x.size(0), K = x.size(1), N = wq.size(0);
  check_rounded(wq, wscale, qbits, N, K);
  TORCH_CHECK(x.scalar_type() == at::ScalarType::BFloat16 &&
              y.scalar_type() == at::ScalarType::BFloat16);
  TORCH_CHECK(x.is_contiguous() && y.is_contiguous() && M >= 1);
  TORCH_CHECK(y.size(0) == M && y.size(1) == N);
  // rows of a block of W are found by 32 bits
  TORCH_CHECK((int64_t)128 * K < (1LL << 31));
  // x and W reach LDS in 16-byte pieces by panels and tiles
  const bool aligned = reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0 &&
                       reinterpret_cast<uintptr_t>(wq.data_ptr()) % 16 == 0;
  const int plan = M > 64 ? gemm_panel_plan(M, N, K, (int)qbits)
                   : aligned && reinterpret_cast<uintptr_t>(y.data_ptr()) % 8 == 0
                       ? gemm_panel_few_plan(M, N, K, (int)qbits) : 0;
  if (plan > 0) {
    TORCH_CHECK(aligned);
    torch::Tensor part;
    launch_gemm_block_q(ptr<__hip_bfloat16>(y), stream_parts(part, x, plan & 255, (int64_t)M * N),
                        cptr<__hip_bfloat16>(x), cptr<unsigned char>(wq),
                        wscale.data_ptr<float>(), (int)qbits, M, N, K, plan, current_stream());
    return;
  }
  const int parts = gemm_stream_parts((int)qbits, M, N, K, false);
  torch::Tensor part;
  launch_gemm_stream_q(ptr<__hip_bfloat16>(y), stream_parts(part, x, parts, (int64_t)M * N),
                       cptr<__hip_bfloat16>(x), cptr<unsigned char>(wq),
                       wscale.data_ptr<float>(), (int)qbits, M, N, K, parts, current_stream());
}

// out [N, K] bf16 = the weights that (wq, wscale) round
void widen_weight(torch::Tensor out, torch::Tensor wq, torch::Tensor wscale, int64_t qbits) {
  const int64_t N = out.size(0), K = out.size(1);
  check_rounded(wq, wscale, qbits, N, K);
  TORCH_CHECK(out.is_cuda() && out.is_contiguous() &&
              out.scalar_type() == at::ScalarType::BFloat16 &&
              reinterpret_cast<uintptr_t>(wq.data_ptr()) % 16 == 0);
  launch_widen_weight(ptr<__hip_bfloat16>(out), cptr<unsigned char>(wq),
                      wscale.data_ptr<float>(), (int)qbits, N * K, (int)K, current_stream());
}

// What the products of one normed row share: x [1, K] (+ residual) -> norm -> w [rows, K] in
// qbits; returns the sum's place (null without a residual).
__hip_bfloat16* check_row_norm(const torch::Tensor& x, const c10::optional<torch::Tensor>& residual,
                               c10::optional<torch::Tensor>& sum, const torch::Tensor& weight,
                               const torch::Tensor& w, const c10::optional<torch::Tensor>& scales,
                               int64_t qbits, int64_t rows) {
  const int64_t K = x.numel();
  auto row = [&](const torch::Tensor& t) {
    TORCH_CHECK(t.is_cuda() && t.scalar_type() == at::ScalarType::BFloat16 && t.is_contiguous() &&
                    t.numel() == K && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0,
                "one dense bf16 row from a 16-byte boundary on");
  };
  row(x);
  row(weight);
  TORCH_CHECK(residual.has_value() == sum.has_value());
  if (residual.has_value()) {
    row(*residual);
    row(*sum);
    TORCH_CHECK(sum->data_ptr() != residual->data_ptr() && sum->data_ptr() != x.data_ptr());
  }
  TORCH_CHECK(rows % 128 == 0 && K % 64 == 0 && gemm_row_fits((int)K));
  TORCH_CHECK(w.is_cuda() && w.dim() == 2 && w.size(0) == rows && w.is_contiguous() &&
              reinterpret_cast<uintptr_t>(w.data_ptr()) % 16 == 0);
  if (qbits == 16) {
    TORCH_CHECK(w.scalar_type() == at::ScalarType::BFloat16 && w.size(1) == K);
  } else {
    TORCH_CHECK(scales.has_value() && scales->is_cuda());
    check_rounded(w, *scales, qbits, rows, K);
  }
  return sum.has_value() ? ptr<__hip_bfloat16>(*sum) : nullptr;
}

const __hip_bfloat16* optional_row(const c10::optional<torch::Tensor>& t) {
  return t.has_value() ? cptr<__hip_bfloat16>(*t) : nullptr;
}

const float* optional_scales(const c10::optional<torch::Tensor>& t, int64_t qbits) {
  return qbits == 16 ? nullptr : t->data_ptr<float>();
}

// y = silu(x Wg^T) * (x Wu^T) for rounded [Wg; Wu] and more than one row, by one launch; false:
// nothing was done, the product's plan has no room for the gate
bool gemm_q_gated(torch::Tensor y, torch::Tensor x, torch::Tensor wq, torch::Tensor wscale,
                  int64_t qbits) {
  const int64_t M = x.size(0), K = x.size(1), N = wq.size(0) / 2;
  const int plan = gemm_panel_gated_plan((int)M, (int)N, (int)K, (int)qbits);
  if (plan == 0) return false;
  check_rounded(wq, wscale, qbits, 2 * N, K);
  TORCH_CHECK(x.is_cuda() && x.scalar_type() == at::ScalarType::BFloat16 &&
              y.scalar_type() == at::ScalarType::BFloat16);
  TORCH_CHECK(x.is_contiguous() && y.is_contiguous() && y.size(0) == M && y.size(1) == N);
  TORCH_CHECK((int64_t)128 * K < (1LL << 31));
  TORCH_CHECK(reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0 &&
              reinterpret_cast<uintptr_t>(wq.data_ptr()) % 16 == 0 &&
              reinterpret_cast<uintptr_t>(y.data_ptr()) % 8 == 0);
  launch_gemm_panel_gated(ptr<__hip_bfloat16>(y), cptr<__hip_bfloat16>(x),
                          cptr<unsigned char>(wq), wscale.data_ptr<float>(), (int)qbits, (int)M,
                          (int)N, (int)K, plan, current_stream());
  return true;
}

// y [1, I] = silu(n Wg^T) * (n Wu^T), n = rmsnorm(x + residual), sum = x + residual
void row_norm_gated(torch::Tensor y, c10::optional<torch::Tensor> sum, torch::Tensor x,
                    c10::optional<torch::Tensor> residual, torch::Tensor weight, double eps,
                    torch::Tensor w, c10::optional<torch::Tensor> scales, int64_t qbits) {
  const int64_t I = y.numel();
  __hip_bfloat16* to = check_row_norm(x, residual, sum, weight, w, scales, qbits, 2 * I);
  TORCH_CHECK(y.is_cuda() && y.scalar_type() == at::ScalarType::BFloat16 && y.is_contiguous() &&
              I % 128 == 0);
  launch_gemm_row_norm_gated(ptr<__hip_bfloat16>(y), to, cptr<__hip_bfloat16>(x),
                             optional_row(residual), cptr<__hip_bfloat16>(weight), (float)eps,
                             w.data_ptr(), optional_scales(scales, qbits), (int)qbits, (int)I,
                             (int)x.numel(), current_stream());
}

// q [1, heads * hd] = the turned queries of n W^T, its turned keys and its values in the cache
void row_norm_turn(torch::Tensor q, c10::optional<torch::Tensor> sum, torch::Tensor x,
                   c10::optional<torch::Tensor> residual, torch::Tensor weight, double eps,
                   torch::Tensor w, c10::optional<torch::Tensor> scales, int64_t qbits,
                   torch::Tensor positions, torch::Tensor slots, torch::Tensor cos_sin,
                   torch::Tensor k_cache, torch::Tensor v_cache) {
  TORCH_CHECK(k_cache.dim() == 4 && k_cache.sizes() == v_cache.sizes());
  const int64_t kvh = k_cache.size(2), hd = k_cache.size(3), heads = q.numel() / hd;
  TORCH_CHECK(q.is_cuda() && q.scalar_type() == at::ScalarType::BFloat16 && q.is_contiguous() &&
              heads * hd == q.numel() && hd >= 32 && (hd & (hd - 1)) == 0);
  __hip_bfloat16* to =
      check_row_norm(x, residual, sum, weight, w, scales, qbits, (heads + 2 * kvh) * hd);
  const bool fp8 = k_cache.scalar_type() == at::ScalarType::Byte;
  for (const auto& c : {k_cache, v_cache})
    TORCH_CHECK(c.is_cuda() && c.is_contiguous() &&
                c.scalar_type() == (fp8 ? at::ScalarType::Byte : at::ScalarType::BFloat16));
  for (const auto& i : {positions, slots})
    TORCH_CHECK(i.is_cuda() && i.scalar_type() == at::ScalarType::Long && i.numel() == 1);
  TORCH_CHECK(cos_sin.is_cuda() && cos_sin.scalar_type() == at::ScalarType::Float &&
              cos_sin.is_contiguous() && cos_sin.size(-1) == hd);
  launch_gemm_row_norm_turn(
      ptr<__hip_bfloat16>(q), to, cptr<__hip_bfloat16>(x), optional_row(residual),
      cptr<__hip_bfloat16>(weight), (float)eps, w.data_ptr(), optional_scales(scales, qbits),
      (int)qbits, (int)x.numel(), positions.data_ptr<long>(), slots.data_ptr<long>(),
      cos_sin.data_ptr<float>(), k_cache.data_ptr(), v_cache.data_ptr(), (int)heads, (int)kvh,
      __builtin_ctzl(hd) - 1, fp8, current_stream());
}

void gemm_skinny_gated(torch::Tensor y, torch::Tensor x, torch::Tensor w13) {
  const int M = x.size(0);
  const int K = x.size(1);
  const int I = w13.size(0) / 2;
  TORCH_CHECK(x.scalar_type() == at::ScalarType::BFloat16 &&
              w13.scalar_type() == at::ScalarType::BFloat16);
  TORCH_CHECK(x.is_contiguous() && w13.is_contiguous() && y.is_contiguous());
  TORCH_CHECK(M >= 1 && I % 128 == 0 && K % 64 == 0);
  TORCH_CHECK(w13.size(0) % 2 == 0 && w13.size(1) == K);
  TORCH_CHECK(y.size(0) == M && y.size(1) == I);
  torch::Tensor part;
  if (M <= 64) {
    if (gemm_ring_wins(M, I, K, true) && on16(x) && on16(w13) && on16(y)) {
      run_ring(y, x, w13, M, I, K, true, gemm_ring_plan(M, I, K, true));
      return;
    }
    const int parts = gemm_stream_parts(16, M, I, K, true);
    launch_gemm_stream_gated(ptr<__hip_bfloat16>(y),
                             stream_parts(part, x, parts, (int64_t)2 * M * I),
                             cptr<__hip_bfloat16>(x), cptr<__hip_bfloat16>(w13), M, I, K, parts,
                             current_stream());
    return;
  }
  const int KS = gemm_skinny_num_ksplit(I, K, M);
  float* pp = nullptr;
  if (KS > 1) {
    part = at::empty({KS, 2, M, I}, x.options().dtype(at::ScalarType::Float));
    pp = part.data_ptr<float>();
  }
  launch_gemm_skinny_gated(
      reinterpret_cast<__hip_bfloat16*>(y.data_ptr()), pp,
      reinterpret_cast<const __hip_bfloat16*>(x.data_ptr()),
      reinterpret_cast<const __hip_bfloat16*>(w13.data_ptr()), M, I, K, KS,
      current_stream());
}

void lora_bgmv(torch::Tensor out, torch::Tensor x, torch::Tensor a_stack,
               torch::Tensor b_stack, torch::Tensor tmp, torch::Tensor slots,
               torch::Tensor scales, int64_t off) {
  const int Tn = x.size(0);
  const int K = x.size(1);
  const int R = a_stack.size(1);
  const int N = b_stack.size(1);
  const int out_w = out.size(1);
  TORCH_CHECK(out.size(0) == Tn && tmp.size(0) == Tn && tmp.size(1) == R);
  TORCH_CHECK(a_stack.size(2) == K && b_stack.size(2) == R);
  TORCH_CHECK(R <= 64 && K % 8 == 0);
  TORCH_CHECK(off + N <= out_w);
  TORCH_CHECK(slots.scalar_type() == at::ScalarType::Int);
  TORCH_CHECK(tmp.scalar_type() == at::ScalarType::Float &&
              scales.scalar_type() == at::ScalarType::Float);
  TORCH_CHECK(x.is_contiguous() && out.is_contiguous() &&
              a_stack.is_contiguous() && b_stack.is_contiguous());
  DISPATCH_FLOATING(x.scalar_type(), {
    launch_lora_shrink<scalar_t>(tmp.data_ptr<float>(), cptr<scalar_t>(x),
                                 cptr<scalar_t>(a_stack),
                                 slots.data_ptr<int>(), Tn, R, K,
                                 current_stream());
    launch_lora_expand<scalar_t>(ptr<scalar_t>(out), tmp.data_ptr<float>(),
                                 cptr<scalar_t>(b_stack),
                                 slots.data_ptr<int>(),
                                 scales.data_ptr<float>(), Tn, R, N, out_w,
                                 (int)off, current_stream());
  });
}

bool on16(const torch::Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; }

// checked: y = x w^T, or the gated product, by gemm_ring.hip's tiles
void run_ring(torch::Tensor& y, const torch::Tensor& x, const torch::Tensor& w, int64_t M,
              int64_t N, int64_t K, bool gated, int plan) {
  torch::Tensor part;
  launch_gemm_ring(ptr<__hip_bfloat16>(y), stream_parts(part, x, plan & 15, M * N),
                   cptr<__hip_bfloat16>(x), cptr<__hip_bfloat16>(w), (int)M, (int)N, (int)K, plan,
                   gated, current_stream());
}

// y = x w^T, or silu(x wg^T) * (x wu^T) for w = [wg; wu], by large tiles; plan: as
// gemm_ring_plan gives it, 0: that one
void gemm_ring(torch::Tensor y, torch::Tensor x, torch::Tensor w, bool gated, int64_t plan) {
  for (const auto& t : {y, x, w})
    TORCH_CHECK(t.is_cuda() && t.scalar_type() == at::ScalarType::BFloat16 &&
                t.is_contiguous() && t.dim() == 2);
  const int64_t M = x.size(0), K = x.size(1), N = y.size(1);
  TORCH_CHECK(y.size(0) == M && w.size(0) == (gated ? 2 : 1) * N && w.size(1) == K);
  TORCH_CHECK(N % 128 == 0 && K % 64 == 0 && M < (1 << 24) && N < (1 << 24) && K < (1 << 23));
  TORCH_CHECK(!gated || (N + 128) * K * 2 < (int64_t)1 << 32, "W is found by 32 bits");
  // both reach LDS in 16-byte pieces
  TORCH_CHECK(on16(x) && on16(w));
  if (M == 0 || N == 0) return;
  if (K == 0) {
    y.zero_();
    return;
  }
  if (plan == 0) plan = gemm_ring_plan((int)M, (int)N, (int)K, gated);
  TORCH_CHECK(gemm_ring_takes((int)N, (int)K, (int)plan, gated), "no such plan");
  // results are stored by 16 bytes
  torch::Tensor to = on16(y) ? y : at::empty_like(y);
  run_ring(to, x, w, M, N, K, gated, (int)plan);
  if (!on16(y)) y.copy_(to);
}

// y = x w^T by large tiles, K cut over workgroups
void gemm_block(torch::Tensor y, torch::Tensor x, torch::Tensor w) {
  gemm_ring(y, x, w, false, 0);
}

LoraCols lora_cols(const std::vector<std::pair<int64_t, int64_t>>& spans, int V, int out_w) {
  LoraCols cols;
  const int P = spans.size();
  int64_t v = 0;
  for (int p = 0; p < 3; ++p) {
    const auto& span = spans[p < P ? p : P - 1];
    if (p < P) {
      TORCH_CHECK(0 <= span.first && span.first <= span.second && span.second <= out_w);
      cols.shift[p] = (int)(span.first - v);
      v += span.second - span.first;
    } else {
      cols.shift[p] = cols.shift[P - 1];
    }
    cols.end[p] = (int)v;
  }
  TORCH_CHECK(v == V);
  return cols;
}

// bf16: out[t, start_p ...] += scale · B_p A_p x[t] for up to three projections of x, whose
// adapters' weights are stacked side by side: a [L, P R, K], b [L, V, R], spans[p] = (start,
// end) in out's columns, V = the sum of their widths.
void lora_delta(torch::Tensor out, torch::Tensor x, torch::Tensor a, torch::Tensor b,
                torch::Tensor slots, torch::Tensor scales,
                const std::vector<std::pair<int64_t, int64_t>>& spans) {
  const int T = x.size(0), K = x.size(1), L = a.size(0), PR = a.size(1), R = b.size(2);
  const int V = b.size(1), out_w = out.size(1), P = spans.size();
  for (const auto& t : {out, x, a, b})
    TORCH_CHECK(t.is_cuda() && t.scalar_type() == at::ScalarType::BFloat16 && t.is_contiguous());
  TORCH_CHECK(P >= 1 && P <= 3 && PR == P * R && (R == 8 || R == 16 || R == 32 || R == 64));
  TORCH_CHECK(a.size(2) == K && K % 8 == 0 && b.size(0) == L && out.size(0) == T);
  TORCH_CHECK(slots.is_cuda() && slots.scalar_type() == at::ScalarType::Int &&
              slots.numel() == T);
  TORCH_CHECK(scales.is_cuda() && scales.scalar_type() == at::ScalarType::Float &&
              scales.numel() >= L);
  slots = slots.contiguous();
  scales = scales.contiguous();
  const LoraCols cols = lora_cols(spans, V, out_w);
  if (T == 0 || V == 0 || L == 0) return;
  const int cuts = lora_shrink_cuts(T, K);
  auto tmp = at::empty({cuts, T, PR}, x.options().dtype(at::ScalarType::Float));
  launch_lora_tiles(ptr<__hip_bfloat16>(out), tmp.data_ptr<float>(), cptr<__hip_bfloat16>(x),
                    cptr<__hip_bfloat16>(a), cptr<__hip_bfloat16>(b), slots.data_ptr<int>(),
                    scales.data_ptr<float>(), cols, T, L, R, PR, V, K, out_w, cuts,
                    current_stream());
}

// bf16: out = the product of x and its deltas as in lora_delta, for all W columns, gated: silu
// of the first half of them times the second.  The product is given (y [T, W]) or made from w
// [W, K] by gemm_ring.hip's tiles.
void lora_product(torch::Tensor out, torch::Tensor x, c10::optional<torch::Tensor> w,
                  c10::optional<torch::Tensor> y, torch::Tensor a, torch::Tensor b,
                  torch::Tensor slots, torch::Tensor scales,
                  const std::vector<std::pair<int64_t, int64_t>>& spans, bool gated) {
  const int T = x.size(0), K = x.size(1), L = a.size(0), PR = a.size(1), R = b.size(2);
  const int V = b.size(1), P = spans.size();
  TORCH_CHECK(w.has_value() != y.has_value());
  const torch::Tensor& given = w.has_value() ? *w : *y;
  for (const auto& t : {out, x, a, b, given})
    TORCH_CHECK(t.is_cuda() && t.scalar_type() == at::ScalarType::BFloat16 && t.is_contiguous() &&
                on16(t));
  const int W = w.has_value() ? w->size(0) : y->size(1);
  TORCH_CHECK(P >= 1 && P <= 3 && PR == P * R && (R == 8 || R == 16 || R == 32 || R == 64));
  TORCH_CHECK(a.size(2) == K && K % 8 == 0 && b.size(0) == L && L >= 1);
  TORCH_CHECK(out.dim() == 2 && out.size(0) == T && W % 2 == 0 &&
              out.size(1) == (gated ? W / 2 : W));
  TORCH_CHECK(slots.is_cuda() && slots.scalar_type() == at::ScalarType::Int &&
              slots.is_contiguous() && slots.numel() == T);
  TORCH_CHECK(scales.is_cuda() && scales.scalar_type() == at::ScalarType::Float &&
              scales.is_contiguous() && scales.numel() >= L);
  for (int p = 1; p < P; ++p) TORCH_CHECK(spans[p - 1].second <= spans[p].first, "spans in order");
  const LoraCols cols = lora_cols(spans, V, W);
  if (T == 0) return;
  const auto f32 = x.options().dtype(at::ScalarType::Float);
  torch::Tensor base, part, tmp;
  int parts = 0, cuts = lora_shrink_cuts(T, K);
  if (y.has_value()) {
    TORCH_CHECK(y->size(0) == T);
    base = *y;
  } else {
    TORCH_CHECK(w->size(1) == K && W % 128 == 0 && K % 64 == 0 && K > 0 && K < (1 << 23));
    const int plan = gemm_ring_plan(T, W, K, false);
    if ((plan & 15) > 1) {
      parts = plan & 15;
      part = at::empty({parts, T, W}, f32);
    } else {
      base = at::empty({T, W}, x.options());
    }
    auto* to = parts ? nullptr : ptr<__hip_bfloat16>(base);
    float* sums = parts ? part.data_ptr<float>() : nullptr;
    if (const int ahead = gemm_ring_lora_cuts(T, K, L, PR, plan)) {
      cuts = ahead;
      tmp = at::empty({cuts, T, PR}, f32);
      launch_gemm_ring_lora(to, sums, cptr<__hip_bfloat16>(x), cptr<__hip_bfloat16>(*w), T, W, K,
                            plan, tmp.data_ptr<float>(), cptr<__hip_bfloat16>(a),
                            slots.data_ptr<int>(), L, PR, cuts, current_stream());
    } else {
      launch_gemm_ring_parts(to, sums, cptr<__hip_bfloat16>(x), cptr<__hip_bfloat16>(*w), T, W, K,
                             plan, current_stream());
    }
  }
  if (!tmp.defined()) {
    tmp = at::empty({cuts, T, PR}, f32);
    launch_lora_shrink_tiles(tmp.data_ptr<float>(), cptr<__hip_bfloat16>(x),
                             cptr<__hip_bfloat16>(a), slots.data_ptr<int>(), T, L, PR, K, cuts,
                             current_stream());
  }
  launch_lora_finish(ptr<__hip_bfloat16>(out), parts ? nullptr : cptr<__hip_bfloat16>(base),
                     parts ? part.data_ptr<float>() : nullptr, tmp.data_ptr<float>(),
                     cptr<__hip_bfloat16>(b), slots.data_ptr<int>(), scales.data_ptr<float>(),
                     cols, T, L, R, PR, V, W, cuts, parts, gated, current_stream());
}

// A captured step's static buffers from a packed pinned host buffer (decode_inputs.hip) of n rows
// and tables of w blocks; rows: of the graph
void decode_inputs(torch::Tensor packed, torch::Tensor ids, torch::Tensor positions,
                   torch::Tensor slots, torch::Tensor lens, c10::optional<torch::Tensor> states,
                   torch::Tensor tables, int64_t n, int64_t w, int64_t rows) {
  TORCH_CHECK(packed.is_pinned() && packed.is_contiguous() &&
              packed.scalar_type() == at::ScalarType::Byte && on16(packed));
  TORCH_CHECK(n >= 1 && w >= 0 && n <= rows && packed.numel() >= n * (32 + 4 * w));
  for (const auto& t : {ids, positions, slots})
    TORCH_CHECK(t.is_cuda() && t.scalar_type() == at::ScalarType::Long && t.is_contiguous() &&
                t.numel() >= rows);
  TORCH_CHECK(lens.is_cuda() && lens.scalar_type() == at::ScalarType::Int &&
              lens.is_contiguous() && lens.numel() >= rows);
  TORCH_CHECK(tables.is_cuda() && tables.scalar_type() == at::ScalarType::Int &&
              tables.is_contiguous() && tables.dim() == 2 && tables.size(0) >= rows &&
              tables.size(1) >= w);
  if (states.has_value())
    TORCH_CHECK(states->is_cuda() && states->scalar_type() == at::ScalarType::Int &&
                states->is_contiguous() && states->numel() >= rows);
  launch_decode_inputs(reinterpret_cast<const long*>(packed.data_ptr()), ids.data_ptr<long>(),
                       positions.data_ptr<long>(), slots.data_ptr<long>(), lens.data_ptr<int>(),
                       states.has_value() ? states->data_ptr<int>() : nullptr,
                       tables.data_ptr<int>(), (int)n, (int)w, (int)rows, (int)tables.size(1),
                       current_stream());
}

// slots[t] = the place of token_ids[t] among ids (64 at most), or -1
void lora_slots(torch::Tensor slots, torch::Tensor token_ids, const std::vector<int>& ids) {
  for (const auto& t : {slots, token_ids})
    TORCH_CHECK(t.is_cuda() && t.scalar_type() == at::ScalarType::Int && t.is_contiguous());
  TORCH_CHECK(slots.numel() == token_ids.numel() && ids.size() <= 64);
  if (slots.numel() == 0) return;
  launch_lora_slots(slots.data_ptr<int>(), token_ids.data_ptr<int>(), ids.data(),
                    (int)ids.size(), (int)slots.numel(), current_stream());
}

void moe_gemm(torch::Tensor y, torch::Tensor x, torch::Tensor w,
              torch::Tensor seg_off, int64_t mode, c10::optional<torch::Tensor> rows) {
  // mode 0: plain, 1: silu(first half) * second half, 2: squared relu
  // rows: sorted row r is x[rows[r]]; without it x is sorted itself
  const int T = rows.has_value() ? rows->numel() : x.size(0);
  const int K = x.size(1);
  const int E = w.size(0);
  const long wn = w.size(1);
  const bool gated = mode == 1;
  const int N = gated ? (int)(wn / 2) : (int)wn;
  TORCH_CHECK(mode >= 0 && mode <= 2);
  TORCH_CHECK(x.scalar_type() == at::ScalarType::BFloat16 &&
              w.scalar_type() == at::ScalarType::BFloat16 &&
              y.scalar_type() == at::ScalarType::BFloat16);
  TORCH_CHECK(seg_off.scalar_type() == at::ScalarType::Int &&
              seg_off.numel() == E + 1);
  TORCH_CHECK(N % 128 == 0 && K % 64 == 0 && w.size(2) == K);
  TORCH_CHECK(y.size(0) == T && y.size(1) == N);
  TORCH_CHECK(x.is_contiguous() && w.is_contiguous() && y.is_contiguous());
  // rows reach LDS in 16-byte pieces
  TORCH_CHECK(reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0 &&
              reinterpret_cast<uintptr_t>(w.data_ptr()) % 16 == 0, "x and w start at 16 bytes");
  const int* rp = nullptr;
  if (rows.has_value()) {
    TORCH_CHECK(rows->is_cuda() && rows->scalar_type() == at::ScalarType::Int &&
                rows->is_contiguous());
    rp = rows->data_ptr<int>();
  }
  if (T == 0) return;
  torch::Tensor scratch;
  if (const long floats = moe_gemm_scratch(E, N, K, T, (int)mode))
    scratch = at::empty({floats}, x.options().dtype(at::ScalarType::Float));
  launch_moe_gemm(ptr<__hip_bfloat16>(y), cptr<__hip_bfloat16>(x), cptr<__hip_bfloat16>(w),
                  seg_off.data_ptr<int>(), rp, E, N, K, T, (int)mode,
                  scratch.defined() ? scratch.data_ptr<float>() : nullptr, current_stream());
}

void moe_topk(torch::Tensor ids, torch::Tensor weights, torch::Tensor x, torch::Tensor gate) {
  const int T = x.size(0), K = x.size(1), E = gate.size(0), top = ids.size(1);
  TORCH_CHECK(x.is_cuda() && x.scalar_type() == at::ScalarType::BFloat16 && x.is_contiguous() &&
              gate.scalar_type() == at::ScalarType::BFloat16 && gate.is_contiguous() &&
              gate.size(1) == K && K % 8 == 0);
  TORCH_CHECK(E >= 1 && E <= moe_topk_max_experts() && top >= 1 && top <= E &&
              top <= moe_topk_max_top());
  TORCH_CHECK(ids.scalar_type() == at::ScalarType::Int && ids.is_contiguous() &&
              ids.size(0) == T && weights.scalar_type() == at::ScalarType::Float &&
              weights.is_contiguous() && weights.sizes() == ids.sizes());
  if (T == 0) return;
  launch_moe_topk(ids.data_ptr<int>(), weights.data_ptr<float>(), cptr<__hip_bfloat16>(x),
                  cptr<__hip_bfloat16>(gate), T, E, K, top, current_stream());
}

void moe_group(torch::Tensor rows, torch::Tensor pos, torch::Tensor seg, torch::Tensor ids) {
  // pairs with ids other than experts 0 .. seg.numel() - 2 are left out
  const int pairs = ids.numel(), E = seg.numel() - 1;
  for (const auto& t : {rows, pos, seg, ids})
    TORCH_CHECK(t.is_cuda() && t.scalar_type() == at::ScalarType::Int && t.is_contiguous());
  TORCH_CHECK(rows.numel() == pairs && pos.numel() == pairs && ids.dim() == 2 && E >= 1 &&
              E <= moe_topk_max_experts());
  launch_moe_group(rows.data_ptr<int>(), pos.data_ptr<int>(), seg.data_ptr<int>(),
                   ids.data_ptr<int>(), pairs, E, (int)ids.size(1), current_stream());
}

void moe_sum(torch::Tensor out, torch::Tensor ye, torch::Tensor pos, torch::Tensor weights) {
  const int T = pos.size(0), top = pos.size(1), H = ye.size(1);
  TORCH_CHECK(ye.is_cuda() && ye.scalar_type() == at::ScalarType::BFloat16 &&
              ye.is_contiguous() && ye.size(0) == (int64_t)T * top && H % 8 == 0);
  TORCH_CHECK(out.scalar_type() == at::ScalarType::BFloat16 && out.is_contiguous() &&
              out.size(0) == T && out.size(1) == H);
  TORCH_CHECK(pos.scalar_type() == at::ScalarType::Int && pos.is_contiguous() &&
              weights.scalar_type() == at::ScalarType::Float && weights.is_contiguous() &&
              weights.sizes() == pos.sizes());
  if (T == 0) return;
  launch_moe_sum(ptr<__hip_bfloat16>(out), cptr<__hip_bfloat16>(ye), pos.data_ptr<int>(),
                 weights.data_ptr<float>(), T, H, top, current_stream());
}

void sample_argmax(torch::Tensor out, torch::Tensor logits,
                   torch::Tensor temps, c10::optional<torch::Tensor> noise) {
  const int N = logits.size(0);
  const int V = logits.size(1);
  TORCH_CHECK(out.scalar_type() == at::ScalarType::Long && out.size(0) == N);
  TORCH_CHECK(temps.scalar_type() == at::ScalarType::Float && temps.size(0) == N);
  TORCH_CHECK(logits.is_contiguous());
  const float* np_ = nullptr;
  if (noise.has_value()) {
    TORCH_CHECK(noise->scalar_type() == at::ScalarType::Float &&
                noise->is_contiguous() && noise->size(0) == N &&
                noise->size(1) == V);
    np_ = noise->data_ptr<float>();
  }
  DISPATCH_FLOATING(logits.scalar_type(), {
    launch_sample_argmax<scalar_t>(out.data_ptr<long>(),
                                   cptr<scalar_t>(logits),
                                   temps.data_ptr<float>(), np_, N, V,
                                   current_stream());
  });
}

void logsoftmax_topk(torch::Tensor topv, torch::Tensor topi,
                     torch::Tensor chosen_lp, torch::Tensor ranks,
                     torch::Tensor logits, torch::Tensor chosen) {
  const int N = logits.size(0);
  const int V = logits.size(1);
  const int K = topv.size(1);
  TORCH_CHECK(logits.scalar_type() == at::ScalarType::BFloat16 &&
              logits.is_contiguous());
  TORCH_CHECK(V % 8 == 0, "vocab must be a multiple of 8");
  TORCH_CHECK(K <= 16, "K <= 16");
  TORCH_CHECK(topv.scalar_type() == at::ScalarType::Float &&
              topi.scalar_type() == at::ScalarType::Int &&
              topv.is_contiguous() && topi.is_contiguous() &&
              topi.size(1) == K && topv.size(0) == N && topi.size(0) == N);
  TORCH_CHECK(chosen_lp.scalar_type() == at::ScalarType::Float &&
              chosen_lp.size(0) == N);
  TORCH_CHECK(ranks.scalar_type() == at::ScalarType::Int && ranks.size(0) == N);
  TORCH_CHECK(chosen.scalar_type() == at::ScalarType::Long &&
              chosen.is_contiguous() && chosen.size(0) == N);
  launch_logsoftmax_topk(
      topv.data_ptr<float>(), topi.data_ptr<int>(),
      chosen_lp.data_ptr<float>(), ranks.data_ptr<int>(),
      reinterpret_cast<const __hip_bfloat16*>(logits.data_ptr()),
      chosen.data_ptr<long>(), N, V, K, current_stream());
}

void mfma_probe(torch::Tensor a, torch::Tensor b, torch::Tensor d, int64_t shape) {
  TORCH_CHECK(a.scalar_type() == at::ScalarType::BFloat16);
  auto* ap = reinterpret_cast<const unsigned short*>(a.data_ptr());
  auto* bp = reinterpret_cast<const unsigned short*>(b.data_ptr());
  auto* dp = d.data_ptr<float>();
  if (shape == 32)
    launch_mfma_probe_32(ap, bp, dp, current_stream());
  else
    launch_mfma_probe_16(ap, bp, dp, current_stream());
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("mfma_probe", &mfma_probe, "MFMA fragment layout probe");
  m.def("rms_norm", &rms_norm, "fused RMSNorm (CDNA4)");
  m.def("fused_add_rms_norm", &fused_add_rms_norm,
        "in-place residual-add + RMSNorm (CDNA4)");
  m.def("silu_and_mul", &silu_and_mul, "SwiGLU activation (CDNA4)");
  m.def("rotary_embedding", &rotary_embedding, "NeoX rotary: q into dense rows, k in place (CDNA4)");
  m.def("reshape_and_cache", &reshape_and_cache, "paged KV cache write (CDNA4)");
  register_attention_ops(m);
  m.def("xar_alloc", &xar_alloc,
        "raw hipMalloc + IPC handle for the xGMI all-reduce staging buffer");
  m.def("xar_open", &xar_open, "open a peer's IPC handle -> device pointer");
  m.def("xgmi_allreduce", &xgmi_allreduce,
        "in-place one-shot all-reduce over peer-mapped xGMI buffers");
  m.def("gemm_tile", &gemm_tile,
        "128x128-tile glds-staged bf16 GEMM for decode batches (CDNA4)");
  m.def("gemm_q", &gemm_q, "product with int8 / 4-bit weights");
  m.def("widen_weight", &widen_weight, "int8 / 4-bit weights to bf16");
  m.def("gemm_skinny", &gemm_skinny,
        "skinny decode GEMM y = x @ w^T, M <= 64 (CDNA4 MFMA)");
  m.def("gemm_q_gated", &gemm_q_gated,
        "gated product with rounded weights, where it is one launch", py::arg("y"),
        py::arg("x"), py::arg("wq"), py::arg("wscale"), py::arg("qbits") = 8);
  m.def("gemm_panel_gated_plan", &gemm_panel_gated_plan, "its plan, or 0", py::arg("m"),
        py::arg("n"), py::arg("k"), py::arg("qbits") = 8);
  m.def("gemm_panel_plan", &gemm_panel_plan,
        "which panel products of many rows with rounded weights take, and parts of K (panel << 8 | "
        "parts)", py::arg("m"), py::arg("n"), py::arg("k"), py::arg("qbits") = 8);
  m.def("gemm_panel_few_plan", &gemm_panel_few_plan, "the same up to 64 rows, 0: no panel");
  m.def("gemm_row_form", &gemm_row_form,
        "waves of a workgroup for products of one row, and those K is dealt to (waves << 4 | those); "
        "mode 0 plain, 1 gated, 2 turned", py::arg("qbits"), py::arg("mode"), py::arg("n"), py::arg("k"));
  m.def("row_norm_gated", &row_norm_gated, "norm and gated product of one row (CDNA4)");
  m.def("row_norm_turn", &row_norm_turn,
        "norm, query / key / value product, rotation and cache write of one row (CDNA4)");
  m.def("gemm_skinny_gated", &gemm_skinny_gated,
        "fused gate/up skinny GEMM + SiLU-mul, M <= 64 (CDNA4 MFMA)");
  m.def("moe_gemm", &moe_gemm,
        "grouped MoE GEMM over expert segments (CDNA4 MFMA)", py::arg("y"), py::arg("x"),
        py::arg("w"), py::arg("seg_off"), py::arg("mode"), py::arg("rows") = py::none());
  m.def("moe_topk", &moe_topk, "router product, choice and weights of a softmax router");
  m.def("moe_group", &moe_group, "token-expert pairs grouped by expert");
  m.def("moe_sum", &moe_sum, "weighted sum of each token's expert results");
  m.def("moe_topk_max_experts", &moe_topk_max_experts);
  m.def("moe_topk_max_top", &moe_topk_max_top);
  m.def("logsoftmax_topk", &logsoftmax_topk,
        "fused log-softmax + top-K + sampled-token rank (one HBM pass)");
  m.def("sample_argmax", &sample_argmax,
        "fused temperature/gumbel-race sampling + greedy argmax (CDNA4)");
  m.def("rotary_cache", &rotary_cache, "rotation of q and k with the cache write");
  m.def("gemm_block", &gemm_block, "product of many rows, large tiles");
  m.def("gemm_ring", &gemm_ring, "product of many rows, large tiles, also gated", py::arg("y"),
        py::arg("x"), py::arg("w"), py::arg("gated") = false, py::arg("plan") = 0);
  m.def("gemm_ring_wins", &gemm_ring_wins, "whether the large tiles are the faster product");
  m.def("moe_tile", &moe_tile, "which tile expert products of many rows take");
  m.def("gemm_tiles_route", &gemm_tiles_route,
        "past 64 rows: 1 for their cut K, 2 otherwise, 0 where the library is faster");
  m.def("gemm_block_takes", &gemm_block_takes, "whether they are for their cut K");
  m.def("gemm_ring_plan", &gemm_ring_plan, "which tile a product takes, and parts of K (form << 4 | parts)");
  m.def("gemm_ring_reads_once", &gemm_ring_reads_once, "whether its weights go past the caches",
        py::arg("m"), py::arg("n"), py::arg("k"), py::arg("plan"), py::arg("gated") = false);
  m.def("decode_inputs", &decode_inputs, "a captured step's inputs from a packed host buffer");
  m.def("lora_product", &lora_product, "a product with its LoRA deltas, also gated");
  m.def("gemm_ring_lora_wins", &gemm_ring_lora_wins, "whether the tiles take a product with adapters",
        py::arg("m"), py::arg("n"), py::arg("k"), py::arg("rank") = 16);
  m.def("gemm_ring_lora_cuts", &gemm_ring_lora_cuts,
        "parts of K of the adapters' shrink beside a product, 0: in a launch of its own");
  m.def("lora_tiles_win", &lora_tiles_win, "whether its deltas are added by the matrix unit");
  m.def("lora_delta", &lora_delta,
        "bf16 multi-LoRA of up to three projections of one input");
  m.def("lora_slots", &lora_slots, "adapter slot of every token");
  m.def("lora_bgmv", &lora_bgmv,
        "batched multi-LoRA shrink+expand for mixed-adapter batches (CDNA4)");
}
