// Test infrastructure: extern "C" launchers for what the product's own library does not launch: the
// engine drop-in (miso_amd/engine/attention.{hpp,hip} against engine_stub/), the 64 x 64 GEMM
// kernel that the engine's own gemm() launches, GEMM batches of any mix, and the host's choices of
// a form. Used only by GPU tests; never linked into the product.

#include "engine/attention.hip"

#include <cstring>

namespace {

// A layer from device weights (r1 rows; q, k, o Q4_K, v Q6_K) and norms, and one sequence of at most
// max_ctx tokens with the scratch of both steps.
struct Engine {
  miso::AttentionLayer layer;
  miso::RopeConfig rope;
  miso::AttentionCache cache;
  miso::AttentionScratch sc;
  miso::AttentionPrefillScratch ps;
};

template <class T>
miso::DeviceBuffer<T> copy(const T* p, std::size_t n) {
  miso::DeviceBuffer<T> b(n);
  MISO_HIP_CHECK(hipMemcpy(b.data(), p, n * sizeof(T), hipMemcpyDeviceToDevice));
  return b;
}

miso::QMatrix matrix(miso::gguf::GgmlType type, unsigned n, unsigned k, const std::uint8_t* p,
                     std::size_t bytes) {
  return {type, n, k, copy(p, bytes)};
}

}  // namespace

extern "C" {

void* drop_engine_new(const std::uint8_t* const* w, const std::uint64_t* bytes,
                      const float* attn_norm, const float* q_norm, const float* k_norm,
                      const float* inv_freq, unsigned max_ctx, unsigned max_tok) {
  using miso::gguf::GgmlType;
  try {
    return new Engine{{matrix(GgmlType::Q4_K, 8192, 2048, w[0], bytes[0]),
                       matrix(GgmlType::Q4_K, 512, 2048, w[1], bytes[1]),
                       matrix(GgmlType::Q6_K, 512, 2048, w[2], bytes[2]),
                       matrix(GgmlType::Q4_K, 2048, 4096, w[3], bytes[3]), copy(attn_norm, 2048),
                       copy(q_norm, 256), copy(k_norm, 256)},
                      {copy(inv_freq, 32)},
                      miso::AttentionCache(max_ctx),
                      {},
                      miso::AttentionPrefillScratch(max_tok)};
  } catch (const std::exception&) {
    return nullptr;
  }
}
void drop_engine_delete(void* e) { delete static_cast<Engine*>(e); }

// One step of n tokens (n == 1 and decode != 0: the decode step) on the null stream; 0 on success.
int drop_engine_step(void* e_, int decode, float* h, const float* delta, float* y, unsigned n,
                     float eps) {
  Engine& e = *static_cast<Engine*>(e_);
  try {
    if (decode != 0)
      miso::attention_decode(e.layer, e.cache, e.sc, e.rope, h, delta, y, eps, nullptr);
    else
      miso::attention_prefill(e.layer, e.cache, e.sc, e.ps, e.rope, h, delta, y, n, eps, nullptr);
  } catch (const std::exception&) {
    return 1;
  }
  return 0;
}

// Copies `n` floats of a scratch member to the host: 's' decode, 'p' prefill, then the member's name
// (pxn, sq, ...); returns its size in floats, 0 for an unknown name.
std::uint64_t drop_engine_read(void* e_, const char* name, float* out, std::uint64_t n) {
  Engine& e = *static_cast<Engine*>(e_);
  const struct {
    const char* name;
    miso::DeviceBuffer<float>& b;
  } members[] = {{"sxn", e.sc.xn},     {"sproj", e.sc.proj}, {"sq", e.sc.q},
                 {"score", e.sc.core}, {"pxn", e.ps.xn},     {"pproj", e.ps.proj},
                 {"pq", e.ps.q},       {"pcore", e.ps.core}, {"pbalance", e.ps.balance}};
  for (const auto& m : members)
    if (std::strcmp(m.name, name) == 0) {
      if (n > m.b.size() ||
          hipMemcpy(out, m.b.data(), n * sizeof(float), hipMemcpyDeviceToHost) != hipSuccess)
        return 0;
      return m.b.size();
    }
  return 0;
}

// qgemm_kernel<F> as the engine launches it (src/engine/weights.hip:306-330); format 0 Q4_K, 1 Q6_K.
int drop_qgemm_kernel(int format, const std::uint8_t* w, const void* xh, const float* xs, float* y,
                      unsigned k, unsigned n_rows, unsigned n_tok, unsigned ldy) {
  namespace K = miso::kernels;
  const K::QGemmParams p{w, static_cast<const _Float16*>(xh), xs, y, k, n_rows, n_tok, ldy};
  const unsigned tiles = K::qgemm_tiles(n_rows, n_tok);
  if (format == 0)
    K::qgemm_kernel<K::QFormat::Q4K><<<tiles, 256>>>(p);
  else
    K::qgemm_kernel<K::QFormat::Q6K><<<tiles, 256>>>(p);
  return static_cast<int>(hipGetLastError());
}

namespace {
miso::kernels::QGemmBatch batch(unsigned count, const int* format, const std::uint8_t* const* w,
                                const void* xh, const float* xs, float* const* y, unsigned k,
                                const unsigned* n_rows, unsigned n_tok, unsigned ldy) {
  namespace K = miso::kernels;
  K::QGemmBatch b{};
  b.count = count;
  for (unsigned i = 0; i < count; ++i) {
    b.m[i] = {w ? w[i] : nullptr, static_cast<const _Float16*>(xh), xs, y ? y[i] : nullptr, k,
              n_rows[i], n_tok, ldy};
    b.format[i] = format[i] == 0 ? K::QFormat::Q4K : K::QFormat::Q6K;
  }
  return b;
}
}  // namespace

// qgemm_launch of up to three products, and the tile shape it takes for them (10 + the shape's index
// where the ring is deep; host only).
int drop_qgemm_batch(unsigned count, const int* format, const std::uint8_t* const* w, const void* xh,
                     const float* xs, float* const* y, unsigned k, const unsigned* n_rows,
                     unsigned n_tok, unsigned ldy) {
  miso::kernels::qgemm_launch(batch(count, format, w, xh, xs, y, k, n_rows, n_tok, ldy), nullptr);
  return static_cast<int>(hipGetLastError());
}
unsigned drop_qgemm_shape(unsigned count, const int* format, const unsigned* n_rows,
                          unsigned n_tok) {
  const auto s = miso::kernels::qgemm_shape(
      batch(count, format, nullptr, nullptr, nullptr, nullptr, 256, n_rows, n_tok, 0));
  return s.index + (s.deep ? 10 : 0);
}

// The form a causal prefill takes: 0 one workgroup per block, 1 balanced pairs, 2 parts, 3 parts with
// two row blocks (host only).
unsigned drop_prefill_form(unsigned pos0, unsigned n, std::uint64_t workspace_bytes) {
  return static_cast<unsigned>(miso::kernels::attn_prefill_form(pos0, n, workspace_bytes));
}

}  // extern "C"
