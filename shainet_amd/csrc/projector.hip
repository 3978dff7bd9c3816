// Row-major projections on the device and small upload helpers.
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <vector>

#include "../../include/shainet_hip_attn.h"
#include "attn_kernels.hpp"
#include "block_kernels.hpp"
#include "gemm_kernel.hpp"
#include "llama_internal.hpp"

void shainet_hip_set_error(int code, const char *msg);  // capi.hip

namespace shainet {

int llama_fail(int code, const std::string &msg) {
  shainet_hip_set_error(code, msg.c_str());
  return code;
}

bool DevF::reserve(size_t n) {
  if (n <= cap) return true;
  size_t want = cap ? cap : 1024;
  while (want < n) want *= 2;
  float *np = nullptr;
  if (hipMalloc((void **)&np, want * sizeof(float)) != hipSuccess) {
    (void)hipGetLastError();
    if (hipMalloc((void **)&np, n * sizeof(float)) != hipSuccess) {
      (void)hipGetLastError();  // (a launch behind this would report it as its own)
      return false;
    }
    want = n;
  }
  if (p) (void)hipFree(p);
  p = np;
  cap = want;
  return true;
}

bool PinnedF::reserve(size_t n) {
  if (n <= cap) return true;
  size_t want = cap ? cap : 4096;
  while (want < n) want *= 2;
  float *np = nullptr;
  if (hipHostMalloc((void **)&np, want * sizeof(float), hipHostMallocDefault) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  if (p) (void)hipHostFree(p);
  p = np;
  cap = want;
  return true;
}

void PinnedF::release() {
  if (p) (void)hipHostFree(p);
  p = nullptr;
  cap = 0;
}

void DevF::release() {
  if (p) (void)hipFree(p);
  p = nullptr;
  cap = 0;
}

// SHAINET_HIP_NO_TRANSPOSED_WEIGHTS: no second, transposed copy of q | k | v, W_o, gate | up and down (the
// products of a single row then run as the split GEMV over the [in, out] matrices, like the rest)
bool transposed_twins_wanted() {
  static const bool wanted = getenv("SHAINET_HIP_NO_TRANSPOSED_WEIGHTS") == nullptr;
  return wanted;
}

// Whether a copy of `bytes` leaves enough device memory to what cannot do without (caches that grow, scratch): an eighth
// of the device's (36 GB), or SHAINET_HIP_TWIN_RESERVE_MB.
static bool twin_leaves_room(size_t bytes) {
  size_t free_bytes = 0, total = 0;
  if (hipMemGetInfo(&free_bytes, &total) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  static const char *const knob = getenv("SHAINET_HIP_TWIN_RESERVE_MB");
  const size_t reserve = knob ? (size_t)strtoull(knob, nullptr, 10) << 20 : total / 8;
  return free_bytes >= bytes && free_bytes - bytes >= reserve;
}

// *twin = src transposed (src: [rows, cols] on the device), allocated on first use.  Returns the
// twin, or null when there is no memory for it (the caller then goes without; *stale false without a twin: not asked
// again until there are new weights).
const float *transposed_twin(float **twin, bool *stale, const float *src, int rows, int cols, hipStream_t stream,
                             const float *row_scale) {
  if (!transposed_twins_wanted() || !src) return nullptr;
  if (!*twin) {
    if (!*stale) return nullptr;
    const size_t bytes = (size_t)rows * cols * sizeof(float);
    if (!twin_leaves_room(bytes) || hipMalloc((void **)twin, bytes) != hipSuccess) {
      (void)hipGetLastError();
      *twin = nullptr;
      *stale = false;
      return nullptr;
    }
  }
  if (*stale) {
    // (waited for, once per set of weights: the copy may next be read on another stream)
    if (launch_transpose(src, *twin, rows, cols, stream, row_scale) != hipSuccess || hipStreamSynchronize(stream) != hipSuccess) {
      (void)hipGetLastError();
      return nullptr;
    }
    *stale = false;
  }
  return *twin;
}

// The flag words are shared by all kernels of this projector: each leaves them zero, and the
// launches of one projector follow each other on one stream.
int Projector::reserve_flags(size_t n_flags, hipStream_t stream) {
  if (n_flags <= flags_cap) return SHAINET_HIP_OK;
  if (!flags) lose_marks = getenv("SHAINET_HIP_TEST_LOSE_PARTIAL_MARKS") != nullptr;
  size_t want = flags_cap ? flags_cap : 4096;
  while (want < n_flags) want *= 2;
  unsigned *np = nullptr;
  // (twice the words: the second half is where the marks go in the test of the give-up path)
  if (hipMalloc((void **)&np, 2 * want * sizeof(unsigned)) != hipSuccess) return llama_fail(SHAINET_HIP_ERR_ALLOC, "hipMalloc failed");
  if (hipMemsetAsync(np, 0, 2 * want * sizeof(unsigned), stream) != hipSuccess) {
    (void)hipFree(np);
    return llama_fail(SHAINET_HIP_ERR_RUNTIME, "hipMemsetAsync(flags) failed");
  }
  if (flags) (void)hipFree(flags);  // hipFree waits for the device
  flags = np;
  flags_cap = want;
  return SHAINET_HIP_OK;
}

// Room for the parts of n floats.  Rows for which there is none stay floats.
bool Projector::reserve_parts(DevF &to, size_t n) {
  if (!asked_parts) no_parts = getenv("SHAINET_HIP_TEST_NO_ROWS_AS_PARTS") != nullptr;
  asked_parts = true;
  return !no_parts && to.reserve(n / 2 * 3);
}

// y = (res +) x W with the library's own MFMA kernel; res == y is allowed.
// swiglu: W is gate | up and y [T, N / 2].
int Projector::gemm(const float *x, long long x_stride, const float *w, float *y, int T, int K, int N,
                    hipStream_t stream, bool w_bf16, const float *res, const float *bias, Activation act, bool swiglu, Handover *next,
                    const GemvPrep *spread, bool planes) {
  const GemmPlan p = plan_gemm(T, K, N, x_stride, w_bf16);
  const bool aligned = !(((uintptr_t)x | (uintptr_t)w | (uintptr_t)y | (uintptr_t)res | (uintptr_t)bias) & 15);
  GemmNext also;
  also.swiglu = swiglu;
  also.prep = spread;
  float *result = y;
  if (spread && !(aligned && gemm_takes_next(p, T, N, also))) return llama_fail(SHAINET_HIP_ERR_ARGUMENT, "this product does not spread heads");
  if (swiglu && !(aligned && gemm_takes_next(p, T, N, also))) {
    if (!wide.reserve((size_t)T * N)) return llama_fail(SHAINET_HIP_ERR_ALLOC, "hipMalloc failed");
    result = wide.p;
    also.swiglu = false;
  }
  if (!scratch.reserve(p.partial_floats)) return llama_fail(SHAINET_HIP_ERR_ALLOC, "hipMalloc failed");
  if (int rc = reserve_flags(p.flag_words, stream)) return rc;
  // (what the product itself needs comes first: without the memory for these rows they are normed in front of the next product, as
  // after one that adds no pieces)
  const bool takes_norm = next && next->norm->kind != kNormNone && !bias && aligned && gemm_takes_next(p, T, N, also);
  const bool as_planes = takes_norm && p.parts == 1 && next->n && gemm_takes_planes(plan_gemm(T, N, next->n, N, next->w_bf16), N) &&
                         reserve_parts(handed, (size_t)T * N);
  if (takes_norm && (as_planes || handed.reserve((size_t)T * N))) {
    also.norm.kind = next->norm->kind;
    also.norm.gamma = next->norm->gamma;
    also.norm.beta = next->norm->beta;
    also.norm.alpha = next->norm->alpha;
    also.norm.eps = next->eps;
    also.norm.rows = handed.p;
    also.norm.planes = next->planes = as_planes;
    next->rows = handed.p;
  }
  if (p.flag_words && !error) return llama_fail(SHAINET_HIP_ERR_RUNTIME, "the projector has no error word");
  hipError_t e = launch_gemm(x, x_stride, w, result, res, scratch.p, flags, error, T, K, N, p, stream,
                             lose_marks ? flags + flags_cap : nullptr, lose_marks ? 2000 : 0, bias, act, also, planes);
  if (e == hipSuccess && swiglu && !also.swiglu) e = launch_swiglu_act(wide.p, y, T, N / 2, stream);
  if (e != hipSuccess) return llama_fail(SHAINET_HIP_ERR_RUNTIME, std::string("gemm launch: ") + hipGetErrorString(e));
  return SHAINET_HIP_OK;
}

bool Projector::spreads(const float *x, const float *w, const float *y, int T, int K, int N, bool w_bf16, const GemvPrep &where) {
  GemmNext next;
  next.prep = &where;
  return !few_rows(T, K, N, K) && !(((uintptr_t)x | (uintptr_t)w | (uintptr_t)y) & 15) && gemm_takes_next(plan_gemm(T, K, N, K, w_bf16), T, N, next);
}

bool Projector::few_rows(int T, int K, int N, long long x_stride) {
  const long long weights = (long long)K * N;
  return T <= 4 || (T <= 6 && weights <= 128 << 10) || (T <= 8 && weights <= 64 << 10) || (T <= 16 && !plan_gemm(T, K, N, x_stride).mfma);
}

int Projector::project(const float *x, long long x_stride, const float *w, float *y, int T, int K, int N,
                       hipStream_t stream, const Fused &f) {
  const bool swiglu = f.epilogue == kGemvSwiglu;
  if (f.next) f.next->rows = nullptr;
  if (f.epilogue == kGemvQkvPrep && (!f.prep || T > 16 || (N & 3)))
    return llama_fail(SHAINET_HIP_ERR_ARGUMENT, "the fused q | k | v epilogue takes at most 16 rows");
  const bool one_row = f.w_t && gemvt_takes(T, K, N, f.epilogue, f.norm, f.prep) && !(((uintptr_t)x | (uintptr_t)f.gamma | (uintptr_t)f.beta) & 15);
  const bool joins = one_row && f.join && f.join->d == K && row_join_fits(*f.join) && gemvt_takes_join(K, N, f.epilogue, f.norm);
  if (f.join && !joins) {
    const hipError_t e = launch_residual(*f.join, stream);
    if (e != hipSuccess) return llama_fail(SHAINET_HIP_ERR_RUNTIME, std::string("residual launch: ") + hipGetErrorString(e));
  }
  if (one_row) {
    GemvArgs a = {};
    if (joins) a.join = *f.join;
    a.x = x;
    a.x_stride = x_stride;
    a.norm = f.norm;
    a.gamma = f.w_t_has_gamma ? nullptr : f.gamma;
    a.beta = f.beta;
    a.alpha = f.alpha;
    a.eps = f.eps;
    a.w = f.w_t;
    a.res = f.res;
    a.bias = f.bias;
    a.act = f.act;
    a.y = y;
    a.T = T;
    a.K = K;
    a.N = N;
    a.epilogue = f.epilogue;
    if (f.prep) a.prep = *f.prep;
    hipError_t e = launch_gemvt(a, stream);
    if (e != hipSuccess)
      return llama_fail(SHAINET_HIP_ERR_RUNTIME, std::string("gemv launch: ") + hipGetErrorString(e));
    return SHAINET_HIP_OK;
  }
  // (an epilogue that only it has, or rows that the MFMA product cannot load or store 16 bytes at a time, keep the
  // split GEMV, too: 8 rows a float off 16 bytes, through a block 2048 wide with a feed-forward of 4096, take 127 us, with
  // a thread per element 564, on 16 bytes 106)
  const bool gemv = f.epilogue == kGemvQkvPrep || f.any_few_rows || few_rows(T, K, swiglu ? 2 * N : N, x_stride) ||
                    (((uintptr_t)x | (uintptr_t)w | (uintptr_t)y | (uintptr_t)f.res | (uintptr_t)f.bias) & 15);
  if (T <= 16 && (N & 3) == 0 && gemv) {
    const float *xin = x;
    long long xs = x_stride;
    int norm = f.norm;
    if (norm == kNormRms && T > 4) {  // every workgroup would redo the sums of squares of all rows: norm them once instead
      if (!normed.reserve((size_t)T * K)) return llama_fail(SHAINET_HIP_ERR_ALLOC, "hipMalloc failed");
      hipError_t e = launch_rmsnorm(x, x_stride, f.gamma, normed.p, T, K, f.eps, stream);
      if (e != hipSuccess) return llama_fail(SHAINET_HIP_ERR_RUNTIME, std::string("rmsnorm launch: ") + hipGetErrorString(e));
      xin = normed.p;
      xs = K;
      norm = kNormNone;
    }
    const GemvPlan p = plan_gemv(T, K, N, f.epilogue, f.prep ? f.prep->hd : 0);
    if (!scratch.reserve(p.partial_floats)) return llama_fail(SHAINET_HIP_ERR_ALLOC, "hipMalloc failed");
    if (p.splits > 1)
      if (int rc = reserve_flags((size_t)p.col_tiles * p.splits, stream)) return rc;
    if (p.splits > 1 && !error) return llama_fail(SHAINET_HIP_ERR_RUNTIME, "the projector has no error word");
    GemvArgs a = {};
    a.x = xin;
    a.x_stride = xs;
    a.norm = norm;
    a.gamma = f.gamma;
    a.beta = f.beta;
    a.alpha = f.alpha;
    a.eps = f.eps;
    a.w = w;
    a.res = f.res;
    a.bias = f.bias;
    a.act = f.act;
    a.y = y;
    a.partials = scratch.p;
    a.flags = flags;
    a.flag_set = lose_marks ? flags + flags_cap : nullptr;
    a.spin_limit = lose_marks ? 2000 : 0;
    a.error = error;
    a.T = T;
    a.K = K;
    a.N = N;
    a.epilogue = f.epilogue;
    if (f.prep) a.prep = *f.prep;
    hipError_t e = launch_gemv(a, p, stream);
    if (e != hipSuccess)
      return llama_fail(SHAINET_HIP_ERR_RUNTIME, std::string("gemv launch: ") + hipGetErrorString(e));
    return SHAINET_HIP_OK;
  }
  // many rows: norm kernel, MFMA product (the residual rides in its epilogue), activation kernel; the latter and the next norm
  // where the pieces of the product's tiles are added, if they are
  const float *xin = x;
  long long xs = x_stride;
  hipError_t e = hipSuccess;
  bool planes = false;
  if (f.norm && f.normed) {
    xin = f.normed;
    xs = K;
    planes = f.normed_planes;
  } else if (f.norm) {
    // (rows that the product copies as their parts are written so: 2048 rows of 2048 -> 16384 319 us and 298, 512 rows 94 and 83, 777 rows
    // 151 and 131, 512 rows of 2048 -> 3072 32.8 and 30.6; a launch of its own for the parts would take 5 to 8 of these)
    planes = (x_stride & 3) == 0 && !(((uintptr_t)x | (uintptr_t)w | (uintptr_t)y | (uintptr_t)f.res | (uintptr_t)f.bias) & 15) &&
             gemm_takes_planes(plan_gemm(T, K, swiglu ? 2 * N : N, K, f.w_bf16), K);
    planes = planes && reserve_parts(normed, (size_t)T * K);
    if (!planes && !normed.reserve((size_t)T * K)) return llama_fail(SHAINET_HIP_ERR_ALLOC, "hipMalloc failed");
    e = f.norm == kNormDynTanh ? launch_dyn_tanh(x, x_stride, f.gamma, f.beta, f.alpha, normed.p, T, K, stream, planes)
                               : launch_rmsnorm(x, x_stride, f.gamma, normed.p, T, K, f.eps, stream, planes);
    if (e != hipSuccess) return llama_fail(SHAINET_HIP_ERR_RUNTIME, std::string("norm launch: ") + hipGetErrorString(e));
    xin = normed.p;
    xs = K;
  }
  if (swiglu) return gemm(xin, xs, w, y, T, K, 2 * N, stream, f.w_bf16, nullptr, nullptr, Activation(), true, nullptr, nullptr, planes);
  return gemm(xin, xs, w, y, T, K, N, stream, f.w_bf16, f.epilogue == kGemvResidual ? f.res : nullptr,
              f.epilogue == kGemvBias ? f.bias : nullptr, f.act, false, f.next, f.spread, planes);
}

void Projector::release() {
  scratch.release();
  normed.release();
  wide.release();
  handed.release();
  if (flags) (void)hipFree(flags);
  flags = nullptr;
  flags_cap = 0;
}

int upload_floats(float **dst, const float *src, size_t n) {
  if (*dst) (void)hipFree(*dst);
  *dst = nullptr;
  if (hipMalloc((void **)dst, n * sizeof(float)) != hipSuccess) return llama_fail(SHAINET_HIP_ERR_ALLOC, "hipMalloc failed");
  if (hipMemcpy(*dst, src, n * sizeof(float), hipMemcpyHostToDevice) != hipSuccess)
    return llama_fail(SHAINET_HIP_ERR_RUNTIME, "hipMemcpy of a weight matrix failed");
  return SHAINET_HIP_OK;
}

int upload_side_by_side(float **dst, const float *const *mats, const int *widths, int count, int rows) {
  if (*dst) (void)hipFree(*dst);
  *dst = nullptr;
  size_t total = 0;
  for (int i = 0; i < count; ++i) total += (size_t)widths[i];
  if (hipMalloc((void **)dst, (size_t)rows * total * sizeof(float)) != hipSuccess)
    return llama_fail(SHAINET_HIP_ERR_ALLOC, "hipMalloc failed");
  const size_t pitch = total * sizeof(float);
  size_t off = 0;
  for (int i = 0; i < count; ++i) {
    const size_t wb = (size_t)widths[i] * sizeof(float);
    if (hipMemcpy2D(*dst + off, pitch, mats[i], wb, wb, rows, hipMemcpyHostToDevice) != hipSuccess)
      return llama_fail(SHAINET_HIP_ERR_RUNTIME, "hipMemcpy2D of a weight matrix failed");
    off += (size_t)widths[i];
  }
  return SHAINET_HIP_OK;
}

}  // namespace shainet

// ---- the product by itself ---------------------------------------------------------------
namespace {
std::mutex g_matmul_lock;
// Grow-only scratch of the handle-less calls (partial products of split shapes, their flag words, the
// error word their kernels report into), one set per stream: calls on different streams may overlap
// on the device and must not share partial products.  Never freed, like the reference's class-level scratch.
std::map<hipStream_t, shainet::Projector> g_matmul;

int describe(int rows, int k, int n, bool w_bf16, int plan[7]) {
  using namespace shainet;
  if (!plan || rows < 1 || k < 1 || n < 1) return llama_fail(SHAINET_HIP_ERR_ARGUMENT, "invalid matmul arguments");
  describe_gemm(plan_gemm(rows, k, n, k, w_bf16), k, plan);
  return SHAINET_HIP_OK;
}

int matmul(const float *x, long long x_stride, const float *w, const float *res, float *y, int rows, int k, int n, void *stream,
           bool w_bf16) {
  using namespace shainet;
  if (!x || !w || !y || rows < 1 || k < 1 || n < 1 || x_stride < k)
    return llama_fail(SHAINET_HIP_ERR_ARGUMENT, "invalid matmul arguments");
  if (!shainet_hip_available()) return llama_fail(SHAINET_HIP_ERR_RUNTIME, "no gfx950 device available");
  std::lock_guard<std::mutex> guard(g_matmul_lock);
  Projector &p = g_matmul[(hipStream_t)stream];
  if (!p.error) p.error = alloc_error_word();
  // what a kernel of an earlier call on this stream reported (a given-up wait for partial sums)
  // is said by the next call, which does nothing else then
  if (int rc = check_error_word(p.error)) return rc;
  Fused f;
  f.any_few_rows = !w_bf16;
  f.w_bf16 = w_bf16;
  if (res) {
    f.epilogue = kGemvResidual;
    f.res = res;
  }
  return p.project(x, x_stride, w, y, rows, k, n, (hipStream_t)stream, f);
}
}  // namespace

extern "C" int shainet_hip_describe_matmul(int rows, int k, int n, int plan[7]) { return describe(rows, k, n, false, plan); }

extern "C" int shainet_hip_describe_matmul_bf16_weights(int rows, int k, int n, int plan[7]) {
  return describe(rows, k, n, true, plan);
}

extern "C" int shainet_hip_matmul_f32(const float *x, long long x_stride, const float *w, const float *res, float *y,
                                      int rows, int k, int n, void *stream) {
  return matmul(x, x_stride, w, res, y, rows, k, n, stream, false);
}

extern "C" int shainet_hip_matmul_bf16_weights_f32(const float *x, long long x_stride, const float *w, const float *res, float *y,
                                                   int rows, int k, int n, void *stream) {
  return matmul(x, x_stride, w, res, y, rows, k, n, stream, true);
}
