// Shared by the host mirrors of LlamaBlock and of the model around it: grow-only
// device buffers and the row-major projection y = x W.
#pragma once
#include <hip/hip_runtime.h>

#include <string>

#include "../../include/shainet_hip_attn.h"
#include "activation.hpp"

namespace shainet {
struct AheadRows;
struct GemvPrep;
struct ResidualArgs;
}
// capi.hip: shainet_attn_forward with the rows of q, k and v at given strides; ahead (nullable): what a decode
// launch also reads
int shainet_attn_forward_strided(shainet_attn_ctx *c, shainet_kv_cache *kc, const int *seq_ids,
                                 const int *new_tokens, int n_seqs, const float *q, const float *k, const float *v,
                                 long long q_stride, long long k_stride, long long v_stride, float *out, int mem,
                                 const shainet::AheadRows *ahead = nullptr);

// capi.hip: the two halves of shainet_attn_forward for one sequence (slot 0 of the
// cache) when the kernel that produces q | k | v also does the bias / QK-norm / RoPE /
// append step (the kGemvQkvPrep epilogue).  Both refuse a cache whose lengths are on the device; begin checks the capacity and says where
// the prepared rows go; finish runs the attention kernel over them and counts the rows
// into the cache.  Both are asynchronous on the context's stream.
int shainet_attn_begin_prepared(shainet_attn_ctx *c, shainet_kv_cache *kc, int new_tokens, shainet::GemvPrep *where);
int shainet_attn_finish_prepared(shainet_attn_ctx *c, shainet_kv_cache *kc, int new_tokens, float *out,
                                 const shainet::AheadRows *ahead = nullptr);
// capi.hip: instead of finish, when the caller's own kernel appended the rows and attended over them
void shainet_attn_commit_prepared(shainet_attn_ctx *c, shainet_kv_cache *kc, int new_tokens);
// capi.hip: the pinned host word a context's kernels report a given-up wait into; a block or a
// model that owns the context makes it the owner's word (null = back to the context's own)
void shainet_attn_adopt_error_word(shainet_attn_ctx *c, int *word);
int *shainet_attn_error_word(shainet_attn_ctx *c);

// Device weight buffers of a block / a model, allocated on first request, for a loader
// that fills them on the device (llama_block.hip, llama_model.hip).
namespace shainet {
struct NormWeights;
struct LatentAttn;
struct Mixer;
struct FeedForward;
}
struct LlamaBlockBuffers {
  float *w_qkv, *w_o, *gate_up, *down;  // w_qkv, w_o: null where the mixer is latent attention; gate_up, down: where there is no feed-forward
  shainet::NormWeights *norm1, *norm2;
  int d_model, q_dim, kv_dim, ff_hidden;
  // for the loader to say: every value of the matrix is a bf16 number (false until then)
  bool *w_qkv_bf16, *w_o_bf16, *gate_up_bf16, *down_bf16;
};
int shainet_llama_block_buffers(shainet_llama_block *b, LlamaBlockBuffers *out);
// A block whose mixer is latent attention (latent_attn.hpp), its norms of one kind (kNorm*), with a
// dense feed-forward or none (ff_hidden 0).  weights_of: the block whose weights it uses, or null.
int shainet_llama_block_create_latent(shainet_llama_block **out, int d_model, const shainet_latent_config &cfg,
                                      int ff_hidden, int norm_kind, double eps, const shainet_llama_block *weights_of);
shainet::LatentAttn *shainet_llama_block_latent_mixer(shainet_llama_block *b);  // null: grouped-query attention
// A block with norms behind its sublayers, too (RMS norms of d_model values), and a causal convolution over time
// of `taps` taps in front of each; ff may be null.  The block takes over mixer and ff, also on failure.
// Its buffers are there at once, for a loader to fill: norms [d], convolutions [taps, d], oldest row's tap first.
int shainet_llama_block_create_wrapped(shainet_llama_block **out, int d_model, shainet::Mixer *mixer, shainet::FeedForward *ff,
                                       int taps, double eps);
struct WrappedBlockBuffers {
  float *norm1, *post1, *conv1, *norm2, *post2, *conv2;  // the last three: null without a feed-forward
};
WrappedBlockBuffers shainet_llama_block_wrapped_buffers(shainet_llama_block *b);
shainet::Mixer *shainet_llama_block_mixer_of(shainet_llama_block *b);  // null: the grouped-query attention of a LLaMA block
namespace shainet {
// The norm of what reads a product's result next, for the product to take along where its last launch holds whole rows.
struct Handover {
  const NormWeights *norm = nullptr;
  double eps = 0.0;
  int n = 0;             // columns of the product that reads these rows, and whether its weights are bf16 numbers (0: it takes the rows as they are)
  bool w_bf16 = false;
  const float *rows = nullptr;  // set by the product: the result's rows behind the norm, dense; null: the norm is still to be taken
  bool planes = false;          // set by the product: as their parts, which that product takes so (gemm_takes_planes)
};

}
// The result of such a block's last sublayer that has not joined the residual yet: the next block's first launch
// does it (shainet_llama_block_forward_device), or shainet_llama_block_join_carry behind the last block.
struct BlockCarry {
  const float *y = nullptr, *post = nullptr;
  // other blocks: the rows behind the block's first norm, if the block before has taken it; and the next block's first norm
  const float *normed = nullptr;
  shainet::Handover next;
};
// A model without blocks yet, and one more block for it (which it then owns), for loaders of designs
// whose layers are not all alike.
int shainet_llama_model_create_empty(shainet_llama_model **out, int vocab, int d_model, double eps,
                                     double embedding_scale, int norm_kind);
int shainet_llama_model_add_block(shainet_llama_model *m, shainet_llama_block *b);
struct LlamaModelBuffers {
  float *embedding;
  shainet::NormWeights *final_norm;
  float *lm_head;
  bool *lm_head_bf16;  // for the loader to say: every value is a bf16 number (false until then)
};
// Position vectors [max_positions, d_model] that are added to the embedding rows: the buffer, allocated on first
// request, for a loader to fill.  A sequence cannot outgrow them.
int shainet_llama_model_position_buffer(shainet_llama_model *m, int max_positions, float **out);
int shainet_llama_model_buffers(shainet_llama_model *m, LlamaModelBuffers *out);

namespace shainet {

struct DevF {
  float *p = nullptr;
  size_t cap = 0;
  bool reserve(size_t n);
  void release();
};

// Grow-only pinned host buffer: host-pointer calls stage their rows through it, so that the
// copies to and from the device run as one asynchronous DMA each instead of the runtime's
// staged copy of pageable memory.
struct PinnedF {
  float *p = nullptr;
  size_t cap = 0;
  bool reserve(size_t n);
  void release();
};

// What rides along with a projection y = x W.
struct Fused {
  int epilogue = 0;            // kGemvPlain, kGemvResidual (y = res + x W), kGemvSwiglu (W = gate | up, [K, 2N]) or kGemvBias
  const float *res = nullptr;  // [T, N]
  const float *bias = nullptr;  // [N]: y = act(x W + bias)
  Activation act;
  int norm = 0;                // kNorm*: applied to the rows of x first
  const float *gamma = nullptr;
  const float *beta = nullptr;  // kNormDynTanh
  float alpha = 0.f;            // kNormDynTanh
  double eps = 0.0;
  const GemvPrep *prep = nullptr;  // kGemvQkvPrep: where the head rows go (y may be null); at most 16 rows
  // the same weights transposed ([N, K]; kGemvSwiglu: [2N, K]) or null: one row of x then takes the
  // product that gives a wavefront whole outputs (launch_gemvt) where its shapes allow
  const float *w_t = nullptr;
  const GemvPrep *spread = nullptr;  // many rows, Projector::spreads: y is q | k | v, whose heads go where it says (y is scratch)
  bool w_bf16 = false;  // every value of W is a bf16 number: half the MFMAs of many rows have nothing to add
  bool any_few_rows = false;  // up to 16 rows run as the split GEMV, not only the ones it is the faster product for
  const float *normed = nullptr;  // [T, K]: the rows of x behind the norm, where an earlier product handed them over (more than a few rows only)
  bool normed_planes = false;     // as their parts (Handover::planes)
  Handover *next = nullptr;       // nullable; for kGemvPlain and kGemvResidual
  const ResidualArgs *join = nullptr;  // x is this row's h, still to be made: in the product's launch where that takes it along (x may stay unwritten then)
  bool w_t_has_gamma = false;  // the rows of w_t were made with gamma multiplied in: the norm's factor 1 / rms is all that is left to apply
};

// The weights of one norm, on the device.
struct NormWeights {
  int kind = 1;            // kNorm*
  float *gamma = nullptr;  // null = ones (kNormRms only)
  float *beta = nullptr;   // kNormDynTanh
  float alpha = 0.f;       // kNormDynTanh
  void apply(Fused &f, double eps) const {  // the norm in front of a product
    f.norm = kind;
    f.gamma = gamma;
    f.beta = beta;
    f.alpha = alpha;
    f.eps = eps;
  }
};

// y[T,N] = epilogue(norm(x)[T,K] * W), all row-major on the device.  A few rows
// (decode; few_rows) run as one hand-written split GEMV with the norm and the epilogue
// inside; more rows run as the MFMA product of gemm_kernel.hip (the counterpart of
// the reference's cuBLAS SGEMM, cuda.cr:237-247) after the separate norm kernel,
// with the residual add in its epilogue.  The SwiGLU activation and the norm of what comes next ride in the kernel that adds
// the pieces of the product's tiles where there is one, and are kernels of their own elsewhere.
struct Projector {
  // Whether T rows run as the split GEMV.  Up to 4 do.  It streams the weights once for up to 16, but its multiply-adds
  // are the vector ALU's, and from 5 rows on the MFMA product is the faster one (a prompt of a 2048 wide model of 4
  // layers: 4 rows 533 | 600 us, 5 rows 701 | 600, 16 rows 962 | 602); it needs K, N and the row stride of x to be
  // multiples of 4.  Small weights wait for launches alone, and the MFMA product has more of them (norm, head rows,
  // activation, the sum of pieces): a block of width 64 | 128 | 256 | 512 takes 90 | 88 | 101 | 103 us for 5 rows if all its
  // products are MFMA's, 68 | 72 | 81 | 93 this way; for 8 rows 84 | 80 | 99 | 98 and 77 | 77 | 93 | 94; from 10 rows on
  // the MFMA product is the faster one at any size (width 128, 12 rows: 80, and 85 with the smallest as the split GEMV).
  static bool few_rows(int T, int K, int N, long long x_stride);
  // Whether the product of many rows [T, K] without gaps puts q | k | v heads where `where` says (Fused::spread).
  static bool spreads(const float *x, const float *w, const float *y, int T, int K, int N, bool w_bf16, const GemvPrep &where);
  DevF scratch, normed, wide, handed;
  // split products: a word per partial that says when it is complete (zero between launches)
  unsigned *flags = nullptr;
  size_t flags_cap = 0;
  // SHAINET_HIP_TEST_LOSE_PARTIAL_MARKS (read when the flag words are first allocated): the marks
  // go to a second set of words nobody reads and waits end after 2000 polls, so that the report
  // of a given-up wait can be exercised without hanging anything
  bool lose_marks = false;
  // SHAINET_HIP_TEST_NO_ROWS_AS_PARTS (read when the first such rows are to be written): as if there were no memory for them
  bool no_parts = false, asked_parts = false;
  // where the split products' kernels report a given-up wait: the owner's pinned host word
  int *error = nullptr;
  // returns a SHAINET_HIP_* status; the message is left for shainet_hip_last_error
  int project(const float *x, long long x_stride, const float *w, float *y, int T, int K, int N, hipStream_t stream,
              const Fused &f = Fused());
  void release();

 private:
  int reserve_flags(size_t n_flags, hipStream_t stream);
  bool reserve_parts(DevF &to, size_t n);
  // res != nullptr: y = res + x W
  int gemm(const float *x, long long x_stride, const float *w, float *y, int T, int K, int N, hipStream_t stream, bool w_bf16,
           const float *res = nullptr, const float *bias = nullptr, Activation act = Activation(), bool swiglu = false, Handover *next = nullptr,
           const GemvPrep *spread = nullptr, bool planes = false);
};

// Replace *dst (device, hipMalloc'ed or null) by a copy of n host floats.
int upload_floats(float **dst, const float *src, size_t n);
// Host matrices [rows, n_i] side by side into one device matrix [rows, sum n_i].
int upload_side_by_side(float **dst, const float *const *mats, const int *widths, int count, int rows);

int llama_fail(int code, const std::string &msg);

// Whether all n device floats are bf16 numbers (the lower half of their bits is zero), waited for: asked once per set of
// weights, whatever they came from, so that equal weights take equal products.
int values_are_bf16(const float *w, size_t n, bool *out);

// Second copies of weight matrices, transposed, for the product of a single row (launch_gemvt).
// SHAINET_HIP_NO_TRANSPOSED_WEIGHTS turns them off.  transposed_twin: *twin = src ([rows, cols] on
// the device) transposed, allocated on first use and made again when *stale; returns the twin, or
// null when they are turned off or there is no memory for one (the caller then goes without).
bool transposed_twins_wanted();
// row_scale (nullable): a factor per row of src, i.e. per input of the product: the RMSNorm weights
// gamma of the norm the product always follows, so that (x gamma) W = x (diag(gamma) W) needs no gamma.
const float *transposed_twin(float **twin, bool *stale, const float *src, int rows, int cols, hipStream_t stream,
                             const float *row_scale = nullptr);

}  // namespace shainet
