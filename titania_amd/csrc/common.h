// Internal definitions shared by the HIP device's translation units.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdarg>
#include <cstddef>
#include <cstdint>

#include "../../include/titania_hip.h"

// Concrete types behind the opaque handles of the C ABI.
struct th_device {
    int ordinal = 0;
    hipStream_t stream = nullptr;
    int num_cus = 0;
    // Device staging for token ids handed over from the host.
    uint32_t *tokens = nullptr;
    size_t tokens_cap = 0;
    // Scratch for partial results (attention splits, argmax partials). Grows on
    // demand outside graph capture.
    void *scratch = nullptr;
    size_t scratch_bytes = 0;
    // Scratch that was outgrown after a capture: graphs hold its address, so it
    // is kept for the device's life. Each block is at least twice the one
    // before, so together they are smaller than the current one.
    void *outgrown[64] = {};
    int n_outgrown = 0;
    // A graph has been captured on this device's stream.
    bool captured = false;
    // The device address of the no-alloc entry points' fixed array (looked up
    // once, at th_device_create, with this device current).
    void *noalloc_scratch = nullptr;
    // Split-K partials of a matmul (th::kPartFloats) and partials of an
    // attention split by rounds (th::kAttnRoundFloats), for the device's life:
    // calls that allocate nothing (a matmul of fewer than 16 tokens, so that
    // it can be captured; th_attention_noalloc) then split like any other, and
    // an allocation costs more than most matmuls.
    float *part = nullptr;
    // One u32 the argmax kernels leave their result in.
    uint32_t *token_out = nullptr;
    // th_timer_begin / th_timer_end.
    hipEvent_t ev_begin = nullptr, ev_end = nullptr;
    // Pinned host memory of kPinnedFloats for the results of calls that wait
    // (th::read_back), then kPinnedTokens token ids for the next launch.
    float *pinned = nullptr;
    // Between th_graph_begin and th_graph_end: the stream is being captured.
    bool capturing = false;
};

// A model takes ownership of weight handles it frees on destruction (the
// handles th_model_load uploads); null entries are skipped.
void th_model_own_weights(th_model *m, th_weight *const *w, size_t n);

struct th_buffer {
    float *ptr = nullptr;
    size_t len = 0;  // current length
    size_t cap = 0;  // length it was allocated with
};

struct th_weight {
    uint16_t *ptr = nullptr;  // bf16 bits, row-major
    size_t ndim = 0;
    size_t shape[2] = {0, 0};
    size_t numel = 0;
};

namespace th {

// Records a printf-style message as the calling thread's last error and returns `code`.
int fail(int code, const char *fmt, ...) __attribute__((format(printf, 2, 3)));
void clear_error();

// Floats and token ids that a device's pinned memory holds.
constexpr size_t kPinnedFloats = (size_t)1 << 18, kPinnedTokens = 256;

// Waits for the stream and copies `len` floats out, and *word (device memory;
// may be null) to *word_out.
int read_back(th_device *dev, const float *src, size_t len, float *out, const unsigned *word = nullptr,
              unsigned *word_out = nullptr);

// Makes sure the device scratch holds at least `bytes`; returns its pointer or null.
void *scratch(th_device *dev, size_t bytes);

// The fixed array of the no-alloc entry points: its size, and its address on
// the current device.
size_t noalloc_scratch_bytes();
int noalloc_scratch_address(void **ptr);

}  // namespace th

#define TH_HIP(call)                                                                            \
    do {                                                                                        \
        hipError_t th_e_ = (call);                                                              \
        if (th_e_ != hipSuccess)                                                                \
            return th::fail(TH_ERR_HIP, "%s failed: %s (%s:%d)", #call, hipGetErrorString(th_e_), \
                            __FILE__, __LINE__);                                                \
    } while (0)

#define TH_REQUIRE(cond, ...)                                  \
    do {                                                       \
        if (!(cond)) return th::fail(TH_ERR_INVALID, __VA_ARGS__); \
    } while (0)

// Calls that allocate, move data to or from the host or wait are refused while
// the device's stream is being captured (th_graph_begin .. th_graph_end).
#define TH_NOT_CAPTURING(dev, what)                                                                        \
    TH_REQUIRE(!(dev)->capturing, "%s cannot run while the device's stream is being captured (th_graph_begin)", \
               what)

// Returns the status of `call` from the enclosing function unless it is TH_OK.
#define TRY(call)                 \
    do {                          \
        int rc_ = (call);         \
        if (rc_ != TH_OK) return rc_; \
    } while (0)

// Kernel launchers (host functions defined next to their kernels). Each queues
// work on `s` and returns the launch status; argument checks happen in the ABI layer.
namespace th {

hipError_t launch_embed(hipStream_t s, float *out, const uint16_t *table, size_t dim, const uint32_t *tokens,
                        size_t n);
hipError_t launch_copy(hipStream_t s, float *dst, const float *src, size_t len);
// dst[i] = src[i] for i < len and, if word is not null, dst[len] = *word, in
// host memory that the device can write (both 16-byte aligned).
hipError_t launch_copy_out(hipStream_t s, float *dst, const float *src, size_t len, const unsigned *word);
hipError_t launch_add(hipStream_t s, float *x, const float *y, size_t len);
hipError_t launch_silu_mul(hipStream_t s, float *gate, const float *up, size_t len);
// silu(gate) * up as split_bf16 terms hi/lo (len a multiple of 4).
hipError_t launch_silu_mul_split(hipStream_t s, const float *gate, const float *up, size_t len, uint16_t *hi,
                                 uint16_t *lo);
hipError_t launch_rmsnorm(hipStream_t s, float *x, size_t rows, const uint16_t *w, size_t dim, float eps);
// xb = rmsnorm(x (+)= y): if y, x += y first; xb may equal x.
hipError_t launch_add_rmsnorm(hipStream_t s, float *x, const float *y, float *xb, size_t rows,
                              const uint16_t *w, size_t dim, float eps);
// The same with the residual summed from ny partials y[z * y_stride] (z in
// order; ny = 0: none), the normalized rows to xb (f32) and/or to hi/lo as
// split_bf16 terms (either may be null, not both).
hipError_t launch_add_rmsnorm_parts(hipStream_t s, float *x, const float *y, int ny, size_t y_stride, float *xb,
                                    uint16_t *hi, uint16_t *lo, size_t rows, const uint16_t *w, size_t dim,
                                    float eps);
hipError_t launch_rope(hipStream_t s, float *x, size_t n, const float *table, size_t pos, size_t n_heads,
                       size_t head_dim);
// Two-pass argmax: partials need argmax_partials(n) u64 of scratch.
size_t argmax_partials(size_t n);
hipError_t launch_argmax(hipStream_t s, const float *x, size_t n, uint64_t *partials, uint32_t *token);
hipError_t launch_argmax_partials(hipStream_t s, const float *x, size_t n, uint64_t *partials);

// The kernel that launch_matmul takes, and its parts of K (kMatmulGemm's are
// gemm_outs_plan's), with room for partials or without.
enum MatmulKernel { kMatmulScalar, kMatmulGemv, kMatmulFew, kMatmulRagged, kMatmulGemm };
struct MatmulRoute {
    MatmulKernel kernel;
    int ksplit;
};
MatmulRoute matmul_route(size_t n, size_t rows, size_t cols, bool part);
// About how long launch_matmul takes, with room for partials.
double matmul_us(size_t n, size_t rows, size_t cols);

// out[t*rows + r] = dot(w[r], x[t]) for t < n. Where it splits K, the partials
// go to part (kPartFloats long; null: it does not split).
hipError_t launch_matmul(hipStream_t s, float *out, const uint16_t *w, size_t rows, size_t cols, const float *x,
                         size_t n, float *part = nullptr);

// Attention over caches addressed as base + pos * pos_stride + head * head_stride
// (elements), f32 or bf16. The position is *pos_dev when pos_dev is not null.
struct AttnKernelArgs {
    float *out;
    const float *q;
    const void *k;
    const void *v;
    int n_heads, n_kv_heads, group;
    long long pos;
    const long long *pos_dev;
    long long pos_stride, head_stride;
    int nsplit;
    int kv_bf16;
    float scale;
    float *part_acc;  // [n][n_heads][nsplit][head_dim] when nsplit > 1
    float *part_ml;   // [n][n_heads][nsplit][2]
    // When set, the output goes here as split_bf16 terms [n][n_heads * head_dim]
    // (the o projection's GEMM input); `out` may then be scratch.
    uint16_t *out_hi, *out_lo;
};
// Splits of the sequence for n tokens (of head_dim) whose contexts reach at
// most max_len.
int attention_splits(size_t n, size_t n_heads, size_t n_kv_heads, size_t max_len, size_t head_dim);
// Splits for n tokens at position pos. Several tokens after a context at least
// as long see about the same number of 64-key tiles each, and a CU holds one
// block of the matrix-core kernels, so the launch takes its rounds of 256
// blocks times the tiles a block walks, and the combine (us with
// attention_splits -> these: 11 tokens at 700 of 32 / 8 heads 18.7 -> 11.8, at
// 4000 38.2 -> 20.0; 64 at 30000 of 16 / 8 222.7 -> 80.3; 300 at 2000 of 32 / 8
// 70.7 -> 55.4). The estimate counts tiles of 3.3 us: two more a round to start
// and end it, and the combine's. Of 1227 calls of seven head layouts, 8 to 500
// tokens at up to 31900, none is more than 3% slower than with attention_splits'
// count (geometric mean 1.54 times as fast). Others as attention_splits. *by_rounds, if not null: whether they are such a count,
// whose partials take at most kAttnRoundFloats.
int attention_splits_at(size_t n, size_t n_heads, size_t n_kv_heads, size_t pos, size_t head_dim,
                        bool *by_rounds = nullptr);
constexpr size_t kAttnRoundFloats = (size_t)1024 * 128 * (128 + 2);  // 1024 blocks of 128 rows, head_dim 128
// Scratch floats the partials of `nsplit` splits take (0 for one split).
size_t attention_scratch(size_t n, size_t n_heads, size_t head_dim, int nsplit);
hipError_t launch_attention(hipStream_t s, const AttnKernelArgs &k, size_t n, size_t head_dim);
// Prefill attention of an f32 cache through bf16 hi/lo planes of the keys and
// values: launch_attention's result, bit for bit, with each key and value
// split once per call instead of once per token tile. `planes` holds
// attention_planes_bytes(max_len, n_kv_heads) bytes of scratch (max_len: the
// positions the caches hold). Host positions only (no pos_dev).
size_t attention_planes_bytes(size_t max_len, size_t n_kv_heads);
bool attention_planes_supported(const AttnKernelArgs &k, size_t n, size_t head_dim);
// With split_kv false the planes already hold positions [0, pos + n): the
// q/k/v GEMM's epilogue wrote the new keys and values (QkvPostArgs::kh ..),
// and launch_kv_planes the earlier ones, before that GEMM.
hipError_t launch_attention_planes(hipStream_t s, const AttnKernelArgs &k, size_t n, size_t head_dim, void *planes,
                                   size_t planes_bytes, size_t max_len, bool split_kv = true);
// The planes of positions [0, valid) from the caches of k (the 64-position
// tile that holds `valid` gets zeros past it).
hipError_t launch_kv_planes(hipStream_t s, const AttnKernelArgs &k, size_t valid, void *planes, size_t planes_bytes,
                            size_t max_len);
// The four planes inside `planes` for caches of max_len positions.
struct PlanePtrs {
    uint16_t *kh, *kl, *vh, *vl;
    long long plane_len;
};
PlanePtrs attention_planes_of(void *planes, size_t max_len, size_t n_kv_heads);
// Merges attention partials of `heads` (token, head) pairs into out (f32) or,
// when hi is set, into hi/lo as split_bf16 terms.
hipError_t launch_attn_combine(hipStream_t s, float *out, const float *part_acc, const float *part_ml, size_t heads,
                               int nsplit, int hd, uint16_t *hi = nullptr, uint16_t *lo = nullptr);

}  // namespace th
