// On-device sampling of the next token (model/sampler.rs:21-59): the top_k
// largest logits under total order (equal logits: the lower token first, an
// order the reference leaves unspecified), a softmax at the temperature over
// them, the shortest prefix whose probability reaches top_p, and a draw from
// that prefix with xorshift64*.
//
// The search starts from the largest (key, inverted index) word of every 16
// consecutive logits, which the decode step's output projection leaves beside
// its logits (elsewhere group_max_kernel makes them). The top_k-th largest of
// these maxima is no larger than the top_k-th largest logit (top_k groups
// each hold one as large), so only the groups whose maximum reaches it can
// hold a candidate: one block finds that threshold, reads those groups and
// ranks what reaches it. The block then does the reference's arithmetic in
// its order (the softmax sum and the cumulative mass are sequential f32
// folds).
//
// Bound by the block's round trips (maxima, logits of the chosen groups) and
// barriers, not by bytes: 13.4 us a draw at 151936 logits and top_k 20, where
// sorting every 8192 logits in LDS and then the blocks' candidates took 72.6
// + 73.6 us in two launches.
#include "common.h"
#include "device_util.h"
#include "sample.h"

namespace th {

namespace {

constexpr int kThreads = 1024, kWaves = kThreads / 64;
// Logits a maximum covers: the rows of a block of launch_step_logits.
constexpr int kGroup = 16;
// Maxima a thread holds: all of them at the largest vocabulary.
constexpr int kMaxPerThread = (int)(kSampleMaxVocab / kGroup / kThreads);
// Most groups that are read, and candidates that are ranked: at least
// kSampleMaxTopK; a power of two, with two or more threads a candidate.
constexpr int kMost = 512;
constexpr int kLogitsPerThread = kMost * kGroup / kThreads;
constexpr int kBins = kThreads;  // a bin a thread
static_assert(kMost >= kSampleMaxTopK && kThreads >= 2 * kMost && kSampleMaxVocab % (kGroup * kThreads) == 0, "");

// argmax_pack's value back.
__device__ __forceinline__ float key_value(uint64_t word) {
    int32_t k = (int32_t)((uint32_t)(word >> 32) ^ 0x80000000u);
    k ^= (int32_t)(((uint32_t)(k >> 31)) >> 1);
    return __int_as_float(k);
}

// groups[g] = the largest word of logits [16 g, 16 g + 16): four lanes a group.
__global__ __launch_bounds__(256) void group_max_kernel(const float *__restrict__ logits, size_t vocab, size_t m,
                                                        uint64_t *__restrict__ groups) {
    const size_t q = (size_t)blockIdx.x * 256 + threadIdx.x, i = q * 4;
    uint64_t best = 0;
    if (i + 4 <= vocab) {
        const float4 v = *reinterpret_cast<const float4 *>(logits + i);
        best = max_u64(max_u64(argmax_pack(v.x, (uint32_t)i), argmax_pack(v.y, (uint32_t)i + 1)),
                       max_u64(argmax_pack(v.z, (uint32_t)i + 2), argmax_pack(v.w, (uint32_t)i + 3)));
    } else {
        for (size_t t = i; t < vocab; ++t) best = max_u64(best, argmax_pack(logits[t], (uint32_t)t));
    }
    best = max_u64(best, __shfl_xor(best, 1, 64));
    best = max_u64(best, __shfl_xor(best, 2, 64));
    if ((q & 3) == 0 && q / 4 < m) groups[q / 4] = best;
}

struct Shared {
    unsigned bins[kBins];
    unsigned wave_sum[kWaves];
    uint64_t wave_hi[kWaves], wave_lo[kWaves];
    unsigned bin, below, upto;   // the bin of the k-th, and the counts before and through it
    unsigned count;              // entries of `chosen`, then of `cand`
    int chosen[kMost];
    alignas(16) uint64_t cand[kMost];
    uint64_t sorted[kSampleMaxTopK];
    alignas(16) float probs[kSampleMaxTopK + 16];
    uint32_t picked;
};

// A word that k to kMost of the block's words (N a thread, 0: none; all
// distinct; at least k of them) reach. Bins the words between the largest
// and the smallest by the leading bits of their distance from the largest,
// and goes into the k-th's bin while the words through it are more than
// kMost. A step keeps 2^-10 of the range, so a 64-bit one ends within seven;
// one is the rule (the maxima of 16 logits lie within a few octaves).
template <int N>
__device__ __forceinline__ uint64_t threshold(const uint64_t (&v)[N], unsigned k, Shared &sh) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    uint64_t hi = 0, lo = ~0ull;
#pragma unroll
    for (int j = 0; j < N; ++j) {
        hi = max_u64(hi, v[j]);
        lo = v[j] && v[j] < lo ? v[j] : lo;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        hi = max_u64(hi, __shfl_xor(hi, o, 64));
        const uint64_t other = __shfl_xor(lo, o, 64);
        lo = other < lo ? other : lo;
    }
    if (lane == 0) {
        sh.wave_hi[wave] = hi;
        sh.wave_lo[wave] = lo;
    }
    sh.bins[tid] = 0;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
        hi = max_u64(hi, sh.wave_hi[w]);
        lo = sh.wave_lo[w] < lo ? sh.wave_lo[w] : lo;
    }
    unsigned above = 0;  // words past hi
    for (;;) {
        const int bits = 64 - __clzll((long long)(hi - lo));
        const int shift = bits > 10 ? bits - 10 : 0;
#pragma unroll
        for (int j = 0; j < N; ++j)
            if (v[j] >= lo && v[j] <= hi) atomicAdd(&sh.bins[(hi - v[j]) >> shift], 1u);
        __syncthreads();
        const unsigned mine = sh.bins[tid];
        unsigned sum = mine;  // inclusive over the wave's bins
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const unsigned t = __shfl_up(sum, o, 64);
            if (lane >= o) sum += t;
        }
        if (lane == 63) sh.wave_sum[wave] = sum;
        __syncthreads();
#pragma unroll
        for (int w = 0; w < kWaves; ++w) sum += w < wave ? sh.wave_sum[w] : 0;
        sum += above;
        if (sum - mine < k && k <= sum) {
            sh.bin = (unsigned)tid;
            sh.below = sum - mine;
            sh.upto = sum;
        }
        sh.bins[tid] = 0;
        __syncthreads();
        const unsigned bin = sh.bin, upto = sh.upto;
        const uint64_t reach = ((uint64_t)(bin + 1) << shift) - 1;  // the bin's last distance from hi
        const uint64_t low = hi - lo <= reach ? lo : hi - reach;
        if (upto <= (unsigned)kMost) return low;
        above = sh.below;
        hi -= (uint64_t)bin << shift;
        lo = low;
        __syncthreads();  // bin, below and upto are read before the next step's are written
    }
}

// Calls f(i, probs[i]) for i < k in order, sixteen read ahead.
template <class F>
__device__ __forceinline__ void in_order(const float *probs, int k, F f) {
    const float4 *p = reinterpret_cast<const float4 *>(probs);
    float4 cur[4] = {p[0], p[1], p[2], p[3]};
    for (int b = 0; b < k; b += 16) {
        p += b + 16 < k ? 4 : 0;
        const float4 next[4] = {p[0], p[1], p[2], p[3]};
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            f(b + 4 * q, cur[q].x);
            f(b + 4 * q + 1, cur[q].y);
            f(b + 4 * q + 2, cur[q].z);
            f(b + 4 * q + 3, cur[q].w);
            cur[q] = next[q];
        }
    }
}

// model/sampler.rs:66-76.
__device__ __forceinline__ uint64_t rng_next_u64(uint64_t &x) {
    x ^= x >> 12;
    x ^= x << 25;
    x ^= x >> 27;
    return x * 0x2545F4914F6CDD1DULL;
}

__device__ __forceinline__ float rng_next_f32(uint64_t &x) {
    return (float)(rng_next_u64(x) >> 40) / (float)(1u << 24);
}

__global__ __launch_bounds__(kThreads) void sample_kernel(const float *__restrict__ logits, size_t vocab,
                                                         const uint64_t *__restrict__ groups, int m,
                                                         SampleState *ss, StepState *st, int advance,
                                                         PickEmbed emb) {
    __shared__ Shared sh;
    const int tid = threadIdx.x;
    // The states, read with the maxima (their waits then end together).
    const SampleState sampler = *ss;
    StepState loc{};
    if (tid == 0 && st) loc = *st;
    const int k = sampler.top_k;
    uint64_t g[kMaxPerThread];
#pragma unroll
    for (int j = 0; j < kMaxPerThread; ++j) g[j] = tid + j * kThreads < m ? groups[tid + j * kThreads] : 0;
    if (tid == 0) sh.count = 0;
    // Every group, or those whose maximum reaches the top_k-th largest.
    uint64_t least = 1;
    if (m > k) least = threshold(g, (unsigned)k, sh);
    else __syncthreads();
#pragma unroll
    for (int j = 0; j < kMaxPerThread; ++j)
        if (g[j] >= least) sh.chosen[atomicAdd(&sh.count, 1u)] = tid + j * kThreads;
    __syncthreads();
    const int n_logits = (int)sh.count * kGroup;
    uint64_t c[kLogitsPerThread];
#pragma unroll
    for (int j = 0; j < kLogitsPerThread; ++j) {
        const int e = tid + j * kThreads;
        const size_t i = e < n_logits ? (size_t)sh.chosen[e / kGroup] * kGroup + e % kGroup : vocab;
        const uint64_t word = i < vocab ? argmax_pack(logits[i], (uint32_t)i) : 0;
        c[j] = word >= least ? word : 0;
    }
    __syncthreads();
    if (tid == 0) sh.count = 0;
    __syncthreads();
    // What reaches the threshold: a few more than top_k, unless the largest
    // logits sit side by side.
    unsigned mine = 0;
#pragma unroll
    for (int j = 0; j < kLogitsPerThread; ++j) mine += c[j] ? 1 : 0;
    if (mine) atomicAdd(&sh.count, mine);
    __syncthreads();
    if (sh.count > (unsigned)kMost) least = threshold(c, (unsigned)k, sh);
    __syncthreads();
    if (tid == 0) sh.count = 0;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kLogitsPerThread; ++j)
        if (c[j] >= least) sh.cand[atomicAdd(&sh.count, 1u)] = c[j];
    __syncthreads();
    // Each candidate's rank, its comparisons dealt to `share` neighbouring lanes.
    const int n = (int)sh.count;
    int share = kThreads / kMost;
    while (share < 64 && n * share * 2 <= kThreads) share *= 2;
    if (tid < n * share) {
        const uint64_t word = sh.cand[tid / share];
        int rank = 0;
        for (int i = tid % share; i < n; i += share) rank += sh.cand[i] > word ? 1 : 0;
        for (int o = 1; o < share; o <<= 1) rank += __shfl_xor(rank, o, 64);
        if (tid % share == 0 && rank < k) sh.sorted[rank] = word;
    }
    __syncthreads();
    if (tid < 64) {
        // model/sampler.rs:35-58, in its order; the exponentials and the
        // quotients, which have none, a lane each, the folds in every lane
        // alike. Zeros past top_k leave the sum as it is.
        const float t = sampler.temperature, top_p = sampler.top_p;
        const float max = key_value(sh.sorted[0]);
        for (int i = tid; i < kSampleMaxTopK + 16; i += 64)
            sh.probs[i] = i < k ? expf((key_value(sh.sorted[i]) - max) / t) : 0.f;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
        float sum = 0.f;
        in_order(sh.probs, k, [&](int, float p) { sum += p; });
        for (int i = tid; i < k; i += 64) sh.probs[i] /= sum;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
        float cumulative = 0.f;
        int kept = 0;
        in_order(sh.probs, k, [&](int i, float p) {
            if (i < k && cumulative < top_p) {
                cumulative += p;
                kept += 1;
            }
        });
        uint64_t x = sampler.rng;
        float r = rng_next_f32(x) * cumulative;
        int at = kept - 1;
        bool drawn = false;
        in_order(sh.probs, kept, [&](int i, float p) {
            if (i < kept && !drawn) {
                r -= p;
                if (r <= 0.f) {
                    at = i;
                    drawn = true;
                }
            }
        });
        if (tid == 0) {
            // Steps after a stop token draw nothing (their picks are dropped).
            if (!loc.stopped) {
                ss->rng_prev = sampler.rng;
                ss->rng = x;
            }
            uint32_t tok = argmax_index(sh.sorted[at]);
            if (st) tok = step_record_from(st, loc, advance, tok);
            else ss->token = tok;
            sh.picked = tok;
        }
    }
    if (!st || !emb.table) return;
    __syncthreads();
    write_embedding(emb, sh.picked);
}

}  // namespace

size_t sample_scratch_bytes(size_t vocab) { return (vocab + kGroup - 1) / kGroup * sizeof(uint64_t); }

hipError_t launch_sample(hipStream_t s, const float *logits, size_t vocab, void *scratch, SampleState *ss,
                         StepState *st, int advance, const PickEmbed &emb, const uint64_t *maxima) {
    if (vocab == 0 || vocab > kSampleMaxVocab || (emb.table && emb.dim % 8) || (uintptr_t)logits % 16)
        return hipErrorInvalidValue;
    const size_t m = (vocab + kGroup - 1) / kGroup;
    if (!maxima) {
        uint64_t *groups = static_cast<uint64_t *>(scratch);
        group_max_kernel<<<(unsigned)((m * 4 + 255) / 256), 256, 0, s>>>(logits, vocab, m, groups);
        maxima = groups;
    }
    sample_kernel<<<1, kThreads, 0, s>>>(logits, vocab, maxima, (int)m, ss, st, advance, emb);
    return hipGetLastError();
}

}  // namespace th
