// Matmuls of a few tokens: out[t][r] = w[r] . x[t] (model/cpu.rs:49-77) for
// tiles of up to 16 tokens, on the matrix cores.
//
// Bound by the weights' bytes, each read once, through the CU's vector-memory
// path, which the activations share: a tile of 16 weight rows needs all of x,
// so reading x again for every tile costs as much as the weights do
// (measured at 11 tokens x 19456 x 2560: 20.7 us for the weights alone, 14.2
// for the activations alone, 33 together). So each wave of a block keeps its
// slice of K of the activations in registers, as matrix operands, and the
// block walks weight tiles, the next tile's rows in flight while one is
// multiplied: 26.7 us (3.7 TB/s), where the GEMV took 46.8 for each 8 tokens.
// The waves' partial tiles meet in LDS, one barrier a tile. A turn of 11
// tokens on four Qwen3-4B layers: 1.120 -> 0.501 ms; 50 tokens x 1000 x 1096:
// 45.0 -> 6.2 us.
//
// The activations enter as three bf16 terms (8 significant bits each, cut off,
// so that their sum is the f32 value exactly), three products a weight
// fragment: measured against 64 bits, the results are as close as the f32
// GEMV's or closer (8.1e-8 against 1.0e-7 at 1096 columns), infinities and
// NaN as the f32 products give them (repair_nan).
#include "few.h"

#include "common.h"
#include "device_util.h"

namespace th {
namespace {

typedef bf16_term8 bf16x8;
typedef f32_acc4 f32x4;

constexpr int kTokens = 16, kTerms = 3;
constexpr unsigned kPastEnd = 0xfffffff0u;  // an offset no descriptor reaches: the load gives zero

struct Args {
    const uint16_t *w[3];
    float *out[3];
    int rows[3];
    int tiles0, tiles1, tiles;  // row tiles of the first, the first two and all matrices
    const float *x;
    int n, cols;
    int ksplit;
};

template <bool NT>
__device__ __forceinline__ uint4 load16(__amdgpu_buffer_rsrc_t r, unsigned off) {
    const th_u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, NT ? kCachePolicyNt : 0);
    return make_uint4(v.x, v.y, v.z, v.w);
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t records(const void *p, unsigned bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, (int)bytes, kBufferRsrcWord3);
}

enum Epi { kRows, kSilu };

// WK waves, each of NKS steps of 32 columns of K, for the 16 tokens of
// blockIdx.y; blockIdx.z takes a part of K (kRows, one matrix: partials).
// The block takes row tiles blockIdx.x, + gridDim.x, ... (kSilu: the gate and
// then the up rows of each). K past WK * NKS steps goes in chunks, x read
// again for each.
template <int NKS, int WK, int EPI, bool NT>
__global__ __launch_bounds__(64 * WK) void few_kernel(Args a) {
    __shared__ f32x4 red[2][WK][64];
    const int lane = threadIdx.x & 63, wk = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int fr = lane & 15, fq = lane >> 4, cols = a.cols, t0 = blockIdx.y * kTokens;
    // This block's K: steps [kb, ke), in chunks of WK * NKS.
    const int steps = (cols + 31) / 32, z = blockIdx.z;
    const int kb = (int)((long long)z * steps / a.ksplit), ke = (int)((long long)(z + 1) * steps / a.ksplit);
    const int chunks = (ke - kb + WK * NKS - 1) / (WK * NKS);
    const float *xb = a.x + (size_t)t0 * cols;
    const unsigned xbytes = (unsigned)(a.n - t0 < kTokens ? a.n - t0 : kTokens) * (unsigned)cols * 4u;

    // Lane (fq, fr) of step k holds columns 32 k + 8 fq .. + 8 of token fr, or
    // of weight row fr. Columns past the row's end (cols is a multiple of 8)
    // and steps past this block's are zero on both sides, tokens and rows
    // past the last by the descriptors' sizes.
    auto column = [&](int chunk, int k) {
        const int step = kb + (chunk * WK + wk) * NKS + k, c = step * 32 + fq * 8;
        return step < ke && c < cols ? c : -1;
    };
    bf16x8 x[NKS][kTerms];
    auto load_x = [&](int chunk) {
        const __amdgpu_buffer_rsrc_t r = records(xb, xbytes);
        uint4 v[NKS][2];
#pragma unroll
        for (int k = 0; k < NKS; ++k) {
            const int c = column(chunk, k);
            const unsigned off = c >= 0 ? ((unsigned)fr * (unsigned)cols + (unsigned)c) * 4u : kPastEnd - 16u;
            v[k][0] = load16<false>(r, off);
            v[k][1] = load16<false>(r, off + 16u);
        }
        return [=](bf16x8(&xs)[NKS][kTerms]) {
#pragma unroll
            for (int k = 0; k < NKS; ++k) split3(v[k][0], v[k][1], xs[k]);
        };
    };
    // The weights of (tile, chunk), `second`: of up. Past the last tile, no
    // records: zeros and no memory access.
    auto load_w = [&](uint4(&w)[NKS], int tile, int chunk, bool second) {
        const bool live = tile < a.tiles;
        const int seg = EPI == kSilu ? (second ? 1 : 0) : tile < a.tiles0 ? 0 : tile < a.tiles1 ? 1 : 2;
        const int r0 = 16 * (EPI == kSilu ? tile : tile - (seg == 0 ? 0 : seg == 1 ? a.tiles0 : a.tiles1));
        const uint16_t *m = seg == 0 ? a.w[0] : seg == 1 ? a.w[1] : a.w[2];
        const int rows = (seg == 0 || EPI == kSilu ? a.rows[0] : seg == 1 ? a.rows[1] : a.rows[2]) - r0;
        const unsigned bytes = live ? (unsigned)(rows < 16 ? rows : 16) * (unsigned)cols * 2u : 0u;
        const __amdgpu_buffer_rsrc_t r = records(live ? m + (size_t)r0 * cols : m, bytes);
#pragma unroll
        for (int k = 0; k < NKS; ++k) {
            const int c = column(chunk, k);
            w[k] = load16<NT>(r, c >= 0 ? ((unsigned)fr * (unsigned)cols + (unsigned)c) * 2u : kPastEnd);
        }
    };

    uint4 w[2][NKS];
    {
        // The activations first: their conversion then runs while the first
        // weights stream in behind.
        auto convert = load_x(0);
        load_w(w[0], blockIdx.x, 0, false);
        convert(x);
    }
    // The first terms of even and odd steps and the others sum apart: shorter
    // chains of dependent products, and of roundings.
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    f32x4 gate = zero, acc[3] = {zero, zero, zero};
    int tile = blockIdx.x, chunk = 0, turn = 0;  // turn: tiles done, deals the sums to the waves
    // Two (tile, chunk)s an iteration, from the two weight buffers; a tile is
    // gate and up with kSilu (chunks are then walked once for each).
    int part2 = 0;  // kSilu: 0 gate, 1 up
    bool nan = false;
    while (tile < a.tiles) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            // The next (tile, chunk)'s weights go out before this one's products.
            int next_tile = tile, next_chunk = chunk + 1, next_part = part2;
            if (next_chunk == chunks) {
                next_chunk = 0;
                if (EPI == kSilu && part2 == 0) {
                    next_part = 1;
                } else {
                    next_part = 0;
                    next_tile += (int)gridDim.x;
                }
            }
            load_w(w[h ^ 1], next_tile, next_chunk, next_part != 0);
#pragma unroll
            for (int k = 0; k < NKS; ++k)
#pragma unroll
                for (int i = 0; i < kTerms; ++i) {
                    f32x4 &to = acc[i == 0 ? k & 1 : 2];
                    to = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[k][i], __builtin_bit_cast(bf16x8, w[h][k]), to, 0, 0,
                                                                 0);
                }
            if (next_chunk == 0) {
                // The tile is whole: the waves' sums meet, in wave order.
                // Buffer h is free: its last readers passed the barrier of
                // the tile between.
                red[turn & 1][wk][lane] = acc[0] + acc[1] + acc[2];
                acc[0] = acc[1] = acc[2] = zero;
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
                __builtin_amdgcn_s_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
                const int owner = (EPI == kSilu ? turn >> 1 : turn) % WK;
                if (wk == owner && tile < a.tiles) {
                    f32x4 s = red[turn & 1][0][lane];
#pragma unroll
                    for (int k = 1; k < WK; ++k) s += red[turn & 1][k][lane];
                    nan |= any_nan(s);
                    if (EPI == kSilu && part2 == 0) {
                        gate = s;
                    } else {
                        // Lane (fq, fr): tokens 4 fq + i of row fr.
                        const int seg = EPI == kSilu || tile < a.tiles0 ? 0 : tile < a.tiles1 ? 1 : 2;
                        const int row = 16 * (tile - (seg == 0 ? 0 : seg == 1 ? a.tiles0 : a.tiles1)) + fr;
                        const int rows = seg == 0 ? a.rows[0] : seg == 1 ? a.rows[1] : a.rows[2];
                        float *out = seg == 0 ? a.out[0] + (size_t)z * a.n * rows : seg == 1 ? a.out[1] : a.out[2];
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const int t = t0 + 4 * fq + i;
                            if (row < rows && t < a.n)
                                out[(size_t)t * rows + row] = EPI == kSilu ? silu(gate[i]) * s[i] : s[i];
                        }
                    }
                }
                turn += 1;
            }
            if (chunks > 1) {
                auto convert = load_x(next_chunk);
                convert(x);
            }
            tile = next_tile;
            chunk = next_chunk;
            part2 = next_part;
        }
    }
    if (__builtin_expect(!nan, 1)) return;
    // This wave's tiles again, for what infinite weights made NaN (here and not
    // in the loop, whose registers and instructions it would add to).
    const int c0 = 32 * kb, c1 = 32 * ke < cols ? 32 * ke : cols;
    unsigned looked = 0;
    for (tile = blockIdx.x + wk * gridDim.x; tile < a.tiles; tile += WK * gridDim.x) {
        const int seg = EPI == kSilu || tile < a.tiles0 ? 0 : tile < a.tiles1 ? 1 : 2;
        const int row = 16 * (tile - (seg == 0 ? 0 : seg == 1 ? a.tiles0 : a.tiles1)) + fr;
        const int rows = seg == 0 ? a.rows[0] : seg == 1 ? a.rows[1] : a.rows[2];
        float *out = seg == 0 ? a.out[0] + (size_t)z * a.n * rows : seg == 1 ? a.out[1] : a.out[2];
        const size_t at = (size_t)(row < rows ? row : rows - 1) * cols;
        const uint16_t *wr = (seg == 0 ? a.w[0] : seg == 1 ? a.w[1] : a.w[2]) + at;
        const uint16_t *up = EPI == kSilu ? a.w[1] + at : wr;
        f32x4 s = zero;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (row < rows && t0 + 4 * fq + i < a.n) s[i] = out[(size_t)(t0 + 4 * fq + i) * rows + row];
        if (!any_nan(s)) continue;
        const f32x4 was = s;
        repair_nan(s, wr, up, row < rows, xb, a.n - t0, cols, c0, c1, fq, looked);
        if (EPI == kSilu) {
            f32x4 u = was;
            repair_nan(u, up, wr, row < rows, xb, a.n - t0, cols, c0, c1, fq, looked);
#pragma unroll
            for (int i = 0; i < 4; ++i) s[i] = silu(s[i]) * u[i];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (was[i] != was[i] && row < rows && t0 + 4 * fq + i < a.n)
                out[(size_t)(t0 + 4 * fq + i) * rows + row] = s[i];
    }
}

// K steps of a wave for a block's K of `steps` steps: the fewest instances
// whose eight waves hold it, since idle steps still issue (11 tokens x 1024 x
// 2048 in four parts of 16 steps: 4.3 / 4.8 / 5.1 / 5.9 / 7.2 us with 2 / 3 /
// 4 / 6 / 10 steps a wave; four waves of 8, 5.7). Past 80, chunks.
constexpr int kWaves = 8, kMaxSteps = 10 * kWaves;

template <int EPI, bool NT>
hipError_t few_launch(hipStream_t s, const Args &a, dim3 grid, int steps) {
    constexpr int kBlock = 64 * kWaves;
    if (steps <= 2 * kWaves) few_kernel<2, kWaves, EPI, NT><<<grid, kBlock, 0, s>>>(a);
    else if (steps <= 3 * kWaves) few_kernel<3, kWaves, EPI, NT><<<grid, kBlock, 0, s>>>(a);
    else if (steps <= 4 * kWaves) few_kernel<4, kWaves, EPI, NT><<<grid, kBlock, 0, s>>>(a);
    else if (steps <= 6 * kWaves) few_kernel<6, kWaves, EPI, NT><<<grid, kBlock, 0, s>>>(a);
    else if (steps <= 8 * kWaves) few_kernel<8, kWaves, EPI, NT><<<grid, kBlock, 0, s>>>(a);
    else few_kernel<10, kWaves, EPI, NT><<<grid, kBlock, 0, s>>>(a);
    return hipGetLastError();
}

template <int EPI>
hipError_t few(hipStream_t s, Args &a) {
    const unsigned y = (unsigned)((a.n + kTokens - 1) / kTokens);
    const int steps = (a.cols + 31) / 32, per = (steps + a.ksplit - 1) / a.ksplit;
    // One block a CU, each walking its share of the tiles: with two, x is
    // read twice as often (11 tokens x 19456 x 2560: 26.7 against 34.8 us; x
    // 6144 x 1024: 6.6 against 8.7).
    const int slots = std::max(1, 256 / (int)(y * a.ksplit));
    const int rounds = (a.tiles + slots - 1) / slots;
    const dim3 grid((unsigned)((a.tiles + rounds - 1) / rounds), y, (unsigned)a.ksplit);
    // Weights that one token tile reads are not kept in the caches.
    return y == 1 ? few_launch<EPI, true>(s, a, grid, per) : few_launch<EPI, false>(s, a, grid, per);
}

}  // namespace

bool few_supported(size_t n, size_t rows, size_t cols) {
    return n >= 1 && n <= 65535 * (size_t)kTokens && rows >= 1 && rows < ((size_t)1 << 30) && cols >= 8 &&
           cols % 8 == 0 && cols < ((size_t)1 << 24);
}

int few_ksplit(size_t n, size_t rows, size_t cols) {
    // Few row tiles leave CUs idle and make each read all of x: K in up to
    // four parts of at least 16 steps (11 tokens, one part / two / four: x
    // 1024 x 2048 8.1 / 6.4 / 4.3 us, 1024 x 3072 16.0 / 7.2 / 5.2, 2560 x
    // 4096 17.7 / 10.1 / 8.6, 2560 x 9728 31.5 / 32.3 / 16.6). And K that the
    // registers do not hold (chunks read x again for every 16 rows), in as many
    // parts as they do: 8 tokens x 8192 x 3072 25.1 -> 15.0 us, x 9001 x 3000 34.2
    // -> 20.1, x 4096 x 8192 32.2 -> 19.3, x 64000 x 4096 172 -> 95.
    const size_t tiles = (rows + 15) / 16 * ((n + kTokens - 1) / kTokens), steps = (cols + 31) / 32;
    int k = 1;
    while (k < kFewMaxSplitK && steps / (2 * k) >= 16 && (tiles * k < 512 || steps > kMaxSteps * k)) k *= 2;
    return k;
}

bool few_preferred(size_t n, size_t rows, size_t cols, int n_outs) {
    if (n < kGemmMinTokens) return true;
    if (n > 64) return false;
    // The GEMM splits the K of a single matrix and reads each weight once for
    // 64 tokens, this kernel once for every 16: so many tiles of 16 tokens
    // times rows. Us, this kernel / that one, weights from HBM: one matrix of
    // 1024 columns, 6144 rows and 33 / 64 tokens 10.8 / 10.0, 11.1 / 12.0;
    // 16384 and 16 / 17 / 64 tokens 10.0 / 12.1, 13.1 / 12.8, 24.5 / 15.1;
    // 151936 and 16 / 64 67.6 / 77.7, 197.7 / 93.5. Of more columns, 1024 x
    // 2048 and 16 tokens 9.0 / 7.4, 2560 x 9728 36.5 / 21.9.
    const size_t work = (n + kTokens - 1) / kTokens * rows;
    if (n_outs == 1) return cols <= 1024 && (n <= (size_t)kTokens || work <= 24576);
    // Several matrices: the GEMM does not split K, and gate and up then take a
    // launch more. Gate and up of 16384 x 1024, 17 / 33 / 64 tokens 21.8 / 19.0,
    // 31.7 / 20.3, 38.7 / 23.9, of 8192 12.6 / 15.0, 19.2 / 15.5, 21.3 / 16.3, of
    // 4096 8.2 / 12.2, 12.2 / 12.4, 12.2 / 12.8; 9728 x 2560, 32 / 33 tokens 35.1
    // / 36.8, 44.5 / 36.9; q, k and v of 6144 x 2560, 64 tokens 25.2 / 30.9, of
    // 12288 x 1024, 33 tokens 20.7 / 14.9. Past 2560 columns it goes in chunks:
    // gate and up of 2048 x 4096, 32 / 33 tokens 31.5 / 41.2, 54.4 / 41.0; of
    // 8192 x 4096, 17 tokens 101.7 / 47.6.
    return work <= (cols > 2560 ? 8192 : n <= 32 ? 40960 : 32768);
}

bool few_together(size_t n, const size_t *rows, int n_outs, size_t cols) {
    size_t total = 0;
    bool whole = true;
    double each = n_outs == 2 ? 3 : 0;  // silu_mul
    for (int i = 0; i < n_outs; ++i) {
        if (n < 2 || !few_supported(n, rows[i], cols)) return false;
        total += rows[i];
        whole = whole && gemm_supported(rows[i], cols);
        each += matmul_us(n, rows[i], cols);
    }
    if (n >= kGemmMinTokens && whole) return few_preferred(n, total, cols, n_outs);
    // Launches together do not split K: past what the registers hold, in
    // chunks. Us together / each: gate and up of 8192 x 4096, 2 / 3 / 8 tokens
    // 40.4 / 32.6, 40.8 / 38.2, 46.5 / 40.0, of 2048 x 4096 22.6 / 18.9, 23.1 /
    // 21.7, 26.1 / 20.5; q, k and v of 12288 x 4096, 2 / 3 tokens 36.7 / 32.7, 36.9
    // / 36.4, of 6144 x 4096 27.6 / 29.2, 28.1 / 33.2, of 10240 x 8192, 3 / 8
    // tokens 64.6 / 66.1, 71.7 / 56.7. And of two tokens the GEMV is as fast where the
    // weights are many: gate and up of 9728 x 2560 28.1 / 26.3, of 3072 x 1024 6.2
    // / 10.2.
    if (n == 2 && (cols > 2560 || total * cols > ((size_t)40 << 20))) return false;
    if (n_outs == 2 && cols > 2560) return false;
    return n == 3 || (n < kGemmMinTokens && cols <= 2560) || few_us(n, total, cols) <= each;
}

double few_us(size_t n, size_t rows, size_t cols, int ksplit) {
    // Rounds of row tiles, past the chunks that the registers hold three times
    // as long a column; besides, the launch and the first read of x, and the
    // sum of the parts.
    const size_t y = (n + kTokens - 1) / kTokens * (size_t)ksplit, slots = std::max<size_t>(1, 256 / y);
    const double rounds = (double)(((rows + 15) / 16 + slots - 1) / slots), c = 1e-3 * (double)cols / ksplit;
    return (c > 2.56 ? 4 + 3 * rounds * c : 4 + 2 * c + rounds * std::max(0.9 * c, 0.5)) + (ksplit > 1 ? 2 : 0);
}

hipError_t launch_few(hipStream_t s, const float *x, size_t n, size_t cols, const GemmOut *outs, int n_outs,
                      float *part, int ksplit) {
    if (n == 0) return hipSuccess;
    if (n_outs < 1 || n_outs > 3 || ksplit < 1 || ksplit > kFewMaxSplitK || (ksplit > 1 && (n_outs != 1 || !part)) ||
        (size_t)ksplit > (cols + 31) / 32 || (uintptr_t)x % 16)
        return hipErrorInvalidValue;
    Args a{};
    a.x = x;
    a.n = (int)n;
    a.cols = (int)cols;
    a.ksplit = ksplit;
    size_t tiles = 0;
    for (int i = 0; i < 3; ++i) {
        if (i < n_outs) {
            if (!few_supported(n, outs[i].rows, cols) || (uintptr_t)outs[i].w % 16) return hipErrorInvalidValue;
            a.w[i] = outs[i].w;
            a.out[i] = ksplit > 1 ? part : outs[i].out;
            a.rows[i] = (int)outs[i].rows;
            tiles += (outs[i].rows + 15) / 16;
        }
        if (i == 0) a.tiles0 = (int)tiles;
        if (i == 1) a.tiles1 = (int)tiles;
    }
    a.tiles = (int)tiles;
    return few<kRows>(s, a);
}

hipError_t launch_few_silu(hipStream_t s, const float *x, size_t n, size_t cols, const uint16_t *gate,
                           const uint16_t *up, size_t inter, float *h) {
    if (n == 0) return hipSuccess;
    if (!few_supported(n, inter, cols) || ((uintptr_t)x | (uintptr_t)gate | (uintptr_t)up) % 16)
        return hipErrorInvalidValue;
    Args a{};
    a.x = x;
    a.n = (int)n;
    a.cols = (int)cols;
    a.ksplit = 1;
    a.w[0] = gate;
    a.w[1] = up;
    a.out[0] = h;
    a.rows[0] = (int)inter;
    a.tiles0 = a.tiles1 = a.tiles = (int)((inter + 15) / 16);
    return few<kSilu>(s, a);
}

}  // namespace th
