// gram_kernel.hpp -- the Gram entries between the markers of a sweep's blocks.
//
// The pipelined sweep (pipe_kernel.hpp) needs, for a marker h whose beta changes, how the dots of the later
// markers of h's block and of all markers of the next block change per unit of beta_old - beta_new:
//   G[h][k] = sum_i u_h(x_hi) w_k(x_ki),
// u_h the residual change per unit (densebayesrkernel.cpp:17-20, raggedbayesrkernel.cpp:10-30) and w_k the dot
// weight (sparsebayesrkernel.cpp:24-27, eigenbayesrkernel.cpp:10-20). They depend on the genotypes and on the
// marker order alone, so one kernel ahead of the sweep forms them for a whole iteration.
//
// u and w are combinations of 1 and at most three small integers per 2-bit code, the marker's bases: G follows in
// FP64 from per-marker sums and the products of the bases' integers, which the i8 matrix cores give exactly. Sparse
// columns have the dosage (0 for a missing call) and the missing-call indicator. Dense columns hold whatever four
// values the caller's table has, so their bases are found from the table: three values at equal steps share one (the
// dosages of a standardised column, under any numbering of its codes), every other value that occurs has its own.
//
// One workgroup per block of up to 64 markers: the 2-bit codes of the block's and the next block's columns
// (128 columns) are staged through LDS in chunks of 1,024 individuals, each of the 8 waves takes 128
// individuals of a chunk, expands the codes to bytes (a byte permute through a 4-entry table) and accumulates
// seven 32 x 32 tiles of the 64 x 128 result (the tile below the diagonal is not needed). The 28 matrix
// instructions of a wave and chunk and their 176 expansion instructions take about as long as each other,
// hence two waves per SIMD. Workgroups of consecutive blocks go to one XCD, whose L2 then serves the shared
// columns. With few blocks the individuals are split over several workgroups (integer atomics, so the sums
// are the same in any order) and gram_finish_kernel forms the entries.
#pragma once

#include "gram_plan.hpp"
#include "sweep_kernel.hpp"

namespace brr {

constexpr int kGramThreads = 512;
constexpr int kGramCols = 2 * kMaxB;              // entries per row: the block's slots, then the next block's
constexpr uint32_t kGramChunkBytes = kGramChunk / 4;
constexpr uint32_t kGramStride = kGramChunkBytes + 16;   // LDS bytes per column: rows start in shifted banks

constexpr int kGramBases = 3;
// Bytes per 2-bit code of the sparse columns' bases: 0 -> dosage 2, 1 missing, 2 -> 1, 3 -> 0.
constexpr uint32_t kDosageTab = 0x00010002u;
constexpr uint32_t kMissingTab = 0x00000100u;

// A marker's share in its row and column entries: value of code v = a + sum_b c[b] (byte v of tab[b]).
struct GramMarker {
    double a, c[kGramBases];        // sparse: mean; 1 / sd, the others unused
    double s[kGramBases];           // sums of the bytes over the individuals
    uint32_t tab[kGramBases];
    int n;                          // bases in use
};

struct GramParams {
    uint32_t N, M, B, iterations;
    int layout;
    uint32_t splits;                // workgroups per block (1: the entries are formed here)
    const uint32_t* codes;          // 2-bit columns, column j at codes + j * col_words
    uint64_t col_words;
    const GramMarker* markers;      // M
    int bases;                      // most bases of a marker of the context
    const uint32_t* order;          // iterations x M
    double* gram;                   // (iterations x M) rows of kGramCols
    int32_t* acc;                   // splits > 1: products x (iterations x M) x kGramCols, zero between launches
    const uint32_t* gate;           // null, or a word that must be 0 for the launch to run
};

// The bases of a dense column from its table (by dosage 0, 1, 2, missing) and counts per code. Codes that do not occur
// have no value: whatever the table holds for them stays out of the sums. Steps count as equal up to the roundings of
// (dosage - mean) / sd, at most 2^-50 of the largest value.
__device__ __forceinline__ void dense_bases(const double* lt, const uint32_t* cnt, GramMarker& g)
{
    const double v[4] = {lt[2], lt[3], lt[1], lt[0]};
    // low, middle and high code of three values at equal steps: a builder's table first
    constexpr uint32_t kTriple[12] = {0x320, 0x312, 0x310, 0x321, 0x301, 0x302, 0x230, 0x231, 0x132, 0x130, 0x031, 0x012};
    g.n = 0;
    uint32_t left = 0u;             // codes that still need a value
#pragma unroll
    for (int c = 0; c < 4; ++c) left |= cnt[c] ? 1u << c : 0u;
    if (!(left & 2u) && left != 13u) {
        // at most two dosages: the dosage as base, whatever its third value would be
        const double step = left == 5u ? v[0] - v[2] : left == 9u ? 0.5 * (v[0] - v[3]) : left == 12u ? v[2] - v[3] : 0.0;
        g.a = left == 5u ? v[2] - step : left & 8u ? v[3] : left & 4u ? v[2] : v[0];
        g.c[0] = step;
        g.tab[0] = kDosageTab;
        g.n = 1;
        return;
    }
    auto value = [&](uint32_t c) { return c == 0u ? v[0] : c == 1u ? v[1] : c == 2u ? v[2] : v[3]; };
    auto add = [&](double c, uint32_t tab) {
#pragma unroll
        for (int b = 0; b < kGramBases; ++b) {
            g.c[b] = g.n == b ? c : g.c[b];
            g.tab[b] = g.n == b ? tab : g.tab[b];
        }
        ++g.n;
    };
    bool steps = false;
    for (int t = 0; t < 12 && !steps; ++t) {
        const uint32_t lo = kTriple[t] >> 8, mid = (kTriple[t] >> 4) & 3u, hi = kTriple[t] & 3u;
        const uint32_t three = 1u << lo | 1u << mid | 1u << hi;
        if ((left & three) != three) continue;
        const double x = value(lo), y = value(mid), z = value(hi);
        if (!(fabs(2.0 * y - x - z) <= 1.7763568394002505e-15 * fmax(fabs(x), fmax(fabs(y), fabs(z))))) continue;   // 2^-49
        g.a = x;
        add(0.5 * (z - x), 1u << (8u * mid) | 2u << (8u * hi));
        left &= ~three;
        steps = true;
    }
    if (!steps) {
        const uint32_t base = left & 8u ? 3u : (uint32_t)__builtin_ctz(left | 8u);
        g.a = value(base);
        left &= ~(1u << base);
    }
#pragma unroll
    for (int c = 0; c < 4; ++c)
        if (((left >> c) & 1u) && v[c] != g.a) add(v[c] - g.a, 1u << (8 * c));
    if (g.n == 0) g.n = 1;          // (one value throughout)
}

// Every marker's GramMarker, and in *kind (0 before) the largest of 2 n, or 2 n + 1 where a marker's n = 1 base is not the
// dosage.
static __global__ void __launch_bounds__(256)
gram_markers_kernel(uint32_t M, int layout, const double* lut, const double* stats, const uint32_t* counts, GramMarker* out,
                    uint32_t* kind)
{
    const uint32_t j = blockIdx.x * 256u + threadIdx.x;
    if (j >= M) return;
    GramMarker g;
    const uint32_t* cnt = counts + 4 * (size_t)j;
#pragma unroll
    for (int b = 0; b < kGramBases; ++b) {
        g.c[b] = 0.0;
        g.tab[b] = 0u;
    }
    if (layout == kLayoutDense) {
        dense_bases(lut + 4 * (size_t)j, cnt, g);
    } else {
        const double* st = stats + 4 * (size_t)j;
        g.a = st[0];
        g.c[0] = 1.0 / st[1];
        g.tab[0] = kDosageTab;
        g.tab[1] = kMissingTab;
        g.n = cnt[1] ? 2 : 1;
    }
#pragma unroll
    for (int b = 0; b < kGramBases; ++b) {
        g.s[b] = 0.0;
#pragma unroll
        for (int v = 0; v < 4; ++v) g.s[b] += (double)cnt[v] * (double)((g.tab[b] >> (8 * v)) & 255u);
    }
    out[j] = g;
    const uint32_t k = 2u * (uint32_t)g.n + (g.n == 1 && g.tab[0] != kDosageTab ? 1u : 0u);
    if (*(volatile uint32_t*)kind < k) atomicMax(kind, k);
}

// The entry's part that does not depend on the products, and the factor of the product of h's base i and k's base j.
__device__ __forceinline__ double gram_base(int layout, double N, const GramMarker& h, const GramMarker& k)
{
    if (layout == kLayoutDense)
        return N * h.a * k.a + h.a * (k.c[0] * k.s[0] + k.c[1] * k.s[1] + k.c[2] * k.s[2]) +
               k.a * (h.c[0] * h.s[0] + h.c[1] * h.s[1] + h.c[2] * h.s[2]);
    if (layout == kLayoutEigen) return -h.a * (k.s[0] + k.a * k.s[1]) * h.c[0];
    return -h.a * k.s[0] * h.c[0];
}
__device__ __forceinline__ double gram_factor(int layout, int i, int j, const GramMarker& h, const GramMarker& k)
{
    if (layout == kLayoutDense) {
        const double fh = i == 0 ? h.c[0] : i == 1 ? h.c[1] : h.c[2];
        const double fk = j == 0 ? k.c[0] : j == 1 ? k.c[1] : k.c[2];
        return fh * fk;
    }
    const double d = h.c[0];
    if (j == 0) return i == 0 ? d : h.a * d;
    return (i == 0 ? k.a : h.a * k.a) * d;   // EigenSparse
}
// Products of contexts whose markers have up to `bases` bases, product i + bases j from h's base i and k's base j: the
// ragged dot weight is the dosage alone.
__host__ __device__ constexpr int gram_weights(int layout, int bases) { return layout == kLayoutRagged ? 1 : bases; }
__host__ __device__ constexpr int gram_products(int layout, int bases) { return bases * gram_weights(layout, bases); }

typedef int int4v __attribute__((ext_vector_type(4)));
typedef int int16v __attribute__((ext_vector_type(16)));

// 16 codes of a word as 16 bytes through a 4-entry table (byte v of `tab` for code v): byte q of result j is
// individual 4 q + j. Both operands of a product use the same order, so the sum over individuals is the same.
__device__ __forceinline__ int4v gram_expand(uint32_t w, uint32_t tab)
{
    int4v r;
#pragma unroll
    for (int j = 0; j < 4; ++j)
        r[j] = (int)__builtin_amdgcn_perm(0u, tab, (w >> (2 * j)) & 0x03030303u);
    return r;
}

struct GramShared {
    union {
        alignas(16) uint8_t col[2][kGramCols][kGramStride];
        int32_t sum[kMaxB][kGramCols];
    };
    uint32_t id[kGramCols];
    GramMarker mk[kGramCols];
    uint32_t tab[kGramBases][kGramCols];   // the bases' bytes per code
    int bases;                             // most bases of the block's and the next block's markers
};

// Work item `item` (block of an iteration, times its split). kMany: some marker of the context has another base than the
// dosage, or more than that (then the blocks that hold one form the other products too). With the dosage alone all
// lanes expand through one constant table: 520 us for 626 blocks at N = 100,000, 530 through the markers' own.
template <bool kMany>
__device__ __forceinline__ void gram_body(const GramParams& p, GramShared& L, uint32_t item)
{
    if (p.gate && __hip_atomic_load(p.gate, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u) return;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t per = (p.M + p.B - 1) / p.B;            // blocks per iteration
    const uint32_t bi = item / p.splits, split = item % p.splits;
    const uint32_t it = bi / per, blk = bi % per;
    const uint32_t b0 = blk * p.B;
    const int nb = (int)min(p.B, p.M - b0);
    const int nn = b0 + p.B < p.M ? (int)min(p.B, p.M - b0 - p.B) : 0;
    const uint32_t* order = p.order + (size_t)it * p.M;
    if (tid == 0) L.bases = 1;
    __syncthreads();
    if (tid < kGramCols) {
        const int k = tid & (kMaxB - 1);
        const bool next = tid >= kMaxB;
        const bool ok = k < (next ? nn : nb);
        L.id[tid] = 0xFFFFFFFFu;
        if (ok) {
            const uint32_t j = order[b0 + (next ? p.B : 0u) + (uint32_t)k];
            L.id[tid] = j;
            const GramMarker g = p.markers[j];
            L.mk[tid] = g;
            if constexpr (kMany) {
#pragma unroll
                for (int b = 0; b < kGramBases; ++b) L.tab[b][tid] = g.tab[b];
                if (g.n > 1) atomicMax(&L.bases, g.n);
            }
        } else if constexpr (kMany) {
#pragma unroll
            for (int b = 0; b < kGramBases; ++b) L.tab[b][tid] = 0u;
        }
    }
    __syncthreads();
    const uint32_t nchunk = (p.N + kGramChunk - 1) / kGramChunk;
    const uint32_t c0 = (uint32_t)((uint64_t)nchunk * split / p.splits);
    const uint32_t c1 = (uint32_t)((uint64_t)nchunk * (split + 1) / p.splits);
    const uint64_t colb = p.col_words * 4;
    const int nu = kMany ? min(L.bases, p.bases) : 1, nw = gram_weights(p.layout, nu);
    // individuals past the last one, staged as code 3, of which the sums know nothing
    const int32_t pads = (int32_t)(nchunk * kGramChunk - p.N);
    const size_t row0 = (size_t)it * p.M + b0;

    // 16-byte pieces of a chunk: thread tid takes pieces tid + 512 q: column (tid >> 4) + 32 q, part tid & 15
    const uint32_t part = (uint32_t)(tid & 15);
    uint4 pre[4];
    auto fetch = [&](uint32_t c) {
        const uint64_t off = (uint64_t)c * kGramChunkBytes + 16u * part;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint32_t j = L.id[(tid >> 4) + 32 * q];
            const bool ok = j != 0xFFFFFFFFu && off < colb;
            pre[q] = *(const uint4*)((const uint8_t*)p.codes + (ok ? (size_t)j * colb + off : 0));
            if (!ok) pre[q] = make_uint4(~0u, ~0u, ~0u, ~0u);
        }
    };
    // code 3 past the last individual
    auto stage = [&](uint32_t c, int buf) {
        const int64_t left = (int64_t)p.N - (int64_t)c * kGramChunk - 64 * (int64_t)part;   // individuals of this piece
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            uint32_t v[4] = {pre[q].x, pre[q].y, pre[q].z, pre[q].w};
            if (left < 64) {
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    const int64_t n = left - 16 * s;
                    if (n <= 0) v[s] = ~0u;
                    else if (n < 16) v[s] |= ~0u << (2 * (uint32_t)n);
                }
            }
            *(uint4*)&L.col[buf][(tid >> 4) + 32 * q][16 * part] = make_uint4(v[0], v[1], v[2], v[3]);
        }
    };

    for (int prod = 0; prod < nu * nw; ++prod) {
        const int bu = prod % nu, bw = prod / nu;
        uint32_t tw[4], tu[2];
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            tw[g] = kMany ? L.tab[bw][32 * g + (lane & 31)] : kDosageTab;
            if (g < 2) tu[g] = kMany ? L.tab[bu][32 * g + (lane & 31)] : kDosageTab;
        }
        int16v acc[7];
#pragma unroll
        for (int t = 0; t < 7; ++t)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[t][r] = 0;
        if (c0 < c1) {
            fetch(c0);
            stage(c0, 0);
            __syncthreads();
        }
        for (uint32_t c = c0; c < c1; ++c) {
            const int buf = (int)((c - c0) & 1u);
            if (c + 1 < c1) fetch(c + 1);
            uint4 w[4];
#pragma unroll
            for (int g = 0; g < 4; ++g)
                w[g] = *(const uint4*)&L.col[buf][32 * g + (lane & 31)][32 * wave + 16 * (lane >> 5)];
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                int4v fb[4], fa[2];
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const uint32_t x = s == 0 ? w[g].x : s == 1 ? w[g].y : s == 2 ? w[g].z : w[g].w;
                    fb[g] = gram_expand(x, tw[g]);
                    if (g < 2) fa[g] = kMany ? gram_expand(x, tu[g]) : fb[g];
                }
                acc[0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[0], fb[0], acc[0], 0, 0, 0);
                acc[1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[0], fb[1], acc[1], 0, 0, 0);
                acc[2] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[1], fb[1], acc[2], 0, 0, 0);
                acc[3] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[0], fb[2], acc[3], 0, 0, 0);
                acc[4] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[0], fb[3], acc[4], 0, 0, 0);
                acc[5] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[1], fb[2], acc[5], 0, 0, 0);
                acc[6] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[1], fb[3], acc[6], 0, 0, 0);
            }
            if (c + 1 < c1) stage(c + 1, buf ^ 1);
            __syncthreads();
        }
        // the waves' sums over their individuals, then the entries (or the shared counts)
        for (int t = tid; t < kMaxB * kGramCols; t += kGramThreads) (&L.sum[0][0])[t] = 0;
        __syncthreads();
        constexpr int kRow[7] = {0, 0, 1, 0, 0, 1, 1}, kCol[7] = {0, 1, 1, 2, 3, 2, 3};
#pragma unroll
        for (int t = 0; t < 7; ++t)
#pragma unroll
            for (int r = 0; r < 16; ++r)
                atomicAdd(&L.sum[32 * kRow[t] + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3)][32 * kCol[t] + (lane & 31)],
                          acc[t][r]);
        __syncthreads();
        for (int t = tid; t < kMaxB * kGramCols; t += kGramThreads) {
            const int h = t / kGramCols, k = t % kGramCols;
            const bool need = h < nb && (k < kMaxB ? (k > h && k < nb) : k - kMaxB < nn);
            if (!need) continue;
            const size_t at = (row0 + (size_t)h) * kGramCols + (size_t)k;
            int32_t s = L.sum[h][k];
            if (kMany && c1 == nchunk) s -= pads * (int32_t)(L.tab[bu][h] >> 24) * (int32_t)(L.tab[bw][k] >> 24);
            if (p.splits > 1) {
                atomicAdd(p.acc + (size_t)(bu + p.bases * bw) * p.iterations * p.M * kGramCols + at, s);
            } else {
                const GramMarker& mh = L.mk[h];
                const GramMarker& mk = L.mk[k];
                const double prev = prod == 0 ? gram_base(p.layout, (double)p.N, mh, mk) : p.gram[at];
                p.gram[at] = prev + gram_factor(p.layout, bu, bw, mh, mk) * (double)s;
            }
        }
        __syncthreads();
    }
}

// Consecutive work items on one XCD (workgroups go round robin over the 8 XCDs).
__device__ __forceinline__ uint32_t gram_item()
{
    const uint32_t n8 = gridDim.x / 8, r8 = gridDim.x % 8, x8 = blockIdx.x % 8;
    return x8 * n8 + min(x8, r8) + blockIdx.x / 8;
}

template <bool kMany>
__global__ void __launch_bounds__(kGramThreads)
gram_kernel(GramParams p)
{
    __shared__ GramShared L;
    gram_body<kMany>(p, L, gram_item());
}

// The blocks of several contexts (cohorts) in one launch: item i belongs to the last entry with first <= i.
struct GramEntry {
    GramParams p;
    uint32_t first;
};

template <bool kMany>
__global__ void __launch_bounds__(kGramThreads)
gram_cohort_kernel(const GramEntry* tab, uint32_t n)
{
    __shared__ GramShared L;
    const uint32_t item = gram_item();
    uint32_t c = 0;
    while (c + 1 < n && item >= tab[c + 1].first) ++c;
    const GramParams p = tab[c].p;
    gram_body<kMany>(p, L, item - tab[c].first);
}

// splits > 1: the entries from the shared counts, which are left zero. One workgroup per row.
static __global__ void __launch_bounds__(kGramCols)
gram_finish_kernel(GramParams p)
{
    if (p.gate && __hip_atomic_load(p.gate, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u) return;
    const uint32_t it = blockIdx.x / p.M, pos = blockIdx.x % p.M;
    const uint32_t b0 = pos / p.B * p.B;
    const int nb = (int)min(p.B, p.M - b0);
    const int nn = b0 + p.B < p.M ? (int)min(p.B, p.M - b0 - p.B) : 0;
    const int h = (int)(pos - b0), k = (int)threadIdx.x;
    if (!(k < kMaxB ? (k > h && k < nb) : k - kMaxB < nn)) return;
    const uint32_t* order = p.order + (size_t)it * p.M;
    const GramMarker& mh = p.markers[order[pos]];
    const GramMarker& mk = p.markers[order[k < kMaxB ? b0 + (uint32_t)k : b0 + p.B + (uint32_t)(k - kMaxB)]];
    const size_t at = (size_t)blockIdx.x * kGramCols + (size_t)k;
    double g = gram_base(p.layout, (double)p.N, mh, mk);
    for (int prod = 0; prod < gram_products(p.layout, p.bases); ++prod) {
        int32_t* s = p.acc + (size_t)prod * p.iterations * p.M * kGramCols + at;
        g += gram_factor(p.layout, prod % p.bases, prod / p.bases, mh, mk) * (double)*s;
        *s = 0;
    }
    p.gram[at] = g;
}

// Individuals per 2-bit value of each column (one workgroup per marker).
static __global__ void __launch_bounds__(256)
marker_counts_kernel(const uint32_t* codes, uint64_t col_words, uint32_t N, uint32_t* counts)
{
    __shared__ uint32_t red[3][4];
    const uint32_t* col = codes + (size_t)blockIdx.x * col_words;
    uint32_t c[3] = {0, 0, 0};
    for (uint32_t t = threadIdx.x; 16u * t < N; t += 256) {
        const uint32_t x = col[t], left = N - 16u * t;
        const uint32_t pm = left < 16u ? 0x55555555u & ((1u << (2u * left)) - 1u) : 0x55555555u;
        const uint32_t l = x & pm, h = (x >> 1) & pm;
        c[0] += (uint32_t)__builtin_popcount(pm & ~(l | h));
        c[1] += (uint32_t)__builtin_popcount(l & ~h);
        c[2] += (uint32_t)__builtin_popcount(h & ~l);
    }
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        for (int o = 32; o > 0; o >>= 1) c[q] += (uint32_t)__shfl_xor((int)c[q], o, 64);
        if ((threadIdx.x & 63) == 0) red[q][threadIdx.x >> 6] = c[q];
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t n[3];
        for (int q = 0; q < 3; ++q) n[q] = red[q][0] + red[q][1] + red[q][2] + red[q][3];
        uint32_t* o = counts + 4 * (size_t)blockIdx.x;
        o[0] = n[0];
        o[1] = n[1];
        o[2] = n[2];
        o[3] = N - n[0] - n[1] - n[2];
    }
}

} // namespace brr
