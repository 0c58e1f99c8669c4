// gram_kernel.hpp -- the Gram entries between the markers of a sweep's blocks.
//
// The pipelined sweep (pipe_kernel.hpp) needs, for a marker h whose beta changes, how the dots of the later
// markers of h's block and of all markers of the next block change per unit of beta_old - beta_new:
//   G[h][k] = sum_i u_h(x_hi) w_k(x_ki),
// u_h the residual change per unit (densebayesrkernel.cpp:17-20, raggedbayesrkernel.cpp:10-30) and w_k the dot
// weight (sparsebayesrkernel.cpp:24-27, eigenbayesrkernel.cpp:10-20). They depend on the genotypes and on the
// marker order alone, so one kernel ahead of the sweep forms them for a whole iteration.
//
// With x the dosage (0 for a missing call) and m the missing-call indicator, u and w are linear in (1, x, m),
// so G follows in FP64 from per-marker sums and the integer products XX = sum x_h x_k, XM = sum x_h m_k,
// MX = sum m_h x_k, MM = sum m_h m_k, which the i8 matrix cores give exactly.
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

struct GramParams {
    uint32_t N, M, B, iterations;
    int layout;
    uint32_t splits;                // workgroups per block (1: the entries are formed here)
    const uint32_t* codes;          // 2-bit columns, column j at codes + j * col_words
    uint64_t col_words;
    const uint32_t* counts;         // M x 4: individuals per 2-bit value
    const double* lut;              // dense: M x 4 by dosage 0, 1, 2, missing
    const double* stats;            // ragged / EigenSparse: M x 4 {mean, sd, sqrdZ, Zsum}
    const uint32_t* order;          // iterations x M
    double* gram;                   // (iterations x M) rows of kGramCols
    int32_t* acc;                   // splits > 1: products x (iterations x M) x kGramCols, zero between launches
    const uint32_t* gate;           // null, or a word that must be 0 for the launch to run
};

// A marker's share in its row and column entries.
struct GramMarker {
    double x, m;       // sums of x and of the missing calls
    double a, d, e;    // dense: value = a + d x + e m; sparse: mean, 1 / sd, unused
};

__device__ __forceinline__ GramMarker gram_marker(const GramParams& p, uint32_t j)
{
    GramMarker g;
    const uint32_t* c = p.counts + 4 * (size_t)j;
    g.x = (double)c[2] + 2.0 * (double)c[0];
    g.m = (double)c[1];
    if (p.layout == kLayoutDense) {
        const double* lt = p.lut + 4 * (size_t)j;
        g.a = lt[0];
        g.d = 0.5 * (lt[2] - lt[0]);
        g.e = lt[3] - lt[0];
    } else {
        const double* st = p.stats + 4 * (size_t)j;
        g.a = st[0];
        g.d = 1.0 / st[1];
        g.e = 0.0;
    }
    return g;
}

// The entry's part that does not depend on the products, and each product's factor (0 XX, 1 MX, 2 XM, 3 MM).
__device__ __forceinline__ double gram_base(int layout, double N, const GramMarker& h, const GramMarker& k)
{
    if (layout == kLayoutDense)
        return N * h.a * k.a + h.a * (k.d * k.x + k.e * k.m) + k.a * (h.d * h.x + h.e * h.m);
    if (layout == kLayoutEigen) return -h.a * (k.x + k.a * k.m) * h.d;
    return -h.a * k.x * h.d;
}
__device__ __forceinline__ double gram_factor(int layout, int prod, const GramMarker& h, const GramMarker& k)
{
    if (layout == kLayoutDense) {
        const double fh = (prod & 1) ? h.e : h.d, fk = (prod & 2) ? k.e : k.d;
        return fh * fk;
    }
    if (prod == 0) return h.d;
    if (prod == 1) return h.a * h.d;
    return (prod == 2 ? k.a : h.a * k.a) * h.d;   // EigenSparse
}
// Products a layout needs when calls are missing.
__host__ __device__ constexpr int gram_products(int layout) { return layout == kLayoutRagged ? 2 : 4; }

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
    int any_miss;
};

// Work item `item` (block of an iteration, times its split). kMiss: some call of the context is missing (then the
// blocks that hold one form the other products too).
template <bool kMiss>
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
    if (tid == 0) L.any_miss = 0;
    __syncthreads();
    if (tid < kGramCols) {
        const int k = tid & (kMaxB - 1);
        const bool next = tid >= kMaxB;
        const bool ok = k < (next ? nn : nb);
        L.id[tid] = 0xFFFFFFFFu;
        if (ok) {
            const uint32_t j = order[b0 + (next ? p.B : 0u) + (uint32_t)k];
            L.id[tid] = j;
            L.mk[tid] = gram_marker(p, j);
            if (L.mk[tid].m != 0.0) L.any_miss = 1;
        } else {
            L.mk[tid] = GramMarker{0.0, 0.0, 0.0, 0.0, 0.0};
        }
    }
    __syncthreads();
    const uint32_t nchunk = (p.N + kGramChunk - 1) / kGramChunk;
    const uint32_t c0 = (uint32_t)((uint64_t)nchunk * split / p.splits);
    const uint32_t c1 = (uint32_t)((uint64_t)nchunk * (split + 1) / p.splits);
    const uint64_t colb = p.col_words * 4;
    const int nprod = (kMiss && L.any_miss) ? gram_products(p.layout) : 1;
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
    // code 3 (dosage 0, not missing) past the last individual
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

    constexpr uint32_t kDosage = 0x00010002u;   // byte per code: 0 -> 2, 1 (missing) -> 0, 2 -> 1, 3 -> 0
    constexpr uint32_t kMissing = 0x00000100u;
    for (int prod = 0; prod < nprod; ++prod) {
        const uint32_t ta = (prod & 1) ? kMissing : kDosage, tb = (prod & 2) ? kMissing : kDosage;
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
                    fb[g] = gram_expand(x, tb);
                    if (g < 2) fa[g] = kMiss ? gram_expand(x, ta) : fb[g];
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
            const int32_t s = L.sum[h][k];
            if (p.splits > 1) {
                atomicAdd(p.acc + (size_t)prod * p.iterations * p.M * kGramCols + at, s);
            } else {
                const GramMarker& mh = L.mk[h];
                const GramMarker& mk = L.mk[k];
                const double prev = prod == 0 ? gram_base(p.layout, (double)p.N, mh, mk) : p.gram[at];
                p.gram[at] = prev + gram_factor(p.layout, prod, mh, mk) * (double)s;
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

template <bool kMiss>
__global__ void __launch_bounds__(kGramThreads)
gram_kernel(GramParams p)
{
    __shared__ GramShared L;
    gram_body<kMiss>(p, L, gram_item());
}

// The blocks of several contexts (cohorts) in one launch: item i belongs to the last entry with first <= i.
struct GramEntry {
    GramParams p;
    uint32_t first;
};

template <bool kMiss>
__global__ void __launch_bounds__(kGramThreads)
gram_cohort_kernel(const GramEntry* tab, uint32_t n)
{
    __shared__ GramShared L;
    const uint32_t item = gram_item();
    uint32_t c = 0;
    while (c + 1 < n && item >= tab[c + 1].first) ++c;
    const GramParams p = tab[c].p;
    gram_body<kMiss>(p, L, item - tab[c].first);
}

// splits > 1: the entries from the shared counts, which are left zero. One workgroup per row.
static __global__ void __launch_bounds__(kGramCols)
gram_finish_kernel(GramParams p, int products)
{
    if (p.gate && __hip_atomic_load(p.gate, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u) return;
    const uint32_t it = blockIdx.x / p.M, pos = blockIdx.x % p.M;
    const uint32_t b0 = pos / p.B * p.B;
    const int nb = (int)min(p.B, p.M - b0);
    const int nn = b0 + p.B < p.M ? (int)min(p.B, p.M - b0 - p.B) : 0;
    const int h = (int)(pos - b0), k = (int)threadIdx.x;
    if (!(k < kMaxB ? (k > h && k < nb) : k - kMaxB < nn)) return;
    const uint32_t* order = p.order + (size_t)it * p.M;
    const GramMarker mh = gram_marker(p, order[pos]);
    const GramMarker mk = gram_marker(p, order[k < kMaxB ? b0 + (uint32_t)k : b0 + p.B + (uint32_t)(k - kMaxB)]);
    const size_t at = (size_t)blockIdx.x * kGramCols + (size_t)k;
    double g = gram_base(p.layout, (double)p.N, mh, mk);
    for (int prod = 0; prod < products; ++prod) {
        int32_t* s = p.acc + (size_t)prod * p.iterations * p.M * kGramCols + at;
        g += gram_factor(p.layout, prod, mh, mk) * (double)*s;
        *s = 0;
    }
    p.gram[at] = g;
}

// Individuals per 2-bit value of each column (one workgroup per marker), and whether any call is missing.
static __global__ void __launch_bounds__(256)
marker_counts_kernel(const uint32_t* codes, uint64_t col_words, uint32_t N, uint32_t* counts, uint32_t* any_miss)
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
        if (n[1]) *any_miss = 1u;
    }
}

} // namespace brr
