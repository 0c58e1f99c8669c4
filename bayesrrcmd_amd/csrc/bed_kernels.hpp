// bed_kernels.hpp -- a PLINK .bed payload decoded on the device.
//
// The reference turns every SNP column of the .bed file into a Marker on the
// host (preprocessgraph.cpp:24-60): the 2-bit decode, then DenseMarkerBuilder
// (densemarkerbuilder.cpp:23-60) or RaggedSparseMarkerBuilder with
// SparseMarker::updateStatistics (raggedsparsemarkerbuilder.cpp:25-55,
// sparsemarker.cpp:8-19). The device holds a column as its 2-bit codes, so the
// decode reduces to: repack each column to a 16-byte-aligned stride, count the
// four code values, and derive the per-marker table (dense) or statistics
// (ragged) from those counts and, for the dense table, from the column sums the
// builder forms in individual order.
//
// 2-bit values (LSB first): 0 = genotype 2, 1 = missing, 2 = genotype 1,
// 3 = genotype 0.
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>

namespace brr {

constexpr int kBedThreads = 256;

__device__ __forceinline__ uint32_t bed_wave_sum_u32(uint32_t v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += (uint32_t)__shfl_xor((int)v, o, 64);
    return v;
}

// One workgroup per marker j. src is the packed payload (column j at byte
// j * cb, cb = ceil(N/4)) read as words; the caller provides at least 20
// readable bytes past M * cb. Output column j is col_words words at
// codes + j * col_words: the column's cb bytes, then zeros. counts[4j + v] =
// number of individuals i < N whose value is v (pad bits ignored). When stats is
// not null, stats[4j..4j+3] = {mean, sd, sqrdZ, Zsum} of SparseMarker and the
// first marker without genotype 1 or 2 calls lowers *bad. eigen = 1: the
// EigenSparse statistics instead (missing calls imputed at the mean,
// eigensparsemarkerbuilder.cpp:41-59), and only a marker without any nonzero
// call (eigensparsemarker.cpp:60-71) lowers *bad.
static __global__ void __launch_bounds__(kBedThreads)
bed_unpack_kernel(const uint32_t* __restrict__ src, uint64_t cb, uint32_t N, uint64_t col_words,
                  uint32_t* __restrict__ codes, uint32_t* __restrict__ counts, double* __restrict__ stats,
                  uint32_t* __restrict__ bad, int eigen)
{
    __shared__ uint32_t red[3][kBedThreads / 64];
    const uint32_t j = blockIdx.x;
    const int tid = threadIdx.x;
    const uint64_t base = (uint64_t)j * cb;
    uint4* dst = reinterpret_cast<uint4*>(codes + (size_t)j * col_words);
    const uint32_t nvec = (uint32_t)(col_words / 4u);
    uint32_t c0 = 0, c1 = 0, c2 = 0;
    for (uint32_t t = (uint32_t)tid; t < nvec; t += kBedThreads) {
        const uint64_t s = base + 16ull * t;                 // first payload byte of this 16-byte chunk
        const uint32_t* wp = src + (s >> 2);
        const uint32_t sh = 8u * (uint32_t)(s & 3u);
        uint32_t w[5];
#pragma unroll
        for (int k = 0; k < 5; ++k) w[k] = wp[k];
        uint32_t out[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            uint32_t x = (uint32_t)((((uint64_t)w[k + 1] << 32) | (uint64_t)w[k]) >> sh);
            const int64_t inside = (int64_t)cb - (int64_t)(16ull * t + 4u * (uint32_t)k);   // bytes of x in the column
            if (inside <= 0) x = 0u;
            else if (inside < 4) x &= (1u << (8 * (uint32_t)inside)) - 1u;
            out[k] = x;
            const int64_t npos = (int64_t)N - (int64_t)(64ull * t + 16u * (uint32_t)k);    // individuals < N in x
            uint32_t pm = 0x55555555u;
            if (npos <= 0) pm = 0u;
            else if (npos < 16) pm &= (1u << (2 * (uint32_t)npos)) - 1u;
            const uint32_t lo = x & pm, hi = (x >> 1) & pm;
            c0 += (uint32_t)__builtin_popcount(pm & ~(lo | hi));
            c1 += (uint32_t)__builtin_popcount(lo & ~hi);
            c2 += (uint32_t)__builtin_popcount(hi & ~lo);
        }
        dst[t] = make_uint4(out[0], out[1], out[2], out[3]);
    }
    c0 = bed_wave_sum_u32(c0);
    c1 = bed_wave_sum_u32(c1);
    c2 = bed_wave_sum_u32(c2);
    if ((tid & 63) == 0) { red[0][tid >> 6] = c0; red[1][tid >> 6] = c1; red[2][tid >> 6] = c2; }
    __syncthreads();
    if (tid == 0) {
        uint32_t n[3];
#pragma unroll
        for (int q = 0; q < 3; ++q) n[q] = red[q][0] + red[q][1] + red[q][2] + red[q][3];
        counts[4 * (size_t)j + 0] = n[0];
        counts[4 * (size_t)j + 1] = n[1];
        counts[4 * (size_t)j + 2] = n[2];
        counts[4 * (size_t)j + 3] = N - n[0] - n[1] - n[2];
        if (stats) {
            // SparseMarker::updateStatistics sums the values 1 and 2 in
            // individual order; the sums are integers, so the counts give them
            // exactly. The rest is the same expression in the same order.
            const uint64_t ones = n[2], twos = n[0], nm = n[1];
            const double numInds = (double)N;
            double Zsum = (double)(ones + 2u * twos);
            double sqrdZ = (double)(ones + 4u * twos);
            const double mean = Zsum / numInds;
            if (eigen) {
                sqrdZ += (mean * mean) * (double)nm;
                Zsum += mean * (double)nm;
            }
            const double sd = sqrt((sqrdZ - 2.0 * mean * Zsum + numInds * mean * mean) / (numInds - 1.0));
            double* st = stats + 4 * (size_t)j;
            st[0] = mean;
            st[1] = sd;
            st[2] = sqrdZ;
            st[3] = Zsum;
            if (ones == 0 && twos == 0 && (!eigen || nm == 0)) atomicMin(bad, j);
        }
    }
}

// The running FP64 sum of tab(v) over the values v of one column's individuals
// 0..N-1, added one at a time in individual order. tab(v) = tabl[v * kBedThreads]:
// the calling thread's entries in LDS, one plane per value so that the lanes of
// a wave read distinct banks whatever their values.
__device__ __forceinline__ double bed_ordered_sum_lane(const uint4* col, uint32_t N, const double* tabl)
{
    double acc = 0.0;
    const uint32_t nfull = N / 64u;
    uint4 next = nfull ? col[0] : make_uint4(0u, 0u, 0u, 0u);
    for (uint32_t q = 0; q < nfull; ++q) {
        const uint4 w = next;
        if (q + 1u < nfull) next = col[q + 1u];
        const uint32_t xs[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
        for (int k = 0; k < 4; ++k)
#pragma unroll
            for (uint32_t e = 0; e < 16u; ++e) acc = acc + tabl[((xs[k] >> (2u * e)) & 3u) * kBedThreads];
    }
    uint32_t rest = N - 64u * nfull;
    if (rest) {
        const uint4 w = col[nfull];
        const uint32_t xs[4] = {w.x, w.y, w.z, w.w};
        for (int k = 0; k < 4 && rest; ++k) {
            const uint32_t n = rest < 16u ? rest : 16u;
            for (uint32_t e = 0; e < n; ++e) acc = acc + tabl[((xs[k] >> (2u * e)) & 3u) * kBedThreads];
            rest -= n;
        }
    }
    return acc;
}

// The running FP64 sum of x[v] >= 0 over the values v of one column's individuals 0..N-1, added one at a time in
// individual order, by one wave; n[v] > 0 tells which values occur. While the sum stays in one binade it is a multiple
// of that binade's unit and each addition adds x[v] rounded to the unit, whatever came before: the sum over a
// stretch is an exact combination of the counts. Only a value half a unit off looks at the last bit (it rounds to
// even, so the bit is 0 after it); the lanes then follow that bit through their individuals for both its values.
// Lane l counts the values of 64 individuals, a scan over the lanes finds the first 64 that leave the binade, and
// only those are added one by one: about a dozen times a column.
__device__ __forceinline__ double bed_ordered_sum(const uint4* col, uint32_t N, const double (&x)[4],
                                                  const uint32_t (&n)[4], int lane)
{
    const uint32_t chunks = (N + 63u) / 64u;
    // (scalar registers: the one-by-one additions then choose their value beside the vector unit)
    const double x0 = lane_read(x[0], 0), x1 = lane_read(x[1], 0), x2 = lane_read(x[2], 0), x3 = lane_read(x[3], 0);
    double acc = 0.0;
    for (uint32_t c0 = 0; c0 < chunks; c0 += 64u) {
        const uint32_t at = c0 + (uint32_t)lane;
        const uint32_t valid = at < chunks ? min(64u, N - 64u * at) : 0u;
        uint32_t w[4] = {0u, 0u, 0u, 0u};
        if (valid) {
            const uint4 q = col[at];
            w[0] = q.x; w[1] = q.y; w[2] = q.z; w[3] = q.w;
        }
        uint32_t n1 = 0, n2 = 0, n3 = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const uint32_t here = valid > 16u * (uint32_t)k ? min(16u, valid - 16u * (uint32_t)k) : 0u;
            const uint32_t m = here == 16u ? 0x55555555u : ((1u << (2u * here)) - 1u) & 0x55555555u;
            const uint32_t lo = w[k] & m, hi = (w[k] >> 1) & m;
            n3 += (uint32_t)__popc(lo & hi);
            n2 += (uint32_t)__popc(hi & ~lo);
            n1 += (uint32_t)__popc(lo & ~hi);
        }
        const uint32_t cnt[4] = {valid - n1 - n2 - n3, n1, n2, n3};
        int start = 0;
        while (start < 64) {
            // the unit's rounding of each value, r (a tie's: downwards), if the sum is far enough from zero; without
            // it (no binade yet, a value above it, not a number) a stretch ends at the first nonzero value
            const uint32_t ex = (uint32_t)(__double_as_longlong(acc) >> 52) & 0x7FFu;
            bool fixed = ex >= 64u && ex < 0x7C0u;
            const double bottom = __longlong_as_double((long long)(fixed ? ex : 1023u) << 52);
            const double unit = bottom * 2.220446049250313e-16, units = 4503599627370496.0 / bottom;   // 2^-52, 2^52
            double add = 0.0;
            bool any = false;
            uint32_t odd = 0, tie = 0;   // values whose r is an odd number of units; that are half a unit off
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const double xv = v == 0 ? x0 : v == 1 ? x1 : v == 2 ? x2 : x3;
                double r = (bottom + xv) - bottom;
                if (n[v]) {
                    if (!(xv < bottom)) fixed = false;
                    else if (fabs(xv - r) == 0.5 * unit) {
                        tie |= 1u << v;
                        r = xv - 0.5 * unit;
                    }
                    if (fixed) odd |= ((uint32_t)(uint64_t)(r * units) & 1u) << v;
                }
                if (cnt[v]) {
                    add += (double)cnt[v] * r;
                    any = any || xv != 0.0;
                }
            }
            if (lane < start) { add = 0.0; any = false; }
            double incl = add;
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) {
                const double y = __shfl_up(incl, off, 64);
                if (lane >= off) incl += y;
            }
            if (fixed && tie) {
                // ups of the ties and the last bit afterwards, by the bit before: up0 | up1 << 13 | bit0 << 26 |
                // bit1 << 27, composed over the lanes
                uint32_t b0 = 0, b1 = 1, up0 = 0, up1 = 0;
                if (lane >= start)
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const uint32_t here = valid > 16u * (uint32_t)k ? min(16u, valid - 16u * (uint32_t)k) : 0u;
                        for (uint32_t e = 0; e < here; ++e) {
                            const uint32_t v = (w[k] >> (2u * e)) & 3u;
                            b0 ^= (odd >> v) & 1u;
                            b1 ^= (odd >> v) & 1u;
                            if ((tie >> v) & 1u) {
                                up0 += b0;
                                up1 += b1;
                                b0 = b1 = 0;
                            }
                        }
                    }
                uint32_t map = up0 | up1 << 13 | b0 << 26 | b1 << 27;
#pragma unroll
                for (int off = 1; off < 64; off <<= 1) {
                    const uint32_t p = (uint32_t)__shfl_up((int)map, off, 64);
                    if (lane >= off) {
                        const uint32_t q0 = (p >> 26) & 1u, q1 = (p >> 27) & 1u;
                        const uint32_t m0 = map & 0x1FFFu, m1 = (map >> 13) & 0x1FFFu, o0 = (map >> 26) & 1u, o1 = (map >> 27) & 1u;
                        map = ((p & 0x1FFFu) + (q0 ? m1 : m0)) | (((p >> 13) & 0x1FFFu) + (q1 ? m1 : m0)) << 13 |
                              (q0 ? o1 : o0) << 26 | (q1 ? o1 : o0) << 27;
                    }
                }
                const bool last = (uint32_t)(uint64_t)(acc * units) & 1u;
                incl += (double)(last ? (map >> 13) & 0x1FFFu : map & 0x1FFFu) * unit;
            }
            const unsigned long long leave = __ballot(fixed ? !(acc + incl < 2.0 * bottom) : any);
            const int f = leave ? (int)__ffsll((long long)leave) - 1 : 64;
            if (fixed && f > start) acc = acc + lane_read(incl, f - 1);
            if (f < 64) {
                const uint32_t left = (uint32_t)lane_read((int)valid, f);
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const uint32_t word = (uint32_t)lane_read((int)w[k], f);
                    const uint32_t here = left > 16u * (uint32_t)k ? min(16u, left - 16u * (uint32_t)k) : 0u;
                    for (uint32_t e = 0; e < here; ++e) {
                        const uint32_t v = (word >> (2u * e)) & 3u;
                        acc = acc + (v < 2u ? (v == 0u ? x0 : x1) : (v == 2u ? x2 : x3));
                    }
                }
            }
            start = f + 1;
        }
    }
    return acc;
}

// DenseMarkerBuilder::endColumn from the counts and the codes: one wave per
// marker (kWave) or one lane. The table holds the standardised value of dosage 0, 1, 2 and of a
// missing call. The mean of the non-missing dosages and, without missing calls,
// the column mean are integer sums (exact from the counts); with missing calls
// the column sum, and always the squared norm, are summed in individual order.
template <bool kWave>
static __global__ void __launch_bounds__(kBedThreads)
bed_dense_table_kernel(const uint32_t* __restrict__ codes, uint64_t col_words, uint32_t N, uint32_t M,
                       const uint32_t* __restrict__ counts, double* __restrict__ lut)
{
    __shared__ double tab[kWave ? 1 : 4 * kBedThreads];   // a lane's entries, value v at [v * kBedThreads]
    const int lane = (int)(threadIdx.x & 63u);
    const uint32_t j = kWave ? blockIdx.x * (kBedThreads / 64u) +
                                   (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6))
                             : blockIdx.x * kBedThreads + threadIdx.x;
    if (j >= M) return;
    const uint4* col = reinterpret_cast<const uint4*>(codes + (size_t)j * col_words);
    const uint32_t n2 = counts[4 * (size_t)j + 0];   // value 0: dosage 2
    const uint32_t nm = counts[4 * (size_t)j + 1];   // value 1: missing
    const uint32_t n1 = counts[4 * (size_t)j + 2];   // value 2: dosage 1
    auto ordered_sum = [&](double x0, double x1, double x2, double x3) {
        if constexpr (kWave) {
            const double x[4] = {x0, x1, x2, x3};
            const uint32_t n[4] = {n2, nm, n1, N - n2 - nm - n1};
            return bed_ordered_sum(col, N, x, n, lane);
        } else {
            double* t = tab + threadIdx.x;
            t[0 * kBedThreads] = x0;
            t[1 * kBedThreads] = x1;
            t[2 * kBedThreads] = x2;
            t[3 * kBedThreads] = x3;
            return bed_ordered_sum_lane(col, N, t);
        }
    };
    const double numInds = (double)N;
    const double sum = (double)((uint64_t)n1 + 2u * (uint64_t)n2);
    const double mean = sum / (numInds - (double)nm);
    double s = sum;                                   // integer terms: the index-order sum is exact
    if (nm) s = ordered_sum(2.0, mean, 1.0, 0.0);
    const double cmean = s / numInds;
    const double d0 = 0.0 - cmean, d1 = 1.0 - cmean, d2 = 2.0 - cmean, dm = mean - cmean;
    const double sqn = ordered_sum(d2 * d2, dm * dm, d1 * d1, d0 * d0);
    const double sigma = 1.0 / (sqrt(sqn / (numInds - 1.0)));
    if (!kWave || lane == 0) {
        double* o = lut + 4 * (size_t)j;
        o[0] = d0 * sigma;
        o[1] = d1 * sigma;
        o[2] = d2 * sigma;
        o[3] = dm * sigma;
    }
}

// A wave per column against a lane per column. A lane takes 13 ns an individual whatever the number of columns (up to
// about 65,000, a wave per SIMD); waves take 27 us and, with the chip full, 8.5 ns + 0.16 ns per 1,000 individuals
// a column more. Measured, wave against lane: 8,000 columns of 100,000 individuals 0.24 / 1.3 ms, 40,000 0.98 / 1.34,
// 100,000 2.45 / 1.95; 8,000 of 3,000 0.105 / 0.044, 500 of 500 0.030 / 0.012.
inline bool bed_wave_sums(uint32_t N, uint32_t M)
{
    return 13.0 * N > 27000.0 + M * (8.5 + 1.6e-4 * N);
}

} // namespace brr
