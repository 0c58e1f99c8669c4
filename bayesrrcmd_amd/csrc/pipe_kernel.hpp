// pipe_kernel.hpp -- the pipelined persistent kernel of the sequential BayesR sweep over 2-bit columns.
//
// What it computes is sweep_kernel.hpp's sequential sweep. How it differs: that kernel goes round a loop of
// dots, grid exchange, decisions and residual update once per block of 64 markers and once more for most beta
// changes, every step waiting for the one before (10.6 us a round, 3.4 of them in the exchange). Here the Gram
// entries between a block's markers and to the next block's (gram_kernel.hpp) turn a change into a correction
// of dots that are already known:
//   - a block is exchanged exactly once, whatever changes in it: after the change of slot h the later slots'
//     dots become dot_k + dBeta_h G[h][k] and they are decided again at once, on one wave, without the grid;
//   - the dots of block b + 1 are formed and exchanged from the residual before block b's changes while block
//     b is decided, and corrected the same way, so the exchange is off the critical path.
// A workgroup is twelve waves with one role each, in lockstep by one barrier per block (step b):
//   waves 0-7   apply block b - 1's changes to their copy of the residual slice, form and publish the partial
//               dots of 8 slots each of block b + 1;
//   wave 8      waits for block b's totals, corrects and decides them (lane = slot) change by change;
//   wave 9      reduces this workgroup's slots of block b + 1 and gathers its totals, as far as they arrive before
//               block b is decided;
//   wave 10     loads the columns of block b + 2 and the Gram rows of block b + 1's in-model slots into LDS and
//               draws block b + 1's u and z;
//   wave 11     constants and pair table of block b + 2, ids of block b + 3, outputs of block b - 1.
// Waves 8 to 11 have a higher wave priority than the dot waves: as the youngest of their SIMDs they were served last
// (a gather took 7.5 us while the dot waves had work, 1.5 us now). A step takes 3.9 us at N = 60,000 dense FP64
// (6.2 us with ten waves at one priority, scattered partials and spilled addresses), 4.3 us at 100,000 ragged FP32:
// apply and dots 2.4 us, their exchange 2.5 us beside the 1.3 us of block b's decisions.
// With at most 16 workgroups every workgroup sums all partials itself and the reduce hop is left out.
// Every workgroup decides from the same totals with the same instructions, so all hold the same bits.
#pragma once

#include "gram_kernel.hpp"

namespace brr {

constexpr int kDotWaves = 8;
constexpr int kDecWave = 8;
constexpr int kRedWave = 9;
constexpr int kLoadWave = 10;
constexpr int kMetaWave = 11;
constexpr int kDotThreads = 64 * kDotWaves;
constexpr int kPipeThreads = kDotThreads + 256;
constexpr int kSlotsPerWave = kMaxB / kDotWaves;
constexpr int kRing = 4;                 // blocks of columns and constants held at once
// Workgroups up to which the partials are summed without a reduce hop. An exchange of 64 slots alone takes 2.1 us at
// 16 workgroups so (2.4 with the hop) and 2.8 us at 24 (2.5 with it): each workgroup reads all partials.
constexpr uint32_t kDirectP = 16;

// Gram rows of a block kept in LDS: those of its first in-model slots; others are loaded when needed. As many
// as 160 KB hold beside the columns and, but for the ragged layout, the pair tables.
template <int R, int kLay>
constexpr int gram_rows()
{
    return kLay == kLayoutRagged ? (R == 1 ? 32 : 16) : (R == 1 ? 24 : 8);
}

// One wave's load from global memory straight into LDS, kBytes (4 or 16) per lane: lane l's bytes go to
// lds + kBytes l (lds is the same in every lane). No register waits for the data; the wave's vector-memory
// counter does.
template <int kBytes>
__device__ __forceinline__ void load_to_lds(const void* src, void* lds)
{
    static_assert(kBytes == 4 || kBytes == 16, "bytes per lane");
    const auto s = (__attribute__((address_space(1))) void*)const_cast<void*>(src);
    const auto d = (__attribute__((address_space(3))) void*)lds;
    if constexpr (kBytes == 4) __builtin_amdgcn_global_load_lds(s, d, 4, 0, 0);
    else __builtin_amdgcn_global_load_lds(s, d, 16, 0, 0);
}

// Waits until at most kLeft of the wave's vector-memory operations are outstanding (they end in order).
template <int kLeft>
__device__ __forceinline__ void wait_vm()
{
    static_assert(kLeft < 16, "the low four bits of the counter's field");
    __builtin_amdgcn_s_waitcnt(0x0F70 | kLeft);   // the other counters at their maxima: not waited for
}

struct PipeMeta {
    uint32_t mk[kMaxB];
    int32_t gr[kMaxB];
    double bo[kMaxB];          // beta before the block
    double w[kMaxB][4];        // dense: column value per 2-bit code; sparse: mean, sd, Zsum, 1 / sd
    double u[kMaxB];           // given u and z (sweep mode)
    double z[kMaxB];
};

template <int R, int kLay, bool kF32>
struct PipeShared {
    static constexpr int kTabs = kLay == kLayoutRagged ? 1 : kMaxB;   // the ragged column values are the same for all
    using E = typename std::conditional<kF32, float, double>::type;
    uint32_t codes[kRing][kMaxB][R][32];
    alignas(16) E pt[2][kTabs][16][2];         // column values by pairs of codes, by block parity
    alignas(16) double rows[2][gram_rows<R, kLay>()][kGramCols];
    PipeMeta meta[kRing];
    uint32_t ids[kRing][kMaxB];
    double du[2][kMaxB], dz[2][kMaxB];         // chain draws, by block parity
    double tots[2][kMaxB];                     // a block's totals gathered ahead, by parity
    // a block's decisions, by parity
    double ob[2][kMaxB], oa[2][kMaxB], on[2][kMaxB];
    int os[2][kMaxB];
    double cdl[2][kMaxB][4];                   // residual change per 2-bit code of each change in order
    int ck[2][kMaxB];                          // its slot
    int nchg[2];
    float fs[kF32 ? 2 : 1][kF32 ? R * kRun : 1];   // refreshed FP32 slice, by step parity
    double ed[kF32 ? R * kRun : 1];                // FP64 slice between iterations
    double mu, sigmaE, epsSum, tot;
    double sigmaG[kMaxG];
    double pi[kMaxG * kMaxK], v[kMaxG * kMaxK], betasqn[kMaxG];
    double cva[kMaxG * (kMaxK - 1)];
    double gc[kMaxG * kMaxK], grd[kMaxG * kMaxK], gbsd[kMaxG * kMaxK], gdg[kMaxG * kMaxK], ghk[kMaxG * kMaxK];
    double gamma[kMaxF];
    uint32_t forder[kMaxF];
    double sigmaF;
    int decided;                               // last block decided
    int got[2];                                // the block whose totals `tots` holds
    int abort;
};

// The parameter block in constant memory. The loops of the sweep read its fields through a pointer that the
// compiler may not see through from step to step: held in scalar registers throughout they spill to vector
// lanes, at 300 moves a step; read again they cost a cached scalar load.
typedef const __attribute__((address_space(4))) SweepParams* ConstParams;

// kParts: launches of a part of an iteration (SweepParams::part). A body of their own: the tests of those flags moved the
// whole one's registers about, 11% of a sweep at N = 100,000 with slices of 400 individuals.
template <int R, int kLay, bool kF32, bool kParts>
__device__ __forceinline__ void pipe_body(const SweepParams& p, ConstParams q, PipeShared<R, kLay, kF32>& L,
                                          const uint32_t w)
{
    using E = typename std::conditional<kF32, float, double>::type;
    constexpr bool dense = kLay == kLayoutDense;
    constexpr int kRows = gram_rows<R, kLay>();
    if (p.gate && __hip_atomic_load(p.gate, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u) return;
    const int tid = threadIdx.x;
    int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t lo = w * p.S;
    const uint32_t hi = min(lo + p.S, p.N);
    const uint32_t P = p.P, B = p.B, M = p.M;
    const int K = (int)p.K;
    const ScalarLayout SL{p.G, p.K};
    const double dN = (double)p.N;
    const bool direct = P <= kDirectP;
    const uint32_t copy = w % kCopies;

    // the residual slice: individual lo + 512 r + 8 lane + e in every dot wave; with an FP32 slice also its
    // FP64 original, spread over the dot waves (individual lo + 512 r + 64 wave + lane)
    E eps[R][8];
    double e64[kF32 ? R : 1];
#pragma unroll
    for (int r = 0; r < R; ++r) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const uint32_t i = lo + (uint32_t)r * kRun + 8u * (uint32_t)lane + (uint32_t)e;
            eps[r][e] = (i < hi) ? (E)p.eps[i] : (E)0;
        }
        if constexpr (kF32) {
            const uint32_t i = lo + (uint32_t)r * kRun + (uint32_t)(tid % kDotThreads);
            e64[r] = (i < hi) ? p.eps[i] : 0.0;
        }
    }

    // body(ed) on the FP64 slice ed[R][8], between iterations (all waves; waves 8 to 11 hold no current slice
    // and store nothing)
    auto fp64_region = [&](auto&& body) -> bool {
        if constexpr (!kF32) {
            return body(eps);
        } else {
            __syncthreads();
            if (wave < kDotWaves)
#pragma unroll
                for (int r = 0; r < R; ++r) L.ed[r * kRun + tid] = e64[r];
            __syncthreads();
            double ed[R][8];
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int e = 0; e < 8; ++e) ed[r][e] = L.ed[r * kRun + 8 * lane + e];
            const bool ok = body(ed);
            __syncthreads();
            if (wave == 0)
#pragma unroll
                for (int r = 0; r < R; ++r)
#pragma unroll
                    for (int e = 0; e < 8; ++e) L.ed[r * kRun + 8 * lane + e] = ed[r][e];
            __syncthreads();
#pragma unroll
            for (int r = 0; r < R; ++r) {
                if (wave < kDotWaves) e64[r] = L.ed[r * kRun + tid];
#pragma unroll
                for (int e = 0; e < 8; ++e) eps[r][e] = (float)ed[r][e];
            }
            return ok;
        }
    };

    if (tid == 0) {
        L.abort = 0;
        L.mu = p.scal[SL.mu()];
        L.sigmaE = p.scal[SL.sigmaE()];
        L.epsSum = p.scal[SL.epsSum()];
        L.sigmaF = p.F ? p.fixed[0] : 1.0;
        L.nchg[0] = L.nchg[1] = 0;
    }
    for (uint32_t t = tid; t < p.G; t += kPipeThreads) {
        L.sigmaG[t] = p.scal[SL.sigmaG() + t];
        L.betasqn[t] = kParts && (q->part & 1u) ? p.scal[SL.betasqn() + t] : 0.0;
    }
    for (uint32_t t = tid; t < p.G * p.K; t += kPipeThreads) {
        L.pi[t] = p.scal[SL.pi() + t];
        L.v[t] = kParts && (q->part & 1u) ? p.scal[SL.v() + t] : 0.0;
    }
    for (uint32_t t = tid; t < p.G * (p.K - 1); t += kPipeThreads) L.cva[t] = p.cva[t];
    for (uint32_t t = tid; t < p.F; t += kPipeThreads) {
        L.gamma[t] = p.fixed[1 + t];
        L.forder[t] = p.forder[t];
    }
    if constexpr (kLay == kLayoutRagged) {
        if (tid < 64) {   // genotype 2 counts 2, genotype 1 counts 1, missing calls and genotype 0 nothing
            const int n = (tid >> 1) & 15, code = (tid & 1) ? n >> 2 : n & 3;
            L.pt[tid >> 5][0][n][tid & 1] = (E)(code == 0 ? 2 : code == 2 ? 1 : 0);
        }
    }
    uint32_t rnd = __hip_atomic_load(p.ctl + kCtlRound, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    unsigned long long n_rounds = 0, n_changes = 0;
    // phase timers of workgroup 0: wave 0 (loads, dots, update, iteration scalars) and wave 8 (exchange, decisions)
    uint64_t tk[kPhases] = {0, 0, 0, 0, 0, 0};
    uint64_t t_last = __builtin_amdgcn_s_memrealtime();
    auto tick = [&](int slot) {
        if (w == 0) {
            const uint64_t now = __builtin_amdgcn_s_memrealtime();
            tk[slot] += now - t_last;
            t_last = now;
        }
    };
    __syncthreads();

    // Slot k's partial of workgroup w2 in round r. Rounds alternate between two buffers: a workgroup publishes round
    // r + 2 only after deciding round r, whose totals show that every partial of it has been read. Without the
    // reduce hop (direct) it only knows that they were written: a workgroup may publish round r + 3 while another
    // still reads round r, so four buffers take turns.
    // Laid out so that a publishing wave writes whole sectors and a reading wave reads them: direct, by workgroup;
    // else by groups of 2 slots (4 with less than 32 workgroups), which one workgroup reduces, and by workgroup
    // within the group.
    const uint32_t gl = direct ? 6u : P >= 32 ? 1u : 2u;   // log2 of the slots in a group
    auto part_slot = [&](uint32_t r, uint32_t k, uint32_t w2) {
        const uint32_t buf = direct ? r & 3u : (r & 1u) * ((uint32_t)kMaxB >> gl);
        return q->xchg1 + 2u * ((((size_t)(buf + (k >> gl)) * P + w2) << gl) + (k & ((1u << gl) - 1u)));
    };
    auto tot_slot = [&](uint32_t r, uint32_t k, uint32_t c) {
        return q->xchg2 + c * kCopyWords + (((size_t)(r & 1u) * kSlots + (size_t)k) * 2u);
    };
    // The sum of the lane's words at offsets at, at + step, .. (n of them, at most kN; cnt is the largest n of a
    // lane) once all carry tag r. A lane without words reads the one at `at` and does not wait. All loads are in
    // flight at once: their addresses come from one register, as each address kept and spilled for itself is a
    // wait for the loads before it. `leave()` ends the wait (for a round that is not needed yet).
    // 1: done, 0: left, -1: abort or timeout.
    auto wait_words = [&](auto kn, const uint64_t* base, uint32_t at, uint32_t step, uint32_t n, uint32_t cnt, uint32_t r,
                          auto&& leave, double* acc) -> int {
        constexpr uint32_t kN = decltype(kn)::value;
        const auto buf = xbuf(base);
        const uint32_t last = at + (n ? n - 1u : 0u) * step;
        u32x4 x[kN];
        for (uint64_t spins = 0;; ++spins) {
            uint32_t from = at;
            asm volatile("" : "+v"(from));   // opaque offset: every poll issues fresh loads
#pragma unroll
            for (uint32_t i = 0; i < kN; ++i)
                if (i < cnt) x[i] = __builtin_amdgcn_raw_buffer_load_b128(buf, min(from + i * step, last), 0, kCpolDevice);
            bool stale = false;
#pragma unroll
            for (uint32_t i = 0; i < kN; ++i)
                if (i < cnt) stale |= x[i].y != r || x[i].w != r;
            if (!__any(stale && n != 0u)) break;
            if (leave()) return 0;
            if (spins > kSpinLimit || ((spins & 255u) == 255u &&
                                       __hip_atomic_load(q->ctl + kCtlAbort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)))
                return -1;
        }
#pragma unroll
        for (uint32_t i = 0; i < kN; ++i)
            if (i < n) *acc += bits_as_double(((uint64_t)x[i].x << 32) | x[i].z);
        return 1;
    };
    // Wave 9 of the workgroups that own a group: its slots of [0, nb), reduced in a fixed order and published.
    auto reduce_round = [&](uint32_t r, int nb, auto&& leave) -> int {
        if (direct || (int)(w << gl) >= nb) return 1;
        const uint32_t k = (w << gl) + ((uint32_t)lane & ((1u << gl) - 1u));
        const uint32_t first = (uint32_t)lane >> gl, stride = 64u >> gl;
        constexpr uint32_t kN = 8;
        static_assert(kN * 32 >= kMaxP, "two slots over 64 lanes");
        double acc = 0.0;
        const int st = wait_words(std::integral_constant<uint32_t, kN>(), q->xchg1,
                                  (uint32_t)((const char*)part_slot(r, k, min(first, P - 1u)) - (const char*)q->xchg1),
                                  16u * 64u, (int)k < nb && first < P ? (P - first + stride - 1u) / stride : 0u,
                                  (P + stride - 1u) / stride, r, leave, &acc);
        if (st != 1) return st;
        acc += lane_xor<32>(acc, lane);
        acc += lane_xor<16>(acc, lane);
        acc += lane_xor<8>(acc, lane);
        acc += lane_xor<4>(acc, lane);
        if (gl == 1) acc += lane_xor<2>(acc, lane);
        if ((int)k < nb && first < (uint32_t)kCopies) publish_pair(q->xchg2, tot_slot(r, k, first), r, acc);
        return 1;
    };
    auto never = [] { return false; };
    // Slot k's total in lane k < nb.
    auto gather_round = [&](uint32_t r, int nb, double* out, auto&& leave) -> int {
        *out = 0.0;
        const bool act = lane < nb;
        if (!direct)
            return wait_words(std::integral_constant<uint32_t, 1>(), q->xchg2,
                              (uint32_t)((const char*)tot_slot(r, (uint32_t)lane, copy) - (const char*)q->xchg2), 0u,
                              act ? 1u : 0u, 1u, r, leave, out);
        int st = 1;
        for (uint32_t w0 = 0; st == 1 && w0 < P; w0 += 8) {
            const uint32_t n = min(P - w0, 8u);
            st = wait_words(std::integral_constant<uint32_t, 8>(), q->xchg1,
                            (uint32_t)((const char*)part_slot(r, (uint32_t)lane, w0) - (const char*)q->xchg1), 16u * kMaxB,
                            act ? n : 0u, n, r, leave, out);
        }
        return st;
    };
    // A scalar all-reduce of wave 0's slice sum (all threads call it).
    auto allreduce = [&](double part, double* total) -> bool {
        part = wave_sum_full(part, lane);
        ++rnd;
        ++n_rounds;
        if (tid == 0) publish_pair(q->xchg1, part_slot(rnd, 0, w), rnd, part);
        if (wave == kRedWave && reduce_round(rnd, 1, never) < 0 && lane == 0) { L.abort = 1; raise_abort(*q, 1); }
        if (wave == kDecWave) {
            double x;
            if (gather_round(rnd, 1, &x, never) < 0) {
                if (lane == 0) { L.abort = 1; raise_abort(*q, 2); }
            } else if (lane == 0) {
                L.tot = x;
            }
        }
        __syncthreads();
        *total = L.tot;
        const bool ok = L.abort == 0;
        __syncthreads();
        return ok;
    };

    if (p.mode == kModeProbe) {
        // exchange rounds of a full block with nothing else; no state is touched
        const int nb = (int)min(B, M);
        for (uint32_t q = 0; q < p.iterations; ++q) {
            ++rnd;
            ++n_rounds;
            if (wave < kDotWaves) {
                const int k = kSlotsPerWave * wave + (lane >> 3);
                if ((lane & 7) == 0 && k < nb) publish_pair(p.xchg1, part_slot(rnd, k, w), rnd, 0.0);
            } else if (wave == kDecWave) {
                double x;
                if (gather_round(rnd, nb, &x, never) < 0 && lane == 0) { L.abort = 1; raise_abort(p, 2); }
            } else if (wave == kRedWave && reduce_round(rnd, nb, never) < 0 && lane == 0) {
                L.abort = 1;
                raise_abort(p, 1);
            }
            __syncthreads();
            if (L.abort) return;
        }
        if (w == 0 && tid == 0) {
            __hip_atomic_store(p.ctl + kCtlRound, rnd, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            p.counters[0] += n_rounds;
        }
        return;
    }

    const uint32_t iters = (p.mode == kModeChain) ? p.iterations : 1u;
    const int nblocks = (int)((M + B - 1) / B);
    auto count = [&](int b) -> int { return b < 0 || b >= nblocks ? 0 : (int)min(B, M - (uint32_t)b * B); };
    for (uint32_t it = 0; it < iters; ++it) {
        const uint32_t iteration = p.iter_base + it;
        const uint32_t* order = p.order + (size_t)it * M;
        const double* gram = p.gram + (size_t)it * M * kGramCols;
        if (p.mode == kModeFixed) {
            if (!fp64_region([&](double (&ed)[R][8]) {
                    return fixed_effects<R>(p, L, ed, iteration, lo, hi, lane, allreduce);
                }))
                goto done;
            break;
        }
        if (p.mode == kModeChain && !(kParts && (q->part & 1u))) {
            // ---- updateMu (DenseBayesRRmz.cpp:36-42 / SparseBayesRRG.cpp:106-113)
            const double old_mu = L.mu;
            double new_mu = 0.0;
            const bool ok = fp64_region([&](double (&ed)[R][8]) {
                double part = 0.0;
#pragma unroll
                for (int r = 0; r < R; ++r)
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const uint32_t i = lo + (uint32_t)r * kRun + 8u * (uint32_t)lane + (uint32_t)e;
                        if (i < hi) ed[r][e] = ed[r][e] + old_mu;
                        part += ed[r][e];
                    }
                double total = L.epsSum + old_mu * dN;
                if (dense && !allreduce(part, &total)) return false;
                new_mu = norm_rng(p.seed, iteration, kDrawMu, p.chain, total / dN, L.sigmaE / dN);
#pragma unroll
                for (int r = 0; r < R; ++r)
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const uint32_t i = lo + (uint32_t)r * kRun + 8u * (uint32_t)lane + (uint32_t)e;
                        if (i < hi) ed[r][e] = ed[r][e] - new_mu;
                    }
                return true;
            });
            if (!ok) goto done;
            __syncthreads();
            if (tid == 0) {
                L.mu = new_mu;
                if (!dense) L.epsSum = (L.epsSum + old_mu * dN) - new_mu * dN;
            }
            for (uint32_t t = tid; t < p.G; t += kPipeThreads) L.betasqn[t] = 0.0;
            for (uint32_t t = tid; t < p.G * p.K; t += kPipeThreads) L.v[t] = 0.0;
        }
        group_constants(p, L);
        if (tid < count(0)) L.ids[0][tid] = order[tid];
        if (tid == 0) L.decided = L.got[0] = L.got[1] = -1;
        __syncthreads();

        double eS = L.epsSum;        // wave 8: epsilonSum
        double xc = 0.0;             // wave 8: correction of the next block's dot in this lane
        const uint32_t rnd0 = rnd + 1;   // block b's exchange round is rnd0 + b
        // the outputs of block b and its counts (wave 11, lane = slot)
        auto outputs = [&](int b) {
            const int nb = count(b), par = b & 1;
            const PipeMeta& m = L.meta[b & (kRing - 1)];
            const bool act = lane < nb;
            const int k = act ? lane : 0;
            const int sel = act ? L.os[par][k] : -1;
            const double bn = L.ob[par][k];
            const int g = m.gr[k];
            // v counts (integer-valued doubles: exact in any order), one add per distinct (group, component)
            const int key = sel >= 0 ? g * K + sel : -1;
            unsigned long long todo = __ballot(key >= 0);
            while (todo) {
                const int kb = lane_read(key, (int)__ffsll((long long)todo) - 1);
                const unsigned long long same = __ballot(key == kb);
                if (lane == 0) L.v[kb] += (double)__popcll(same);
                todo &= ~same;
            }
            // betasqnG += beta^2 in marker order (BayesRBase.cpp:353)
            unsigned long long sq = __ballot(sel > 0);
            while (sq) {
                const int i = (int)__ffsll((long long)sq) - 1;
                const double bb = lane_read(bn, i);
                const int gb = lane_read(g, i);
                if (lane == 0) L.betasqn[gb] += bb * bb;
                sq &= sq - 1;
            }
            // slot k's outputs are written by workgroup k % P, with agent-scope stores: a marker's writer
            // changes between iterations and the XCD L2s are not coherent with each other
            if (act && ((uint32_t)k < P ? (uint32_t)k == w : (uint32_t)k % P == w)) {
                const uint32_t j = m.mk[k];
                st_agent((uint64_t*)(q->beta + j), double_as_bits(bn));
                if (sel >= 0) __hip_atomic_store(q->comp + j, sel, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                st_agent((uint64_t*)(q->acum + j), double_as_bits(L.oa[par][k]));
                if (q->num_out) st_agent((uint64_t*)(q->num_out + j), double_as_bits(L.on[par][k]));
            }
        };
        // block b's changes on the slice, in order (dot waves)
        auto apply = [&](int b) {
            const int par = b & 1, n = L.nchg[par];
            n_changes += (unsigned long long)n;
            for (int i = 0; i < n; ++i) {
                const int k = L.ck[par][i];
                const double d0 = L.cdl[par][i][0], d1 = L.cdl[par][i][1], d2 = L.cdl[par][i][2], d3 = L.cdl[par][i][3];
                const E f0 = (E)d0, f1 = (E)d1, f2 = (E)d2, f3 = (E)d3;
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const uint32_t* cw = L.codes[b & (kRing - 1)][k][r];
                    const uint32_t bits = cw[lane >> 1] >> (16 * (lane & 1));
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const uint32_t at = lo + (uint32_t)r * kRun + 8u * (uint32_t)lane + (uint32_t)e;
                        const E x = eps[r][e] + wt_t((bits >> (2 * e)) & 3u, f0, f1, f2, f3);
                        eps[r][e] = at < hi ? x : (E)0;
                    }
                    if constexpr (kF32) {
                        const uint32_t at = lo + (uint32_t)r * kRun + (uint32_t)tid;
                        const uint32_t c = (cw[4 * wave + (lane >> 4)] >> (2 * (lane & 15))) & 3u;
                        const double x = e64[r] + wt_of(c, d0, d1, d2, d3);
                        e64[r] = at < hi ? x : 0.0;
                    }
                }
            }
        };
        // block b's decisions (wave 8, lane = slot), BayesRBase.cpp:300-378
        auto decide = [&](int b, auto kc, auto exact) {
            constexpr int kK = decltype(kc)::value;
            const int nb = count(b), nn = count(b + 1), par = b & 1;
            const PipeMeta& m = L.meta[b & (kRing - 1)];
            const bool act0 = lane < nb;
            const int k = act0 ? lane : 0;
            const double bo = act0 ? m.bo[k] : 0.0;
            const double u = q->mode == kModeChain ? L.du[par][k] : m.u[k];
            const double z = q->mode == kModeChain ? L.dz[par][k] : m.z[k];
            const double w0 = m.w[k][0], w1 = m.w[k][1], w2 = m.w[k][2], w3 = m.w[k][3];
            const int g = m.gr[k];
            // the group's constants: in registers for up to 4 components, else read from LDS when needed
            constexpr bool kRegs = kK <= 4;
            constexpr int kC = kRegs ? kK : 1;
            double dg[kC], hk[kC], lc[kC], zs[kC], rd[kC];
            const int gk = g * K;
            if constexpr (kRegs) {
#pragma unroll
                for (int c = 0; c < kK; ++c) {
                    const int at = gk + (c < K ? c : 0);
                    dg[c] = L.gdg[at];
                    hk[c] = L.ghk[at];
                    lc[c] = L.gc[at];
                    zs[c] = z * L.gbsd[at];
                    rd[c] = L.grd[at];
                }
            }
            const double base = bo * (double)(q->N - 1u);
            // epsilonSum's change per unit of beta (sparsebayesrkernel.cpp:29-34)
            const double dS = dense ? 0.0 : w2 * w3 - w0 * (double)q->N * w3;
            const unsigned long long im = __ballot(bo != 0.0);
            double dot;
            if (__builtin_amdgcn_readfirstlane(L.got[par]) == b) {
                dot = L.tots[par][lane];
            } else if (gather_round(rnd0 + (uint32_t)b, nb, &dot, never) < 0) {
                if (lane == 0) { L.abort = 1; raise_abort(*q, 2); }
                return;
            }
            tick(2);
            dot += xc;
            xc = 0.0;
            int start = 0, sel = -1;
            unsigned long long chm = 0;      // slots whose beta changes
            double bnew = bo, e0 = 0.0, es = 1.0, numk = 0.0;
            while (start < nb) {
                const bool act = lane >= start && act0;
                const double num = dense ? dot + base : __builtin_fma(dot - w0 * eS, w3, base);
                const MixDraw md = mix_draw<kK, decltype(exact)::value>(
                    K, num * num, u, [&](int c) { return kRegs ? dg[kRegs ? c : 0] : L.gdg[gk + c]; },
                    [&](int c) { return kRegs ? hk[kRegs ? c : 0] : L.ghk[gk + c]; },
                    [&](int c) { return kRegs ? lc[kRegs ? c : 0] : L.gc[gk + c]; });
                // the beta draw of the chosen component (BayesRBase.cpp:343-352)
                double bn = md.sel == 0 ? 0.0 : bo;
                if constexpr (kRegs) {
#pragma unroll
                    for (int c = 1; c < kK; ++c) bn = md.sel == c ? __builtin_fma(num, rd[c], zs[c]) : bn;
                } else {
                    const int at = gk + (md.sel > 0 ? md.sel : 0);
                    const double b2 = __builtin_fma(num, L.grd[at], z * L.gbsd[at]);
                    bn = md.sel > 0 ? b2 : bn;
                }
                if (act) {
                    sel = md.sel;
                    e0 = md.e0;
                    es = md.s;
                    numk = num;
                    bnew = bn;
                }
                const unsigned long long cm = __ballot(act && bn != bo);
                if (!cm) break;
                // the first change: its residual change, and what it does to the later dots
                const int c = (int)__ffsll((long long)cm) - 1;
                const int rank = (int)__popcll(im & ((1ull << c) - 1ull));
                double gi, gx;
                if (((im >> c) & 1ull) && rank < kRows) {
                    gi = L.rows[par][rank][lane];
                    gx = L.rows[par][rank][kMaxB + lane];
                } else {
                    const double* row = gram + ((size_t)b * B + (size_t)c) * kGramCols;
                    gi = row[lane];
                    gx = row[kMaxB + lane];
                }
                const double dB = bo - bnew;
                chm |= 1ull << c;
                const double D = lane_read(dB, c);
                if (!dense) {
                    eS = eS + lane_read(dB * dS, c);
                }
                // entries left of the diagonal or past the block are not formed: selected away, not multiplied
                const double d2 = __builtin_fma(D, gi, dot), x2 = __builtin_fma(D, gx, xc);
                dot = lane > c ? d2 : dot;
                xc = lane < nn ? x2 : 0.0;
                start = c + 1;
            }
            // the changes in order, with their residual change per 2-bit code
            if ((chm >> lane) & 1ull) {
                const int n = (int)__popcll(chm & ((1ull << lane) - 1ull));
                const double dB = bo - bnew;
                L.ck[par][n] = lane;
                if (dense) {
                    L.cdl[par][n][0] = dB * w0;
                    L.cdl[par][n][1] = dB * w1;
                    L.cdl[par][n][2] = dB * w2;
                    L.cdl[par][n][3] = dB * w3;
                } else {
                    // raggedbayesrkernel.cpp:10-30
                    const double meanAdjustment = dB * w0 * w3;
                    const double oneAdjustment = dB * w3;
                    L.cdl[par][n][0] = -meanAdjustment + 2 * oneAdjustment;
                    L.cdl[par][n][1] = 0.0;
                    L.cdl[par][n][2] = -meanAdjustment + oneAdjustment;
                    L.cdl[par][n][3] = -meanAdjustment;
                }
            }
            if (act0) {
                L.ob[par][k] = bnew;
                L.oa[par][k] = MixDraw::prob0(e0, es);
                L.on[par][k] = numk;
                L.os[par][k] = sel;
            }
            if (lane == 0) L.nchg[par] = (int)__popcll(chm);
            tick(3);
        };

        tick(5);
        // ---- the sweep (AnalysisGraph::exec over the order). Step b decides block b; steps -2 and -1 fill
        // the pipeline.
        if (wave >= kDotWaves) {
            // these waves hold no slice from here on: none of its registers is kept over their loops
#pragma unroll
            for (int r = 0; r < R; ++r) {
#pragma unroll
                for (int e = 0; e < 8; ++e) eps[r][e] = 0;
                if constexpr (kF32) e64[r] = 0.0;
            }
        }
        if (wave < kDotWaves) {
            // blocks until the FP32 slice is re-rounded: half the interval asked for, since the re-rounding reaches
            // the dots two steps after the block that it follows
            const int every = (int)max((q->refresh_blocks + 1u) / 2u, 1u);
            int due = every;
            bool fresh = false;
            for (int b = -2; b < nblocks; ++b) {
                asm volatile("" : "+s"(q), "+v"(lane));
                const int nb1 = count(b + 1);
                const int b1 = b + 1;
                if (wave == 0) tick(0);
                if (b >= 1) {
                    if constexpr (kF32) {
                        // the slice re-rounded from the FP64 residual in the step before
                        if (fresh) {
#pragma unroll
                            for (int r = 0; r < R; ++r)
#pragma unroll
                                for (int e = 0; e < 8; ++e) eps[r][e] = L.fs[(b - 1) & 1][r * kRun + 8 * lane + e];
                        }
                    }
                    apply(b - 1);
                    if constexpr (kF32) {
                        fresh = --due == 0;
                        if (fresh) due = every;
                        if (fresh)
#pragma unroll
                            for (int r = 0; r < R; ++r) L.fs[b & 1][r * kRun + tid] = (float)e64[r];
                    }
                }
                if (wave == 0) tick(4);

                // ---- partial dots of block b + 1's slots over the slice: 8 slots per wave, the column values
                // from the pair table, two per LDS load, products summed in individual order
                if (kSlotsPerWave * wave < nb1) {
                    E part[kSlotsPerWave];
                    uint32_t bits[kSlotsPerWave][R];
#pragma unroll
                    for (int j = 0; j < kSlotsPerWave; ++j) {
                        const int k = kSlotsPerWave * wave + j;
#pragma unroll
                        for (int r = 0; r < R; ++r)
                            bits[j][r] = L.codes[b1 & (kRing - 1)][k][r][lane >> 1] >> (16 * (lane & 1));
                    }
#pragma unroll
                    for (int j = 0; j < kSlotsPerWave; ++j) {
                        const int k = kSlotsPerWave * wave + j;
                        const E* tab = &L.pt[b1 & 1][kLay == kLayoutRagged ? 0 : k][0][0];
                        E s = 0;
#pragma unroll
                        for (int r = 0; r < R; ++r) {
                            using E2 = typename std::conditional<kF32, flt2, dbl2>::type;
                            E2 x[4];
#pragma unroll
                            for (int i = 0; i < 4; ++i)
                                x[i] = *reinterpret_cast<const E2*>(tab + 2 * ((bits[j][r] >> (4 * i)) & 15u));
#pragma unroll
                            for (int i = 0; i < 4; ++i) {
                                s = fma_t(x[i].x, eps[r][2 * i], s);
                                s = fma_t(x[i].y, eps[r][2 * i + 1], s);
                            }
                        }
                        part[j] = s;
                        // four slots' table loads in flight at most (all eight spill)
                        if (j == kSlotsPerWave / 2 - 1) __builtin_amdgcn_sched_barrier(0);
                    }
                    double tot;
                    if constexpr (kF32) tot = transpose_reduce8_c(part, lane);
                    else tot = transpose_reduce8(part, lane);
                    const int k = kSlotsPerWave * wave + (lane >> 3);
                    if ((lane & 7) == 0 && k < nb1)
                        publish_pair(q->xchg1, part_slot(rnd0 + (uint32_t)b1, k, w), rnd0 + (uint32_t)b1, tot);
                }
                if (wave == 0) tick(1);
                __syncthreads();
                if (L.abort) goto done;
            }
        } else if (wave == kDecWave) {
            __builtin_amdgcn_s_setprio(3);
            __syncthreads();
            __syncthreads();
            for (int b = 0; b < nblocks; ++b) {
                asm volatile("" : "+s"(q), "+v"(lane));
                t_last = w == 0 ? __builtin_amdgcn_s_memrealtime() : 0;
                with_components(K, [&](auto kc, auto exact) { decide(b, kc, exact); });
                if (lane == 0) L.decided = b;
                __syncthreads();
                if (L.abort) goto done;
            }
        } else if (wave == kRedWave) {
            __builtin_amdgcn_s_setprio(2);
            bool reduced = true;             // block b's slots were reduced in the step before
            for (int b = -2; b < nblocks; ++b) {
                asm volatile("" : "+s"(q), "+v"(lane));
                const int b1 = b + 1, nb1 = count(b1);
                int st = 1;
                if (!reduced) st = reduce_round(rnd0 + (uint32_t)b, count(b), never);
                reduced = true;
                if (st > 0 && b1 >= 0 && nb1 > 0) {
                    // block b + 1 already in this step, as far as its words arrive before block b is decided
                    const volatile int* dec = &L.decided;
                    auto leave = [&] { return *dec >= b; };
                    st = reduce_round(rnd0 + (uint32_t)b1, nb1, leave);
                    reduced = st == 1;
                    double x;
                    if (st == 1 && b >= 0 && (st = gather_round(rnd0 + (uint32_t)b1, nb1, &x, leave)) == 1) {
                        L.tots[b1 & 1][lane] = x;
                        if (lane == 0) L.got[b1 & 1] = b1;
                    }
                }
                if (st < 0 && lane == 0) {
                    L.abort = 1;
                    raise_abort(*q, 1);
                }
                __syncthreads();
                if (L.abort) goto done;
            }
        } else if (wave == kLoadWave) {
            __builtin_amdgcn_s_setprio(2);
            for (int b = -2; b < nblocks; ++b) {
                asm volatile("" : "+s"(q), "+v"(lane));
                const int b1 = b + 1, b2 = b + 2;
                const int nb1 = count(b1), nb2 = count(b2);
                // columns of block b + 2, the flattened [slot][R][32] words: four to a lane where slices start on 16
                // bytes of their columns. A load past the column's end is of its last words, of individuals that
                // hold no residual; a slot past the block is column 0.
                if (nb2 > 0) {
                    const uint32_t* ids = L.ids[b2 & (kRing - 1)];
                    uint32_t* dst = &L.codes[b2 & (kRing - 1)][0][0][0];
                    auto columns = [&](auto wc) {
                        constexpr uint32_t kWords = decltype(wc)::value, per = (uint32_t)R * 32u / kWords;
                        const uint32_t words = (uint32_t)q->col_words;
                        const uint32_t at = min((lo >> 4) + kWords * ((uint32_t)lane % per), words - kWords);
#pragma unroll 8
                        for (uint32_t i = 0; i < per; ++i) {
                            const uint32_t k = ((uint32_t)lane + 64u * i) / per;
                            const uint32_t j = k < (uint32_t)nb2 ? ids[k] : 0u;
                            load_to_lds<4 * (int)kWords>(q->dense + (size_t)j * words + at, dst + 64u * kWords * i);
                        }
                    };
                    if (p.S % 64u == 0u) columns(std::integral_constant<uint32_t, 4>());
                    else columns(std::integral_constant<uint32_t, 1>());
                }
                // Gram rows of block b + 1's in-model slots
                if (nb1 > 0) {
                    const PipeMeta& m = L.meta[b1 & (kRing - 1)];
                    const bool in = lane < nb1 && m.bo[lane < nb1 ? lane : 0] != 0.0;
                    unsigned long long im = __ballot(in);
                    const int have = min((int)__popcll(im), kRows);
                    for (int i = 0; i < have; ++i, im &= im - 1) {
                        const int h = (int)__ffsll((long long)im) - 1;
                        load_to_lds<16>(gram + ((size_t)b1 * B + (size_t)h) * kGramCols + 2 * lane, &L.rows[b1 & 1][i][0]);
                    }
                }
                if (q->mode == kModeChain && lane < nb1) {
                    double u;
                    uint64_t zw;
                    chain_draws(*q, L.ids[b1 & (kRing - 1)][lane], iteration, u, zw);
                    L.du[b1 & 1][lane] = u;
                    L.dz[b1 & 1][lane] = bits_as_double(zw);
                }
                wait_vm<0>();   // the loads into LDS are done
                __syncthreads();
                if (L.abort) goto done;
            }
        } else {
            __builtin_amdgcn_s_setprio(2);
            for (int b = -2; b < nblocks; ++b) {
                asm volatile("" : "+s"(q), "+v"(lane));
                const int b2 = b + 2, b3 = b + 3;
                const int nb2 = count(b2);
                // constants of block b + 2 and ids of block b + 3
                const uint32_t j = lane < nb2 ? L.ids[b2 & (kRing - 1)][lane] : 0u;
                const uint64_t bo = ld_agent((const uint64_t*)(q->beta + j));
                const int32_t g = q->group ? q->group[j] : 0;
                const double u_ = q->u[j], z_ = q->z[j];
                double m0, m1, m2, m3 = 0.0;
                if constexpr (dense) {
                    const double* lt = q->lut + 4 * (size_t)j;
                    m0 = lt[2];
                    m1 = lt[3];
                    m2 = lt[1];
                    m3 = lt[0];
                } else {
                    const double* st = q->stats + 4 * (size_t)j;
                    m0 = st[0];
                    m1 = st[1];
                    m2 = st[3];
                }
                const uint32_t id = order[min((uint32_t)b3 * B + (uint32_t)lane, M - 1u)];
                if (lane < nb2) {
                    PipeMeta& m = L.meta[b2 & (kRing - 1)];
                    m.mk[lane] = j;
                    m.gr[lane] = g;
                    m.bo[lane] = bits_as_double(bo);
                    m.w[lane][0] = m0;
                    m.w[lane][1] = m1;
                    m.w[lane][2] = m2;
                    m.w[lane][3] = dense ? m3 : 1.0 / m1;
                    m.u[lane] = u_;
                    m.z[lane] = z_;
                    if constexpr (kLay != kLayoutRagged) {
                        // EigenBayesRKernel: missing calls at the mean
                        const double t0 = dense ? m0 : 2.0, t1 = dense ? m1 : m0, t2 = dense ? m2 : 1.0, t3 = dense ? m3 : 0.0;
                        // (entry order turned by the lane: the lanes' tables are a multiple of all banks apart)
#pragma unroll 4
                        for (int i = 0; i < 16; ++i) {
                            const uint32_t n = (uint32_t)(i + lane) & 15u;
                            L.pt[b2 & 1][lane][n][0] = (E)wt_of(n & 3u, t0, t1, t2, t3);
                            L.pt[b2 & 1][lane][n][1] = (E)wt_of(n >> 2, t0, t1, t2, t3);
                        }
                    }
                }
                if (lane < count(b3)) L.ids[b3 & (kRing - 1)][lane] = id;
                if (b >= 1) outputs(b - 1);
                __syncthreads();
                if (L.abort) goto done;
            }
        }
        rnd += (uint32_t)nblocks;
        n_rounds += (unsigned long long)nblocks;
        if (wave < kDotWaves) {
            apply(nblocks - 1);
        } else if (wave == kMetaWave) {
            outputs(nblocks - 1);
        } else if (wave == kDecWave && lane == 0) {
            L.epsSum = eS;
        }
        // other workgroups read this workgroup's beta stores only in the block loads of the next iteration,
        // which follow this workgroup's next publish
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();

        if (p.mode == kModeChain && !(kParts && (q->part & 2u))) {
            double e2 = 0.0;
            const bool ok = fp64_region([&](double (&ed)[R][8]) {
                // ---- fixed effects (BayesRBase.cpp:212-235)
                if (p.F && !fixed_effects<R>(p, L, ed, iteration, lo, hi, lane, allreduce)) return false;
                // ---- |eps|^2 of the sigmaE draw
                double part = 0.0;
#pragma unroll
                for (int r = 0; r < R; ++r)
#pragma unroll
                    for (int e = 0; e < 8; ++e) part += ed[r][e] * ed[r][e];
                return allreduce(part, &e2);
            });
            if (!ok) goto done;
            scalar_draws(p, L, iteration, it, e2, w);
            if (wave == 0) tick(5);
        }
    }

done:
    __syncthreads();
    if (L.abort == 0) {
        if constexpr (kF32) {
            if (wave < kDotWaves)
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const uint32_t i = lo + (uint32_t)r * kRun + (uint32_t)tid;
                    if (i < hi) p.eps[i] = e64[r];
                }
        } else if (wave == 0) {
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const uint32_t i = lo + (uint32_t)r * kRun + 8u * (uint32_t)lane + (uint32_t)e;
                    if (i < hi) p.eps[i] = (double)eps[r][e];
                }
        }
        if (w == 0) {
            if (tid == 0) {
                p.scal[SL.mu()] = L.mu;
                p.scal[SL.sigmaE()] = L.sigmaE;
                p.scal[SL.epsSum()] = L.epsSum;
                __hip_atomic_store(p.ctl + kCtlRound, rnd, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                // (added to: a chain may take several launches)
                p.counters[0] += n_rounds;
                p.counters[1] += n_changes;
                p.counters[2] += tk[0];
                p.counters[3] += tk[1];
                p.counters[6] += tk[4];
                p.counters[7] += tk[5];
            }
            if (wave == kDecWave && lane == 0) {
                p.counters[4] += tk[2];
                p.counters[5] += tk[3];
            }
            for (uint32_t t = tid; t < p.G; t += kPipeThreads) {
                p.scal[SL.sigmaG() + t] = L.sigmaG[t];
                p.scal[SL.betasqn() + t] = L.betasqn[t];
            }
            for (uint32_t t = tid; t < p.G * p.K; t += kPipeThreads) {
                p.scal[SL.pi() + t] = L.pi[t];
                p.scal[SL.v() + t] = L.v[t];
            }
            if (p.F && tid == 0) p.fixed[0] = L.sigmaF;
            for (uint32_t t = tid; t < p.F; t += kPipeThreads) {
                p.fixed[1 + t] = L.gamma[t];
                p.forder[t] = L.forder[t];
            }
        }
    }
}

template <int R, int kLay, bool kF32, bool kParts>
__global__ void __launch_bounds__(kPipeThreads)
bayesr_pipe_kernel(SweepParams p)
{
    __shared__ PipeShared<R, kLay, kF32> L;
    pipe_body<R, kLay, kF32, kParts>(p, (ConstParams)__builtin_amdgcn_kernarg_segment_ptr(), L, blockIdx.x);
}

// ------------------------------------------------------- cohorts in one launch --

// Independent single-chain contexts (cohorts of uneven N and M) in one persistent cooperative launch: cohort c
// owns workgroups [first[c], first[c+1]) and runs its own context's chain on them -- its own slices, exchange
// words, state and counters -- so small cohorts, whose steps cost as much as a large one's, run side by side.
// Every cohort of a launch has the same lane runs R and residual precision; the layout is per cohort.
constexpr int kMaxCohorts = 64;

struct CohortTable {
    const SweepParams* params;          // device array, one per cohort
    uint32_t n;
    uint32_t first[kMaxCohorts + 1];    // first workgroup of each cohort; first[n] = grid size
};

template <int R, bool kF32, bool kParts>
__global__ void __launch_bounds__(kPipeThreads)
bayesr_cohort_kernel(CohortTable t)
{
    __shared__ union {
        PipeShared<R, kLayoutDense, kF32> d;
        PipeShared<R, kLayoutEigen, kF32> e;
        PipeShared<R, kLayoutRagged, kF32> r;
    } L;
    uint32_t c = 0;
    while (c + 1 < t.n && blockIdx.x >= t.first[c + 1]) ++c;
    const SweepParams p = t.params[c];
    const ConstParams q = (ConstParams)(uint64_t)(t.params + c);   // (not written while the kernel runs)
    const uint32_t w = blockIdx.x - t.first[c];
    if (p.layout == kLayoutDense) pipe_body<R, kLayoutDense, kF32, kParts>(p, q, L.d, w);
    else if (p.layout == kLayoutEigen) pipe_body<R, kLayoutEigen, kF32, kParts>(p, q, L.e, w);
    else pipe_body<R, kLayoutRagged, kF32, kParts>(p, q, L.r, w);
}

} // namespace brr
