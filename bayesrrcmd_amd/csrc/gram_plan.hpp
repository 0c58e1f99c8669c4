// gram_plan.hpp -- how the Gram rows of a call's iterations are cut into launches, and the workspace these use.
#pragma once

#include <stddef.h>
#include <stdint.h>

#include <algorithm>
#include <vector>

namespace brr {

constexpr uint32_t kGramChunk = 1024;   // individuals that a Gram workgroup stages at once
// Rows of the Gram workspace one launch may fill when it runs several iterations (1 KB a row): what bounds the
// workspace of a long chain (a chain of more is cut into launches), and a thousand blocks fill the chip.
constexpr size_t kGramRowsPerLaunch = 65536;
// Rows of the workspace at most: an iteration of more markers is swept in parts, a launch each. An iteration of 64
// individuals and 300,000 markers takes 21.3 ms in two parts, 22.1 ms in one with 300 MB of rows.
constexpr size_t kGramRowsMost = 262144;
// Rows that a step of several contexts may take (8 GB; more markers in parts, which change a chain's roundings).
constexpr size_t kCohortRowsMost = 8388608;
// Rows below which a workspace that the device has no room for is not halved any more.
constexpr size_t kGramRowsLeast = 8192;
// Blocks from which a Gram launch is not split over the individuals. At N = 100,000 a sweep of 125 blocks takes
// 648 us with its Gram launch split in two (716 unsplit, and 219 instead of 70 at 4 blocks); of 250 blocks 1,265 us
// unsplit and 1,332 split: the products then go through memory and a second launch.
constexpr uint32_t kGramBlocks = 128;

struct GramPlan {
    uint32_t total;       // iterations of the call
    uint32_t step;        // iterations of a launch; the last one may have fewer
    uint32_t parts;       // launches of an iteration (more than one: step is 1)
    uint32_t part;        // markers of a launch's iterations; the last part may have fewer
    uint32_t splits;      // workgroups per block, in every launch
    size_t rows;          // Gram rows of a launch, at most
    size_t acc_rows;      // rows of shared counts that a launch uses, at most (0: no block is split)

    uint32_t iterations(uint32_t first) const { return std::min(step, total - first); }
    uint32_t markers(uint32_t M, uint32_t q) const { return std::min(part, M - q * part); }   // of part q
};

// The launches of `total` iterations over M markers in blocks of B, with a workspace of `most` rows (at least B). They
// are of nearly equal length and split alike: a last one that decided for itself would have few blocks, and split them,
// where the others need no shared counts at all.
inline GramPlan gram_plan(uint32_t N, uint32_t M, uint32_t B, uint32_t total, size_t most)
{
    GramPlan p{};
    p.total = total;
    const uint32_t blocks1 = (M + B - 1) / B;             // of an iteration
    if (M > most) {
        const uint32_t fit = (uint32_t)std::max<size_t>(1, most / B);
        p.step = 1;
        p.parts = (blocks1 + fit - 1) / fit;
        p.part = (blocks1 + p.parts - 1) / p.parts * B;
        p.parts = (M + p.part - 1) / p.part;
    } else {
        const uint32_t fit = (uint32_t)std::min<size_t>(total, std::max<size_t>(1, std::min(most, kGramRowsPerLaunch) / M));
        const uint32_t launches = (total + fit - 1) / fit;
        p.step = (total + launches - 1) / launches;
        p.parts = 1;
        p.part = M;
    }
    p.rows = (size_t)p.step * std::min(p.part, M);
    const uint64_t blocks = (uint64_t)p.step * ((p.part + B - 1) / B);
    const uint64_t chunks = (N + kGramChunk - 1) / kGramChunk;
    p.splits = blocks >= kGramBlocks ? 1u : (uint32_t)std::max<uint64_t>(1, std::min(2 * kGramBlocks / blocks, chunks));
    p.acc_rows = p.splits > 1 ? p.rows : 0;
    return p;
}

// The steps of a call over several contexts whose Gram rows share one workspace: `step` iterations each or, where one
// iteration of all takes more than `most` rows, an iteration in `parts` of each context's blocks (a context with few blocks
// sits out some of them).
struct CohortPlan {
    uint32_t step, parts;
    size_t rows;          // rows of a step, at most

    // first marker of part `part` of M markers in blocks of B (parts: M)
    uint32_t first(uint32_t M, uint32_t B, uint32_t part) const
    {
        const uint64_t blocks = (M + B - 1) / B;
        return (uint32_t)std::min<uint64_t>(M, blocks * part / parts * B);
    }
};

inline CohortPlan cohort_plan(const std::vector<uint32_t>& M, const std::vector<uint32_t>& B, uint32_t total, size_t most)
{
    CohortPlan p{};
    size_t rows1 = 0;
    for (uint32_t m : M) rows1 += m;
    if (rows1 <= most) {
        const uint32_t fit = (uint32_t)std::min<size_t>(total, most / rows1);
        const uint32_t steps = (total + fit - 1) / fit;
        p.step = (total + steps - 1) / steps;
        p.parts = 1;
        p.rows = p.step * rows1;
    } else {
        p.step = 1;
        p.parts = (uint32_t)((rows1 + most - 1) / most);
        for (uint32_t part = 0; part < p.parts; ++part) {
            size_t rows = 0;
            for (size_t q = 0; q < M.size(); ++q) rows += p.first(M[q], B[q], part + 1) - p.first(M[q], B[q], part);
            p.rows = std::max(p.rows, rows);
        }
    }
    return p;
}

} // namespace brr
