// gram_plan.hpp -- how the Gram rows of a call's iterations are cut into launches, and the workspace these use.
#pragma once

#include <stddef.h>
#include <stdint.h>

#include <algorithm>

namespace brr {

constexpr uint32_t kGramChunk = 1024;   // individuals that a Gram workgroup stages at once
// Rows of the Gram workspace one launch may fill when it runs several iterations (1 KB a row): what bounds the
// workspace of a long chain (a chain of more is cut into launches), and a thousand blocks fill the chip.
constexpr size_t kGramRowsPerLaunch = 65536;
// Blocks from which a Gram launch is not split over the individuals. At N = 100,000 a sweep of 125 blocks takes
// 648 us with its Gram launch split in two (716 unsplit, and 219 instead of 70 at 4 blocks); of 250 blocks 1,265 us
// unsplit and 1,332 split: the products then go through memory and a second launch.
constexpr uint32_t kGramBlocks = 128;

struct GramPlan {
    uint32_t total;       // iterations of the call
    uint32_t step;        // iterations of a launch; the last one may have fewer
    uint32_t splits;      // workgroups per block, in every launch
    size_t rows;          // Gram rows of a launch, at most
    size_t acc_rows;      // rows of shared counts that a launch uses, at most (0: no block is split)

    uint32_t iterations(uint32_t first) const { return std::min(step, total - first); }
};

// The launches are of nearly equal length and split alike: a last one that decided for itself would have few blocks,
// and split them, where the others need no shared counts at all.
inline GramPlan gram_plan(uint32_t N, uint32_t M, uint32_t B, uint32_t total)
{
    GramPlan p{};
    p.total = total;
    const uint32_t most = (uint32_t)std::min<size_t>(total, std::max<size_t>(1, kGramRowsPerLaunch / M));
    const uint32_t launches = (total + most - 1) / most;
    p.step = (total + launches - 1) / launches;
    p.rows = (size_t)p.step * M;
    const uint64_t blocks = (uint64_t)p.step * ((M + B - 1) / B);
    const uint64_t chunks = (N + kGramChunk - 1) / kGramChunk;
    p.splits = blocks >= kGramBlocks ? 1u : (uint32_t)std::max<uint64_t>(1, std::min(2 * kGramBlocks / blocks, chunks));
    p.acc_rows = p.splits > 1 ? p.rows : 0;
    return p;
}

} // namespace brr
