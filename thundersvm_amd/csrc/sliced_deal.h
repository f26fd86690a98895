// How the sliced CSR kernel's work is dealt to workgroups.  Host and device, no HIP calls.
#pragma once
#include <algorithm>
#include <cstdint>

#if defined(__HIPCC__)
#define SLICED_HD __host__ __device__ __forceinline__
#else
#define SLICED_HD inline
#endif

// A block is sixteen working rows against all slices of 64 stored rows.  It is cut into per_block parts, `larger` of them of slices + 1
// slices, the others of `slices`; and the parts, block after block, are dealt to the workgroups in runs, to `longer` of them run + 1, to
// the others run.  Larger parts and longer runs are spread evenly (with the longer runs all on the first dies 7,000 x 10,000
// took 606 us, not 563).  All numbers are below 2^31; larger is 0 or per_block no more than 2,048.
struct SlicedDeal {
    unsigned per_block, slices, larger, workgroups, run, longer;
};

// One workgroup's way through its run: a stretch of slices of one block at a time.
struct SlicedWalk {
    unsigned t, end;
    SLICED_HD SlicedWalk(const SlicedDeal &d, unsigned w) {
        if (d.run == 1 && d.longer == 0) {
            // a part each: neighbours (of a die) take the same slices of one block after another, which its L2 then has (18,000 stored
            // rows, 512 working rows, seven parts a block: 105 us, 108 with the parts of a block side by side)
            const unsigned n_blocks = d.workgroups / d.per_block;
            t = w % n_blocks * d.per_block + w / n_blocks;
            end = t + 1;
            return;
        }
        t = w * d.run + w * d.longer / d.workgroups;
        end = (w + 1) * d.run + (w + 1) * d.longer / d.workgroups;
    }
    // slices slice0 .. slice1 - 1 of block `block`; false behind the last
    SLICED_HD bool next(const SlicedDeal &d, unsigned &block, unsigned &slice0, unsigned &slice1) {
        if (t >= end) return false;
        block = t / d.per_block;
        const unsigned from = t - block * d.per_block, here = d.per_block - from < end - t ? d.per_block - from : end - t;
        const unsigned to = from + here;
        slice0 = from * d.slices + from * d.larger / d.per_block;
        slice1 = to * d.slices + to * d.larger / d.per_block;
        t += here;
        return true;
    }
};

// `places`: workgroups that run at a time, one a CU.  256; 224 on a stream that leaves CUs out: workgroups are dealt to a die's four groups
// of eight CUs in turn, whether or not a group lacks one, so that of 232 or more some wait, as a rule, until another has ended (1,024
// rows of 18,000 columns on 255 CUs, 192 / 224 / 240 / 248 / 256 workgroups: 202 / 201 / 203 or 339 / 336 / 323 us).
//
// How a block is cut is the least of a model's time: the slices of the longest run and, for each block that it may touch, as much as
// SLICED_TILE slices for the tile (stored rows of some fifty entries: 17 us a tile, 1.9 a slice).  Cut finely, every workgroup has as
// much to do as the others but builds tiles that others have built as well; cut into few parts, it has whole blocks, and as workgroups
// then go through the same slices side by side, which the L2 is for, runs that begin anywhere count a tenth more.  us by runs of slices
// / halves / whole blocks, stored rows x working rows: 300 x 10,000 110 / - / 88; 7,000 x 4,099 250 / 346 / 386, x 6,000 383 / 345 / 431,
// x 8,000 488 / 463 / 434, x 20,000 1,132 / 1,116 / 1,078; 18,000 x 300 on 255 CUs 103, in eleven parts a block 77.  Over some 110
// sizes the choice is within 1.5 % of the best of these.  (Panels of stored rows that an L2 holds never were: 200,000 x 1,024 in one
// panel 1,695, in two to twenty-eight 1,726 to 2,252.)
// Against a run of slices for each of min(248, slices x blocks / 16) workgroups in such panels: 64 x 4,099 416 -> 52 us, 1,000 x 10,000 138 -> 113,
// 7,000 x 4,099 291 -> 248, x 10,000 618 -> 562, x 20,000 1,178 -> 1,077; on 255 CUs 18,000 x 300 121 -> 74, x 512 102 -> 105, x 1,024 336 -> 199.
constexpr unsigned SLICED_TILE = 10;

// n, n_blocks >= 1
inline SlicedDeal sliced_deal(int64_t n, int64_t n_blocks, unsigned places) {
    const int64_t slices = (n + 63) / 64;
    SlicedDeal best{};
    uint64_t best_cost = ~0ull;
    const auto consider = [&](int64_t parts) {
        const int64_t all = parts * n_blocks, run = (all + places - 1) / places, touched = (run - 1 + parts - 1) / parts + 1;
        if (all >= 0x7fffffff) return;
        uint64_t cost = (uint64_t) (run * ((slices + parts - 1) / parts) + SLICED_TILE * touched) * 10;
        if (run > 1 && parts > 4) cost += cost / 10;
        if (cost >= best_cost) return;
        best_cost = cost;
        const int64_t wgs = std::min<int64_t>(places, all);
        best = SlicedDeal{(unsigned) parts, (unsigned) (slices / parts), (unsigned) (slices % parts), (unsigned) wgs, (unsigned) (all / wgs), (unsigned) (all % wgs)};
    };
    // (for runs of one to eight parts the most parts that make them, or up to sixteen parts a block: as cheap as the best of all numbers of
    // parts at every size looked at, 0.1 us in place of 1.8)
    const bool few = n_blocks < places;
    for (int64_t i = 1; i <= (few ? 8 : 16); ++i) consider(std::min<int64_t>(slices, few ? i * places / n_blocks : i));
    consider(slices);
    return best;
}
