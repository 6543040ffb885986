/*
 * Sources per part of the factorised correlators (shared by the one-call
 * and batch forms of xcorr_factorised.hip and by xcorr_stations.hip).
 */
#ifndef OSKAR_AMD_FACT_PARTS_H_
#define OSKAR_AMD_FACT_PARTS_H_

#include <math.h>

#include <algorithm>

namespace oskar_amd {

constexpr int PART_SLOTS = 512;     /* 256 CUs x two workgroups */

/* Workgroup tiles of 64 x 64 stations that hold a p > q pair. */
inline long long part_tiles(int num_stations)
{
    const long long nb = (num_stations + 63) / 64;
    return nb * (nb + 1) / 2;
}

/* Sources per part, at most max_part (the caller's limit on what is summed
 * in FP32) and a multiple of unit, for one (channel, time) unit.
 *
 * A workgroup takes one tile of one part, 8 sources per step.  At max_part,
 * 97 stations x 12,007 sources were 6 workgroups on 256 CUs (0.81 ms).
 *  - Fewer workgroups than the chip runs at once: a step takes about
 *    0.8 us on its own, so the parts of S / 8 steps cost 0.8 (S / 8) / parts
 *    us, and 0.064 us per tile and part for the 128 KB of partial sums
 *    written and read (4 TB/s); least at sqrt(12.5 (S / 8) / tiles) parts,
 *    and no more than one round of workgroups.
 *  - Otherwise: as many parts as whole rounds hold (512 stations x 1M
 *    sources: 128 parts in 9 rounds instead of 123 in 8.65). */
inline int part_sources(int num_sources, int num_stations, int max_part,
        int unit)
{
    const long long tiles = part_tiles(num_stations);
    const long long least = ((long long) num_sources + max_part - 1) /
            max_part;
    long long parts = least;
    if (tiles * least < PART_SLOTS)
    {
        const double steps = num_sources / 8.0;
        parts = std::max(least, std::min((long long) sqrt(12.5 * steps /
                (double) tiles), PART_SLOTS / tiles));
    }
    else
    {
        const long long rounds = (tiles * least + PART_SLOTS - 1) /
                PART_SLOTS;
        parts = std::max(least, PART_SLOTS * rounds / tiles);
    }
    /* The parts are a grid's y. */
    parts = std::min(parts, std::max(least, 65535LL));
    const long long part = (num_sources + parts - 1) / parts;
    return (int) std::min((long long) max_part,
            std::max((long long) unit, (part + unit - 1) / unit * unit));
}

} /* namespace oskar_amd */

#endif /* OSKAR_AMD_FACT_PARTS_H_ */
