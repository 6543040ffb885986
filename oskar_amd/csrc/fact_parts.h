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
 *    sources: 128 parts in 9 rounds instead of 123 in 8.65).  Where those are
 *    no more than parts of max_part, a short last part can end the last round
 *    sooner than equal ones: it does if all work in full rounds and that part
 *    take less than the rounds of equal parts (2048 x 20,000, 3 parts in 3.1
 *    rounds: 3734 against 4005 us; 1500 x 40,000, 5 parts in 2.93: 3837
 *    against 3786, equal). */
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
        const double last = (double) num_sources - (least - 1.0) * max_part;
        if (parts == least && (double) tiles * num_sources / PART_SLOTS +
                last < (double) rounds * ((double) num_sources / parts))
            return max_part;
    }
    /* The parts are a grid's y. */
    parts = std::min(parts, std::max(least, 65535LL));
    const long long part = (num_sources + parts - 1) / parts;
    return (int) std::min((long long) max_part,
            std::max((long long) unit, (part + unit - 1) / unit * unit));
}

/* Whether the units of a batch take part_sources(), which sizes the parts of
 * a unit as if it had the chip to itself, in place of parts of max_part.
 *
 * max_part: rounds of workgroups, each as long as the longest part, 1.1 us
 * per step of a round that is not full and 1.25 us of a full one.
 * part_sources: the work in full rounds, and 0.03 us per tile and part for
 * the partial sums.  Past two rounds of max_part little is idle: no (200
 * units of 97 stations x 12,007 sources: 2835 against 3578 us).  Measured, us (max_part -> part_sources): 97 stations x
 * 12,007 sources, 16 units 1095 -> 335, 64 units 1170 -> 1177, 170 units 2490
 * -> 3086; 30 x 2,000, 64 units 319 -> 152, 512 units 371 -> 1127; 300 x 500,
 * 32 units 191 -> 299.  Where it does not pay it also costs memory: 512 units
 * of 30 x 2,000 took 3.2 GB of partial sums for 0.1 GB. */
template <typename Sources>
bool part_sources_pay(int num_units, Sources sources, int num_stations,
        int max_part, int unit)
{
    const double tiles = (double) part_tiles(num_stations);
    double items = 0.0, work = 0.0, partials = 0.0, longest = 0.0;
    for (int u = 0; u < num_units; ++u)
    {
        const int S = sources(u);
        if (S <= 0) continue;
        const int part = part_sources(S, num_stations, max_part, unit);
        items += tiles * (double) (((long long) S + max_part - 1) / max_part);
        partials += tiles * (double) (((long long) S + part - 1) / part);
        work += tiles * (S / 8.0);
        longest = std::max(longest, std::min(S, max_part) / 8.0);
    }
    if (items >= 2 * PART_SLOTS) return false;
    const double whole = items <= PART_SLOTS ? 1.1 * longest :
            1.25 * longest * ceil(items / PART_SLOTS);
    return 1.25 * work / PART_SLOTS + 0.03 * partials < whole;
}

} /* namespace oskar_amd */

#endif /* OSKAR_AMD_FACT_PARTS_H_ */
