/*
 * work_items.h -- order of the (unit, sample) items of a launch.
 *
 * A unit is a detector pair, a group of pairs or a strip of the samples' discs;
 * a "sample" may stand for a block's samples.  Samples are taken in chunks, and
 * within a chunk all items of one unit before the next.  The XCD-aware block
 * order hands each XCD a contiguous stretch of the items: consecutive waves
 * share one unit's part of the beam, and samples close in the scan.  The last
 * chunk is short, so that the nsamp * nunits items are all work and no XCD is
 * left with padding.
 */
#ifndef PISCO_WORK_ITEMS_H
#define PISCO_WORK_ITEMS_H

namespace pisco {

__host__ __device__ inline long work_items(long nsamp, long nunits) { return nsamp * nunits; }

/* Item w; false beyond the last one. */
__host__ __device__ inline bool work_item(long w, long nsamp, long nunits, long chunk, long &unit,
                                          long &sample)
{
    const long per = chunk * nunits, c = w / per, rem = w - c * per, first = c * chunk;
    const long len = nsamp - first < chunk ? nsamp - first : chunk;
    if (len <= 0 || rem >= len * nunits)
        return false;
    unit = rem / len;
    sample = first + (rem - unit * len);
    return true;
}

} /* namespace pisco */

#endif
