/* The items of a launch (work_items.h) on the host: the unit and sample of every
 * item of its grid; returns the grid's size. */
#define __host__
#define __device__
#include "work_items.h"

extern "C" long launch_items(long nsamp, long nunits, long chunk, long cap, long *unit,
                             long *sample)
{
    const long n = pisco::work_items(nsamp, nunits);
    for (long w = 0; w < n && w < cap; w++) {
        unit[w] = sample[w] = -1;
        pisco::work_item(w, nsamp, nunits, chunk, unit[w], sample[w]);
    }
    return n;
}
