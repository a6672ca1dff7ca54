/*
 * visit_marks.h -- index arithmetic of the walk's run marks.
 *
 * A pass's visits are numbered 0 .. total-1; pref[i] is the first visit of run
 * i.  A lane finds its visit's run by counting the marks of the runs that start
 * at or before it.  The marks cover a segment of visits from seg0 on: bit
 * v - 1 - seg0 marks a run that starts at visit v > seg0.
 */
#ifndef PISCO_VISIT_MARKS_H
#define PISCO_VISIT_MARKS_H

namespace pisco {

/* The run of a segment's first visit, of `started` runs that start at or before
 * it.  A lane group without a run in the pass has 0: it idles beside groups
 * with several segments, and reads (and discards) entry 0. */
__host__ __device__ inline int segment_base(int started) { return started > 0 ? started - 1 : 0; }

/* The mark of a run that starts o > 0 visits after the segment's first. */
__host__ __device__ inline int mark_word(int o) { return (o - 1) >> 5; }
__host__ __device__ inline unsigned mark_bit(int o) { return 1u << ((o - 1) & 31); }

/* Runs that start within the `lane` visits after the first of a block of at most
 * 32, whose marks are the low bits of m. */
__host__ __device__ inline int marks_below(unsigned m, int lane)
{
    return __builtin_popcount(m & ((1u << (lane & 31)) - 1u));
}

} /* namespace pisco */

#endif
