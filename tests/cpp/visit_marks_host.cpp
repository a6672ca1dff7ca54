/* The runs that the lanes of a lane group find for visits 0 .. wtot-1 of a pass,
 * from the kernels' own index arithmetic (visit_marks.h), on the host: one group
 * of `lanes` lanes whose pass has nrun runs (visit offsets pref[0 .. nrun],
 * pref[nrun] its visits), in a wave whose longest pass has wtot visits, with
 * marks over vcap visits at a time. */
#define __host__
#define __device__
#include <algorithm>
#include <vector>

#include "visit_marks.h"

extern "C" void visit_runs(int lanes, int vcap, int nrun, const int *pref, int wtot, int *run)
{
    std::vector<unsigned> bits(vcap / 32);
    for (int seg0 = 0; seg0 < wtot; seg0 += vcap) {
        std::fill(bits.begin(), bits.end(), 0u);
        int started = 0;
        for (int i = 0; i < nrun; i++) {
            const int o = pref[i] - seg0;
            started += o <= 0;
            if (o > 0 && o <= vcap)
                bits[pisco::mark_word(o)] |= pisco::mark_bit(o);
        }
        int base = pisco::segment_base(started);
        for (int k = 0; k < std::min(vcap, wtot - seg0); k += lanes) {
            const unsigned m = bits[k >> 5] >> (k & 31);
            for (int l = 0; l < lanes && seg0 + k + l < wtot; l++)
                run[seg0 + k + l] = base + pisco::marks_below(m, l);
            base += lanes == 32 ? __builtin_popcount(m) : pisco::marks_below(m, lanes);
        }
    }
}
