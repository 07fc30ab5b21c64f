// mf_pivots.h — the column loop of a front whose columns are spread over the
// four wavefronts of a workgroup, apart from the arithmetic, so that its
// order of barriers can be run on the host as well.
#pragma once

#if defined(__HIPCC__)
#define MF_PIVOTS_FN __host__ __device__ __forceinline__
#else
#define MF_PIVOTS_FN inline
#endif

namespace mf {

// Wavefront g of four runs the columns [0, nn) of one front; column k belongs
// to wavefront k mod 4.
//   own(k)     the owner factors column k; false: its pivot has failed
//   fail       the front's shared record, 0 before: set(v) by an owner, get()
//   barrier()  of the whole workgroup
//   update(k)  every wavefront takes column k off its later columns
//   closed     one more barrier a column: update(k) reads what own(k + 1)
//              overwrites
// False after a failed pivot.  The record is the failing column + 1 and ends
// the front at that column only: one barrier a column lets the owner of column
// k + 1 run ahead and record its failure while another wavefront has yet to
// look at column k's, and a plain flag would send that one away a barrier
// early (the next ticket then starts with three wavefronts out of step).
template <typename Own, typename Fail, typename Barrier, typename Update>
MF_PIVOTS_FN bool pivot_columns(int nn, int g, bool closed, Own own, Fail fail, Barrier barrier, Update update) {
    for (int k = 0; k < nn; ++k) {
        if (g == (k & 3) && !own(k)) fail.set(k + 1);
        barrier();
        if (fail.get() == k + 1) return false;
        update(k);
        if (closed) barrier();
    }
    return true;
}

}  // namespace mf
