// Host side of the resident solves (persist.h): when a result stands.  Plain
// C++, so it can be compiled and tested without a GPU.
#pragma once

namespace xcal {

// Whether a case's resident solve is complete, from its state after the
// launch: `stop` says that the case's first workgroup finished, `gave_up` that
// some workgroup of it left early, without its rows of the solution.  Both can
// be set, when the one that left had published its last sums: the solve is
// then incomplete whatever `stop` says.  Launch chains never set `gave_up`.
inline bool resident_done(int stop, int gave_up) { return stop != 0 && gave_up == 0; }

}  // namespace xcal
