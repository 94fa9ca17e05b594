// stop_mark.h -- which launch ended a scene's CG loop (InstDev::stopped)
//
// A kernel that records the end of a loop does so while waves of the same launch, each on its own, read the
// flag at their head: a workgroup whose waves saw both values would lose some of them before its barriers.
// So `stopped` says which launch recorded it -- 1: before the first iteration, stop_mark(it, phase): the
// operator side (phase 0) or the update (1) of iteration `it` -- and a kernel leaves at its head for
// earlier marks only.  What its own launch records, every workgroup finds by the same test on the same sums.
#pragma once

namespace sofa_amd {

constexpr int stop_mark(int it, int phase) { return 2 * it + phase; }
// whether a launch before that of `mark` stopped the scene (mark 0, a launch that records nothing: any launch)
constexpr bool stopped_before(int stopped, int mark) {
    return (unsigned)(stopped - 1) < (unsigned)(mark - 1);
}

}  // namespace sofa_amd
