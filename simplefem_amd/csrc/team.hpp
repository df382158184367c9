// team.hpp -- host interface of the one-launch solves by a team of workgroups
// (team.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "kernels.hpp"

namespace sfa {

constexpr int kTeamWaves = 8;        // wavefronts per workgroup
constexpr int kTeamMaxBlocks = 256;  // one workgroup per CU
constexpr int kTeamMaxGroups = 512;  // groups of a sweep (kept in LDS)
constexpr int kTeamSyncWords = 1024; // unsigned words of TeamArgs::sync

// A group of a sweep.  turn: which wavefront of a workgroup takes the first of
// the workgroup's slices; it moves on from group to group, so that a
// wavefront has several steps of the chain to load its next slice in, and is
// the same for both steps of a colour.
struct TeamGroup {
    SweepGroup g;
    int turn, pad;
};

// A system as the kernel takes it: the vectors, partials and state of the
// launches of an iteration (kernels.hpp), and a second z.
template <typename T>
struct TeamArgs {
    SellViewT<T> full, lower, upper;
    const TeamGroup* groups;   // gl forward groups, then gu backward groups
    int gl, gu;
    int fuse;        // the first backward group is the last forward one's rows, without entries
    int same_wave;   // a row's forward and backward steps fall to one wavefront (colours)
    int full_slices, full_row0;
    int n, n_active;
    T *x, *r, *d, *d1, *z, *z0, *m, *q;
    T* rs;           // !same_wave: r once more, for the backward rows' z.r
    const T* diag;
    T omega, c2;
    SolveState* st;
    double *ps, *pb, *grp;
    unsigned* sync;
    int max_iters;   // even
};

// Runs iterations from parity 0 until the loop ends or max_iters of them have
// run, in one launch of `blocks` workgroups (a power of two, 8 to
// kTeamMaxBlocks) that must all be resident at once: the caller sees to that
// (team_acquire).  When a wait lasts too long -- something else holds the
// CUs -- the launch gives up and sets SolveState::team_lost; the state and the
// vectors are then to be set up again.
template <typename T>
hipError_t launch_team(hipStream_t s, const TeamArgs<T>& a, int blocks);

// Takes `blocks` of the device's CUs for a team; false when other teams of
// this process hold too many.
bool team_acquire(int device, int blocks);
void team_release(int device, int blocks);

// Counts the solves under way on a device in this process.  A team fills the
// chip and would hold up solves on other streams, which overlap well as
// launches, so it runs only for a solve that is alone.
struct SolveGuard {
    explicit SolveGuard(int device);
    ~SolveGuard();
    SolveGuard(const SolveGuard&) = delete;
    SolveGuard& operator=(const SolveGuard&) = delete;
    static bool alone(int device);

private:
    int device_;
};

}  // namespace sfa
