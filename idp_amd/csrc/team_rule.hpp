// Rules of the one-kernel PCG solve (k_pcg_team) that need no device code.
#pragma once

namespace idp {

constexpr int TEAM_MAX = 256;   // workgroups of a launch at most: one per CU of the whole chip
constexpr int TEAM_ROWS = 128;  // rows of a workgroup: two per 8 lanes in the SpMV, 4 lanes a row in the update

// Workgroups that can run together: a team of several waits for all of its
// members, so a launch with such a team has to fit the compute units that the
// device shows (a partition of the chip shows fewer than 256); teams of one
// wait for nobody.
inline bool team_fits(int workgroups, bool all_of_one, int resident)
{
    return workgroups <= TEAM_MAX && (all_of_one || workgroups <= resident);
}

// The kernel's vectors are buffers with 32-bit byte offsets over the whole
// context, the two copies of p (48 bytes a vertex) the longest of them: a
// batch of more than 89 million vertices, however few of its solves run, is
// out of their range.
inline bool team_addresses(long long nV) { return 48 * nV <= 0xffffffffll; }

// Looks of the batched hand-over: both PCG loops look at the solves of a call
// after 8, 24, 56, 120, 248, 504, 760, ... iterations of it (the two-kernel
// loop's chunks of 8, 16, ... 256).  At the first look b by which half of the
// solves have stopped, the others get as many iterations again and are handed
// over after 2 b.
constexpr int HAND_FIRST = 8;
constexpr int HAND_LOOKS = 48;  // looks that a launch keeps count of: the last is at 11,256 iterations
#ifdef __HIPCC__
__host__ __device__
#endif
inline int hand_next(int b)
{
    return b < 504 ? 2 * b + 8 : b + 256;
}

// Starts of the one-kernel solves of a context.  A team whose workgroups do
// not all become resident in time (other work holds compute units) leaves its
// solve to the two-kernel loop after TEAM_WAIT polls, about a millisecond: as
// long as a short solve takes.  While starts go on failing, the next 1, 3, 7,
// ... 63 solves take that loop without a try, so a GPU that is busy for long
// costs a context next to nothing; the results are the same either way.
constexpr long TEAM_WAIT = 1000;
struct TeamStarts {
    int failed = 0, skip = 0;
    bool now()
    {
        if (skip == 0) return true;
        --skip;
        return false;
    }
    void ended(bool started)
    {
        failed = started ? 0 : failed < 6 ? failed + 1 : 6;
        skip = (1 << failed) - 1;
    }
};

}  // namespace idp
