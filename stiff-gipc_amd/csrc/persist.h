// persist.h -- the FP64 PCG solve of a small or medium system as one launch
// (persist.hip).
#pragma once

#include "linsys.h"

namespace sgipc
{

// Static part of the one-launch solve, made once per matrix pattern: the
// workgroups' row ranges (cut at MAS banks), and for each the columns outside
// its range (its halo) with every stored block's column renumbered to
// [own rows | halo].
class PersistPlan
{
  public:
    // part_first: first row of each MAS part (size parts + 1), empty for the
    // block-Jacobi preconditioner
    void build(const Bsr& A, const std::vector<int>& part_first, hipStream_t s);
    bool ready() const { return groups > 0 && polls != 0; }
    // most polls of a wait at a grid barrier; 0: not this way, -1: the default
    void set_polls(int n)
    {
        SG_CHECK(n >= -1, -1, "the number of polls is -1, 0 or positive");
        polls = n < 0 ? kPolls : n;
        pause = skip = 0;
    }

    // about a second; the workgroups meet within microseconds once all of them run
    static constexpr int kPolls = 1 << 20;
    int polls = kPolls;
    // After a wait that ran out the next solves, 16 and doubling up to 1024 while
    // it happens again, do not try: each attempt costs kPolls polls, and what kept
    // a workgroup from running (another program's work on the device) may last.
    int pause = 0, skip = 0;

    int groups = 0;                            // workgroups (0: not this way)
    int dev = 0, units = 0;                    // device, its compute units per XCD
    int rows = 0, halo = 0, banks = 0;         // most of one workgroup
    DBuf<int>            rstart, bstart;       // groups + 1: rows, level-0 banks
    DBuf<int>            hptr, hcol;           // groups + 1; halo columns
    DBuf<unsigned short> lcol;                 // per stored block
    // exchange slots of the grid barrier, control words and results
    DBuf<unsigned long long> slots;
    DBuf<int>                ctl;
    DBuf<double>             out;
};

struct PersistResult
{
    int    stop_at = 0;    // stopping check iteration (0: none)
    int    bad     = 0;    // 1: non-finite r.z
    double rz0 = 0, rz = 0;
};

// true: the solve ran (result in *res, x complete); false: this system or
// device does not take it, its contact rows are better served by a launch per
// operation, or a wait ran out, and x is still to be solved for
bool persist_solve(PersistPlan& plan, const SysView& S, Mas* mas, const double* dinv,
                   const double* b, double* x, double* z, double* p0, double* p1,
                   const PcgConfig& cfg, int maxit, int every, PersistResult* res, hipStream_t s,
                   Profiler* prof);

}  // namespace sgipc
