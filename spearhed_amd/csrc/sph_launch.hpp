// sph_launch.hpp -- host-side launch interface of the gfx950 kernels (internal to the library).
#pragma once

#include <hip/hip_runtime.h>

#include "sph_device.hpp"

namespace sph {

struct LaunchCtx {
    const RunDev* runs;  // device run table
    int nruns;
    int ncell_tot;
    int nkb;             // particle-kernel blocks (run-aligned, 256 particles each)
    int mixed;
    int has_mhd;
    int has_state = 1;  // 0: velocity, u and rho are not part of the state (the resort leaves them alone)
    int force_chunk;
    int kmax;     // max lanes per target in the pair passes
    int balance;  // pair_balance: 1 = the force pass shares a target's accepted pairs among its K lanes,
                  // 2 = whole-supercell neighbour lists
    int kern;     // smoothing kernel of every run (SPH_KERNEL_*), or -1 when runs differ
    int one_h;    // every run's particles share one smoothing length (the run's own)
    int rmax;     // largest stencil reach of the runs: 1 (supercells of edge >= H) or 2 (edge >= H/2; pair
                  // passes take the chunked lane loop, pair_balance 0)
    int persistent_waves;  // pair passes: 0 = one wave per supercell; else a persistent grid of this many
                           // waves (a multiple of 8) walking the supercells at a stride of the grid
    StateBuf S;          // current buffer set
    WorkBuf W;
    hipStream_t stream;
};

// Columns copied by one launch (launch_copy_columns): any alignment and length >= 1, no overlaps; destinations
// on the device or in pinned host memory.
struct CopyTable {
    struct Col {
        void* dst;
        const void* src;
        int64_t bytes;
    };
    int n;
    Col col[32];  // a response has at most 29 columns and the conserved sums
};
// Largest response that a kernel writes to pinned host memory (launch_copy_out). One launch takes 6 us of host
// time and 8 us on the stream at 0.28 MB where the copies of 13 columns take 34 and 75. With several contexts
// keeping the link busy the runtime's copies win beyond it, since a kernel's writes hold up the other streams'
// kernels (evaluations of 20^3 / 32^3 / 44^3 / 56^3 / 62^3 / 70^3 / 80^3 particles in turn, 0.35 to 23 MB each: 31 /
// 56 / 122 / 191 / 260 / 325 / 464 us by copies, 31 / 55 / 101 / 185 / 235 / 334 / 492 us by the kernels; 13.2 MB
// beside the cubic kernel 260 to 299 by copies, 297 by the kernels).
constexpr int64_t kKernelCopyBytes = int64_t(12) << 20;
// The same for copies out of a pool's ring, which run beside the next steps on their own stream: 8.9 MB after
// seven steps of 131,044 particles, 804 us by the kernel, 937 us by copies.
constexpr int64_t kRingCopyBytes = int64_t(16) << 20;
// Responses up to this size are written by all XCDs (0.35 MB 31 us a pass instead of 36, 1.4 MB the same).
constexpr int64_t kWideCopyBytes = int64_t(1) << 20;

hipError_t launch_copy_columns(const CopyTable& t, hipStream_t s);
hipError_t launch_copy_out(const CopyTable& t, hipStream_t s);
hipError_t launch_fill_u32(uint32_t* p, uint32_t v, int64_t n, hipStream_t s);
// Copy the state of n_keep runs from A to B: run k's particles [src, src + count) to [dst, dst + count),
// with (dst, src, count) at tab[3k..3k+2] on the device, dst ascending from 0 and runs contiguous.
// Per-run dt, time and priming flag of a new run set of n_new runs from the n_old old ones (W.run_src:
// the old run each new run continues, or -1 for a fresh run); runs is the new run table.
hipError_t launch_remap_runs(const RunDev* runs, const WorkBuf& W, int n_old, int n_new, hipStream_t s);
// New initial data for one run: time 0, dt its fixed dt or 0, primed by its next step.
hipError_t launch_restart_run(const RunDev* runs, const WorkBuf& W, int run, hipStream_t s);
hipError_t launch_move_runs(const StateBuf& A, const StateBuf& B, const int64_t* tab, int n_keep, int64_t total,
                            int mixed, int mhd, hipStream_t s);
// Without store, launch_scatter_gather has to be given the same drift.
hipError_t launch_drift_bin(const LaunchCtx& c, double dt_host, int do_drift, bool store = true);
hipError_t launch_scan(const LaunchCtx& c);
hipError_t launch_scatter_gather(const LaunchCtx& c, const StateBuf& Snew, double dt_host = 0.0, int do_drift = 0);
hipError_t launch_density(const LaunchCtx& c);
hipError_t launch_forces(const LaunchCtx& c);
hipError_t launch_kick(const LaunchCtx& c, double dt_host, int do_kick);

}  // namespace sph
