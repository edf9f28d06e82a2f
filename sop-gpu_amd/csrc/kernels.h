// kernels.h -- host-side launchers for the kernels in kernels.hip.
#pragma once
#include <hip/hip_runtime.h>

#include "jobdesc.h"

namespace sop {

// Launch shapes of the LDS step and list kernels that the autotuner picks
// (none of them changes any result): threads of a step unit (its Verlet
// rows), Verlet entries fetched ahead per lane in the step, 64-entry chunks
// in flight per row in the Verlet build, and the row-sort cadence (every
// k-th Verlet rebuild).  split_rows (4, 8 or 16; 0: off) steps the LDS-step
// jobs by k_step_rows instead, that many rows per wavefront (two instead of
// four in the smallest launches) with each row's force terms spread over its
// lanes, and builds their lists one wavefront per row; split_global steps the
// jobs above the LDS limit the same way.  -1 (not in a shape that is launched):
// chosen by the rows of the launch.
struct StepShape {
    int unit_rows = kLdsUnit;
    int pair_batch = 6;
    int verlet_chunk = 8;
    int sort_every = kSortEvery;
    int split_rows = -1;
    int split_global = -1;
};
// The rule for the spread step where its rows are not asked for (measurements at
// Engine::effective_shape): rows of the launch up to which a wavefront takes
// two, four and eight rows (sixteen above), the rows of LDS-step jobs and of the
// others up to which they are spread at all, and the beads of a job whose lists
// are too short for less than eight rows per wavefront.
constexpr int kRowsTwo = 4500, kRowsFour = 17000, kRowsEight = 34000, kRowsMaxLds = 90000, kRowsMaxGlobal = 220000;
constexpr int kRowsShort = 28;
// A block of steps in one launch (k_block_rows; measurements at
// Engine::block_rows): beads of a job up to which it is possible, beads up to
// which it pays for any number of jobs, jobs of the largest size (by rows)
// from which it pays past that, and steps of one launch.
constexpr int kBlockBeads = 256, kBlockShort = 32, kBlockJobs = 100, kBlockSteps = 250;
// The autotuner tries split_rows only where the launch has at most this many
// 64-row tiles.
constexpr int kSplitMaxTiles = 1536;

// One Langevin step (local step = state.step + kstep) of every job that owns
// a tile.  max_blocks caps the persistent grid (0 = one block per 4 tiles).
// Jobs flagged lds_step are stepped by the LDS kernel over `units` (first
// segment, segment count) of `segs` (job slot, first row, rows, LDS offset
// in float4; lds_beads = the largest LDS use of a unit), the others by the
// tile kernel (launched when any_global is set).  With shape.split_rows set
// (split_global) the LDS-step (other) jobs are stepped by k_step_rows over the
// tiles instead, from the step records `descs` (one: the record, in host
// memory, where the launch has a single job; else null).
hipError_t launch_step(const DevJob* jobs, const StepDesc* descs, const StepDesc* one, const DevJobState* st,
                       const int2* tiles, int ntiles, int any_global,
                       const int2* units, const int4* segs, int nunits, int lds_beads, int kstep, int max_blocks,
                       hipStream_t stream, const StepShape& shape);
// List rebuilds for jobs whose cadence is due (force != 0: rebuild all).
// boxes: jobs with tile boxes build their possible list by them (BOXES_NEAR) or,
// the wide ones, by their cell grid (BOXES_WIDE, cell_words bitmap words --
// ceil(n/64) -- of the largest); 0: every job by the all-pairs scan.
// sunits/segs/nsunits/lds_beads: the LDS step plan (see launch_step), whose
// jobs get their possible lists scanned from LDS-staged coordinates
// (nsunits = 0: all jobs by the tile kernels); any_global: some job is
// outside that plan (the tile kernel is launched only then).
enum { BOXES_NEAR = 1, BOXES_WIDE = 2 };
hipError_t launch_possible(const DevJob* jobs, DevJobState* st, const int2* tiles, int ntiles, int njobs, int boxes,
                           int cell_words, int any_global, const int2* sunits, const int4* segs, int nsunits,
                           int lds_beads, int force, hipStream_t stream, const StepShape& shape);
// Largest cell_words launch_possible accepts (the LDS bitmap of one wavefront).
constexpr int kMaxCellWords = 8192;
// The rows of units (job, first row) re-sorted by list length, where due.
hipError_t launch_sort_rows(const DevJob* jobs, DevJobState* st, const int2* units, int nunits, int force,
                            hipStream_t stream, const StepShape& shape);
// any_idx32: some job of the launch stores its lists as int32 (n >= 65536).
// units (job, first row) of the jobs whose rows are re-sorted first;
// sunits/segs/nsunits/lds_beads: the LDS step plan (see launch_step), whose
// jobs get their lists built from LDS-staged coordinates (nsunits = 0: all
// jobs by the tile kernel); any_global: some job is outside that plan.
hipError_t launch_verlet(const DevJob* jobs, DevJobState* st, const int2* tiles, int ntiles, int any_idx32,
                         int any_global, const int2* units, int nunits, const int2* sunits, const int4* segs,
                         int nsunits, int lds_beads, int force, hipStream_t stream, const StepShape& shape);
// Per-job updaters at a block start, and the step counter advance.
hipError_t launch_job_update(const DevJob* jobs, DevJobState* st, int njobs, hipStream_t stream, int mask = 7);
// A job's current coordinates (n beads) into pinned host memory: the kernel
// takes the buffer by the job's step on the device, so one launch and one wait
// replace reading the state first, and stores `ticket` to *done (pinned host
// memory) behind them.  One read takes 12 us at 22 beads, 17 at 1,000 and 31
// at 16,384; the state's copy, then the coordinates', 26, 33 and 43.  Past
// kStageBeads the copies stay: the gap closes and the staging memory grows.
constexpr int kStageBeads = 16384;
hipError_t launch_read_coords(const DevJob* job, const DevJobState* st, int n, float4* host, unsigned* done,
                              unsigned ticket, hipStream_t stream);
hipError_t launch_job_advance(const DevJob* jobs, DevJobState* st, int njobs, int nsteps, hipStream_t stream);
// Output / parity hooks.
hipError_t launch_energies(const DevJob* jobs, const DevJobState* st, int job, int n, hipStream_t stream);
// Steps state.step + kstep .. + nsteps - 1 of njobs jobs of at most `beads`
// beads, R = 8 or 16 rows per wavefront (ceil(beads / R) <= 16), in one launch,
// which then adds `advance` to the step counters.  begin: the launch starts with
// the pulling and heating updaters and the Verlet lists of the jobs due.
enum { BLOCK_UPDATE = 1, BLOCK_VERLET = 2 };
hipError_t launch_block_rows(const DevJob* jobs, const StepDesc* descs, DevJobState* st, int njobs, int beads, int R,
                             int kstep, int nsteps, int advance, int begin, hipStream_t stream);
// Forces only (the step kernels' force terms, no state change) of the jobs
// of the given tiles / LDS plan, into out[bead] (one job per launch).
hipError_t launch_forces(const DevJob* jobs, const StepDesc* descs, const StepDesc* one, const DevJobState* st,
                         const int2* tiles, int ntiles, int any_global,
                         const int2* units, const int4* segs, int nunits, int lds_beads, float4* out,
                         hipStream_t stream, const StepShape& shape);
hipError_t launch_rng_probe(uint4* state, int n, int count, int gaussian, float* out, hipStream_t stream);
// Counts (into *bad, device) the b bit patterns in [lo, hi) times numerators
// a[0..na) (device) whose short division differs from the IEEE quotient.
hipError_t launch_division_check(unsigned lo, unsigned hi, const float* a, int na, unsigned long long* bad,
                                 hipStream_t stream);
const void* step_kernel_symbol();
hipError_t launch_copy(const float4* src, float4* dst, size_t n, hipStream_t stream);

}  // namespace sop
