// kernels.h -- launch tables shared by kernels.hip and runtime.hip.
#pragma once
#include <hip/hip_runtime.h>
#include "rig.h"

namespace sister {

enum Stage {
    kStageCensus = 0,
    kStageWta,          // WTA: the rows of frames 0/2
    kStageWtaV,         // the rows of frames 1/3
    kStageWtaFill,      // the WTA maps' deep padding bands, copied from their first rows
    kStageMedianPrep,
    kStageMask,
    kNumStages
};

// Launches whose code depends on the disparity count (cost sum, SGM) run per
// group of rigs with the same D.
enum GroupKernel {
    kGPaths = 0,                          // SGM chains (ahead of the fused sweep: the rows family's)
    kGWinner,                             // S and the winner from the chains' bytes
    kGCost,                               // cost sum, per tile
    kGVSweep,                             // fused vertical SGM families, per column block
    kNumGroupKernels
};
struct DGroup {
    const RigDesc* rigs;     // device pointer to the group's first rig
    int nrig;
    int D, Dp;
    const int* bs[kNumGroupKernels];   // block starts per kernel, nrig+1 entries each
    int blocks[kNumGroupKernels];
    int vcols;               // fused vertical sweep: owned columns per block (0: separate families)
    int maxHp;               // tallest padded rig of the group
    int joined;              // paths: some family of some rig in the joined form
};
constexpr int kMaxDGroups = 16;

// Everything one launch of a stage needs for a set of rigs (device pointers).
struct LaunchSet {
    const RigDesc* rigs;
    int nrig;
    const int* bs[kNumStages];      // block-start tables, nrig+1 entries each
    int blocks[kNumStages];         // total blocks per stage
    uint64_t* const* scratch;       // per rig: 8 median order-statistic maps
    int maxD;
    int maxCols;                    // max frame width over the rigs
    int med_waves;                  // waves per block of k_median
    int maxWp, maxHp;               // max padded width / height over the rigs
    int ngroups;
    DGroup groups[kMaxDGroups];
};

// individual kernels, for per-kernel event timing
enum KernelId {
    kKCensus = 0, kKWta, kKMedianPrep, kKMedianSerial, kKMask, kKMsum,
    kKRows, kKPaths, kKWinner, kKVSweep, kNumKernels
};
extern const char* const kKernelNames[kNumKernels];

// optional hook called around every kernel launch
struct KernelTimer {
    virtual void begin(int kernel, hipStream_t st) = 0;
    virtual void end(int kernel, hipStream_t st) = 0;
    virtual ~KernelTimer() {}
    long dispatched[kNumKernels] = {};   // kernel dispatches issued, per kernel
};

void stage_blocks(const RigDesc& g, int out[kNumStages]);
int wta_fill_blocks(const RigDesc& g);
int wta_setup(int lds_limit);
// paths.hip: blocks of the chains of a rig's first nfam families (whole: over
// the padded frame, debug sums) and of the winner
int path_blocks(const RigDesc& g, int nfam, bool whole);
int winner_blocks(const RigDesc& g, bool whole);
size_t path_state_total(int W, int H, int D, int f);
int path_waves(int W, int H, int f);
int cost_blocks(const RigDesc& g);
int path_pairs(int Dp);   // pairs of disparities per lane (16 lanes) of the path kernels
// fused vertical sweep: owned columns per block for a group whose rigs have
// `cols` padded columns in all and disparity count D (0: not used)
int vsweep_pick_cols(long cols, int D, int choice);
bool vsweep_in_place(int D);
int vsweep_blocks(const RigDesc& g, int vcols);
// per-device set-up of kernel attributes (dynamic LDS above 64 KB); call with
// the device current.  0 on success.
int kernels_setup(int device);
void launch_census(const LaunchSet& ls, hipStream_t st, KernelTimer* t);
void launch_wta(const LaunchSet& ls, hipStream_t st, KernelTimer* t);
int median_setup(int lds_limit);
int median_waves(const RigDesc& g);
extern int g_num_cu;    // compute units of the device (kernels_setup)
void launch_median(const LaunchSet& ls, hipStream_t st, KernelTimer* t);
void launch_mask(const LaunchSet& ls, int fmask, hipStream_t st, KernelTimer* t);
void launch_msum(const LaunchSet& ls, int fuse, hipStream_t st, KernelTimer* t);
void launch_paths(const DGroup& G, int keep_sum, hipStream_t st);
void launch_winner(const DGroup& G, int mode, int keep_sum, hipStream_t st);
// keep_sum: also store the final S of every cell (debug)
void launch_sgm(const LaunchSet& ls, int mode, int keep_sum, hipStream_t st, KernelTimer* t);

}  // namespace sister
