// Host-side FR helpers of the product library (no GPU needed).
#pragma once

#include <cstdint>
#include <string>
#include <utility>
#include <vector>

#include "umpalumpa_amd.h"

namespace umpa::host {

// AFR::CreateConstants (afr.cpp:6-19)
umpa_fr_constants create_constants(uint64_t volumeX, uint64_t volumeY, uint64_t tableElems,
                                   const umpa_fr_settings &s);

// AFR::FillBlobTable (afr.cpp:22-34)
void fill_blob_table(float *table, uint64_t n, uint64_t volumeX, uint64_t volumeY,
                     const umpa_fr_settings &s);

// ComputeTraverseSpace (traverse_space_generator.hpp:94-145)
void compute_traverse_space(uint32_t imgSizeX, uint32_t imgSizeY, const float transform[9],
                            umpa_traverse_space &space, uint32_t maxVolumeIndexX,
                            uint32_t maxVolumeIndexYZ, bool useFast, float blobRadius,
                            float weight);

// Width of the unrolled candidate box for blob radius r: floor(2r) + 1 columns (with a margin
// for rounding at the blob edge; 2r where that is 3 or 5), clamped to the kernels' widths 3..6;
// wider footprints take the generic gather.
int footprint(const umpa_fr_settings &s);

// May the candidate box slide inside the slice (no per-candidate masking)?  Slices of at least
// footprint(s) pixels each way, and a footprint that holds the blob's whole bounding box.
bool box_can_shift(const umpa_fr_settings &s, uint64_t sliceX, uint64_t sliceY);

// One work item of the insertion kernel: the origin of an 8 x 8 x D brick of job `job`
// (z | job << 16) and w = D | heavy << 4 | parts << 8 | part << 16 (a brick split into `parts`
// slice ranges is accumulated by `parts` wavefronts, which merge their sums with atomics).
struct BrickOrigin {
  int x, y, z, w;
  float est;  // estimated cost, for ordering only
};

// Tunable knobs of the work-item schedule and of the kernel (the autotuner's search space).
struct SchedParams {
  float depthScale = 1.f;  // brick depth 8 / 4 / 2 / 1 beyond radius 48 / 24 / 12 times this
                           // (times the launch's own scale: *_depth_scale)
  bool priority = true;    // run bricks above a quarter of a wave's fair share at priority 2
  int maxParts = 16;       // split heavy bricks into at most this many slice ranges (fast math)
  float splitAt = 0.5f;    // ... when their cost exceeds splitAt times a wave's fair share
  int kernel = 0;          // UMPA_FR_KERNEL_*
  bool tableGlobal = false;  // blob table from global memory
  bool boxFixed = false;     // candidate box kept at the blob's bounding box
};

// The C struct's knobs in range (finite, positive scales; flags 0 / 1)?
bool sched_params_valid(const umpa_fr_sched_params &p);
SchedParams from_c(const umpa_fr_sched_params &p);
umpa_fr_sched_params to_c(const SchedParams &p);

// The bricks covering a vx*vy*vz volume with their estimated cost per inserted slice.
struct BrickCand {
  int x, y, z, d;
  float est;
};
// 8 x 8 x 8 blocks up to `core` from the centre are left out.
std::vector<BrickCand> brick_candidates(int vx, int vy, int vz, float depthScale = 1.f,
                                        float core = 0.f);
// The core radius of a volume for plain exact launches, and its cells of 2 x 2 x 2 voxels, two ints
// each: x | y << 16 and z.
float core_radius(int vx, int vy, int vz);
std::vector<int> core_cells(int vx, int vy, int vz, float core);

// Scale of the brick depths' radii: of a plain operation's launches of up to `spaces` spaces (what
// Init was told, which also decides shared cells: launches of fewer run the same schedule), by the
// blob (of the settings) and whether heavy bricks are split; of a volume in a batch's launch, by
// whether that is bounded and heavy bricks are split.
float plain_depth_scale(int vx, int vy, int vz, uint64_t spaces, const umpa_fr_settings &s,
                        bool split);
float batch_depth_scale(int vx, int vy, int vz, bool bounded, bool split);

// A volume's bricks sorted by estimated cost (heaviest first, ties in brick order) and the
// costs' sum: what make_schedule needs of a volume, built once per volume shape.
struct BrickSet {
  std::vector<BrickCand> sorted;
  double estSum = 0;
};
BrickSet make_brick_set(int vx, int vy, int vz, float depthScale = 1.f, float core = 0.f);

// The bricks of one job in a launch, `scale` = slices the launch inserts for it.
struct JobWork {
  const BrickSet *set;
  int job;
  double scale;
};

// Work items of one launch over several jobs, heaviest first (equal costs in job order, then
// brick order).  `splitHeavy` splits the heaviest bricks' slice ranges (changes the summation
// order: fast-math strategies only).
std::vector<BrickOrigin> make_schedule(const std::vector<JobWork> &jobs, bool splitHeavy,
                                       const SchedParams &sp = SchedParams());
// The same into `out` (its storage reused from call to call).
void make_schedule(const std::vector<JobWork> &jobs, bool splitHeavy, const SchedParams &sp,
                   std::vector<BrickOrigin> &out);

// make_schedule for a single job
std::vector<BrickOrigin> make_brick_schedule(int vx, int vy, int vz, bool splitHeavy,
                                             const SchedParams &sp = SchedParams(),
                                             float core = 0.f);

// The blocks covering a volume, the costliest first, two ints each: x | y << 16 and z | edge << 16
// (the small-problem kernel's work items).  With `share` (share_cells: by volume, spaces and blob)
// those at the centre are of 4 x 2 x 2 voxels, edge 2, whose cells four wavefronts share.
bool share_cells(int vx, int vy, int vz, uint64_t spaces, const umpa_fr_settings &s);
std::vector<int> make_cell_blocks(int vx, int vy, int vz, bool share);

// Persisted tuning results: one "key depthScale priority maxParts splitAt kernel tableGlobal
// boxFixed ms" line per key in $UMPA_TUNING_DIR/fr_tuning.txt (default
// $HOME/.cache/umpalumpa_amd); keys carry a tag, so lines of another format, or whose knobs meant
// other launches, are skipped.
bool tuning_cache_lookup(const std::string &key, SchedParams &out);
void tuning_cache_store(const std::string &key, const SchedParams &p, double ms);

// Rotation matrices (row-major 3x3, FP64) of the point group C_n or D_n ('C' / 'D'); the
// number is written to *count (n or 2n); out == nullptr only queries it.  0 on success.
int symmetry_operators(char family, int n, double *out, uint32_t cap, uint32_t *count);

// The autotuner's first-stage candidates for a strategy: exact, every schedule (no splitting)
// with every kernel knob; fast math, the schedules with default kernel knobs.
std::vector<SchedParams> tuning_candidates(bool fastMath);
// Second stage (fast math only, else empty): the kernel knobs over the schedule `base`.
std::vector<SchedParams> kernel_candidates(const SchedParams &base, bool fastMath);

// The first stage for an operation.  Where `cells` (its launch may be the small-problem kernel,
// which UMPA_FR_KERNEL_AUTO then means, whatever the schedule), the schedules name the brick kernel
// that AUTO means otherwise, so that what is timed is theirs.
std::vector<SchedParams> op_tuning_candidates(bool fastMath, bool half, bool cells);

// Keys of the tuning results: all that a launch of given knobs depends on.  An operation's: mode,
// precision and footprint, volume, launched spaces (to a power of two), and what Init decided by the
// spaces it was told of: the launch's own depth scale and shared cells.  A batch's: also whether its
// launches are bounded, and the first step's (volume, spaces), sorted.
std::string op_tuning_key(int numCUs, int mode, bool fastMath, bool half, int nb, int vx,
                          uint64_t spaces, float depthScale, bool sharedCells);
std::string batch_tuning_key(int numCUs, int mode, bool fastMath, bool half, int nb, bool bounded,
                             const std::vector<std::pair<int, int>> &shape);

// The kernel that UMPA_FR_KERNEL_AUTO means in a batch's launch (per pair where the carried queues
// do not cover the launch).
int batch_auto_kernel(bool fastMath, bool half, bool bounded);
// The batch tuner's first stage: the distinct schedules of tuning_candidates, all run by `kernel`,
// which fast math names; then (fast math only, else empty) the other kernel and boxes over the
// schedule `best`.
std::vector<SchedParams> batch_tuning_candidates(bool fastMath, int kernel);
std::vector<SchedParams> batch_kernel_candidates(const SchedParams &best, bool fastMath);

}  // namespace umpa::host
