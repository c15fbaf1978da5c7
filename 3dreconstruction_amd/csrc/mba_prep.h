// Device-side construction of a problem's index structures (mba_prep.hip):
// prefix sums, a stable radix sort, and the coupled-row-pair list of the
// explicit Schur complement.
#ifndef MBA_PREP_H_
#define MBA_PREP_H_

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <functional>
#include <string>
#include <vector>

#include "../../include/mba.h"

namespace mba {

// Sets the calling thread's message (mba_last_error).
void set_last_error(const std::string& msg);

// Device memory that outlives the call (the context's); the structure
// builders free what they use for themselves.
using DeviceAlloc = std::function<mba_status(void** out, size_t bytes)>;

// The blocks (fa, fb), fa >= fb, of the reduced camera matrix that points
// couple, and for each the pairs (a, b) of point-major rows of a common point
// with F blocks fa and fb (both orders when fa == fb), sorted by block and, in
// a block, by point and row.
struct SPairs {
  int64_t npairs = 0, nblk = 0, nitems = 0, nsplit = 0, nslots = 0, nmerged = 0;
  int2* pair = nullptr;                              // npairs
  int32_t *blk_fa = nullptr, *blk_fb = nullptr;      // nblk
  int32_t* blk_cross = nullptr;                      // nblk, grouped layout (else null)
  // Work items: a block, or a slice of at most split_pairs of its pairs,
  // whose sums go to scratch slot item_slot (-1: a whole block); blocks cut
  // into slices with their slots [split_lo, split_hi).
  int32_t *item_blk = nullptr, *item_slot = nullptr;
  int64_t *item_p0 = nullptr, *item_p1 = nullptr;
  int32_t *split_blk = nullptr, *split_lo = nullptr, *split_hi = nullptr;
  // Grouped layout: merged group rows (virtual rows nrows + m).
  int32_t *m_start = nullptr, *m_row = nullptr;
};

// The device layout of one call's problems, concatenated: rows (observations)
// grouped by point in the device point order, points in that order, and the
// camera-major order of the rows.
struct Layout {
  int32_t *row_cam = nullptr, *row_e = nullptr, *pt_start = nullptr, *e_to_pt = nullptr;
  int32_t* of_e = nullptr;     // window of each point block (several windows only)
  int32_t* cm_src = nullptr;   // camera-major slot -> row
  double *obs = nullptr, *pts = nullptr;  // rows' observations, points' positions
};

// Layout construction on the device, in two steps with a host decision in
// between.  measure() sorts the observations by point (descending observation
// index within a point) and reports what the Schur ordering is decided on;
// arrange(), given the order of the camera-side blocks, puts points, rows and
// camera-major rows in device order.
class LayoutBuilder {
 public:
  // All device arrays, problems concatenated; indices are global (a window's
  // cameras and points start at its offsets).
  struct In {
    hipStream_t stream = nullptr;
    int32_t W = 1, nc = 0, np = 0, ng = 0;
    int64_t n = 0;
    const int32_t *cam = nullptr, *pt = nullptr, *grp = nullptr;  // per observation (grp: grouped layout)
    const double *obs = nullptr, *pts = nullptr, *cams = nullptr, *intr = nullptr;
    int64_t ncams64 = 0, nintr64 = 0;                              // doubles in cams / intr
    const uint8_t *cam_const = nullptr, *grp_const = nullptr;      // or null
    const int32_t* pt_off = nullptr;                               // W + 1 (several windows)
  };
  // Per camera / group: distinct points of non-constant blocks (degree in the
  // Hessian graph but for camera-group edges), first observation (INT32_MAX:
  // none); per window the largest point degree and the observed points.  With
  // a track beyond kLayoutMaxTrack only max_track is meaningful.
  struct Stats {
    std::vector<int32_t> cam_deg, cam_first, grp_deg, grp_first, cam_grp, win_max_deg, win_points;
    int32_t max_track = 0;
    bool finite = true;       // every parameter is
    bool repeated = false;    // some camera observes a point twice
    bool two_groups = false;  // some camera is observed with two groups
  };
  explicit LayoutBuilder(const In& in);
  ~LayoutBuilder();
  mba_status measure(Stats* out);
  // cam_key: camera-major key of each camera (its F block, or -1: its rows
  // are left out), nkeys keys; nq > 1: each key's rows are also cut at the
  // bounds of nq point ranges of equal row count (split: nq + 1 bounds per
  // key).  track_hist: points per track length (0: unobserved).
  mba_status arrange(const std::vector<int32_t>& cam_key, int32_t nkeys, int32_t nq, int32_t max_deg,
                     const DeviceAlloc& alloc, Layout* out, std::vector<int32_t>* split,
                     std::vector<int32_t>* track_hist);

 private:
  struct State;
  State* st_;
};

// Longest track the builder takes (a thread walks a point's rows).
constexpr int32_t kLayoutMaxTrack = 512;

// Items 0 .. n - 1 listed by bucket (in order within one): start (nbuckets + 1)
// and list, allocated by `alloc`.
mba_status bucket_lists(hipStream_t s, int64_t n, const int32_t* bucket, int32_t nbuckets, const DeviceAlloc& alloc,
                        int32_t** start, int32_t** list);

struct SPairsIn {
  hipStream_t stream = nullptr;
  int32_t ne = 0, nf = 0, nc = 0, nrows = 0;
  int32_t f_span = 0;  // the most F blocks of one problem
  bool grouped = false;
  const int32_t *pt_start = nullptr, *row_cam = nullptr, *cam_to_f = nullptr, *cam_gf = nullptr, *f_to_cam = nullptr;
  int64_t split_pairs = 0;
};

mba_status build_s_pairs(const SPairsIn& in, const DeviceAlloc& alloc, SPairs* out);

}  // namespace mba

#endif  // MBA_PREP_H_
