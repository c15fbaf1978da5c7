// Device-side construction of a problem's index structures (mba_prep.hip):
// prefix sums, a stable radix sort, and the coupled-row-pair list of the
// explicit Schur complement.
#ifndef MBA_PREP_H_
#define MBA_PREP_H_

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <functional>
#include <string>

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
  // Grouped layout: merged group rows (virtual rows 2 nrows + m).
  int32_t *m_start = nullptr, *m_row = nullptr;
};

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
