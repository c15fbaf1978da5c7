// Sort key of a point in the device layout: track length, window, degree, first
// observation (the device order: the reference's elimination order, stably by
// track length); unobserved points last, as the all-ones key.
#ifndef MBA_POINT_KEY_H_
#define MBA_POINT_KEY_H_

#include <stdint.h>

#if defined(__HIPCC__)
#define MBA_POINT_KEY __host__ __device__
#else
#define MBA_POINT_KEY
#endif

namespace mba {

inline int bits_for(uint64_t largest) {
  int b = 0;
  while (b < 64 && (largest >> b) != 0) ++b;
  return b;
}

struct PointKey {
  int first_bits, deg_bits, win_bits, len_bits;
  // n observations, W windows, the largest degree and track of a point.
  PointKey(int64_t n, int32_t W, int32_t max_deg, int32_t max_track)
      : first_bits(bits_for((uint64_t)n)),
        deg_bits(bits_for((uint64_t)max_deg)),
        win_bits(bits_for((uint64_t)W - 1)),
        len_bits(bits_for((uint64_t)max_track + 1)) {}  // max_track + 1: unobserved
  MBA_POINT_KEY int bits() const { return first_bits + deg_bits + win_bits + len_bits; }
  // Whether it can be sorted on the device (millions of windows of many
  // observations in one call do not fit: the host's order is by comparison).
  bool fits() const { return bits() <= 64; }
};

}  // namespace mba

#endif  // MBA_POINT_KEY_H_
