// Device-side construction of a problem's index structures: exclusive prefix
// sums, a stable least-significant-digit radix sort, and the coupled-row-pair
// list of the explicit Schur complement.  Everything is deterministic: the
// same problem gives the same order whatever the launch's timing.
#include "mba_prep.h"

#include "mba_point_key.h"
#include "mba_pool.h"

#include <algorithm>
#include <string>
#include <vector>

namespace mba {
namespace {

constexpr int kThreads = 256, kWaves = kThreads / 64;
constexpr int kPer = 16, kTile = kThreads * kPer;  // items per thread and per workgroup of a sweep

mba_status fail(mba_status s, const std::string& msg) {
  set_last_error(msg);
  return s;
}
#define PREP_TRY(expr)                                                                      \
  do {                                                                                      \
    const hipError_t e_ = (expr);                                                           \
    if (e_ != hipSuccess)                                                                   \
      return fail(e_ == hipErrorOutOfMemory ? MBA_ERR_OUT_OF_MEMORY : MBA_ERR_DEVICE,       \
                  std::string(#expr) + ": " + hipGetErrorString(e_));                       \
  } while (0)
#define PREP_OK(expr)            \
  do {                           \
    const mba_status s_ = (expr); \
    if (s_ != MBA_OK) return s_; \
  } while (0)

inline unsigned blocks_of(int64_t n, int64_t per) { return (unsigned)std::max<int64_t>(1, (n + per - 1) / per); }

// Temporaries of one build, given back when it ends, after the stream has
// drained.
struct Temps {
  DevicePool mem;
  hipStream_t s;
  explicit Temps(hipStream_t stream) : s(stream) {}
  ~Temps() {
    (void)hipStreamSynchronize(s);
    mem.release();
  }
  template <typename X>
  mba_status get(X** out, size_t n) {
    void* p = nullptr;
    PREP_TRY(mem.raw(&p, std::max<size_t>(1, n) * sizeof(X)));
    *out = (X*)p;
    return MBA_OK;
  }
};

template <typename X>
mba_status keep(const DeviceAlloc& alloc, X** out, size_t n) {
  void* p = nullptr;
  PREP_OK(alloc(&p, std::max<size_t>(1, n) * sizeof(X)));
  *out = (X*)p;
  return MBA_OK;
}

// ------------------------------------------------------------ prefix sums
// Inclusive scan over a wave.
template <typename A>
__device__ __forceinline__ A wave_scan(A v) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const A u = __shfl_up(v, o, 64);
    if (lane >= o) v += u;
  }
  return v;
}
// Exclusive scan of one value per thread over the workgroup (lds: kWaves
// values); *total receives the sum.  Two barriers.
template <typename A>
__device__ __forceinline__ A block_scan(A v, A* lds, A* total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const A inc = wave_scan(v);
  if (lane == 63) lds[wave] = inc;
  __syncthreads();
  A base = A(0), sum = A(0);
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    if (w < wave) base += lds[w];
    sum += lds[w];
  }
  __syncthreads();
  *total = sum;
  return base + inc - v;
}

// Exclusive scan out[0..n) of in[0..n) (in and out may be the same array),
// the total to out[n].  Sweep 1 sums tiles, sweep 3 scans them from the
// scanned tile sums; each thread takes kPer consecutive values.
template <typename V, typename A>
__global__ __launch_bounds__(kThreads) void k_scan_sums(int64_t n, const V* __restrict__ in, A* __restrict__ sums) {
  __shared__ A lds[kWaves];
  const int64_t b = blockIdx.x * (int64_t)kTile;
  A v = A(0);
  for (int k = 0; k < kPer; ++k) {
    const int64_t i = b + k * kThreads + threadIdx.x;
    if (i < n) v += (A)in[i];
  }
  A total;
  (void)block_scan(v, lds, &total);
  if (threadIdx.x == 0) sums[blockIdx.x] = total;
}
template <typename V, typename A>
__global__ __launch_bounds__(kThreads) void k_scan_tiles(int64_t n, const V* in, const A* __restrict__ base, A* out) {
  __shared__ A lds[kWaves];
  __shared__ A tile[kTile + kTile / 16];  // padded: thread t reads kPer values from kPer t
  const int64_t b = blockIdx.x * (int64_t)kTile;
  for (int k = 0; k < kPer; ++k) {
    const int i = k * kThreads + threadIdx.x;
    tile[i + (i >> 4)] = b + i < n ? (A)in[b + i] : A(0);
  }
  __syncthreads();
  A v[kPer], sum = A(0);
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int i = kPer * threadIdx.x + k;
    v[k] = tile[i + (i >> 4)];
    sum += v[k];
  }
  A total;
  A run = block_scan(sum, lds, &total) + (base ? base[blockIdx.x] : A(0));
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int i = kPer * threadIdx.x + k;
    tile[i + (i >> 4)] = run;
    run += v[k];
  }
  __syncthreads();
  for (int k = 0; k < kPer; ++k) {
    const int i = k * kThreads + threadIdx.x;
    if (b + i < n) out[b + i] = tile[i + (i >> 4)];
  }
  if (threadIdx.x == kThreads - 1 && b + kTile >= n) out[n] = run;
}
template <typename V, typename A>
mba_status scan(Temps& t, int64_t n, const V* in, A* out) {
  const unsigned nb = blocks_of(n, kTile);
  A* sums = nullptr;
  if (nb > 1) {
    PREP_OK(t.get(&sums, (size_t)nb + 1));
    hipLaunchKernelGGL((k_scan_sums<V, A>), dim3(nb), dim3(kThreads), 0, t.s, n, in, sums);
    PREP_OK((scan<A, A>(t, nb, sums, sums)));
  }
  hipLaunchKernelGGL((k_scan_tiles<V, A>), dim3(nb), dim3(kThreads), 0, t.s, n, in, (const A*)sums, out);
  PREP_TRY(hipGetLastError());
  return MBA_OK;
}

// -------------------------------------------------------------- radix sort
// Stable sort of (key, value) by key bits [0, bits), digits of up to 8 bits.
// A pass counts each 4,096-item tile's digits (hist[digit][tile]), scans the
// counts, and scatters: within a tile an item's rank among its digit's items
// comes from per-wave counters and, inside 64 items, from the lanes that hold
// the same digit (a ballot per digit bit); the tile is put in digit order in
// LDS first so that the stores run along the digits' destinations.
// Memory bound: a pass reads the keys twice and moves key and value once.
constexpr int kDigits = 256;
template <typename K>
__global__ __launch_bounds__(kThreads) void k_sort_hist(int64_t n, const K* __restrict__ key, int shift,
                                                        uint32_t mask, int64_t ntiles, uint32_t* __restrict__ hist) {
  __shared__ uint32_t cnt[kWaves][kDigits];
  for (int w = 0; w < kWaves; ++w) cnt[w][threadIdx.x] = 0;
  __syncthreads();
  const int64_t b = blockIdx.x * (int64_t)kTile;
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int64_t i = b + k * kThreads + threadIdx.x;
    if (i < n) atomicAdd(&cnt[threadIdx.x >> 6][(uint32_t)(key[i] >> shift) & mask], 1u);
  }
  __syncthreads();
  if (threadIdx.x <= mask) {
    uint32_t s = 0;
    for (int w = 0; w < kWaves; ++w) s += cnt[w][threadIdx.x];
    hist[(int64_t)threadIdx.x * ntiles + blockIdx.x] = s;
  }
}

template <typename K, typename P>
__global__ __launch_bounds__(kThreads) void k_sort_scatter(int64_t n, const K* __restrict__ key,
                                                           const P* __restrict__ val, int shift, uint32_t mask,
                                                           int nbits, int64_t ntiles,
                                                           const uint32_t* __restrict__ offs,
                                                           K* __restrict__ key_out, P* __restrict__ val_out) {
  __shared__ uint32_t cnt[kWaves][kDigits];  // counts, then each wave's first place per digit
  __shared__ uint32_t start[kDigits];        // the digit's first place in the tile
  __shared__ uint32_t gbase[kDigits];
  __shared__ uint32_t lds[kWaves];
  __shared__ K lk[kTile];
  __shared__ P lv[kTile];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int w = 0; w < kWaves; ++w) cnt[w][threadIdx.x] = 0;
  __syncthreads();
  // Wave w takes the tile's items [1024 w, 1024 (w + 1)), 64 at a time.
  const int64_t b = blockIdx.x * (int64_t)kTile + wave * (kTile / kWaves);
  K k[kPer];
  P v[kPer];
  uint16_t rank[kPer];
#pragma unroll
  for (int q = 0; q < kPer; ++q) {
    const int64_t i = b + 64 * q + lane;
    k[q] = i < n ? key[i] : K(0);
    if (i < n) v[q] = val[i];
  }
  const unsigned long long below = (1ull << lane) - 1ull;
#pragma unroll
  for (int q = 0; q < kPer; ++q) {
    const bool on = b + 64 * q + lane < n;
    const uint32_t d = (uint32_t)(k[q] >> shift) & mask;
    unsigned long long peers = __ballot(on);
    for (int bit = 0; bit < nbits; ++bit) {
      const unsigned long long set = __ballot((d >> bit) & 1u);
      peers &= ((d >> bit) & 1u) ? set : ~set;
    }
    if (on) {
      rank[q] = (uint16_t)(cnt[wave][d] + __popcll(peers & below));
      __builtin_amdgcn_wave_barrier();
      if ((peers & below) == 0ull) cnt[wave][d] += (uint32_t)__popcll(peers);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
  __syncthreads();
  {
    const uint32_t d = threadIdx.x;
    uint32_t c[kWaves], sum = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      c[w] = cnt[w][d];
      sum += c[w];
    }
    uint32_t total;
    uint32_t run = block_scan(sum, lds, &total);
    start[d] = run;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      cnt[w][d] = run;
      run += c[w];
    }
    gbase[d] = d <= mask ? offs[(int64_t)d * ntiles + blockIdx.x] : 0u;
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < kPer; ++q)
    if (b + 64 * q + lane < n) {
      const uint32_t at = cnt[wave][(uint32_t)(k[q] >> shift) & mask] + rank[q];
      lk[at] = k[q];
      lv[at] = v[q];
    }
  __syncthreads();
  const int m = (int)min((int64_t)kTile, n - blockIdx.x * (int64_t)kTile);
  for (int i = threadIdx.x; i < m; i += kThreads) {
    const K kk = lk[i];
    const uint32_t d = (uint32_t)(kk >> shift) & mask;
    const size_t dst = (size_t)gbase[d] + (uint32_t)(i - (int)start[d]);
    key_out[dst] = kk;
    val_out[dst] = lv[i];
  }
}

// Sorts key[0] / val[0] (n < 2^32 items) with key[1] / val[1] as the other
// buffers; returns which of the two holds the result.
template <typename K, typename P>
mba_status radix_sort(Temps& t, int64_t n, int bits, K* const key[2], P* const val[2], int* where) {
  *where = 0;
  if (n <= 1 || bits == 0) return MBA_OK;
  const int passes = (bits + 7) / 8;
  const int64_t ntiles = (n + kTile - 1) / kTile;
  uint32_t* hist = nullptr;
  const int width = (bits + passes - 1) / passes;
  PREP_OK(t.get(&hist, (size_t)ntiles * ((size_t)1 << width) + 1));
  for (int p = 0, shift = 0; p < passes; ++p, shift += width) {
    const int nb = std::min(width, bits - shift);
    const uint32_t mask = (1u << nb) - 1u;
    const int a = *where;
    hipLaunchKernelGGL(k_sort_hist<K>, dim3((unsigned)ntiles), dim3(kThreads), 0, t.s, n, (const K*)key[a], shift,
                       mask, ntiles, hist);
    PREP_OK((scan<uint32_t, uint32_t>(t, ntiles * (int64_t)(mask + 1), hist, hist)));
    hipLaunchKernelGGL((k_sort_scatter<K, P>), dim3((unsigned)ntiles), dim3(kThreads), 0, t.s, n, (const K*)key[a],
                       (const P*)val[a], shift, mask, nb, ntiles, (const uint32_t*)hist, key[1 - a], val[1 - a]);
    *where = 1 - a;
  }
  PREP_TRY(hipGetLastError());
  return MBA_OK;
}

// ---------------------------------------------------------------- layout
// key[k] = bucket of item k (reversed: of item n - 1 - k), val[k] = the item.
template <bool kReverse>
__global__ __launch_bounds__(kThreads) void k_keys(int64_t n, const int32_t* __restrict__ bucket,
                                                   uint32_t* __restrict__ key, uint32_t* __restrict__ val) {
  const int64_t k = blockIdx.x * (int64_t)kThreads + threadIdx.x;
  if (k >= n) return;
  const int64_t i = kReverse ? n - 1 - k : k;
  key[k] = (uint32_t)bucket[i];
  val[k] = (uint32_t)i;
}
// First place of every key 0 .. nkeys in sorted keys (start[nkeys] = n).
__global__ __launch_bounds__(kThreads) void k_bounds(int64_t n, const uint32_t* __restrict__ key, int32_t nkeys,
                                                     int32_t* __restrict__ start) {
  const int64_t k = blockIdx.x * (int64_t)kThreads + threadIdx.x;
  if (k > n) return;
  const int64_t prev = k > 0 ? (int64_t)key[k - 1] : -1;
  const int64_t cur = k < n ? (int64_t)key[k] : nkeys;
  for (int64_t q = prev + 1; q <= cur && q <= nkeys; ++q) start[q] = (int32_t)k;
}

// Counters of measure(), in one array: [cam_deg nc | cam_first nc | grp_deg ng
// | grp_first ng | grp_lo nc | grp_hi nc (grouped) | win_max W | win_points W |
// max_track | bad | repeated].
struct StatsAt {
  int32_t nc, ng, W;
  __host__ __device__ int64_t cam_first() const { return nc; }
  __host__ __device__ int64_t grp_deg() const { return 2 * (int64_t)nc; }
  __host__ __device__ int64_t grp_first() const { return grp_deg() + ng; }
  __host__ __device__ int64_t grp_lo() const { return grp_first() + ng; }
  __host__ __device__ int64_t grp_hi() const { return grp_lo() + (ng ? nc : 0); }
  __host__ __device__ int64_t win_max() const { return grp_hi() + (ng ? nc : 0); }
  __host__ __device__ int64_t win_points() const { return win_max() + W; }
  __host__ __device__ int64_t max_track() const { return win_points() + W; }
  __host__ __device__ int64_t bad() const { return max_track() + 1; }
  __host__ __device__ int64_t repeated() const { return max_track() + 2; }
  __host__ __device__ int64_t size() const { return max_track() + 3; }
};
__global__ __launch_bounds__(kThreads) void k_stats_init(StatsAt at, int32_t* __restrict__ s) {
  for (int64_t i = blockIdx.x * (int64_t)kThreads + threadIdx.x; i < at.size(); i += (int64_t)gridDim.x * kThreads) {
    const bool big = (i >= at.cam_first() && i < at.grp_deg()) || (i >= at.grp_first() && i < at.grp_hi());
    s[i] = big ? INT32_MAX : (i >= at.grp_hi() && i < at.win_max() ? -1 : 0);
  }
}
__global__ __launch_bounds__(kThreads) void k_finite(int64_t n, const double* __restrict__ v, int32_t* __restrict__ bad) {
  int any = 0;
  for (int64_t i = blockIdx.x * (int64_t)kThreads + threadIdx.x; i < n; i += (int64_t)gridDim.x * kThreads)
    any |= !isfinite(v[i]);
  if (any) *bad = 1;
}
// Atomic minimum / maximum, skipped when a (possibly stale) read shows that it
// would change nothing.
__device__ __forceinline__ void lower(int32_t* p, int32_t v) {
  if (v < *p) atomicMin(p, v);
}
__device__ __forceinline__ void raise(int32_t* p, int32_t v) {
  if (v > *p) atomicMax(p, v);
}
// Cameras (and groups) counted in LDS.
constexpr int kLdsBlocks = 4096;
// The least and greatest group of each camera's observations: per workgroup in
// LDS if there are at most kLdsBlocks cameras (every observation compared with
// the one value in memory: 320 us at 600,000 observations of 300 cameras,
// mostly the first ones' atomics on the same words; 16).
template <bool kLds>
__global__ __launch_bounds__(kThreads) void k_cam_groups(int64_t n, const int32_t* __restrict__ cam,
                                                         const int32_t* __restrict__ grp, StatsAt at,
                                                         int32_t* __restrict__ s) {
  __shared__ int32_t lo[kLds ? kLdsBlocks : 1], hi[kLds ? kLdsBlocks : 1];
  if (kLds) {
    for (int c = threadIdx.x; c < at.nc; c += kThreads) {
      lo[c] = INT32_MAX;
      hi[c] = -1;
    }
    __syncthreads();
  }
  for (int64_t i = blockIdx.x * (int64_t)kThreads + threadIdx.x; i < n; i += (int64_t)gridDim.x * kThreads) {
    const int c = cam[i], g = grp[i];
    lower(kLds ? lo + c : s + at.grp_lo() + c, g);
    raise(kLds ? hi + c : s + at.grp_hi() + c, g);
  }
  if (kLds) {
    __syncthreads();
    for (int c = threadIdx.x; c < at.nc; c += kThreads) {
      if (hi[c] < 0) continue;
      lower(s + at.grp_lo() + c, lo[c]);
      raise(s + at.grp_hi() + c, hi[c]);
    }
  }
}

// Window of point p.
__device__ __forceinline__ int window_of(int p, const int32_t* __restrict__ off, int W) {
  int lo = 0, hi = W;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (off[mid] <= p) lo = mid;
    else hi = mid;
  }
  return lo;
}

// A thread walks its points' rows: the point's degree (distinct non-constant
// cameras and groups it meets), its first observation (the list's last), and
// the cameras' and groups' degrees and first observations.  The latter are
// counted in LDS (thousands of observations share a camera): all cameras and
// groups if they are at most kLdsBlocks, else (ranged; a batch of windows,
// whose points and cameras are numbered window by window) the range of
// cameras that the workgroup's points meet if it fits, else in global memory
// (2.0 ms at 512 windows of 40 cameras, 1.1 with ranges).  Whether a row's
// camera came before in the point is looked up only when its bit in a 128-bit
// hash of the cameras so far is set (4.0M rows: 465 us with the look-up for
// every row, 268).
template <bool kLds>
__global__ __launch_bounds__(kThreads) void k_point_stats(
    int np, const int32_t* __restrict__ pstart, const uint32_t* __restrict__ rows, const int32_t* __restrict__ cam,
    const int32_t* __restrict__ grp, const uint8_t* __restrict__ cam_const, const uint8_t* __restrict__ grp_const,
    const int32_t* __restrict__ pt_off, StatsAt at, int32_t* s, int32_t* __restrict__ pdeg, int ranged) {
  __shared__ int32_t l_deg[kLds ? kLdsBlocks : 1], l_first[kLds ? kLdsBlocks : 1];
  __shared__ int32_t l_range[2];
  // The workgroup's points.
  const int tiles = (np + kThreads - 1) / kThreads, per = (tiles + (int)gridDim.x - 1) / (int)gridDim.x;
  const int64_t p0 = (int64_t)per * kThreads * blockIdx.x;
  const int p1 = (int)(p0 + (int64_t)per * kThreads < np ? p0 + (int64_t)per * kThreads : np);
  int base = 0, nb = at.nc + at.ng;  // cameras, then groups
  bool lds = kLds;
  if (kLds && ranged) {
    if (threadIdx.x == 0) {
      l_range[0] = INT32_MAX;
      l_range[1] = -1;
    }
    __syncthreads();
    int lo = INT32_MAX, hi = -1;
    if (p0 < p1)
      for (int r = pstart[p0] + (int)threadIdx.x; r < pstart[p1]; r += kThreads) {
        const int c = cam[rows[r]];
        lo = min(lo, c);
        hi = max(hi, c);
      }
    atomicMin(&l_range[0], lo);
    atomicMax(&l_range[1], hi);
    __syncthreads();
    base = l_range[0];
    nb = l_range[1] < 0 ? 0 : l_range[1] - base + 1;
    lds = nb <= kLdsBlocks;
  }
  if (kLds && lds) {
    for (int i = threadIdx.x; i < nb; i += kThreads) {
      l_deg[i] = 0;
      l_first[i] = INT32_MAX;
    }
    __syncthreads();
  }
  auto add = [&](int b) {
    if (kLds && lds) atomicAdd(&l_deg[b - base], 1);
    else atomicAdd(s + (b < at.nc ? b : at.grp_deg() + (b - at.nc)), 1);
  };
  auto seen_at = [&](int b, int i) {
    if (kLds && lds) {
      if (i < l_first[b - base]) atomicMin(&l_first[b - base], i);
    } else {
      lower(s + (b < at.nc ? at.cam_first() + b : at.grp_first() + (b - at.nc)), i);
    }
  };
  for (int p = (int)p0 + (int)threadIdx.x; p < p1; p += kThreads) {
    const int r0 = pstart[p], r1 = pstart[p + 1];
    int deg = 0;
    unsigned long long met[2] = {0, 0};
    const int rend = r1 - r0 > kLayoutMaxTrack ? r0 : r1;  // too long a walk: the host's path
    for (int r = r0; r < rend; ++r) {
      const int i = (int)rows[r], c = cam[i];
      seen_at(c, i);
      bool rep = false;
      const unsigned h = (unsigned)c * 2654435769u >> 25;
      const unsigned long long bit = 1ull << (h & 63);
      if ((h < 64 ? met[0] : met[1]) & bit)
        for (int q = r0; q < r && !rep; ++q) rep = cam[rows[q]] == c;
      if (h < 64) met[0] |= bit;
      else met[1] |= bit;
      if (rep) s[at.repeated()] = 1;
      if (!rep && !(cam_const && cam_const[c])) {
        ++deg;
        add(c);
      }
      if (grp) {
        const int g = grp[i];
        seen_at(at.nc + g, i);
        bool again = grp_const && grp_const[g];
        for (int q = r0; q < r && !again; ++q) again = grp[rows[q]] == g;
        if (!again) {
          ++deg;
          add(at.nc + g);
        }
      }
    }
    pdeg[p] = deg;
    if (r1 > r0) {
      const int w = pt_off ? window_of(p, pt_off, at.W) : 0;
      raise(s + at.win_max() + w, deg);
      raise(s + at.max_track(), r1 - r0);
      if (pt_off) atomicAdd(s + at.win_points() + w, 1);
    }
  }
  if (kLds && lds) {
    __syncthreads();
    for (int i = threadIdx.x; i < nb; i += kThreads) {
      const int b = base + i;
      if (l_deg[i]) atomicAdd(s + (b < at.nc ? b : at.grp_deg() + (b - at.nc)), l_deg[i]);
      if (l_first[i] != INT32_MAX)
        atomicMin(s + (b < at.nc ? at.cam_first() + b : at.grp_first() + (b - at.nc)), l_first[i]);
    }
  }
}

__global__ __launch_bounds__(kThreads) void k_point_keys(int np, const int32_t* __restrict__ pstart,
                                                         const uint32_t* __restrict__ rows,
                                                         const int32_t* __restrict__ pdeg,
                                                         const int32_t* __restrict__ pt_off, int W, PointKey pk,
                                                         uint64_t* __restrict__ key, uint32_t* __restrict__ val,
                                                         int max_track, int32_t* __restrict__ hist) {
  __shared__ int32_t h[kLayoutMaxTrack + 1];
  for (int i = threadIdx.x; i <= max_track; i += kThreads) h[i] = 0;
  __syncthreads();
  for (int p = blockIdx.x * kThreads + threadIdx.x; p < np; p += gridDim.x * kThreads) {
    const int r0 = pstart[p], len = pstart[p + 1] - r0;
    uint64_t k = ~0ull;
    if (len > 0) {
      k = (uint64_t)len;
      k = (k << pk.win_bits) | (uint64_t)(pt_off ? window_of(p, pt_off, W) : 0);
      k = (k << pk.deg_bits) | (uint64_t)pdeg[p];
      k = (k << pk.first_bits) | (uint64_t)rows[r0 + len - 1];
    }
    key[p] = k;
    val[p] = (uint32_t)p;
    atomicAdd(&h[len], 1);
  }
  __syncthreads();
  for (int i = threadIdx.x; i <= max_track; i += kThreads)
    if (h[i]) atomicAdd(hist + i, h[i]);
}
__global__ __launch_bounds__(kThreads) void k_point_order(int ne, const uint32_t* __restrict__ perm,
                                                          const int32_t* __restrict__ pstart,
                                                          const double* __restrict__ pts_in,
                                                          const int32_t* __restrict__ pt_off, int W,
                                                          int32_t* __restrict__ e_to_pt, int32_t* __restrict__ len,
                                                          double* __restrict__ pts, int32_t* __restrict__ of_e) {
  const int e = blockIdx.x * kThreads + threadIdx.x;
  if (e >= ne) return;
  const int p = (int)perm[e];
  e_to_pt[e] = p;
  len[e] = pstart[p + 1] - pstart[p];
  for (int k = 0; k < 3; ++k) pts[3 * (size_t)e + k] = pts_in[3 * (size_t)p + k];
  if (of_e) of_e[e] = window_of(p, pt_off, W);
}
// Point of each row, and the row's place in the by-point list.
__global__ __launch_bounds__(kThreads) void k_row_points(int ne, const int32_t* __restrict__ pt_start,
                                                         int32_t* __restrict__ row_e) {
  // 16 lanes per point: short tracks fill a cache line together.
  const int64_t t = blockIdx.x * (int64_t)kThreads + threadIdx.x;
  const int e = (int)(t >> 4), sub = (int)(t & 15);
  if (e >= ne) return;
  for (int r = pt_start[e] + sub; r < pt_start[e + 1]; r += 16) row_e[r] = e;
}
__global__ __launch_bounds__(kThreads) void k_rows(int64_t n, const int32_t* __restrict__ row_e,
                                                   const int32_t* __restrict__ pt_start,
                                                   const int32_t* __restrict__ e_to_pt,
                                                   const int32_t* __restrict__ pstart,
                                                   const uint32_t* __restrict__ rows, const int32_t* __restrict__ cam,
                                                   const double2* __restrict__ obs_in,
                                                   const int32_t* __restrict__ cam_key, int32_t nkeys,
                                                   int32_t* __restrict__ row_cam, double2* __restrict__ obs,
                                                   uint32_t* __restrict__ key, uint32_t* __restrict__ val) {
  const int64_t r = blockIdx.x * (int64_t)kThreads + threadIdx.x;
  if (r >= n) return;
  const int e = row_e[r];
  const uint32_t i = rows[pstart[e_to_pt[e]] + ((int)r - pt_start[e])];
  const int c = cam[i];
  row_cam[r] = c;
  obs[r] = obs_in[i];
  const int k = cam_key[c];
  key[r] = (uint32_t)(k < 0 ? nkeys : k);
  val[r] = (uint32_t)r;
}
// First row of point range q = 1 .. nq - 1 (equal row counts), 0 and n at the
// ends.
__global__ void k_range_rows(int64_t n, int ne, const int32_t* __restrict__ pt_start, int nq,
                             int32_t* __restrict__ range_row) {
  const int q = threadIdx.x;
  if (q > nq) return;
  const int64_t target = n * q / nq;
  int lo = 0, hi = ne + 1;  // first e with pt_start[e] >= target
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (pt_start[mid] < target) lo = mid + 1;
    else hi = mid;
  }
  range_row[q] = q == 0 ? 0 : (q == nq ? (int32_t)n : pt_start[min(lo, ne)]);
}
__global__ __launch_bounds__(kThreads) void k_split(int32_t nkeys, int nq, const int32_t* __restrict__ start,
                                                    const uint32_t* __restrict__ cm_src,
                                                    const int32_t* __restrict__ range_row,
                                                    int32_t* __restrict__ split) {
  const int64_t t = blockIdx.x * (int64_t)kThreads + threadIdx.x;
  const int64_t f = t / (nq + 1);
  const int q = (int)(t % (nq + 1));
  if (f >= nkeys) return;
  int lo = start[f], hi = start[f + 1];
  if (q == nq) lo = hi;
  else if (q > 0) {
    const uint32_t bound = (uint32_t)range_row[q];
    while (lo < hi) {
      const int mid = lo + ((hi - lo) >> 1);
      if (cm_src[mid] < bound) lo = mid + 1;
      else hi = mid;
    }
  }
  split[t] = lo;
}

// ------------------------------------------------- coupled-row-pair list
// Virtual rows of the explicit S, point by point: the point's rows (in row
// order; F block -1 for a constant camera) and, in the grouped layout, one
// merged row per intrinsic group the point meets (summing the point's group
// parts in that group: Z is linear in the rows, so the group blocks of S pair
// merged rows).  v_f: F block, v_id: the row of the Z
// array it stands for (a merged row m: nrows + m), v_e: its point.

// Whether row r is the first of its point with its camera's group block.
__device__ __forceinline__ bool first_of_group(int r0, int r, int g, const int32_t* row_cam, const int32_t* cam_gf) {
  for (int q = r0; q < r; ++q)
    if (cam_gf[row_cam[q]] == g) return false;
  return true;
}
__global__ __launch_bounds__(kThreads) void k_merge_count(int ne, const int32_t* __restrict__ pt_start,
                                                          const int32_t* __restrict__ row_cam,
                                                          const int32_t* __restrict__ cam_gf,
                                                          uint32_t* __restrict__ nm, uint32_t* __restrict__ nr) {
  const int e = blockIdx.x * kThreads + threadIdx.x;
  if (e >= ne) return;
  uint32_t m = 0, k = 0;
  const int r0 = pt_start[e], r1 = pt_start[e + 1];
  for (int r = r0; r < r1; ++r) {
    const int g = cam_gf[row_cam[r]];
    if (g < 0) continue;
    ++k;
    m += first_of_group(r0, r, g, row_cam, cam_gf);
  }
  nm[e] = m;
  nr[e] = k;
}
__global__ __launch_bounds__(kThreads) void k_merge_fill(int ne, int nrows, const int32_t* __restrict__ pt_start,
                                                         const int32_t* __restrict__ row_cam,
                                                         const int32_t* __restrict__ cam_gf,
                                                         const uint32_t* __restrict__ m0,
                                                         const uint32_t* __restrict__ k0, int32_t* __restrict__ m_start,
                                                         int32_t* __restrict__ m_row, int32_t* __restrict__ v_f,
                                                         int32_t* __restrict__ v_id, int32_t* __restrict__ v_e) {
  const int e = blockIdx.x * kThreads + threadIdx.x;
  if (e >= ne) return;
  const int r0 = pt_start[e], r1 = pt_start[e + 1];
  uint32_t m = m0[e], k = k0[e];
  if (e == 0) m_start[0] = 0;
  for (int r = r0; r < r1; ++r) {
    const int g = cam_gf[row_cam[r]];
    if (g < 0 || !first_of_group(r0, r, g, row_cam, cam_gf)) continue;
    for (int q = r; q < r1; ++q)
      if (cam_gf[row_cam[q]] == g) m_row[k++] = q;
    const size_t v = (size_t)r1 + m;  // after the rows up to r1 and the merged rows before m
    v_f[v] = g;
    v_id[v] = nrows + (int)m;
    v_e[v] = e;
    m_start[++m] = (int)k;
  }
}
__global__ __launch_bounds__(kThreads) void k_vrows(int ne, const int32_t* __restrict__ pt_start,
                                                    const int32_t* __restrict__ row_cam,
                                                    const int32_t* __restrict__ cam_to_f,
                                                    const uint32_t* __restrict__ m0, int32_t* __restrict__ v_start,
                                                    int32_t* __restrict__ v_f, int32_t* __restrict__ v_id,
                                                    int32_t* __restrict__ v_e) {
  const int e = blockIdx.x * kThreads + threadIdx.x;
  if (e >= ne) return;
  const int shift = m0 ? (int)m0[e] : 0;
  v_start[e] = pt_start[e] + shift;
  if (e == ne - 1) v_start[ne] = pt_start[ne] + (m0 ? (int)m0[ne] : 0);
  for (int r = pt_start[e]; r < pt_start[e + 1]; ++r) {
    v_f[r + shift] = cam_to_f[row_cam[r]];
    v_id[r + shift] = r;
    v_e[r + shift] = e;
  }
}

// Key of block (fa, fb): fa above fb's place in the `span` F blocks that end
// with fa (span: the most F blocks of one problem of the call, so a batch of
// many small problems has a short low part).
struct BlockKey {
  int lbits, span;
  template <typename K>
  __host__ __device__ K make(int fa, int fb) const {
    return ((K)(uint32_t)fa << lbits) | (K)(uint32_t)(fb - fa + span - 1);
  }
  template <typename K>
  __host__ __device__ int fa(K k) const { return (int)(k >> lbits); }
  template <typename K>
  __host__ __device__ int fb(K k) const { return (int)(k & (((K)1 << lbits) - 1)) + fa(k) - (span - 1); }
};

// Row a pairs with the rows b of its point whose F block is not above its
// own (itself included); pairs come out point by point, a by a, b by b.
__global__ __launch_bounds__(kThreads) void k_pair_count(int64_t nv, const int32_t* __restrict__ v_start,
                                                         const int32_t* __restrict__ v_f,
                                                         const int32_t* __restrict__ v_e, uint32_t* __restrict__ cnt) {
  const int64_t a = blockIdx.x * (int64_t)kThreads + threadIdx.x;
  if (a >= nv) return;
  const int fa = v_f[a], e = v_e[a];
  uint32_t c = 0;
  if (fa >= 0)
    for (int b = v_start[e]; b < v_start[e + 1]; ++b) c += (uint32_t)v_f[b] <= (uint32_t)fa;  // -1 is above all
  cnt[a] = c;
}
template <typename K>
__global__ __launch_bounds__(kThreads) void k_pair_fill(int64_t nv, const int32_t* __restrict__ v_start,
                                                        const int32_t* __restrict__ v_f,
                                                        const int32_t* __restrict__ v_id,
                                                        const int32_t* __restrict__ v_e,
                                                        const uint64_t* __restrict__ off, BlockKey bk,
                                                        K* __restrict__ key, int2* __restrict__ pair) {
  const int64_t a = blockIdx.x * (int64_t)kThreads + threadIdx.x;
  if (a >= nv) return;
  const int fa = v_f[a], e = v_e[a], ia = v_id[a];
  if (fa < 0) return;
  uint64_t o = off[a];
  for (int b = v_start[e]; b < v_start[e + 1]; ++b) {
    const int fb = v_f[b];
    if ((uint32_t)fb > (uint32_t)fa) continue;
    key[o] = bk.make<K>(fa, fb);
    pair[o] = make_int2(ia, v_id[b]);
    ++o;
  }
}

// Heads of runs of equal keys: counted per tile, then written at the tile's
// offset (position and key of each run).
template <typename K>
__global__ __launch_bounds__(kThreads) void k_head_count(int64_t n, const K* __restrict__ key,
                                                         uint32_t* __restrict__ cnt) {
  __shared__ uint32_t lds[kWaves];
  const int64_t b = blockIdx.x * (int64_t)kTile;
  uint32_t c = 0;
  for (int k = 0; k < kPer; ++k) {
    const int64_t i = b + k * kThreads + threadIdx.x;
    if (i < n) c += i == 0 || key[i] != key[i - 1];
  }
  uint32_t total;
  (void)block_scan(c, lds, &total);
  if (threadIdx.x == 0) cnt[blockIdx.x] = total;
}
template <typename K>
__global__ __launch_bounds__(kThreads) void k_head_write(int64_t n, const K* __restrict__ key,
                                                         const uint32_t* __restrict__ off, BlockKey bk,
                                                         int64_t* __restrict__ start, int32_t* __restrict__ fa,
                                                         int32_t* __restrict__ fb) {
  __shared__ uint32_t lds[kWaves];
  const int64_t b = blockIdx.x * (int64_t)kTile;
  uint32_t run = off[blockIdx.x];
  for (int k = 0; k < kPer; ++k) {
    const int64_t i = b + k * kThreads + threadIdx.x;
    const bool head = i < n && (i == 0 || key[i] != key[i - 1]);
    uint32_t total;
    const uint32_t at = run + block_scan((uint32_t)head, lds, &total);
    if (head) {
      start[at] = i;
      fa[at] = bk.fa(key[i]);
      fb[at] = bk.fb(key[i]);
    }
    run += total;
  }
}

// Work items, slots and split blocks of every block, packed as three counts.
__global__ __launch_bounds__(kThreads) void k_item_count(int64_t nblk, int64_t npairs,
                                                         const int64_t* __restrict__ start, int64_t split,
                                                         uint32_t* __restrict__ items, uint32_t* __restrict__ slots,
                                                         uint32_t* __restrict__ splits) {
  const int64_t b = blockIdx.x * (int64_t)kThreads + threadIdx.x;
  if (b >= nblk) return;
  const int64_t n = (b + 1 < nblk ? start[b + 1] : npairs) - start[b];
  const uint32_t parts = (uint32_t)((n + split - 1) / split);
  items[b] = parts;
  slots[b] = parts > 1 ? parts : 0u;
  splits[b] = parts > 1;
}
__global__ __launch_bounds__(kThreads) void k_item_fill(
    int64_t nblk, int64_t npairs, const int64_t* __restrict__ start, int64_t split, const uint32_t* __restrict__ items,
    const uint32_t* __restrict__ slots, const uint32_t* __restrict__ splits, const int32_t* __restrict__ blk_fa,
    const int32_t* __restrict__ blk_fb, const int32_t* __restrict__ f_to_cam, const int32_t* __restrict__ cam_gf, int nc,
    int32_t* __restrict__ item_blk, int64_t* __restrict__ p0, int64_t* __restrict__ p1, int32_t* __restrict__ item_slot,
    int32_t* __restrict__ split_blk, int32_t* __restrict__ split_lo, int32_t* __restrict__ split_hi,
    int32_t* __restrict__ blk_cross) {
  const int64_t b = blockIdx.x * (int64_t)kThreads + threadIdx.x;
  if (b >= nblk) return;
  const int64_t q0 = start[b], q1 = b + 1 < nblk ? start[b + 1] : npairs;
  const uint32_t parts = items[b + 1] - items[b];
  for (uint32_t k = 0; k < parts; ++k) {
    const uint32_t i = items[b] + k;
    item_blk[i] = (int32_t)b;
    p0[i] = q0 + k * split;
    p1[i] = min(q1, q0 + (k + 1) * split);
    item_slot[i] = parts > 1 ? (int32_t)(slots[b] + k) : -1;
  }
  if (parts > 1) {
    split_blk[splits[b]] = (int32_t)b;
    split_lo[splits[b]] = (int32_t)slots[b];
    split_hi[splits[b]] = (int32_t)(slots[b] + parts);
  }
  if (blk_cross) {
    // Camera / group pairs: 2 c (+ 1 when the group block is fa).
    const int a = f_to_cam[blk_fa[b]], g = f_to_cam[blk_fb[b]];
    int x = -1;
    if (a < nc && g >= nc && cam_gf[a] == blk_fb[b]) x = 2 * a;
    else if (g < nc && a >= nc && cam_gf[g] == blk_fa[b]) x = 2 * g + 1;
    blk_cross[b] = x;
  }
}

// Device value(s) to the host (waits for the stream).
template <typename X>
mba_status read_back(hipStream_t s, const X* dev, X* host) {
  PREP_TRY(hipMemcpyAsync(host, dev, sizeof(X), hipMemcpyDeviceToHost, s));
  PREP_TRY(hipStreamSynchronize(s));
  return MBA_OK;
}

}  // namespace

// Built on the device: every point's pairs are written point by point, sorted
// by (fa, fb) -- stable, so a block's pairs stay in point and row order -- and
// cut into blocks and work items.  4.0M observations, 47M pairs: 284 ms on 16
// host threads with a bucket per fa; the whole solve (two LM iterations) 354
// -> 76 ms so, bit-identical.
mba_status build_s_pairs(const SPairsIn& in, const DeviceAlloc& alloc, SPairs* out) {
  const hipStream_t s = in.stream;
  Temps t(s);
  if ((in.grouped ? 3 : 1) * (int64_t)in.nrows > 0x7fffffffLL)
    return fail(MBA_ERR_UNSUPPORTED, "explicit Schur: too many rows");
  const unsigned ge = blocks_of(in.ne, kThreads);
  uint32_t *m0 = nullptr, *k0 = nullptr;
  uint32_t nmerged = 0;
  if (in.grouped) {
    PREP_OK(t.get(&m0, (size_t)in.ne + 1));
    PREP_OK(t.get(&k0, (size_t)in.ne + 1));
    if (in.ne > 0)
      hipLaunchKernelGGL(k_merge_count, dim3(ge), dim3(kThreads), 0, s, in.ne, in.pt_start, in.row_cam, in.cam_gf, m0,
                         k0);
    PREP_OK((scan<uint32_t, uint32_t>(t, in.ne, m0, m0)));
    PREP_OK((scan<uint32_t, uint32_t>(t, in.ne, k0, k0)));
    uint32_t members = 0;
    PREP_OK(read_back(s, (const uint32_t*)(m0 + in.ne), &nmerged));
    PREP_OK(read_back(s, (const uint32_t*)(k0 + in.ne), &members));
    PREP_OK(keep(alloc, &out->m_start, (size_t)nmerged + 1));
    PREP_OK(keep(alloc, &out->m_row, (size_t)members));
  }
  out->nmerged = nmerged;
  const int64_t nv = (int64_t)in.nrows + nmerged;
  if (2 * (int64_t)in.nrows + nmerged > 0x7fffffffLL) return fail(MBA_ERR_UNSUPPORTED, "explicit Schur: too many rows");
  int32_t *v_start, *v_f, *v_id, *v_e;
  uint32_t* cnt;
  uint64_t* off;
  PREP_OK(t.get(&v_start, (size_t)in.ne + 1));
  PREP_OK(t.get(&v_f, (size_t)nv));
  PREP_OK(t.get(&v_id, (size_t)nv));
  PREP_OK(t.get(&v_e, (size_t)nv));
  PREP_OK(t.get(&cnt, (size_t)nv));
  PREP_OK(t.get(&off, (size_t)nv + 1));
  uint64_t npairs = 0;
  const unsigned gv = blocks_of(nv, kThreads);
  if (in.ne > 0) {
    hipLaunchKernelGGL(k_vrows, dim3(ge), dim3(kThreads), 0, s, in.ne, in.pt_start, in.row_cam, in.cam_to_f,
                       (const uint32_t*)m0, v_start, v_f, v_id, v_e);
    if (in.grouped)
      hipLaunchKernelGGL(k_merge_fill, dim3(ge), dim3(kThreads), 0, s, in.ne, in.nrows, in.pt_start, in.row_cam,
                         in.cam_gf, (const uint32_t*)m0, (const uint32_t*)k0, out->m_start, out->m_row, v_f, v_id, v_e);
    hipLaunchKernelGGL(k_pair_count, dim3(gv), dim3(kThreads), 0, s, nv, (const int32_t*)v_start, (const int32_t*)v_f,
                       (const int32_t*)v_e, cnt);
    PREP_OK((scan<uint32_t, uint64_t>(t, nv, cnt, off)));
    PREP_OK(read_back(s, (const uint64_t*)(off + nv), &npairs));
  }
  if (npairs > 0x7fffffffull) return fail(MBA_ERR_UNSUPPORTED, "explicit Schur: more than 2^31-1 coupled row pairs");
  out->npairs = (int64_t)npairs;
  const BlockKey bk{bits_for((uint64_t)std::max(0, in.f_span - 1)), std::max(1, in.f_span)};
  const int bits = bk.lbits + bits_for((uint64_t)std::max(0, in.nf - 1));
  int64_t* start;
  uint32_t nblk = 0;
  auto sorted = [&](auto zero) -> mba_status {
    using K = decltype(zero);
    K* key[2];
    int2* pair[2];
    PREP_OK(t.get(&key[0], (size_t)npairs));
    PREP_OK(t.get(&key[1], (size_t)npairs));
    // The result ends in buffer passes % 2: the kept one.
    const int last = npairs > 1 ? ((bits + 7) / 8) & 1 : 0;
    PREP_OK(keep(alloc, &pair[last], (size_t)npairs));
    PREP_OK(t.get(&pair[1 - last], (size_t)npairs));
    int at = 0;
    if (npairs > 0) {
      hipLaunchKernelGGL(k_pair_fill<K>, dim3(gv), dim3(kThreads), 0, s, nv, (const int32_t*)v_start,
                         (const int32_t*)v_f, (const int32_t*)v_id, (const int32_t*)v_e, (const uint64_t*)off, bk,
                         key[0], pair[0]);
      PREP_OK((radix_sort<K, int2>(t, (int64_t)npairs, bits, key, pair, &at)));
    }
    if (at != last) return fail(MBA_ERR_DEVICE, "pair sort ended in the other buffer");
    out->pair = pair[last];
    const unsigned gt = blocks_of((int64_t)npairs, kTile);
    uint32_t* heads;
    PREP_OK(t.get(&heads, (size_t)gt + 1));
    if (npairs > 0) {
      hipLaunchKernelGGL(k_head_count<K>, dim3(gt), dim3(kThreads), 0, s, (int64_t)npairs, (const K*)key[at], heads);
      PREP_OK((scan<uint32_t, uint32_t>(t, gt, heads, heads)));
      PREP_OK(read_back(s, (const uint32_t*)(heads + gt), &nblk));
    }
    PREP_OK(t.get(&start, (size_t)nblk));
    PREP_OK(keep(alloc, &out->blk_fa, nblk));
    PREP_OK(keep(alloc, &out->blk_fb, nblk));
    if (nblk > 0)
      hipLaunchKernelGGL(k_head_write<K>, dim3(gt), dim3(kThreads), 0, s, (int64_t)npairs, (const K*)key[at],
                         (const uint32_t*)heads, bk, start, out->blk_fa, out->blk_fb);
    return MBA_OK;
  };
  PREP_OK(bits <= 32 ? sorted(uint32_t(0)) : sorted(uint64_t(0)));
  out->nblk = nblk;
  if (in.grouped) PREP_OK(keep(alloc, &out->blk_cross, nblk));
  uint32_t *items, *slots, *splits, total[3] = {0, 0, 0};
  PREP_OK(t.get(&items, (size_t)nblk + 1));
  PREP_OK(t.get(&slots, (size_t)nblk + 1));
  PREP_OK(t.get(&splits, (size_t)nblk + 1));
  const unsigned gb = blocks_of(nblk, kThreads);
  if (nblk > 0) {
    hipLaunchKernelGGL(k_item_count, dim3(gb), dim3(kThreads), 0, s, (int64_t)nblk, (int64_t)npairs,
                       (const int64_t*)start, in.split_pairs, items, slots, splits);
    uint32_t* const a[3] = {items, slots, splits};
    for (int k = 0; k < 3; ++k) {
      PREP_OK((scan<uint32_t, uint32_t>(t, nblk, a[k], a[k])));
      PREP_TRY(hipMemcpyAsync(&total[k], a[k] + nblk, sizeof(uint32_t), hipMemcpyDeviceToHost, s));
    }
    PREP_TRY(hipStreamSynchronize(s));
  }
  out->nitems = total[0];
  out->nslots = total[1];
  out->nsplit = total[2];
  PREP_OK(keep(alloc, &out->item_blk, total[0]));
  PREP_OK(keep(alloc, &out->item_p0, total[0]));
  PREP_OK(keep(alloc, &out->item_p1, total[0]));
  PREP_OK(keep(alloc, &out->item_slot, total[0]));
  PREP_OK(keep(alloc, &out->split_blk, total[2]));
  PREP_OK(keep(alloc, &out->split_lo, total[2]));
  PREP_OK(keep(alloc, &out->split_hi, total[2]));
  if (nblk > 0)
    hipLaunchKernelGGL(k_item_fill, dim3(gb), dim3(kThreads), 0, s, (int64_t)nblk, (int64_t)npairs,
                       (const int64_t*)start, in.split_pairs, (const uint32_t*)items, (const uint32_t*)slots,
                       (const uint32_t*)splits, (const int32_t*)out->blk_fa, (const int32_t*)out->blk_fb, in.f_to_cam,
                       in.cam_gf, in.nc, out->item_blk, out->item_p0, out->item_p1, out->item_slot, out->split_blk,
                       out->split_lo, out->split_hi, out->blk_cross);
  PREP_TRY(hipGetLastError());
  return MBA_OK;
}

// ---------------------------------------------------------------- layout
struct LayoutBuilder::State {
  In in;
  Temps t;
  int32_t *pstart = nullptr, *pdeg = nullptr;
  uint32_t* rows = nullptr;  // observations by point, descending within one
  int32_t max_track = 0;
  explicit State(const In& i) : in(i), t(i.stream) {}
};
LayoutBuilder::LayoutBuilder(const In& in) : st_(new State(in)) {}
LayoutBuilder::~LayoutBuilder() { delete st_; }

mba_status LayoutBuilder::measure(Stats* out) {
  State& S = *st_;
  const In& in = S.in;
  Temps& t = S.t;
  const hipStream_t s = in.stream;
  uint32_t *key[2], *val[2];
  for (int k = 0; k < 2; ++k) {
    PREP_OK(t.get(&key[k], (size_t)in.n));
    PREP_OK(t.get(&val[k], (size_t)in.n));
  }
  hipLaunchKernelGGL(k_keys<true>, dim3(blocks_of(in.n, kThreads)), dim3(kThreads), 0, s, in.n, in.pt, key[0], val[0]);
  int at = 0;
  PREP_OK((radix_sort<uint32_t, uint32_t>(t, in.n, bits_for((uint64_t)in.np - 1), key, val, &at)));
  S.rows = val[at];
  PREP_OK(t.get(&S.pstart, (size_t)in.np + 1));
  PREP_OK(t.get(&S.pdeg, (size_t)in.np));
  hipLaunchKernelGGL(k_bounds, dim3(blocks_of(in.n + 1, kThreads)), dim3(kThreads), 0, s, in.n,
                     (const uint32_t*)key[at], in.np, S.pstart);
  const StatsAt sa{in.nc, in.ng, in.W};
  int32_t* st;
  PREP_OK(t.get(&st, (size_t)sa.size()));
  hipLaunchKernelGGL(k_stats_init, dim3((unsigned)std::min<int64_t>(256, blocks_of(sa.size(), kThreads))),
                     dim3(kThreads), 0, s, sa, st);
  const std::pair<const double*, int64_t> params[3] = {
      {in.pts, 3 * (int64_t)in.np}, {in.cams, in.ncams64}, {in.intr, in.nintr64}};
  for (const auto& v : params)
    if (v.second > 0)
      hipLaunchKernelGGL(k_finite, dim3((unsigned)std::min<int64_t>(512, blocks_of(v.second, kThreads))),
                         dim3(kThreads), 0, s, v.second, v.first, st + sa.bad());
  if (in.grp)
    hipLaunchKernelGGL((in.nc <= kLdsBlocks ? k_cam_groups<true> : k_cam_groups<false>),
                       dim3((unsigned)std::min<int64_t>(in.nc <= kLdsBlocks ? 256 : 8192, blocks_of(in.n, kThreads))),
                       dim3(kThreads), 0, s, in.n, in.cam, in.grp, sa, st);
  const bool ranged = in.nc + in.ng > kLdsBlocks && in.W > 1 && !in.grp;
  const bool lds = in.nc + in.ng <= kLdsBlocks || ranged;
  const unsigned g = (unsigned)std::min<int64_t>(lds ? 1024 : 8192, blocks_of(in.np, kThreads));
  hipLaunchKernelGGL((lds ? k_point_stats<true> : k_point_stats<false>), dim3(g), dim3(kThreads), 0, s, in.np,
                     (const int32_t*)S.pstart, (const uint32_t*)S.rows, in.cam, in.grp, in.cam_const, in.grp_const,
                     in.W > 1 ? in.pt_off : nullptr, sa, st, S.pdeg, (int)ranged);
  PREP_TRY(hipGetLastError());
  std::vector<int32_t> h((size_t)sa.size());
  PREP_TRY(hipMemcpyAsync(h.data(), st, h.size() * sizeof(int32_t), hipMemcpyDeviceToHost, s));
  PREP_TRY(hipStreamSynchronize(s));
  auto part = [&](int64_t from, int64_t n) { return std::vector<int32_t>(h.begin() + from, h.begin() + from + n); };
  out->cam_deg = part(0, in.nc);
  out->cam_first = part(sa.cam_first(), in.nc);
  out->grp_deg = part(sa.grp_deg(), in.ng);
  out->grp_first = part(sa.grp_first(), in.ng);
  out->win_max_deg = part(sa.win_max(), in.W);
  out->win_points = part(sa.win_points(), in.W);  // (several windows)
  out->max_track = S.max_track = h[sa.max_track()];
  out->finite = h[sa.bad()] == 0;
  out->repeated = h[sa.repeated()] != 0;
  if (in.grp) {
    out->cam_grp.assign(in.nc, -1);
    for (int32_t c = 0; c < in.nc; ++c) {
      const int32_t lo = h[sa.grp_lo() + c], hi = h[sa.grp_hi() + c];
      if (hi < 0) continue;
      out->cam_grp[c] = lo;
      out->two_groups = out->two_groups || lo != hi;
    }
  }
  return MBA_OK;
}

mba_status LayoutBuilder::arrange(const std::vector<int32_t>& cam_key, int32_t nkeys, int32_t nq, int32_t max_deg,
                                  const DeviceAlloc& alloc, Layout* out, std::vector<int32_t>* split,
                                  std::vector<int32_t>* track_hist) {
  State& S = *st_;
  const In& in = S.in;
  Temps& t = S.t;
  const hipStream_t s = in.stream;
  if (S.max_track > kLayoutMaxTrack) return fail(MBA_ERR_UNSUPPORTED, "track too long for the device layout");
  const PointKey pk(in.n, in.W, max_deg, S.max_track);
  if (!pk.fits()) return fail(MBA_ERR_UNSUPPORTED, "point key too wide for the device layout");
  uint64_t* pkey[2];
  uint32_t* perm[2];
  for (int k = 0; k < 2; ++k) {
    PREP_OK(t.get(&pkey[k], (size_t)in.np));
    PREP_OK(t.get(&perm[k], (size_t)in.np));
  }
  const int32_t* off = in.W > 1 ? in.pt_off : nullptr;
  int32_t* hist;
  PREP_OK(t.get(&hist, (size_t)S.max_track + 1));
  PREP_TRY(hipMemsetAsync(hist, 0, sizeof(int32_t) * ((size_t)S.max_track + 1), s));
  hipLaunchKernelGGL(k_point_keys, dim3((unsigned)std::min<int64_t>(1024, blocks_of(in.np, kThreads))), dim3(kThreads),
                     0, s, in.np, (const int32_t*)S.pstart, (const uint32_t*)S.rows, (const int32_t*)S.pdeg, off, in.W,
                     pk, pkey[0], perm[0], S.max_track, hist);
  int at = 0;
  PREP_OK((radix_sort<uint64_t, uint32_t>(t, in.np, pk.bits(), pkey, perm, &at)));
  track_hist->resize((size_t)S.max_track + 1);
  PREP_TRY(hipMemcpyAsync(track_hist->data(), hist, sizeof(int32_t) * track_hist->size(), hipMemcpyDeviceToHost, s));
  PREP_TRY(hipStreamSynchronize(s));
  const int32_t ne = in.np - (*track_hist)[0];
  int32_t* len;
  PREP_OK(t.get(&len, (size_t)ne));
  PREP_OK(keep(alloc, &out->e_to_pt, (size_t)ne));
  PREP_OK(keep(alloc, &out->pts, 3 * (size_t)ne));
  PREP_OK(keep(alloc, &out->pt_start, (size_t)ne + 1));
  if (in.W > 1) PREP_OK(keep(alloc, &out->of_e, (size_t)ne));
  hipLaunchKernelGGL(k_point_order, dim3(blocks_of(ne, kThreads)), dim3(kThreads), 0, s, ne, (const uint32_t*)perm[at],
                     (const int32_t*)S.pstart, in.pts, off, in.W, out->e_to_pt, len, out->pts, out->of_e);
  PREP_OK((scan<int32_t, int32_t>(t, ne, len, out->pt_start)));
  PREP_OK(keep(alloc, &out->row_e, (size_t)in.n));
  PREP_OK(keep(alloc, &out->row_cam, (size_t)in.n));
  PREP_OK(keep(alloc, &out->obs, 2 * (size_t)in.n));
  hipLaunchKernelGGL(k_row_points, dim3(blocks_of(16 * (int64_t)ne, kThreads)), dim3(kThreads), 0, s, ne,
                     (const int32_t*)out->pt_start, out->row_e);
  int32_t *ck, *start;
  PREP_OK(t.get(&ck, cam_key.size()));
  PREP_TRY(hipMemcpyAsync(ck, cam_key.data(), sizeof(int32_t) * cam_key.size(), hipMemcpyHostToDevice, s));
  uint32_t *key[2], *src[2];
  const int bits = bits_for((uint64_t)nkeys);  // key nkeys: rows left out
  const int last = in.n > 1 ? ((bits + 7) / 8) & 1 : 0;
  for (int k = 0; k < 2; ++k) PREP_OK(t.get(&key[k], (size_t)in.n));
  PREP_OK(keep(alloc, &src[last], (size_t)in.n));
  PREP_OK(t.get(&src[1 - last], (size_t)in.n));
  hipLaunchKernelGGL(k_rows, dim3(blocks_of(in.n, kThreads)), dim3(kThreads), 0, s, in.n, (const int32_t*)out->row_e,
                     (const int32_t*)out->pt_start, (const int32_t*)out->e_to_pt, (const int32_t*)S.pstart,
                     (const uint32_t*)S.rows, in.cam, (const double2*)in.obs, (const int32_t*)ck, nkeys, out->row_cam,
                     (double2*)out->obs, key[0], src[0]);
  PREP_OK((radix_sort<uint32_t, uint32_t>(t, in.n, bits, key, src, &at)));
  if (at != last) return fail(MBA_ERR_DEVICE, "row sort ended in the other buffer");
  out->cm_src = (int32_t*)src[at];
  PREP_OK(t.get(&start, (size_t)nkeys + 2));
  hipLaunchKernelGGL(k_bounds, dim3(blocks_of(in.n + 1, kThreads)), dim3(kThreads), 0, s, in.n,
                     (const uint32_t*)key[at], nkeys + 1, start);
  int32_t *range_row, *sp;
  const size_t nsp = (size_t)nkeys * ((size_t)nq + 1);
  PREP_OK(t.get(&range_row, (size_t)nq + 1));
  PREP_OK(t.get(&sp, nsp));
  hipLaunchKernelGGL(k_range_rows, dim3(1), dim3(64), 0, s, in.n, ne, (const int32_t*)out->pt_start, nq, range_row);
  split->resize(nsp);
  if (nsp > 0) {
    hipLaunchKernelGGL(k_split, dim3(blocks_of((int64_t)nsp, kThreads)), dim3(kThreads), 0, s, nkeys, nq,
                       (const int32_t*)start, (const uint32_t*)out->cm_src, (const int32_t*)range_row, sp);
    PREP_TRY(hipMemcpyAsync(split->data(), sp, sizeof(int32_t) * nsp, hipMemcpyDeviceToHost, s));
  }
  PREP_TRY(hipGetLastError());
  PREP_TRY(hipStreamSynchronize(s));
  return MBA_OK;
}

mba_status bucket_lists(hipStream_t s, int64_t n, const int32_t* bucket, int32_t nbuckets, const DeviceAlloc& alloc,
                        int32_t** start, int32_t** list) {
  Temps t(s);
  uint32_t *key[2], *val[2];
  const int bits = bits_for((uint64_t)std::max(0, nbuckets - 1));
  const int last = n > 1 ? ((bits + 7) / 8) & 1 : 0;
  for (int k = 0; k < 2; ++k) PREP_OK(t.get(&key[k], (size_t)n));
  PREP_OK(keep(alloc, &val[last], (size_t)n));
  PREP_OK(t.get(&val[1 - last], (size_t)n));
  PREP_OK(keep(alloc, start, (size_t)nbuckets + 1));
  int at = 0;
  if (n > 0) {
    hipLaunchKernelGGL(k_keys<false>, dim3(blocks_of(n, kThreads)), dim3(kThreads), 0, s, n, bucket, key[0], val[0]);
    PREP_OK((radix_sort<uint32_t, uint32_t>(t, n, bits, key, val, &at)));
  }
  if (at != last) return fail(MBA_ERR_DEVICE, "bucket sort ended in the other buffer");
  hipLaunchKernelGGL(k_bounds, dim3(blocks_of(n + 1, kThreads)), dim3(kThreads), 0, s, n, (const uint32_t*)key[at],
                     nbuckets, *start);
  PREP_TRY(hipGetLastError());
  *list = (int32_t*)val[last];
  return MBA_OK;
}

}  // namespace mba
