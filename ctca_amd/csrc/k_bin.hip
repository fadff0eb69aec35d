// k_bin.hip -- FP64 particles in no spatial order binned by tiles of kBinTile^3
// cells, for the kernels that then work tile by tile in LDS (the adjoint step,
// the charge of an unsorted state):
//   k_bin_count  particles per tile (a block's counts in LDS, one atomic per
//                block and tile), then a scan;
//   k_bin        position and index of each particle, 32 bytes, to its tile's
//                range, a block's records of one tile in one run.
// 8.8M particles in 512 tiles: 0.08 + 0.26 ms.  With more than kBinLds tiles a
// block's LDS counters would not fit, and each particle takes one global atomic
// on its tile's counter.
#include <algorithm>

#include "emg_internal.h"

namespace emg {
namespace {

constexpr int kBinLds = 4096;                     // 16 KB of LDS counters
constexpr int64_t kBinMax = int64_t(1) << 24;     // records per pass (512 MB)

__device__ __forceinline__ int bin_of(const BinTiles &a, const Grid &g, double x, double y,
                                      double z) {
  const int i = min(max((int)x, 0), g.nx - 1), j = min(max((int)y, 0), g.ny - 1),
            k = min(max((int)z, 0), g.nz - 1);
  return ((k / kBinTile) * a.nty + j / kBinTile) * a.ntx + i / kBinTile;
}

// The particles of a pass: [lo, hi) of each species, as indices of the state
// arrays.  A block takes kBlock P of species blockIdx.y.
struct BinPass {
  int64_t lo[EMG_MAX_SPECIES], hi[EMG_MAX_SPECIES];
};

template <int P>
__global__ __launch_bounds__(kBlock) void k_bin_count(State64 s, BinPass ps, BinTiles at, Grid g,
                                                      int32_t *count) {
  extern __shared__ int32_t hist[];
  const int is = blockIdx.y;
  const int64_t beg = ps.lo[is] + (int64_t)blockIdx.x * (kBlock * P);
  if (beg >= ps.hi[is]) return;  // uniform over the block
  const bool lds = at.n <= kBinLds;
  if (lds) {
    for (int t = threadIdx.x; t < at.n; t += kBlock) hist[t] = 0;
    __syncthreads();
  }
#pragma unroll 4
  for (int q = 0; q < P; q++) {
    const int64_t m = beg + q * kBlock + threadIdx.x;
    if (m < ps.hi[is]) {
      const int tl = bin_of(at, g, s.x[m], s.y[m], s.z[m]);
      if (lds) atomicAdd(&hist[tl], 1);
      else atomicAdd(&count[tl], 1);
    }
  }
  if (lds) {
    __syncthreads();
    for (int t = threadIdx.x; t < at.n; t += kBlock)
      if (hist[t]) atomicAdd(&count[t], hist[t]);
  }
}

template <int P>
__global__ __launch_bounds__(kBlock) void k_bin(State64 s, BinPass ps, BinTiles at, Grid g,
                                                const int64_t *__restrict__ start,
                                                int32_t *__restrict__ cursor,
                                                BinRec *__restrict__ rec) {
  // a tile's count, then its first record of this block; then each particle's
  // tile and rank
  extern __shared__ int32_t hist[];
  static_assert(kBinLds <= 1 << 16 && kBlock * P <= 1 << 16, "tile and rank in one word");
  uint32_t *mine = reinterpret_cast<uint32_t *>(hist + at.n) + threadIdx.x;
  const int is = blockIdx.y;
  const int64_t beg = ps.lo[is] + (int64_t)blockIdx.x * (kBlock * P);
  if (beg >= ps.hi[is]) return;  // uniform over the block
  const bool lds = at.n <= kBinLds;
  if (lds) {
    for (int t = threadIdx.x; t < at.n; t += kBlock) hist[t] = 0;
    __syncthreads();
#pragma unroll 4
    for (int q = 0; q < P; q++) {
      const int64_t m = beg + q * kBlock + threadIdx.x;
      if (m < ps.hi[is]) {
        const int tl = bin_of(at, g, s.x[m], s.y[m], s.z[m]);
        mine[q * kBlock] = ((uint32_t)tl << 16) | (uint32_t)atomicAdd(&hist[tl], 1);
      }
    }
    __syncthreads();
    for (int t = threadIdx.x; t < at.n; t += kBlock)
      if (hist[t]) hist[t] = (int32_t)start[t] + atomicAdd(&cursor[t], hist[t]);
    __syncthreads();
  }
#pragma unroll 4
  for (int q = 0; q < P; q++) {
    const int64_t m = beg + q * kBlock + threadIdx.x;
    if (m < ps.hi[is]) {
      const double x = s.x[m], y = s.y[m], z = s.z[m];
      int64_t d;
      if (lds) {
        const uint32_t tr = mine[q * kBlock];
        d = hist[tr >> 16] + (int)(tr & 0xffffu);
      } else {
        const int tl = bin_of(at, g, x, y, z);
        d = start[tl] + atomicAdd(&cursor[tl], 1);
      }
      double2 *r = reinterpret_cast<double2 *>(rec + d);
      r[0] = make_double2(x, y);
      r[1] = make_double2(z, __longlong_as_double(m | ((int64_t)is << 56)));
    }
  }
}

template <int P>
void launch_bin(emg_ctx *c, const BinPass &ps, int64_t most) {
  const TileBins &B = c->bins;
  const BinTiles at = bin_tiles(c->g);
  const dim3 grid((unsigned)((most + kBlock * P - 1) / (kBlock * P)), c->sp.nspec);
  const size_t lds = at.n <= kBinLds ? sizeof(int32_t) * at.n : 0;
  launch_zero(B.count, sizeof(int32_t) * 2 * at.n, c->stream);
  hipLaunchKernelGGL(k_bin_count<P>, grid, dim3(kBlock), lds, c->stream, c->s64, ps, at, c->g,
                     B.count);
  exclusive_scan_i32(B.count, B.start, at.n, c->scan_tmp, c->stream);
  hipLaunchKernelGGL(k_bin<P>, grid, dim3(kBlock), lds ? lds + sizeof(int32_t) * kBlock * P : 0,
                     c->stream, c->s64, ps, at, c->g, B.start, B.count + at.n, B.rec);
}

}  // namespace

BinTiles bin_tiles(const Grid &g) {
  BinTiles a;
  a.ntx = (g.nx + kBinTile - 1) / kBinTile;
  a.nty = (g.ny + kBinTile - 1) / kBinTile;
  a.ntz = (g.nz + kBinTile - 1) / kBinTile;
  a.n = a.ntx * a.nty * a.ntz;
  return a;
}

// the workspace, kept with the context: the tile counters and starts, and the
// records of one pass (halved until they can be allocated: more passes then)
int bins_alloc(emg_ctx *c) {
  TileBins &B = c->bins;
  if (B.rec) return EMG_OK;
  const int64_t n = bin_tiles(c->g).n;
  if (!B.count && !dev_malloc(c, &B.count, sizeof(int32_t) * 2 * n))
    return set_error(EMG_ERR_NOMEM, "tile counters");
  if (!B.start && !dev_malloc(c, &B.start, sizeof(int64_t) * (n + 1)))
    return set_error(EMG_ERR_NOMEM, "tile starts");
  const int rc = scan_tmp_alloc(c, n);
  if (rc) return rc;
  int64_t len = std::min(std::max<int64_t>(c->cap_total, 1), kBinMax);
  while (!dev_malloc(c, &B.rec, sizeof(BinRec) * len)) {
    if (len <= 65536) return set_error(EMG_ERR_NOMEM, "tile records");
    len /= 2;
  }
  B.len = len;
  return EMG_OK;
}

// The records, up to 512 MB, are a workspace that is had again when it is next
// needed: what else the context allocates comes first (unless a graph holds their
// address).
bool bins_give_back(emg_ctx *c) {
  TileBins &B = c->bins;
  if (!B.rec || B.recorded || capturing(c)) return false;
  (void)hipStreamSynchronize(c->stream);
  (void)hipFree(B.rec);
  B.rec = nullptr;
  B.len = 0;
  return true;
}

int64_t bin_pass(emg_ctx *c, int64_t done[EMG_MAX_SPECIES]) {
  BinPass ps{};
  int64_t room = c->bins.len, most = 0;
  for (int s = 0; s < c->sp.nspec; s++) {
    const int64_t k = std::min(room, c->sp.cnt[s] - done[s]);
    ps.lo[s] = c->sp.off[s] + done[s];
    ps.hi[s] = ps.lo[s] + k;
    done[s] += k;
    room -= k;
    most = std::max(most, k);
  }
  if (most == 0) return 0;
  c->bins.recorded = c->bins.recorded || capturing(c);
  const int64_t total = c->bins.len - room;
  // 16 particles per thread make a block's records of a tile a run of several;
  // small populations need the blocks more
  if (total >= (int64_t)kBlock * 16 * 512)
    launch_bin<16>(c, ps, most);
  else
    launch_bin<4>(c, ps, most);
  return total;
}

}  // namespace emg
