// Device neighbour list: the cell-list search of fc_neighbor_list (fc_neighbors.cpp) on the
// GPU, for structures whose positions already live in HBM (an MD step, a batch built on
// the device). Replaces NeighborList.build (reference src/flashcart/data/neighbors.py:56-77,
// :120-143) like the host list, and returns the same pairs in the same order:
// (i, j, S) with |pos[j] - pos[i] + S.cell| < cutoff, self pairs with S = 0 removed,
// sorted by (i, j, Sx, Sy, Sz).
//
// Same edge set as the host list, bit for bit: fractional coordinates, wrapping, image
// positions and squared distances are evaluated in float64 with the host's expressions
// and operation order, and without fused multiply-adds (this file is compiled with
// -ffp-contract=off; the host build has none), so every comparison with cutoff^2 takes
// the same branch.
//
// Steps (one stream, one small device-to-host read; two with open axes):
//   range: min / max of the fractional coordinates along open axes (read back)
//   bin:   bins of fractional width >= reach (cutoff / plane spacing) over the unit cell
//          (periodic axes) or [min, max] (open axes); counting sort of the atoms by bin, after
//          which wrapped coordinates, integer offsets and atom numbers stand in bin order
//   count: one wave per receiver visits its (2D+1)^3 neighbouring bins, periodic bins
//          through their image shift (virtual bin v = bin + shift * bins, so every
//          (atom, image) candidate appears once), and counts the pairs (ballot)
//   scan:  receiver offsets (read back: the number of pairs)
//   fill:  one wave per receiver collects its pairs' keys (j, S) in LDS, sorts them
//          (bitonic) and writes them at its offset.
//
// Neighbouring bins along the last axis are neighbours in memory too, so a receiver's candidates are
// (2D+1)^2 runs (more where a run crosses a periodic boundary), whose ends the lanes look up side by
// side. Walking bin by bin, 27 chains of bin, atom number and coordinate, bounded both searches by
// latency.
#include <cmath>
#include <mutex>

#include "fc_common.h"

namespace fc {

constexpr int kNLMaxPerAtom = 1024;  // pairs per receiver held in LDS by the fill kernel
constexpr int kNLShiftBias = 512;    // shift components packed in 10 bits each: |S| < 512
// A cell far thinner than the cutoff is left to the host list before anything is launched: beyond 2^20 bins
// to one side, or 2^18 runs of candidates (nl_visit) for a receiver. Lists of at most 1,024 pairs an atom and 511 images
// an axis need some 10,000 runs (1,023 x 9 for one thin axis, 4 x 1,024 / pi x 3 for two), more in skewed cells only. A
// wave takes 1 s for the 3 million runs of a cell of 8 x 0.008 x 0.008 under a cutoff of 4, each with an atom in it.
constexpr double kNLMaxBinsAway = 1 << 20, kNLMaxRuns = 1 << 18;

struct NLPlan {
  double cell[9], inv[9];
  double base[3], width[3];
  double c2;
  int32_t nb[3], D[3], pbc[3];
  int32_t ns2;  // images that the bins of one column, v2 in [b2 - D2, b2 + D2], can lie in
  int64_t n;
};

__device__ __forceinline__ int nl_bin_of(double f, double base, double width, int nb) {
  int v = (int)floor((f - base) / width);
  return v < 0 ? 0 : (v >= nb ? nb - 1 : v);
}

// Wrapped fractional coordinates of atom i and the integer offsets taken out. Computed from the positions
// wherever they are needed, always with these operations.
__device__ __forceinline__ void nl_wrap(const NLPlan& p, const double* __restrict__ pos, int64_t i, double (&w)[3],
                                        int (&off)[3]) {
  for (int k = 0; k < 3; ++k) {
    const double f = pos[3 * i] * p.inv[k] + pos[3 * i + 1] * p.inv[3 + k] + pos[3 * i + 2] * p.inv[6 + k];
    const double fl = p.pbc[k] ? floor(f) : 0.0;
    w[k] = p.pbc[k] ? f - fl : f;
    off[k] = (int32_t)fl;
  }
}

// min / max of the fractional coordinates per axis (one workgroup of 256 threads).
__global__ void __launch_bounds__(256) nl_range_kernel(NLPlan p, const double* __restrict__ pos,
                                                       double* __restrict__ out) {
  __shared__ double lo[3][256], hi[3][256];
  const int t = threadIdx.x;
  double l[3] = {1e300, 1e300, 1e300}, h[3] = {-1e300, -1e300, -1e300};
  for (int64_t i = t; i < p.n; i += 256) {
    double w[3];
    int off[3];
    nl_wrap(p, pos, i, w, off);
    for (int k = 0; k < 3; ++k) {
      l[k] = fmin(l[k], w[k]);
      h[k] = fmax(h[k], w[k]);
    }
  }
  for (int k = 0; k < 3; ++k) {
    lo[k][t] = l[k];
    hi[k][t] = h[k];
  }
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (t < s)
      for (int k = 0; k < 3; ++k) {
        lo[k][t] = fmin(lo[k][t], lo[k][t + s]);
        hi[k][t] = fmax(hi[k][t], hi[k][t + s]);
      }
    __syncthreads();
  }
  if (t < 3) {
    out[t] = lo[t][0];
    out[3 + t] = hi[t][0];
  }
}

__global__ void nl_init_kernel(int64_t n, int32_t* __restrict__ hist, int32_t* __restrict__ status) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) hist[i] = 0;
  if (i < 2) status[i] = 0;
}

__global__ void nl_bin_kernel(NLPlan p, const double* __restrict__ pos, int32_t* __restrict__ bin,
                              int32_t* __restrict__ hist) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= p.n) return;
  double w[3];
  int off[3], b[3];
  nl_wrap(p, pos, i, w, off);
  for (int k = 0; k < 3; ++k) b[k] = nl_bin_of(w[k], p.base[k], p.width[k], p.nb[k]);
  const int id = (b[0] * p.nb[1] + b[1]) * p.nb[2] + b[2];
  bin[i] = id;
  atomicAdd(&hist[id], 1);
}

// Counting sort by bin. The order of atoms inside a bin depends on scheduling; the fill kernel sorts
// every receiver's pairs, so the output does not. Takes the bin counts back down to zero.
__global__ void nl_scatter_kernel(NLPlan p, const double* __restrict__ pos, const int32_t* __restrict__ bin,
                                  const int64_t* __restrict__ head, int32_t* __restrict__ hist,
                                  double* __restrict__ w, int32_t* __restrict__ off, int32_t* __restrict__ order) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= p.n) return;
  const int id = bin[i];
  const int64_t slot = head[id] + atomicAdd(&hist[id], -1) - 1;
  double wi[3];
  int oi[3];
  nl_wrap(p, pos, i, wi, oi);
  for (int k = 0; k < 3; ++k) {
    w[3 * slot + k] = wi[k];
    off[3 * slot + k] = oi[k];
  }
  order[slot] = (int32_t)i;
}

// Exclusive prefix sum of n counts into out[0..n] (out[n] = total, also *total). One workgroup of 1024
// threads goes through the counts 4096 at a time, four to a thread, the next tile's loads under way while
// this one is summed across lanes and waves. (25,000 counts and
// 1,350 bins, both scans: 44 us with a contiguous share of the counts to each thread, now 20.)
__global__ void __launch_bounds__(1024) nl_scan_kernel(int64_t n, const int32_t* __restrict__ in,
                                                        int64_t* __restrict__ out, int64_t* __restrict__ total) {
  __shared__ int64_t part[2][16];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  int64_t carry = 0;
  struct Four {
    int32_t x, y, z, w;
  };  // (aligned as its members: a workspace need not be to 16 bytes)
  auto load = [&](int64_t a) {
    Four v{0, 0, 0, 0};
    if (a + 4 <= n) {
      v = *reinterpret_cast<const Four*>(in + a);
    } else {
      if (a < n) v.x = in[a];
      if (a + 1 < n) v.y = in[a + 1];
      if (a + 2 < n) v.z = in[a + 2];
    }
    return v;
  };
  Four next = load(4 * t);
  for (int64_t base = 0, k = 0; base < n; base += 4096, k ^= 1) {
    const int64_t a = base + 4 * t;
    const Four v = next;
    next = load(a + 4096);
    const int64_t s = (int64_t)v.x + v.y + v.z + v.w;
    int64_t x = s;  // inclusive over the lanes of the wave
    for (int o = 1; o < 64; o <<= 1) {
      const int64_t u = __shfl_up((long long)x, o);
      if (lane >= o) x += u;
    }
    if (lane == 63) part[k][wave] = x;
    __syncthreads();  // (two buffers: the next tile's sums do not wait for this tile's readers)
    int64_t before = carry, all = 0;
    for (int q = 0; q < 16; ++q) {
      const int64_t u = part[k][q];
      if (q < wave) before += u;
      all += u;
    }
    carry += all;
    int64_t run = before + x - s;
    if (a < n) out[a] = run;
    if (a + 1 < n) out[a + 1] = run + v.x;
    if (a + 2 < n) out[a + 2] = run + v.x + v.y;
    if (a + 3 < n) out[a + 3] = run + v.x + v.y + v.z;
  }
  if (t == 0) {
    out[n] = carry;
    if (total) *total = carry;
  }
}

// Visit every candidate (j, image) of the receiver in `slot` (bin order) of bin b0; calls hit(ok, j, S) with ok
// for the pairs within the cutoff. Lane r holds run r of the candidates: the bins v2 in [b2 - D2, b2 + D2] of
// one image of one column (v0, v1), a range of slots. At most ns2 images meet a column, and 64 runs are looked
// up at a time; lanes stride over the atoms of each run in turn.
template <class F>
__device__ __forceinline__ void nl_visit(const NLPlan& p, int64_t slot, int bin, const double* __restrict__ w,
                                         const int32_t* __restrict__ off, const int64_t* __restrict__ head,
                                         const int32_t* __restrict__ order, int lane, F&& hit) {
  double xi[3];
  for (int k = 0; k < 3; ++k)
    xi[k] = w[3 * slot] * p.cell[k] + w[3 * slot + 1] * p.cell[3 + k] + w[3 * slot + 2] * p.cell[6 + k];
  const int oi[3] = {off[3 * slot], off[3 * slot + 1], off[3 * slot + 2]};
  const int b01 = bin / p.nb[2];
  const int b[3] = {b01 / p.nb[1], b01 % p.nb[1], bin % p.nb[2]};
  const int n1 = 2 * p.D[1] + 1;
  const int v2lo = p.pbc[2] ? b[2] - p.D[2] : max(b[2] - p.D[2], 0);
  const int v2hi = p.pbc[2] ? b[2] + p.D[2] : min(b[2] + p.D[2], p.nb[2] - 1);
  auto image = [](int v, int nb) {  // of virtual bin v: floor(v / nb), divided out for few lanes
    return v >= 0 && v < nb ? 0 : (v >= 0 ? v : v - nb + 1) / nb;
  };
  const int s2lo = image(v2lo, p.nb[2]);
  const unsigned ns2 = p.ns2, runs = (unsigned)(2 * p.D[0] + 1) * n1 * ns2;
  for (unsigned r0 = 0; r0 < runs; r0 += 64) {
    const unsigned id = r0 + lane;
    int first = 0, len = 0, s[3] = {0, 0, 0};
    if (id < runs) {
      const unsigned c = id / ns2;
      const int v0 = b[0] - p.D[0] + (int)(c / (unsigned)n1), v1 = b[1] - p.D[1] + (int)(c % (unsigned)n1);
      s[2] = s2lo + (int)(id % ns2);
      const bool in = (p.pbc[0] || (v0 >= 0 && v0 < p.nb[0])) && (p.pbc[1] || (v1 >= 0 && v1 < p.nb[1]));
      const int a2 = max(v2lo - s[2] * p.nb[2], 0), e2 = min(v2hi - s[2] * p.nb[2], p.nb[2] - 1);
      if (in && a2 <= e2) {
        s[0] = image(v0, p.nb[0]);
        s[1] = image(v1, p.nb[1]);
        const int col = ((v0 - s[0] * p.nb[0]) * p.nb[1] + v1 - s[1] * p.nb[1]) * p.nb[2];
        first = (int)head[col + a2];
        len = (int)head[col + e2 + 1] - first;
      }
    }
    for (uint64_t m = __ballot(len > 0); m; m &= m - 1) {
      const int r = __builtin_ctzll(m);
      const int q0 = __builtin_amdgcn_readlane(first, r), q1 = q0 + __builtin_amdgcn_readlane(len, r);
      const int s0 = __builtin_amdgcn_readlane(s[0], r), s1 = __builtin_amdgcn_readlane(s[1], r);
      const int s2 = __builtin_amdgcn_readlane(s[2], r);
      for (int q = q0; q < q1; q += 64) {  // wave-uniform trip count
        const int64_t c = q + lane;
        bool ok = false;
        int j = 0;
        int S[3] = {0, 0, 0};
        if (c < q1) {
          const double f[3] = {w[3 * c] + s0, w[3 * c + 1] + s1, w[3 * c + 2] + s2};
          double d2 = 0.0;
          for (int k = 0; k < 3; ++k) {
            const double xk = f[0] * p.cell[k] + f[1] * p.cell[3 + k] + f[2] * p.cell[6 + k];
            d2 += (xk - xi[k]) * (xk - xi[k]);
          }
          ok = d2 < p.c2 && !(c == slot && s0 == 0 && s1 == 0 && s2 == 0);
          if (ok) {
            j = order[c];
            S[0] = s0 - off[3 * c] + oi[0];
            S[1] = s1 - off[3 * c + 1] + oi[1];
            S[2] = s2 - off[3 * c + 2] + oi[2];
          }
        }
        hit(ok, j, S);
      }
    }
  }
}

// One wave per receiver: counts[i] = pairs of i. status[0] = 1 if any receiver exceeds the per-receiver
// capacity of the fill kernel or a shift does not fit the packed key, status[1] = the largest count.
// (25,000 atoms, 84 pairs each: 180 us bin by bin, 58 us by runs.)
__global__ void __launch_bounds__(256) nl_count_kernel(NLPlan p, const double* __restrict__ w,
                                                       const int32_t* __restrict__ off,
                                                       const int64_t* __restrict__ head,
                                                       const int32_t* __restrict__ order,
                                                       const int32_t* __restrict__ bin, int32_t* __restrict__ counts,
                                                       int32_t* __restrict__ status) {
  __shared__ int most[4];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int64_t at = (int64_t)blockIdx.x * 4 + wave;
  int cnt = 0;
  if (at < p.n) {
    const int i = order[at];
    bool bad = false;
    nl_visit(p, at, bin[i], w, off, head, order, lane, [&](bool ok, int, const int* S) {
      cnt += __popcll(__ballot(ok));
      if (ok)
        for (int k = 0; k < 3; ++k) bad |= S[k] <= -kNLShiftBias || S[k] >= kNLShiftBias;
    });
    bad = __any(bad) || cnt > kNLMaxPerAtom;
    if (lane == 0) {
      counts[i] = cnt;
      if (bad) atomicOr(status, 1);
    }
  }
  if (lane == 0) most[wave] = cnt;
  __syncthreads();
  if (threadIdx.x == 0) {
    const int m = max(max(most[0], most[1]), max(most[2], most[3]));
    if (m > status[1]) atomicMax(status + 1, m);  // (a stale read costs an atomic, no more)
  }
}

// One 64-thread workgroup per receiver: collect the (j, S) keys in LDS (room for the largest count, rounded
// up to a power of two), sort, write. (25,000 atoms, 84 pairs each: 218 us bin by bin, 94 us by runs.)
__global__ void __launch_bounds__(64) nl_fill_kernel(NLPlan p, const double* __restrict__ w,
                                                     const int32_t* __restrict__ off, const int64_t* __restrict__ head,
                                                     const int32_t* __restrict__ order,
                                                     const int32_t* __restrict__ bin,
                                                     const int64_t* __restrict__ rowptr, int64_t* __restrict__ out_i,
                                                     int64_t* __restrict__ out_j, int32_t* __restrict__ out_shift) {
  extern __shared__ uint64_t keys[];
  const int lane = threadIdx.x;
  const int64_t slot = blockIdx.x;
  const int i = order[slot];
  const int64_t start = rowptr[i];
  const int cnt = (int)(rowptr[i + 1] - start);
  int fillc = 0;
  nl_visit(p, slot, bin[i], w, off, head, order, lane, [&](bool ok, int j, const int* S) {
    const uint64_t m = __ballot(ok);
    if (ok) {
      const int at = fillc + __popcll(m & ((1ull << lane) - 1ull));
      keys[at] = ((uint64_t)(uint32_t)j << 32) | ((uint64_t)(S[0] + kNLShiftBias) << 20) |
                 ((uint64_t)(S[1] + kNLShiftBias) << 10) | (uint64_t)(S[2] + kNLShiftBias);
    }
    fillc += __popcll(m);
  });
  int P = 1;
  while (P < cnt) P <<= 1;
  for (int t = cnt + lane; t < P; t += 64) keys[t] = ~0ull;
  __syncthreads();
  for (int k = 2; k <= P; k <<= 1)
    for (int jj = k >> 1; jj > 0; jj >>= 1) {
      for (int h = lane; h < P / 2; h += 64) {  // pair h of this step: t and t + jj
        const int t = ((h & ~(jj - 1)) << 1) | (h & (jj - 1)), u = t + jj;
        const uint64_t a = keys[t], b = keys[u];
        const bool up = (t & k) == 0;
        if ((a > b) == up) {
          keys[t] = b;
          keys[u] = a;
        }
      }
      __syncthreads();
    }
  for (int t = lane; t < cnt; t += 64) {
    const uint64_t key = keys[t];
    out_i[start + t] = i;
    out_j[start + t] = (int64_t)(key >> 32);
    out_shift[3 * (start + t)] = (int32_t)((key >> 20) & 1023u) - kNLShiftBias;
    out_shift[3 * (start + t) + 1] = (int32_t)((key >> 10) & 1023u) - kNLShiftBias;
    out_shift[3 * (start + t) + 2] = (int32_t)(key & 1023u) - kNLShiftBias;
  }
}

static void nl_cross(const double* a, const double* b, double* c) {
  c[0] = a[1] * b[2] - a[2] * b[1];
  c[1] = a[2] * b[0] - a[0] * b[2];
  c[2] = a[0] * b[1] - a[1] * b[0];
}

// What the host reads before the fill: status (see nl_count_kernel) and the number of pairs.
struct NLResult {
  int32_t status[2];
  int64_t total;
};

// Workspace layout (bytes, 256-aligned pieces); the bin count is capped at 4n + 64.
struct NLWorkspace {
  double* w;
  double* range;
  int32_t* off;
  int32_t* bin;
  int32_t* order;
  int32_t* hist;
  int32_t* counts;
  NLResult* status;
  int64_t* head;
  int64_t* rowptr;
};

static int64_t nl_max_bins(int64_t n) { return 4 * n + 64; }

static int64_t nl_layout(int64_t n, char* base, NLWorkspace* ws) {
  int64_t o = 0;
  auto take = [&](int64_t bytes) {
    const int64_t at = o;
    o += (bytes + 255) / 256 * 256;
    return base ? base + at : nullptr;
  };
  const int64_t nb = nl_max_bins(n);
  NLWorkspace t{};
  t.w = reinterpret_cast<double*>(take(3 * n * sizeof(double)));
  t.range = reinterpret_cast<double*>(take(6 * sizeof(double)));
  t.off = reinterpret_cast<int32_t*>(take(3 * n * sizeof(int32_t)));
  t.bin = reinterpret_cast<int32_t*>(take(n * sizeof(int32_t)));
  t.order = reinterpret_cast<int32_t*>(take(n * sizeof(int32_t)));
  t.hist = reinterpret_cast<int32_t*>(take((nb + 1) * sizeof(int32_t)));
  t.counts = reinterpret_cast<int32_t*>(take((n + 1) * sizeof(int32_t)));
  t.status = reinterpret_cast<NLResult*>(take(sizeof(NLResult)));
  t.head = reinterpret_cast<int64_t*>(take((nb + 1) * sizeof(int64_t)));
  t.rowptr = reinterpret_cast<int64_t*>(take((n + 1) * sizeof(int64_t)));
  if (ws) *ws = t;
  return o;
}

}  // namespace fc

using namespace fc;

extern "C" int64_t fc_neighbor_list_device_workspace(int64_t n) {
  if (n < 0) return -FC_ERR_SHAPE;
  return nl_layout(n, nullptr, nullptr);
}

namespace fc {

// The list from positions in HBM, with its working arrays laid out from `workspace` (at least
// nl_layout(n) bytes, already checked by the caller). Returns the pair count or -fc_status.
static int64_t nl_build(int64_t n, const double* pos, const double* cell, const int32_t* pbc, double cutoff,
                        int64_t capacity, int64_t* out_i, int64_t* out_j, int32_t* out_shift, void* workspace,
                        hipStream_t s) {
  NLWorkspace ws;
  nl_layout(n, reinterpret_cast<char*>(workspace), &ws);

  NLPlan p{};
  p.n = n;
  for (int k = 0; k < 9; ++k) p.cell[k] = cell[k];
  for (int k = 0; k < 3; ++k) p.pbc[k] = pbc[k] ? 1 : 0;
  const double* m = cell;
  const double det = m[0] * (m[4] * m[8] - m[5] * m[7]) - m[1] * (m[3] * m[8] - m[5] * m[6]) +
                     m[2] * (m[3] * m[7] - m[4] * m[6]);
  if (std::fabs(det) < 1e-300) return -FC_ERR_BAD_DESC;
  {  // the host list's inverse, operation for operation
    const double id = 1.0 / det;
    p.inv[0] = (m[4] * m[8] - m[5] * m[7]) * id;
    p.inv[1] = (m[2] * m[7] - m[1] * m[8]) * id;
    p.inv[2] = (m[1] * m[5] - m[2] * m[4]) * id;
    p.inv[3] = (m[5] * m[6] - m[3] * m[8]) * id;
    p.inv[4] = (m[0] * m[8] - m[2] * m[6]) * id;
    p.inv[5] = (m[2] * m[3] - m[0] * m[5]) * id;
    p.inv[6] = (m[3] * m[7] - m[4] * m[6]) * id;
    p.inv[7] = (m[1] * m[6] - m[0] * m[7]) * id;
    p.inv[8] = (m[0] * m[4] - m[1] * m[3]) * id;
  }
  double reach[3];
  {
    double vv[3];
    nl_cross(cell + 3, cell + 6, vv);
    const double vol = std::fabs(cell[0] * vv[0] + cell[1] * vv[1] + cell[2] * vv[2]);
    for (int k = 0; k < 3; ++k) {
      double c[3];
      nl_cross(cell + 3 * ((k + 1) % 3), cell + 3 * ((k + 2) % 3), c);
      reach[k] = cutoff / (vol / std::sqrt(c[0] * c[0] + c[1] * c[1] + c[2] * c[2]));
    }
  }
  p.c2 = cutoff * cutoff;
  const int bs = 256;
  const unsigned g_atoms = (unsigned)((n + bs - 1) / bs);
  double lo[3] = {0, 0, 0}, hi[3] = {1, 1, 1};
  if (!(p.pbc[0] && p.pbc[1] && p.pbc[2])) {
    double r[6];
    hipLaunchKernelGGL(nl_range_kernel, dim3(1), dim3(256), 0, s, p, pos, ws.range);
    if (hipGetLastError() != hipSuccess) return -FC_ERR_LAUNCH;
    if (hipMemcpyAsync(r, ws.range, sizeof(r), hipMemcpyDeviceToHost, s) != hipSuccess ||
        hipStreamSynchronize(s) != hipSuccess)
      return -FC_ERR_LAUNCH;
    for (int k = 0; k < 3; ++k)
      if (!p.pbc[k]) { lo[k] = r[k]; hi[k] = r[3 + k]; }
  }
  // Bins of fractional width >= reach (1e-6 margin: rounding of the coordinates never puts
  // two atoms closer than the cutoff two bins apart). Periodic axes: D = ceil(reach / width)
  // neighbouring bins each way (several images when the cell is thinner than the cutoff).
  for (int k = 0; k < 3; ++k) {
    const double span = hi[k] - lo[k], fit = std::floor(span / (reach[k] * (1.0 + 1e-6)));
    p.nb[k] = !(fit > 1) ? 1 : (fit > 512 ? 512 : (int)fit);
    p.base[k] = lo[k];
  }
  while ((int64_t)p.nb[0] * p.nb[1] * p.nb[2] > nl_max_bins(n)) {  // coarser bins for sparse systems
    int k = 0;
    for (int q = 1; q < 3; ++q)
      if (p.nb[q] > p.nb[k]) k = q;
    p.nb[k] = (p.nb[k] + 1) / 2;
  }
  for (int k = 0; k < 3; ++k) {
    const double span = hi[k] - lo[k];
    p.width[k] = span > 0 ? span / p.nb[k] : 1.0;
    const double away = p.pbc[k] ? std::ceil(reach[k] / p.width[k]) : 1.0;
    if (!(away <= kNLMaxBinsAway)) return -FC_ERR_SHAPE;  // (before it is an integer)
    p.D[k] = (int)away;
  }
  const int64_t nbins = (int64_t)p.nb[0] * p.nb[1] * p.nb[2];
  p.ns2 = p.pbc[2] ? (2 * p.D[2] + p.nb[2] - 1) / p.nb[2] + 1 : 1;
  if ((2.0 * p.D[0] + 1.0) * (2.0 * p.D[1] + 1.0) * p.ns2 > kNLMaxRuns) return -FC_ERR_SHAPE;
  int32_t* const status = ws.status->status;
  hipLaunchKernelGGL(nl_init_kernel, dim3((unsigned)((nbins + bs - 1) / bs)), dim3(bs), 0, s, nbins, ws.hist, status);
  hipLaunchKernelGGL(nl_bin_kernel, dim3(g_atoms), dim3(bs), 0, s, p, pos, ws.bin, ws.hist);
  hipLaunchKernelGGL(nl_scan_kernel, dim3(1), dim3(1024), 0, s, nbins, ws.hist, ws.head, (int64_t*)nullptr);
  hipLaunchKernelGGL(nl_scatter_kernel, dim3(g_atoms), dim3(bs), 0, s, p, pos, ws.bin, ws.head, ws.hist, ws.w, ws.off,
                     ws.order);
  hipLaunchKernelGGL(nl_count_kernel, dim3((unsigned)((n + 3) / 4)), dim3(256), 0, s, p, ws.w, ws.off, ws.head,
                     ws.order, ws.bin, ws.counts, status);
  hipLaunchKernelGGL(nl_scan_kernel, dim3(1), dim3(1024), 0, s, n, ws.counts, ws.rowptr, &ws.status->total);
  if (hipGetLastError() != hipSuccess) return -FC_ERR_LAUNCH;
  NLResult res{};
  if (hipMemcpyAsync(&res, ws.status, sizeof(res), hipMemcpyDeviceToHost, s) != hipSuccess ||
      hipStreamSynchronize(s) != hipSuccess)
    return -FC_ERR_LAUNCH;
  const int64_t total = res.total;
  if (res.status[0]) return -FC_ERR_SHAPE;  // > 1024 pairs for one atom, or |S| >= 512
  if (total > capacity || total == 0) return total;
  if (!out_i || !out_j || !out_shift) return -FC_ERR_NULL;
  unsigned room = 64;
  while (room < (unsigned)res.status[1]) room <<= 1;
  hipLaunchKernelGGL(nl_fill_kernel, dim3((unsigned)n), dim3(64), room * sizeof(uint64_t), s, p, ws.w, ws.off, ws.head,
                     ws.order, ws.bin, ws.rowptr, out_i, out_j, out_shift);
  if (hipGetLastError() != hipSuccess) return -FC_ERR_LAUNCH;
  return total;
}

static int64_t nl_check_args(int64_t n, const double* pos, const double* cell, const int32_t* pbc, double cutoff) {
  if (n < 0 || !(cutoff > 0.0) || !cell || !pbc) return -FC_ERR_BAD_DESC;
  if (n > 0x7fffffff || (n > 0 && !pos)) return -FC_ERR_SHAPE;
  return 0;
}

// Working memory of the allocation-free entry point: one copy of this array per device (a module
// global), held until the process ends. Host code never passes `scratch` itself to a kernel or a
// copy (in host code the name is only a stand-in for the symbol): it uses the device address that
// hipGetSymbolAddress returns for the current device, kept in g_scratch_ptr.
constexpr int64_t kNLScratchBytes = int64_t(64) << 20;
static __device__ __align__(256) char scratch[kNLScratchBytes];

constexpr int kMaxDevices = 64;
static std::mutex g_scratch_mu;
static void* g_scratch_ptr[kMaxDevices];

// The current device's address of `scratch` (looked up once per device, with that device current).
static int nl_scratch_address(void** out) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return FC_ERR_LAUNCH;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return FC_ERR_LAUNCH;
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return FC_OK;
}

}  // namespace fc

extern "C" int64_t fc_neighbor_list_device(int64_t n, const double* pos, const double* cell, const int32_t* pbc,
                                           double cutoff, int64_t capacity, int64_t* out_i, int64_t* out_j,
                                           int32_t* out_shift, void* workspace, int64_t workspace_bytes,
                                           void* stream) {
  const int64_t bad = nl_check_args(n, pos, cell, pbc, cutoff);
  if (bad) return bad;
  if (n == 0) return 0;
  if (!workspace || workspace_bytes < nl_layout(n, nullptr, nullptr)) return -FC_ERR_WORKSPACE;
  return nl_build(n, pos, cell, pbc, cutoff, capacity, out_i, out_j, out_shift, workspace, (hipStream_t)stream);
}

extern "C" int64_t fc_neighbor_list_device_noalloc_max_atoms(void) {
  int64_t lo = 0, hi = int64_t(1) << 31;  // largest n whose working arrays fit the scratch array
  while (lo < hi) {
    const int64_t mid = (lo + hi + 1) / 2;
    if (nl_layout(mid, nullptr, nullptr) <= kNLScratchBytes) lo = mid; else hi = mid - 1;
  }
  return lo;
}

extern "C" int64_t fc_neighbor_list_device_noalloc(int64_t n, const double* pos, const double* cell,
                                                   const int32_t* pbc, double cutoff, int64_t capacity,
                                                   int64_t* out_i, int64_t* out_j, int32_t* out_shift,
                                                   void* stream) {
  const int64_t bad = nl_check_args(n, pos, cell, pbc, cutoff);
  if (bad) return bad;
  if (n == 0) return 0;
  if (nl_layout(n, nullptr, nullptr) > kNLScratchBytes) return -FC_ERR_SCRATCH_LIMIT;
  void* base = nullptr;
  const int st = nl_scratch_address(&base);
  if (st != FC_OK) return -st;
  return nl_build(n, pos, cell, pbc, cutoff, capacity, out_i, out_j, out_shift, base, (hipStream_t)stream);
}
