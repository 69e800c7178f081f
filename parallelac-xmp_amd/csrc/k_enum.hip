/*
 * k_enum.hip -- binning, candidate enumeration and the alpha filters.
 *
 * Waves enumerate the candidates of a ball or of 64 alpha edges or
 * triangles (cells of the stencil, rows in each other by bitmaps and masks),
 * 64 at a time whatever item they belong to, classify each with one precision
 * stage (FP32 on the staged path, FP64 on the plain path) and append undecided
 * candidates to a queue.  The escalation kernel re-decides them in FP64 then double-double;
 * what is still undecided goes to the wide-integer kernel.
 *
 * Reference kernels restated (AlphaComplexLargeData.cu unless noted):
 *   k_cell_key           computeCellIndex :65-78
 *   k_edge_count, k_edge_enum_filter  computePossibleEdgeCount / fillPotentialEdges
 *                        :80-165 + markRealEdges :167-190 (fused)
 *   k_tri_hits, k_tri_enum_filter  computePossibleTriangleCount / fillPossibleTriangles
 *                        :192-296 + markRealTriangles :298-348 (fused)
 *   k_tet_enum_filter    computePossibleTetCount / fillPossibleTets :350-529
 *                        + markRealTets :531-591 (fused)
 */
#include "pac_dev.h"
#include "pac_wide.h"

namespace pac {
namespace PAC_V {

/* ------------------------------------------------------------------ */
/* bounds / keys / gather                                              */
/* ------------------------------------------------------------------ */
__device__ __forceinline__ int neg_lsb_exp(float v) {
  uint32_t b = __float_as_uint(v) & 0x7fffffffu;
  if (b == 0) return 0;
  uint32_t E = b >> 23, m = b & 0x7fffffu;
  int e;
  if (E == 0) {
    e = -149;
  } else {
    m |= 0x800000u;
    e = (int)E - 150;
  }
  int lsb = e + __builtin_ctz(m);
  return lsb < 0 ? -lsb : 0;
}

__device__ __forceinline__ int neg_lsb_exp(double v) {
  uint64_t b = (uint64_t)__double_as_longlong(v) & 0x7fffffffffffffffull;
  if (b == 0) return 0;
  uint32_t E = (uint32_t)(b >> 52);
  uint64_t m = b & ((1ull << 52) - 1);
  int e;
  if (E == 0) {
    e = -1074;
  } else {
    m |= 1ull << 52;
    e = (int)E - 1075;
  }
  int lsb = e + __builtin_ctzll(m);
  return lsb < 0 ? -lsb : 0;
}
/* r = r_raw + solvent as the reference computes it (FP32 add,
 * AlphaComplexParallel.cu:1086), or in FP64 for FP64 balls */
__device__ __forceinline__ float add_r(float a, float s) { return __fadd_rn(a, s); }
__device__ __forceinline__ double add_r(double a, double s) { return a + s; }

struct BRed {
  Real v[9];  /* minx miny minz -maxx -maxy -maxz -maxrawr -maxr -maxabs */
  int shift, nonfinite;
};
__device__ void bred_init(BRed& b) {
#pragma unroll
  for (int q = 0; q < 9; ++q) b.v[q] = INFINITY;
  b.shift = 0;
  b.nonfinite = 0;
}
__device__ void bred_merge(BRed& a, const BRed& b) {
#pragma unroll
  for (int q = 0; q < 9; ++q) a.v[q] = fmin(a.v[q], b.v[q]);
  a.shift = max(a.shift, b.shift);
  a.nonfinite += b.nonfinite;
}
__device__ void bred_ball(BRed& b, const Ball& a, Real solvent) {
  if (!isfinite(a.x) || !isfinite(a.y) || !isfinite(a.z) || !isfinite(a.w)) {
    b.nonfinite++;
    return;
  }
  Real r = add_r(a.w, solvent);
  b.v[0] = fmin(b.v[0], a.x);
  b.v[1] = fmin(b.v[1], a.y);
  b.v[2] = fmin(b.v[2], a.z);
  b.v[3] = fmin(b.v[3], -a.x);
  b.v[4] = fmin(b.v[4], -a.y);
  b.v[5] = fmin(b.v[5], -a.z);
  b.v[6] = fmin(b.v[6], -a.w);
  b.v[7] = fmin(b.v[7], -fabs(r));
  b.v[8] = fmin(b.v[8], -fmax(fabs(a.x), fmax(fabs(a.y), fabs(a.z))));
  int s = max(max(neg_lsb_exp(a.x), neg_lsb_exp(a.y)),
              max(neg_lsb_exp(a.z), neg_lsb_exp(r)));
  b.shift = max(b.shift, s);
}
__device__ Bounds bred_out(const BRed& b) {
  Bounds o;
  o.minx = b.v[0];
  o.miny = b.v[1];
  o.minz = b.v[2];
  o.maxx = -b.v[3];
  o.maxy = -b.v[4];
  o.maxz = -b.v[5];
  o.max_raw_r = -b.v[6];
  o.max_r = -b.v[7];
  o.max_abs = -b.v[8];
  o.shift = b.shift;
  o.nonfinite = b.nonfinite;

  return o;
}
__device__ void bred_block(BRed& mine, BRed* sh) {
  sh[threadIdx.x] = mine;
  __syncthreads();
  for (int s = blockDim.x / 2; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) bred_merge(sh[threadIdx.x], sh[threadIdx.x + s]);
    __syncthreads();
  }
  mine = sh[0];
}

/* the reduced bounds to `out`, and posted */
__device__ __forceinline__ void bounds_done(const BRed& b, Bounds* out,
                                            const Post& post, Bounds* s_b,
                                            unsigned long long began) {
  if (threadIdx.x == 0) {
    *s_b = bred_out(b);
    *out = *s_b;
    if (post.box)
      *reinterpret_cast<unsigned long long*>(post.box + kBoxSpan) =
          wall_clock64() - began;
  }
  if (!post.box) return;
  __syncthreads();
  constexpr int kW = sizeof(Bounds) / sizeof(unsigned);
  static_assert(sizeof(Bounds) % sizeof(unsigned) == 0 && kW <= 64, "one wave");
  if (threadIdx.x < kW)
    post.box[kBoxData + threadIdx.x] =
        reinterpret_cast<const unsigned*>(s_b)[threadIdx.x];
  if (threadIdx.x < 64) {
    __threadfence_system();
    if (threadIdx.x == 0)
      __hip_atomic_store(
          reinterpret_cast<unsigned long long*>(post.box + kBoxTicket),
          post.ticket, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}
/* Bounds of the balls; a run's first kernel, so it also clears the run's
 * control words (ctl) and keeps the balls in input order with their final
 * radii (orig, for alpha values and the adjoint), each where given.  A
 * single block's partial is the result. */
__global__ __launch_bounds__(kBlock) void k_bounds_part(
    const Ball* raw, int64_t n, Real solvent, BRed* part, Bounds* out,
    double4* orig, unsigned long long* ctl, int ctl_words, Post post) {
  __shared__ BRed sh[kBlock];
  __shared__ Bounds s_b;
  const unsigned long long began = wall_clock64();
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  if (ctl) {
    for (int64_t i = gtid(); i < ctl_words; i += stride)
      ctl[i] = i == ctl_words - kStamps + TS_GRID ? began : 0ull;
  }
  BRed b;
  bred_init(b);
  for (int64_t i = gtid(); i < n; i += stride) {
    const Ball a = raw[i];
    bred_ball(b, a, solvent);
    if (orig)
      orig[i] = make_double4(a.x, a.y, a.z, (double)add_r(a.w, solvent));
  }
  bred_block(b, sh);
  if (gridDim.x == 1)
    bounds_done(b, out, post, &s_b, began);
  else if (threadIdx.x == 0)
    part[blockIdx.x] = b;
}
__global__ __launch_bounds__(kBlock) void k_bounds_final(const BRed* part,
                                                         int np, Bounds* out,
                                                         const uint64_t* ts,
                                                         Post post) {
  __shared__ BRed sh[kBlock];
  __shared__ Bounds s_b;
  const unsigned long long began = ts ? ts[TS_GRID] : wall_clock64();
  BRed b;
  bred_init(b);
  for (int i = threadIdx.x; i < np; i += blockDim.x) bred_merge(b, part[i]);
  bred_block(b, sh);
  bounds_done(b, out, post, &s_b, began);
}
void launch_bounds(const Ball* raw, int64_t n, Real solvent, Bounds* part,
                   Bounds* out, double4* orig, unsigned long long* ctl,
                   int ctl_words, Post post, PipeLaunch L) {
  /* one block up to 2048 balls: a second launch costs more than 8 balls a
   * thread */
  int nb = n <= 2048 ? 1
                     : (int)std::min<int64_t>(1024, (n + kBlock - 1) / kBlock);
  hipLaunchKernelGGL(k_bounds_part, dim3(nb), dim3(kBlock), 0, L.s, raw, n,
                     solvent, (BRed*)part, out, orig, ctl, ctl_words, post);
  if (nb > 1)
    hipLaunchKernelGGL(k_bounds_final, dim3(1), dim3(kBlock), 0, L.s,
                       (const BRed*)part, nb, out,
                       ctl ? (const uint64_t*)ctl + ctl_words - kStamps
                           : nullptr, post);
}

/* Per-molecule bounds of a batch: block m reduces the balls of molecule m
 * (a few hundred to tens of thousands each). */
__global__ __launch_bounds__(kBlock) void k_bounds_mol(const Ball* raw,
                                                       const uint32_t* moff,
                                                       Real solvent,
                                                       Bounds* out,
                                                       unsigned long long* ts) {
  stamp(ts, TS_GRID);
  __shared__ BRed sh[kBlock];
  const uint32_t m = blockIdx.x, b0 = moff[m], b1 = moff[m + 1];
  BRed b;
  bred_init(b);
  for (uint32_t i = b0 + threadIdx.x; i < b1; i += blockDim.x)
    bred_ball(b, raw[i], solvent);
  bred_block(b, sh);
  if (threadIdx.x == 0) out[m] = bred_out(b);
}
void launch_bounds_mol(const Ball* raw, const uint32_t* moff, int64_t nmol,
                       Real solvent, Bounds* out, unsigned long long* ts,
                       PipeLaunch L) {
  if (nmol <= 0) return;
  hipLaunchKernelGGL(k_bounds_mol, dim3((unsigned)nmol), dim3(kBlock), 0, L.s,
                     raw, moff, solvent, out, ts);
}

__global__ __launch_bounds__(kBlock) void k_mol_ids(const uint32_t* moff,
                                                    int64_t nmol, int64_t n,
                                                    uint32_t* mol) {
  int64_t i = gtid();
  if (i >= n) return;
  /* last m with moff[m] <= i */
  int64_t lo = 0, hi = nmol - 1;
  while (lo < hi) {
    int64_t mid = (lo + hi + 1) >> 1;
    if ((int64_t)moff[mid] <= i) lo = mid;
    else hi = mid - 1;
  }
  mol[i] = (uint32_t)lo;
}
void launch_mol_ids(const uint32_t* moff, int64_t nmol, int64_t n,
                    uint32_t* mol, PipeLaunch L) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_mol_ids, dim3((unsigned)((n + kBlock - 1) / kBlock)),
                     dim3(kBlock), 0, L.s, moff, nmol, n, mol);
}

/* computeCellIndex (LD:65-78): FP32 subtract, IEEE divide, truncate; in a
 * batch the molecule's first global cell id is added.  idx: the ball, or
 * with the cells' counts (cleared) its place among the balls of its cell, in
 * the order they arrive, counted a run of lanes at a time: 20,000 balls in one
 * cell 6 us, 230 with an atomic each. */
__global__ __launch_bounds__(kBlock) void k_cell_key(const Ball* raw,
                                                     int64_t n, GridP g1,
                                                     const GridP* grids,
                                                     const uint32_t* mol,
                                                     uint32_t* key,
                                                     uint32_t* idx,
                                                     uint32_t* cnt) {
  int64_t i = gtid();
  if (i >= n) return;
  const GridP g = mol ? grids[mol[i]] : g1;
  Ball a = raw[i];
  /* FP64 balls are keyed by their FP32 roundings (monotone, so every key
   * stays inside the grid; the host widens the search margin by the
   * rounding) */
  int cx = (int)__fdiv_rn(__fsub_rn((float)a.x, g.minx), g.step);
  int cy = (int)__fdiv_rn(__fsub_rn((float)a.y, g.miny), g.step);
  int cz = (int)__fdiv_rn(__fsub_rn((float)a.z, g.minz), g.step);
  /* balls always key inside the grid planned from their own bounds; the
   * clamp only keeps a recorded pipeline in bounds after its input moved
   * (that run is then reported stale) */
  cx = min(max(cx, 0), g.ex - 1);
  cy = min(max(cy, 0), g.ey - 1);
  cz = min(max(cz, 0), g.ez - 1);
  const uint32_t c = g.cbase + (uint32_t)(cx + g.ex * cy + g.ex * g.ey * cz);
  key[i] = c;
  idx[i] = cnt ? count_run(cnt, c) : (uint32_t)i;
}
void launch_cell_key(const Ball* raw, int64_t n, GridP g,
                     const GridP* grids, const uint32_t* mol, uint32_t* key,
                     uint32_t* idx, uint32_t* cnt, PipeLaunch L) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_cell_key, dim3((unsigned)((n + kBlock - 1) / kBlock)),
                     dim3(kBlock), 0, L.s, raw, n, g, grids, mol, key, idx, cnt);
}

/* the balls by cell, in each cell as they arrived, and their cells */
__global__ __launch_bounds__(kBlock) void k_cell_put(int64_t n,
                                                     const uint32_t* key,
                                                     const uint32_t* place,
                                                     const uint32_t* cstart,
                                                     uint32_t* sidx,
                                                     uint32_t* cellk) {
  const int64_t i = gtid();
  if (i >= n) return;
  const uint32_t c = key[i], at = cstart[c] + place[i];
  sidx[at] = (uint32_t)i;
  cellk[at] = c;
}
void launch_cell_put(int64_t n, const uint32_t* key, const uint32_t* place,
                     const uint32_t* cstart, uint32_t* sidx, uint32_t* cellk,
                     PipeLaunch L) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_cell_put, dim3((unsigned)((n + kBlock - 1) / kBlock)),
                     dim3(kBlock), 0, L.s, n, key, place, cstart, sidx, cellk);
}
struct __attribute__((packed, aligned(4))) U4a4 { /* 16 bytes at any word */
  uint32_t x, y, z, w;
};
/* Each ball to its place by cell and id: as many after its cell's start as
 * the cell holds smaller ids.  A cell of m balls walks m^2 ids and has
 * m (m - 1) / 2 edge candidates: this runs after the candidates were counted
 * and found below 2^32, so at most 2^33 ids in all.  A cell of 20,000: 296 us
 * with 32 ids in flight a thread, 1,496 one by one. */
__global__ __launch_bounds__(kBlock) void k_cell_order(
    const Ball* raw, int64_t n, const uint32_t* sidx, const uint32_t* cellk,
    const uint32_t* cstart, Real solvent, Ball* ball, uint32_t* perm,
    unsigned long long* ts) {
  stamp(ts, TS_ORDER);
  const int64_t s = gtid();
  if (s >= n) return;
  const uint32_t o = sidx[s];
  const Ball a = raw[o];
  const uint32_t c = cellk[s], b = cstart[c], e = cstart[c + 1];
  uint32_t at = b, t = b;
  for (; t + 32 <= e; t += 32) {
    U4a4 x[8];
#pragma unroll
    for (int k = 0; k < 8; ++k)
      x[k] = *reinterpret_cast<const U4a4*>(sidx + t + 4 * k);
#pragma unroll
    for (int k = 0; k < 8; ++k)
      at += (x[k].x < o) + (x[k].y < o) + (x[k].z < o) + (x[k].w < o);
  }
  for (; t < e; t += 8) {
    uint32_t x[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) x[k] = sidx[t + k < e ? t + k : b];
#pragma unroll
    for (int k = 0; k < 8; ++k) at += t + k < e && x[k] < o;
  }
  ball[at] = Ball{a.x, a.y, a.z, add_r(a.w, solvent)};
  perm[at] = o;
}
void launch_cell_order(const Ball* raw, int64_t n, const uint32_t* sidx,
                       const uint32_t* cellk, const uint32_t* cstart,
                       Real solvent, Ball* ball, uint32_t* perm,
                       unsigned long long* ts, PipeLaunch L) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_cell_order, dim3((unsigned)((n + kBlock - 1) / kBlock)),
                     dim3(kBlock), 0, L.s, raw, n, sidx, cellk, cstart, solvent,
                     ball, perm, ts);
}

__global__ __launch_bounds__(kBlock) void k_gather(const Ball* raw,
                                                   const uint32_t* sidx,
                                                   const uint32_t* skey,
                                                   int64_t n, Real solvent,
                                                   Ball* ball, uint32_t* perm,
                                                   uint32_t* cellk) {
  int64_t s = gtid();
  if (s >= n) return;
  uint32_t o = sidx[s];
  Ball a = raw[o];
  ball[s] = Ball{a.x, a.y, a.z, add_r(a.w, solvent)};
  perm[s] = o;
  cellk[s] = skey[s];
}
void launch_gather(const Ball* raw, const uint32_t* sidx,
                   const uint32_t* skey, int64_t n, Real solvent,
                   Ball* ball, uint32_t* perm, uint32_t* cellk,
                   PipeLaunch L) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_gather, dim3((unsigned)((n + kBlock - 1) / kBlock)),
                     dim3(kBlock), 0, L.s, raw, sidx, skey, n, solvent, ball,
                     perm, cellk);
}

/* cstart[c] = first sorted ball with key >= c, for c in [0, G]: one
 * thread per cell, binary search over the sorted keys (neighbouring cells
 * share the first probes, so the search runs from cache; a grid that is
 * mostly empty -- a chunk's sub-input on the whole input's grid -- costs no
 * serial fill of its empty runs) */
__global__ __launch_bounds__(kBlock) void k_cell_starts(const uint32_t* cellk,
                                                        int64_t n, int64_t G,
                                                        uint32_t* cstart) {
  const int64_t c = gtid();
  if (c > G) return;
  int64_t lo = 0, hi = n;
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if ((int64_t)cellk[mid] < c)
      lo = mid + 1;
    else
      hi = mid;
  }
  cstart[c] = (uint32_t)lo;
}
void launch_cell_starts(const uint32_t* cellk, int64_t n, int64_t G,
                        uint32_t* cstart, PipeLaunch L) {
  hipLaunchKernelGGL(k_cell_starts,
                     dim3((unsigned)((G + 1 + kBlock - 1) / kBlock)),
                     dim3(kBlock), 0, L.s, cellk, n, G, cstart);
}

/* Fine scan grid: each reference cell split into kx cells along x.  One
 * thread per reference cell partitions its balls (in order) by x
 * sub-cell, (x - minx) * kx / step in double clamped into the cell: a ball
 * the FP32 key put in a neighbouring cell is off by less than the grid's
 * margin, which every scan radius includes. */
__global__ __launch_bounds__(kBlock) void k_fine_split(
    const Ball* ball, const uint32_t* cstart, int64_t G, int kx, GridP g1,
    const GridP* grids, const uint32_t* mol, Ball* fball, uint32_t* fid,
    uint32_t* fstart) {
  const int64_t c = gtid();
  if (c >= G) return;
  const uint32_t b0 = cstart[c], b1 = cstart[c + 1];
  uint32_t cnt[kMaxFine];
#pragma unroll
  for (int q = 0; q < kMaxFine; ++q) cnt[q] = 0;
  int base = 0;
  GridP g = g1;
  if (b1 > b0) {
    if (mol) g = grids[mol[b0]];
    /* g is the fine grid: its cell ids and x extent are kx times the
     * reference grid's */
    const int64_t local = c - (int64_t)(g.cbase / (uint32_t)kx);
    base = (int)(local % (g.ex / kx)) * kx; /* first fine x index of the cell */
    for (uint32_t i = b0; i < b1; ++i) {
      const double q = ((double)ball[i].x - (double)g.minx) * g.inv_step - base;
      const int s = q >= 1.0 ? min((int)fmin(q, 64.0), kx - 1) : 0;
#pragma unroll
      for (int t = 0; t < kMaxFine; ++t) cnt[t] += (t == s);
    }
  }
  uint32_t off[kMaxFine];
  uint32_t acc = b0;
#pragma unroll
  for (int t = 0; t < kMaxFine; ++t) {
    off[t] = acc;
    if (t < kx) fstart[c * kx + t] = acc;
    acc += cnt[t];
  }
  if (c == G - 1) fstart[G * kx] = b1;
  for (uint32_t i = b0; i < b1; ++i) {
    const double q = ((double)ball[i].x - (double)g.minx) * g.inv_step - base;
    const int s = q >= 1.0 ? min((int)fmin(q, 64.0), kx - 1) : 0;
    uint32_t at = 0;
#pragma unroll
    for (int t = 0; t < kMaxFine; ++t)
      if (t == s) at = off[t]++;
    fball[at] = ball[i];
    fid[at] = i;
  }
}
void launch_fine_split(const Ball* ball, const uint32_t* cstart, int64_t G,
                       int kx, GridP g, const GridP* grids,
                       const uint32_t* mol, Ball* fball, uint32_t* fid,
                       uint32_t* fstart, PipeLaunch L) {
  if (G <= 0) return;
  hipLaunchKernelGGL(k_fine_split, dim3((unsigned)((G + kBlock - 1) / kBlock)),
                     dim3(kBlock), 0, L.s, ball, cstart, G, kx, g, grids, mol,
                     fball, fid, fstart);
}

/* ------------------------------------------------------------------ */
/* filter decisions (one stage) and exact decisions                    */
/* ------------------------------------------------------------------ */
template <class T>
__device__ int edge_code(const Ball& a, const Ball& b, Real alpha) {
  T v = edge_val(Ld<T>::p(a), Ld<T>::w(a), Ld<T>::p(b), Ld<T>::w(b),
                 Al<T>::c(alpha));
  return code_of(fe_sign(v));
}
/* exact decisions over the wavefront-cooperative integers (every lane of
 * a group of kTPI lanes calls them with the same balls) */
using XI = CW<kTPI>;
__device__ int edge_exact(const Ball& a, const Ball& b,
                          const ExactScale& X) {
  if (same_pos(a, b)) return REJECT;
  const LdCW<kTPI> L{X.S};
  XI v = edge_val(L.p(a), L.w(a), L.p(b), L.w(b), cw_of<kTPI>(X.alpha));
  return fe_sign(v) >= 0 ? KEEP : REJECT;
}

template <class T>
__device__ int tri_code(const Ball& a, const Ball& b, const Ball& c,
                        Real alpha) {
  T nn;
  T v = tri_val(Ld<T>::p(a), Ld<T>::w(a), Ld<T>::p(b), Ld<T>::w(b),
                Ld<T>::p(c), Ld<T>::w(c), Al<T>::c(alpha), &nn);
  if (fe_sign(nn) <= 0) return UNDEC;
  return code_of(fe_sign(v));
}
__device__ int tri_exact(const Ball& a, const Ball& b, const Ball& c,
                         const ExactScale& X) {
  const LdCW<kTPI> L{X.S};
  XI nn;
  XI v = tri_val(L.p(a), L.w(a), L.p(b), L.w(b), L.p(c), L.w(c),
                 cw_of<kTPI>(X.alpha), &nn);
  if (fe_sign(nn) == 0) return REJECT;
  return fe_sign(v) >= 0 ? KEEP : REJECT;
}

template <class T>
__device__ int tet_code(const Ball& a, const Ball& b, const Ball& c,
                        const Ball& d, Real alpha) {
  T D;
  V3<T> N;
  T wa = Ld<T>::w(a);
  tet_DN(Ld<T>::p(a), wa, Ld<T>::p(b), Ld<T>::w(b), Ld<T>::p(c), Ld<T>::w(c),
         Ld<T>::p(d), Ld<T>::w(d), &D, &N);
  if (fe_sign(D) == 0) return UNDEC;
  return code_of(fe_sign(tet_val(D, N, wa, Al<T>::c(alpha))));
}
/* The first stages of the edge and triangle filters, semi-static as
 * tet_dn_ss: each value evaluated once in precision R together with its
 * permanent (the same expression on absolute values, subtractions made
 * additions), its bound the rounding count k times u times the permanent
 * (ss_fe), leaves u, v = p - p_a and w = r^2 rounded once, alpha exact,
 * products by 2 and 4 exact.
 *   edge: V = 4 |u|^2 (w_a + alpha) - A^2, A = |u|^2 + w_a - w_b: A^2 15,
 *   V 16;
 *   triangle: |n|^2 (n = u x v) 11, and V = 4 |n|^2 (w_a + alpha) -
 *   (A^2 |v|^2 - 2 A B u.v + B^2 |u|^2), A = |u|^2 + w_a - w_b,
 *   B = |v|^2 + w_a - w_c: A^2 |v|^2 21, its sum 23, V 24.
 * The same values as edge_val / tri_val; the bound replaces a running
 * error per operation (~4x the instructions for triangles). */
template <class R>
__device__ __forceinline__ int edge_code_ss(const Ball& a, const Ball& b,
                                            Real alpha) {
  const R ux = (R)b.x - (R)a.x, uy = (R)b.y - (R)a.y, uz = (R)b.z - (R)a.z;
  const R wa = (R)a.w * (R)a.w, wb = (R)b.w * (R)b.w, al = (R)alpha;
  const R uu = dot3(ux, uy, uz, ux, uy, uz);
  const R A = (uu + wa) - wb, Ap = (uu + wa) + wb;
  const R u4 = (R)4 * uu;
  const R V = fmaR(u4, wa + al, -(A * A));
  const R Vp = fmaR(u4, wa + fabs(al), Ap * Ap);
  return code_of(fe_sign(ss_fe(SS<R>{V, Vp}, 16)));
}
/* A rejected triangle (a, b, c) also tells which of its edges one ball
 * covers.  The points of equal power to a and b with that power <= alpha
 * are a disk around the edge's centre; c's power minus theirs is affine on
 * the disk's plane and vanishes nowhere on the disk (such a point would be
 * a common orthocentre of value <= alpha), so its sign at the edge's
 * centre, the sign of c's barycentric coordinate of the triangle's
 * orthocentre, is its sign on the whole disk.  Negative: every alpha
 * simplex with the edge ab has its orthocentre on the disk, where c's
 * power is strictly below the simplex's value, and is not empty.
 * The coordinates (times 2 |n|^2 > 0): b: A |v|^2 - B u.v, c: B |u|^2 -
 * A u.v, a: 2 |n|^2 minus both; at most 17 roundings on any path of the
 * last (A 7, |v|^2 - u.v 6, their product 14 and two sums; 14 of the
 * others).
 * cover: bit q set when vertex q (a, b, c) certainly covers the opposite
 * edge; set only with the result REJECT. */
template <class R>
__device__ __forceinline__ int tri_code_ss(const Ball& a, const Ball& b,
                                           const Ball& c, Real alpha,
                                           unsigned& cover) {
  cover = 0u;
  const R ax = a.x, ay = a.y, az = a.z;
  const R ux = (R)b.x - ax, uy = (R)b.y - ay, uz = (R)b.z - az;
  const R vx = (R)c.x - ax, vy = (R)c.y - ay, vz = (R)c.z - az;
  const R wa = (R)a.w * (R)a.w, wb = (R)b.w * (R)b.w, wc = (R)c.w * (R)c.w;
  const R n0 = det2(uy, vz, uz, vy), n1 = det2(uz, vx, ux, vz),
          n2 = det2(ux, vy, uy, vx);
  /* permanents of n by max norms, as in tet_dn_ss: 2 |u|_inf |v|_inf each,
   * 12 (|u|_inf |v|_inf)^2 for |n|^2 */
  const R pm = max3(fabs(ux), fabs(uy), fabs(uz)) *
               max3(fabs(vx), fabs(vy), fabs(vz));
  const R nn = dot3(n0, n1, n2, n0, n1, n2);
  const R nnp = ((R)12 * pm) * pm;
  if (fe_sign(ss_fe(SS<R>{nn, nnp}, 11)) <= 0) return UNDEC;
  const R uu = dot3(ux, uy, uz, ux, uy, uz);
  const R vv = dot3(vx, vy, vz, vx, vy, vz);
  const R uv = dot3(ux, uy, uz, vx, vy, vz);
  const R uvp = (R)3 * pm;
  const R A = (uu + wa) - wb, Ap = (uu + wa) + wb;
  const R B = (vv + wa) - wc, Bp = (vv + wa) + wc;
  const R lhs = fmaR(A * A, vv, fmaR(B * B, uu, -((((R)2 * A) * B) * uv)));
  const R lhsp = fmaR(Ap * Ap, vv, fmaR(Bp * Bp, uu, (((R)2 * Ap) * Bp) * uvp));
  const R al = (R)alpha;
  const R V = fmaR((R)4 * nn, wa + al, -lhs);
  const R Vp = fmaR((R)4 * nnp, wa + fabs(al), lhsp);
  const int r = code_of(fe_sign(ss_fe(SS<R>{V, Vp}, 24)));
  if (r == REJECT) {
    const SS<R> lb{det2(A, vv, B, uv), fmaR(Ap, vv, Bp * uvp)};
    const SS<R> lc{det2(B, uu, A, uv), fmaR(Bp, uu, Ap * uvp)};
    const SS<R> la{fmaR(A, uv - vv, fmaR(B, uv - uu, (R)2 * nn)),
                   fmaR(Ap, uvp + vv, fmaR(Bp, uvp + uu, (R)2 * nnp))};
    cover = (fe_sign(ss_fe(la, 18)) < 0 ? 1u : 0u) |
            (fe_sign(ss_fe(lb, 18)) < 0 ? 2u : 0u) |
            (fe_sign(ss_fe(lc, 18)) < 0 ? 4u : 0u);
  }
  return r;
}
/* the first stage of the tet filter: D and N with a-priori error bounds
 * (tet_dn_ss: one extra operation per operation, on absolute values),
 * the final 4 D^2 (w_a + alpha) - |N|^2 with one bound (tet_val_ss) */
template <class R>
__device__ __forceinline__ int tet_code_ss(const Ball* v, Real alpha) {
  TetCert<R> T;
  tet_dn_ss(v, T);
  if (fe_sign(T.D) == 0) return UNDEC;
  return code_of(tet_val_ss(T, (R)alpha));
}
__device__ int tet_exact(const Ball& a, const Ball& b, const Ball& c,
                         const Ball& d, const ExactScale& X) {
  const LdCW<kTPI> L{X.S};
  XI D;
  V3<XI> N;
  XI wa = L.w(a);
  tet_DN(L.p(a), wa, L.p(b), L.w(b), L.p(c), L.w(c), L.p(d), L.w(d), &D, &N);
  if (fe_sign(D) == 0) return REJECT;
  return fe_sign(tet_val(D, N, wa, cw_of<kTPI>(X.alpha))) >= 0 ? KEEP : REJECT;
}

/* ------------------------------------------------------------------ */
/* edges                                                               */
/* ------------------------------------------------------------------ */
__device__ __forceinline__ void cell_xyz(uint32_t c, const GridP& g, int& x,
                                         int& y, int& z) {
  x = (int)(c % (uint32_t)g.ex);
  uint32_t t = c / (uint32_t)g.ex;
  y = (int)(t % (uint32_t)g.ey);
  z = (int)(t / (uint32_t)g.ey);
}

__global__ __launch_bounds__(kBlock) void k_edge_count(Stage S, uint32_t* cnt) {
  stamp(S.ts, TS_EDGES);
  int64_t i = gtid();
  if (i >= S.n) return;
  const GridP g = grid_of(S, (uint32_t)i);
  uint32_t c = S.cellk[i];
  int gx, gy, gz;
  cell_xyz(c - g.cbase, g, gx, gy, gz);
  const int k = g.k_enum;
  uint32_t total = 0;
  for (int z = max(gz - k, 0); z <= min(gz + k, g.ez - 1); ++z)
    for (int y = max(gy - k, 0); y <= min(gy + k, g.ey - 1); ++y) {
      int64_t row = (int64_t)g.cbase + (int64_t)g.ex * (y + (int64_t)g.ey * z);
      int x0 = max(gx - k, 0), x1 = min(gx + k, g.ex - 1);
      int64_t c0 = row + x0, c1 = row + x1;
      if (c1 < (int64_t)c) continue;
      uint32_t b = S.cstart[c0], e = S.cstart[c1 + 1];
      if (b < (uint32_t)i + 1) b = (uint32_t)i + 1;
      if (e > b) total += e - b;
    }
  cnt[i] = total;
}
void launch_edge_count(const Stage& S, uint32_t* cnt, PipeLaunch L) {
  if (S.n <= 0) return;
  hipLaunchKernelGGL(k_edge_count, dim3((unsigned)((S.n + kBlock - 1) / kBlock)),
                     dim3(kBlock), 0, L.s, S, cnt);
}

/* ------------------------------------------------------------------ */
/* triangles: k in row(i) after j and in row(j); tets: l in T(i,j)     */
/* after k, T(i,k), T(j,k)                                             */
/* ------------------------------------------------------------------ */
/* Tet slots of the alpha triangles of a chunk sub-input: the row tail of each,
 * but no slots for the triangles (i,j,k) none of whose vertices is owned --
 * every tet they start has its three lowest vertices unowned, and no owned
 * simplex depends on it */
__global__ __launch_bounds__(kBlock) void k_tail_caps_own(
    Stage S, Cnt c_m, const uint64_t* row, const uint32_t* owner,
    const uint32_t* eleft, const uint32_t* ecol, const uint32_t* tk,
    uint32_t* cap) {
  const int64_t m = c_m.get();
  int64_t q = gtid();
  if (q >= m) return;
  const uint32_t e = owner[q];
  const uint32_t i = eleft[e], j = ecol[e], k = tk[q] & ~kDeadBit;
  const bool need = (i >= S.own_lo && i < S.own_hi) ||
                    (j >= S.own_lo && j < S.own_hi) ||
                    (k >= S.own_lo && k < S.own_hi);
  cap[q] = need ? (uint32_t)(row[e + 1] - (uint64_t)q - 1) : 0u;
}
void launch_tet_caps(const Stage& S, Cnt m, const uint64_t* trow,
                     const uint32_t* tedge, const uint32_t* eleft,
                     const uint32_t* ecol, const uint32_t* tk, uint32_t* cap,
                     PipeLaunch L) {
  if (m.cap <= 0) return;
  hipLaunchKernelGGL(k_tail_caps_own,
                     dim3((unsigned)((m.cap + kBlock - 1) / kBlock)),
                     dim3(kBlock), 0, L.s, S, m, trow, tedge, eleft, ecol, tk,
                     cap);
}

/* orders a wave's LDS and global accesses before those after it */
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}
/* inclusive sum over the lanes */
__device__ __forceinline__ uint32_t wave_prefix(uint32_t x) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const uint32_t y = (uint32_t)__shfl_up((int)x, d, 64);
    if (lane >= d) x += y;
  }
  return x;
}
/* of n entries from base on, those below lim (the arrays' end, which only a
 * recorded pass over its capacity reaches) */
__device__ __forceinline__ uint32_t cut_at(uint32_t n, uint64_t base,
                                           uint64_t lim) {
  const uint64_t room = base < lim ? lim - base : 0;
  return n < room ? n : (uint32_t)room;
}
/* the third vertices of alpha edge (i, j) are row(i) after j, from a on,
 * merged with row(j): hit(k, a, b) for each; two steps a round, each row's
 * next id loaded with its current one (~0 past the end) */
template <class F>
__device__ __forceinline__ void merge_rows(const uint32_t* ecol, uint32_t a,
                                           uint32_t ae, uint32_t b,
                                           uint32_t be, F&& hit) {
  while (a < ae && b < be) {
    const uint32_t x0 = ecol[a], y0 = ecol[b];
    const uint32_t x1 = a + 1u < ae ? ecol[a + 1u] : ~0u;
    const uint32_t y1 = b + 1u < be ? ecol[b + 1u] : ~0u;
    if (x0 == y0) hit(x0, a, b);
    const bool sa = x0 <= y0, sb = y0 <= x0;
    a += sa;
    b += sb;
    const uint32_t x = sa ? x1 : x0, y = sb ? y1 : y0;
    if (x == y && x != ~0u) hit(x, a, b);
    a += (x <= y);
    b += (y <= x);
  }
}
/* the first of the ascending ids at(lo), .. at(hi - 1) not below v, or hi */
template <class F>
__device__ __forceinline__ uint32_t first_from(uint32_t lo, uint32_t hi,
                                               uint32_t v, F&& at) {
  while (lo < hi) {
    const uint32_t m = (lo + hi) >> 1;
    const bool c = at(m) < v;
    lo = c ? m + 1u : lo;
    hi = c ? hi : m;
  }
  return lo;
}
/* Triangle candidates of the alpha edges (computePossibleTriangleCount,
 * Parallel:232-266), a wave per kTriSeg = 64 edges, an edge q = (i, j) a
 * lane: bit t of hits[q] is set if the t-th of row(j) may be in row(i), and
 * cnt[seg] is the wave's number of such bits.
 * The rows of a wave's few i are contiguous in ecol: each goes into an LDS
 * bitmap over the ids modulo its size (512 words shared by the wave's i, so
 * usually 4,096 bits for the ~20 ids of a row), and a lane tests its row(j),
 * four ids a load, instead of merging it with row(i).  The few false hits
 * are dropped by the enumeration; they cost a slot each.  EXACT: they are
 * dropped here, for a recorded pass, whose capacity is one of triangles (how
 * many hits are false also depends on which rows share a wave): an id's bits
 * above its word's place in the bitmap are compared too, and only hits in
 * words that ids of several such values share are looked up in row(i); 61 us
 * for 42 at 100k balls, 120 with every hit of a long row looked up.
 * A wave with a row(j) of more than 128 ids counts by merges and leaves its
 * edges' counts for bits.  39 us at 100k balls (10.6 at 16068), 85 (20) with
 * every lane merging its rows; the loads of the rows and the LDS reads bound
 * it.  ecol is readable up to kEcolPad words past its end. */
template <bool EXACT>
__global__ __launch_bounds__(kBlock) void k_tri_hits(
    Cnt c_ne, const uint64_t* erow, const uint32_t* ecol,
    const uint32_t* eleft, ulonglong2* hits, uint32_t* cnt,
    unsigned long long* ts) {
  static_assert(kTriSeg == 64, "an edge a lane");
  stamp(ts, TS_TRIS);
  constexpr int W = 512; /* words of a wave's bitmaps */
  constexpr int E = EXACT ? 2 : 1; /* words of an entry */
  __shared__ uint4 s_raw[kBlock / 64][W * E / 4];
  const int64_t ne = c_ne.get();
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int64_t seg = gtid() >> 6, q = gtid();
  if (seg * kTriSeg >= ne) { /* a segment past the (device) count */
    if (lane == 0 && seg * kTriSeg < c_ne.cap) cnt[seg] = 0;
    return;
  }
  const bool act = q < ne;
  uint32_t i = ~0u, j = 0, b = 0, len = 0;
  if (act) {
    i = eleft[q];
    j = ecol[q];
    b = (uint32_t)erow[j];
    len = (uint32_t)erow[j + 1] - b;
  }
  uint32_t n = 0;
  if (__ballot(len > 128u) != 0) {
    if (act)
      merge_rows(ecol, (uint32_t)q + 1u, (uint32_t)erow[i + 1], b, b + len,
                 [&](uint32_t, uint32_t, uint32_t) { ++n; });
    if (act) hits[q] = make_ulonglong2(n, 0);
  } else {
    /* the wave's different i: this lane's is number `rank` of them */
    const uint32_t pi = (uint32_t)__shfl_up((int)i, 1, 64);
    const uint64_t heads = __ballot(act && (lane == 0 || i != pi));
    const int nd = __popcll(heads);
    const int rank = __popcll(heads & (~0ull >> (63 - lane))) - 1;
    const int sh = nd > 1 ? 9 - (32 - __builtin_clz((unsigned)nd - 1u)) : 9;
    const uint32_t wm = (1u << sh) - 1u;
    uint32_t* const bm = reinterpret_cast<uint32_t*>(s_raw[wv]);
#pragma unroll
    for (int t = 0; t < W * E / 256; ++t)
      s_raw[wv][64 * t + lane] = make_uint4(0u, 0u, 0u, 0u);
    wave_sync();
    /* the wave's ids of each row: this lane's, and the rest of the last row */
    auto each_id = [&](auto&& f) {
      if (act) f(rank << sh, j);
      if (seg * kTriSeg + 64 < ne) {
        const uint32_t il = (uint32_t)__builtin_amdgcn_readlane((int)i, 63);
        const uint32_t ae = (uint32_t)erow[il + 1];
        for (uint32_t a = (uint32_t)(seg * kTriSeg) + 64u + (uint32_t)lane;
             a < ae; a += 64)
          f((nd - 1) << sh, ecol[a]);
      }
    };
    /* EXACT: beside each word the ids' bits above it, or kMixed where two ids
     * of the row in that word differ there */
    constexpr uint32_t kMixed = ~0u;
    each_id([&](int row, uint32_t y) {
      const uint32_t at = (uint32_t)row + ((y >> 5) & wm);
      atomicOr(&bm[E * at], 1u << (y & 31u));
      if (EXACT) bm[E * at + 1] = y >> (5 + sh);
    });
    wave_sync();
    if constexpr (EXACT) {
      each_id([&](int row, uint32_t y) {
        const uint32_t at = (uint32_t)row + ((y >> 5) & wm);
        if (bm[E * at + 1] != y >> (5 + sh)) bm[E * at + 1] = kMixed;
      });
      wave_sync();
    }
    const uint32_t* const mine = bm + (act ? E * (rank << sh) : 0);
    /* bit 0: a hit; bit 16: a hit in a mixed word */
    auto test = [&](uint32_t y) -> uint32_t {
      const uint32_t at = (y >> 5) & wm;
      if (!EXACT) return (mine[at] >> (y & 31u)) & 1u;
      const uint2 m = reinterpret_cast<const uint2*>(mine)[at];
      const uint32_t in = (m.x >> (y & 31u)) & 1u, p = m.y;
      return p == y >> (5 + sh) ? in : (p == kMixed ? in | in << 16 : 0u);
    };
    uint32_t h[4] = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      if (__ballot(len > 32u * w) == 0) break;
      uint32_t x = 0, mixed = 0;
      for (uint32_t t = 0; t < 32 && __ballot(len > 32u * w + t) != 0; t += 4) {
        U4a4 y = {0u, 0u, 0u, 0u};
        if (32u * w + t < len)
          y = *reinterpret_cast<const U4a4*>(ecol + b + 32u * w + t);
        const uint32_t in =
            test(y.x) | test(y.y) << 1 | test(y.z) << 2 | test(y.w) << 3;
        x |= (in & 15u) << t;
        if (EXACT) mixed |= (in >> 16) << t;
      }
      /* (the ids past the row's end) */
      const uint32_t left = len > 32u * w ? len - 32u * w : 0u;
      const uint32_t in_row = left >= 32u ? ~0u : (1u << left) - 1u;
      h[w] = x & in_row;
      if constexpr (EXACT) {
        for (uint32_t m = mixed & in_row; m; m &= m - 1) {
          const uint32_t t = (uint32_t)__builtin_ctz(m);
          const uint32_t k = ecol[b + 32u * w + t], end = (uint32_t)erow[i + 1];
          const uint32_t a = first_from((uint32_t)q + 1u, end, k,
                                        [&](uint32_t c) { return ecol[c]; });
          if (a >= end || ecol[a] != k) h[w] &= ~(1u << t);
        }
      }
      n += (uint32_t)__popc(h[w]);
    }
    if (act)
      hits[q] = make_ulonglong2((uint64_t)h[1] << 32 | h[0],
                                (uint64_t)h[3] << 32 | h[2]);
  }
  n = wave_prefix(n);
  if (lane == 63) cnt[seg] = n;
}
void launch_tri_hits(Cnt ne, const uint64_t* erow, const uint32_t* ecol,
                     const uint32_t* eleft, ulonglong2* hits, uint32_t* cnt,
                     bool exact, unsigned long long* ts, PipeLaunch L) {
  if (ne.cap <= 0) return;
  auto kf = exact ? k_tri_hits<true> : k_tri_hits<false>;
  hipLaunchKernelGGL(kf, dim3((unsigned)((ne.cap + kBlock - 1) / kBlock)),
                     dim3(kBlock), 0, L.s, ne, erow, ecol, eleft, hits, cnt, ts);
}

/* ------------------------------------------------------------------ */
/* alpha filters, one thread per candidate (uniform work per lane)     */
/* ------------------------------------------------------------------ */
/* vertices of candidate (seg, val): KIND 1 edge (seg = ball), 2 triangle
 * (seg = alpha edge), 3 tet (seg = alpha triangle) */
template <int KIND>
__device__ __forceinline__ void cand_balls(const Stage& S, const CandCtx& C,
                                           int64_t o, uint32_t seg,
                                           uint32_t val, Ball* v) {
  if (KIND == 3) {
    const uint4 t = C.ctet[o];
    v[0] = S.ball[t.x];
    v[1] = S.ball[t.y];
    v[2] = S.ball[t.z];
    v[3] = S.ball[t.w];
  } else if (KIND == 1) {
    v[0] = S.ball[seg];
    v[1] = S.ball[val];
  } else if (KIND == 2) {
    v[0] = S.ball[C.eleft[seg]];
    v[1] = S.ball[C.ecol[seg]];
    v[2] = S.ball[val];
  }
}
template <int KIND, class T>
__device__ __forceinline__ int filter_code(const Ball* v, Real alpha) {
  if (KIND == 1) return same_pos(v[0], v[1]) ? REJECT : edge_code<T>(v[0], v[1], alpha);
  if (KIND == 2) return tri_code<T>(v[0], v[1], v[2], alpha);
  return tet_code<T>(v[0], v[1], v[2], v[3], alpha);
}
/* Degenerate candidates (collinear triangle centres: n = u x v = 0;
 * coplanar tet centres: D = u . (v x t) = 0), which the filter rejects,
 * decided in 128-bit integers on the coordinates scaled by 2^S when their
 * differences fit 40 bits (n's components stay below 2^81, D below 2^123):
 * 1 degenerate, 0 not, -1 out of that range.  Lattice inputs send millions
 * of such candidates past the float stages (D or |n|^2 exactly 0). */
template <int KIND>
__device__ __forceinline__ int degenerate_i128(const Ball* v, int S) {
  constexpr int NB = KIND == 3 ? 4 : 3;
  int64_t d[NB - 1][3];
  double o[3] = {(double)v[0].x, (double)v[0].y, (double)v[0].z};
  int64_t q0[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const double sv = __builtin_ldexp(o[a], S);
    if (!(fabs(sv) < 0x1p62)) return -1;
    q0[a] = (int64_t)sv;
  }
#pragma unroll
  for (int i = 1; i < NB; ++i) {
    const double c[3] = {(double)v[i].x, (double)v[i].y, (double)v[i].z};
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const double sv = __builtin_ldexp(c[a], S);
      if (!(fabs(sv) < 0x1p62)) return -1;
      d[i - 1][a] = (int64_t)sv - q0[a];
      if (d[i - 1][a] >= ((int64_t)1 << 40) || d[i - 1][a] <= -((int64_t)1 << 40))
        return -1;
    }
  }
  const int64_t *u = d[0], *w = d[1];
  const __int128 nx = (__int128)u[1] * w[2] - (__int128)u[2] * w[1];
  const __int128 ny = (__int128)u[2] * w[0] - (__int128)u[0] * w[2];
  const __int128 nz = (__int128)u[0] * w[1] - (__int128)u[1] * w[0];
  if (KIND == 2) return nx == 0 && ny == 0 && nz == 0;
  /* D = t . (u x w), the same determinant as u . (w x t) */
  const int64_t* t = d[NB - 2];
  const __int128 D = (__int128)t[0] * nx + (__int128)t[1] * ny +
                     (__int128)t[2] * nz;
  return D == 0;
}

template <int KIND>
__device__ __forceinline__ int filter_exact(const Ball* v,
                                            const ExactScale& X) {
  if (KIND == 1) return edge_exact(v[0], v[1], X);
  if (KIND == 2) return tri_exact(v[0], v[1], v[2], X);
  return tet_exact(v[0], v[1], v[2], v[3], X);
}
constexpr int fam_of(int KIND) {
  return KIND == 1 ? FAM_EDGE : (KIND == 2 ? FAM_TRI : FAM_TET);
}

/* Tets of alpha triangle q = (i,j,k): l in T(i,j) after k, T(i,k), T(j,k)
 * (computePossibleTetCount / fillPossibleTets, Parallel:418-543), fused
 * with the tet filter's first stage (markRealTets, :531-591).
 * A wave takes kTetSeg = 64 triangles, one a lane, whose candidate slots
 * are one contiguous range.  The masks that k_tri_seg_copy left per alpha
 * edge give each triangle the l in both T(i,j) after k and T(i,k) as the set
 * bits of one 64-bit word; the wave lists them in LDS and takes them 64 at a
 * time, whatever triangle they belong to: is (j,k,l) a triangle (a bit of
 * the third mask), then the filter.  The kept and undecided ones are written
 * compacted, in order, from the wave's first slot on, with their flags.
 * No barrier: a wave waits for no other until the counters are summed.
 * A wave with a triangle whose row is cut off in a mask (a third vertex 63
 * or more edges on: dense inputs) merges the three rows instead, each lane
 * its own, into fourth vertices in LDS (928 of them, the rest in the
 * candidates' own array).
 * At 100k balls 266 us; 395 with all waves merging, whose rounds last as
 * long as their longest rows; 523 with blocks of 256 triangles filtering
 * every slot.  200k balls with a lattice block: 1.39 ms against 1.70 and
 * 9.6.  The vector ALU bounds it, the filter's 114 instructions being half
 * of a round.
 * A candidate with a covered edge (kDeadBit of one of its triangles in
 * tk, carried with the fourth vertex) is filtered like any other, but an
 * alpha tet among them is only counted (CTR_DROP), not written: it cannot
 * be empty.  On the 100k globule 4.6M of the 19.1M alpha tets are written. */
/* First slot of alpha triangle q without a per-triangle offset array:
 * the triangles of edge e occupy rows trow[e] .. trow[e+1]-1 and each has
 * its row's tail after it as slots, so triangle s + k of a row of L = trow
 * [e+1] - s triangles starts k (L - 1) - k (k - 1) / 2 slots into the
 * edge's range, which begins at the sum of L (L - 1) / 2 over the edges
 * before: roff[] of the segment of kTriSeg edges plus epre[e] within it. */
__device__ __forceinline__ uint64_t tet_slot_off(const uint64_t* roff,
                                                 const uint32_t* epre,
                                                 const uint64_t* trow,
                                                 uint32_t e, uint32_t q) {
  const uint64_t s = trow[e], L = trow[e + 1] - s, k = (uint64_t)q - s;
  return roff[e / kTriSeg] + epre[e] + k * (L - 1) - k * (k - 1) / 2;
}
/* FP32 first stage: 8 waves per SIMD (at most 64 VGPRs, no spills; the
 * LDS stage admits 8 blocks per CU); FP64: the compiler's choice */
template <class R, bool BUF>
__global__ __launch_bounds__(kBlock)
__attribute__((amdgpu_waves_per_eu(sizeof(R) == 4 ? 8 : 1))) void k_tet_enum_filter(
    Stage S, Cnt c_nt, const uint64_t* trow, const uint32_t* tk,
    const uint32_t* tedge, const uint32_t* teik, const uint32_t* tejk,
    const uint32_t* eleft, const uint32_t* ecol, const ulonglong2* emask,
    const uint64_t* off, const uint64_t* roff, const uint32_t* epre,
    uint64_t* bbase, uint4* ctet, uint8_t* flag, uint32_t* bcnt,
    uint32_t* bkeep, Queue q1, uint64_t lim) {
  static_assert(kTetSeg == 64, "a triangle a lane");
  stamp(S.ts, TS_TETS);
  /* LDS of a wave, 4,992 bytes (8 blocks per CU): by masks, three rows of
   * 16 bytes a triangle and the listed bits; by merges, the stage of fourth
   * vertices and the lanes' prefix counts */
  constexpr uint32_t RAW = 312, LIST = (RAW - 192) * 8, CAP = 928;
  __shared__ uint4 s_raw[kBlock / 64][RAW];
  const int64_t nt = c_nt.get();
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int64_t seg = gtid() >> 6, q = gtid();
  unsigned found = 0, dropped = 0;
  if (seg * kTetSeg >= nt) {
    /* a segment past the (device) count */
    if (lane == 0 && seg * kTetSeg < c_nt.cap) {
      bcnt[seg] = bkeep[seg] = 0;
      bbase[seg] = 0;
    }
  } else {
    constexpr uint32_t kEnd = ~kDeadBit;
    uint32_t eij = 0, eik = 0, ejk = 0, i = 0, j = 0, kd = 0;
    ulonglong2 mij = make_ulonglong2(0, 0), mik = mij, mjk = mij;
    if (q < nt) {
      eij = tedge[q];
      eik = teik[q];
      ejk = tejk[q];
      kd = tk[q];
      i = eleft[eij];
      j = ecol[eij];
      mij = emask[eij];
      mik = emask[eik];
      mjk = emask[ejk];
    }
    const uint32_t k = kd & kEnd;
    /* the wave's first slot */
    const uint32_t q0 = __builtin_amdgcn_readfirstlane((uint32_t)q);
    const uint32_t e0 = __builtin_amdgcn_readfirstlane(eij);
    const uint64_t base = off ? off[q0] : tet_slot_off(roff, epre, trow, e0, q0);
    const uint64_t lt = lane ? (~0ull >> (64 - lane)) : 0ull;
    uint32_t run = 0; /* kept + undecided written so far (wave-uniform) */
    bool und = false;
    /* candidates 0 .. total - 1 of the wave, `step` at a time */
    const bool masks = __ballot((mij.x | mik.x | mjk.x) >> 63) == 0;
    uint4* const tab = s_raw[wv];
    uint16_t* const list = reinterpret_cast<uint16_t*>(s_raw[wv] + 192);
    uint32_t* const s_l = reinterpret_cast<uint32_t*>(s_raw[wv]);
    uint32_t* const s_end = s_l + CAP;
    uint32_t* const s_off = s_end + 64;
    uint32_t* const spill = reinterpret_cast<uint32_t*>(ctet + base);
    uint32_t total, step, at = 0, lo = 0, hi = 0;
    bool spilled = false;
    if (masks) {
      /* By masks: l in T(i,j) after k and in T(i,k) are the common bits of
       * the two edges' masks, both over the edges (i,.) that follow (i,k);
       * l is the next triangle of T(i,j) but as many as `after` has bits
       * before it, and the edge (j,l) recorded there has its bit in the
       * mask of (j,k) if (j,k,l) is a triangle.  A triangle without slots
       * (a chunk sub-input's unowned one) has no candidates. */
      const uint32_t d = (eik - eij) & 63u; /* 1 .. 63 */
      const uint64_t after = mij.x >> d;
      const uint64_t dead = (mij.y >> d) | mik.y | ((kd & kDeadBit) ? ~0ull : 0ull);
      uint64_t both = after & mik.x;
      if (off && q < nt && off[q] == off[q + 1]) both = 0;
      tab[3 * lane] = make_uint4((uint32_t)after, (uint32_t)(after >> 32),
                                 (uint32_t)dead, (uint32_t)(dead >> 32));
      tab[3 * lane + 1] =
          make_uint4((uint32_t)mjk.x, (uint32_t)(mjk.x >> 32),
                     (uint32_t)mjk.y, (uint32_t)(mjk.y >> 32));
      tab[3 * lane + 2] = make_uint4(i, j, k, ejk + 1u);
      const uint32_t incl = wave_prefix((uint32_t)__popcll(both));
      at = incl - (uint32_t)__popcll(both);
      total = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
      step = LIST;
      lo = (uint32_t)both;
      hi = (uint32_t)(both >> 32);
    } else {
      /* By merges, where a row is too long for some mask: the three rows
       * are merged by each lane into a stage of fourth vertices from its
       * triangle's first slot on.
       * the triangle's slots [o, oe): off[] per triangle, or (roff) the
       * closed form, a triangle's slots being its row's tail */
      uint64_t o = 0, oe = 0;
      if (q < nt) {
        if (off) {
          o = off[q];
          oe = off[q + 1];
        } else {
          o = tet_slot_off(roff, epre, trow, eij, (uint32_t)q);
          oe = o + (trow[eij + 1] - (uint64_t)q - 1);
        }
      }
      /* the wave's slots, numbered from its first one; [rel, end) this
       * lane's, cut at the arrays' end */
      const uint32_t rel = (uint32_t)(o - base);
      const uint32_t end =
          o >= lim ? rel : rel + (uint32_t)((oe < lim ? oe : lim) - o);
      at = rel;
      auto put = [&](uint32_t v) {
        ++found;
        if (at < end) {
          if (at < CAP) s_l[at] = v;
          else spill[4 * (uint64_t)at] = v;
          ++at;
        }
      };
      /* two merge steps a round: each list's next element is loaded with
       * its current one (kEnd past the row's end, above every ball id) */
      if (o < oe) {
        if constexpr (BUF) {
          /* byte offsets into tk (below 4 GiB): no 64-bit address
           * arithmetic per load */
          const BufU32 K{tk, (uint32_t)(c_nt.cap * 4)};
          uint32_t a = ((uint32_t)q + 1u) << 2, ae = (uint32_t)trow[eij + 1] << 2;
          uint32_t b = (uint32_t)trow[eik] << 2, be = (uint32_t)trow[eik + 1] << 2;
          uint32_t c = (uint32_t)trow[ejk] << 2, ce = (uint32_t)trow[ejk + 1] << 2;
          while (a < ae && b < be && c < ce) {
            const uint32_t xd0 = K.at(a), yd0 = K.at(b), zd0 = K.at(c);
            const uint32_t xd1 = a + 4u < ae ? K.at(a + 4u) : kEnd;
            const uint32_t yd1 = b + 4u < be ? K.at(b + 4u) : kEnd;
            const uint32_t zd1 = c + 4u < ce ? K.at(c + 4u) : kEnd;
            const uint32_t x0 = xd0 & kEnd, y0 = yd0 & kEnd, z0 = zd0 & kEnd;
            const uint32_t m0 = max(x0, max(y0, z0));
            const bool all0 = x0 == m0 && y0 == m0 && z0 == m0;
            if (all0) put(m0 | ((kd | xd0 | yd0 | zd0) & kDeadBit));
            const bool sa = all0 || x0 < m0, sb = all0 || y0 < m0,
                       sc = all0 || z0 < m0;
            const uint32_t xd = sa ? xd1 : xd0, yd = sb ? yd1 : yd0,
                           zd = sc ? zd1 : zd0;
            const uint32_t x = xd & kEnd, y = yd & kEnd, z = zd & kEnd;
            const uint32_t m = max(x, max(y, z));
            const bool all = x == m && y == m && z == m;
            if (all && m != kEnd) put(m | ((kd | xd | yd | zd) & kDeadBit));
            a += (sa ? 4u : 0u) + ((all || x < m) ? 4u : 0u);
            b += (sb ? 4u : 0u) + ((all || y < m) ? 4u : 0u);
            c += (sc ? 4u : 0u) + ((all || z < m) ? 4u : 0u);
          }
        } else {
          /* alpha-triangle ids fit 32 bits (the slot count is checked below
           * 2^32): 32-bit cursors halve the merge's index arithmetic */
          uint32_t a = (uint32_t)q + 1, ae = (uint32_t)trow[eij + 1];
          uint32_t b = (uint32_t)trow[eik], be = (uint32_t)trow[eik + 1];
          uint32_t c = (uint32_t)trow[ejk], ce = (uint32_t)trow[ejk + 1];
          while (a < ae && b < be && c < ce) {
            const uint32_t xd = tk[a], yd = tk[b], zd = tk[c];
            const uint32_t x = xd & kEnd, y = yd & kEnd, z = zd & kEnd;
            const uint32_t m = max(x, max(y, z));
            if (x == m && y == m && z == m) {
              put(m | ((kd | xd | yd | zd) & kDeadBit));
              ++a;
              ++b;
              ++c;
            } else {
              a += (x < m);
              b += (y < m);
              c += (z < m);
            }
          }
        }
      }
      const uint32_t mine = at - rel;
      const uint32_t incl = wave_prefix(mine);
      total = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
      step = total;
      spilled = __ballot(at > CAP) != 0; /* wave-uniform */
      s_end[lane] = incl;
      s_off[lane] = rel - (incl - mine);
      s_off[64 + lane] = i;
      s_off[128 + lane] = j;
      s_off[192 + lane] = k;
    }
    /* A written position is at most the number of the candidate it holds,
     * and that at most its slot: an unread spilled candidate lies past
     * every position written before it. */
    for (uint32_t w0 = 0; w0 < total; w0 += step) {
      const uint32_t wn = min(total - w0, step), we = w0 + wn;
      if (masks) { /* list the bits of this pass: (triangle, bit) */
        while (lo && at < we) {
          list[at - w0] = (uint16_t)(lane << 6 | __builtin_ctz(lo));
          lo &= lo - 1;
          ++at;
        }
        while (!lo && hi && at < we) {
          list[at - w0] = (uint16_t)(lane << 6 | 32 | __builtin_ctz(hi));
          hi &= hi - 1;
          ++at;
        }
      }
      wave_sync();
      for (uint32_t d0 = 0; d0 < wn; d0 += 64) {
        const uint32_t d = d0 + (uint32_t)lane;
        uint4 v = make_uint4(0u, 0u, 0u, 0u);
        bool have = d < wn, dead = false;
        if (masks) {
          if (have) {
            const uint32_t e = list[d], t = e >> 6, b = e & 63u;
            const uint4 x = tab[3 * t], y = tab[3 * t + 1], z = tab[3 * t + 2];
            const uint64_t ax = (uint64_t)x.y << 32 | x.x;
            /* (bit b of `after` is set: the count includes it) */
            const uint32_t tl = q0 + t + (uint32_t)__popcll(ax << (63u - b));
            const uint32_t p = tejk[tl] - z.w, ld = tk[tl];
            const uint32_t mm = p & 32u ? y.y : y.x, md = p & 32u ? y.w : y.z;
            have = p < 63u && ((mm >> (p & 31u)) & 1u);
            dead = (((b & 32u ? x.w : x.z) >> (b & 31u)) | (md >> (p & 31u))) & 1u;
            v = make_uint4(z.x, z.y, z.z, ld & kEnd);
            found += have;
          }
        } else {
          /* of the first lane whose inclusive count exceeds d, at slot
           * d + s_off of that lane */
          int t = 0; /* last lane with an inclusive count <= d, plus one */
#pragma unroll
          for (int h = 32; h >= 1; h >>= 1)
            t += s_end[t + h - 1] <= d ? h : 0;
          t &= 63; /* (d past the last candidate) */
          if (have) {
            const uint32_t slot = d + s_off[t];
            uint32_t ld = 0;
            /* (two branches: one load through a selected pointer would be a
             * flat one) */
            if (!spilled) {
              ld = s_l[slot];
            } else {
              if (slot < CAP) ld = s_l[slot];
              if (slot >= CAP) ld = spill[4 * (uint64_t)slot];
            }
            dead = (ld & kDeadBit) != 0;
            v = make_uint4(s_off[64 + t], s_off[128 + t], s_off[192 + t],
                           ld & kEnd);
          }
        }
        /* the first precision stage */
        int r = REJECT;
        if (have) {
          const Ball bv[4] = {S.ball[v.x], S.ball[v.y], S.ball[v.z],
                              S.ball[v.w]};
          /* the weights are first used after the test of D's sign; left
           * alone, the compiler loads them there, a second round trip per
           * round; used here (an empty asm), each ball is one 16-byte load */
#pragma unroll
          for (int z = 0; z < 4; ++z) asm volatile("" ::"v"(bv[z].w));
          r = tet_code_ss<R>(bv, S.alpha);
          if (dead && r == KEEP) { /* alpha, certainly not empty */
            ++dropped;
            r = REJECT;
          }
        }
        const uint64_t bm = __ballot(r != REJECT);
        if (r != REJECT) {
          const uint64_t w = base + run + (uint32_t)__popcll(bm & lt);
          if (w < lim) {
            ctet[w] = v;
            flag[w] = (uint8_t)r;
            if (r == UNDEC) push_q(q1, (uint32_t)w, v.x);
          }
        }
        und |= __ballot(r == UNDEC) != 0;
        run += (uint32_t)__popcll(bm);
      }
      wave_sync(); /* the next pass rewrites the list */
    }
    run = cut_at(run, base, lim);
    if (lane == 0) {
      bbase[seg] = base;
      bcnt[seg] = run;
      bkeep[seg] = und ? kRecount : run;
    }
  }
  block_flush(S.ctr, CTR_CAND + 2, found);
  block_flush(S.ctr, CTR_DROP, dropped);
}
void launch_tet_enum_filter(const Stage& S, Cnt nt, const uint64_t* trow,
                            const uint32_t* tk, const uint32_t* tedge,
                            const uint32_t* teik, const uint32_t* tejk,
                            const uint32_t* eleft, const uint32_t* ecol,
                            const ulonglong2* emask, const uint64_t* off,
                            const uint64_t* roff, const uint32_t* epre,
                            uint64_t* bbase, uint4* ctet, uint8_t* flag,
                            uint32_t* bcnt, uint32_t* bkeep, Queue q1,
                            PipeLaunch L, uint64_t lim) {
  if (nt.cap <= 0) return;
  dim3 gr((unsigned)((nt.cap + kBlock - 1) / kBlock));
  /* byte offsets into tk while it stays below 4 GiB */
  const bool buf = nt.cap < ((int64_t)1 << 30);
  if constexpr (!kBallF64) {
    if (S.staged) {
      auto kf = buf ? k_tet_enum_filter<float, true>
                    : k_tet_enum_filter<float, false>;
      hipLaunchKernelGGL(kf, gr, dim3(kBlock), 0, L.s, S, nt, trow, tk, tedge,
                         teik, tejk, eleft, ecol, emask, off, roff, epre, bbase, ctet,
                         flag, bcnt, bkeep, q1, lim);
      return;
    }
  }
  auto kd = buf ? k_tet_enum_filter<double, true>
                : k_tet_enum_filter<double, false>;
  hipLaunchKernelGGL(kd, gr, dim3(kBlock), 0, L.s, S, nt, trow, tk, tedge, teik,
                     tejk, eleft, ecol, emask, off, roff, epre, bbase, ctet, flag,
                     bcnt, bkeep, q1, lim);
}

/* kSegLanes lanes per enumeration segment in the two kernels below: a tet
 * segment holds ~26 entries on a globule, and whole waves left most lanes
 * idle.  A segment's lanes stay together; seg_ballot is their ballot. */
constexpr int kSegLanes = 16;
__device__ __forceinline__ unsigned seg_ballot(bool p) {
  const int first = (threadIdx.x & 63) & ~(kSegLanes - 1);
  return (unsigned)(__ballot(p) >> first) & ((1u << kSegLanes) - 1u);
}
/* After the ladder: the kept candidates of each enumeration segment of
 * `seg` items (its first bcnt[b] positions from off[b] on hold its
 * kept and formerly undecided ones) to kept[b].  The marks in bkeep stay: the
 * ladder may decide more of them and count again. */
__global__ __launch_bounds__(kBlock) void k_seg_kept(
    Cnt c_n, int seg, const uint64_t* off, const uint32_t* bcnt,
    const uint8_t* flag, const uint32_t* bkeep, uint32_t* kept) {
  __shared__ uint8_t s_list[kBlock / 64][64];
  const int64_t n = c_n.get();
  const int64_t nseg = (c_n.cap + seg - 1) / seg;
  const int64_t b = gtid(), b0 = b & ~(int64_t)63;
  if (b0 >= nseg) return; /* a whole wave */
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  /* a segment that queued no undecided candidate kept all it wrote: its
   * enumeration left that count.  The wave's others are listed and counted
   * by kSegLanes lanes each. */
  const uint32_t c = b < nseg ? bkeep[b] : 0u;
  const bool count = c == kRecount && b * seg < n;
  if (b < nseg && !count) kept[b] = c == kRecount ? 0u : c;
  const uint64_t todo = __ballot(count);
  if (!todo) return;
  const uint64_t lt = lane ? (~0ull >> (64 - lane)) : 0ull;
  if (count) s_list[wv][__popcll(todo & lt)] = (uint8_t)lane;
  wave_sync();
  const int m = __popcll(todo);
  const uint32_t sub = lane & (kSegLanes - 1);
  for (int k0 = 0; k0 < m; k0 += 64 / kSegLanes) {
    const int k = k0 + lane / kSegLanes;
    const int64_t q = b0 + (k < m ? s_list[wv][k] : 0);
    const uint64_t base = k < m ? off[q] : 0;
    const uint32_t cnt = k < m ? bcnt[q] : 0;
    unsigned sum = 0;
    for (uint32_t t = sub; t < cnt; t += 8 * kSegLanes) {
      uint8_t f[8]; /* in flight together */
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const uint32_t x = t + u * kSegLanes;
        f[u] = flag[base + (x < cnt ? x : sub)];
      }
#pragma unroll
      for (int u = 0; u < 8; ++u)
        sum += t + u * kSegLanes < cnt && f[u] == KEEP;
    }
#pragma unroll
    for (int d = 1; d < kSegLanes; d <<= 1)
      sum += (unsigned)__shfl_xor((int)sum, d, 64);
    if (k < m && sub == 0) kept[q] = sum;
  }
}
/* the kept tets of segment b to tets[bout[b], ...), in order */
__global__ __launch_bounds__(kBlock) void k_tet_seg_copy(
    Cnt c_nt, const uint64_t* bbase, const uint32_t* bcnt, const uint4* ctet,
    const uint8_t* flag, const uint64_t* bout, uint4* tets, uint64_t ocap) {
  const int64_t nt = c_nt.get();
  const int64_t b = gtid() / kSegLanes;
  const uint32_t sub = threadIdx.x & (kSegLanes - 1);
  if (b * kTetSeg >= nt) return;
  const uint64_t base = bbase[b];
  const uint32_t n = bcnt[b];
  uint64_t o = bout[b];
  if (bout[b + 1] - o == n) { /* every entry kept: a straight copy */
    for (uint32_t t = sub; t < n; t += kSegLanes)
      if (o + t < ocap) tets[o + t] = ctet[base + t];
    return;
  }
  for (uint32_t r0 = 0; r0 < n; r0 += kSegLanes) {
    const uint32_t t = r0 + sub;
    bool keep = false;
    uint4 v = make_uint4(0u, 0u, 0u, 0u);
    if (t < n) { /* both loads in flight together */
      v = ctet[base + t];
      keep = flag[base + t] == KEEP;
    }
    const unsigned bm = seg_ballot(keep);
    const uint64_t pre = o + (unsigned)__popc(bm & ((1u << sub) - 1u));
    if (keep && pre < ocap) tets[pre] = v;
    o += (unsigned)__popc(bm);
  }
}
void launch_seg_kept(Cnt n, int seg, const uint64_t* off, const uint32_t* bcnt,
                     const uint8_t* flag, const uint32_t* bkeep, uint32_t* kept,
                     PipeLaunch L) {
  if (n.cap <= 0) return;
  const int64_t nseg = (n.cap + seg - 1) / seg;
  hipLaunchKernelGGL(k_seg_kept,
                     dim3((unsigned)((nseg + kBlock - 1) / kBlock)),
                     dim3(kBlock), 0, L.s, n, seg, off, bcnt, flag, bkeep,
                     kept);
}
void launch_tet_seg_copy(Cnt nt, const uint64_t* bbase, const uint32_t* bcnt,
                         const uint4* ctet, const uint8_t* flag,
                         const uint64_t* bout, uint4* tets, PipeLaunch L,
                         uint64_t ocap) {
  if (nt.cap <= 0) return;
  const int64_t nseg = (nt.cap + kTetSeg - 1) / kTetSeg;
  hipLaunchKernelGGL(
      k_tet_seg_copy,
      dim3((unsigned)((nseg * kSegLanes + kBlock - 1) / kBlock)), dim3(kBlock),
      0, L.s, nt, bbase, bcnt, ctet, flag, bout, tets, ocap);
}

/* Edge candidates of ball i (j > i in the stencil rows, Parallel:122-201)
 * fused with the edge filter's first stage (markRealEdges,
 * Parallel:1229-1250).  One wave per ball: lane r finds stencil row r's
 * candidate range (64 rows per pass), a wave prefix sum lays the ranges
 * end to end, and the lanes test the concatenation 64 candidates at a
 * time (a row of ~15 candidates would leave most lanes idle); the kept
 * and undecided ones are written compacted, in order, from the ball's
 * first slot on (a ballot prefix per 64), with their flags; nothing is
 * written for the others. */
constexpr int kEdgeBallsPerBlock = kBlock / 64;
template <class R>
__global__ __launch_bounds__(kBlock) void k_edge_enum_filter(
    Stage S, const uint64_t* off, uint32_t* cval, uint8_t* flag,
    uint32_t* bcnt, uint32_t* bkeep, Queue q1, uint64_t lim) {
  stamp(S.ts, TS_ENUM);
  const int64_t iw = (int64_t)blockIdx.x * kEdgeBallsPerBlock + (threadIdx.x >> 6);
  if (iw >= S.n) return; /* a whole wave */
  const uint32_t i = __builtin_amdgcn_readfirstlane((uint32_t)iw);
  const int lane = threadIdx.x & 63;
  const uint64_t lt = lane ? (~0ull >> (64 - lane)) : 0ull;
  const GridP g = grid_of(S, i);
  const uint32_t c = S.cellk[i];
  int gx, gy, gz;
  cell_xyz(c - g.cbase, g, gx, gy, gz);
  const int k = g.k_enum;
  const int z0 = max(gz - k, 0), y0 = max(gy - k, 0);
  const int nz = min(gz + k, g.ez - 1) - z0 + 1, ny = min(gy + k, g.ey - 1) - y0 + 1;
  const int x0 = max(gx - k, 0), x1 = min(gx + k, g.ex - 1);
  const Ball bi = S.ball[i];
  const uint64_t o0 = off[i];
  uint64_t o = o0; /* next compacted position */
  bool und = false;
  __shared__ uint32_t s_end[kEdgeBallsPerBlock][64], s_beg[kEdgeBallsPerBlock][64];
  const int wv = threadIdx.x >> 6;
  for (int r0 = 0; r0 < ny * nz; r0 += 64) {
    /* this lane's row: candidates [b, b + len) */
    uint32_t b = 0, len = 0;
    const int r = r0 + lane;
    if (r < ny * nz) {
      const int y = y0 + r % ny, z = z0 + r / ny;
      const int64_t row = (int64_t)g.cbase + (int64_t)g.ex * (y + (int64_t)g.ey * z);
      const int64_t c0 = row + x0, c1 = row + x1;
      if (c1 >= (int64_t)c) {
        b = S.cstart[c0];
        const uint32_t e = S.cstart[c1 + 1];
        if (b < i + 1) b = i + 1;
        len = e > b ? e - b : 0u;
      }
    }
    /* inclusive prefix of the lengths: row r's candidates are positions
     * [incl - len, incl) of the pass; the rows' ends and starts go to LDS
     * for the lanes' searches */
    uint32_t incl = len;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const uint32_t y = (uint32_t)__shfl_up((int)incl, d, 64);
      if (lane >= d) incl += y;
    }
    const uint32_t total = (uint32_t)__shfl((int)incl, 63, 64);
    s_end[wv][lane] = incl;
    s_beg[wv][lane] = b - (incl - len); /* j = s_beg[row] + f */
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    int rr = 0; /* the row of this lane's candidate: first with end > f */
    for (uint32_t f0 = 0; f0 < total; f0 += 64) {
      const uint32_t f = f0 + (uint32_t)lane;
      int code = REJECT;
      uint32_t j = 0;
      if (f < total) {
        while (s_end[wv][rr] <= f) ++rr; /* f < total = s_end[63] */
        j = s_beg[wv][rr] + f;
        const Ball bj = S.ball[j];
        code = same_pos(bi, bj) ? REJECT : edge_code_ss<R>(bi, bj, S.alpha);
      }
      const uint64_t m = __ballot(code != REJECT);
      und |= __ballot(code == UNDEC) != 0;
      if (code != REJECT) {
        const uint64_t w = o + (uint64_t)__popcll(m & lt);
        if (w < lim) {
          cval[w] = j;
          flag[w] = (uint8_t)code;
          if (code == UNDEC) push_q(q1, (uint32_t)w, i);
        }
      }
      o += (uint64_t)__popcll(m);
    }
    /* the next pass rewrites the tables */
    __builtin_amdgcn_wave_barrier();
  }
  if (lane == 0) {
    const uint32_t c = cut_at((uint32_t)(o - o0), o0, lim);
    bcnt[i] = c;
    bkeep[i] = und ? kRecount : c;
  }
}
void launch_edge_enum_filter(const Stage& S, const uint64_t* off,
                             uint32_t* cval, uint8_t* flag,
                             uint32_t* bcnt, uint32_t* bkeep, Queue q1,
                             PipeLaunch L, uint64_t lim) {
  if (S.n <= 0) return;
  dim3 gr((unsigned)((S.n + kEdgeBallsPerBlock - 1) / kEdgeBallsPerBlock));
  if (S.staged)
    hipLaunchKernelGGL(k_edge_enum_filter<float>, gr, dim3(kBlock), 0, L.s, S,
                       off, cval, flag, bcnt, bkeep, q1, lim);
  else
    hipLaunchKernelGGL(k_edge_enum_filter<double>, gr, dim3(kBlock), 0, L.s, S,
                       off, cval, flag, bcnt, bkeep, q1, lim);
}
/* ball i's kept edges (one wave per ball) to (ecol, eleft)[erow[i], ...),
 * their marks in edead (if given; for the triangle stage) and edge_in (the
 * closure) cleared; erow cut at the arrays' end */
__global__ __launch_bounds__(kBlock) void k_edge_copy(
    int64_t n, const uint64_t* off, const uint32_t* bcnt, const uint32_t* cval,
    const uint8_t* flag, uint64_t* erow, uint32_t* ecol, uint32_t* eleft,
    uint8_t* edead, uint8_t* edge_in, uint64_t ocap) {
  const int64_t iw = (int64_t)blockIdx.x * kEdgeBallsPerBlock + (threadIdx.x >> 6);
  if (iw >= n) return;
  const uint32_t i = __builtin_amdgcn_readfirstlane((uint32_t)iw);
  const uint32_t lane = threadIdx.x & 63;
  const uint64_t lt = lane ? (~0ull >> (64 - lane)) : 0ull;
  const uint64_t base = off[i];
  const uint32_t m = bcnt[i];
  uint64_t o = erow[i];
  /* (a recorded pass over its capacity: rows end at the arrays' end) */
  if (lane == 0 && o > ocap) erow[i] = ocap;
  if (lane == 0 && i + 1 == n && erow[n] > ocap) erow[n] = ocap;
  for (uint32_t t0 = 0; t0 < m; t0 += 64) {
    const uint32_t t = t0 + lane;
    const bool keep = t < m && flag[base + t] == KEEP;
    const uint64_t bm = __ballot(keep);
    if (keep) {
      const uint64_t w = o + (uint64_t)__popcll(bm & lt);
      if (w < ocap) {
        ecol[w] = cval[base + t];
        eleft[w] = i;
        if (edead) edead[w] = 0;
        edge_in[w] = 0;
      }
    }
    o += (uint64_t)__popcll(bm);
  }
}
void launch_edge_copy(int64_t n, const uint64_t* off, const uint32_t* bcnt,
                      const uint32_t* cval, const uint8_t* flag,
                      uint64_t* erow, uint32_t* ecol, uint32_t* eleft,
                      uint8_t* edead, uint8_t* edge_in, PipeLaunch L,
                      uint64_t ocap) {
  if (n <= 0) return;
  hipLaunchKernelGGL(
      k_edge_copy,
      dim3((unsigned)((n + kEdgeBallsPerBlock - 1) / kEdgeBallsPerBlock)),
      dim3(kBlock), 0, L.s, n, off, bcnt, cval, flag, erow, ecol, eleft, edead,
      edge_in, ocap);
}

/* a triangle candidate's edge within its segment, and how far edge (i, k) lies
 * after it in row(i), in one word (a row of 2^26 edges has more candidate
 * pairs among its balls than a run accepts) */
static_assert(kTriSeg == 64, "six bits for the edge");
__device__ __forceinline__ uint32_t tri_pos(uint32_t edge, uint32_t ahead) {
  return edge << 26 | ahead;
}
__device__ __forceinline__ uint32_t tri_seg_edge(uint32_t x) { return x >> 26; }
__device__ __forceinline__ uint32_t tri_ahead(uint32_t x) {
  return x & 0x3ffffffu;
}
/* Triangles of alpha edge q = (i, j) -- k in row(i) after j and in row(j),
 * the positions of k in the two rows being the alpha-edge ids of (i, k)
 * and (j, k), recorded for the tet stage and the closure -- fused with the
 * triangle filter's first stage (markRealTriangles, Parallel:1294-1340).
 * A wave takes the kTriSeg edges and hits of k_tri_hits: it lists the hits
 * (edge, position in row(j)) in LDS and takes them 64 at a time: k's
 * position in row(i) by a binary search in the wave's part of ecol, which is
 * in LDS unless a row is long (none: a false hit), then the filter; the kept
 * and undecided ones are written compacted, in order, from the wave's first
 * slot on, three words and the flag.
 * 113 us at 100k balls (30 at 16068), 211 (48) for blocks of 256 edges that
 * merged the rows into LDS and filtered them from there, waiting for their
 * longest rows and at two barriers a round.
 * A ball with 4,000 edges to small ones of short rows: 45 us (and 18 for the
 * hits), 1,948 with its waves, whose rows do not fit the LDS, merging; merges
 * throughout took 889 and 341.
 * A wave with a row too long for the hits merges its rows into
 * the slots themselves and filters them from there: each round's 64 are read
 * before any is written, to positions not past them.
 * edead (alpha edges, cleared; may be null): set for the edges a rejected
 * candidate shows covered by one ball (tri_code_ss): no simplex with such
 * an edge is empty. */
template <class R>
__global__ __launch_bounds__(kBlock) void k_tri_enum_filter(
    Stage S, Cnt c_ne, const uint64_t* erow, const uint32_t* ecol,
    const uint32_t* eleft, const ulonglong2* hits, const uint64_t* off,
    uint32_t* cval, uint32_t* cpos, uint32_t* ceb, uint8_t* flag,
    uint32_t* bcnt, uint32_t* bkeep, uint8_t* edead, Queue q1, uint64_t lim) {
  /* with the tables 4,096 bytes of LDS a wave: 8 blocks per CU */
  constexpr uint32_t LIST = 1152, COLS = 192;
  __shared__ uint4 s_tab[kBlock / 64][64];
  __shared__ uint32_t s_col[kBlock / 64][COLS];
  __shared__ uint16_t s_list[kBlock / 64][LIST];
  const int64_t ne = c_ne.get();
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int64_t seg = gtid() >> 6, q = gtid();
  unsigned found = 0;
  if (seg * kTriSeg >= ne) { /* a segment past the (device) count */
    if (lane == 0 && seg * kTriSeg < c_ne.cap) bcnt[seg] = bkeep[seg] = 0;
  } else {
    const uint32_t q0 = __builtin_amdgcn_readfirstlane((uint32_t)q);
    const uint64_t base = off[seg];
    uint32_t i = 0, j = 0, b = 0, len = 0, ae = 0;
    ulonglong2 h = make_ulonglong2(0, 0);
    if (q < ne) {
      i = eleft[q];
      j = ecol[q];
      b = (uint32_t)erow[j];
      len = (uint32_t)erow[j + 1] - b;
      ae = (uint32_t)erow[i + 1];
      h = hits[q];
    }
    const bool listed = __ballot(len > 128u) == 0;
    /* the wave's rows end within the LDS */
    const bool near = __ballot(q < ne && ae - q0 > COLS) == 0;
    const uint64_t lt = lane ? (~0ull >> (64 - lane)) : 0ull;
    uint32_t w4[4] = {0u, 0u, 0u, 0u};
    uint32_t total, step, at = 0;
    if (listed) {
      w4[0] = (uint32_t)h.x;
      w4[1] = (uint32_t)(h.x >> 32);
      w4[2] = (uint32_t)h.y;
      w4[3] = (uint32_t)(h.y >> 32);
      const uint32_t n = (uint32_t)(__popcll(h.x) + __popcll(h.y));
      const uint32_t incl = wave_prefix(n);
      at = incl - n;
      total = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
      step = LIST;
      s_tab[wv][lane] = make_uint4(i, j, ae - q0, b);
      s_col[wv][lane] = j;
      /* the rest of the last row */
      const int last = ne - q0 < 64 ? (int)(ne - q0) - 1 : 63;
      const uint32_t end = (uint32_t)__builtin_amdgcn_readlane((int)ae, last);
      if (near)
        for (uint32_t t = 64u + (uint32_t)lane; q0 + t < end; t += 64)
          s_col[wv][t] = ecol[q0 + t];
    } else {
      const uint32_t n = (uint32_t)h.x;
      const uint32_t incl = wave_prefix(n);
      total = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
      uint64_t o = base + (incl - n);
      if (q < ne)
        merge_rows(ecol, (uint32_t)q + 1u, ae, b, b + len,
                   [&](uint32_t k, uint32_t a, uint32_t bb) {
                     if (o < lim) {
                       cval[o] = k;
                       cpos[o] = tri_pos((uint32_t)lane, a - (uint32_t)q);
                       ceb[o] = bb;
                     }
                     ++o;
                   });
      total = cut_at(total, base, lim);
      step = total;
    }
    uint32_t run = 0; /* kept + undecided written so far (wave-uniform) */
    bool und = false;
    for (uint32_t w0 = 0; w0 < total; w0 += step) {
      const uint32_t wn = min(total - w0, step), we = w0 + wn;
      if (listed) { /* list the hits of this pass */
        bool open = true; /* (all bits of the words before are listed) */
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          while (open && w4[w] && at < we) {
            s_list[wv][at - w0] =
                (uint16_t)(lane << 7 | w << 5 | __builtin_ctz(w4[w]));
            w4[w] &= w4[w] - 1;
            ++at;
          }
          open = open && !w4[w];
        }
      }
      wave_sync();
      for (uint32_t d0 = 0; d0 < wn; d0 += 64) {
        const uint32_t d = d0 + (uint32_t)lane;
        bool have = d < wn;
        uint32_t vi = 0, vj = 0, k = 0, e = 0, ea = 0, eb = 0;
        if (listed) {
          if (have) {
            const uint32_t x = s_list[wv][d], t = x >> 7;
            const uint4 T = s_tab[wv][t];
            eb = T.w + (x & 127u);
            k = ecol[eb];
            /* k among the ids after (i, j) in row(i) */
            uint32_t lo;
            if (near) {
              lo = first_from(t + 1u, T.z, k,
                              [&](uint32_t m) { return s_col[wv][m]; });
              have = lo < T.z && s_col[wv][lo] == k;
            } else {
              lo = first_from(t + 1u, T.z, k,
                              [&](uint32_t m) { return ecol[q0 + m]; });
              have = lo < T.z && ecol[q0 + lo] == k;
            }
            vi = T.x;
            vj = T.y;
            e = q0 + t;
            ea = q0 + lo;
          }
        } else if (have) {
          k = cval[base + d];
          const uint32_t x = cpos[base + d];
          e = q0 + tri_seg_edge(x);
          ea = e + tri_ahead(x);
          eb = ceb[base + d];
          vi = eleft[e];
          vj = ecol[e];
        }
        int r = REJECT;
        if (have) {
          ++found;
          const Ball b0 = S.ball[vi], b1 = S.ball[vj], b2 = S.ball[k];
          /* weights used here: one 16-byte load per ball (as for tets) */
          asm volatile("" ::"v"(b0.w), "v"(b1.w), "v"(b2.w));
          unsigned cover;
          r = tri_code_ss<R>(b0, b1, b2, S.alpha, cover);
          if (cover && edead) { /* opposite edges: (j, k), (i, k), (i, j) */
            if (cover & 1u) edead[eb] = 1;
            if (cover & 2u) edead[ea] = 1;
            if (cover & 4u) edead[e] = 1;
          }
        }
        const uint64_t bm = __ballot(r != REJECT);
        if (r != REJECT) {
          const uint64_t o = base + run + (uint32_t)__popcll(bm & lt);
          if (o < lim) {
            cval[o] = k;
            cpos[o] = tri_pos(e - q0, ea - e);
            ceb[o] = eb;
            flag[o] = (uint8_t)r;
            if (r == UNDEC) push_q(q1, (uint32_t)o, e);
          }
        }
        und |= __ballot(r == UNDEC) != 0;
        run += (uint32_t)__popcll(bm);
      }
      wave_sync(); /* the next pass rewrites the list */
    }
    run = cut_at(run, base, lim);
    if (lane == 0) {
      bcnt[seg] = run;
      bkeep[seg] = und ? kRecount : run;
    }
  }
  block_flush(S.ctr, CTR_CAND + 1, found);
}
void launch_tri_enum_filter(const Stage& S, Cnt ne, const uint64_t* erow,
                            const uint32_t* ecol, const uint32_t* eleft,
                            const ulonglong2* hits, const uint64_t* off,
                            uint32_t* cval, uint32_t* cpos, uint32_t* ceb,
                            uint8_t* flag, uint32_t* bcnt,
                            uint32_t* bkeep, uint8_t* edead, Queue q1,
                            PipeLaunch L, uint64_t lim) {
  if (ne.cap <= 0) return;
  dim3 gr((unsigned)((ne.cap + kBlock - 1) / kBlock));
  auto kf = S.staged ? k_tri_enum_filter<float> : k_tri_enum_filter<double>;
  hipLaunchKernelGGL(kf, gr, dim3(kBlock), 0, L.s, S, ne, erow, ecol, eleft,
                     hits, off, cval, cpos, ceb, flag, bcnt, bkeep, edead,
                     q1, lim);
}
/* the kept triangles of segment b to (tk, tedge, teik, tejk)[bout[b], ...)
 * in order, a wave each; trow[e] for its edges e (and trow[ne], by the wave
 * holding index ne) = bout[b] + the kept triangles of its edges before e.
 * tk has kDeadBit set where one of the triangle's edges is marked in edead
 * (if given); tri_in (the closure's marks) cleared.  emask[e], e = (i,j): x
 * has bit r if (i, j, k) is a triangle and (i, k) the (r + 1)th edge after e,
 * y the bits of those with kDeadBit; bit 63 is set if some r is 63 or more.  spair, epre (if given):
 * the tet slots of the segment's triangles (each one's row tail), and of
 * those of its edges before e.  Grid: a wave per segment and one more; bout
 * has one entry more than segments. */
__global__ __launch_bounds__(kBlock) void k_tri_seg_copy(
    Cnt c_ne, const uint64_t* off, const uint32_t* bcnt, const uint32_t* cval,
    const uint32_t* cpos, const uint32_t* ceb, const uint8_t* flag,
    const uint64_t* bout, const uint8_t* edead, uint32_t* tk, uint32_t* tedge, uint32_t* teik,
    uint32_t* tejk, uint64_t* trow, uint64_t* spair, uint32_t* epre,
    ulonglong2* emask, uint8_t* tri_in, uint64_t ocap) {
  __shared__ uint32_t s_cnt[kBlock / 64][64];
  __shared__ unsigned long long s_mask[2][kBlock / 64][64];
  const int64_t ne = c_ne.get();
  const int64_t b = gtid() >> 6, q0 = b * kTriSeg;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  if (q0 > ne) { /* a segment past the (device) count */
    if (spair && lane == 0 && q0 < c_ne.cap) spair[b] = 0;
    return;
  }
  s_cnt[wv][lane] = 0;
  s_mask[0][wv][lane] = s_mask[1][wv][lane] = 0;
  wave_sync();
  const uint64_t lt = lane ? (~0ull >> (64 - lane)) : 0ull;
  const uint64_t o0 = bout[b];
  if (q0 < ne) {
    const uint64_t base = off[b];
    const uint32_t n = bcnt[b];
    /* every entry kept (bout's step equals the written count): no flag is
     * read */
    const bool all = bout[b + 1] - o0 == n;
    uint64_t o = o0;
    /* kU entries a lane in flight together: the rounds' chains of loads are
     * what the kernel waits for (139 us at 100k balls one by one, 122 by
     * two, 115 by four; 94 with 12 bytes read and 17 written a triangle for
     * 16 and 21) */
    constexpr int kU = 4;
    for (uint32_t r0 = 0; r0 < n; r0 += 64 * kU) {
      /* an entry's arrays are read whether or not it is kept (all were
       * written) */
      uint32_t fv[kU], sv[kU], xv[kU], av[kU], bv[kU];
      bool dead[kU];
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        const uint32_t t = r0 + 64u * u + (uint32_t)lane;
        const uint64_t at = base + (t < n ? t : n - 1);
        fv[u] = all ? (uint32_t)KEEP : flag[at];
        const uint32_t x = cpos[at];
        sv[u] = (uint32_t)q0 + tri_seg_edge(x);
        xv[u] = cval[at];
        av[u] = sv[u] + tri_ahead(x);
        bv[u] = ceb[at];
        if (t >= n) fv[u] = REJECT;
      }
#pragma unroll
      for (int u = 0; u < kU; ++u)
        dead[u] = edead && (edead[sv[u]] | edead[av[u]] | edead[bv[u]]);
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        if (r0 + 64u * u >= n) break;
        const bool keep = fv[u] == KEEP;
        const uint32_t seg = keep ? sv[u] : 0xffffffffu;
        /* entries come in edge order: one LDS add per run of lanes with
         * the same edge (its first lane adds the run's length) instead of
         * one per lane on the same counter */
        const uint32_t prev = (uint32_t)__shfl_up((int)seg, 1, 64);
        const uint64_t heads = __ballot(lane == 0 || prev != seg);
        const uint64_t bm = __ballot(keep);
        if (keep) {
          const uint32_t e = seg - (uint32_t)q0;
          if ((heads >> lane) & 1ull) {
            const uint64_t later = lane == 63 ? 0ull : heads >> (lane + 1);
            const unsigned len = later ? (unsigned)__builtin_ctzll(later) + 1u
                                       : 64u - (unsigned)lane;
            atomicAdd(&s_cnt[wv][e], len);
          }
          const uint64_t w = o + (uint64_t)__popcll(bm & lt);
          if (w < ocap) {
            tk[w] = xv[u] | (dead[u] ? kDeadBit : 0u);
            tedge[w] = seg;
            teik[w] = av[u];
            tejk[w] = bv[u];
            tri_in[w] = 0;
            const uint32_t r = av[u] - seg - 1u;
            const unsigned long long bit = 1ull << (r < 63u ? r : 63u);
            atomicOr(&s_mask[0][wv][e], bit);
            if (dead[u]) atomicOr(&s_mask[1][wv][e], bit);
          }
        }
        o += (uint64_t)__popcll(bm);
      }
    }
  }
  wave_sync(); /* the per-edge counts and masks complete */
  const uint32_t c = s_cnt[wv][lane];
  const int64_t e = q0 + lane;
  const uint64_t v = o0 + (wave_prefix(c) - c);
  if (e <= ne) trow[e] = v < ocap ? v : ocap;
  if (e < ne)
    emask[e] = make_ulonglong2(s_mask[0][wv][lane], s_mask[1][wv][lane]);
  if (spair) {
    const uint64_t m = c ? (uint64_t)c * (c - 1) / 2 : 0;
    uint64_t x = m;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const uint64_t y = (uint64_t)__shfl_up((unsigned long long)x, d, 64);
      if (lane >= d) x += y;
    }
    /* (2^32 slots or more end the run after their scan) */
    if (e < ne) epre[e] = (uint32_t)(x - m);
    if (lane == 63 && q0 < c_ne.cap) spair[b] = x;
  }
}
void launch_tri_seg_copy(Cnt ne, const uint64_t* off, const uint32_t* bcnt,
                         const uint32_t* cval, const uint32_t* cpos,
                         const uint32_t* ceb, const uint8_t* flag,
                         const uint64_t* bout, const uint8_t* edead,
                         uint32_t* tk, uint32_t* tedge, uint32_t* teik, uint32_t* tejk,
                         uint64_t* trow, uint64_t* spair, uint32_t* epre,
                         ulonglong2* emask, uint8_t* tri_in, PipeLaunch L,
                         uint64_t ocap) {
  const int64_t nseg = (std::max<int64_t>(ne.cap, 0) + kTriSeg - 1) / kTriSeg;
  hipLaunchKernelGGL(k_tri_seg_copy,
                     dim3((unsigned)((nseg + kBlock / 64) / (kBlock / 64))),
                     dim3(kBlock), 0, L.s, ne, off, bcnt, cval, cpos, ceb,
                     flag, bout, edead, tk, tedge, teik, tejk, trow, spair,
                     epre, emask, tri_in, ocap);
}

template <int KIND>
__global__ __launch_bounds__(kBlock) void k_filter_esc(Stage S, CandCtx C,
                                                       QRef qr,
                                                       const uint32_t* cval,
                                                       uint8_t* flag,
                                                       Queue q2) {
  __shared__ uint32_t s_off[QSLOTS + 1];
  const QTab q = q_table(qr, s_off);
  StageCnt sc;
  for_queue(q, [&](uint32_t t) {
    QEntry e = q.at(t);
    Ball v[4];
    cand_balls<KIND>(S, C, e.item, e.aux, KIND == 3 ? 0u : cval[e.item], v);
    sc.c[1]++;
    int r = filter_code<KIND, FE<double>>(v, S.alpha);
    if (KIND > 1 && r == UNDEC && degenerate_i128<KIND>(v, S.ex.S) == 1) {
      sc.c[3]++; /* decided exactly, in 128-bit integers */
      r = REJECT;
    }
    if (r == UNDEC) {
      sc.c[2]++;
      r = filter_code<KIND, FEDD>(v, S.alpha);
    }
    if (r == UNDEC)
      push_q(q2, e.item, e.aux);
    else
      flag[e.item] = (uint8_t)r;
  });
  sc.flush(S.ctr, fam_of(KIND));
}
/* Exact filter decisions in two steps per wave: every lane takes one
 * queued candidate and settles degenerate ones (collinear / coplanar
 * centres) in 128-bit integers; the wave's other candidates are listed in
 * LDS and taken 4 at a time by its groups of kTPI lanes for the
 * wavefront-cooperative wide-integer evaluation. */
template <int KIND>
__global__ __launch_bounds__(kBlock) void k_filter_exact(Stage S, CandCtx C,
                                                         QRef qr,
                                                         const uint32_t* cval,
                                                         uint8_t* flag) {
  __shared__ uint32_t s_off[QSLOTS + 1];
  const QTab q = q_table(qr, s_off);
  __shared__ uint32_t s_pend[kBlock / 64][64];
  unsigned cnt = 0;
  const uint32_t n = q.size();
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const uint64_t lt = lane ? (~0ull >> (64 - lane)) : 0ull;
  const uint64_t waves = (uint64_t)gridDim.x * (blockDim.x >> 6);
  uint32_t* const pend_list = s_pend[w];
  /* wave-uniform loop over 64 entries at a time */
  for (uint64_t base = ((uint64_t)blockIdx.x * (blockDim.x >> 6) + w) * 64;
       base < n; base += waves * 64) {
    const uint32_t t = (uint32_t)(base + lane);
    bool pend = false;
    if (t < n) {
      pend = true;
      if (KIND > 1) {
        const QEntry e = q.at(t);
        Ball v[4];
        cand_balls<KIND>(S, C, e.item, e.aux, KIND == 3 ? 0u : cval[e.item], v);
        if (degenerate_i128<KIND>(v, S.ex.S) == 1) {
          flag[e.item] = REJECT;
          ++cnt;
          pend = false;
        }
      }
    }
    const uint64_t m = __ballot(pend);
    if (pend) pend_list[__popcll(m & lt)] = t;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int np = __popcll(m);
    /* group-uniform loop: group g takes the pending entries g, g + 4, ... */
    for (int k = lane / kTPI; k < np; k += 64 / kTPI) {
      const QEntry e = q.at(pend_list[k]);
      Ball v[4];
      cand_balls<KIND>(S, C, e.item, e.aux, KIND == 3 ? 0u : cval[e.item], v);
      const int r = filter_exact<KIND>(v, S.ex);
      if (Grp<kTPI>::idx() == 0) {
        flag[e.item] = (uint8_t)r;
        ++cnt;
      }
    }
    /* the list is rewritten next round: every group is done with it */
    __builtin_amdgcn_wave_barrier();
  }
  flush_ctr(S.ctr, CTR_STAGE + fam_of(KIND) * 4 + 3, cnt);
}

void launch_filter_esc(const Stage& S, int kind, CandCtx C, QRef q, const uint32_t* cval, uint8_t* flag,
                       Queue q2, PipeLaunch L) {
  if (!q.launch_items()) return;
  dim3 gr = qgrid(q, kEscBlocks);
  if (kind == 1)
    hipLaunchKernelGGL(k_filter_esc<1>, gr, dim3(kBlock), 0, L.s, S, C, q,
                       cval, flag, q2);
  else if (kind == 2)
    hipLaunchKernelGGL(k_filter_esc<2>, gr, dim3(kBlock), 0, L.s, S, C, q,
                       cval, flag, q2);
  else
    hipLaunchKernelGGL(k_filter_esc<3>, gr, dim3(kBlock), 0, L.s, S, C, q,
                       cval, flag, q2);
}
void launch_filter_exact(const Stage& S, int kind, CandCtx C, QRef q, const uint32_t* cval, uint8_t* flag,
                         PipeLaunch L) {
  if (!q.launch_items()) return;
  dim3 gr = qgrid(q, kExactBlocks); /* one entry per lane in the first step */
  if (kind == 1)
    hipLaunchKernelGGL(k_filter_exact<1>, gr, dim3(kBlock), 0, L.s, S, C, q,
                       cval, flag);
  else if (kind == 2)
    hipLaunchKernelGGL(k_filter_exact<2>, gr, dim3(kBlock), 0, L.s, S, C, q,
                       cval, flag);
  else
    hipLaunchKernelGGL(k_filter_exact<3>, gr, dim3(kBlock), 0, L.s, S, C, q,
                       cval, flag);
}

}  // namespace PAC_V
}  // namespace pac
