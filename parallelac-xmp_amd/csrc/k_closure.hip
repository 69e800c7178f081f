/*
 * k_closure.hip -- closure of the complex and output emission.
 *
 * The reference builds the faces of the final tets and the edges of the
 * final triangles, sorts and de-duplicates them and merges them with the
 * surviving dangling simplices (AlphaComplexParallel.cu:1490-1632,
 * :1646-1788; generateTrisInTets / markTrisForDeletion / generateEdgesInTris
 * / markEdgesForDeletion, AlphaComplexLargeData.cu:737-926).  Every such
 * face is itself an alpha simplex, so here each final tet (triangle) marks
 * its faces (edges) in the already sorted alpha lists by CSR lookup; the
 * final lists are then a stable compaction of the alpha lists and come out
 * in the reference's lexicographic order with no sort or merge.
 */
#include "pac_dev.h"
#include "pac_tiles.h"

namespace pac {
using namespace PAC_V; /* type-independent device helpers */

/* out[i] = a[i] | b[i] (flags) */
__global__ __launch_bounds__(kBlock) void k_or_flags(Cnt c_n, const uint8_t* a,
                                                     const uint8_t* b,
                                                     uint8_t* out) {
  const int64_t n = c_n.get();
  const int64_t i = gtid();
  if (i >= n) return;
  out[i] = (a[i] | b[i]) != 0;
}
void launch_or_flags(Cnt n, const uint8_t* a, const uint8_t* b, uint8_t* out,
                     PipeLaunch L) {
  if (n.cap <= 0) return;
  hipLaunchKernelGGL(k_or_flags, dim3((unsigned)((n.cap + kBlock - 1) / kBlock)),
                     dim3(kBlock), 0, L.s, n, a, b, out);
}
/* The final tets out of the alpha tets' flags, a tile of flags a block: each
 * kept tet in original ids to out, and its faces marked in tri_in (cleared).
 * t = (i, j, k, l), i < j < k < l: one pass over row i finds the edges ij, ik
 * and il; the faces ijk and ijl are in the triangle row of ij, ikl in that of
 * ik, jkl in that of jk, each at the number of bits before its own in the
 * edge's mask (emask), and the edges jk and jl are recorded with the first
 * two.  A row that its mask cuts off is searched instead. */
__global__ __launch_bounds__(kBlock) void k_tile_tets(
    Cnt c_nk, const uint4* tets, const uint8_t* flag, const uint64_t* offs,
    const uint64_t* erow, const uint32_t* ecol, const ulonglong2* emask,
    const uint64_t* trow, const uint32_t* tk, const uint32_t* tejk,
    const uint32_t* perm, uint8_t* tri_in, int4* out, uint64_t ocap,
    unsigned long long* ts) {
  stamp(ts, TS_TRI_AC2);
  /* the triangle of edge e whose third vertex is v, e2 = (i, v) for e =
   * (i, .); -1 if there is none (a recorded pass over its capacities) */
  auto face = [&](uint32_t e, uint32_t e2, uint32_t v) -> int64_t {
    const uint64_t m = emask[e].x, r0 = trow[e];
    if (m >> 63) return find_row(tk, r0, trow[e + 1], v, ~kDeadBit);
    const uint32_t r = e2 - e - 1u;
    if (r >= 63u || !((m >> r) & 1)) return -1;
    return (int64_t)(r0 + (uint64_t)__popcll(m & ((1ull << r) - 1)));
  };
  tile_each(flag, c_nk.get(), offs, [&](int64_t id, uint64_t p) {
    if (p >= ocap) return;
    const uint4 t = tets[id];
    out[p] = make_int4((int)perm[t.x], (int)perm[t.y], (int)perm[t.z],
                       (int)perm[t.w]);
    int64_t eij, eik, eil;
    find_row3(ecol, erow[t.x], erow[t.x + 1], t.y, t.z, t.w, eij, eik, eil);
    if (eij < 0 || eik < 0 || eil < 0) return;
    const int64_t f = face((uint32_t)eij, (uint32_t)eik, t.z);
    const int64_t g = face((uint32_t)eij, (uint32_t)eil, t.w);
    const int64_t h = face((uint32_t)eik, (uint32_t)eil, t.w);
    if (f >= 0) tri_in[f] = 1;
    if (g >= 0) tri_in[g] = 1;
    if (h >= 0) tri_in[h] = 1;
    if (f < 0 || g < 0) return;
    const int64_t q = face(tejk[f], tejk[g], t.w);
    if (q >= 0) tri_in[q] = 1;
  });
}
void launch_tile_tets(Cnt nk, const uint4* tets, const uint8_t* flag,
                      const uint64_t* offs, const uint64_t* erow,
                      const uint32_t* ecol, const ulonglong2* emask,
                      const uint64_t* trow, const uint32_t* tk,
                      const uint32_t* tejk, const uint32_t* perm,
                      uint8_t* tri_in, int32_t* out, unsigned long long* ts,
                      PipeLaunch L, uint64_t ocap) {
  if (nk.cap <= 0) return;
  hipLaunchKernelGGL(k_tile_tets, tiles_of(nk), dim3(kBlock), 0, L.s, nk, tets,
                     flag, offs, erow, ecol, emask, trow, tk, tejk, perm,
                     tri_in, (int4*)out, ocap, ts);
}

/* the same for the final triangles, which mark their edges in edge_in
 * (edge ids recorded at enumeration: (i,j) = tedge, (i,k) = teik, (j,k) =
 * tejk) */
__global__ __launch_bounds__(kBlock) void k_tile_tris(
    Cnt c_nt, const uint8_t* flag, const uint64_t* offs, const uint32_t* ecol,
    const uint32_t* eleft, const uint32_t* tk, const uint32_t* tedge,
    const uint32_t* teik, const uint32_t* tejk, const uint32_t* perm,
    uint8_t* edge_in, int32_t* out, uint64_t ocap, unsigned long long* ts) {
  stamp(ts, TS_EDGE_AC2);
  tile_each(flag, c_nt.get(), offs, [&](int64_t t, uint64_t p) {
    if (p >= ocap) return;
    const uint32_t e = tedge[t];
    edge_in[e] = 1;
    edge_in[teik[t]] = 1;
    edge_in[tejk[t]] = 1;
    out[3 * p] = (int32_t)perm[eleft[e]];
    out[3 * p + 1] = (int32_t)perm[ecol[e]];
    out[3 * p + 2] = (int32_t)perm[tk[t] & ~kDeadBit];
  });
}
void launch_tile_tris(Cnt nt, const uint8_t* flag, const uint64_t* offs,
                      const uint32_t* ecol, const uint32_t* eleft,
                      const uint32_t* tk, const uint32_t* tedge,
                      const uint32_t* teik, const uint32_t* tejk,
                      const uint32_t* perm, uint8_t* edge_in, int32_t* out,
                      unsigned long long* ts, PipeLaunch L, uint64_t ocap) {
  if (nt.cap <= 0) return;
  hipLaunchKernelGGL(k_tile_tris, tiles_of(nt), dim3(kBlock), 0, L.s, nt, flag,
                     offs, ecol, eleft, tk, tedge, teik, tejk, perm, edge_in,
                     out, ocap, ts);
}

}  // namespace pac
