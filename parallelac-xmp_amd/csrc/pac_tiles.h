/*
 * pac_tiles.h -- block scans, and the kept entries of a flag array by tiles
 * of kTile flags (one block each) whose offsets flag_tile_offsets computed.
 */
#ifndef PAC_TILES_H
#define PAC_TILES_H
#include "pac_internal.h"

namespace pac {

__device__ __forceinline__ uint64_t wave_incl_scan_u64(uint64_t v) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    uint64_t o = __shfl_up(v, d, 64);
    if (lane >= d) v += o;
  }
  return v;
}

/* block-wide exclusive scan of one value per thread; returns block total */
__device__ __forceinline__ uint64_t block_excl_scan_u64(uint64_t v,
                                                        uint64_t* total) {
  __shared__ uint64_t wsum[kBlock / 64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  uint64_t inc = wave_incl_scan_u64(v);
  if (lane == 63) wsum[w] = inc;
  __syncthreads();
  uint64_t base = 0, tot = 0;
#pragma unroll
  for (int q = 0; q < kBlock / 64; ++q) {
    if (q < w) base += wsum[q];
    tot += wsum[q];
  }
  __syncthreads();
  *total = tot;
  return base + inc - v;
}

__device__ __forceinline__ unsigned nz_bytes(uint32_t x) {
  /* high bit of each byte set iff the byte is nonzero */
  const uint32_t y = ((x & 0x7f7f7f7fu) + 0x7f7f7f7fu) | x;
  return (unsigned)__popc(y & 0x80808080u);
}
__device__ __forceinline__ uint2 load_flags8(const uint8_t* in, int64_t i0,
                                             int64_t n) {
  if (i0 + 8 <= n) return *reinterpret_cast<const uint2*>(in + i0);
  uint32_t w[2] = {0u, 0u};
  for (int q = 0; q < 8; ++q)
    if (i0 + q < n) w[q >> 2] |= (uint32_t)in[i0 + q] << (8 * (q & 3));
  return make_uint2(w[0], w[1]);
}

/* emit(i, p) for the kept entries i of this block's tile, p being the rank
 * among all kept entries: their ids are gathered in LDS first, so that
 * consecutive lanes take consecutive ranks however sparse the flags are */
template <class F>
__device__ __forceinline__ void tile_each(const uint8_t* flag, int64_t n,
                                          const uint64_t* offs, F&& emit) {
  __shared__ uint16_t s_kept[kTile];
  const int64_t base = (int64_t)blockIdx.x * kTile;
  const uint2 f = load_flags8(flag, base + (int64_t)threadIdx.x * 8, n);
  uint64_t tot;
  uint32_t p =
      (uint32_t)block_excl_scan_u64(nz_bytes(f.x) + nz_bytes(f.y), &tot);
#pragma unroll
  for (int q = 0; q < 8; ++q)
    if ((((q < 4 ? f.x : f.y) >> (8 * (q & 3))) & 0xffu) != 0)
      s_kept[p++] = (uint16_t)(threadIdx.x * 8 + q);
  __syncthreads();
  const uint64_t p0 = offs[blockIdx.x];
  for (uint32_t t = threadIdx.x; t < (uint32_t)tot; t += kBlock)
    emit(base + s_kept[t], p0 + t);
}
inline dim3 tiles_of(Cnt n) {
  return dim3((unsigned)((n.cap + kTile - 1) / kTile));
}

}  // namespace pac
#endif
