// Transfer of host arrays in the reference's layout ((i,k,j) with j
// contiguous, species last; src/wrf_jax/core/conversion.py:62-67 fills its
// state from such arrays) to and from the registry's layout in HBM.
//
// The arrays cross PCIe as they are, through pinned chunks, and k_layout
// turns them on the device: a plane of one level is a 2-D transpose through
// LDS, read along j and written along i, or back.  Turning them on the host
// (one strided pass per array on one core) took 85 % of a 64x48x30
// step_em_core_once: 26.9 ms a call, 3.5 ms this way (1 ms of it the step).
#pragma once
#include "wrfdc_common.h"

// A run of i of one array.  Registry element (s, p, j, i) is at reg + s*rs +
// p*rp + j*rj + i0 + i, the reference's at ref + i*si + p*sp + j*sj + slot.
// A species stack of n has n + 1 slots, slot = s + 1; its slot 0 has no
// registry element (not even a buffer where n = 0), is skipped on the way up
// and read back as 0.  i in [ni, nipad) are the pitch's pad columns, which an
// upload clears.
struct LayoutSeg {
  float *reg;
  unsigned ref;  // element offset in the chunk
  int i0, ni, nipad, nj, np, nslot, species;
  unsigned si, sj, sp;
  size_t rj, rp, rs;
  unsigned tile0;  // first tile of the launch that is this segment's
};
constexpr int kLayoutSegs = 24;  // segments per launch (kernel arguments of about 2 KB)
struct LayoutList {
  LayoutSeg s[kLayoutSegs];
  int n;
};
constexpr int kLayoutTile = 32;
__host__ inline unsigned layout_tiles(const LayoutSeg &g) {
  return (unsigned)((g.nipad + kLayoutTile - 1) / kLayoutTile) * (unsigned)((g.nj + kLayoutTile - 1) / kLayoutTile) * (unsigned)(g.np * g.nslot);
}

// block (32, 8): one 32 x 32 tile (i, j) of one plane
template <bool UP>
__global__ void __launch_bounds__(256) k_layout(LayoutList L, float *__restrict__ chunk) {
  __shared__ float t[kLayoutTile][kLayoutTile + 1];
  int n = 0;
  while (n + 1 < L.n && L.s[n + 1].tile0 <= blockIdx.x) n++;
  const LayoutSeg &g = L.s[n];
  unsigned b = blockIdx.x - g.tile0;
  const unsigned ti = (unsigned)((g.nipad + kLayoutTile - 1) / kLayoutTile), tj = (unsigned)((g.nj + kLayoutTile - 1) / kLayoutTile);
  const int ib = (int)(b % ti) * kLayoutTile, jb = (int)(b / ti % tj) * kLayoutTile;
  b = b / ti / tj;
  const unsigned p = b % (unsigned)g.np, slot = b / (unsigned)g.np;
  const bool empty = g.species && slot == 0;  // the unused species slot
  if (UP && empty) return;
  const unsigned ref = g.ref + p * g.sp + slot;
  float *reg = g.reg + (g.species && !empty ? (size_t)(slot - 1) * g.rs : 0) + (size_t)p * g.rp + (size_t)g.i0;
  const int x = (int)threadIdx.x, y = (int)threadIdx.y;
  if (UP) {
    for (int q = y; q < kLayoutTile; q += 8)
      if (ib + q < g.ni && jb + x < g.nj) t[q][x] = chunk[ref + (unsigned)(ib + q) * g.si + (unsigned)(jb + x) * g.sj];
    __syncthreads();
    for (int q = y; q < kLayoutTile; q += 8)
      if (ib + x < g.nipad && jb + q < g.nj) reg[(size_t)(jb + q) * g.rj + (size_t)(ib + x)] = ib + x < g.ni ? t[x][q] : 0.f;
  } else {
    for (int q = y; q < kLayoutTile; q += 8)
      if (ib + x < g.ni && jb + q < g.nj) t[x][q] = empty ? 0.f : reg[(size_t)(jb + q) * g.rj + (size_t)(ib + x)];
    __syncthreads();
    for (int q = y; q < kLayoutTile; q += 8)
      if (ib + q < g.ni && jb + x < g.nj) chunk[ref + (unsigned)(ib + q) * g.si + (unsigned)(jb + x) * g.sj] = t[q][x];
  }
}
