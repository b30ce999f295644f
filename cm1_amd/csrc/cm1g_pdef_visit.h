// The points whose marks pdef_fix (cm1g_adv.hip) reads besides a tile's own
// 64-column word, and the halo mapping they use.  Host and device: the CPU
// test enumerates them over all widths with g++.
#pragma once

#if defined(__HIP__) || defined(__HIPCC__)
#define CM1_VISIT __host__ __device__ __forceinline__
#else
#define CM1_VISIT inline
#endif

// halo point of the horizontal fill (bcs, src/bc.F:180-364) -> the
// interior point whose value it holds
CM1_VISIT int pdef_wrap(int m, int n, bool periodic) {
  if (m < 1) return periodic ? (m + n < 1 ? 1 : m + n) : 1;
  if (m > n) return periodic ? (m - n > n ? n : m - n) : n;  // (past the halo: any point)
  return m;
}

// the column beside the tile of columns i0..i0+63 (the last tile ends with
// column ni, whose right neighbour is ni+1, wherever the 64 would end)
CM1_VISIT int pdef_side_col(int i0, int ni, bool right, bool periodic) {
  const int m = right ? (i0 + 64 < ni + 1 ? i0 + 64 : ni + 1) : i0 - 1;
  return pdef_wrap(m, ni, periodic);
}
