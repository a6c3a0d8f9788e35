// Order of workgroups over tiles and chunks of columns.
#pragma once

namespace gdtp {

// Tile (or block of rows) of workgroup b when the eight XCDs (workgroup b runs on XCD b % 8) each
// take a contiguous eighth of the n tiles, in order: XCD x owns tiles [x per + min(x, rem), ...),
// per + (x < rem) of them (a bijection on [0, n)).  Neighbouring tiles then share an L2, so the halo
// texels a tile reads from its neighbours are mostly L2 hits instead of HBM re-reads.
__device__ __forceinline__ int XcdTile(int b, int n) {
  const int x = b % 8, k = b / 8, per = n / 8, rem = n % 8;
  return x * per + min(x, rem) + k;
}

// Columns in chunks of up to kMax, a chunk per workgroup: workgroups are numbered tile by tile and
// within a tile chunk by chunk, in XCD-contiguous order, so that a tile's chunks run on one XCD one
// after another and read its stencil, masks and row tables from that XCD's L2.  (With the chunks in a
// loop inside the workgroup, each waited for the one before it: 3.0 M texels x 64 columns, V-cycle
// residual of level 0 1027 us, 896 so; one colour pair of level 0, 16 launches, 554 us, one launch 448; a
// solve pair 348 to 292 ms.)
struct TileChunk {
  int tile, c0;
};
__device__ __forceinline__ TileChunk TileOf(int width, int b, int nTiles, int K) {
  const int chunks = (K + width - 1) / width;
  if (chunks == 1) return {XcdTile(b, nTiles), 0};
  const int v = XcdTile(b, nTiles * chunks);
  return {v / chunks, v % chunks * width};
}
template <int kMax>
__device__ __forceinline__ TileChunk TileOf(int b, int nTiles, int K) {
  return TileOf(kMax, b, nTiles, K);
}
template <int kMax>
static inline unsigned ChunkBlocks(long blocks, int K) { return (unsigned)(blocks * ((K + kMax - 1) / kMax)); }

}  // namespace gdtp
