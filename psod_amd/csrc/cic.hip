// cic.hip -- a2 CIC deposit, a3 CIC^-1 (+ FoF seeds), a4 density order.
//
// Deposit (main file:1077-1265).  One workgroup owns the (8*TB*R)^3 nodes of
// a tile of TB^3 8^3-cell blocks (R = ng/nx in {1, 2}).  A node receives
// mass from the cells on both sides of it, so the workgroup reads its own
// blocks' particles (TB^2 contiguous runs of the cell-sorted records) plus
// the particles of the lower-neighbour boundary cells, and accumulates only
// the nodes it owns.  Every node is written exactly once with a plain
// store: no zero-fill and no global atomics.
//
// Node sums are 64-bit fixed point (weights * 2^36) in LDS, exact sums of
// the float32 weights and independent of particle order.  A particle's
// offset in its CIC cell is exact: the record holds u in [0, 8) relative to
// its 8^3 block, and R*u - floor(R*u) is exact for R in {1, 2}.  Each lane
// takes K consecutive particles of the sorted list and keeps the 8 node sums
// in registers while they share the same lower node (dense cells), adding
// them to LDS only when it changes.  Tiles are dispatched densest first, so
// that the long tiles of halo cores overlap the rest; the largest are cut
// into pieces whose node sums meet in memory.
#include "psod_internal.h"

#include <algorithm>
#include <mutex>

int psod_fill_i32(psod_ctx *c, int32_t *p, int64_t n, int32_t v);
int psod_fill_u64(psod_ctx *c, uint64_t *p, int64_t n, uint64_t v);

// weights in 2^-36 units: a node holds up to 2^28 unit weights
constexpr float FIX_SCALE = 68719476736.0f;  // 2^36
constexpr double FIX_INV = 1.0 / 68719476736.0;

// Tile of TB^3 blocks (8*TB cells per axis), R nodes per cell per axis.
// Halo ranges: the boundary cells of the lower-neighbour blocks of the tile,
// enumerated per neighbour block type; see tile_seg().
template <int TB>
struct TileSegs {
  static constexpr int NA = TB * TB * 64;  // x-1 face: single cells
  static constexpr int NB = TB * TB * 8;   // y-1 face: rows of 8 cells
  static constexpr int NC = TB * TB;       // z-1 face: 64-cell slabs
  static constexpr int ND = TB * 8;        // x-1,y-1 edge: single cells
  static constexpr int NE = TB * 8;        // x-1,z-1 edge: single cells
  static constexpr int NF = TB;            // y-1,z-1 edge: rows of 8
  static constexpr int N = NA + NB + NC + ND + NE + NF + 1;
};

// s-th halo range of a tile: neighbour block offset (in blocks, relative to
// the tile's first block), local cell key inside it and run length
template <int TB>
__device__ inline void tile_seg(int s, int *bi, int *bj, int *bk, int *loc,
                                int *len) {
  using T = TileSegs<TB>;
  if (s < T::NA) {  // lx=7 of block (-1, j, k); cell (ly, lz)
    const int j = (s >> 6) % TB, k = (s >> 6) / TB, c = s & 63;
    *bi = -1; *bj = j; *bk = k;
    *loc = ((c >> 3) * 8 + (c & 7)) * 8 + 7; *len = 1; return;
  }
  s -= T::NA;
  if (s < T::NB) {  // ly=7 of block (i, -1, k); row lz
    const int i = (s >> 3) % TB, k = (s >> 3) / TB, lz = s & 7;
    *bi = i; *bj = -1; *bk = k;
    *loc = (lz * 8 + 7) * 8; *len = 8; return;
  }
  s -= T::NB;
  if (s < T::NC) {  // lz=7 of block (i, j, -1)
    *bi = s % TB; *bj = s / TB; *bk = -1;
    *loc = 7 * 64; *len = 64; return;
  }
  s -= T::NC;
  if (s < T::ND) {  // lx=7, ly=7 of block (-1, -1, k); cell lz
    *bi = -1; *bj = -1; *bk = s >> 3;
    *loc = ((s & 7) * 8 + 7) * 8 + 7; *len = 1; return;
  }
  s -= T::ND;
  if (s < T::NE) {  // lx=7, lz=7 of block (-1, j, -1); cell ly
    *bi = -1; *bj = s >> 3; *bk = -1;
    *loc = (7 * 8 + (s & 7)) * 8 + 7; *len = 1; return;
  }
  s -= T::NE;
  if (s < T::NF) {  // ly=7, lz=7 of block (i, -1, -1)
    *bi = s; *bj = -1; *bk = -1;
    *loc = (7 * 8 + 7) * 8; *len = 8; return;
  }
  *bi = -1; *bj = -1; *bk = -1;  // corner cell
  *loc = 511; *len = 1;
}

constexpr int DEP_T = 512;  // threads of a deposit workgroup (one tile)
constexpr int DEP_K = 4;  // consecutive particles per lane
constexpr int32_t DEP_CAPD = 8192;  // dense tiles dispatched first, at most
// Tiles of at least DEP_BIG own particles are deposited in pieces of about
// DEP_PIECE of them, one workgroup each: a 6e6-particle halo's central tile
// alone held the launch for 2.6 ms (1.1 for the rest of 512^3).
constexpr int32_t DEP_BIG = 1 << 17, DEP_PIECE = 1 << 15, DEP_BIGCAP = 512;

// Tiles cut into pieces: count[0] tiles (slots), count[1] pieces; slot s is
// tile[s], in np[s] pieces, done[s] of them finished, its node sums in
// acc[s * 4096 ..]; unit[u] = (slot, piece), or (-1, ..): nothing.  cap = 0:
// none.  The lists are sized by the npart of the call; a tile whose pieces
// would not fit (cell_start counts more records) is not cut.
struct BigTiles {
  int32_t cap, ucap;
  int32_t *count, *tile, *np, *done;
  int2 *unit;
  unsigned long long *acc;
};

// Dense tiles (at least dense_tile own particles, a tunable) are listed so
// that they are dispatched first: their long runs then overlap the rest
// instead of trailing it.  listed[tile] = 1 for a tile in dlist or in B.
// Clears the node sums of B's slots as well (any grid of at least ntile
// threads).
__global__ void k_tile_dense(const int32_t *__restrict__ cell_start,
                             int32_t nb, int32_t TB, int32_t ntile, int32_t capd,
                             int32_t dense_tile,
                             int32_t *__restrict__ listed,
                             int32_t *__restrict__ dcount,
                             int32_t *__restrict__ dlist, BigTiles B) {
  const int32_t tile = blockIdx.x * blockDim.x + threadIdx.x;
  for (int32_t i = tile; i < B.cap * 4096; i += gridDim.x * blockDim.x)
    B.acc[i] = 0ull;
  if (tile >= ntile) return;
  const int32_t nt = nb / TB;
  const int tx = tile % nt, ty = (tile / nt) % nt, tz = tile / (nt * nt);
  int32_t n = 0;
  for (int k = 0; k < TB; k++)
    for (int j = 0; j < TB; j++) {
      const int32_t b0 = ((tz * TB + k) * nb + (ty * TB + j)) * nb + tx * TB;
      n += cell_start[(b0 + TB) * BS3] - cell_start[b0 * BS3];
    }
  int32_t f = 0;
  if (B.cap > 0 && n >= DEP_BIG) {
    const int32_t s = atomicAdd(&B.count[0], 1);
    if (s < B.cap) {
      const int32_t np = (n + DEP_PIECE - 1) / DEP_PIECE,
                    u = atomicAdd(&B.count[1], np);
      const bool fits = u <= B.ucap - np;
      B.tile[s] = tile;
      B.np[s] = np;
      B.done[s] = 0;
      for (int32_t i = 0; i < np && u + i < B.ucap; i++)
        B.unit[u + i] = make_int2(fits ? s : -1, i);
      f = fits;
    }
  }
  if (!f && n >= dense_tile) {
    const int32_t k = atomicAdd(dcount, 1);
    if (k < capd) {
      dlist[k] = tile;
      f = 1;
    }
  }
  listed[tile] = f;
}

// Tile of workgroup b: b < capd takes the b-th listed dense tile; the others
// take the remaining tiles in an XCD-aware order (workgroups go round-robin
// over the 8 XCDs, each with its own L2: XCD x sweeps a contiguous slab of
// tiles, so that a tile finds its neighbours' boundary cells in its L2).
__device__ inline int32_t tile_of_block(int32_t b, int32_t ntile, int32_t capd,
                                        const int32_t *dcount,
                                        const int32_t *dlist,
                                        const int32_t *listed) {
  if (b < capd) return b < min(*dcount, capd) ? dlist[b] : -1;
  const int32_t q = b - capd;
  const int32_t tile = ntile % 8 == 0 ? (q % 8) * (ntile / 8) + q / 8 : q;
  return (capd > 0 && listed[tile]) ? -1 : tile;
}

// x within [0,1]; 0 for NaN
__device__ inline float clamp01(float x) {
  return __builtin_amdgcn_fmed3f(x, 0.0f, 1.0f);
}

// Deposit of the (8*TB*R)^3 nodes owned by one tile.  Own particles come
// from the TB^3 blocks, in runs of TB; halo particles from the ranges of
// tile_seg(), found by binary search on their prefix counts.  The first
// B.ucap workgroups take the pieces of the tiles in B.
//
// A weight becomes 2^36 fixed point by one rounding to an integer float
// (v_rndne) and an FP64 add onto 2^52: the low bits of the sum are the
// integer sum, exact up to 2^16 unit weights, and leave the register by one
// 64-bit subtraction.  Bound by VALU issue (85 %) and the LDS atomics
// together, at 2.1 TB/s of positions and nodes (12 bytes a particle, 4 a node;
// 4.0 TB/s of what it moves): 1024^3 8.66 -> 8.1 ms, zoom
// catalogue at 512^3 (with the pieces) 2.66 -> 1.10 ms, 256^3 on 512^3 nodes
// 0.42 -> 0.40 ms.  Slower at 1024^3: a margin of nodes in LDS instead of the
// bounds checks (9.2: fewer waves fit), 2, 3 or 8 particles per lane (9.0,
// 8.7, 10.9), the upper x plane kept in registers when the next particle lies
// in the next cell (8.2), workgroups of 1024 (11.0).
template <int R, int TB>
__global__ void __launch_bounds__(DEP_T)
k_cic_deposit(const int32_t *__restrict__ cell_start,
              const float4 *__restrict__ rec, int32_t nx, int32_t ng,
              int32_t shift, double norm, int32_t capd,
              const int32_t *__restrict__ dcount,
              const int32_t *__restrict__ dlist,
              const int32_t *__restrict__ listed, BigTiles B,
              float *__restrict__ grid) {
  constexpr int NN = 8 * TB * R;  // owned nodes per axis
  constexpr int NS = TileSegs<TB>::N;
  constexpr int NB = TB * TB * TB;  // own blocks
  __shared__ unsigned long long acc[NN * NN * NN];
  __shared__ int32_t hstart[NS];
  __shared__ int32_t hpre[NS + 1];
  __shared__ uint16_t hoff[NS];  // block offset, each axis + 2 in 4 bits
  __shared__ int32_t ostart[NB], opre[NB + 1];  // own blocks, x fastest
  __shared__ int32_t wtot[DEP_T / 64], lastpiece;
  const int32_t nb = nx >> 3;
  const int32_t nt = nb / TB;  // tiles per axis
  int32_t tile, slot = -1, piece = 0, np = 1;
  if ((int32_t)blockIdx.x < B.ucap) {
    if ((int32_t)blockIdx.x >= B.count[1]) return;
    const int2 u = B.unit[blockIdx.x];
    if (u.x < 0) return;
    slot = u.x;
    piece = u.y;
    np = B.np[slot];
    tile = B.tile[slot];
  } else {
    tile = tile_of_block((int32_t)blockIdx.x - B.ucap, nt * nt * nt, capd,
                         dcount, dlist, listed);
  }
  if (tile < 0) return;  // uniform per workgroup: before any barrier
  const int tx = tile % nt, ty = (tile / nt) % nt, tz = tile / (nt * nt);
  const int bx0 = tx * TB, by0 = ty * TB, bz0 = tz * TB;
  const int l = threadIdx.x & 63;
  for (int i = threadIdx.x; i < NN * NN * NN; i += DEP_T) acc[i] = 0ull;
  if (threadIdx.x < NB) {
    const int q = threadIdx.x % TB, j = (threadIdx.x / TB) % TB,
              k = threadIdx.x / (TB * TB);
    const int32_t b0 = ((bz0 + k) * nb + (by0 + j)) * nb + bx0 + q;
    ostart[threadIdx.x] = cell_start[b0 * BS3];
    opre[threadIdx.x + 1] = cell_start[(b0 + 1) * BS3];
  }
  // halo ranges and their prefix counts (blocks of DEP_T ranges)
  int32_t carry = 0;
  for (int base = 0; base < NS; base += DEP_T) {
    const int s = base + threadIdx.x;
    int32_t cnt = 0;
    if (s < NS) {
      int bi, bj, bk, loc, len;
      tile_seg<TB>(s, &bi, &bj, &bk, &loc, &len);
      const int32_t nbk = (wrapi(bz0 + bk, nb) * nb + wrapi(by0 + bj, nb)) * nb +
                          wrapi(bx0 + bi, nb);
      const int32_t k0 = nbk * BS3 + loc;
      const int32_t a = cell_start[k0];
      cnt = cell_start[k0 + len] - a;
      hstart[s] = a;
      // offset of the neighbour block relative to the tile origin, blocks
      hoff[s] = (uint16_t)(((bk + 2) << 8) | ((bj + 2) << 4) | (bi + 2));
    }
    const int w = threadIdx.x >> 6;
    const int32_t inc = wave_incl_scan(cnt);
    if (l == 63) wtot[w] = inc;
    __syncthreads();
    int32_t off = carry;
    for (int i = 0; i < w; i++) off += wtot[i];
    if (s < NS) hpre[s] = off + inc - cnt;
    for (int i = 0; i < DEP_T / 64; i++) carry += wtot[i];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    hpre[NS] = carry;
    opre[0] = 0;
    // prefix of the own blocks (their ends were stored in opre[1..])
    int32_t p = 0;
    for (int r = 0; r < NB; r++) {
      p += opre[r + 1] - ostart[r];
      opre[r + 1] = p;
    }
  }
  __syncthreads();
  const int32_t nown = opre[NB];
  const int32_t ntot = nown + hpre[NS];
  // register sums of the current lower node (2^52 + integer) and their flush
  // to LDS
  constexpr double MAGIC = 4503599627370496.0;  // 2^52
  double ra[8];
#pragma unroll
  for (int c = 0; c < 8; c++) ra[c] = MAGIC;
  int32_t rid = -1, rix = 0, riy = 0, riz = 0, run = 0;
  auto flush = [&]() {
    if (rid < 0) return;
#pragma unroll
    for (int c = 0; c < 8; c++) {
      const int ax = rix + (c & 1), ay = riy + ((c >> 1) & 1), az = riz + (c >> 2);
      if ((unsigned)ax < (unsigned)NN && (unsigned)ay < (unsigned)NN &&
          (unsigned)az < (unsigned)NN)
        atomicAdd(&acc[(az * NN + ay) * NN + ax],
                  (unsigned long long)(__double_as_longlong(ra[c]) -
                                       __double_as_longlong(MAGIC)));
    }
  };
  // this workgroup's share of the list: all of it, or a piece
  const int32_t per = ((ntot + np - 1) / np + DEP_T * DEP_K - 1) /
                      (DEP_T * DEP_K) * (DEP_T * DEP_K);
  const int32_t lo0 = min(piece * (int64_t)per, (int64_t)ntot),
                hi0 = min((int64_t)lo0 + per, (int64_t)ntot);
  // lane l of wave w takes list positions base + w*64*K + l*K + j, j < K.
  // All K records of a lane are requested before the first is used, so that
  // a wave keeps K loads per lane in flight.
  const int wv = threadIdx.x >> 6;
  for (int32_t base = lo0; base < hi0; base += DEP_T * DEP_K) {
    float4 rv[DEP_K];
    int32_t ob[DEP_K];  // block offset of the record, packed; 0 = none
    int32_t send = -1, sdel = 0, soff = 0;  // end of the segment at hand
#pragma unroll
    for (int j = 0; j < DEP_K; j++) {
      const int32_t t = base + wv * 64 * DEP_K + l * DEP_K + j;
      ob[j] = 0;
      if (t < hi0) {
        if (t >= send) {  // the next segment: record = t + sdel
          if (t < nown) {
            int lo = 0;  // last own block with opre <= t
#pragma unroll
            for (int o = NB / 2; o > 0; o >>= 1)
              if (opre[lo + o] <= t) lo += o;
            send = opre[lo + 1];
            sdel = ostart[lo] - opre[lo];
            soff = ((lo / (TB * TB) + 2) << 8) | ((lo / TB % TB + 2) << 4) |
                   (lo % TB + 2);
          } else {
            const int32_t th = t - nown;
            int lo = 0, hi = NS;  // last s with hpre[s] <= th
            while (hi - lo > 1) {
              const int mid = (lo + hi) >> 1;
              if (hpre[mid] <= th) lo = mid; else hi = mid;
            }
            send = nown + hpre[lo + 1];
            sdel = hstart[lo] - hpre[lo] - nown;
            soff = hoff[lo];
          }
        }
        ob[j] = soff;
        rv[j] = rec[t + sdel];
      }
    }
    // sums of one node stay below 2^52
    run += DEP_K;
    if (run > 32768) {
      flush();
      rid = -1;
#pragma unroll
      for (int c = 0; c < 8; c++) ra[c] = MAGIC;
      run = DEP_K;
    }
#pragma unroll
    for (int j = 0; j < DEP_K; j++) {
      if (ob[j] == 0) break;
      // lower node (tile-relative) and exact offsets
      const float4 r = rv[j];
      const float qx = (float)R * r.x, qy = (float)R * r.y, qz = (float)R * r.z;
      const float fx0 = floorf(qx), fy0 = floorf(qy), fz0 = floorf(qz);
      const int32_t ix = 8 * R * ((ob[j] & 15) - 2) + (int32_t)fx0;
      const int32_t iy = 8 * R * (((ob[j] >> 4) & 15) - 2) + (int32_t)fy0;
      const int32_t iz = 8 * R * ((ob[j] >> 8) - 2) + (int32_t)fz0;
      const float fx = qx - fx0, fy = qy - fy0, fz = qz - fz0;
      const int32_t id = ((iz + 16) * 64 + (iy + 16)) * 64 + (ix + 16);
      if (id != rid) {
        flush();
#pragma unroll
        for (int c = 0; c < 8; c++) ra[c] = MAGIC;
        run = DEP_K;
        rid = id;
        rix = ix;
        riy = iy;
        riz = iz;
      }
      // (wx wy) wz with the scale, a power of two, in wz
      // (a position that is not finite has offsets NaN: weight 0, by the clamp)
      const float wx[2] = {clamp01(1.0f - fx), clamp01(fx)},
                  wy[2] = {clamp01(1.0f - fy), clamp01(fy)},
                  wz[2] = {clamp01(1.0f - fz) * FIX_SCALE,
                           clamp01(fz) * FIX_SCALE};
#pragma unroll
      for (int c = 0; c < 8; c++)
        ra[c] += (double)rintf(wx[c & 1] * wy[(c >> 1) & 1] * wz[c >> 2]);
    }
  }
  flush();
  __syncthreads();
  const int32_t gx0 = bx0 * 8 * R, gy0 = by0 * 8 * R, gz0 = bz0 * 8 * R;
  unsigned long long *bacc = B.acc + (int64_t)max(slot, 0) * 4096;
  if (slot >= 0) {
    // the pieces' sums meet in memory (integers: any order); the last piece
    // to finish writes the tile
    for (int i = threadIdx.x; i < NN * NN * NN; i += DEP_T)
      if (acc[i]) atomicAdd(&bacc[i], acc[i]);
    __threadfence();
    __syncthreads();
    if (threadIdx.x == 0)
      lastpiece = atomicAdd(&B.done[slot], 1) == np - 1;
    __syncthreads();
    if (!lastpiece) return;
    __threadfence();
  }
  for (int i = threadIdx.x; i < NN * NN * NN; i += DEP_T) {
    const int ax = i % NN, ay = (i / NN) % NN, az = i / (NN * NN);
    const int32_t gx = (gx0 + ax + shift) & (ng - 1);
    const int32_t gy = (gy0 + ay + shift) & (ng - 1);
    const int32_t gz = (gz0 + az + shift) & (ng - 1);
    const unsigned long long v =
        slot >= 0 ? __hip_atomic_load(&bacc[i], __ATOMIC_RELAXED,
                                      __HIP_MEMORY_SCOPE_AGENT)
                  : acc[i];
    grid[((int64_t)gz * ng + gy) * ng + gx] =
        (float)((double)v * FIX_INV * norm);
  }
}

// A block of more than INT_CH records is shared by several workgroups: the
// first INT_CH of them by its own, the rest by one extra each, listed here as
// (block, piece).  A halo core's block alone held the launch: zoom catalogue
// at 512^3 2.30 -> 0.87 ms, 1024^3 8.5 -> 6.9, 128^3 70 -> 21 us, with the
// keys below (pieces of 2^14: 35 us at 128^3).
constexpr int32_t INT_CH = 1 << 12;
// From 2^21 particles on.  The list costs two short launches and the idle
// workgroups of its capacity, 4-7 us; what it saves depends on the densest
// block, which the host does not know.  Calls with seed keys, us without / with
// it, at 128^3 cells: uniform 45.3 / 51.3 (1.0e6 particles), 50.7 / 57.4 (2.1e6);
// clumps of at most 1% of the particles 47.4 / 50.7 (8e5), 50.7 / 54.2 (1.0e6),
// 53.0 / 55.9 (1.6e6), 66.5 / 60.2 (2.1e6, 15643 records in the densest block);
// 5% in one halo 52.2 / 54.7 (1.0e6), 59.1 / 56.8 (1.6e6), 67.5 / 60.0 (2.1e6).
// Blocks above about 10^4 records pay for it at any count (30% in one halo:
// 2.6e5 58.1 / 56.7, 1.0e6 102 / 71; half of 2.1e6 221 / 66): the line is where
// ordinary catalogues have them.
constexpr int64_t INT_SPLIT_MIN = 1 << 21;
__global__ void __launch_bounds__(256)
k_interp_split(const int32_t *__restrict__ cell_start, int32_t nblk,
               int32_t ucap, int32_t *__restrict__ count,
               int2 *__restrict__ unit) {
  const int32_t b = blockIdx.x * 256 + threadIdx.x;
  if (b >= nblk) return;
  const int32_t n = cell_start[b * BS3 + BS3] - cell_start[b * BS3];
  if (n <= INT_CH) return;
  const int32_t ne = (n - 1) / INT_CH;
  const int32_t u = atomicAdd(count, ne);
  for (int32_t i = 0; i < ne && u + i < ucap; i++)
    unit[u + i] = make_int2(b, i + 1);
}

// CIC^-1 of the block's own particles from its (8R+1)^3 nodes.  Workgroups
// before ucap take the extra pieces; no block is shared where ucap = 0 or
// where the pieces are more than ucap (cell_start counts more records than
// the npart of the call, which sized the list).
template <int R>
__global__ void __launch_bounds__(256)
k_cic_interp(const int32_t *__restrict__ cell_start,
             const float4 *__restrict__ rec, int32_t nx, int32_t ng,
             int32_t shift, const float *__restrict__ grid,
             float *__restrict__ rho_sorted, float *__restrict__ rho,
             const int32_t *__restrict__ lab_sorted, int64_t nhalo,
             unsigned long long *__restrict__ seed_key, int32_t ucap,
             const int32_t *__restrict__ ucount,
             const int2 *__restrict__ unit) {
  constexpr int NN = 8 * R + 1;
  __shared__ float g[NN * NN * NN];
  const int32_t nb = nx >> 3;
  int32_t blk = (int32_t)blockIdx.x - ucap, piece = 0;
  const int32_t nu = ucap > 0 ? ucount[0] : 0;
  const bool shared = ucap > 0 && nu <= ucap;
  if (blk < 0) {
    if (!shared || (int32_t)blockIdx.x >= nu) return;
    const int2 u = unit[blockIdx.x];
    blk = u.x;
    piece = u.y;
  } else if (nb >= 4) {
    // workgroups go round-robin over the 8 XCDs: row r of blocks along x
    // goes to XCD r % 8, whose L2 then serves the 128-byte lines that the
    // node rows of 4 blocks share (1024^3: 47 -> 27 GB read, 6.9 -> 6.4 ms;
    // into the particles' order at 1e8 3.7 -> 3.2 ms for the two launches)
    const int32_t j = blk >> 3;
    blk = ((j / nb) * 8 + (blk & 7)) * nb + j % nb;
  }
  const int bx = blk % nb, by = (blk / nb) % nb, bz = blk / (nb * nb);
  const int32_t gx0 = bx * 8 * R, gy0 = by * 8 * R, gz0 = bz * 8 * R;
  const bool seeds = seed_key && lab_sorted;
  // The block's record range first; then the first round's record and label
  // are requested before the nodes are staged, and each round requests the
  // next round's before its own are used, so that the loads of a block are
  // in flight together rather than one after the other.
  const int32_t s0 = cell_start[blk * BS3] + piece * INT_CH,
                sb = cell_start[blk * BS3 + BS3],
                s1 = shared ? min(sb, s0 + INT_CH) : sb;
  float4 r = make_float4(0.f, 0.f, 0.f, 0.f);
  int32_t h = -1;
  if (s0 + (int32_t)threadIdx.x < s1) {
    r = rec[s0 + threadIdx.x];
    if (seeds) h = lab_sorted[s0 + threadIdx.x];
  }
  for (int i = threadIdx.x; i < NN * NN * NN; i += 256) {
    const int ax = i % NN, ay = (i / NN) % NN, az = i / (NN * NN);
    const int32_t gx = (gx0 + ax + shift) & (ng - 1);
    const int32_t gy = (gy0 + ay + shift) & (ng - 1);
    const int32_t gz = (gz0 + az + shift) & (ng - 1);
    g[i] = grid[((int64_t)gz * ng + gy) * ng + gx];
  }
  __syncthreads();
  // the label at hand (uniform over the wave; -1: none), each lane's best key
  // of it, and the wave's maximum of them, given to the label
  int32_t held = -1;
  unsigned long long hkey = 0ull;
  auto give = [&]() {
    if (held < 0) return;
    const uint32_t kh = (uint32_t)(hkey >> 32);
    const uint32_t mh = wave_max_u32(kh);
    const uint32_t ml = wave_max_u32(kh == mh ? (uint32_t)hkey : 0u);
    if ((threadIdx.x & 63) == 0)
      atomicMax(&seed_key[held], ((unsigned long long)mh << 32) | ml);
  };
  // uniform trip count so that every lane of a wave takes part in the
  // reduction of the seed keys
  for (int32_t base = s0; base < s1; base += 256) {
    const int32_t k = base + threadIdx.x;
    const bool ok = k < s1;
    float4 rn = make_float4(0.f, 0.f, 0.f, 0.f);
    int32_t hn = -1;
    if (k + 256 < s1) {
      rn = rec[k + 256];
      if (seeds) hn = lab_sorted[k + 256];
    }
    float rf = 0.0f;
    int32_t idx = 0;
    if (ok) {
      const float qx = (float)R * r.x, qy = (float)R * r.y, qz = (float)R * r.z;
      const float fx0 = floorf(qx), fy0 = floorf(qy), fz0 = floorf(qz);
      const int ix = (int)fx0, iy = (int)fy0, iz = (int)fz0;
      const float fx = qx - fx0, fy = qy - fy0, fz = qz - fz0;
      const double wx[2] = {1.0 - (double)fx, (double)fx};
      const double wy[2] = {1.0 - (double)fy, (double)fy};
      const double wz[2] = {1.0 - (double)fz, (double)fz};
      double acc = 0.0;
#pragma unroll
      for (int c = 0; c < 8; c++) {
        const int ax = ix + (c & 1), ay = iy + ((c >> 1) & 1),
                  az = iz + (c >> 2);
        acc += (double)g[(az * NN + ay) * NN + ax] * wx[c & 1] *
               wy[(c >> 1) & 1] * wz[c >> 2];
      }
      rf = (float)acc;
      idx = __float_as_int(r.w);
      if (rho_sorted) rho_sorted[k] = rf;
      if (rho) rho[idx] = rf;
    }
    if (seeds) {
      const bool mem = ok && h >= 0 && h < nhalo;
      const unsigned long long key =
          mem ? (((unsigned long long)__float_as_uint(rf) << 32) |
                 (unsigned long long)(0xFFFFFFFFu - (uint32_t)idx))
              : 0ull;
      // Members of a halo are neighbours in cell order: each lane keeps its
      // best key of the label at hand, and the wave reduces them only when
      // other labels appear (a 64-bit shuffle maximum per round and label:
      // zoom catalogue at 512^3 1.6 ms against 0.9).
      if (mem && h == held) hkey = key > hkey ? key : hkey;
      uint64_t todo = __ballot(mem && h != held);
      while (todo) {
        give();
        held = __builtin_amdgcn_readlane(h, __ffsll((unsigned long long)todo) - 1);
        const bool mine = mem && h == held;
        hkey = mine ? key : 0ull;
        todo &= ~__ballot(mine);
      }
    }
    r = rn;
    h = hn;
  }
  give();
}

static int check_grid_args(int32_t nx, int32_t ng, int32_t shift) {
  if (nx < 8 || nx > 1024 || (nx & (nx - 1)))
    return psod_set_error(PSOD_E_ARG, "nx=%d must be a power of two in [8,1024]",
                          nx);
  if (ng != nx && ng != 2 * nx)
    return psod_set_error(PSOD_E_ARG, "ng=%d must be nx or 2*nx (nx=%d)", ng,
                          nx);
  if (shift < 0 || shift >= ng)
    return psod_set_error(PSOD_E_ARG, "shift=%d outside [0, ng)", shift);
  return PSOD_OK;
}

// Tiles of a deposit launch and the length of its tile list (ints): the
// listed flags of every tile, the dense-tile count and the dense-tile list.
static int32_t deposit_tiles(int32_t nx, int32_t ng, int32_t *TB,
                             int32_t *ntile, int32_t *capd) {
  const int32_t nb = nx / 8;
  *TB = (ng == nx && nb % 2 == 0) ? 2 : 1;
  *ntile = (nb / *TB) * (nb / *TB) * (nb / *TB);
  *capd = std::min<int32_t>(*ntile, DEP_CAPD);
  return *ntile + *capd + 64;
}

// Queues the deposit on the context's stream with `listed` as its tile list
// (deposit_tiles() ints); returns without waiting.
static int deposit_queue(psod_ctx *ctx, int64_t npart, int32_t nx,
                         const int32_t *d_cell_start, const float *d_rec,
                         int32_t ng, int32_t shift, float *d_grid,
                         int32_t *listed, const BigTiles &B) {
  int32_t TB, ntile, capd;
  (void)deposit_tiles(nx, ng, &TB, &ntile, &capd);
  const int32_t nb = nx / 8;
  const double norm = (double)ng * (double)ng * (double)ng / (double)npart;
  int32_t *dcount = listed + ntile, *dlist = dcount + 32;
  hipStream_t st = ctx->stream;
  const unsigned nblk = (unsigned)(B.ucap + ntile + capd);
  if (capd > 0) {
    PSOD_TRY(psod_fill_i32(ctx, dcount, 3, 0));
    k_tile_dense<<<std::max(grid_for(ntile, 256), 4u * (unsigned)B.cap), 256, 0,
                   st>>>(
        d_cell_start, nb, TB, ntile, capd,
        psod_tunables_for(ctx, nx).dense_tile, listed, dcount, dlist, B);
    PSOD_LAUNCH_CHECK();
  }
  if (ng == nx && TB == 2)
    k_cic_deposit<1, 2><<<nblk, DEP_T, 0, st>>>(
        d_cell_start, (const float4 *)d_rec, nx, ng, shift, norm, capd, dcount,
        dlist, listed, B, d_grid);
  else if (ng == nx)
    k_cic_deposit<1, 1><<<nblk, DEP_T, 0, st>>>(
        d_cell_start, (const float4 *)d_rec, nx, ng, shift, norm, capd, dcount,
        dlist, listed, B, d_grid);
  else
    k_cic_deposit<2, 1><<<nblk, DEP_T, 0, st>>>(
        d_cell_start, (const float4 *)d_rec, nx, ng, shift, norm, capd, dcount,
        dlist, listed, B, d_grid);
  PSOD_LAUNCH_CHECK();
  return PSOD_OK;
}

extern "C" int psod_cic_deposit(psod_ctx *ctx, int64_t npart, int32_t nx,
                                const int32_t *d_cell_start,
                                const float *d_rec, int32_t ng, int32_t shift,
                                float *d_grid) {
  PSOD_TRY(psod_use_device(ctx));
  PSOD_TRY(check_grid_args(nx, ng, shift));
  if (npart <= 0 || !d_cell_start || !d_rec || !d_grid)
    return psod_set_error(PSOD_E_ARG, "psod_cic_deposit: bad arguments");
  int32_t TB, ntile, capd;
  const size_t nlist = (size_t)deposit_tiles(nx, ng, &TB, &ntile, &capd);
  // the tile list, then the tiles in pieces: 3 ints per slot, their units
  // and their node sums
  BigTiles B = {};
  B.cap = (int32_t)std::min<int64_t>(std::min<int64_t>(ntile, DEP_BIGCAP),
                                     npart / DEP_BIG);
  B.ucap = B.cap > 0 ? (int32_t)(npart / DEP_PIECE) + B.cap : 0;
  const size_t o1 = (nlist * 4 + 255) & ~(size_t)255,
               o2 = o1 + (((size_t)B.cap * 12 + 255) & ~(size_t)255),
               o3 = o2 + (((size_t)B.ucap * 8 + 255) & ~(size_t)255);
  char *buf = (char *)psod_scratch(ctx, S_TILE, o3 + (size_t)B.cap * 4096 * 8);
  if (!buf) return PSOD_E_NOMEM;
  B.count = (int32_t *)buf + ntile + 1;  // beside the dense-tile count
  B.tile = (int32_t *)(buf + o1);
  B.np = B.tile + B.cap;
  B.done = B.np + B.cap;
  B.unit = (int2 *)(buf + o2);
  B.acc = (unsigned long long *)(buf + o3);
  PSOD_TRY(deposit_queue(ctx, npart, nx, d_cell_start, d_rec, ng, shift,
                         d_grid, (int32_t *)buf, B));
  return psod_finish(ctx);
}

// ---------------------------------------------------------------------------
// The deposit for callers that cannot allocate device memory.  Its tile list
// lives in `scratch`, a fixed array of every device the library runs on,
// large enough for the largest valid grid (nx = 1024, ng = 2048: 2^21 tiles).
// In host code the array's name is not a device address: psod_create
// resolves the array of its device once (hipGetSymbolAddress, with that
// device current) and the entry point passes only that address on.
// ---------------------------------------------------------------------------
constexpr int32_t STATIC_TILE_INTS = (1 << 21) + DEP_CAPD + 64;
constexpr int PSOD_MAX_DEVICES = 64;
static __device__ __align__(256) int32_t scratch[STATIC_TILE_INTS];
static int32_t *g_scratch[PSOD_MAX_DEVICES];
static std::mutex g_scratch_mu;

// Called by psod_create with `device` current.
int psod_static_scratch_init(int device) {
  if (device < 0 || device >= PSOD_MAX_DEVICES)
    return psod_set_error(PSOD_E_ARG, "device %d beyond the %d the library "
                          "supports", device, PSOD_MAX_DEVICES);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch[device]) return PSOD_OK;
  void *p = nullptr;
  PSOD_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
  if (!p)
    return psod_set_error(PSOD_E_DEVICE, "no address for the fixed tile "
                          "list of device %d", device);
  g_scratch[device] = (int32_t *)p;
  return PSOD_OK;
}

extern "C" int psod_cic_deposit_noalloc(psod_ctx *ctx, int64_t npart,
                                        int32_t nx,
                                        const int32_t *d_cell_start,
                                        const float *d_rec, int32_t ng,
                                        int32_t shift, float *d_grid) {
  PSOD_TRY(psod_use_device(ctx));
  PSOD_TRY(check_grid_args(nx, ng, shift));
  if (npart <= 0 || !d_cell_start || !d_rec || !d_grid)
    return psod_set_error(PSOD_E_ARG, "psod_cic_deposit_noalloc: bad "
                          "arguments");
  int32_t TB, ntile, capd;
  const int32_t nlist = deposit_tiles(nx, ng, &TB, &ntile, &capd);
  if (nlist > STATIC_TILE_INTS)
    return psod_set_error(PSOD_E_CAPACITY, "psod_cic_deposit_noalloc: %d "
                          "tile-list entries exceed the fixed %d", nlist,
                          STATIC_TILE_INTS);
  int32_t *listed = nullptr;
  {
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (ctx->device >= 0 && ctx->device < PSOD_MAX_DEVICES)
      listed = g_scratch[ctx->device];
  }
  if (!listed)
    return psod_set_error(PSOD_E_DEVICE, "psod_cic_deposit_noalloc: the "
                          "fixed tile list of device %d is not set up",
                          ctx->device);
  // no tiles in pieces: their sums would need memory
  return deposit_queue(ctx, npart, nx, d_cell_start, d_rec, ng, shift, d_grid,
                       listed, BigTiles{});
}

extern "C" int psod_cic_interp(psod_ctx *ctx, int64_t npart, int32_t nx,
                               const int32_t *d_cell_start, const float *d_rec,
                               int32_t ng, int32_t shift, const float *d_grid,
                               float *d_rho_sorted, float *d_rho,
                               const int32_t *d_lab_sorted, int64_t nhalo,
                               uint64_t *d_seed_key) {
  PSOD_TRY(psod_use_device(ctx));
  PSOD_TRY(check_grid_args(nx, ng, shift));
  if (npart <= 0 || !d_cell_start || !d_rec || !d_grid)
    return psod_set_error(PSOD_E_ARG, "psod_cic_interp: bad arguments");
  const int32_t nb = nx / 8;
  const unsigned nblk = (unsigned)nb * nb * nb;
  // the keys are maxima over the members: clear them on this stream, so
  // that no fill queued elsewhere can race the atomics below
  if (d_seed_key && d_lab_sorted && nhalo > 0)
    PSOD_TRY(psod_fill_u64(ctx, d_seed_key, nhalo, 0));
  int32_t ucap = 0, *ucount = nullptr;
  int2 *unit = nullptr;
  if (npart >= INT_SPLIT_MIN) {
    const int32_t cap = (int32_t)(npart / INT_CH + 7) & ~7;  // whole rounds of XCDs
    ucount = (int32_t *)psod_scratch(ctx, S_TILE, 256 + (size_t)cap * 8);
    if (!ucount) return PSOD_E_NOMEM;
    ucap = cap;
    unit = (int2 *)(ucount + 64);
    PSOD_TRY(psod_fill_i32(ctx, ucount, 1, 0));
    k_interp_split<<<grid_for(nblk, 256), 256, 0, ctx->stream>>>(
        d_cell_start, (int32_t)nblk, ucap, ucount, unit);
    PSOD_LAUNCH_CHECK();
  }
  if (ng == nx)
    k_cic_interp<1><<<nblk + (unsigned)ucap, 256, 0, ctx->stream>>>(
        d_cell_start, (const float4 *)d_rec, nx, ng, shift, d_grid,
        d_rho_sorted, d_rho, d_lab_sorted, nhalo,
        (unsigned long long *)d_seed_key, ucap, ucount, unit);
  else
    k_cic_interp<2><<<nblk + (unsigned)ucap, 256, 0, ctx->stream>>>(
        d_cell_start, (const float4 *)d_rec, nx, ng, shift, d_grid,
        d_rho_sorted, d_rho, d_lab_sorted, nhalo,
        (unsigned long long *)d_seed_key, ucap, ucount, unit);
  PSOD_LAUNCH_CHECK();
  return psod_finish(ctx);
}

__global__ void k_seed_index(const unsigned long long *__restrict__ key,
                             int64_t n, int32_t *__restrict__ seed) {
  const int64_t h = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (h >= n) return;
  const unsigned long long k = key[h];
  seed[h] = (k == 0ull) ? -1
                        : (int32_t)(0xFFFFFFFFu - (uint32_t)(k & 0xFFFFFFFFull));
}

extern "C" int psod_seed_index(psod_ctx *ctx, int64_t nhalo,
                               const uint64_t *d_seed_key, int32_t *d_seed) {
  PSOD_TRY(psod_use_device(ctx));
  if (nhalo <= 0) return PSOD_OK;
  k_seed_index<<<grid_for(nhalo, 256), 256, 0, ctx->stream>>>(
      (const unsigned long long *)d_seed_key, nhalo, d_seed);
  PSOD_LAUNCH_CHECK();
  return psod_finish(ctx);
}

// Members of a label come in runs (a halo's members are neighbours in cell
// order, and catalogues list each group's members together), so each wave
// adds its 64 labels with one atomic per distinct label of the wave; after
// LC_RUNS distinct labels the remaining lanes add their own.  One atomic per
// particle ran at 85 GB/s on 1024^3 particles.  Each wave takes a contiguous
// range of the labels and holds the count of its current label across its
// rounds, adding it when another label's run starts: a halo of 5e7 members
// costs one atomic per wave that meets it, not one per 64 members (all on
// one counter: 9.3 ms for the zoom catalogue's central halo).
constexpr int LC_RUNS = 4;
__global__ void __launch_bounds__(256)
k_label_counts(const int32_t *__restrict__ lab, int64_t n, int64_t nhalo,
               int32_t *__restrict__ cnt) {
  const int l = threadIdx.x & 63;
  const int64_t nw = (int64_t)gridDim.x * (blockDim.x >> 6);
  const int64_t w = (int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  const int64_t per = ((n + nw - 1) / nw + 63) & ~(int64_t)63;
  const int64_t lo = w * per, hi = min(n, lo + per);
  int32_t hold = -1, hcnt = 0;  // wave-uniform: the label held and its count
  // uniform trip count per wave: every lane takes part in the ballots
  for (int64_t b = lo; b < hi; b += 64) {
    const int64_t i = b + l;
    const int32_t h = i < hi ? lab[i] : -1;
    const bool mem = h >= 0 && h < nhalo;
    uint64_t todo = __ballot(mem);
    for (int r = 0; todo; r++) {
      if (r == LC_RUNS) {
        if ((todo >> l) & 1) atomicAdd(&cnt[h], 1);
        break;
      }
      const int leader = __ffsll((unsigned long long)todo) - 1;
      const int32_t hl = __shfl(h, leader, 64);
      const uint64_t same = __ballot(mem && h == hl);
      const int32_t c = (int32_t)__popcll(same);
      if (hl == hold) {
        hcnt += c;
      } else {
        if (l == 0 && hcnt > 0) atomicAdd(&cnt[hold], hcnt);
        hold = hl;
        hcnt = c;
      }
      todo &= ~same;
    }
  }
  if (l == 0 && hcnt > 0) atomicAdd(&cnt[hold], hcnt);
}

extern "C" int psod_label_counts(psod_ctx *ctx, int64_t npart,
                                 const int32_t *d_labels, int64_t nhalo,
                                 int32_t *d_nmem) {
  PSOD_TRY(psod_use_device(ctx));
  PSOD_TRY(psod_fill_i32(ctx, d_nmem, nhalo, 0));
  if (npart > 0) {
    k_label_counts<<<grid_for(npart, 256, (int64_t)ctx->num_cus * 64), 256, 0,
                     ctx->stream>>>(d_labels, npart, nhalo, d_nmem);
    PSOD_LAUNCH_CHECK();
  }
  return psod_finish(ctx);
}

// ---------------------------------------------------------------------------
// a4: density order.  Ascending sort of (0xFFFFFFFF - float bits of rho)
// with the particle index as a stable payload = decreasing rho, ties by
// index; npart_new = #(rho > threshold) + 1 (main file:1029-1032).
// ---------------------------------------------------------------------------
extern "C" int psod_density_order(psod_ctx *ctx, int64_t npart,
                                  const float *d_rho, double threshold,
                                  int32_t *d_isort, int64_t *npart_new) {
  PSOD_TRY(psod_use_device(ctx));
  if (npart <= 0 || !d_rho || !d_isort || !npart_new)
    return psod_set_error(PSOD_E_ARG, "psod_density_order: bad arguments");
  unsigned long long *cnt =
      (unsigned long long *)psod_scratch(ctx, S_MISC, 256);
  if (!cnt) return PSOD_E_NOMEM;
  PSOD_TRY(psod_fill_u64(ctx, (uint64_t *)cnt, 1, 0));
  // float threshold: rho > thr in float equals rho > threshold for the
  // thresholds used (exactly representable, e.g. 100)
  PSOD_TRY(psod_order_by_density(ctx, npart, d_rho, (float)threshold, cnt,
                                 d_isort));
  unsigned long long h = 0;
  PSOD_HIP(hipMemcpyAsync(&h, cnt, 8, hipMemcpyDeviceToHost, ctx->stream));
  PSOD_HIP(hipStreamSynchronize(ctx->stream));
  int64_t nn = (int64_t)h + 1;
  if (nn > npart) nn = npart;
  *npart_new = nn;
  return PSOD_OK;
}
