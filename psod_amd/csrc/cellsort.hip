// cellsort.hip -- a5: cell bucketing as an integer counting sort.
//
// Replaces main file:1561-1604 (cell key, quick_sort of the keys as reals,
// run-length first_ngp/num_ngp): an MSD radix sort of the particles' 8^3
// blocks, a counting sort by cell inside small groups of blocks, and the
// offsets of every cell.  The output records hold the particle position
// relative to the origin of its 8^3-cell block:
// u = x*nx - 8*floor(floor(x*nx)/8), exact in float32 (a multiple-of-8
// subtraction from x*nx, itself exact for a power-of-two nx).
#include "psod_internal.h"

#include <algorithm>

__global__ void k_fill_i32(int32_t *__restrict__ p, int64_t n, int32_t v) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    p[i] = v;
}

__global__ void k_fill_u64(uint64_t *__restrict__ p, int64_t n, uint64_t v) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    p[i] = v;
}

int psod_fill_i32(psod_ctx *c, int32_t *p, int64_t n, int32_t v) {
  if (n <= 0) return PSOD_OK;
  k_fill_i32<<<grid_for(n, 256, 8192), 256, 0, c->stream>>>(p, n, v);
  PSOD_LAUNCH_CHECK();
  return PSOD_OK;
}

int psod_fill_u64(psod_ctx *c, uint64_t *p, int64_t n, uint64_t v) {
  if (n <= 0) return PSOD_OK;
  k_fill_u64<<<grid_for(n, 256, 8192), 256, 0, c->stream>>>(p, n, v);
  PSOD_LAUNCH_CHECK();
  return PSOD_OK;
}

// scaled coordinate in [0, nx) and its cell
__device__ inline float scaled_wrap(float x, int32_t nx, int32_t *cell) {
  float xs = x * (float)nx;
  if (xs >= (float)nx) xs -= (float)nx;
  if (xs < 0.0f) xs += (float)nx;
  int32_t c = (int32_t)floorf(xs);
  if (c >= nx) { c -= nx; xs -= (float)nx; }
  *cell = c;
  return xs;
}

// Block of a particle (8^3 cells), its scaled coordinates and cell
struct PartCell {
  float xs, ys, zs;
  int32_t cx, cy, cz, blk;
};

__device__ inline PartCell part_cell3(float x, float y, float z, int32_t nx) {
  PartCell p;
  p.xs = scaled_wrap(x, nx, &p.cx);
  p.ys = scaled_wrap(y, nx, &p.cy);
  p.zs = scaled_wrap(z, nx, &p.cz);
  const int32_t nb = nx >> 3;
  p.blk = ((p.cz >> 3) * nb + (p.cy >> 3)) * nb + (p.cx >> 3);
  return p;
}

__device__ inline PartCell part_cell(const float *pos, int64_t i, int32_t nx) {
  return part_cell3(pos[3 * i + 0], pos[3 * i + 1], pos[3 * i + 2], nx);
}

__device__ inline int32_t block_of(const float4 &v, int32_t nx) {
  return part_cell3(v.x, v.y, v.z, nx).blk;
}

// ---------------------------------------------------------------------------
// Particles into groups of blocks: an MSD radix sort in at most two passes
// of at most CS_DB bits (1024^3 cells: 2^21 blocks, groups of 4, so 10 and
// 9 bits).  Elements travel as raw positions with their index, and labels;
// the block is recomputed from the position wherever it is needed.  A
// workgroup sorts a chunk of CH elements by digit in LDS and writes it in
// digit order.  The places come from a counter per digit (from the digit
// counts of the pass, counted down): the order inside a bucket does not
// matter, so no per-tile counts are kept, and a digit's runs of successive
// chunks are neighbours in memory.
//
// At 1024^3 the sort takes 37.0 ms (hist 2.4, scatter 10.6, hist 1.0, scatter
// 9.0, final 8.4, large groups 3.8, subsort 1.7); three passes of 7 bits with
// per-tile counts and a block sort took 55.  What bounds it is HBM: a pass
// moves 40 bytes per particle (4.1-5.2 TB/s in the scatters, 4.8 in
// k_cs_final).  A chunk's run of one digit is short (CH / 2^bits elements, 4 to 16), so its first and
// last 128-byte lines are partial, and so are most lines of the 4-byte
// labels.  They reach memory whole when the neighbouring runs are written
// through the same L2 soon after: each XCD has its own L2, and workgroups go
// round-robin over the 8 XCDs.  In the first pass the chunks c = x (mod 8)
// therefore have counters of their own per digit; in the second an XCD takes
// a contiguous eighth of the chunks (bucket after bucket).
// ---------------------------------------------------------------------------
constexpr int CS_DB = 10;  // digit bits of a pass, at most
constexpr int CS_XCD = 8;

// chunk of workgroup w of a pass over nc chunks (-1: none): round-robin
// (first pass) or an eighth of the chunks per XCD
template <bool FROM_POS>
__device__ inline int32_t cs_chunk(int32_t w, int32_t nc) {
  if (FROM_POS) return w < nc ? w : -1;
  const int32_t per = (nc + CS_XCD - 1) / CS_XCD;
  const int32_t c = (w % CS_XCD) * per + w / CS_XCD;
  return w / CS_XCD < per && c < nc ? c : -1;
}

// Digit counts of the first pass, per digit and chunk class (chunk mod 8):
// H[digit * 8 + class].  A workgroup counts many chunks of one class.
template <int CH>
__global__ void __launch_bounds__(256)
k_cs_hist1(const float *__restrict__ pos, int64_t n, int32_t nx, int shift,
           int dbits, int32_t *__restrict__ H) {
  __shared__ int32_t hist[1 << CS_DB];
  const int32_t nd = 1 << dbits;
  for (int d = threadIdx.x; d < nd; d += 256) hist[d] = 0;
  __syncthreads();
  // gridDim.x is a multiple of 8: the class stays
  for (int64_t c0 = (int64_t)blockIdx.x * CH; c0 < n;
       c0 += (int64_t)gridDim.x * CH) {
    const int64_t c1 = min(n, c0 + CH);
    for (int64_t k = c0 + threadIdx.x; k < c1; k += 256)
      atomicAdd(&hist[(part_cell(pos, k, nx).blk >> shift) & (nd - 1)], 1);
  }
  __syncthreads();
  for (int d = threadIdx.x; d < nd; d += 256)
    if (hist[d]) atomicAdd(&H[d * CS_XCD + blockIdx.x % CS_XCD], hist[d]);
}

// Starts of the first pass from its counts (one workgroup): S[digit*8+class],
// bucket starts bs[0..nd], and for the second pass the chunks of each bucket,
// their prefix cb[0..nd] and the bucket of each chunk.
__global__ void __launch_bounds__(1024)
k_cs_starts(const int32_t *__restrict__ H, int32_t nd, int32_t n, int32_t ch,
            int32_t *__restrict__ S, int32_t *__restrict__ bs,
            int32_t *__restrict__ cb, int32_t *__restrict__ cmap) {
  __shared__ int32_t wsum[16];
  const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
  auto scan = [&](int32_t v) {  // exclusive over the workgroup
    const int32_t inc = wave_incl_scan(v);
    __syncthreads();
    if (l == 63) wsum[w] = inc;
    __syncthreads();
    int32_t off = 0;
    for (int i = 0; i < w; i++) off += wsum[i];
    return off + inc - v;
  };
  const int32_t d = threadIdx.x;  // nd <= 1024
  int32_t h[CS_XCD], tot = 0;
  for (int x = 0; x < CS_XCD; x++) {
    h[x] = d < nd ? H[d * CS_XCD + x] : 0;
    tot += h[x];
  }
  int32_t e = scan(tot);
  if (d < nd) {
    bs[d] = e;
    for (int x = 0; x < CS_XCD; x++) {
      S[d * CS_XCD + x] = e;
      e += h[x];
    }
  }
  if (d == 0) bs[nd] = n;
  if (!cb) return;  // uniform
  const int32_t k = (tot + ch - 1) / ch;
  const int32_t c = scan(k);
  if (d < nd) cb[d] = c;
  if (d == nd - 1) cb[nd] = c + k;
  __syncthreads();
  __threadfence_block();
  // chunks of a bucket, written by its wave of 64 lanes
  for (int32_t q = w; q < nd; q += 16) {
    const int32_t a = cb[q], b = cb[q + 1];
    for (int32_t i = a + l; i < b; i += 64) cmap[i] = q;
  }
}

// Digit counts of the second pass, H[bucket * nd + digit], from the 16-bit
// keys the first pass left.  A workgroup takes `per` consecutive chunks and
// adds its counts when the bucket changes.  The key array is 16-byte aligned.
__global__ void __launch_bounds__(256)
k_cs_hist2(const uint16_t *__restrict__ key, int shift, int dbits,
           const int32_t *__restrict__ bs, int32_t nbk,
           const int32_t *__restrict__ cb, const int32_t *__restrict__ cmap,
           int32_t ch, int32_t per, int32_t *__restrict__ H) {
  __shared__ int32_t hist[1 << CS_DB];
  const int32_t nd = 1 << dbits, nc = cb[nbk];
  const int32_t c0 = blockIdx.x * per, c1 = min(nc, c0 + per);
  if (c0 >= c1) return;  // uniform
  for (int d = threadIdx.x; d < nd; d += 256) hist[d] = 0;
  __syncthreads();
  const uint4 *key8 = reinterpret_cast<const uint4 *>(key);
  int32_t b = cmap[c0];
  for (int32_t c = c0; c < c1; c++) {
    const int32_t k0 = bs[b] + (c - cb[b]) * ch, k1 = min(bs[b + 1], k0 + ch);
    // 8 keys per load: the aligned words that meet [k0, k1)
    for (int32_t w = (k0 >> 3) + (int32_t)threadIdx.x; w << 3 < k1; w += 256) {
      const uint4 q = key8[w];
      const uint32_t p[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
      for (int j = 0; j < 8; j++) {
        const uint32_t kv = (p[j >> 1] >> ((j & 1) * 16)) & 0xFFFFu;
        const int32_t k = (w << 3) + j;
        if (k >= k0 && k < k1) atomicAdd(&hist[(kv >> shift) & (nd - 1)], 1);
      }
    }
    const int32_t bn = c + 1 < c1 ? cmap[c + 1] : -1;
    if (bn != b) {
      __syncthreads();
      for (int d = threadIdx.x; d < nd; d += 256) {
        const int32_t v = hist[d];
        if (v) atomicAdd(&H[(int64_t)b * nd + d], v);
        hist[d] = 0;
      }
      __syncthreads();
      b = bn;
    }
  }
}

// One chunk: elements sorted by digit in LDS and written in digit order.
// Reads positions and labels (first pass) or the elements of bucket cmap[c]
// (second pass).  H counts the free places of a digit down to zero; kout
// (first pass of two) receives the low 16 bits of the block.
template <bool FROM_POS, int CH, int TH>
__global__ void __launch_bounds__(TH)
k_cs_scatter(const float *__restrict__ pos, const float4 *__restrict__ sin,
             const int32_t *__restrict__ lin, int64_t n, int32_t nx, int shift,
             int dbits, const int32_t *__restrict__ bs, int32_t nbk,
             const int32_t *__restrict__ cb, const int32_t *__restrict__ cmap,
             const int32_t *__restrict__ S, int32_t *__restrict__ H,
             float4 *__restrict__ sout, int32_t *__restrict__ lout,
             uint16_t *__restrict__ kout) {
  constexpr int U = CH / TH;
  __shared__ float4 ex[CH];  // the chunk in digit order, then its labels
  __shared__ int32_t lcnt[1 << CS_DB], lst[1 << CS_DB], gb[1 << CS_DB];
  __shared__ int32_t wsum[TH / 64];
  int32_t *exi = reinterpret_cast<int32_t *>(ex);
  const int32_t nd = 1 << dbits;
  int64_t k0;
  int32_t cn;
  int64_t tab;  // first entry of the chunk's counters
  int32_t step;
  if (FROM_POS) {
    const int32_t c = cs_chunk<true>(blockIdx.x, (int32_t)((n + CH - 1) / CH));
    if (c < 0) return;
    k0 = (int64_t)c * CH;
    cn = (int32_t)min((int64_t)CH, n - k0);
    tab = c % CS_XCD;
    step = CS_XCD;
  } else {
    const int32_t c = cs_chunk<false>(blockIdx.x, cb[nbk]);
    if (c < 0) return;
    const int32_t b = cmap[c];
    k0 = bs[b] + (c - cb[b]) * CH;
    cn = min(CH, bs[b + 1] - (int32_t)k0);
    tab = (int64_t)b * nd;
    step = 1;
  }
  for (int d = threadIdx.x; d < nd; d += TH) lcnt[d] = 0;
  __syncthreads();
  float4 v[U];
  int32_t ll[U], sd[U];  // label; digit << 16 | rank within the digit
#pragma unroll
  for (int u = 0; u < U; u++) {
    const int32_t i = threadIdx.x + TH * u;
    if (i < cn) {
      if (FROM_POS) {
        const float *p = pos + 3 * (k0 + i);
        v[u].x = p[0];
        v[u].y = p[1];
        v[u].z = p[2];
        v[u].w = __int_as_float((int32_t)(k0 + i));
      } else {
        // component-wise, so that the chunk stays in registers
        const float4 r = sin[k0 + i];
        v[u].x = r.x;
        v[u].y = r.y;
        v[u].z = r.z;
        v[u].w = r.w;
      }
      ll[u] = lin ? lin[k0 + i] : -1;
    }
  }
#pragma unroll
  for (int u = 0; u < U; u++) {
    sd[u] = 0;
    if (threadIdx.x + TH * u < cn) {
      const int32_t d = (block_of(v[u], nx) >> shift) & (nd - 1);
      sd[u] = (d << 16) | atomicAdd(&lcnt[d], 1);
    }
  }
  __syncthreads();
  // exclusive scan of the counts; a digit's places are taken at once
  constexpr int DV = (1 << CS_DB) / TH > 1 ? (1 << CS_DB) / TH : 1;
  int32_t c[DV], tot = 0;
  for (int i = 0; i < DV; i++) {
    const int32_t d = threadIdx.x * DV + i;
    c[i] = d < nd ? lcnt[d] : 0;
    tot += c[i];
  }
  const int32_t inc = wave_incl_scan(tot);
  if ((threadIdx.x & 63) == 63) wsum[threadIdx.x >> 6] = inc;
  int32_t place[DV];
  for (int i = 0; i < DV; i++) {
    const int64_t t = tab + (int64_t)(threadIdx.x * DV + i) * step;
    place[i] = 0;
    if (c[i] > 0) place[i] = S[t] + atomicSub(&H[t], c[i]) - c[i];
  }
  __syncthreads();
  int32_t e = inc - tot;
  for (int i = 0; i < (int)(threadIdx.x >> 6); i++) e += wsum[i];
  for (int i = 0; i < DV; i++) {
    const int32_t d = threadIdx.x * DV + i;
    if (d < nd) lst[d] = e;
    e += c[i];
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < U; u++)
    if (threadIdx.x + TH * u < cn) {
      sd[u] = lst[sd[u] >> 16] + (sd[u] & 0xFFFF);  // its slot
      ex[sd[u]] = v[u];
    }
  for (int i = 0; i < DV; i++) {
    const int32_t d = threadIdx.x * DV + i;
    if (d < nd) gb[d] = place[i] - lst[d];
  }
  __syncthreads();
  int32_t dst[U];
#pragma unroll
  for (int u = 0; u < U; u++) {
    const int32_t i = threadIdx.x + TH * u;
    if (i < cn) {
      const float4 r = ex[i];
      const int32_t blk = block_of(r, nx);
      dst[u] = gb[(blk >> shift) & (nd - 1)] + i;
      sout[dst[u]] = r;
      if (kout) kout[dst[u]] = (uint16_t)blk;
    }
  }
  if (lout) {
    __syncthreads();
#pragma unroll
    for (int u = 0; u < U; u++)
      if (threadIdx.x + TH * u < cn) exi[sd[u]] = ll[u];
    __syncthreads();
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int32_t i = threadIdx.x + TH * u;
      if (i < cn) lout[dst[u]] = exi[i];
    }
  }
}

// Dense cells (at least DENSE records) are reordered after the sort; those
// of at most SUB_REG records fit the registers of one workgroup.
constexpr int DENSE = 64;
// cells of at most SUB_REG records are sorted in registers, SUB_V records
// per thread: one wave per cell up to SUB_W records, SUB_T threads above
constexpr int SUB_V = 8, SUB_T = 512, SUB_REG = SUB_T * SUB_V,
              SUB_W = 64 * SUB_V;

// Groups of 2^g blocks into cell order, one workgroup per group: a counting
// sort of its records by cell, the final records and the group's cell
// offsets.  A group of at most CF_CAP records is read once into registers,
// placed in LDS in cell order and written out as one contiguous run; a
// larger one is cut into tiles for the k_cs_big launches.  Groups of 4
// blocks (2048 cells) keep two workgroups per CU, and save the radix pass
// that sorting down to single blocks takes at 1024^3.
constexpr int CF_T = 512, CF_U = 6, CF_CAP = CF_T * CF_U;
constexpr int CF_G = 2;                  // log2 of the blocks of a group, at most
constexpr int CF_CELLS = BS3 << CF_G;
constexpr int CB_T = 1024, CB_U = 8, CB_TILE = CB_T * CB_U;

// a record from a raw element, and its cell inside its group
__device__ inline int32_t group_cell(const float4 &v, int32_t nx, int g,
                                     float4 *r) {
  const PartCell p = part_cell3(v.x, v.y, v.z, nx);
  r->x = p.xs - (float)(p.cx & ~7);
  r->y = p.ys - (float)(p.cy & ~7);
  r->z = p.zs - (float)(p.cz & ~7);
  r->w = v.w;
  return ((p.blk & ((1 << g) - 1)) << 9) | ((p.cz & 7) << 6) |
         ((p.cy & 7) << 3) | (p.cx & 7);
}

// Cell offsets of a group from its counts cnt[0..512 << g) in LDS: cnt
// becomes the exclusive scan, and the dense cells go to their lists by size
// (one atomic per wave and list).  All CF_T threads.
__device__ inline void group_cells(int32_t *cnt, int32_t *wsum, int g,
                                   int64_t cell0, int32_t *__restrict__ dlist,
                                   int32_t *__restrict__ dmid,
                                   int32_t *__restrict__ dbig,
                                   int32_t *__restrict__ dcnt, int32_t dcap) {
  const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
  constexpr int V = 1 << CF_G;
  const int nv = 1 << g;
  int32_t v[V], s = 0;
  int nr = 0, nm = 0, ng = 0;  // this lane's dense cells, by list
#pragma unroll
  for (int k = 0; k < V; k++) {
    v[k] = k < nv ? cnt[threadIdx.x * nv + k] : 0;
    s += v[k];
    nr += v[k] >= DENSE && v[k] <= SUB_W;
    nm += v[k] > SUB_W && v[k] <= SUB_REG;
    ng += v[k] > SUB_REG;
  }
  const int32_t inc = wave_incl_scan(s);
  if (l == 63) wsum[w] = inc;
  __syncthreads();
  int32_t e = inc - s;
  for (int i = 0; i < w; i++) e += wsum[i];
#pragma unroll
  for (int k = 0; k < V; k++)
    if (k < nv) {
      cnt[threadIdx.x * nv + k] = e;
      e += v[k];
    }
  if (__ballot(nr + nm + ng > 0)) {  // uniform per wave
    const int32_t ir = wave_incl_scan(nr), im = wave_incl_scan(nm),
                  ig = wave_incl_scan(ng);
    const int32_t tr = __shfl(ir, 63, 64), tm = __shfl(im, 63, 64),
                  tg = __shfl(ig, 63, 64);
    int32_t br = 0, bm = 0, bg = 0;
    if (l == 0) {
      if (tr > 0) br = atomicAdd(&dcnt[0], tr);
      if (tg > 0) bg = atomicAdd(&dcnt[2], tg);
      if (tm > 0) bm = atomicAdd(&dcnt[4], tm);
    }
    br = __shfl(br, 0, 64) + ir - nr;
    bm = __shfl(bm, 0, 64) + im - nm;
    bg = __shfl(bg, 0, 64) + ig - ng;
#pragma unroll
    for (int k = 0; k < V; k++) {
      const int32_t cell = (int32_t)(cell0 + threadIdx.x * nv + k);
      if (v[k] >= DENSE && v[k] <= SUB_W) {
        if (br < dcap) dlist[br] = cell;
        br++;
      } else if (v[k] > SUB_W && v[k] <= SUB_REG) {
        if (bm < dcap) dmid[bm] = cell;
        bm++;
      } else if (v[k] > SUB_REG) {
        if (bg < dcap) dbig[bg] = cell;
        bg++;
      }
    }
  }
  __syncthreads();
}

// dcnt[6]: large groups, dcnt[7]: their tiles; biggrp[s]: the s-th large
// group, bigcnt[s * CF_CELLS ..]: its cell counts (cleared here), tiles[t] =
// (s, first element).
__global__ void __launch_bounds__(CF_T)
k_cs_final(const int32_t *__restrict__ gs, int64_t ngrp, int g, int32_t nx,
           int64_t npart, const float4 *__restrict__ stage,
           const int32_t *__restrict__ stage_lab,
           int32_t *__restrict__ cell_start, float4 *__restrict__ rec,
           int32_t *__restrict__ perm, int32_t *__restrict__ lab_sorted,
           int32_t *__restrict__ dlist, int32_t *__restrict__ dmid,
           int32_t *__restrict__ dbig, int32_t *__restrict__ dcnt,
           int32_t dcap, int32_t *__restrict__ biggrp,
           int32_t *__restrict__ bigcnt, int2 *__restrict__ tiles) {
  __shared__ int32_t cnt[CF_CELLS];
  __shared__ float4 sr[CF_CAP];
  __shared__ int32_t sl[CF_CAP];
  __shared__ int32_t wsum[CF_T / 64], bslot, btile;
  const int32_t ncell = BS3 << g;
  // A group's records are requested one group ahead (while the group before
  // is placed), and group ranges two ahead, so that the loads of a group
  // are not waited for one after the other.
  auto load = [&](int32_t a, int32_t n, float4 *rr, int32_t *ll) {
    if (n > CF_CAP) return;
#pragma unroll
    for (int k = 0; k < CF_U; k++) {
      const int32_t t = threadIdx.x + CF_T * k;
      if (t < n) {
        const float4 v = stage[a + t];
        rr[k].x = v.x;
        rr[k].y = v.y;
        rr[k].z = v.z;
        rr[k].w = v.w;
        ll[k] = stage_lab ? stage_lab[a + t] : 0;
      }
    }
  };
  if (blockIdx.x == 0 && threadIdx.x == 0)
    cell_start[ngrp * ncell] = (int32_t)npart;
  const int64_t G = gridDim.x;
  int64_t b = blockIdx.x;
  int32_t a = 0, n = 0, an = 0, nn = 0;
  if (b < ngrp) {
    a = gs[b];
    n = gs[b + 1] - a;
  }
  if (b + G < ngrp) {
    an = gs[b + G];
    nn = gs[b + G + 1] - an;
  }
  float4 rr[CF_U];
  int32_t ll[CF_U];
  load(a, n, rr, ll);
  for (; b < ngrp; b += G) {
    float4 rn[CF_U];
    int32_t ln[CF_U];
    load(an, nn, rn, ln);
    int32_t a2 = 0, n2 = 0;
    if (b + 2 * G < ngrp) {
      a2 = gs[b + 2 * G];
      n2 = gs[b + 2 * G + 1] - a2;
    }
    if (n > CF_CAP) {
      const int32_t nt = (n + CB_TILE - 1) / CB_TILE;
      if (threadIdx.x == 0) {
        bslot = atomicAdd(&dcnt[6], 1);
        btile = atomicAdd(&dcnt[7], nt);
        biggrp[bslot] = (int32_t)b;
      }
      __syncthreads();
      for (int i = threadIdx.x; i < ncell; i += CF_T)
        bigcnt[(int64_t)bslot * CF_CELLS + i] = 0;
      for (int32_t t = threadIdx.x; t < nt; t += CF_T)
        tiles[btile + t] = make_int2(bslot, a + t * CB_TILE);
      __syncthreads();
    } else {
      for (int i = threadIdx.x; i < ncell; i += CF_T) cnt[i] = 0;
      __syncthreads();
      int32_t dd[CF_U];  // cell << 16 | rank
#pragma unroll
      for (int k = 0; k < CF_U; k++)
        if (threadIdx.x + CF_T * k < n) {
          float4 r;
          const int32_t c = group_cell(rr[k], nx, g, &r);
          rr[k].x = r.x;
          rr[k].y = r.y;
          rr[k].z = r.z;
          dd[k] = (c << 16) | atomicAdd(&cnt[c], 1);
        }
      __syncthreads();
      group_cells(cnt, wsum, g, b * ncell, dlist, dmid, dbig, dcnt, dcap);
#pragma unroll
      for (int k = 0; k < CF_U; k++)
        if (threadIdx.x + CF_T * k < n) {
          const int32_t p = cnt[dd[k] >> 16] + (dd[k] & 0xFFFF);
          sr[p] = rr[k];
          sl[p] = ll[k];
        }
      for (int i = threadIdx.x; i < ncell; i += CF_T)
        cell_start[b * ncell + i] = a + cnt[i];
      __syncthreads();
      for (int32_t t = threadIdx.x; t < n; t += CF_T) {
        const float4 r = sr[t];
        rec[a + t] = r;
        if (perm) perm[a + t] = __float_as_int(r.w);
        if (lab_sorted) lab_sorted[a + t] = sl[t];
      }
      __syncthreads();
    }
    a = an;
    n = nn;
    an = a2;
    nn = n2;
#pragma unroll
    for (int k = 0; k < CF_U; k++) {
      rr[k] = rn[k];
      ll[k] = ln[k];
    }
  }
}

// Large groups, CB_TILE elements per step of a workgroup: cell counts, the
// group's offsets (one workgroup per group), then the records to their
// cells, each tile taking its places of a cell at once.  Groups share no
// workgroup, so a halo core of 10^5 and more records is spread over the
// GPU.
__global__ void __launch_bounds__(CB_T)
k_cs_big_count(const int32_t *__restrict__ gs, int g, int32_t nx,
               const float4 *__restrict__ stage,
               const int32_t *__restrict__ dcnt,
               const int32_t *__restrict__ biggrp,
               int32_t *__restrict__ bigcnt, const int2 *__restrict__ tiles) {
  __shared__ int32_t cnt[CF_CELLS];
  const int32_t nt = dcnt[7], ncell = BS3 << g;
  for (int32_t t = blockIdx.x; t < nt; t += gridDim.x) {
    const int2 tl = tiles[t];
    const int32_t m = min(gs[biggrp[tl.x] + 1] - tl.y, CB_TILE);
    for (int i = threadIdx.x; i < ncell; i += CB_T) cnt[i] = 0;
    __syncthreads();
    float4 v[CB_U];
#pragma unroll
    for (int k = 0; k < CB_U; k++) {
      const int32_t i = threadIdx.x + CB_T * k;
      if (i < m) v[k] = stage[tl.y + i];
    }
#pragma unroll
    for (int k = 0; k < CB_U; k++)
      if (threadIdx.x + CB_T * k < m) {
        float4 r;
        atomicAdd(&cnt[group_cell(v[k], nx, g, &r)], 1);
      }
    __syncthreads();
    for (int i = threadIdx.x; i < ncell; i += CB_T)
      if (cnt[i]) atomicAdd(&bigcnt[(int64_t)tl.x * CF_CELLS + i], cnt[i]);
    __syncthreads();
  }
}

__global__ void __launch_bounds__(CF_T)
k_cs_big_cells(const int32_t *__restrict__ gs, int g,
               int32_t *__restrict__ cell_start, int32_t *__restrict__ dlist,
               int32_t *__restrict__ dmid, int32_t *__restrict__ dbig,
               int32_t *__restrict__ dcnt, int32_t dcap,
               const int32_t *__restrict__ biggrp,
               int32_t *__restrict__ bigcnt) {
  __shared__ int32_t cnt[CF_CELLS];
  __shared__ int32_t wsum[CF_T / 64];
  const int32_t nb = dcnt[6], ncell = BS3 << g;
  for (int32_t s = blockIdx.x; s < nb; s += gridDim.x) {
    int32_t *bc = bigcnt + (int64_t)s * CF_CELLS;
    for (int i = threadIdx.x; i < ncell; i += CF_T) cnt[i] = bc[i];
    __syncthreads();
    const int64_t b = biggrp[s];
    const int32_t a = gs[b];
    group_cells(cnt, wsum, g, b * ncell, dlist, dmid, dbig, dcnt, dcap);
    for (int i = threadIdx.x; i < ncell; i += CF_T) {
      cell_start[b * ncell + i] = a + cnt[i];
      bc[i] = a + cnt[i];  // next free place of the cell
    }
    __syncthreads();
  }
}

__global__ void __launch_bounds__(CB_T)
k_cs_big_place(const int32_t *__restrict__ gs, int g, int32_t nx,
               const float4 *__restrict__ stage,
               const int32_t *__restrict__ stage_lab,
               const int32_t *__restrict__ dcnt,
               const int32_t *__restrict__ biggrp,
               int32_t *__restrict__ bigcnt, const int2 *__restrict__ tiles,
               float4 *__restrict__ rec, int32_t *__restrict__ perm,
               int32_t *__restrict__ lab_sorted) {
  __shared__ int32_t cnt[CF_CELLS];
  const int32_t nt = dcnt[7], ncell = BS3 << g;
  for (int32_t t = blockIdx.x; t < nt; t += gridDim.x) {
    const int2 tl = tiles[t];
    const int32_t m = min(gs[biggrp[tl.x] + 1] - tl.y, CB_TILE);
    for (int i = threadIdx.x; i < ncell; i += CB_T) cnt[i] = 0;
    __syncthreads();
    float4 v[CB_U];
    int32_t lv[CB_U], dd[CB_U];
#pragma unroll
    for (int k = 0; k < CB_U; k++) {
      const int32_t i = threadIdx.x + CB_T * k;
      if (i < m) {
        const float4 r = stage[tl.y + i];
        v[k].x = r.x;
        v[k].y = r.y;
        v[k].z = r.z;
        v[k].w = r.w;
        lv[k] = stage_lab ? stage_lab[tl.y + i] : 0;
      }
    }
#pragma unroll
    for (int k = 0; k < CB_U; k++)
      if (threadIdx.x + CB_T * k < m) {
        float4 r;
        const int32_t c = group_cell(v[k], nx, g, &r);
        v[k].x = r.x;
        v[k].y = r.y;
        v[k].z = r.z;
        dd[k] = (c << 16) | atomicAdd(&cnt[c], 1);
      }
    __syncthreads();
    for (int i = threadIdx.x; i < ncell; i += CB_T)
      if (cnt[i])
        cnt[i] = atomicAdd(&bigcnt[(int64_t)tl.x * CF_CELLS + i], cnt[i]);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < CB_U; k++)
      if (threadIdx.x + CB_T * k < m) {
        const int32_t d = cnt[dd[k] >> 16] + (dd[k] & 0xFFFF);
        rec[d] = v[k];
        if (perm) perm[d] = __float_as_int(v[k].w);
        if (lab_sorted) lab_sorted[d] = lv[k];
      }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// Dense cells (>= 64 particles) are reordered by the Morton key of the
// particle's 1/8-cell sub-cell, so that any 64 consecutive particles of a
// dense cell occupy a compact box.  The order inside a cell carries no
// meaning elsewhere; the centre search uses the compact chunks to skip
// neighbour chunks beyond its 1-cell reach.
// ---------------------------------------------------------------------------
constexpr int64_t SUB_TMP = 1 << 18;  // records per workgroup slice

__device__ inline uint32_t spread3(uint32_t v) {
  return (v & 1) | ((v & 2) << 2) | ((v & 4) << 4);
}
__device__ inline uint32_t morton9(const float4 &r) {
  const uint32_t qx = (uint32_t)((r.x - floorf(r.x)) * 8.0f) & 7;
  const uint32_t qy = (uint32_t)((r.y - floorf(r.y)) * 8.0f) & 7;
  const uint32_t qz = (uint32_t)((r.z - floorf(r.z)) * 8.0f) & 7;
  return spread3(qx) | (spread3(qy) << 1) | (spread3(qz) << 2);
}

// Cells of at most T * SUB_V records (BIG false): the records read once into
// registers (SUB_V per thread) and placed in place; one wave per cell up to
// SUB_W records, SUB_T threads up to SUB_REG (8 records per thread keep the
// registers to a quarter of the file: 16 took all of it).  Larger cells (BIG true):
// SUB_TB threads, staged through the workgroup's slice, each pass issuing a
// thread's SUB_U records before using them (that launch: 0.88 -> 0.42 ms at
// 1024^3).  A cell's steps are serial round trips to memory, so the
// launches over the many small cells are bound by the cells in flight: one
// 256-thread workgroup per cell of up to 4096 records took 5.7 ms.
constexpr int SUB_TB = 1024, SUB_U = 4;

template <int T, bool BIG>
__global__ void __launch_bounds__(T)
k_subsort(const int32_t *__restrict__ cs, const int32_t *__restrict__ list,
          const int32_t *__restrict__ nlist, int32_t cap,
          int32_t *__restrict__ queue,
          float4 *__restrict__ rec, int32_t *__restrict__ perm,
          int32_t *__restrict__ lab, float4 *__restrict__ trec,
          int32_t *__restrict__ tperm, int32_t *__restrict__ tlab,
          int64_t tcap) {
  __shared__ int32_t hist[512];
  __shared__ int32_t item;
  const int32_t nl = min(*nlist, cap);
  float4 *tr = BIG ? trec + (int64_t)blockIdx.x * tcap : nullptr;
  int32_t *tp = BIG && tperm ? tperm + (int64_t)blockIdx.x * tcap : nullptr;
  int32_t *tl = BIG && tlab ? tlab + (int64_t)blockIdx.x * tcap : nullptr;
  // Cells are taken several at a time where there are many: one counter is
  // shared by every workgroup of the launch, hundreds of thousands of small
  // cells at 1024^3.  Where there are few, 16 at a time left them to a few
  // workgroups in turn (2^21 particles: 73 -> 48 us and, above SUB_W
  // records, 51 -> 9 us).
  const int32_t SUB_B =
      BIG ? 1 : min(16, max(1, nl / (int32_t)(2 * gridDim.x)));
  int32_t it = 0, end = 0;
  for (;;) {
    if (it == end) {
      if (threadIdx.x == 0) item = atomicAdd(queue, SUB_B);
      __syncthreads();
      it = item;
      end = it + SUB_B;
      __syncthreads();
    }
    for (int i = threadIdx.x; i < 512; i += T) hist[i] = 0;
    __syncthreads();
    if (it >= nl) break;
    const int32_t c = list[it++];
    const int32_t a = cs[c], n = cs[c + 1] - a;
    if (BIG ? n > tcap : n > T * SUB_V) {
      // would not fit: keep the scatter order
      __syncthreads();
      continue;
    }
    // the register path reads its records here, once
    float4 rr[BIG ? 1 : SUB_V];
    int32_t pp[BIG ? 1 : SUB_V], ll[BIG ? 1 : SUB_V];
    if constexpr (BIG) {
      for (int32_t t0 = threadIdx.x; t0 < n; t0 += T * SUB_U) {
        float4 r[SUB_U];
#pragma unroll
        for (int k = 0; k < SUB_U; k++)
          if (t0 + k * T < n) r[k] = rec[a + t0 + k * T];
#pragma unroll
        for (int k = 0; k < SUB_U; k++)
          if (t0 + k * T < n) atomicAdd(&hist[morton9(r[k])], 1);
      }
    } else {
#pragma unroll
      for (int k = 0; k < SUB_V; k++) {
        const int32_t t = threadIdx.x + k * T;
        if (t < n) {
          rr[k] = rec[a + t];
          pp[k] = perm ? perm[a + t] : 0;
          ll[k] = lab ? lab[a + t] : 0;
        }
      }
#pragma unroll
      for (int k = 0; k < SUB_V; k++)
        if (threadIdx.x + k * T < n) atomicAdd(&hist[morton9(rr[k])], 1);
    }
    __syncthreads();
    if (threadIdx.x < 64) {  // exclusive scan of 512 counters by one wave
      int32_t v[8], s = 0;
      for (int k = 0; k < 8; k++) { v[k] = hist[threadIdx.x * 8 + k]; s += v[k]; }
      const int32_t inc = wave_incl_scan(s);
      int32_t e = inc - s;
      for (int k = 0; k < 8; k++) { hist[threadIdx.x * 8 + k] = e; e += v[k]; }
    }
    __syncthreads();
    if constexpr (!BIG) {
      // in place: everything was read into registers before any write
      int32_t dd[SUB_V];
#pragma unroll
      for (int k = 0; k < SUB_V; k++)
        if (threadIdx.x + k * T < n) dd[k] = atomicAdd(&hist[morton9(rr[k])], 1);
      __syncthreads();
#pragma unroll
      for (int k = 0; k < SUB_V; k++) {
        const int32_t t = threadIdx.x + k * T;
        if (t < n) {
          rec[a + dd[k]] = rr[k];
          if (perm) perm[a + dd[k]] = pp[k];
          if (lab) lab[a + dd[k]] = ll[k];
        }
      }
    } else {
      for (int32_t t0 = threadIdx.x; t0 < n; t0 += T * SUB_U) {
        float4 r[SUB_U];
        int32_t pv[SUB_U], lv[SUB_U];
#pragma unroll
        for (int k = 0; k < SUB_U; k++) {
          const int32_t t = t0 + k * T;
          if (t < n) {
            r[k] = rec[a + t];
            pv[k] = perm ? perm[a + t] : 0;
            lv[k] = lab ? lab[a + t] : 0;
          }
        }
#pragma unroll
        for (int k = 0; k < SUB_U; k++) {
          if (t0 + k * T < n) {
            const int32_t d = atomicAdd(&hist[morton9(r[k])], 1);
            tr[d] = r[k];
            if (perm) tp[d] = pv[k];
            if (lab) tl[d] = lv[k];
          }
        }
      }
      __threadfence_block();
      __syncthreads();
      for (int32_t t0 = threadIdx.x; t0 < n; t0 += T * SUB_U) {
        float4 r[SUB_U];
        int32_t pv[SUB_U], lv[SUB_U];
#pragma unroll
        for (int k = 0; k < SUB_U; k++) {
          const int32_t t = t0 + k * T;
          if (t < n) {
            r[k] = tr[t];
            pv[k] = perm ? tp[t] : 0;
            lv[k] = lab ? tl[t] : 0;
          }
        }
#pragma unroll
        for (int k = 0; k < SUB_U; k++) {
          const int32_t t = t0 + k * T;
          if (t < n) {
            rec[a + t] = r[k];
            if (perm) perm[a + t] = pv[k];
            if (lab) lab[a + t] = lv[k];
          }
        }
      }
    }
    __syncthreads();
  }
}

extern "C" int psod_cell_sort(psod_ctx *ctx, int64_t npart, const float *d_pos,
                              const int32_t *d_labels, int32_t nx,
                              int32_t *d_cell_start, int32_t *d_perm,
                              float *d_rec, int32_t *d_lab_sorted) {
  PSOD_TRY(psod_check_npart("psod_cell_sort", npart));
  PSOD_TRY(psod_use_device(ctx));
  if (npart < 0 || !d_pos || !d_cell_start || !d_rec)
    return psod_set_error(PSOD_E_ARG, "psod_cell_sort: bad arguments");
  if (nx < 8 || nx > 1024 || (nx & (nx - 1)))
    return psod_set_error(PSOD_E_ARG,
                          "psod_cell_sort: nx=%d must be a power of two in "
                          "[8, 1024]", nx);
  const int64_t ncell = (int64_t)nx * nx * nx;
  const int64_t nblk = ncell / BS3;
  hipStream_t st = ctx->stream;
  const int64_t n = npart;
  int bits = 0;
  while ((int64_t)1 << bits < nblk) bits++;
  // Groups of 2^g blocks for the last step: as many as hold about 2/3 of
  // CF_CAP records at the mean density, at most 4 blocks.
  int g = std::min(CF_G, bits);
  while (g > 0 && n > (int64_t)(CF_CAP / 3 * 2) * (nblk >> g)) g--;
  const int gbits = bits - g;  // bits of the group, sorted in at most 2 passes
  const int64_t ngrp = nblk >> g;
  const int db1 = gbits <= CS_DB ? gbits : gbits / 2, db2 = gbits - db1;
  const int32_t nd1 = 1 << db1, nd2 = 1 << db2;
  // Chunks of 8192 elements in the first pass (runs of 16 at 1024^3; with
  // chunks of 4096: 11.7 against 10.4 ms there, and 13.5 with 10 bits in it)
  // and of 4096, two workgroups per CU, in the second; of 1024 where those
  // would leave CUs without work (2^21 particles: chunks of 8192 25 us, of
  // 1024 58 us, whose 1024 counters per chunk then cost more than the copy).
  const bool small = n < (int64_t)ctx->num_cus * 4096;
  const int32_t ch1 = small ? 1024 : 8192, ch = small ? 1024 : 4096;
  const int64_t nch1 = (n + ch1 - 1) / ch1, nch2 = (n + ch - 1) / ch + nd1;
  // counts of both passes, cleared together; starts; chunk tables
  const int64_t nh1 = (int64_t)nd1 * CS_XCD, nh2 = db2 > 0 ? ngrp + 1 : 0;
  int32_t *hb = (int32_t *)psod_scratch(
      ctx, S_CS_H, (size_t)(2 * nh1 + 2 * nh2 + 2 * (nd1 + 64) + nch2 + 256) * 4);
  float4 *sa = (float4 *)psod_scratch(ctx, S_CS_A, (size_t)(n > 0 ? n : 1) * 22 + 64);
  float4 *sc = nullptr;
  if (db2 > 0)
    sc = (float4 *)psod_scratch(ctx, S_CS_C, (size_t)(n > 0 ? n : 1) * 20);
  if (!hb || !sa || (db2 > 0 && !sc)) return PSOD_E_NOMEM;
  int32_t *H1 = hb, *H2 = H1 + nh1, *S1 = H2 + nh2, *S2 = S1 + nh1,
          *bs = S2 + nh2, *cb = bs + nd1 + 64, *cmap = cb + nd1 + 64;
  int32_t *la = d_lab_sorted ? (int32_t *)(sa + n) : nullptr;
  // 16-byte aligned, with room for the last word of 8
  uint16_t *key = (uint16_t *)(((uintptr_t)((int32_t *)(sa + n) + n) + 15) &
                               ~(uintptr_t)15);
  PSOD_TRY(psod_fill_i32(ctx, H1, nh1 + nh2, 0));
  const int sh1 = bits - db1;
  const float4 *stage = sa;
  const int32_t *slab = la;
  const int32_t *gs = bs;  // ngrp + 1 group starts
  if (n > 0) {
    // a multiple of 8 workgroups, each with chunks of one class; few enough
    // that a workgroup counts at least 8 elements per digit that it adds
    // (2^21 particles, 1024 digits: 38 -> 18 us)
    const int64_t want = std::min<int64_t>(
        std::min<int64_t>(nch1, n / (8 * nd1) + 1), (int64_t)ctx->num_cus * 8);
    const unsigned nw1 = (unsigned)((want + CS_XCD - 1) / CS_XCD * CS_XCD);
    if (small)
      k_cs_hist1<1024><<<nw1, 256, 0, st>>>(d_pos, n, nx, sh1, db1, H1);
    else
      k_cs_hist1<8192><<<nw1, 256, 0, st>>>(d_pos, n, nx, sh1, db1, H1);
    PSOD_LAUNCH_CHECK();
  }
  k_cs_starts<<<1, 1024, 0, st>>>(H1, nd1, (int32_t)n, ch, S1, bs,
                                  db2 > 0 ? cb : nullptr, cmap);
  PSOD_LAUNCH_CHECK();
  if (n > 0) {
    uint16_t *ko = db2 > 0 ? key : nullptr;
    if (small)
      k_cs_scatter<true, 1024, 256><<<(unsigned)nch1, 256, 0, st>>>(
          d_pos, nullptr, d_labels, n, nx, sh1, db1, nullptr, 0, nullptr,
          nullptr, S1, H1, sa, la, ko);
    else
      k_cs_scatter<true, 8192, 1024><<<(unsigned)nch1, 1024, 0, st>>>(
          d_pos, nullptr, d_labels, n, nx, sh1, db1, nullptr, 0, nullptr,
          nullptr, S1, H1, sa, la, ko);
    PSOD_LAUNCH_CHECK();
  }
  if (db2 > 0) {
    const int sh2 = g;
    if (n > 0) {
      const int32_t per = (int32_t)std::max<int64_t>(
          1, nch2 / ((int64_t)ctx->num_cus * 8));
      k_cs_hist2<<<(unsigned)((nch2 + per - 1) / per), 256, 0, st>>>(
          key, sh2, db2, bs, nd1, cb, cmap, ch, per, H2);
      PSOD_LAUNCH_CHECK();
    }
    PSOD_TRY(psod_scan_i32(ctx, H2, S2, ngrp + 1, nullptr));
    if (n > 0) {
      int32_t *lc = d_lab_sorted ? (int32_t *)(sc + n) : nullptr;
      const unsigned nw2 = (unsigned)((nch2 + CS_XCD - 1) / CS_XCD * CS_XCD);
      if (small)
        k_cs_scatter<false, 1024, 256><<<nw2, 256, 0, st>>>(
            nullptr, sa, la, n, nx, sh2, db2, bs, nd1, cb, cmap, S2, H2, sc,
            lc, nullptr);
      else
        k_cs_scatter<false, 4096, 512><<<nw2, 512, 0, st>>>(
            nullptr, sa, la, n, nx, sh2, db2, bs, nd1, cb, cmap, S2, H2, sc,
            lc, nullptr);
      PSOD_LAUNCH_CHECK();
      stage = sc;
      slab = lc;
    }
    gs = S2;
  }
  // lists of the dense cells by size, filled with the cell offsets: ctl[0],
  // ctl[4] and ctl[2] count them (up to SUB_W, up to SUB_REG, larger
  // records), ctl[1], ctl[5] and ctl[3] are the subsort's queues (at most
  // npart / DENSE cells are dense); then the groups of more than CF_CAP
  // records (ctl[6]), their tiles (ctl[7]) and their cell counts
  const int32_t cap = (int32_t)std::min<int64_t>(ncell, npart / DENSE + 32);
  const int64_t bgcap = std::min<int64_t>(ngrp, n / CF_CAP + 1);
  const int64_t btcap = n / CB_TILE + bgcap + 1;
  int32_t *list = (int32_t *)psod_scratch(
      ctx, S_HIST, (size_t)(3 * (int64_t)cap + 128 + bgcap * (CF_CELLS + 1) +
                            2 * btcap + 64) * 4);
  int32_t *ctl = (int32_t *)psod_scratch(ctx, S_MISC, 64);
  if (!list || !ctl) return PSOD_E_NOMEM;
  int32_t *big = list + cap + 32;
  int32_t *mid = big + cap + 32;
  int2 *tiles = (int2 *)(((uintptr_t)(mid + cap + 32) + 15) & ~(uintptr_t)15);
  int32_t *biggrp = (int32_t *)(tiles + btcap), *bigcnt = biggrp + bgcap;
  PSOD_TRY(psod_fill_i32(ctx, ctl, 8, 0));
  k_cs_final<<<grid_for(ngrp, 1, (int64_t)ctx->num_cus * 4), CF_T, 0, st>>>(
      gs, ngrp, g, nx, npart, stage, slab, d_cell_start, (float4 *)d_rec,
      d_perm, d_lab_sorted, list, mid, big, ctl, cap, biggrp, bigcnt, tiles);
  PSOD_LAUNCH_CHECK();
  if (n > CF_CAP) {
    const unsigned nbw = grid_for(btcap, 1, ctx->num_cus * 2);
    k_cs_big_count<<<nbw, CB_T, 0, st>>>(gs, g, nx, stage, ctl, biggrp, bigcnt,
                                         tiles);
    PSOD_LAUNCH_CHECK();
    k_cs_big_cells<<<grid_for(bgcap, 1, ctx->num_cus * 4), CF_T, 0, st>>>(
        gs, g, d_cell_start, list, mid, big, ctl, cap, biggrp, bigcnt);
    PSOD_LAUNCH_CHECK();
    k_cs_big_place<<<nbw, CB_T, 0, st>>>(gs, g, nx, stage, slab, ctl, biggrp,
                                         bigcnt, tiles, (float4 *)d_rec,
                                         d_perm, d_lab_sorted);
    PSOD_LAUNCH_CHECK();
  }
  if (npart > 0) {
    // Morton order of the 1/8-cell sub-cells inside dense cells
    // cells that fit the registers: one wave per cell up to SUB_W records,
    // SUB_T threads up to SUB_REG, no staging slices; larger cells: one
    // workgroup per CU, each with a staging slice
    k_subsort<64, false><<<(unsigned)ctx->num_cus * 12, 64, 0, st>>>(
        d_cell_start, list, ctl, cap, ctl + 1, (float4 *)d_rec, d_perm,
        d_lab_sorted, nullptr, nullptr, nullptr, 0);
    PSOD_LAUNCH_CHECK();
    k_subsort<SUB_T, false><<<(unsigned)ctx->num_cus * 2, SUB_T, 0, st>>>(
        d_cell_start, mid, ctl + 4, cap, ctl + 5, (float4 *)d_rec, d_perm,
        d_lab_sorted, nullptr, nullptr, nullptr, 0);
    PSOD_LAUNCH_CHECK();
    // cells above SUB_REG records: at most npart / SUB_REG of them, each
    // staged in a slice of at most min(SUB_TMP, npart) records
    const int64_t tcap = std::min<int64_t>(SUB_TMP, npart);
    const unsigned nsub = (unsigned)std::min<int64_t>(ctx->num_cus,
                                                      npart / SUB_REG + 1);
    char *tmp = (char *)psod_scratch(ctx, S_KEYS, (size_t)nsub * tcap * 24);
    if (!tmp) return PSOD_E_NOMEM;
    k_subsort<SUB_TB, true><<<nsub, SUB_TB, 0, st>>>(
        d_cell_start, big, ctl + 2, cap, ctl + 3, (float4 *)d_rec, d_perm,
        d_lab_sorted, (float4 *)tmp, (int32_t *)(tmp + (size_t)nsub * tcap * 16),
        (int32_t *)(tmp + (size_t)nsub * tcap * 20), tcap);
    PSOD_LAUNCH_CHECK();
  }
  return psod_finish(ctx);
}
