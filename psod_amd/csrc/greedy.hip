// greedy.hip -- `spherover` (main file:1396-2201) with the reference's
// greedy semantics: seeds in decreasing density, a seed is skipped when an
// earlier sphere captured it, and every grown sphere removes its particles
// (accepted or not) before later seeds gather.
//
// Exact sequential semantics in parallel: seed s only reads and writes the
// (2 ncut + 1)^3 cells around its cell, so two seeds whose cubes do not
// intersect commute.  Each round marks, per small block of cells, the
// earliest unprocessed live seed; a seed runs in this round when no earlier
// unprocessed live seed lies in the blocks within 2 ncut cells of it.
// Rounds repeat until every seed up to npart_new is processed or dead.
// Per-seed arithmetic is FP64 on the float32 positions scaled by nx, as in
// the reference.
//
// A round has few ready seeds (tens on a 128^3 catalogue), and the largest
// of them holds almost all of its work, so a round is a chain of launches
// that each spread one step over the GPU: gather (one workgroup per seed),
// centre search (64 candidates per workgroup), growth (one workgroup per
// seed, keys sorted in LDS).  One workgroup per seed for everything took
// 5.2 ms a round, 290-350 ms for the 66 rounds of the 128^3 catalogue: FP64
// square roots and divisions of every candidate pair on one CU, then a
// bitonic sort of all gathered particles in global memory.  The staged
// rounds, at most 24 there (smaller marking blocks let more seeds run side by
// side), take 7.2 ms with the transfers: 3.3 of it kernels, the rest pageable
// copies and the waits.
//
// A seed that fails ends the zone at its place in the order: the seeds
// before it run on, and where seeds after it had run too, those before it
// run a second time by themselves.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <numeric>
#include <vector>

#include "sod_common.h"

int psod_fill_i32(psod_ctx *c, int32_t *p, int64_t n, int32_t v);

namespace {

constexpr int64_t GCAP = 1 << 18;  // gathered particles per seed, at most
// particles gathered in one round, at most: a ready seed that does not fit
// waits for the next round (one seed always fits)
constexpr int64_t GPOOL = (int64_t)1 << 25;
constexpr int64_t GWIN = 1 << 16;  // seeds looked at per round
constexpr int GROUNDS = 8;         // rounds queued before the host looks (even)

struct GreedyCfg {
  int32_t nx, ncut, nbins;
  int32_t bsh, nb;  // marking blocks of 2^bsh cells per side, nb per axis
  double seuil, seuil2, mmin, lr0, lr1, rmaxf;
  int64_t nsel;
};

// Progress of the rounds, on the device.  Entries [2] alternate between
// rounds: a round of parity p resets its own entries in k_mark and reads
// the window start that the round before left in first[1 - p].
struct GState {
  unsigned long long fail;       // smallest (seed order << 8 | code), or ~0
  unsigned long long cursor[2];  // pool entries handed out
  int32_t first[2];              // first unprocessed seed order
  int32_t nready[2], nunits[2];
  int32_t total, nrec;           // ready seeds so far, records so far
  int32_t last;                  // largest order of a seed with a record
};
enum { GF_NSEL = 1, GF_GCAP = 2, GF_UNCLOSED = 3 };

// End of the orders still to run, within the window from lo: a failed seed
// ends the zone, but the seeds before it that wait on their neighbours run
// on (one of them may be the first to fail); those after it do not count.
__device__ inline int32_t window_end(const GState *S, int32_t npart_new,
                                     int32_t lo) {
  const int64_t end = (int64_t)min((unsigned long long)npart_new, S->fail >> 8);
  return (int32_t)min(end, lo + GWIN);
}

// One ready seed of a round: its pool entries [off, off + n1), of which the
// first nnear / ncand entries of the near / candidate lists are set; its
// centre-search units [unit0, unit0 + ceil(ncand / 64)); n1 = 0: nothing to
// do this round.
struct GInfo {
  int64_t off;
  int32_t n1, nnear, ncand, unit0;
  unsigned long long best;  // largest lower bound of S, as double bits
};

// Pool arrays, one entry per gathered particle
struct GPoolPtrs {
  float4 *p;       // block-relative position, particle index
  int32_t *slot;   // its place in cell order
  int32_t *cell;   // offset of its cell from the seed cell, 10 bits per axis
  float4 *near;    // within 2 cells: position relative to the seed cell,
                   // place in p
  int32_t *cand;   // within 1 cell: place in near
  double *upper;   // per candidate: bound of its S
  uint64_t *d2;    // squared distance from the centre (double bits)
  uint64_t *key;   // sort area: d2 bits and place in p
  uint32_t *ord;
};

struct GRec {
  int64_t ipart, seed, centre, iamas, masse, masse2;
  double amass, xc, yc, zc, rayon, overdens, overdens2;
  int32_t accepted, pad;
};

__device__ inline int32_t pack_off(int di, int dj, int dk) {
  return (di + 511) | ((dj + 511) << 10) | ((dk + 511) << 20);
}
__device__ inline void unpack_off(int32_t v, int *o) {
  o[0] = (v & 1023) - 511;
  o[1] = ((v >> 10) & 1023) - 511;
  o[2] = (v >> 20) - 511;
}

__global__ void k_inverse_perm(const int32_t *__restrict__ perm, int64_t n,
                               int32_t *__restrict__ slot_of) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n) slot_of[perm[k]] = (int32_t)k;
}

__global__ void k_set_u8(uint8_t *__restrict__ p, int64_t n, uint8_t v) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    p[i] = v;
}

__device__ inline void seed_cell(const float *pos, int32_t s, int32_t nx,
                                 int32_t *cs) {
  for (int d = 0; d < 3; d++) {
    float f;
    split_coord(pos[3 * (int64_t)s + d], nx, &cs[d], &f);
  }
}

// per block: smallest order of an unprocessed live seed of the window
__global__ void __launch_bounds__(256)
k_mark(GreedyCfg c, const int32_t *__restrict__ isort,
       const int32_t *__restrict__ slot_of, const float *__restrict__ pos,
       const uint8_t *__restrict__ alive, const uint8_t *__restrict__ done,
       int32_t npart_new, int par, GState *__restrict__ S,
       int32_t *__restrict__ bmin) {
  const int32_t lo = S->first[1 - par];
  const int32_t hi = window_end(S, npart_new, lo);
  const int64_t o = lo + (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    S->total += S->nready[1 - par];
    S->first[par] = hi;
    S->nready[par] = 0;
    S->nunits[par] = 0;
    S->cursor[par] = 0;
  }
  if (o >= hi || done[o]) return;
  const int32_t s = isort[o] - 1;
  if (!alive[slot_of[s]]) return;
  int32_t b[3];
  seed_cell(pos, s, c.nx, b);
  for (int d = 0; d < 3; d++) b[d] >>= c.bsh;
  atomicMin(&bmin[(b[2] * c.nb + b[1]) * c.nb + b[0]], (int32_t)o);
}

// Ready seeds: live, unprocessed, and no earlier unprocessed live seed in
// the blocks within 2 ncut cells (cubes intersect only if the seed cells
// are at most 2 ncut apart).  Also the first unprocessed seed, the start of
// the next round's window (seeds that run in this round count as
// unprocessed until the next).
__global__ void __launch_bounds__(256)
k_ready(GreedyCfg c, const int32_t *__restrict__ isort,
        const int32_t *__restrict__ slot_of, const float *__restrict__ pos,
        const uint8_t *__restrict__ alive, uint8_t *__restrict__ done,
        int32_t npart_new, int par, GState *__restrict__ S,
        const int32_t *__restrict__ bmin, int32_t *__restrict__ ready) {
  const int32_t lo = S->first[1 - par];
  const int32_t hi = window_end(S, npart_new, lo);
  const int64_t o = lo + (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int32_t open = INT32_MAX;
  bool go = false;
  if (o < hi && !done[o]) {
    const int32_t s = isort[o] - 1;
    if (!alive[slot_of[s]]) {  // captured earlier: nothing to do (:1628)
      done[o] = 1;
    } else {
      open = (int32_t)o;
      go = true;
      int32_t cs[3], b0[3], nb[3];
      seed_cell(pos, s, c.nx, cs);
      for (int d = 0; d < 3; d++) {
        b0[d] = (cs[d] - 2 * c.ncut) >> c.bsh;
        nb[d] = min(((cs[d] + 2 * c.ncut) >> c.bsh) - b0[d] + 1, c.nb);
      }
      for (int i = 0; i < nb[2] && go; i++)
        for (int j = 0; j < nb[1] && go; j++) {
          const int32_t row = (wrapi(b0[2] + i, c.nb) * c.nb +
                               wrapi(b0[1] + j, c.nb)) * c.nb;
          for (int k = 0; k < nb[0]; k++)
            go = go && bmin[row + wrapi(b0[0] + k, c.nb)] >= open;
        }
    }
  }
  const int l = threadIdx.x & 63;
  const uint64_t mo = __ballot(open != INT32_MAX);
  if (mo && l == __ffsll((unsigned long long)mo) - 1)
    atomicMin(&S->first[par], open);  // orders ascend with the lane
  const uint64_t m = __ballot(go);
  int32_t base = 0;
  if (l == 0 && m) base = atomicAdd(&S->nready[par], (int32_t)__popcll(m));
  base = __shfl(base, 0, 64);
  if (go)
    ready[base + __popcll(m & (l == 0 ? 0ull : (~0ull >> (64 - l))))] = open;
}

constexpr int GA_T = 1024;  // threads of a gather workgroup

// exclusive prefix of v over the GA_T threads; *tot the sum
__device__ inline int32_t ga_scan(int32_t v, int32_t *wsum, int32_t *tot) {
  const int w = threadIdx.x >> 6;
  const int32_t inc = wave_incl_scan(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 63) wsum[w] = inc;
  __syncthreads();
  int32_t off = 0, t = 0;
  for (int i = 0; i < GA_T / 64; i++) {
    if (i < w) off += wsum[i];
    t += wsum[i];
  }
  *tot = t;
  return off + inc - v;
}

// S1: live particles of the (2ncut+1)^3 cells of each ready seed in walk
// order, x outermost (main file:1658-1716): the gathered list keeps the
// reference's order, which decides exact ties.  One workgroup per seed: the
// cells' ranges GA_T at a time, their records in flat order (a lane per
// record: a thread per cell walked a dense cell's thousands of records
// alone), ranks from ballots.
__global__ void __launch_bounds__(GA_T)
k_greedy_gather(GreedyCfg c, const int32_t *__restrict__ isort,
                const int32_t *__restrict__ cell_start,
                const float4 *__restrict__ rec, const float *__restrict__ pos,
                const uint8_t *__restrict__ alive, uint8_t *__restrict__ done,
                int par, GState *__restrict__ S,
                const int32_t *__restrict__ ready, GInfo *__restrict__ info,
                int2 *__restrict__ units, GPoolPtrs G, int64_t pcap) {
  __shared__ int32_t pre[GA_T + 1], st[GA_T], wsum[GA_T / 64];
  __shared__ int32_t wc[GA_T / 64][3];
  __shared__ long long soff;
  const int32_t nr = S->nready[par];
  const int side = 2 * c.ncut + 1;
  const int32_t ncell = side * side * side;
  const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
  const uint64_t below = l == 0 ? 0ull : (~0ull >> (64 - l));
  for (int32_t it = blockIdx.x; it < nr; it += gridDim.x) {
    const int32_t o = ready[it];
    int32_t cs[3];
    seed_cell(pos, isort[o] - 1, c.nx, cs);
    // pool entries: every particle of the cells, a power of two (the sort's
    // padding)
    int64_t all = 0;
    for (int32_t base = 0; base < ncell; base += GA_T) {
      const int32_t q = base + threadIdx.x;
      int32_t n = 0, a = 0;
      if (q < ncell) {
        int di, dj, dk;
        int32_t lc[3];
        walk_off(q, c.ncut, &di, &dj, &dk);
        const int32_t key = key_at(c.nx, cs, di, dj, dk, lc);
        a = cell_start[key];
        n = cell_start[key + 1] - a;
      }
      int32_t tot;
      const int32_t ex = ga_scan(n, wsum, &tot);
      pre[threadIdx.x] = ex;  // kept when there is one batch of cells
      st[threadIdx.x] = a;
      if (threadIdx.x == 0) pre[GA_T] = tot;
      all += tot;
    }
    int64_t cap = 64;
    while (cap < all && cap < GCAP) cap <<= 1;
    if (threadIdx.x == 0) {
      const long long off = (long long)atomicAdd(&S->cursor[par],
                                                 (unsigned long long)cap);
      soff = off + cap <= pcap ? off : -1;
    }
    __syncthreads();
    const int64_t off = soff;
    GInfo gi;
    gi.off = off;
    gi.n1 = gi.nnear = gi.ncand = gi.unit0 = 0;
    gi.best = 0;
    if (off < 0) {  // the pool is full: next round
      if (threadIdx.x == 0) info[it] = gi;
      __syncthreads();
      continue;
    }
    int64_t n1 = 0;
    int32_t nnear = 0, ncand = 0;
    for (int32_t base = 0; base < ncell; base += GA_T) {
      if (ncell > GA_T) {
        const int32_t q = base + threadIdx.x;
        int32_t n = 0, a = 0;
        if (q < ncell) {
          int di, dj, dk;
          int32_t lc[3];
          walk_off(q, c.ncut, &di, &dj, &dk);
          const int32_t key = key_at(c.nx, cs, di, dj, dk, lc);
          a = cell_start[key];
          n = cell_start[key + 1] - a;
        }
        int32_t tot;
        const int32_t ex = ga_scan(n, wsum, &tot);
        pre[threadIdx.x] = ex;
        st[threadIdx.x] = a;
        if (threadIdx.x == 0) pre[GA_T] = tot;
      }
      __syncthreads();
      const int32_t tot = pre[GA_T];
      for (int32_t j0 = 0; j0 < tot; j0 += GA_T) {
        const int32_t j = j0 + threadIdx.x;
        bool live = false, near = false, cand = false;
        int di = 0, dj = 0, dk = 0;
        int32_t k = 0;
        if (j < tot) {
          int lo = 0, hi = GA_T;  // last cell with pre <= j (empty cells: the
          while (hi - lo > 1) {   // last of equal entries holds j)
            const int mid = (lo + hi) >> 1;
            if (pre[mid] <= j) lo = mid; else hi = mid;
          }
          k = st[lo] + (j - pre[lo]);
          live = alive[k] != 0;
          walk_off(base + lo, c.ncut, &di, &dj, &dk);
          const int cheb = max(abs(di), max(abs(dj), abs(dk)));
          near = live && cheb <= 2;
          cand = live && cheb <= 1;
        }
        const uint64_t ml = __ballot(live), mn = __ballot(near),
                       mc = __ballot(cand);
        if (l == 0) {
          wc[w][0] = __popcll(ml);
          wc[w][1] = __popcll(mn);
          wc[w][2] = __popcll(mc);
        }
        __syncthreads();
        int32_t t0 = 0, t1 = 0, t2 = 0, e0 = 0, e1 = 0, e2 = 0;
        for (int i = 0; i < GA_T / 64; i++) {
          if (i == w) {
            e0 = t0;
            e1 = t1;
            e2 = t2;
          }
          t0 += wc[i][0];
          t1 += wc[i][1];
          t2 += wc[i][2];
        }
        if (live) {
          const int64_t e = n1 + e0 + __popcll(ml & below);
          if (e < cap && e < c.nsel) {
            const float4 r = rec[k];
            G.p[off + e] = r;
            G.slot[off + e] = k;
            G.cell[off + e] = pack_off(di, dj, dk);
            if (near) {
              const int32_t en = nnear + e1 + __popcll(mn & below);
              G.near[off + en] = make_float4(
                  rel1(r.x, (cs[0] + di) & 7, di, 0.f),
                  rel1(r.y, (cs[1] + dj) & 7, dj, 0.f),
                  rel1(r.z, (cs[2] + dk) & 7, dk, 0.f),
                  __int_as_float((int32_t)e));
              if (cand) G.cand[off + ncand + e2 + __popcll(mc & below)] = en;
            }
          }
        }
        n1 += t0;
        nnear += t1;
        ncand += t2;
        __syncthreads();
      }
    }
    if (threadIdx.x == 0) {
      if (n1 > c.nsel || n1 > GCAP) {  // "Increase Nsel" (main file:1681)
        const int code = n1 > c.nsel ? GF_NSEL : GF_GCAP;
        atomicMin(&S->fail, ((unsigned long long)o << 8) | code);
      } else if (!((double)n1 >= c.mmin)) {
        done[o] = 1;  // Mtotsel >= Mmin with unit masses (main file:1759)
      } else {
        gi.n1 = (int32_t)n1;
        gi.nnear = nnear;
        gi.ncand = ncand;
        const int32_t ng = (ncand + 63) >> 6;
        gi.unit0 = atomicAdd(&S->nunits[par], ng);
        for (int32_t g = 0; g < ng; g++)
          units[gi.unit0 + g] = make_int2(it, g);
      }
      info[it] = gi;
    }
    __syncthreads();
  }
}

// Centre search (main file:1799-1875) in two launches.  The first bounds
// every candidate's S in FP32: relative coordinates and their differences
// are good to 4e-7 cells, so a term 1/sqrt(d2 + 2^-12) is good to 2.3e-5
// and d2 to 3e-6; sums of 64 FP32 terms add at most 4e-6 and are folded in
// FP64.  S lies between (1 - 1e-4) times the terms of d2 <= 1 - 1e-5 and
// (1 + 1e-4) times the terms of d2 <= 1 + 1e-5.  The second launch
// evaluates in FP64 only the candidates whose upper bound reaches the
// largest lower bound (no other can hold or tie the maximum): a few of
// thousands, in place of an FP64 square root and division per pair.
// One workgroup takes 64 candidates, its 8 waves a share of the
// neighbours each.
constexpr int GC_T = 512;

__global__ void __launch_bounds__(GC_T)
k_greedy_bound(int par, GState *__restrict__ S, GInfo *__restrict__ info,
               const int2 *__restrict__ units, GPoolPtrs G) {
  __shared__ float4 tile[GC_T];
  __shared__ double red[GC_T / 64][64][2];
  const int l = threadIdx.x & 63,
            w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int32_t nu = S->nunits[par];
  for (int32_t u = blockIdx.x; u < nu; u += gridDim.x) {
    const int2 un = units[u];
    const GInfo gi = info[un.x];
    const int32_t cd = un.y * 64 + l;
    float4 p = make_float4(1e30f, 1e30f, 1e30f, 0.f);
    if (cd < gi.ncand) p = G.near[gi.off + G.cand[gi.off + cd]];
    double lo = 0.0, up = 0.0;
    for (int32_t b = 0; b < gi.nnear; b += GC_T) {
      __syncthreads();
      const int32_t j = b + (int32_t)threadIdx.x;
      // entries past the end lie beyond every cutoff
      tile[threadIdx.x] = j < gi.nnear ? G.near[gi.off + j]
                                       : make_float4(-1e30f, 0.f, 0.f, 0.f);
      __syncthreads();
      float sl = 0.f, su = 0.f;
#pragma unroll 8
      for (int i = 0; i < 64; i++) {
        const float4 q = tile[64 * w + i];
        const float dx = q.x - p.x, dy = q.y - p.y, dz = q.z - p.z;
        const float d2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
        const float t = __builtin_amdgcn_rsqf(d2 + 1.0f / 4096.0f);
        sl += d2 <= 1.0f - 1e-5f ? t : 0.f;
        su += d2 <= 1.0f + 1e-5f ? t : 0.f;
      }
      lo += (double)sl;
      up += (double)su;
    }
    red[w][l][0] = lo;
    red[w][l][1] = up;
    __syncthreads();
    if (w == 0) {
      for (int i = 1; i < GC_T / 64; i++) {
        lo += red[i][l][0];
        up += red[i][l][1];
      }
      if (cd < gi.ncand) G.upper[gi.off + cd] = up * (1.0 + 1e-4);
      unsigned long long v =
          cd < gi.ncand ? (unsigned long long)__double_as_longlong(
                              lo * (1.0 - 1e-4))
                        : 0ull;
      for (int sh = 32; sh > 0; sh >>= 1) {
        const unsigned long long x = __shfl_xor(v, sh, 64);
        v = x > v ? x : v;
      }
      if (l == 0) atomicMax(&info[un.x].best, v);
    }
    __syncthreads();
  }
}

// position of pool entry e relative to the box origin (FP64)
__device__ inline void entry_pos(const GPoolPtrs &G, int64_t e,
                                 const int32_t *cs, double *x, int *off) {
  const float4 r = G.p[e];
  unpack_off(G.cell[e], off);
  const double u[3] = {(double)r.x, (double)r.y, (double)r.z};
  for (int d = 0; d < 3; d++)
    x[d] = (double)cs[d] + (double)off[d] +
           (u[d] - (double)((cs[d] + off[d]) & 7));
}

// FP64 S of the candidates left, one wave each, terms in parallel and their
// sum in gather order (the reference's); first strict maximum in walk
// order.  ures[u] = best (S bits, key) of unit u, key = walk rank of the
// candidate's cell << 32 | particle index.  Also clears the marks for the
// next round.
__global__ void __launch_bounds__(256)
k_greedy_centre(GreedyCfg c, const int32_t *__restrict__ isort,
                const float *__restrict__ pos, int par,
                const GState *__restrict__ S, const int32_t *__restrict__ ready,
                const GInfo *__restrict__ info, const int2 *__restrict__ units,
                GPoolPtrs G, uint64_t *__restrict__ ures,
                int32_t *__restrict__ bmin, int32_t nbk) {
  __shared__ uint64_t mask;
  __shared__ double term[4][64];
  __shared__ double ws[4];
  __shared__ int64_t wk[4];
  for (int32_t i = blockIdx.x * 256 + threadIdx.x; i < nbk;
       i += gridDim.x * 256)
    bmin[i] = INT32_MAX;
  const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
  const uint64_t below = l == 0 ? 0ull : (~0ull >> (64 - l));
  const double taille = (double)c.nx;
  const int32_t nu = S->nunits[par];
  for (int32_t u = blockIdx.x; u < nu; u += gridDim.x) {
    const int2 un = units[u];
    const GInfo gi = info[un.x];
    if (w == 0) {
      const int32_t cd = un.y * 64 + l;
      const bool left =
          cd < gi.ncand &&
          G.upper[gi.off + cd] >= __longlong_as_double((long long)gi.best);
      const uint64_t m = __ballot(left);
      if (l == 0) mask = m;
    }
    __syncthreads();
    uint64_t todo = mask;
    for (int i = 0; i < w && todo; i++) todo &= todo - 1;
    double bs = 0.0;
    int64_t bk = INT64_MAX;
    int32_t cs[3];
    if (todo) seed_cell(pos, isort[ready[un.x]] - 1, c.nx, cs);
    while (todo) {  // survivors w, w + 4, ... of the unit
      const int32_t cd = un.y * 64 + __ffsll((unsigned long long)todo) - 1;
      const int64_t ce = gi.off + __float_as_int(
          G.near[gi.off + G.cand[gi.off + cd]].w);
      double pc[3];
      int po[3];
      entry_pos(G, ce, cs, pc, po);
      double acc = 0.0;
      for (int32_t b = 0; b < gi.nnear; b += 64) {
        bool in = false;
        double t = 0.0;
        if (b + l < gi.nnear) {
          double q[3], dd[3];
          int qo[3];
          entry_pos(G, gi.off + __float_as_int(G.near[gi.off + b + l].w), cs, q,
                    qo);
          for (int d = 0; d < 3; d++) {
            dd[d] = fabs(q[d] - pc[d]);
            dd[d] = fmin(dd[d], taille - dd[d]);
          }
          const double d2 = __dadd_rn(__dadd_rn(__dmul_rn(dd[0], dd[0]),
                                                __dmul_rn(dd[1], dd[1])),
                                      __dmul_rn(dd[2], dd[2]));
          in = d2 <= 1.0;
          if (in) t = 1.0 / sqrt(d2 + (1.0 / 64.0) * (1.0 / 64.0));
        }
        const uint64_t mi = __ballot(in);
        if (in) term[w][__popcll(mi & below)] = t;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        const int n = __popcll(mi);
#pragma unroll 8
        for (int i = 0; i < n; i++) acc += term[w][i];
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      }
      const int64_t rank = (po[0] + 1) * 9 + (po[1] + 1) * 3 + (po[2] + 1);
      const int64_t key =
          (rank << 32) | (uint32_t)__float_as_int(G.p[ce].w);
      if (acc > bs || (acc == bs && key < bk)) {
        bs = acc;
        bk = key;
      }
      for (int i = 0; i < 4 && todo; i++) todo &= todo - 1;
    }
    if (l == 0) {
      ws[w] = bs;
      wk[w] = bk;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      for (int i = 1; i < 4; i++)
        if (ws[i] > bs || (ws[i] == bs && wk[i] < bk)) {
          bs = ws[i];
          bk = wk[i];
        }
      ures[2 * (int64_t)u] = (uint64_t)__double_as_longlong(bs);
      ures[2 * (int64_t)u + 1] = (uint64_t)bk;
    }
    __syncthreads();
  }
}

// Growth, one workgroup per seed.  The particles that can be ranked up to
// the crossing are sorted by (d2, gather order) in LDS: all of them when
// they are at most GS_CAP, otherwise those of the radial bins (uniform in
// r^3 up to ncut) up to the first one inside which a crossing is sure; only
// seeds with more than GS_CAP of those sort in global memory (steps within
// GS_CAP keys still in LDS).
constexpr int GG_T = 512, GS_CAP = 8192, GS_BINS = 4096;

struct GrowLds {
  uint64_t key[GS_CAP];
  uint32_t ord[GS_CAP];
  int32_t hist[GS_BINS];
  int64_t red_l[GG_T / 64];
  int32_t n;
};

__device__ inline int64_t gg_min(int64_t v, GrowLds &S) {
  for (int o = 32; o > 0; o >>= 1) v = min(v, (int64_t)__shfl_xor(v, o, 64));
  __syncthreads();
  if ((threadIdx.x & 63) == 0) S.red_l[threadIdx.x >> 6] = v;
  __syncthreads();
  int64_t r = S.red_l[0];
  for (int i = 1; i < GG_T / 64; i++) r = min(r, S.red_l[i]);
  __syncthreads();
  return r;
}

// one step of the bitonic network on keys in LDS: pairs (i, i + j) of the
// nk keys, whose place in the whole sequence starts at g0
__device__ inline void gg_step(GrowLds &S, int32_t nk, int64_t g0, int64_t k,
                               int32_t j) {
  for (int32_t t = threadIdx.x; t < nk / 2; t += GG_T) {
    const int32_t i = ((t & ~(j - 1)) << 1) | (t & (j - 1)), p = i + j;
    const uint64_t a = S.key[i], b = S.key[p];
    const uint32_t oa = S.ord[i], ob = S.ord[p];
    const bool gt = a > b || (a == b && oa > ob);
    if (gt == (((g0 + i) & k) == 0)) {
      S.key[i] = b;
      S.key[p] = a;
      S.ord[i] = ob;
      S.ord[p] = oa;
    }
  }
  __syncthreads();
}

// sorts n keys ascending by (key, ord): keys already in LDS when n <= GS_CAP,
// else in gk / go (space for the next power of two)
__device__ inline void gg_sort(GrowLds &S, uint64_t *gk, uint32_t *go,
                               int32_t n) {
  int32_t np = 64;
  while (np < n) np <<= 1;
  if (n <= GS_CAP) {
    for (int32_t t = n + threadIdx.x; t < np; t += GG_T) {
      S.key[t] = ~0ull;
      S.ord[t] = ~0u;
    }
    __syncthreads();
    for (int32_t k = 2; k <= np; k <<= 1)
      for (int32_t j = k >> 1; j > 0; j >>= 1) gg_step(S, np, 0, k, j);
    return;
  }
  for (int32_t t = n + threadIdx.x; t < np; t += GG_T) {
    gk[t] = ~0ull;
    go[t] = ~0u;
  }
  __threadfence_block();
  __syncthreads();
  // stages k <= GS_CAP and the steps j < GS_CAP of later stages, block by
  // block in LDS
  for (int64_t k = GS_CAP; k <= np; k <<= 1) {
    for (int32_t j = (int32_t)(k >> 1); j >= GS_CAP; j >>= 1) {
      for (int32_t t = threadIdx.x; t < np / 2; t += GG_T) {
        const int32_t i = ((t & ~(j - 1)) << 1) | (t & (j - 1)), p = i + j;
        const uint64_t a = gk[i], b = gk[p];
        const uint32_t oa = go[i], ob = go[p];
        const bool gt = a > b || (a == b && oa > ob);
        if (gt == ((i & k) == 0)) {
          gk[i] = b;
          gk[p] = a;
          go[i] = ob;
          go[p] = oa;
        }
      }
      __threadfence_block();
      __syncthreads();
    }
    for (int32_t g0 = 0; g0 < np; g0 += GS_CAP) {
      for (int32_t t = threadIdx.x; t < GS_CAP; t += GG_T) {
        S.key[t] = gk[g0 + t];
        S.ord[t] = go[g0 + t];
      }
      __syncthreads();
      if (k == GS_CAP)
        for (int32_t k2 = 2; k2 < GS_CAP; k2 <<= 1)
          for (int32_t j = k2 >> 1; j > 0; j >>= 1)
            gg_step(S, GS_CAP, g0, k2, j);
      for (int32_t j = GS_CAP >> 1; j > 0; j >>= 1)
        gg_step(S, GS_CAP, g0, k, j);
      for (int32_t t = threadIdx.x; t < GS_CAP; t += GG_T) {
        gk[g0 + t] = S.key[t];
        go[g0 + t] = S.ord[t];
      }
      __threadfence_block();
      __syncthreads();
    }
  }
}

__global__ void __launch_bounds__(GG_T)
k_greedy_grow(GreedyCfg c, const int32_t *__restrict__ isort,
              const float *__restrict__ pos, const int64_t *__restrict__ ids,
              uint8_t *__restrict__ alive, uint8_t *__restrict__ done, int par,
              GState *__restrict__ St, const int32_t *__restrict__ ready,
              const GInfo *__restrict__ info, const uint64_t *__restrict__ ures,
              GPoolPtrs G, int64_t *__restrict__ structure,
              GRec *__restrict__ recs, double *__restrict__ radb,
              int32_t *__restrict__ massb) {
  __shared__ GrowLds S;
  const int l = threadIdx.x & 63;
  const uint64_t below = l == 0 ? 0ull : (~0ull >> (64 - l));
  const double taille = (double)c.nx;
  const int32_t nr = St->nready[par];
  for (int32_t it = blockIdx.x; it < nr; it += gridDim.x) {
    const GInfo gi = info[it];
    if (gi.n1 == 0) continue;
    const int32_t o = ready[it];
    const int32_t n1 = gi.n1;
    uint64_t *d2 = G.d2 + gi.off, *gk = G.key + gi.off;
    uint32_t *go = G.ord + gi.off;
    // the best candidate over the seed's units (S > 0: as integers)
    uint64_t bs = 0;
    int64_t bk = INT64_MAX;
    for (int32_t g = threadIdx.x; g < (gi.ncand + 63) >> 6; g += GG_T) {
      const uint64_t s = ures[2 * (int64_t)(gi.unit0 + g)];
      const int64_t k = (int64_t)ures[2 * (int64_t)(gi.unit0 + g) + 1];
      if (s > bs || (s == bs && k < bk)) {
        bs = s;
        bk = k;
      }
    }
    const int64_t top = -gg_min(-(int64_t)bs, S);
    const int64_t kbest = gg_min((int64_t)bs == top ? bk : INT64_MAX, S);
    const int32_t centre = (int32_t)(kbest & 0xFFFFFFFF);
    double xc[3];
    centre_scaled(pos, centre, c.nx, xc);
    // distances (main file:2002-2020)
    const bool lds = n1 <= GS_CAP;
    const double nc = (double)c.ncut, bscale = GS_BINS / (nc * nc * nc);
    auto bin = [&](uint64_t bits) {
      const double x = __longlong_as_double((long long)bits);
      const double b = x * sqrt(x) * bscale;  // grows with x
      return b < (double)GS_BINS ? (int32_t)b : GS_BINS;
    };
    if (!lds)
      for (int32_t t = threadIdx.x; t < GS_BINS; t += GG_T) S.hist[t] = 0;
    __syncthreads();
    for (int32_t t = threadIdx.x; t < n1; t += GG_T) {
      const int64_t j = __float_as_int(G.p[gi.off + t].w);
      double dd[3];
      for (int a = 0; a < 3; a++) {
        dd[a] = fabs((double)(pos[3 * j + a] * (float)c.nx) - xc[a]);
        dd[a] = fmin(dd[a], taille - dd[a]);
      }
      const uint64_t v = (uint64_t)__double_as_longlong(
          __dadd_rn(__dadd_rn(__dmul_rn(dd[0], dd[0]), __dmul_rn(dd[1], dd[1])),
                    __dmul_rn(dd[2], dd[2])));
      if (lds) {
        S.key[t] = v;
        S.ord[t] = (uint32_t)t;
      } else {
        d2[t] = v;
        const int32_t b = bin(v);
        if (b < GS_BINS) atomicAdd(&S.hist[b], 1);
      }
    }
    __threadfence_block();
    __syncthreads();
    // The last bin to sort: the first one whose particles must lie below the
    // threshold, O(k) <= (particles up to the bin) / volume(its lower edge),
    // and whose first particle is at least the 10th.
    int32_t blast = GS_BINS;
    if (!lds) {
      // inclusive scan of the bins, GS_BINS / GG_T per thread
      constexpr int V = GS_BINS / GG_T;
      int32_t v[V], s = 0;
      for (int i = 0; i < V; i++) s += v[i] = S.hist[threadIdx.x * V + i];
      const int32_t inc = wave_incl_scan(s);
      if ((threadIdx.x & 63) == 63) S.red_l[threadIdx.x >> 6] = inc;
      __syncthreads();
      int32_t cum = inc - s;
      for (int i = 0; i < (int)(threadIdx.x >> 6); i++)
        cum += (int32_t)S.red_l[i];
      int64_t first = GS_BINS;
      for (int i = 0; i < V; i++) {
        const int32_t b = threadIdx.x * V + i;
        const double vol = 2.0 / 3.0 * TWOPI_REF * ((double)b / bscale);
        if (v[i] > 0 && cum >= 9 && first == GS_BINS &&
            (double)(cum + v[i]) <= c.seuil * vol * (1.0 - 1e-9))
          first = b;
        cum += v[i];
      }
      blast = (int32_t)gg_min(first, S);
    }
    int32_t ns = n1;  // keys sorted
    const uint64_t *SK = S.key;
    const uint32_t *SO = S.ord;
    int64_t stop = INT64_MAX;
    for (;;) {
      if (lds) {
        gg_sort(S, gk, go, n1);
      } else {
        // collect the bins up to blast (all keys: blast = GS_BINS)
        if (threadIdx.x == 0) S.n = 0;
        __syncthreads();
        int32_t cnt = 0;
        for (int32_t t = threadIdx.x; t < n1; t += GG_T)
          cnt += bin(d2[t]) <= blast;
        cnt = wave_sum(cnt);
        if (l == 0 && cnt) atomicAdd(&S.n, cnt);
        __syncthreads();
        ns = S.n;
        __syncthreads();
        if (threadIdx.x == 0) S.n = 0;
        __syncthreads();
        const bool in = ns <= GS_CAP;
        for (int32_t t0 = 0; t0 < n1; t0 += GG_T) {  // uniform trip count
          const int32_t t = t0 + (int32_t)threadIdx.x;
          const bool take = t < n1 && bin(d2[t]) <= blast;
          const uint64_t m = __ballot(take);  // one counter update per wave
          int32_t e = 0;
          if (l == 0 && m) e = atomicAdd(&S.n, (int32_t)__popcll(m));
          e = __shfl(e, 0, 64) + __popcll(m & below);
          if (take && in) {
            S.key[e] = d2[t];
            S.ord[e] = (uint32_t)t;
          } else if (take) {
            gk[e] = d2[t];
            go[e] = (uint32_t)t;
          }
        }
        __threadfence_block();
        __syncthreads();
        gg_sort(S, gk, go, ns);
        SK = in ? S.key : gk;
        SO = in ? S.ord : go;
      }
      // growth (main file:2040-2051): stop at the first i >= 10 with
      // O(i) <= seuil, i == npart_sel or r_i >= ncut
      stop = INT64_MAX;
      for (int64_t i = 10 + threadIdx.x; i <= ns; i += GG_T) {
        const double r = sqrt(__longlong_as_double((long long)SK[i - 1]));
        if (od_k(i, 1.0, r) <= c.seuil || i >= n1 || r >= nc)
          stop = min(stop, i);
      }
      stop = gg_min(stop, S);
      if (stop != INT64_MAX || ns == n1) break;
      blast = GS_BINS;  // not in those bins: every key
    }
    auto rad = [&](int64_t i) {
      return sqrt(__longlong_as_double((long long)SK[i]));
    };
    if (stop == INT64_MAX || od_k(stop, 1.0, rad(stop - 1)) > c.seuil) {
      // "Increase selection radius" (main file:2072-2089)
      if (threadIdx.x == 0)
        atomicMin(&St->fail, ((unsigned long long)o << 8) | GF_UNCLOSED);
      __syncthreads();
      continue;
    }
    // second threshold: last i in [2, stop] above seuil2 (:2062-2069)
    int64_t m2 = 0;
    for (int64_t i = 2 + threadIdx.x; i <= stop; i += GG_T)
      if (od_k(i, 1.0, rad(i - 1)) > c.seuil2) m2 = max(m2, i);
    m2 = -gg_min(-m2, S);
    const int64_t masse = stop - 1;
    const double rayon = rad(masse - 1);
    const double volume = 2.0 / 3.0 * TWOPI_REF * (rayon * rayon * rayon);
    const double amass = (double)masse;
    if (threadIdx.x == 0) {
      S.n = atomicAdd(&St->nrec, 1);
      atomicMax(&St->last, o);
    }
    __syncthreads();
    const int64_t row = S.n;
    // profile (main file:2103-2115): counts of r < r_j.  Every particle
    // closer than the last one sorted is sorted; a radius beyond it counts
    // the unsorted ones too.
    const double rlast = rad(ns - 1);
    for (int j = threadIdx.x; j < c.nbins; j += GG_T) {
      // the last radius is rayon * rmax_frac exactly
      const double rj =
          j == c.nbins - 1 ? rayon * c.rmaxf
                           : rayon * exp(c.lr0 + (double)j * (c.lr1 - c.lr0) /
                                                     ((double)c.nbins - 1.0));
      int32_t lo2 = 0, hi2 = ns;
      if (ns == n1 || rj <= rlast) {
        while (lo2 < hi2) {
          const int32_t mid = (lo2 + hi2) >> 1;
          if (rad(mid) < rj) lo2 = mid + 1; else hi2 = mid;
        }
      } else {
        for (int32_t t = 0; t < n1; t++)
          lo2 += sqrt(__longlong_as_double((long long)d2[t])) < rj;
      }
      radb[row * c.nbins + j] = rj;
      massb[row * c.nbins + j] = lo2;
    }
    const bool acc = amass >= c.mmin && xc[0] <= taille && xc[0] > 0.0 &&
                     xc[1] <= taille && xc[1] > 0.0 && xc[2] <= taille &&
                     xc[2] > 0.0;
    const int64_t iamas = ids ? ids[centre] : (int64_t)centre;
    // exclusion of the first masse particles, accepted or not
    for (int64_t t = threadIdx.x; t < masse; t += GG_T) {
      const int64_t e = gi.off + SO[t];
      alive[G.slot[e]] = 0;
      structure[__float_as_int(G.p[e].w)] = acc ? iamas : 0;
    }
    if (threadIdx.x == 0) {
      GRec R;
      R.ipart = (int64_t)o + 1;
      R.seed = isort[o] - 1;
      R.centre = centre;
      R.iamas = iamas;
      R.masse = masse;
      R.masse2 = m2;
      R.amass = amass;
      R.xc = xc[0];
      R.yc = xc[1];
      R.zc = xc[2];
      R.rayon = rayon;
      R.overdens = volume > 0.0 ? amass / volume : 0.0;
      R.overdens2 = 0.0;
      if (m2 > 0) {
        const double r2 = rad(m2 - 1);
        R.overdens2 = r2 > 1e-30 ? od_k(m2, 1.0, r2) : 0.0;
      }
      R.accepted = acc ? 1 : 0;
      R.pad = 0;
      recs[row] = R;
      done[o] = 1;
    }
    __syncthreads();
  }
}

__global__ void k_alive_orig(const uint8_t *__restrict__ alive_s,
                             const int32_t *__restrict__ perm, int64_t n,
                             uint8_t *__restrict__ alive) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n) alive[perm[k]] = alive_s[k];
}

}  // namespace

extern "C" int psod_host_spherover(psod_ctx *ctx, int64_t npart,
                                   const float *pos, const int64_t *ids,
                                   const int32_t *isort, int64_t npart_new,
                                   const psod_greedy_params *p, int64_t maxrec,
                                   int64_t *nrec, int64_t *rec_i64,
                                   double *rec_f64, double *rad_bins,
                                   int32_t *mass_bins, uint8_t *alive,
                                   int64_t *structure) {
  PSOD_TRY(psod_check_npart("spherover", npart));
  PSOD_TRY(psod_use_device(ctx));
  if (!pos || !isort || !p || !nrec || npart <= 0 || npart_new < 0)
    return psod_set_error(PSOD_E_ARG, "spherover: bad arguments");
  if (p->nx < 8 || p->nx > 1024 || (p->nx & (p->nx - 1)) || p->ncut < 1 ||
      2 * p->ncut + 1 > p->nx || p->nbins < 2 || p->nsel < 1 ||
      !(p->rmin_frac > 0.0) || !(p->rmax_frac > 0.0))
    return psod_set_error(PSOD_E_ARG, "spherover: bad parameters");
  *nrec = 0;
  if (npart_new > npart) npart_new = npart;
  // the seeds index the device's particle arrays: reject any outside them
  // before anything is queued
  for (int64_t o = 0; o < npart_new; o++)
    if (isort[o] < 1 || isort[o] > npart)
      return psod_set_error(PSOD_E_ARG,
                            "spherover: isort(%lld) = %d outside [1, %lld]",
                            (long long)(o + 1), isort[o], (long long)npart);
  GreedyCfg c;
  c.nx = p->nx;
  c.ncut = p->ncut;
  c.nbins = p->nbins;
  // marking blocks of 4^3 cells, of 8^3 where a seed's reach spans many
  c.bsh = p->ncut <= 8 ? 2 : 3;
  c.nb = p->nx >> c.bsh;
  c.seuil = p->seuil;
  c.seuil2 = p->seuil2;
  c.mmin = p->mmin;
  c.lr0 = log(p->rmin_frac);
  c.lr1 = log(p->rmax_frac);
  c.rmaxf = p->rmax_frac;
  c.nsel = p->nsel;
  hipStream_t st = ctx->stream;
  const int64_t ncellt = (int64_t)p->nx * p->nx * p->nx;
  const int64_t nn = npart_new > 0 ? npart_new : 1;
  // every record removes at least 9 particles (its count starts at 10)
  const int64_t rcap = std::min<int64_t>(nn, npart / 9 + 1);
  float *dpos = (float *)psod_scratch(ctx, S_HOST_A, (size_t)npart * 12);
  int32_t *cs = (int32_t *)psod_scratch(ctx, S_HOST_B, (size_t)(ncellt + 1) * 4);
  int32_t *perm = (int32_t *)psod_scratch(ctx, S_HOST_C, (size_t)npart * 4);
  float *drec = (float *)psod_scratch(ctx, S_HOST_D, (size_t)npart * 16);
  char *A = (char *)psod_scratch(ctx, S_GREEDY,
                                 (size_t)npart * (4 + 1 + 8 + 8 + 1) +
                                     (size_t)nn * (4 + 1) + 4096);
  if (!dpos || !cs || !perm || !drec || !A) return PSOD_E_NOMEM;
  int32_t *slot_of = (int32_t *)A;
  int64_t *dstruct = (int64_t *)(A + (((size_t)npart * 4 + 255) & ~(size_t)255));
  int64_t *dids = dstruct + npart;
  uint8_t *alive_s = (uint8_t *)(dids + npart);
  uint8_t *alive_o = alive_s + npart;
  int32_t *dseeds = (int32_t *)(((uintptr_t)(alive_o + npart) + 255) & ~(uintptr_t)255);
  uint8_t *done = (uint8_t *)(dseeds + nn);
  const int32_t nbk = c.nb * c.nb * c.nb;
  // the pool holds a round's gathered particles: at most every ready seed's
  // cells, and one seed's whole slice
  int64_t pcap = GCAP;
  while (pcap < GPOOL && pcap < 16 * npart) pcap <<= 1;
  const int64_t ucap = pcap / 64 + GWIN;
  constexpr size_t PER = 16 + 4 + 4 + 16 + 4 + 8 + 8 + 8 + 4;
  char *B = (char *)psod_scratch(
      ctx, S_GREEDY2,
      (size_t)pcap * PER + (size_t)ucap * (16 + 8) +
          (size_t)GWIN * (sizeof(GInfo) + 4) + (size_t)nbk * 4 + 8192);
  char *R = (char *)psod_scratch(ctx, S_GREEDY3,
                                 (size_t)rcap * (sizeof(GRec) +
                                                 (size_t)p->nbins * 12) + 512);
  if (!B || !R) return PSOD_E_NOMEM;
  GPoolPtrs G;
  GState *S = (GState *)B;
  G.p = (float4 *)(B + 256);
  G.near = G.p + pcap;
  G.upper = (double *)(G.near + pcap);
  G.d2 = (uint64_t *)(G.upper + pcap);
  G.key = G.d2 + pcap;
  uint64_t *ures = G.key + pcap;
  int2 *units = (int2 *)(ures + 2 * ucap);
  GInfo *info = (GInfo *)(units + ucap);
  G.slot = (int32_t *)(info + GWIN);
  G.cell = G.slot + pcap;
  G.cand = G.cell + pcap;
  G.ord = (uint32_t *)(G.cand + pcap);
  int32_t *ready = (int32_t *)(G.ord + pcap);
  int32_t *bmin = ready + GWIN;
  GRec *recs = (GRec *)R;
  double *radb = (double *)(recs + rcap);
  int32_t *massb = (int32_t *)(radb + (size_t)rcap * p->nbins);

  PSOD_HIP(hipMemcpyAsync(dpos, pos, (size_t)npart * 12, hipMemcpyHostToDevice, st));
  PSOD_TRY(psod_cell_sort(ctx, npart, dpos, nullptr, p->nx, cs, perm, drec,
                          nullptr));
  if (ids)
    PSOD_HIP(hipMemcpyAsync(dids, ids, (size_t)npart * 8, hipMemcpyHostToDevice, st));
  k_inverse_perm<<<grid_for(npart, 256), 256, 0, st>>>(perm, npart, slot_of);
  PSOD_LAUNCH_CHECK();
  // isort: 1-based particle indices
  if (npart_new > 0)
    PSOD_HIP(hipMemcpyAsync(dseeds, isort, (size_t)npart_new * 4,
                            hipMemcpyHostToDevice, st));
  // The seeds of orders below nnew, from the start: rounds over a sliding
  // window of seeds, GROUNDS of them queued at a time; the window, the counts
  // and the work lists stay on the device.
  GState hs;
  auto run = [&](int32_t nnew) -> int {
    k_set_u8<<<grid_for(npart, 256, 4096), 256, 0, st>>>(alive_s, npart, 1);
    PSOD_LAUNCH_CHECK();
    PSOD_HIP(hipMemsetAsync(dstruct, 0, (size_t)npart * 8, st));
    PSOD_HIP(hipMemsetAsync(done, 0, (size_t)nn, st));
    PSOD_TRY(psod_fill_i32(ctx, bmin, nbk, INT32_MAX));
    memset(&hs, 0, sizeof(hs));
    hs.fail = ~0ull;
    hs.last = -1;
    PSOD_HIP(hipMemcpyAsync(S, &hs, sizeof(hs), hipMemcpyHostToDevice, st));
    PSOD_HIP(hipStreamSynchronize(st));
    int32_t lo = 0, end = nnew;
    int64_t ran = 0;  // ready seeds so far
    while (lo < end) {
      const int32_t lo0 = lo, end0 = end;
      for (int r = 0; r < GROUNDS; r++) {
        const int par = r & 1;
        // the window starts at lo0 or later
        const unsigned gw = grid_for(std::min<int64_t>(GWIN, nnew - lo0), 256);
        k_mark<<<gw, 256, 0, st>>>(c, dseeds, slot_of, dpos, alive_s, done,
                                   nnew, par, S, bmin);
        PSOD_LAUNCH_CHECK();
        k_ready<<<gw, 256, 0, st>>>(c, dseeds, slot_of, dpos, alive_s, done,
                                    nnew, par, S, bmin, ready);
        PSOD_LAUNCH_CHECK();
        k_greedy_gather<<<(unsigned)ctx->num_cus, GA_T, 0, st>>>(
            c, dseeds, cs, (const float4 *)drec, dpos, alive_s, done, par, S,
            ready, info, units, G, pcap);
        PSOD_LAUNCH_CHECK();
        k_greedy_bound<<<(unsigned)ctx->num_cus * 4, GC_T, 0, st>>>(
            par, S, info, units, G);
        PSOD_LAUNCH_CHECK();
        k_greedy_centre<<<(unsigned)ctx->num_cus * 4, 256, 0, st>>>(
            c, dseeds, dpos, par, S, ready, info, units, G, ures, bmin, nbk);
        PSOD_LAUNCH_CHECK();
        k_greedy_grow<<<(unsigned)ctx->num_cus, GG_T, 0, st>>>(
            c, dseeds, dpos, ids ? dids : nullptr, alive_s, done, par, S,
            ready, info, ures, G, dstruct, recs, radb, massb);
        PSOD_LAUNCH_CHECK();
      }
      PSOD_HIP(hipMemcpyAsync(&hs, S, sizeof(hs), hipMemcpyDeviceToHost, st));
      PSOD_HIP(hipStreamSynchronize(st));
      lo = hs.first[(GROUNDS - 1) & 1];
      end = (int32_t)std::min<uint64_t>((uint64_t)nnew, hs.fail >> 8);
      const int64_t r1 = (int64_t)hs.total + hs.nready[(GROUNDS - 1) & 1];
      if (lo < end && lo == lo0 && r1 == ran && end == end0)
        return psod_set_error(PSOD_E_DEVICE, "spherover: no progress");
      ran = r1;
    }
    return PSOD_OK;
  };
  PSOD_TRY(run((int32_t)npart_new));
  // Every seed before the failing one has run now.  Where seeds after it did
  // too, in rounds before it, the seeds before it run again by themselves: the
  // zone ends with the particles that these captured, no others.
  const uint64_t fail = hs.fail;
  if (fail != ~0ull && hs.last > (int64_t)(fail >> 8)) {
    PSOD_TRY(run((int32_t)(fail >> 8)));
    if (hs.fail != ~0ull)
      return psod_set_error(PSOD_E_DEVICE, "spherover: seed %lld failed in a "
                            "second run only", (long long)(hs.fail >> 8) + 1);
  }
  // records, in seed order up to the first failing seed
  const int64_t nr = hs.nrec;
  std::vector<GRec> hr((size_t)nr);
  std::vector<double> hrb((size_t)nr * p->nbins);
  std::vector<int32_t> hmb((size_t)nr * p->nbins);
  if (nr > 0) {
    PSOD_HIP(hipMemcpyAsync(hr.data(), recs, (size_t)nr * sizeof(GRec),
                            hipMemcpyDeviceToHost, st));
    PSOD_HIP(hipMemcpyAsync(hrb.data(), radb, hrb.size() * 8,
                            hipMemcpyDeviceToHost, st));
    PSOD_HIP(hipMemcpyAsync(hmb.data(), massb, hmb.size() * 4,
                            hipMemcpyDeviceToHost, st));
  }
  if (alive) {
    k_alive_orig<<<grid_for(npart, 256), 256, 0, st>>>(alive_s, perm, npart,
                                                       alive_o);
    PSOD_LAUNCH_CHECK();
    PSOD_HIP(hipMemcpyAsync(alive, alive_o, (size_t)npart,
                            hipMemcpyDeviceToHost, st));
  }
  if (structure)
    PSOD_HIP(hipMemcpyAsync(structure, dstruct, (size_t)npart * 8,
                            hipMemcpyDeviceToHost, st));
  PSOD_HIP(hipStreamSynchronize(st));
  const int64_t upto = fail == ~0ull ? npart_new : (int64_t)(fail >> 8);
  std::vector<int32_t> order((size_t)nr);
  std::iota(order.begin(), order.end(), 0);
  std::sort(order.begin(), order.end(), [&](int32_t a, int32_t b) {
    return hr[(size_t)a].ipart < hr[(size_t)b].ipart;
  });
  int64_t k = 0;
  for (int64_t i = 0; i < nr; i++) {
    const int64_t o = order[(size_t)i];
    const GRec &g = hr[(size_t)o];
    if (g.ipart > upto) break;
    if (k >= maxrec) return psod_set_error(PSOD_E_CAPACITY,
                                           "spherover: more than %lld records",
                                           (long long)maxrec);
    if (rec_i64) {
      int64_t *ri = rec_i64 + 6 * k;
      ri[0] = g.ipart; ri[1] = g.seed; ri[2] = g.centre; ri[3] = g.iamas;
      ri[4] = g.masse; ri[5] = g.masse2;
    }
    if (rec_f64) {
      double *rf = rec_f64 + 8 * k;
      rf[0] = g.amass; rf[1] = g.xc; rf[2] = g.yc; rf[3] = g.zc;
      rf[4] = g.rayon; rf[5] = g.overdens; rf[6] = g.overdens2;
      rf[7] = g.accepted;
    }
    if (rad_bins)
      memcpy(rad_bins + k * p->nbins, &hrb[(size_t)o * p->nbins],
             sizeof(double) * p->nbins);
    if (mass_bins)
      memcpy(mass_bins + k * p->nbins, &hmb[(size_t)o * p->nbins],
             sizeof(int32_t) * p->nbins);
    k++;
  }
  *nrec = k;
  if (fail != ~0ull) {
    const long long seed1 = (long long)(fail >> 8) + 1;
    const int code = (int)(fail & 255);
    if (code == GF_GCAP)
      return psod_set_error(PSOD_E_CAPACITY,
                            "spherover: seed %lld gathers more than %lld "
                            "particles (device slice)", seed1, (long long)GCAP);
    if (code == GF_NSEL)
      return psod_set_error(PSOD_E_CAPACITY,
                            "spherover: Nsel exceeded at seed %lld", seed1);
    return psod_set_error(PSOD_E_UNCLOSED,
                          "spherover: sphere of seed %lld not closed within "
                          "ncut", seed1);
  }
  return PSOD_OK;
}
