// ctx.hip -- context, errors, scratch, scan and radix sort primitives.
#include <cstdarg>
#include <cstdlib>
#include <cstring>

#include "psod_internal.h"

#include <utility>

static thread_local char g_err[1024] = "";

int psod_set_error(int code, const char *fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

extern "C" const char *psod_last_error(void) { return g_err; }

extern "C" int psod_create(int device, psod_ctx **out) {
  if (!out) return psod_set_error(PSOD_E_ARG, "psod_create: out is NULL");
  *out = nullptr;
  int n = 0;
  hipError_t e = hipGetDeviceCount(&n);
  if (e != hipSuccess || n == 0)
    return psod_set_error(PSOD_E_DEVICE,
                          "psod_create: no HIP device (%s)",
                          hipGetErrorString(e));
  if (device < 0 || device >= n)
    return psod_set_error(PSOD_E_ARG, "psod_create: device %d of %d", device,
                          n);
  PSOD_HIP(hipSetDevice(device));
  psod_ctx *c = (psod_ctx *)calloc(1, sizeof(psod_ctx));
  c->device = device;
  hipError_t es = hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking);
  if (es != hipSuccess) {
    free(c);
    return psod_set_error(PSOD_E_DEVICE, "hipStreamCreate: %s",
                          hipGetErrorString(es));
  }
  if (hipEventCreate(&c->ev[0]) != hipSuccess ||
      hipEventCreate(&c->ev[1]) != hipSuccess ||
      hipEventCreateWithFlags(&c->fork, hipEventDisableTiming) != hipSuccess ||
      hipEventCreateWithFlags(&c->join, hipEventDisableTiming) != hipSuccess ||
      hipStreamCreateWithFlags(&c->side, hipStreamNonBlocking) != hipSuccess) {
    hipStreamDestroy(c->stream);
    free(c);
    return psod_set_error(PSOD_E_DEVICE, "hipEventCreate failed");
  }
  // the fixed tile list of psod_cic_deposit_noalloc on this device
  const int rs = psod_static_scratch_init(device);
  if (rs != PSOD_OK) {
    hipEventDestroy(c->ev[0]);
    hipEventDestroy(c->ev[1]);
    hipEventDestroy(c->fork);
    hipEventDestroy(c->join);
    hipStreamDestroy(c->side);
    hipStreamDestroy(c->stream);
    free(c);
    return rs;
  }
  hipDeviceProp_t prop;
  if (hipGetDeviceProperties(&prop, device) == hipSuccess) {
    c->num_cus = prop.multiProcessorCount;
    snprintf(c->device_name, sizeof(c->device_name), "%s", prop.gcnArchName);
  } else {
    c->num_cus = 256;
    snprintf(c->device_name, sizeof(c->device_name), "unknown");
  }
  // names are single words in the tuning file
  for (char *q = c->device_name; *q; q++)
    if (*q == ' ' || *q == '\t') *q = '_';
  *out = c;
  if (const char *tf = getenv("PSOD_TUNE_FILE")) {
    int32_t nl = 0;
    const int rl = psod_load_tunables(c, tf, &nl);
    if (rl != PSOD_OK) {
      psod_destroy(c);
      *out = nullptr;
      return rl;
    }
  }
  return PSOD_OK;
}

extern "C" int psod_destroy(psod_ctx *c) {
  if (!c) return PSOD_OK;
  hipSetDevice(c->device);
  hipStreamSynchronize(c->stream);
  hipStreamSynchronize(c->side);
  psod_graph_release(c);
  for (int s = 0; s < S_NSLOT; s++)
    if (c->slot[s]) hipFree(c->slot[s]);
  hipEventDestroy(c->ev[0]);
  hipEventDestroy(c->ev[1]);
  hipEventDestroy(c->fork);
  hipEventDestroy(c->join);
  hipStreamDestroy(c->side);
  hipStreamDestroy(c->stream);
  free(c);
  return PSOD_OK;
}

extern "C" int psod_synchronize(psod_ctx *c) {
  if (!c) return psod_set_error(PSOD_E_ARG, "null context");
  PSOD_HIP(hipStreamSynchronize(c->stream));
  PSOD_HIP(hipStreamSynchronize(c->side));
  return PSOD_OK;
}

extern "C" void *psod_stream(psod_ctx *c) { return c ? (void *)c->stream : nullptr; }

extern "C" int64_t psod_scratch_bytes(psod_ctx *c) {
  int64_t s = 0;
  if (c)
    for (int i = 0; i < S_NSLOT; i++) s += (int64_t)c->cap[i];
  return s;
}

extern "C" int psod_sod_stats(psod_ctx *c, int64_t *out, int32_t n) {
  if (!c || !out || n < 0) return psod_set_error(PSOD_E_ARG, "psod_sod_stats: bad arguments");
  for (int i = 0; i < n && i < 13; i++) out[i] = c->sod_stat[i];
  return PSOD_OK;
}

int psod_use_device(psod_ctx *c) {
  if (!c) return psod_set_error(PSOD_E_ARG, "null context");
  if (c->capturing) return PSOD_OK;  // the capturing call made it current
  PSOD_HIP(hipSetDevice(c->device));
  return PSOD_OK;
}

int psod_finish(psod_ctx *c) {
  if (c->capturing || c->queueing) return PSOD_OK;
  PSOD_HIP(hipStreamSynchronize(c->stream));
  return PSOD_OK;
}

void *psod_scratch(psod_ctx *c, int slot, size_t bytes) {
  if (bytes == 0) bytes = 256;
  if (c->cap[slot] >= bytes) return c->slot[slot];
  if (c->capturing) {
    psod_set_error(PSOD_E_CAPACITY, "scratch slot %d would grow from %zu to "
                   "%zu bytes while the pass is captured", slot, c->cap[slot],
                   bytes);
    return nullptr;
  }
  // a captured pass holds the old buffer's address: it is dropped (and
  // captured again by the next psod_pass_graph call)
  psod_graph_release(c);
  if (c->slot[slot]) {
    hipStreamSynchronize(c->stream);
    hipStreamSynchronize(c->side);
    hipFree(c->slot[slot]);
    c->slot[slot] = nullptr;
    c->cap[slot] = 0;
  }
  size_t want = bytes + bytes / 8;
  void *p = nullptr;
  if (hipMalloc(&p, want) != hipSuccess) {
    (void)hipGetLastError();
    if (hipMalloc(&p, bytes) != hipSuccess) {
      (void)hipGetLastError();
      psod_set_error(PSOD_E_NOMEM, "device allocation of %zu bytes failed",
                     bytes);
      return nullptr;
    }
    want = bytes;
  }
  c->slot[slot] = p;
  c->cap[slot] = want;
  return p;
}

int psod_fill_i32(psod_ctx *c, int32_t *p, int64_t n, int32_t v);

// ---------------------------------------------------------------------------
// exclusive scan of int32, 256 threads x 16 elements per block
// ---------------------------------------------------------------------------
constexpr int SCAN_T = 256, SCAN_V = 16, SCAN_TILE = SCAN_T * SCAN_V;

__device__ inline int32_t block_excl_scan(int32_t v, int32_t *total) {
  __shared__ int32_t wsum[SCAN_T / 64];
  const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
  int32_t inc = wave_incl_scan(v);
  if (l == 63) wsum[w] = inc;
  __syncthreads();
  int32_t off = 0, tot = 0;
  for (int i = 0; i < SCAN_T / 64; i++) {
    if (i < w) off += wsum[i];
    tot += wsum[i];
  }
  __syncthreads();
  if (total) *total = tot;
  return off + inc - v;
}

__global__ void __launch_bounds__(SCAN_T)
k_scan_reduce(const int32_t *__restrict__ in, int64_t n,
              int32_t *__restrict__ part) {
  const int64_t base = (int64_t)blockIdx.x * SCAN_TILE;
  int32_t s = 0;
  for (int k = 0; k < SCAN_V; k++) {
    const int64_t i = base + (int64_t)k * SCAN_T + threadIdx.x;
    if (i < n) s += in[i];
  }
  int32_t tot;
  (void)block_excl_scan(s, &tot);
  if (threadIdx.x == 0) part[blockIdx.x] = tot;
}

__global__ void __launch_bounds__(SCAN_T)
k_scan_apply(const int32_t *__restrict__ in, int64_t n,
             const int32_t *__restrict__ partscan, int32_t *__restrict__ out) {
  const int64_t base = (int64_t)blockIdx.x * SCAN_TILE +
                       (int64_t)threadIdx.x * SCAN_V;
  int32_t v[SCAN_V];
  int32_t s = 0;
  for (int k = 0; k < SCAN_V; k++) {
    const int64_t i = base + k;
    v[k] = (i < n) ? in[i] : 0;
    s += v[k];
  }
  int32_t ex = block_excl_scan(s, nullptr) + (partscan ? partscan[blockIdx.x] : 0);
  for (int k = 0; k < SCAN_V; k++) {
    const int64_t i = base + k;
    if (i < n) out[i] = ex;
    ex += v[k];
  }
}

__global__ void k_scan_total(const int32_t *in, const int32_t *out, int64_t n,
                             int32_t *total) {
  if (threadIdx.x == 0 && blockIdx.x == 0) *total = out[n - 1] + in[n - 1];
}

int psod_scan_i32(psod_ctx *c, const int32_t *in, int32_t *out, int64_t n,
                  int32_t *total) {
  if (n <= 0) return PSOD_OK;
  if (in == out)
    return psod_set_error(PSOD_E_ARG, "psod_scan_i32 is out of place");
  // level sizes: n, ceil(n/T), ceil(n/T^2), ... down to one tile
  int64_t len[8];
  int nlev = 0;
  len[nlev++] = n;
  while (len[nlev - 1] > SCAN_TILE) {
    if (nlev == 8) return psod_set_error(PSOD_E_ARG, "scan too long");
    len[nlev] = (len[nlev - 1] + SCAN_TILE - 1) / SCAN_TILE;
    nlev++;
  }
  // one buffer for the partials (part) and their scans (ps) of every level
  int64_t need = 0;
  for (int l = 1; l < nlev; l++) need += 2 * (len[l] + 64);
  int32_t *buf = (int32_t *)psod_scratch(c, S_SCAN, (size_t)(need + 64) * 4);
  if (!buf) return PSOD_E_NOMEM;
  const int32_t *lin[8];
  int32_t *lout[8];
  lin[0] = in;
  lout[0] = out;
  int64_t o = 0;
  for (int l = 1; l < nlev; l++) {
    lin[l] = buf + o;
    o += len[l] + 64;
    lout[l] = buf + o;
    o += len[l] + 64;
  }
  // reduce down the levels
  for (int l = 0; l + 1 < nlev; l++) {
    k_scan_reduce<<<(unsigned)len[l + 1], SCAN_T, 0, c->stream>>>(
        lin[l], len[l], (int32_t *)lin[l + 1]);
    PSOD_LAUNCH_CHECK();
  }
  // top level in one tile, then apply back up
  k_scan_apply<<<1, SCAN_T, 0, c->stream>>>(lin[nlev - 1], len[nlev - 1],
                                             nullptr, lout[nlev - 1]);
  PSOD_LAUNCH_CHECK();
  for (int l = nlev - 2; l >= 0; l--) {
    k_scan_apply<<<(unsigned)len[l + 1], SCAN_T, 0, c->stream>>>(
        lin[l], len[l], lout[l + 1], lout[l]);
    PSOD_LAUNCH_CHECK();
  }
  if (total) {
    k_scan_total<<<1, 64, 0, c->stream>>>(in, out, n, total);
    PSOD_LAUNCH_CHECK();
  }
  return PSOD_OK;
}

// ---------------------------------------------------------------------------
// LSD radix sort, 8-bit digits, u32 or u64 keys + u32 values, stable.
// Per pass: (1) per-tile digit histograms stored digit-major, (2) exclusive
// scan over [digit][tile], (3) stable scatter.  A tile is RS_TILE keys, a
// contiguous 64 * RS_V of them per wave.  A wave ranks its keys 64 at a time
// (the lanes of equal digit from ballots, a running count per digit in its
// own LDS row), so that ranking needs no barrier; the tile then goes through
// LDS into digit order and is written in runs of 32 keys per digit on
// average.  The tiles of an XCD are contiguous, so that neighbouring runs of
// a digit meet in its L2.  What bounds it is HBM: 4 + 16 bytes per u32 key
// and pass.  Writing each round of 256 keys where it went, 12-byte elements
// for 32-bit keys, took 1.52 ms per pass of 1e8 keys; now 0.36-0.60.
// ---------------------------------------------------------------------------
constexpr int RS_T = 512, RS_V = 16, RS_TILE = RS_T * RS_V, RS_R = 256,
              RS_W = RS_T / 64;

// Tile of workgroup b (-1: none): the tiles of an XCD are contiguous, so that
// neighbouring runs and table entries are written through one L2.
__device__ inline int64_t rs_tile(uint32_t b, int64_t ntile) {
  const int64_t per = (ntile + 7) / 8, t = (int64_t)(b % 8) * per + b / 8;
  return b / 8 < per && t < ntile ? t : -1;
}

// key of the density order: decreasing rho (clamped at 0)
__device__ inline uint32_t rho_key(float r) {
  return 0xFFFFFFFFu - __float_as_uint(fmaxf(r, 0.0f));
}

// RHO: keys come from the densities; also counts those above thr
template <typename K, bool RHO>
__global__ void __launch_bounds__(RS_T)
k_rs_hist(const K *__restrict__ keys, const float *__restrict__ rho, float thr,
          unsigned long long *__restrict__ nabove, int64_t n, int shift,
          int32_t *__restrict__ hist, int64_t ntile) {
  __shared__ int32_t h[RS_R], above;
  const int64_t tile = rs_tile(blockIdx.x, ntile);
  if (tile < 0) return;
  if (threadIdx.x < RS_R) h[threadIdx.x] = 0;
  if (threadIdx.x == 0) above = 0;
  __syncthreads();
  const int64_t base = tile * RS_TILE;
  int32_t cnt = 0;
  K k[RS_V];
#pragma unroll
  for (int j = 0; j < RS_V; j++) {
    const int64_t i = base + (int64_t)j * RS_T + threadIdx.x;
    if (i < n) {
      if constexpr (RHO) {
        const float r = rho[i];
        cnt += r > thr;
        k[j] = rho_key(r);
      } else {
        k[j] = keys[i];
      }
    }
  }
#pragma unroll
  for (int j = 0; j < RS_V; j++)
    if (base + (int64_t)j * RS_T + threadIdx.x < n)
      atomicAdd(&h[(k[j] >> shift) & 0xFF], 1);
  if constexpr (RHO) {
    cnt = wave_sum(cnt);
    if ((threadIdx.x & 63) == 0 && cnt) atomicAdd(&above, cnt);
  }
  __syncthreads();
  if (threadIdx.x < RS_R)
    hist[(int64_t)threadIdx.x * ntile + tile] = h[threadIdx.x];
  if constexpr (RHO)
    if (threadIdx.x == 0 && above)
      atomicAdd(nabove, (unsigned long long)above);
}

// FIRST: values are the keys' places (and, with RHO, the keys come from the
// densities); LAST: only the values are written, plus 1 (1-based order)
template <typename K, bool RHO, bool LAST>
__global__ void __launch_bounds__(RS_T)
k_rs_scatter(const K *__restrict__ kin, const float *__restrict__ rho,
             const uint32_t *__restrict__ vin, int64_t n, int shift,
             const int32_t *__restrict__ offs, int64_t ntile,
             K *__restrict__ kout, uint32_t *__restrict__ vout) {
  __shared__ K ex[RS_TILE];
  __shared__ int32_t wcnt[RS_W][RS_R];
  __shared__ int32_t tbase[RS_R], gof[RS_R], wsum[RS_W];
  uint32_t *exv = reinterpret_cast<uint32_t *>(ex);
  const int64_t tile = rs_tile(blockIdx.x, ntile);
  if (tile < 0) return;
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  const uint64_t lower = l == 0 ? 0ull : (~0ull >> (64 - l));
  const int64_t base = tile * RS_TILE;
  const int32_t m = (int32_t)min((int64_t)RS_TILE, n - base);
  for (int d = l; d < RS_R; d += 64) wcnt[w][d] = 0;
  K key[RS_V];
  uint32_t val[RS_V];
  int32_t rk[RS_V];
#pragma unroll
  for (int j = 0; j < RS_V; j++) {
    const int32_t i = w * 64 * RS_V + j * 64 + l;
    key[j] = 0;
    val[j] = (uint32_t)(base + i);
    if (i < m) {
      if constexpr (RHO) key[j] = rho_key(rho[base + i]);
      else key[j] = kin[base + i];
      if (vin) val[j] = vin[base + i];
    }
  }
#pragma unroll
  for (int j = 0; j < RS_V; j++) {
    const bool ok = w * 64 * RS_V + j * 64 + l < m;
    const uint32_t dg = (uint32_t)((key[j] >> shift) & 0xFF);
    // lanes of this wave with the same digit
    uint64_t same = ballot64(ok);
#pragma unroll
    for (int b = 0; b < 8; b++) {
      const uint64_t bb = ballot64(ok && ((dg >> b) & 1));
      same &= ((dg >> b) & 1) ? bb : ~bb;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int32_t c0 = wcnt[w][dg];
    rk[j] = c0 + __popcll(same & lower);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (ok && (same & lower) == 0) wcnt[w][dg] = c0 + __popcll(same);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
  __syncthreads();
  // exclusive over the waves per digit, then over the digits
  int32_t tot = 0;
  if (threadIdx.x < RS_R)
    for (int i = 0; i < RS_W; i++) {
      const int32_t c = wcnt[i][threadIdx.x];
      wcnt[i][threadIdx.x] = tot;
      tot += c;
    }
  const int32_t inc = wave_incl_scan(tot);
  if (l == 63) wsum[w] = inc;
  __syncthreads();
  if (threadIdx.x < RS_R) {
    int32_t e = inc - tot;
    for (int i = 0; i < w; i++) e += wsum[i];
    tbase[threadIdx.x] = e;
    gof[threadIdx.x] = offs[(int64_t)threadIdx.x * ntile + tile] - e;
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < RS_V; j++)
    if (w * 64 * RS_V + j * 64 + l < m) {
      const uint32_t dg = (uint32_t)((key[j] >> shift) & 0xFF);
      rk[j] += tbase[dg] + wcnt[w][dg];
      ex[rk[j]] = key[j];
    }
  __syncthreads();
  int32_t dst[RS_V];
#pragma unroll
  for (int j = 0; j < RS_V; j++) {
    const int32_t i = j * RS_T + threadIdx.x;
    if (i < m) {
      const K k = ex[i];
      dst[j] = gof[(k >> shift) & 0xFF] + i;
      if constexpr (!LAST) kout[dst[j]] = k;
    }
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < RS_V; j++)
    if (w * 64 * RS_V + j * 64 + l < m) exv[rk[j]] = val[j];
  __syncthreads();
#pragma unroll
  for (int j = 0; j < RS_V; j++) {
    const int32_t i = j * RS_T + threadIdx.x;
    if (i < m) vout[dst[j]] = LAST ? exv[i] + 1u : exv[i];
  }
}

// Tile histograms and their scan for one pass; *offs the scanned table.
template <typename K, bool RHO>
static int rs_offsets(psod_ctx *c, const K *keys, const float *rho, float thr,
                      unsigned long long *nabove, int64_t n, int shift,
                      int64_t ntile, int32_t **offs) {
  const int64_t hn = ntile * RS_R;
  int32_t *hist = (int32_t *)psod_scratch(c, S_HIST, (size_t)hn * 8 + 64);
  if (!hist) return PSOD_E_NOMEM;
  *offs = hist + hn;
  k_rs_hist<K, RHO><<<(unsigned)((ntile + 7) / 8 * 8), RS_T, 0, c->stream>>>(
      keys, rho, thr, nabove, n, shift, hist, ntile);
  PSOD_LAUNCH_CHECK();
  return psod_scan_i32(c, hist, *offs, hn, nullptr);
}

int psod_radix_sort_u64(psod_ctx *c, int64_t n, uint64_t *keys,
                        uint32_t *vals, bool order) {
  if (n <= 1) {
    if (order && n == 1) return psod_fill_i32(c, (int32_t *)vals, 1, 1);
    return PSOD_OK;
  }
  const int64_t ntile = (n + RS_TILE - 1) / RS_TILE;
  const unsigned nwg = (unsigned)((ntile + 7) / 8 * 8);
  uint64_t *k2 = (uint64_t *)psod_scratch(c, S_KEYS2, (size_t)n * 8);
  uint32_t *v2 = (uint32_t *)psod_scratch(c, S_VALS2, (size_t)n * 4);
  if (!k2 || !v2) return PSOD_E_NOMEM;
  uint64_t *ka = keys, *kb = k2;
  uint32_t *va = vals, *vb = v2;
  for (int p = 0; p < 8; p++) {  // even: the result is back in keys, vals
    int32_t *offs;
    const int shift = 8 * p;
    PSOD_TRY((rs_offsets<uint64_t, false>(c, ka, nullptr, 0.f, nullptr, n,
                                          shift, ntile, &offs)));
    const uint32_t *vin = order && p == 0 ? nullptr : va;
    if (order && p == 7)
      k_rs_scatter<uint64_t, false, true><<<nwg, RS_T, 0, c->stream>>>(
          ka, nullptr, vin, n, shift, offs, ntile, kb, vb);
    else
      k_rs_scatter<uint64_t, false, false><<<nwg, RS_T, 0, c->stream>>>(
          ka, nullptr, vin, n, shift, offs, ntile, kb, vb);
    PSOD_LAUNCH_CHECK();
    std::swap(ka, kb);
    std::swap(va, vb);
  }
  return PSOD_OK;
}

int psod_order_by_density(psod_ctx *c, int64_t n, const float *rho, float thr,
                          unsigned long long *nabove, int32_t *isort) {
  const int64_t ntile = (n + RS_TILE - 1) / RS_TILE;
  const unsigned nwg = (unsigned)((ntile + 7) / 8 * 8);
  uint32_t *kb[2] = {(uint32_t *)psod_scratch(c, S_KEYS, (size_t)n * 4),
                     (uint32_t *)psod_scratch(c, S_KEYS2, (size_t)n * 4)};
  uint32_t *vb[2] = {(uint32_t *)psod_scratch(c, S_VALS, (size_t)n * 4),
                     (uint32_t *)psod_scratch(c, S_VALS2, (size_t)n * 4)};
  if (!kb[0] || !kb[1] || !vb[0] || !vb[1]) return PSOD_E_NOMEM;
  int32_t *offs;
  PSOD_TRY((rs_offsets<uint32_t, true>(c, nullptr, rho, thr, nabove, n, 0,
                                       ntile, &offs)));
  k_rs_scatter<uint32_t, true, false><<<nwg, RS_T, 0, c->stream>>>(
      nullptr, rho, nullptr, n, 0, offs, ntile, kb[0], vb[0]);
  PSOD_LAUNCH_CHECK();
  for (int p = 1; p < 4; p++) {
    const int a = (p - 1) & 1, b = p & 1;
    PSOD_TRY((rs_offsets<uint32_t, false>(c, kb[a], nullptr, 0.f, nullptr, n,
                                          8 * p, ntile, &offs)));
    if (p < 3)
      k_rs_scatter<uint32_t, false, false><<<nwg, RS_T, 0, c->stream>>>(
          kb[a], nullptr, vb[a], n, 8 * p, offs, ntile, kb[b], vb[b]);
    else
      k_rs_scatter<uint32_t, false, true><<<nwg, RS_T, 0, c->stream>>>(
          kb[a], nullptr, vb[a], n, 8 * p, offs, ntile, nullptr,
          (uint32_t *)isort);
    PSOD_LAUNCH_CHECK();
  }
  return PSOD_OK;
}
