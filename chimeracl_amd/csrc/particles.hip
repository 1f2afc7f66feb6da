// Particle kernels: coordinate push, cell keys + stable counting sort,
// longitudinal density profile.  gfx950, wave64.
//
// Sort design (replaces index_and_sum_in_cell + PyOpenCL cumsum + the
// atomic `sort` kernel, particles_generic.cl:88-126, 186-200):
//   1. key kernel: cell key per particle (optionally fused with the
//      coordinate push), no atomics
//   2. stable sort of the keys with the particle index as value, by passes of
//      up to 11-bit digits: per tile of 4096..16384 keys an LDS digit
//      histogram, a column scan of the tiles' counts, then a scatter that
//      sorts the tile in LDS (ballot-matched digits per wave) and writes runs
//      of consecutive slots.  One pass up to 11-bit keys, a bucket sort (high
//      bits, then low bits inside each bucket) up to 22 bits, else LSD passes;
//      the last pass also writes the sorted keys
//   3. cell_offset[c] = lower bound of c in the sorted keys, Np_stay: from the
//      digit counts, or after LSD passes from the slots where the sorted key
//      changes
// The result is exactly numpy.argsort(key, kind='stable') and the
// reference's cell_offset; no global atomics, no order fix-up.
#include "chm_common.h"

#include <mutex>
#include <type_traits>

#define SORT_BS 256
#define RS_ITEMS 16
// From RS_BIG keys on the tiles are larger: 16384 keys in the first pass
// (fewer rows of counts), 8192 in the second.  Measured on the 66.8M keys of
// the 4096 x 512 workload half a cell of drift after a realignment, us:
//   first pass, tiles of 4096 / 8192 / 16384:  counts and their scan 170 /
//   154 / 120, scatter 205 / 190 / 188
//   second, 8192 / 16384: scatter 306 / 425
#define RS_BIG ((int64_t)1 << 23)
// keys per bucket from which the bucket sort is taken, and the larger tiles
// of its second pass
#define RS_BUCKET ((int64_t)2048)
#define RS_TILES2 ((int64_t)16384)
#define RS_NT1 1024
#define RS_NT2 512
// copies of a tile's histogram, 8 banks apart: lanes with equal digits are
// what its LDS adds wait for
#define RS_COPIES 4
#define RS_PAD 8

// ------------------------------------------------------------------ push
template <typename T>
__global__ void __launch_bounds__(256) k_push_x(T *__restrict__ x, T *__restrict__ y, T *__restrict__ z,
                                                const T *__restrict__ px, const T *__restrict__ py,
                                                const T *__restrict__ pz, const T *__restrict__ g_inv,
                                                T dt, int64_t Np) {
  int64_t ip = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (ip >= Np) return;
  // particles_generic.cl:143-151, same rounding order
  T dt_g = dt * g_inv[ip];
  T dx = px[ip] * dt_g;
  T dy = py[ip] * dt_g;
  T dz = pz[ip] * dt_g;
  x[ip] = x[ip] + dx;
  y[ip] = y[ip] + dy;
  z[ip] = z[ip] + dz;
}

template <typename T>
static int push_x(T *x, T *y, T *z, const T *px, const T *py, const T *pz, const T *g_inv, T dt,
                  int64_t Np, void *stream) {
  if (Np < 0) return CHM_EINVAL;
  if (Np == 0) return CHM_OK;
  k_push_x<T><<<chm_blocks(Np, 256), 256, 0, (hipStream_t)stream>>>(x, y, z, px, py, pz, g_inv, dt, Np);
  CHM_CHECK_LAUNCH();
  return CHM_OK;
}

// Two pushes by dt one after the other, the positions after each stored
// (k_push_x's operations): the adjoint step's x1 and x2 from the recorded x0.
template <typename T>
__global__ void __launch_bounds__(256) k_push_x_twice(const T *__restrict__ x0, const T *__restrict__ y0,
                                                      const T *__restrict__ z0, const T *__restrict__ px,
                                                      const T *__restrict__ py, const T *__restrict__ pz,
                                                      const T *__restrict__ g_inv, T dt, int64_t Np,
                                                      T *__restrict__ x1, T *__restrict__ y1,
                                                      T *__restrict__ z1, T *__restrict__ x2,
                                                      T *__restrict__ y2, T *__restrict__ z2) {
  const int64_t ip = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (ip >= Np) return;
  const T dt_g = dt * g_inv[ip];
  const T dx = px[ip] * dt_g, dy = py[ip] * dt_g, dz = pz[ip] * dt_g;
  const T xa = x0[ip] + dx, ya = y0[ip] + dy, za = z0[ip] + dz;
  x1[ip] = xa;
  y1[ip] = ya;
  z1[ip] = za;
  x2[ip] = xa + dx;
  y2[ip] = ya + dy;
  z2[ip] = za + dz;
}
template <typename T>
static int push_x_twice(const T *x0, const T *y0, const T *z0, const T *px, const T *py, const T *pz,
                        const T *g_inv, T dt, int64_t Np, T *x1, T *y1, T *z1, T *x2, T *y2, T *z2,
                        void *stream) {
  if (Np < 0) return CHM_EINVAL;
  if (Np == 0) return CHM_OK;
  k_push_x_twice<T><<<chm_blocks(Np, 256), 256, 0, (hipStream_t)stream>>>(
      x0, y0, z0, px, py, pz, g_inv, dt, Np, x1, y1, z1, x2, y2, z2);
  CHM_CHECK_LAUNCH();
  return CHM_OK;
}
extern "C" int chm_push_x_twice_f64(const double *x0, const double *y0, const double *z0,
                                    const double *px, const double *py, const double *pz,
                                    const double *g_inv, double dt, int64_t Np, double *x1, double *y1,
                                    double *z1, double *x2, double *y2, double *z2, void *stream) {
  return push_x_twice<double>(x0, y0, z0, px, py, pz, g_inv, dt, Np, x1, y1, z1, x2, y2, z2, stream);
}
extern "C" int chm_push_x_twice_f32(const float *x0, const float *y0, const float *z0, const float *px,
                                    const float *py, const float *pz, const float *g_inv, float dt,
                                    int64_t Np, float *x1, float *y1, float *z1, float *x2, float *y2,
                                    float *z2, void *stream) {
  return push_x_twice<float>(x0, y0, z0, px, py, pz, g_inv, dt, Np, x1, y1, z1, x2, y2, z2, stream);
}

extern "C" int chm_push_x_f64(double *x, double *y, double *z, const double *px, const double *py,
                              const double *pz, const double *g_inv, double dt, int64_t Np,
                              void *stream) {
  return push_x<double>(x, y, z, px, py, pz, g_inv, dt, Np, stream);
}
extern "C" int chm_push_x_f32(float *x, float *y, float *z, const float *px, const float *py,
                              const float *pz, const float *g_inv, float dt, int64_t Np,
                              void *stream) {
  return push_x<float>(x, y, z, px, py, pz, g_inv, dt, Np, stream);
}

// ------------------------------------------------------------------ align
// data_align_dbl / data_align_int, particles_generic.cl:156-186:
// dst[i] = src[sort_indx[i]], i < n, for 8- or 4-byte elements.
template <typename E>
__global__ void __launch_bounds__(256) k_align(const uint32_t *__restrict__ idx, int64_t n,
                                               const E *__restrict__ src, E *__restrict__ dst) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) dst[i] = src[idx[i]];
}

extern "C" int chm_align_elems(const uint32_t *sort_indx, int64_t n, const void *src, void *dst,
                               int32_t elem_bytes, void *stream) {
  if (n < 0 || (elem_bytes != 4 && elem_bytes != 8) || (n > 0 && (!sort_indx || !src || !dst)) ||
      (src == dst && n > 0))
    return CHM_EINVAL;
  if (n == 0) return CHM_OK;
  hipStream_t st = (hipStream_t)stream;
  if (elem_bytes == 8)
    k_align<uint64_t><<<chm_blocks(n, 256), 256, 0, st>>>(sort_indx, n, (const uint64_t *)src,
                                                          (uint64_t *)dst);
  else
    k_align<uint32_t><<<chm_blocks(n, 256), 256, 0, st>>>(sort_indx, n, (const uint32_t *)src,
                                                          (uint32_t *)dst);
  CHM_CHECK_LAUNCH();
  return CHM_OK;
}

// Several arrays permuted by one launch: the slot's index is read once and
// the loads of all arrays are in flight together.
struct AlignSet {
  const void *src[CHM_ALIGN_MAXARR];
  void *dst[CHM_ALIGN_MAXARR];
  int eb[CHM_ALIGN_MAXARR];
  int narr;
};

__global__ void __launch_bounds__(256) k_align_multi(const uint32_t *__restrict__ idx, int64_t n,
                                                     AlignSet as) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const uint32_t p = idx[i];
  uint64_t v[CHM_ALIGN_MAXARR];
#pragma unroll
  for (int a = 0; a < CHM_ALIGN_MAXARR; a++)
    if (a < as.narr)
      v[a] = as.eb[a] == 8 ? ((const uint64_t *)as.src[a])[p]
                           : (uint64_t)((const uint32_t *)as.src[a])[p];
#pragma unroll
  for (int a = 0; a < CHM_ALIGN_MAXARR; a++)
    if (a < as.narr) {
      if (as.eb[a] == 8) ((uint64_t *)as.dst[a])[i] = v[a];
      else ((uint32_t *)as.dst[a])[i] = (uint32_t)v[a];
    }
}

extern "C" int chm_align_multi(const uint32_t *sort_indx, int64_t n, int32_t narr,
                               const void *const *src, void *const *dst,
                               const int32_t *elem_bytes, void *stream) {
  if (n < 0 || narr < 1 || narr > CHM_ALIGN_MAXARR || !src || !dst || !elem_bytes)
    return CHM_EINVAL;
  AlignSet as = {};
  as.narr = narr;
  for (int a = 0; a < narr; a++) {
    if ((elem_bytes[a] != 4 && elem_bytes[a] != 8) || (n > 0 && (!src[a] || !dst[a])))
      return CHM_EINVAL;
    as.src[a] = src[a];
    as.dst[a] = dst[a];
    as.eb[a] = elem_bytes[a];
  }
  // no destination may be read by the same launch
  for (int a = 0; a < narr; a++)
    for (int b = 0; b < narr; b++)
      if (n > 0 && (dst[a] == src[b] || (a != b && dst[a] == dst[b]))) return CHM_EINVAL;
  if (n == 0) return CHM_OK;
  if (!sort_indx) return CHM_EINVAL;
  k_align_multi<<<chm_blocks(n, 256), 256, 0, (hipStream_t)stream>>>(sort_indx, n, as);
  CHM_CHECK_LAUNCH();
  return CHM_OK;
}

// ------------------------------------------------------------------ keys
// Wave-aggregated increment: lanes with act and equal consecutive values form
// runs; a run of lanes i..j adds j + 1 - i as j + 1 at its last lane and -i
// at its first (lane i - 1 and i + 1 by DPP, no bit scans).
__device__ __forceinline__ void run_add(uint32_t *slot_base, bool act, uint32_t v, int lane) {
  const uint32_t rv = act ? v : 0xFFFFFFFFu;
  // wave_shr:1 / wave_shl:1; the lane shifted in keeps ~rv, never a neighbour
  const uint32_t below = (uint32_t)__builtin_amdgcn_update_dpp((int)~rv, (int)rv, 0x138, 0xF, 0xF, false);
  const uint32_t above = (uint32_t)__builtin_amdgcn_update_dpp((int)~rv, (int)rv, 0x130, 0xF, 0xF, false);
  const bool head = below != rv, tail = above != rv;
  if (act && (head || tail))
    atomicAdd(&slot_base[v], (tail ? (uint32_t)lane + 1u : 0u) - (head ? (uint32_t)lane : 0u));
}

// With PUSH, the coordinate push of push_xyz (same rounding order) is applied
// first and the key is taken from the pushed position.  Keys only: the cell
// offsets come from the sorted keys, so this pass has no atomics and its cost
// does not depend on the particles' order.
template <typename T, bool PUSH>
__global__ void __launch_bounds__(SORT_BS) k_cell_key(T *__restrict__ x, T *__restrict__ y,
                                                      T *__restrict__ z, const T *__restrict__ px,
                                                      const T *__restrict__ py, const T *__restrict__ pz,
                                                      const T *__restrict__ g_inv, T dt, int64_t Np,
                                                      int Nx, int Nr, T xmin, T dx_inv, T rmin, T dr_inv,
                                                      uint32_t *__restrict__ key_out) {
  const int Nx_loc = Nx - 1, Nr_loc = Nr - 1;
  const int64_t ip = (int64_t)blockIdx.x * SORT_BS + threadIdx.x;
  if (ip >= Np) return;
  T xp = x[ip], yp = y[ip], zp = z[ip];
  if (PUSH) {
    T dt_g = dt * g_inv[ip];
    T dx = px[ip] * dt_g;
    T dy = py[ip] * dt_g;
    T dz = pz[ip] * dt_g;
    xp = xp + dx;
    yp = yp + dy;
    zp = zp + dz;
    x[ip] = xp;
    y[ip] = yp;
    z[ip] = zp;
  }
  key_out[ip] = cell_key<T>(xp, yp, zp, Nx_loc, Nr_loc, xmin, dx_inv, rmin, dr_inv);
}

// ------------------------------------------------------------------ offsets
// cell_offset[c] = first sorted slot whose key is >= c, c = 0..nbins, and
// Np_stay = cell_offset[nbins - 1], the start of the out-of-domain bin.
// Slot s starts the cells key[s-1] < c <= key[s] (key[-1] = -1,
// key[Np] = nbins); these intervals partition 0..nbins.  A slot writes the
// cells of its interval, at most OFF_RUN of them; the rest of a longer
// interval (a long stretch of empty cells, e.g. the invalid last row before
// the out-of-domain bin) goes to a short list that k_offsets_gaps fills.  If
// the list overflows, k_offsets_gaps recomputes every cell by bisection.
// gl[0] = entries, gl[1] = overflow; both cleared earlier in the same stream
// (k_rs_colscan of the first LSD pass, or k_list_clear where there is none);
// entries (s, first cell, last cell) from gl[2].
#define OFF_RUN 32
#define OFF_LIST 1024

// OFF_PER consecutive slots per lane (two 16-byte key loads).
#define OFF_PER 8
__global__ void __launch_bounds__(256) k_offsets_bounds(const uint32_t *__restrict__ skey, int64_t Np,
                                                        int64_t nbins,
                                                        uint32_t *__restrict__ cell_offset,
                                                        uint32_t *__restrict__ np_stay,
                                                        uint32_t *__restrict__ gl) {
  const int64_t s0 = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * OFF_PER;
  if (s0 > Np) return;
  uint32_t kv[OFF_PER];
  if (s0 + OFF_PER <= Np) {
    const uint4 a = *(const uint4 *)(skey + s0), b = *(const uint4 *)(skey + s0 + 4);
    kv[0] = a.x; kv[1] = a.y; kv[2] = a.z; kv[3] = a.w;
    kv[4] = b.x; kv[5] = b.y; kv[6] = b.z; kv[7] = b.w;
  } else {
#pragma unroll
    for (int i = 0; i < OFF_PER; i++) kv[i] = s0 + i < Np ? skey[s0 + i] : 0u;
  }
  int64_t prev = s0 > 0 ? (int64_t)skey[s0 - 1] : -1;
#pragma unroll
  for (int i = 0; i < OFF_PER; i++) {
    const int64_t s = s0 + i;
    if (s > Np) break;
    const int64_t cur = s < Np ? (int64_t)kv[i] : nbins;
    if (cur > prev) {
      int64_t hi = cur;
      if (hi > prev + OFF_RUN) {
        hi = prev + OFF_RUN;
        const uint32_t e = atomicAdd(&gl[0], 1u);
        if (e < OFF_LIST) {
          gl[2 + 3 * e] = (uint32_t)s;
          gl[3 + 3 * e] = (uint32_t)(hi + 1);
          gl[4 + 3 * e] = (uint32_t)cur;
        } else {
          gl[1] = 1u;
        }
      }
      for (int64_t c = prev + 1; c <= hi; c++) {
        cell_offset[c] = (uint32_t)s;
        if (c == nbins - 1) *np_stay = (uint32_t)s;
      }
    }
    prev = cur;
  }
}

// Fixed grid; every lane strides over the listed cells (or, after an
// overflow of the list, over all cells with a bisection each).
__global__ void k_offsets_gaps(const uint32_t *__restrict__ skey, int64_t Np, int64_t nbins,
                               uint32_t *__restrict__ cell_offset, uint32_t *__restrict__ np_stay,
                               const uint32_t *__restrict__ gl) {
  const int64_t t0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t nt = (int64_t)gridDim.x * blockDim.x;
  if (gl[1] != 0u) {
    for (int64_t c = t0; c <= nbins; c += nt) {
      int64_t lo = 0, hi = Np;
      while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if ((int64_t)skey[mid] < c) lo = mid + 1;
        else hi = mid;
      }
      cell_offset[c] = (uint32_t)lo;
      if (c == nbins - 1) *np_stay = (uint32_t)lo;
    }
    return;
  }
  const uint32_t ne = gl[0] < OFF_LIST ? gl[0] : OFF_LIST;
  for (uint32_t e = 0; e < ne; e++) {
    const uint32_t sv = gl[2 + 3 * e];
    const int64_t c0 = gl[3 + 3 * e], c1 = gl[4 + 3 * e];
    for (int64_t c = c0 + t0; c <= c1; c += nt) {
      cell_offset[c] = sv;
      if (c == nbins - 1) *np_stay = sv;
    }
  }
}

__global__ void k_list_clear(uint32_t *__restrict__ gl) { gl[threadIdx.x] = 0u; }

// ------------------------------------------------------------------ radix sort
// A pass of digits of nbits <= RB bits over tiles of NT * RS_ITEMS items:
//   k_rs_upsweep    the tile's digit counts, counts[tile * nd + d] (16 bits: a
//                   tile holds at most 16384 items)
//   k_rs_colscan    offs[tile * nd + d] = items with digit d in earlier tiles,
//                   and the digit totals
//   k_rs_plan       the digits' first positions (and, for the second pass of
//                   the bucket sort, the tiles of every bucket)
//   k_rs_downsweep  the stable scatter
// SECOND: the second pass of the bucket sort.  Its tiles do not cross the
// buckets the first pass made; tile -> bucket from tmap.
// The count rows of a bucket of many tiles (a beam in a few grid rows, a
// species that has left the grid) would be walked one by one by k_rs_cells:
// the tiles are also counted in chunks of RS_CHUNK, chunk c = tiles c RS_CHUNK
// and on, a row of counts for each chunk that lies inside one bucket.
#define RS_CHUNK 32u
struct RsTiles {
  const uint32_t *tmap, *tfirst, *hbase;  // SECOND only
  int nbk;
  uint32_t per;  // > 0: consecutive tiles on one XCD, per of them on each
  uint32_t *chunk;  // rows of the chunks; the first pass clears them
  uint32_t nchunk;  // chunks that the tiles can make
};
// whether chunk c lies inside the bucket, whose tiles are [t0, t1)
__device__ __forceinline__ bool in_bucket(uint32_t c, uint32_t t0, uint32_t t1) {
  return c * RS_CHUNK >= t0 && (c + 1u) * RS_CHUNK <= t1;
}
// items [first, end) of a tile, and the tiles [t0, t1) of its bucket; false
// when the block has none
template <bool SECOND, int TILE>
__device__ __forceinline__ bool tile_range(const RsTiles &tl, int64_t n, uint32_t &tile, int64_t &first,
                                           int64_t &end, uint32_t &bucket, uint32_t &t0, uint32_t &t1) {
  tile = blockIdx.x;
  if (SECOND && tl.per) tile = (blockIdx.x & 7) * tl.per + (blockIdx.x >> 3);
  if constexpr (SECOND) {
    if (tile >= tl.tfirst[tl.nbk]) return false;
    bucket = tl.tmap[tile];
    const uint32_t b0 = tl.hbase[bucket], b1 = tl.hbase[bucket + 1];
    t0 = tl.tfirst[bucket];
    t1 = t0 + (b1 - b0 + TILE - 1u) / TILE;
    first = (int64_t)b0 + (int64_t)(tile - t0) * TILE;
    end = first + TILE < b1 ? first + TILE : b1;
  } else {
    bucket = t0 = t1 = 0;
    first = (int64_t)tile * TILE;
    end = first + TILE < n ? first + TILE : n;
  }
  return true;
}

template <int RB, int NT, bool SECOND, typename K>
__global__ void __launch_bounds__(NT) k_rs_upsweep(const K *__restrict__ keys, int64_t n, int shift,
                                                   int nbits, uint16_t *__restrict__ counts, RsTiles tl) {
  constexpr int NB = 1 << RB;
  __shared__ uint32_t h[RS_COPIES][NB + RS_PAD];
  int64_t first, end;
  uint32_t bucket, tile, t0, t1;
  if (!tile_range<SECOND, NT * RS_ITEMS>(tl, n, tile, first, end, bucket, t0, t1)) return;
  const int nd = 1 << nbits;
  const uint32_t mask = (uint32_t)nd - 1u;
  const int lane = threadIdx.x & 63;
  uint32_t kk[RS_ITEMS];
#pragma unroll
  for (int i = 0; i < RS_ITEMS; i++) {
    const int64_t idx = first + (int64_t)i * NT + threadIdx.x;
    kk[i] = idx < end ? (uint32_t)keys[idx] : 0u;
  }
  if (!SECOND && tl.nchunk) {
    // (rows of the second pass's digits)
    const int64_t words = (int64_t)tl.nchunk << RB;
    for (int64_t e = (int64_t)tile * NT + threadIdx.x; e < words; e += (int64_t)gridDim.x * NT) tl.chunk[e] = 0u;
  }
  for (int e = threadIdx.x; e < RS_COPIES * (NB + RS_PAD); e += NT) (&h[0][0])[e] = 0;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < RS_ITEMS; i++) {
    const int64_t idx = first + (int64_t)i * NT + threadIdx.x;
    run_add(h[lane & (RS_COPIES - 1)], idx < end, (kk[i] >> shift) & mask, lane);
  }
  __syncthreads();
  auto total = [&](int d) {
    uint32_t c = 0;
#pragma unroll
    for (int q = 0; q < RS_COPIES; q++) c += h[q][d];
    return c;
  };
  for (int d = threadIdx.x; d < nd; d += NT) counts[(int64_t)tile * nd + d] = (uint16_t)total(d);
  if (SECOND && in_bucket(tile / RS_CHUNK, t0, t1)) {
    uint32_t *row = tl.chunk + (int64_t)(tile / RS_CHUNK) * nd;
    for (int d = threadIdx.x; d < nd; d += NT)
      if (const uint32_t c = total(d)) atomicAdd(&row[d], c);
  }
}

// Lanes of the wave holding the same digit d (among the active ones): one
// ballot for each digit bit that is not the same in the whole wave.  The keys
// are nearly sorted in earnest, so these are few; finding them is a
// reduction over the wave by DPP.
__device__ __forceinline__ uint2 match_peers(uint32_t d, bool act) {
  const unsigned long long am = __ballot(act);
  uint32_t lo = (uint32_t)am, hi = (uint32_t)(am >> 32);
  const uint32_t d0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)d);  // active lanes are a prefix
  uint32_t x = act ? d ^ d0 : 0u;
#define OR_DPP(ctrl, rows) x |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, ctrl, rows, 0xF, false)
  OR_DPP(0x111, 0xF);  // row_shr:1, 2, 4, 8: lane 15 of each row of 16
  OR_DPP(0x112, 0xF);
  OR_DPP(0x114, 0xF);
  OR_DPP(0x118, 0xF);
  OR_DPP(0x142, 0xA);  // row_bcast:15, row_bcast:31: lane 63
  OR_DPP(0x143, 0xC);
#undef OR_DPP
  uint32_t vary = (uint32_t)__builtin_amdgcn_readlane((int)x, 63);
  while (vary) {
    const int b = __builtin_ctz(vary);
    vary &= vary - 1u;
    const uint32_t m = (uint32_t)__builtin_amdgcn_sbfe((int)d, b, 1);
    const unsigned long long bal = __ballot(m != 0u);
    lo &= ~(m ^ (uint32_t)bal);
    hi &= ~(m ^ (uint32_t)(bal >> 32));
  }
  return make_uint2(lo, hi);
}

// Exclusive prefix over the block of one value per thread (NT threads).
template <int NT> __device__ __forceinline__ uint32_t block_excl_scan(uint32_t v, uint32_t *wsum) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint32_t inc = v;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const uint32_t t = (uint32_t)__shfl_up((int)inc, d);
    if (lane >= d) inc += t;
  }
  if (lane == 63) wsum[wave] = inc;
  __syncthreads();
  uint32_t wpre = 0;
  for (int w = 0; w < wave; w++) wpre += wsum[w];
  __syncthreads();
  return wpre + inc - v;
}

// The digits' first positions from their totals (nd <= 2048, in total[]),
// by one block of 1024 threads.  With tmap, the tiles of `tile2` items of
// every bucket: tfirst[h] = first tile, tmap[tile] = h.  With cell_offset (a
// sort of a single pass), the digits are the cells themselves.
struct RsPlanOut {
  uint32_t *hbase, *tfirst, *tmap, *cell_offset, *np_stay;
  int64_t nbins;
  int tile2;
};
__device__ __forceinline__ void rs_plan_block(const uint32_t *total, int nd, const RsPlanOut &o,
                                              uint32_t *wsum) {
  const int t = threadIdx.x;
  uint32_t c[2], nt[2];
#pragma unroll
  for (int i = 0; i < 2; i++) {
    c[i] = 2 * t + i < nd ? total[2 * t + i] : 0u;
    nt[i] = o.tmap ? (c[i] + (uint32_t)o.tile2 - 1u) / (uint32_t)o.tile2 : 0u;
  }
  uint32_t pos = block_excl_scan<1024>(c[0] + c[1], wsum);
  uint32_t tile = o.tmap ? block_excl_scan<1024>(nt[0] + nt[1], wsum) : 0u, at[2] = {0u, 0u};
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const int d = 2 * t + i;
    if (d < nd) {
      o.hbase[d] = pos;
      if (o.cell_offset && d <= o.nbins) {
        o.cell_offset[d] = pos;
        if (d == o.nbins - 1) *o.np_stay = pos;
      }
      if (o.tmap) {
        o.tfirst[d] = tile;
        if (nt[i] <= RS_CHUNK)
          for (uint32_t k = 0; k < nt[i]; k++) o.tmap[tile + k] = (uint32_t)d;
        at[i] = tile;
        tile += nt[i];
      }
      pos += c[i];
      if (d == nd - 1) {
        o.hbase[nd] = pos;
        if (o.tmap) o.tfirst[nd] = tile;
        if (o.cell_offset && nd == o.nbins) o.cell_offset[nd] = pos;
      }
    }
  }
  // buckets of many tiles: the whole wave fills their part of the map
  const int lane = t & 63;
#pragma unroll
  for (int i = 0; i < 2; i++)
    for (unsigned long long big = __ballot(nt[i] > RS_CHUNK); big; big &= big - 1) {
      const int l = __ffsll(big) - 1;
      const uint32_t n = (uint32_t)__shfl((int)nt[i], l), a = (uint32_t)__shfl((int)at[i], l);
      for (uint32_t k = lane; k < n; k += 64) o.tmap[a + k] = (uint32_t)(2 * (t - lane + l) + i);
    }
}

// Column scan of the tile counts: a block of 1024 threads takes db digits,
// 1024 / db groups of consecutive tiles each.  A launch of a single block
// (db = nd) also runs the plan: for a few tiles the launches are what a pass
// costs (60 tiles: six launches instead of fourteen a sort).
__global__ void __launch_bounds__(1024) k_rs_colscan(const uint16_t *__restrict__ counts, int64_t nblk,
                                                     int nbits, int db, uint32_t *__restrict__ offs,
                                                     uint32_t *__restrict__ total, RsPlanOut plan,
                                                     uint32_t *__restrict__ clear) {
  __shared__ uint32_t part[1024], tot[1024], wsum[16];
  const int nd = 1 << nbits, t = threadIdx.x, dl = t & (db - 1), grp = t / db, ng = 1024 / db;
  const int d = blockIdx.x * db + dl;
  if (clear && blockIdx.x == 0 && t < 2) clear[t] = 0u;
  const int64_t per = (nblk + ng - 1) / ng;
  const int64_t t0 = grp * per, t1 = t0 + per < nblk ? t0 + per : nblk;
  uint32_t s = 0;
#pragma unroll 8
  for (int64_t i = t0; i < t1; i++) s += counts[i * nd + d];
  part[t] = s;
  __syncthreads();
  uint32_t run = 0;
  for (int q = 0; q < grp; q++) run += part[q * db + dl];
  if (grp == ng - 1) {
    tot[dl] = run + s;
    total[d] = run + s;
  }
#pragma unroll 8
  for (int64_t i = t0; i < t1; i++) {
    const uint32_t v = counts[i * nd + d];
    offs[i * nd + d] = run;
    run += v;
  }
  if (gridDim.x == 1) {
    __syncthreads();
    rs_plan_block(tot, nd, plan, wsum);
  }
}

__global__ void __launch_bounds__(1024) k_rs_plan(const uint32_t *__restrict__ total, int nd,
                                                  RsPlanOut plan) {
  __shared__ uint32_t wsum[16];
  rs_plan_block(total, nd, plan, wsum);
}

// Second pass of the bucket sort, one block per bucket, then one per chunk:
// the first slot of each of the bucket's cells (cell_offset itself) and, per
// tile, the slots its items of each cell start at.  The block of a bucket
// writes those of the tiles outside the bucket's chunks, the block of a chunk
// those of its tiles.  A bucket of T tiles is thus T / RS_CHUNK + 2 RS_CHUNK
// rows one after the other, not 2 T.  Sorts, us, by one block a bucket -> this
// (LSD passes): 67M keys in one grid row 2862 -> 659 (1543), 90% outside the
// grid 2593 -> 658 (832), 30% 1244 -> 628 (972), over the whole grid 556 (982);
// 4.2M in four rows 245 -> 107 (152), 90% outside 325 -> 87 (84).
__global__ void __launch_bounds__(1024) k_rs_cells(const uint16_t *__restrict__ counts, int nbits,
                                                   RsTiles tl, int nbk, uint32_t *__restrict__ offs,
                                                   uint32_t *__restrict__ cell_offset,
                                                   uint32_t *__restrict__ np_stay, int64_t nbins,
                                                   int64_t Np) {
  __shared__ uint32_t wsum[16];
  const int nd = 1 << nbits, t = threadIdx.x;
  int h = blockIdx.x;
  const bool own = h >= nbk;  // a chunk's block
  const uint32_t mine = own ? (uint32_t)(h - nbk) : 0u;
  if (own) {
    if ((mine + 1u) * RS_CHUNK > tl.tfirst[tl.nbk]) return;
    h = (int)tl.tmap[mine * RS_CHUNK];
  }
  const uint32_t t0 = tl.tfirst[h], t1 = tl.tfirst[h + 1];
  if (own && !in_bucket(mine, t0, t1)) return;
  // tiles [t0, ta), chunks [ca, cb), tiles [tb, t1)
  uint32_t ca = (t0 + RS_CHUNK - 1u) / RS_CHUNK, cb = t1 / RS_CHUNK, ta = ca * RS_CHUNK, tb = cb * RS_CHUNK;
  if (ca >= cb) {
    ca = cb = 0u;
    ta = tb = t1;
  }
  // two adjacent digits a thread
  uint32_t c[2] = {0u, 0u}, before[2] = {0u, 0u};
  const bool on = 2 * t < nd;
  auto count = [&](uint32_t i) { return *(const uint32_t *)(counts + (int64_t)i * nd + 2 * t); };
  auto chunk = [&](uint32_t i) { return *(const uint2 *)(tl.chunk + (int64_t)i * nd + 2 * t); };
  if (on) {
#pragma unroll 4
    for (uint32_t i = t0; i < ta; i++) {
      const uint32_t v = count(i);
      c[0] += v & 0xFFFFu;
      c[1] += v >> 16;
    }
#pragma unroll 4
    for (uint32_t i = ca; i < cb; i++) {
      const uint2 v = chunk(i);
      if (i == mine) {
        before[0] = c[0];
        before[1] = c[1];
      }
      c[0] += v.x;
      c[1] += v.y;
    }
#pragma unroll 4
    for (uint32_t i = tb; i < t1; i++) {
      const uint32_t v = count(i);
      c[0] += v & 0xFFFFu;
      c[1] += v >> 16;
    }
  }
  uint32_t pos = block_excl_scan<1024>(c[0] + c[1], wsum) + tl.hbase[h];
  if (blockIdx.x == 0 && t == 0) cell_offset[nbins] = (uint32_t)Np;
  if (!on) return;
  uint32_t run[2] = {pos, pos + c[0]};
  auto place = [&](uint32_t i) {
    const uint32_t v = count(i);
    *(uint2 *)(offs + (int64_t)i * nd + 2 * t) = make_uint2(run[0], run[1]);
    run[0] += v & 0xFFFFu;
    run[1] += v >> 16;
  };
  if (own) {
    run[0] += before[0];
    run[1] += before[1];
#pragma unroll 4
    for (uint32_t i = mine * RS_CHUNK; i < (mine + 1u) * RS_CHUNK; i++) place(i);
    return;
  }
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const int64_t cell = ((int64_t)h << nbits) + 2 * t + i;
    if (cell < nbins) {
      cell_offset[cell] = run[i];
      if (cell == nbins - 1) *np_stay = run[i];
    }
  }
#pragma unroll 4
  for (uint32_t i = t0; i < ta; i++) place(i);
  if (tb < t1) {
#pragma unroll 4
    for (uint32_t i = ca; i < cb; i++) {
      const uint2 v = chunk(i);
      run[0] += v.x;
      run[1] += v.y;
    }
  }
#pragma unroll 4
  for (uint32_t i = tb; i < t1; i++) place(i);
}

// Stable scatter of one tile of NT * IT items.  Wave w owns the tile's items
// w*IT*64 .. (w+1)*IT*64 - 1, visited in index order (round r,
// lane l: item r*64 + l of the wave's range).  Counting loop: each wave counts
// its digits (one LDS add per set of equal digits of a round), which gives
// every item its place among the wave's items of its digit; with the counts
// of the waves and digits before it, its place in the tile's own sorted
// order.  The items then go through LDS into that order, keys first and
// indices after them through the same words, and consecutive lanes write
// consecutive slots: written straight from the counting order the scatter is
// bound by the number of separate L2 writes, up to one per item and array.
// Within a wave LDS operations take effect in order.  The waves' counts and
// positions are 16 bits, two digits a word (at most 16384 items a tile).
// MODE 0: one pass of an LSD sort (32-bit keys out).
// MODE 1: first pass of the bucket sort: the low `shift` bits go out in 16
//         bits, the digit is implied by the position from here on.
// MODE 2: second pass: 16-bit keys in, full keys out.
template <int RB, int NT, int IT, int MODE>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(NT == 1024 ? 8 : 6))) k_rs_downsweep(
    const void *__restrict__ kin_, const uint32_t *__restrict__ vin, int64_t n, int shift, int nbits,
    const uint32_t *__restrict__ offs, const uint32_t *__restrict__ hbase, void *__restrict__ kout_,
    uint32_t *__restrict__ vout, RsTiles tl) {
  typedef typename std::conditional<MODE == 2, uint16_t, uint32_t>::type KI;
  constexpr int NB = 1 << RB;
  constexpr int NW = NT / CHM_WAVE;
  constexpr int TILE = NT * IT;
  constexpr int WORDS = NW * (NB / 2) > TILE ? NW * (NB / 2) : TILE;
  constexpr int WPT = (NB / 2 + NT - 1) / NT;  // count words a thread sums
  __shared__ uint32_t buf[WORDS];
  __shared__ uint32_t base[NB];
  __shared__ uint32_t wsum[NW];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int64_t first, end;
  uint32_t bucket, tile, t0, t1;
  if (!tile_range<MODE == 2, TILE>(tl, n, tile, first, end, bucket, t0, t1)) return;
  const int nd = 1 << nbits;
  const uint32_t mask = (uint32_t)nd - 1u;
  const int sh = MODE == 2 ? 0 : shift;
  // the wave's items, by 32-bit offsets from a scalar base
  const int64_t wbase = first + (int64_t)wave * (IT * CHM_WAVE);
  const int lim = (int)(end - wbase < IT * CHM_WAVE ? end - wbase : IT * CHM_WAVE) - lane;
  const KI *kin = (const KI *)kin_ + wbase;
  const bool given = MODE == 2 || (MODE == 0 && vin);  // else the index is the position
  uint32_t kk[IT], vv[IT], rc[IT / 2];
#pragma unroll
  for (int r = 0; r < IT; r++)
    kk[r] = r * CHM_WAVE < lim ? (uint32_t)kin[r * CHM_WAVE + lane] : 0u;
  if (given) {
    const uint32_t *vi = vin + wbase;
#pragma unroll
    for (int r = 0; r < IT; r++) vv[r] = r * CHM_WAVE < lim ? vi[r * CHM_WAVE + lane] : 0u;
  }
  for (int e = tid; e < NW * (NB / 2); e += NT) buf[e] = 0u;
  __syncthreads();
  uint32_t *h = buf + wave * (NB / 2);
#pragma unroll
  for (int r = 0; r < IT; r++) {
    const bool act = r * CHM_WAVE < lim;
    const uint32_t d = (kk[r] >> sh) & mask;
    const uint2 peers = match_peers(d, act);
    const uint32_t rank = __builtin_amdgcn_mbcnt_hi(peers.y, __builtin_amdgcn_mbcnt_lo(peers.x, 0u));
    // the first lane of each digit adds the digit's lanes to the wave's count
    // and hands the count before it to the others
    uint32_t old = 0;
    if (act && rank == 0)
      old = atomicAdd(&h[d >> 1], (uint32_t)(__popc(peers.x) + __popc(peers.y)) << ((d & 1) * 16));
    const int head = peers.x ? __ffs((int)peers.x) - 1 : 31 + __ffs((int)peers.y);
    old = (uint32_t)__builtin_amdgcn_ds_bpermute(head << 2, (int)old);
    const uint32_t v = ((old >> ((d & 1) * 16)) & 0xFFFFu) + rank;
    rc[r >> 1] = (r & 1) ? rc[r >> 1] | (v << 16) : v;
    if (r & 1) __asm__ __volatile__("" : "+v"(rc[r >> 1]));
  }
  __syncthreads();
  // counts -> places in the tile's sorted order; base[] = slot of the tile's
  // sorted item 0, were all of its items of this digit
  uint32_t sum[WPT], tot = 0;
#pragma unroll
  for (int i = 0; i < WPT; i++) {
    const int e = tid * WPT + i;
    sum[i] = 0;
    if (e < nd / 2) {
#pragma unroll
      for (int w = 0; w < NW; w++) {
        const uint32_t c = buf[w * (NB / 2) + e];
        buf[w * (NB / 2) + e] = sum[i];
        sum[i] += c;
      }
    }
    tot += (sum[i] & 0xFFFFu) + (sum[i] >> 16);
  }
  uint32_t ex = block_excl_scan<NT>(tot, wsum);
#pragma unroll
  for (int i = 0; i < WPT; i++) {
    const int e = tid * WPT + i;
    if (e < nd / 2) {
      const uint32_t e0 = ex, e1 = ex + (sum[i] & 0xFFFFu);
#pragma unroll
      for (int w = 0; w < NW; w++) buf[w * (NB / 2) + e] += e0 | (e1 << 16);
      uint2 o = *(const uint2 *)(offs + (int64_t)tile * nd + 2 * e);
      if (MODE != 2) {
        o.x += hbase[2 * e];
        o.y += hbase[2 * e + 1];
      }
      base[2 * e] = o.x - e0;
      base[2 * e + 1] = o.y - e1;
      ex = e1 + (sum[i] >> 16);
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < IT; r++) {
    // the digit is formed again: kept from the counting loop, digits and LDS
    // addresses are 64 registers, spilled
    __asm__ __volatile__("" : "+v"(kk[r]));
    const uint32_t d = (kk[r] >> sh) & mask;
    const uint32_t at = (h[d >> 1] >> ((d & 1) * 16)) & 0xFFFFu;
    rc[r >> 1] += (r & 1) ? at << 16 : at;
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < IT; r++)
    if (r * CHM_WAVE < lim) buf[(rc[r >> 1] >> ((r & 1) * 16)) & 0xFFFFu] = kk[r];
  __syncthreads();
  const int cnt = (int)(end - first) - tid;
#pragma unroll
  for (int r = 0; r < IT; r++) {
    const uint32_t k = buf[r * NT + tid];
    const uint32_t dest = base[(k >> sh) & mask] + (uint32_t)(r * NT + tid);
    kk[r] = dest;
    if (r * NT < cnt) {
      if (MODE == 1) ((uint16_t *)kout_)[dest] = (uint16_t)(k & ((1u << shift) - 1u));
      else if (MODE == 2) ((uint32_t *)kout_)[dest] = (bucket << nbits) | k;
      else ((uint32_t *)kout_)[dest] = k;
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < IT; r++)
    if (r * CHM_WAVE < lim)
      buf[(rc[r >> 1] >> ((r & 1) * 16)) & 0xFFFFu] =
          given ? vv[r] : (uint32_t)wbase + (uint32_t)(r * CHM_WAVE + lane);
  __syncthreads();
#pragma unroll
  for (int r = 0; r < IT; r++)
    if (r * NT < cnt) vout[kk[r]] = buf[r * NT + tid];
}

// How keys of `bits` bits are sorted (n items, nbins bins):
//   one pass up to 11 bits: the digit is the cell, cell_offset comes from the
//     digit totals;
//   bucket sort up to 22 bits (nbk > 0): a stable pass over the high bits,
//     then one over the low `lo` bits inside each bucket.  The particles are
//     nearly in cell order in earnest, so both passes write long runs (an LSD
//     sort scatters by the low bits first: every tile writes to hundreds of
//     places in both passes); the second pass carries 16-bit keys, and
//     cell_offset comes from its counts.  Not where the buckets would hold
//     less than half a tile of 4096 on average (few particles on many cells:
//     the tiles' count rows would be the most of the work and the workspace);
//   LSD passes of at most 11 bits (8 up to 16 bits) otherwise.
struct RsPlan {
  int npass, rb, nb[3], nbk, lo, nt1, nt2;
};
static RsPlan rs_plan(int bits, int64_t n, int64_t nbins) {
  RsPlan p = {};
  if (bits < 1) bits = 1;
  p.rb = bits <= 8 || (bits > 11 && bits <= 16) ? 8 : 11;
  p.nt1 = p.nt2 = n >= RS_BIG ? RS_NT1 : 256;
  if (bits <= 11) {
    p.npass = 1;
    p.nb[0] = bits;
    return p;
  }
  if (bits <= 22) {
    const int lo = p.rb;
    const int64_t nbk = (nbins + ((int64_t)1 << lo) - 1) >> lo;
    if (n >= RS_BUCKET * nbk) {
      p.npass = 2;
      p.nbk = (int)nbk;
      p.lo = lo;
      p.nb[0] = bits - lo;
      p.nb[1] = lo;
      p.nt2 = n >= RS_BIG && n >= RS_TILES2 * nbk ? RS_NT2 : 256;
      return p;
    }
  }
  p.npass = bits <= 22 ? 2 : 3;
  int left = bits;
  for (int i = 0; i < p.npass; i++) {
    int w = (left + (p.npass - i) - 1) / (p.npass - i);
    p.nb[i] = w;
    left -= w;
  }
  return p;
}
static int key_bits(int64_t nbins) {
  int bits = 0;
  while (((int64_t)1 << bits) < nbins) bits++;  // keys are < nbins
  return bits < 1 ? 1 : bits;
}

// ------------------------------------------------------------------ driver
struct SortWs {
  uint16_t *counts, *low;
  uint32_t *offs, *total, *hbase, *tfirst, *tmap, *kA, *kB, *vA, *vB, *trunc;
  int64_t nblk, ntile2;
};

static size_t sort_layout(int64_t Np, int64_t nbins, SortWs *w, void *base) {
  const RsPlan plan = rs_plan(key_bits(nbins), Np, nbins);
  const int64_t tile1 = plan.nt1 * RS_ITEMS, tile2 = plan.nt2 * RS_ITEMS;
  int64_t nblk = (Np + tile1 - 1) / tile1;
  if (nblk < 1) nblk = 1;
  const int64_t nd1 = (int64_t)1 << (plan.nbk ? plan.nb[0] : plan.rb);
  const int64_t ntile2 = plan.nbk ? Np / tile2 + plan.nbk : 0;
  // the second pass's count rows take the place of the first's
  const int64_t c1 = nd1 * nblk, c2 = ntile2 << plan.nb[1];
  const int64_t ncounts = c1 > c2 ? c1 : c2;
  size_t off = 0;
  size_t o_counts = off; off += chm_align(ncounts * 2);
  size_t o_offs = off; off += chm_align(ncounts * 4);
  size_t o_total = off; off += chm_align(nd1 * 4);
  size_t o_hbase = off; off += chm_align((nd1 + 1) * 4);
  size_t o_tfirst = off; off += chm_align((nd1 + 1) * 4);
  size_t o_tmap = off; off += chm_align((ntile2 + 1) * 4);
  // sorted keys, and what lies between the passes: 16-bit keys and indices
  // of the bucket sort, or a second pair of buffers
  size_t o_kA = off; off += chm_align(Np * 4);
  size_t o_kB = off; off += chm_align(plan.npass == 1 ? 0 : plan.nbk ? Np * 2 : Np * 4);
  size_t o_vA = off; off += chm_align(plan.npass == 1 ? 0 : Np * 4);
  size_t o_vB = off; off += chm_align(plan.npass > 2 ? Np * 4 : 0);
  size_t o_t = off; off += chm_align((2 + 3 * OFF_LIST) * 4);
  if (w) {
    char *b = (char *)base;
    w->counts = (uint16_t *)(b + o_counts);
    w->offs = (uint32_t *)(b + o_offs);
    w->total = (uint32_t *)(b + o_total);
    w->hbase = (uint32_t *)(b + o_hbase);
    w->tfirst = (uint32_t *)(b + o_tfirst);
    w->tmap = (uint32_t *)(b + o_tmap);
    w->kA = (uint32_t *)(b + o_kA);
    w->kB = (uint32_t *)(b + o_kB);
    w->low = (uint16_t *)(b + o_kB);
    w->vA = (uint32_t *)(b + o_vA);
    w->vB = (uint32_t *)(b + o_vB);
    w->trunc = (uint32_t *)(b + o_t);
    w->nblk = nblk;
    w->ntile2 = ntile2;
  }
  return off;
}

// Enough for every sort of up to Np keys: the layout grows with the keys as
// long as the plan stays the same, and may shrink where rs_plan goes over to
// the next one, so the last number of keys of each plan counts too.
extern "C" size_t chm_sort_workspace_bytes(int64_t Np, int64_t nbins) {
  size_t need = sort_layout(Np, nbins, nullptr, nullptr);
  const int lo = rs_plan(key_bits(nbins), (int64_t)1 << 40, nbins).lo;
  const int64_t nbk = lo ? (nbins + ((int64_t)1 << lo) - 1) >> lo : 0;
  for (const int64_t next : {RS_BIG, RS_BUCKET * nbk, RS_TILES2 * nbk})
    if (next > 1 && next <= Np) {
      const size_t n = sort_layout(next - 1, nbins, nullptr, nullptr);
      need = n > need ? n : need;
    }
  return need;
}

// Stage 1: the cell keys (+ the push with PUSH).
template <typename T, bool PUSH>
static int sort_keys(T *x, T *y, T *z, const T *px, const T *py, const T *pz, const T *g_inv, T dt,
                     int64_t Np, const chm_grid_t *g, uint32_t *indx_in_cell, void *ws, size_t ws_bytes,
                     void *stream) {
  if (!g || Np < 0 || Np > 0x7FFFFFF0ll || g->Nx < 4 || g->Nr < 3) return CHM_EINVAL;
  int64_t nbins = (int64_t)(g->Nx - 1) * (g->Nr - 1) + 1;
  SortWs w;
  if (sort_layout(Np, nbins, &w, ws) > ws_bytes || !ws) return CHM_EWORKSPACE;
  hipStream_t st = (hipStream_t)stream;
  if (Np > 0)
    k_cell_key<T, PUSH><<<chm_blocks(Np, SORT_BS), SORT_BS, 0, st>>>(
        x, y, z, px, py, pz, g_inv, dt, Np, g->Nx, g->Nr, (T)g->xmin, (T)g->dx_inv, (T)g->rmin,
        (T)g->dr_inv, indx_in_cell);
  CHM_CHECK_LAUNCH();
  return CHM_OK;
}

template <int RB, int NT, int IT, int MODE>
static void rs_scatter(const void *kin, const uint32_t *vin, int64_t n, int shift, int nbits,
                       const SortWs &w, void *kout, uint32_t *vout, const RsTiles &tl, int64_t nblk,
                       hipStream_t st) {
  k_rs_downsweep<RB, NT, IT, MODE><<<(unsigned)nblk, NT, 0, st>>>(kin, vin, n, shift, nbits, w.offs, w.hbase,
                                                              kout, vout, tl);
}
template <int MODE>
static void rs_scatter(const RsPlan &p, int nt, const void *kin, const uint32_t *vin, int64_t n,
                       int shift, int nbits, const SortWs &w, void *kout, uint32_t *vout,
                       const RsTiles &tl, int64_t nblk, hipStream_t st) {
  constexpr int NTB = MODE == 2 ? RS_NT2 : RS_NT1;
#define DOWN(RB, NT, IT) \
  rs_scatter<RB, NT, IT, MODE>(kin, vin, n, shift, nbits, w, kout, vout, tl, nblk, st)
  // tiles of 4096: what a tile costs is the serial counting of its waves'
  // items, so the fewer tiles there are the more waves share one (sorts of
  // 250 thousand, 1.0 and 3.0 million keys: 36.8, 46.3, 76.7 us with 256 threads
  // of 16 items; 31.4, 39.6, 75.0 with 512 of 8; 29.7, 41.7, 76.0 with 1024
  // of 4)
  const bool few = nblk <= 128;
  if (p.rb == 8 && nt == 256 && few) DOWN(8, 1024, 4);
  else if (p.rb == 8 && nt == 256) DOWN(8, 512, 8);
  else if (p.rb == 8) DOWN(8, NTB, RS_ITEMS);
  else if (nt == 256 && few) DOWN(11, 1024, 4);
  else if (nt == 256) DOWN(11, 512, 8);
  else DOWN(11, NTB, RS_ITEMS);
#undef DOWN
}
template <bool SECOND, typename K>
static void rs_count(const RsPlan &p, int nt, const K *kin, int64_t n, int shift, int nbits,
                     const SortWs &w, const RsTiles &tl, int64_t nblk, hipStream_t st) {
  constexpr int NTB = SECOND ? RS_NT2 : RS_NT1;
#define UP(RB, NT) \
  k_rs_upsweep<RB, NT, SECOND, K><<<(unsigned)nblk, NT, 0, st>>>(kin, n, shift, nbits, w.counts, tl)
  if (p.rb == 8 && nt == 256) UP(8, 256);
  else if (p.rb == 8) UP(8, NTB);
  else if (nt == 256) UP(11, 256);
  else UP(11, NTB);
#undef UP
}

// Column scan and plan of a pass: one launch where the count matrix is small.
static void rs_scan(int64_t nblk, int nbits, const SortWs &w, const RsPlanOut &po, uint32_t *clear,
                    hipStream_t st) {
  const int nd = 1 << nbits;
  if (nd <= 1024 && nblk * nd <= 32768) {
    k_rs_colscan<<<1, 1024, 0, st>>>(w.counts, nblk, nbits, nd, w.offs, w.total, po, clear);
    return;
  }
  const int db = nd < 32 ? nd : 32;
  // a launch of one block runs the plan itself
  k_rs_colscan<<<nd / db, 1024, 0, st>>>(w.counts, nblk, nbits, db, w.offs, w.total, po, clear);
  if (nd / db > 1) k_rs_plan<<<1, 1024, 0, st>>>(w.total, nd, po);
}

// Stage 2: the stable sort of the keys of stage 1 and the cell offsets.
static int sort_from_keys(int64_t Np, const chm_grid_t *g, const uint32_t *indx_in_cell,
                          uint32_t *cell_offset, uint32_t *sort_indx, uint32_t *np_stay, void *ws,
                          size_t ws_bytes, void *stream) {
  if (!g || Np < 0 || Np > 0x7FFFFFF0ll || g->Nx < 4 || g->Nr < 3) return CHM_EINVAL;
  int64_t nbins = (int64_t)(g->Nx - 1) * (g->Nr - 1) + 1;
  SortWs w;
  if (sort_layout(Np, nbins, &w, ws) > ws_bytes || !ws) return CHM_EWORKSPACE;
  hipStream_t st = (hipStream_t)stream;
  const RsPlan plan = rs_plan(key_bits(nbins), Np, nbins);
  RsTiles tl = {w.tmap, w.tfirst, w.hbase, plan.nbk, 0u, nullptr, 0u};
  if (Np > 0 && plan.nbk) {
    // The chunk rows are where the second scatter, after their last use,
    // leaves the sorted keys: ntile2 / RS_CHUNK rows of 2^lo words are at most
    // Np / (2 RS_CHUNK) + 2^lo nbk / RS_CHUNK < Np words, as Np >= 2048 nbk.
    tl.chunk = w.kA;
    tl.nchunk = (uint32_t)(w.ntile2 / RS_CHUNK);
    RsPlanOut po = {w.hbase, w.tfirst, w.tmap, nullptr, nullptr, nbins, plan.nt2 * RS_ITEMS};
    rs_count<false>(plan, plan.nt1, indx_in_cell, Np, plan.lo, plan.nb[0], w, tl, w.nblk, st);
    rs_scan(w.nblk, plan.nb[0], w, po, nullptr, st);
    rs_scatter<1>(plan, plan.nt1, indx_in_cell, nullptr, Np, plan.lo, plan.nb[0], w, w.low, w.vA, tl,
                  w.nblk, st);
    tl.nbk = 1 << plan.nb[0];  // totals and tiles exist for every high digit
    // The tiles of a bucket write interleaved pieces of the same lines: on
    // one XCD its L2 joins them (66.8M keys: scatter 418 -> 306 us, 3.0M:
    // 44 -> 31).  Not for so few tiles that the XCDs would share them unevenly
    // (380 tiles: +2 us).
    const int64_t nt2 = (w.ntile2 + 7) / 8 * 8;
    if (nt2 >= 512) tl.per = (uint32_t)(nt2 / 8);
    rs_count<true>(plan, plan.nt2, w.low, Np, 0, plan.lo, w, tl, nt2, st);
    k_rs_cells<<<plan.nbk + tl.nchunk, 1024, 0, st>>>(w.counts, plan.lo, tl, plan.nbk, w.offs, cell_offset,
                                                      np_stay, nbins, Np);
    rs_scatter<2>(plan, plan.nt2, w.low, w.vA, Np, 0, plan.lo, w, w.kA, sort_indx, tl,
                  nt2, st);
    CHM_CHECK_LAUNCH();
    return CHM_OK;
  }
  if (Np > 0 && plan.npass == 1) {
    RsPlanOut po = {w.hbase, nullptr, nullptr, cell_offset, np_stay, nbins, 0};
    rs_count<false>(plan, plan.nt1, indx_in_cell, Np, 0, plan.nb[0], w, tl, w.nblk, st);
    rs_scan(w.nblk, plan.nb[0], w, po, nullptr, st);
    rs_scatter<0>(plan, plan.nt1, indx_in_cell, nullptr, Np, 0, plan.nb[0], w, w.kA, sort_indx, tl,
                  w.nblk, st);
    CHM_CHECK_LAUNCH();
    return CHM_OK;
  }
  const uint32_t *skey = indx_in_cell;
  if (Np > 0) {
    RsPlanOut po = {w.hbase, nullptr, nullptr, nullptr, nullptr, nbins, 0};
    const uint32_t *kin = indx_in_cell, *vin = nullptr;
    int shift = 0;
    for (int p = 0; p < plan.npass; p++) {
      const int nb = plan.nb[p];
      const bool last = p == plan.npass - 1;
      // the last pass leaves the sorted keys in kA
      uint32_t *kout = ((plan.npass - 1 - p) & 1) ? w.kB : w.kA;
      uint32_t *vout = last ? sort_indx : ((p & 1) ? w.vB : w.vA);
      rs_count<false>(plan, plan.nt1, kin, Np, shift, nb, w, tl, w.nblk, st);
      rs_scan(w.nblk, nb, w, po, p == 0 ? w.trunc : nullptr, st);
      rs_scatter<0>(plan, plan.nt1, kin, vin, Np, shift, nb, w, kout, vout, tl, w.nblk, st);
      kin = kout;
      vin = vout;
      shift += nb;
    }
    skey = kin;
  }
  if (Np == 0) k_list_clear<<<1, 2, 0, st>>>(w.trunc);  // no radix pass cleared it
  k_offsets_bounds<<<chm_blocks(Np / OFF_PER + 1, 256), 256, 0, st>>>(skey, Np, nbins, cell_offset,
                                                                       np_stay, w.trunc);
  k_offsets_gaps<<<256, 256, 0, st>>>(skey, Np, nbins, cell_offset, np_stay, w.trunc);
  CHM_CHECK_LAUNCH();
  return CHM_OK;
}

template <typename T>
static int index_sort(const T *x, const T *y, const T *z, int64_t Np, const chm_grid_t *g,
                      uint32_t *indx_in_cell, uint32_t *cell_offset, uint32_t *sort_indx,
                      uint32_t *np_stay, void *ws, size_t ws_bytes, void *stream) {
  int rc = sort_keys<T, false>((T *)x, (T *)y, (T *)z, nullptr, nullptr, nullptr, nullptr, (T)0, Np, g,
                               indx_in_cell, ws, ws_bytes, stream);
  if (rc) return rc;
  return sort_from_keys(Np, g, indx_in_cell, cell_offset, sort_indx, np_stay, ws, ws_bytes, stream);
}

extern "C" int chm_index_sort_f64(const double *x, const double *y, const double *z, int64_t Np,
                                  const chm_grid_t *g, uint32_t *indx_in_cell, uint32_t *cell_offset,
                                  uint32_t *sort_indx, uint32_t *np_stay, void *ws, size_t ws_bytes,
                                  void *stream) {
  return index_sort<double>(x, y, z, Np, g, indx_in_cell, cell_offset, sort_indx, np_stay, ws,
                            ws_bytes, stream);
}
extern "C" int chm_index_sort_f32(const float *x, const float *y, const float *z, int64_t Np,
                                  const chm_grid_t *g, uint32_t *indx_in_cell, uint32_t *cell_offset,
                                  uint32_t *sort_indx, uint32_t *np_stay, void *ws, size_t ws_bytes,
                                  void *stream) {
  return index_sort<float>(x, y, z, Np, g, indx_in_cell, cell_offset, sort_indx, np_stay, ws,
                           ws_bytes, stream);
}

extern "C" int chm_push_x_keys_f64(double *x, double *y, double *z, const double *px, const double *py,
                                   const double *pz, const double *g_inv, double dt, int64_t Np,
                                   const chm_grid_t *g, uint32_t *indx_in_cell, void *ws,
                                   size_t ws_bytes, void *stream) {
  return sort_keys<double, true>(x, y, z, px, py, pz, g_inv, dt, Np, g, indx_in_cell, ws, ws_bytes,
                                 stream);
}
extern "C" int chm_push_x_keys_f32(float *x, float *y, float *z, const float *px, const float *py,
                                   const float *pz, const float *g_inv, float dt, int64_t Np,
                                   const chm_grid_t *g, uint32_t *indx_in_cell, void *ws,
                                   size_t ws_bytes, void *stream) {
  return sort_keys<float, true>(x, y, z, px, py, pz, g_inv, dt, Np, g, indx_in_cell, ws, ws_bytes,
                                stream);
}
// Where the last pass left the sorted keys in a sort workspace.
extern "C" const uint32_t *chm_sort_sorted_keys(const void *ws, int64_t Np, const chm_grid_t *g) {
  if (!ws || !g || Np <= 0 || Np > 0x7FFFFFF0ll || g->Nx < 4 || g->Nr < 3) return nullptr;
  const int64_t nbins = (int64_t)(g->Nx - 1) * (g->Nr - 1) + 1;
  SortWs w;
  sort_layout(Np, nbins, &w, (void *)ws);
  return w.kA;
}

extern "C" int chm_sort_from_keys(int64_t Np, const chm_grid_t *g, const uint32_t *indx_in_cell,
                                  uint32_t *cell_offset, uint32_t *sort_indx, uint32_t *np_stay,
                                  void *ws, size_t ws_bytes, void *stream) {
  return sort_from_keys(Np, g, indx_in_cell, cell_offset, sort_indx, np_stay, ws, ws_bytes, stream);
}

// ------------------------------------------------------------------ sort without allocation
// chm_index_sort_f64_noalloc takes its sort workspace from `scratch`, a fixed
// array in device memory (one copy per GPU, held until the process ends).
// In host code `scratch` only names the symbol: its device address on the
// current GPU comes from hipGetSymbolAddress, looked up once per device on
// the first call there, and only that address is handed to kernels.  Nothing
// left by an earlier call is read: the count rows of the tiles that a pass has
// are written before its scan reads them, and the scan writes their offsets,
// the digit totals, first positions and the buckets' tiles; the 16-bit keys
// and indices between the passes are written whole by the first scatter, the
// chunk rows are cleared by the first count, and the offsets' list (LSD passes
// only) by the first pass's scan or by k_list_clear.
static __device__ __align__(256) unsigned char scratch[CHM_SORT_SCRATCH_BYTES];

#define CHM_MAX_DEVICES 64
static std::mutex scratch_mu;
static void *scratch_dev[CHM_MAX_DEVICES];

static int scratch_ptr(void **out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return (int)e;
  if (dev < 0 || dev >= CHM_MAX_DEVICES) return CHM_EUNSUPPORTED;
  std::lock_guard<std::mutex> lock(scratch_mu);
  if (!scratch_dev[dev]) {
    void *p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return (int)e;
    if (!p) return CHM_EINVAL;
    scratch_dev[dev] = p;
  }
  *out = scratch_dev[dev];
  return CHM_OK;
}

extern "C" int chm_index_sort_f64_noalloc(const double *x, const double *y, const double *z,
                                          int64_t Np, const chm_grid_t *g, uint32_t *indx_in_cell,
                                          uint32_t *cell_offset, uint32_t *sort_indx,
                                          uint32_t *np_stay, void *stream) {
  if (!g || Np < 0 || Np > 0x7FFFFFF0ll || g->Nx < 4 || g->Nr < 3) return CHM_EINVAL;
  const int64_t nbins = (int64_t)(g->Nx - 1) * (g->Nr - 1) + 1;
  const size_t need = sort_layout(Np, nbins, nullptr, nullptr);
  if (need > (size_t)CHM_SORT_SCRATCH_BYTES) return CHM_ESCRATCH;
  void *ws = nullptr;
  int rc = scratch_ptr(&ws);
  if (rc) return rc;
  return index_sort<double>(x, y, z, Np, g, indx_in_cell, cell_offset, sort_indx, np_stay, ws, need,
                            stream);
}

// ------------------------------------------------------------------ profile
// profile_by_interpolant, particles_generic.cl:6-30, constant extension
// outside the knots (where the reference reads past the knot array).
template <typename T>
__global__ void __launch_bounds__(256) k_dens_profile(const T *__restrict__ x, T *__restrict__ w,
                                                      int64_t Np, const double *__restrict__ xx,
                                                      const double *__restrict__ ff,
                                                      const double *__restrict__ dxm1, int n) {
  int64_t ip = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (ip >= Np) return;
  double xp = (double)x[ip];
  if (xp < xx[0]) xp = xx[0];
  if (xp > xx[n - 1]) xp = xx[n - 1];
  int ix = 0;
  if (xp > xx[0])
    for (ix = 0; ix < n - 2; ix++)
      if (xp > xx[ix] && xp <= xx[ix + 1]) break;
  double f_minus = ff[ix] * dxm1[ix];
  double f_plus = ff[ix + 1] * dxm1[ix];
  double f = f_minus * (xx[ix + 1] - xp) + f_plus * (xp - xx[ix]);
  w[ip] = (T)((double)w[ip] * f);
}

template <typename T>
static int dens_profile(const T *x, T *w, int64_t Np, const double *xx, const double *ff,
                        const double *dxm1, int n, void *stream) {
  if (Np < 0 || n < 2) return CHM_EINVAL;
  if (Np == 0) return CHM_OK;
  k_dens_profile<T><<<chm_blocks(Np, 256), 256, 0, (hipStream_t)stream>>>(x, w, Np, xx, ff, dxm1, n);
  CHM_CHECK_LAUNCH();
  return CHM_OK;
}

extern "C" int chm_dens_profile_f64(const double *x, double *w, int64_t Np, const double *xx,
                                    const double *ff, const double *dxm1, int32_t nknots,
                                    void *stream) {
  return dens_profile<double>(x, w, Np, xx, ff, dxm1, nknots, stream);
}
extern "C" int chm_dens_profile_f32(const float *x, float *w, int64_t Np, const double *xx,
                                    const double *ff, const double *dxm1, int32_t nknots,
                                    void *stream) {
  return dens_profile<float>(x, w, Np, xx, ff, dxm1, nknots, stream);
}

// ------------------------------------------------------------------ domain fill
// Deterministic building blocks shared with the CPU oracle (which evaluates
// the same expressions in the same order, so the results are bit-identical):
//   rng_u01   splitmix64 (Steele, Lea, Flood 2014) of seed + (counter+1)*golden,
//             top 53 bits -> [0, 1)
//   det_sincos sin and cos from IEEE +, -, *, / only: Cody-Waite reduction by
//             pi/2 with the three-part constant of fdlibm (k*P1, k*P2 exact for
//             |k| < 2^20), Taylor polynomials to r^17 / r^18 on |r| <= pi/4.
__device__ __forceinline__ double rng_u01(uint64_t seed, uint64_t counter) {
  uint64_t z = seed + (counter + 1ull) * 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  z = z ^ (z >> 31);
  return (double)(z >> 11) * (1.0 / 9007199254740992.0);
}

__device__ __forceinline__ void det_sincos(double a, double *s_out, double *c_out) {
  const double P1 = 1.57079632673412561417e+00, P2 = 6.07710050630396597660e-11,
               P2T = 2.02226624879595063154e-21;
  const double k = floor(a * (2.0 / 3.14159265358979323846) + 0.5);
  const double r = ((a - k * P1) - k * P2) - k * P2T;
  const double r2 = r * r;
  double s = 1.0 / 355687428096000.0;                 // 1/17!
  s = (-1.0 / 1307674368000.0) + r2 * s;              // 1/15!
  s = (1.0 / 6227020800.0) + r2 * s;                  // 1/13!
  s = (-1.0 / 39916800.0) + r2 * s;                   // 1/11!
  s = (1.0 / 362880.0) + r2 * s;                      // 1/9!
  s = (-1.0 / 5040.0) + r2 * s;                       // 1/7!
  s = (1.0 / 120.0) + r2 * s;                         // 1/5!
  s = (-1.0 / 6.0) + r2 * s;                          // 1/3!
  s = r + r * (r2 * s);
  double c = -1.0 / 6402373705728000.0;               // -1/18!
  c = (1.0 / 20922789888000.0) + r2 * c;              // 1/16!
  c = (-1.0 / 87178291200.0) + r2 * c;                // -1/14!
  c = (1.0 / 479001600.0) + r2 * c;                   // 1/12!
  c = (-1.0 / 3628800.0) + r2 * c;                    // -1/10!
  c = (1.0 / 40320.0) + r2 * c;                       // 1/8!
  c = (-1.0 / 720.0) + r2 * c;                        // -1/6!
  c = (1.0 / 24.0) + r2 * c;                          // 1/4!
  c = (-0.5) + r2 * c;                                // -1/2!
  c = 1.0 + r2 * c;
  const int q = (int)((int64_t)k & 3);
  double sv, cv;
  if (q == 0) { sv = s; cv = c; }
  else if (q == 1) { sv = c; cv = -s; }
  else if (q == 2) { sv = -s; cv = -c; }
  else { sv = -c; cv = s; }
  *s_out = sv;
  *c_out = cv;
}

// log from IEEE operations and the exact frexp split, as the CPU oracle
// evaluates it: x = m 2^e with m in [sqrt(1/2), sqrt(2)), log m = 2 atanh(f),
// f = (m-1)/(m+1), series to f^19 (|f| <= 0.172); e ln2 with fdlibm's
// two-part ln2.
__device__ __forceinline__ double det_log(double x) {
  int e;
  double m = frexp(x, &e);
  if (m < 0.70710678118654752440) {
    m = m * 2.0;
    e -= 1;
  }
  const double f = (m - 1.0) / (m + 1.0);
  const double f2 = f * f;
  double s = 1.0 / 19.0;
  s = (1.0 / 17.0) + f2 * s;
  s = (1.0 / 15.0) + f2 * s;
  s = (1.0 / 13.0) + f2 * s;
  s = (1.0 / 11.0) + f2 * s;
  s = (1.0 / 9.0) + f2 * s;
  s = (1.0 / 7.0) + f2 * s;
  s = (1.0 / 5.0) + f2 * s;
  s = (1.0 / 3.0) + f2 * s;
  const double lm = 2.0 * (f + f * (f2 * s));
  const double de = (double)e;
  return de * 6.93147180369123816490e-01 + (lm + de * 1.90821492927058770002e-10);
}

// Two independent standard normals from counters (c, c+1) (Box-Muller).
__device__ __forceinline__ void det_normal2(uint64_t seed, uint64_t c, double *z0, double *z1) {
  const double u1 = rng_u01(seed, c), u2 = rng_u01(seed, c + 1);
  const double rad = sqrt(-2.0 * det_log(1.0 - u1));
  double s, co;
  det_sincos((2.0 * 3.14159265358979323846) * u2, &s, &co);
  *z0 = rad * co;
  *z1 = rad * s;
}

// fill_grid, particles_generic.cl:33-84: per cell (ix, ir) of the local
// grids (xgrid [Nx_loc], rgrid), Nppc_th x Nppc_r x Nppc_x particles at the
// regular sub-positions, the theta set rotated by a per-cell uniform offset
// in [0, 2 pi) (theta_variator, particles_methods_cl.py:95-98, here from
// rng_u01(seed, counter0 + cell)); weights r * w0 (:103); momenta
// (:111-147): p_c, plus dp times a standard normal per particle and
// component when a spread dp is given (_fill_arr_randn(mu = p_c, sigma =
// dp)); particle ip draws its normals from counters counter_p + 4 ip .. + 2
// (two Box-Muller pairs, the fourth value unused); g_inv from the momenta.
template <typename T>
__global__ void __launch_bounds__(256)
    k_fill_domain(T *__restrict__ x, T *__restrict__ y, T *__restrict__ z, T *__restrict__ w,
                  T *__restrict__ px, T *__restrict__ py, T *__restrict__ pz,
                  T *__restrict__ g_inv, const double *__restrict__ xgrid,
                  const double *__restrict__ rgrid, int Nx, int64_t ncells, int npx, int npr,
                  int npt, double w0, double pxc, double pyc, double pzc, double dpx,
                  double dpy, double dpz, int moving, uint64_t seed, uint64_t counter0,
                  uint64_t counter_p) {
  const int64_t i_cell = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i_cell >= ncells) return;
  const int Nx_cell = Nx - 1;
  const int ir = (int)(i_cell / Nx_cell), ix = (int)(i_cell - (int64_t)ir * Nx_cell);
  int64_t ip = i_cell * (int64_t)(npx * npr * npt);
  const double xmin = xgrid[ix], rmin = rgrid[ir];
  const double thmin = (2.0 * 3.14159265358979323846) * rng_u01(seed, counter0 + (uint64_t)i_cell);
  const double Lx = xgrid[ix + 1] - xgrid[ix];
  const double Lr = rgrid[ir + 1] - rgrid[ir];
  const double dx = 1. / ((double)npx);
  const double dr = 1. / ((double)npr);
  const double dth = 2 * 3.14159265358979323846 / ((double)npt);
  const bool thermal = dpx != 0.0 || dpy != 0.0 || dpz != 0.0;
  double g = 1.0;
  if (pxc != 0.0 || pyc != 0.0 || pzc != 0.0) g = 1. / sqrt(1 + pxc * pxc + pyc * pyc + pzc * pzc);
  for (int it = 0; it < npt; it++) {
    const double th = thmin + it * dth;
    double sin_th, cos_th;
    det_sincos(th, &sin_th, &cos_th);
    for (int irr = 0; irr < npr; irr++) {
      const double rp = rmin + (0.5 + irr) * dr * Lr;
      const double rp_s = rp * sin_th;
      const double rp_c = rp * cos_th;
      for (int ixx = 0; ixx < npx; ixx++) {
        x[ip] = (T)(xmin + (0.5 + ixx) * dx * Lx);
        y[ip] = (T)rp_s;
        z[ip] = (T)rp_c;
        w[ip] = (T)(rp * w0);
        if (moving) {
          if (thermal) {
            double n0, n1, n2, n3;
            const uint64_t c = counter_p + 4ull * (uint64_t)ip;
            det_normal2(seed, c, &n0, &n1);
            det_normal2(seed, c + 2, &n2, &n3);
            const double ux = pxc + dpx * n0, uy = pyc + dpy * n1, uz = pzc + dpz * n2;
            px[ip] = (T)ux;
            py[ip] = (T)uy;
            pz[ip] = (T)uz;
            g_inv[ip] = (T)(1. / sqrt(1 + ux * ux + uy * uy + uz * uz));
          } else {
            px[ip] = (T)pxc;
            py[ip] = (T)pyc;
            pz[ip] = (T)pzc;
            g_inv[ip] = (T)g;
          }
        }
        ip += 1;
      }
    }
  }
}

template <typename T>
static int fill_domain(T *x, T *y, T *z, T *w, T *px, T *py, T *pz, T *g_inv, const double *xgrid,
                       const double *rgrid, int32_t Nx_loc, int64_t ncells, int32_t npx,
                       int32_t npr, int32_t npt, double w0, double pxc, double pyc, double pzc,
                       double dpx, double dpy, double dpz, uint64_t seed, uint64_t counter0,
                       void *stream) {
  if (!x || !y || !z || !w || !xgrid || !rgrid || Nx_loc < 2 || ncells < 0 || npx < 1 || npr < 1 ||
      npt < 1)
    return CHM_EINVAL;
  const int moving = px != nullptr;
  if (moving && (!py || !pz || !g_inv)) return CHM_EINVAL;
  if (ncells == 0) return CHM_OK;
  k_fill_domain<T><<<chm_blocks(ncells, 256), 256, 0, (hipStream_t)stream>>>(
      x, y, z, w, px, py, pz, g_inv, xgrid, rgrid, Nx_loc, ncells, npx, npr, npt, w0, pxc, pyc, pzc,
      dpx, dpy, dpz, moving, seed, counter0, counter0 + (uint64_t)ncells);
  CHM_CHECK_LAUNCH();
  return CHM_OK;
}

extern "C" int chm_fill_domain_f64(double *x, double *y, double *z, double *w, double *px,
                                   double *py, double *pz, double *g_inv, const double *xgrid,
                                   const double *rgrid, int32_t Nx_loc, int64_t ncells,
                                   int32_t npx, int32_t npr, int32_t npt, double w0, double pxc,
                                   double pyc, double pzc, double dpx, double dpy, double dpz,
                                   uint64_t seed, uint64_t counter0, void *stream) {
  return fill_domain<double>(x, y, z, w, px, py, pz, g_inv, xgrid, rgrid, Nx_loc, ncells, npx, npr,
                             npt, w0, pxc, pyc, pzc, dpx, dpy, dpz, seed, counter0, stream);
}
extern "C" int chm_fill_domain_f32(float *x, float *y, float *z, float *w, float *px, float *py,
                                   float *pz, float *g_inv, const double *xgrid,
                                   const double *rgrid, int32_t Nx_loc, int64_t ncells,
                                   int32_t npx, int32_t npr, int32_t npt, double w0, double pxc,
                                   double pyc, double pzc, double dpx, double dpy, double dpz,
                                   uint64_t seed, uint64_t counter0, void *stream) {
  return fill_domain<float>(x, y, z, w, px, py, pz, g_inv, xgrid, rgrid, Nx_loc, ncells, npx, npr,
                            npt, w0, pxc, pyc, pzc, dpx, dpy, dpz, seed, counter0, stream);
}

// ------------------------------------------------------------------ beam
// make_new_beam, particles_methods_cl.py:149-177: Gaussian positions and
// momenta, equal weights, g_inv from the momenta.  Particle p draws its six
// normals from counters counter0 + 6p .. + 5.
template <typename T>
__global__ void __launch_bounds__(256)
    k_fill_beam(T *__restrict__ x, T *__restrict__ y, T *__restrict__ z, T *__restrict__ px,
                T *__restrict__ py, T *__restrict__ pz, T *__restrict__ w, T *__restrict__ g_inv,
                int64_t Np, chm_beam_t b, uint64_t seed, uint64_t counter0) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= Np) return;
  const uint64_t c = counter0 + 6ull * (uint64_t)p;
  double n[6];
  det_normal2(seed, c, &n[0], &n[1]);
  det_normal2(seed, c + 2, &n[2], &n[3]);
  det_normal2(seed, c + 4, &n[4], &n[5]);
  const double xv = b.c[0] + b.L[0] * n[0], yv = b.c[1] + b.L[1] * n[1],
               zv = b.c[2] + b.L[2] * n[2];
  const double ux = b.pc[0] + b.dp[0] * n[3], uy = b.pc[1] + b.dp[1] * n[4],
               uz = b.pc[2] + b.dp[2] * n[5];
  x[p] = (T)xv;
  y[p] = (T)yv;
  z[p] = (T)zv;
  px[p] = (T)ux;
  py[p] = (T)uy;
  pz[p] = (T)uz;
  w[p] = (T)b.w;
  g_inv[p] = (T)(1. / sqrt(1 + ux * ux + uy * uy + uz * uz));
}

template <typename T>
static int fill_beam(T *x, T *y, T *z, T *px, T *py, T *pz, T *w, T *g_inv, int64_t Np,
                     const chm_beam_t *b, uint64_t seed, uint64_t counter0, void *stream) {
  if (!b || Np < 0 || !x || !y || !z || !px || !py || !pz || !w || !g_inv) return CHM_EINVAL;
  if (Np == 0) return CHM_OK;
  k_fill_beam<T><<<chm_blocks(Np, 256), 256, 0, (hipStream_t)stream>>>(x, y, z, px, py, pz, w,
                                                                       g_inv, Np, *b, seed, counter0);
  CHM_CHECK_LAUNCH();
  return CHM_OK;
}

extern "C" int chm_fill_beam_f64(double *x, double *y, double *z, double *px, double *py,
                                 double *pz, double *w, double *g_inv, int64_t Np,
                                 const chm_beam_t *b, uint64_t seed, uint64_t counter0,
                                 void *stream) {
  return fill_beam<double>(x, y, z, px, py, pz, w, g_inv, Np, b, seed, counter0, stream);
}
extern "C" int chm_fill_beam_f32(float *x, float *y, float *z, float *px, float *py, float *pz,
                                 float *w, float *g_inv, int64_t Np, const chm_beam_t *b,
                                 uint64_t seed, uint64_t counter0, void *stream) {
  return fill_beam<float>(x, y, z, px, py, pz, w, g_inv, Np, b, seed, counter0, stream);
}
