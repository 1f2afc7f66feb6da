// Discrete Hankel transform products on the matrix cores (gfx950 MFMA).
//
//   C[M x N] = A[M x K] @ B[K x N]      (row-major, A = a DHT-type matrix)
//
// A is a per-mode real matrix (DHT, DHT_inv, dDHT+-) stored zero-padded to
// [round_up(M, 64)][lda], lda = round_up(K, 64), so A tiles load without
// bounds checks in 16-byte vectors.  B is either a real field [K][N] (mode 0),
// or a complex field [K][Nx] read as N = 2*Nx real columns, optionally formed
// on the fly as alpha*X + beta*Y with either operand read through the
// m = -1 map F_{-1}[k][x] = -conj(F_1[k][-x]) (get_m1,
// transformer_generic.cl:3-24).  This replaces Reikna's MatrixMul
// (transformer_methods_cl.py:458-472) and the axpy/get_m1 kernels that fed it.
//
// Three arithmetic forms, 256 threads, 64 x 64 output tile per block, wave w
// owning the 32 x 32 quadrant (w/2, w%2); the next K-step is loaded into
// registers while the current one is multiplied:
//   f64    : v_mfma_f64_16x16x4f64 (plain form)
//   f32    : v_mfma_f32_16x16x4f32 (mixed form, CHM_DHT_F32)
//   bf16x3 : v_mfma_f32_16x16x32_bf16 on split operands, A = Ah + Al,
//            B = Bh + Bl, C = Ah*Bh + (Ah*Bl + Al*Bh), the two small terms
//            accumulated apart and added at the end (mixed, CHM_DHT_BF16X3).
#include "gemm.h"

#include <mutex>
#include <type_traits>
#include <vector>

typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef unsigned short us8 __attribute__((ext_vector_type(8)));
typedef unsigned short us4 __attribute__((ext_vector_type(4)));

#define BM 64
#define BN 64

// ---------------------------------------------------------------- tiles
// The output tile of a block.  One launch takes the items of all modes (a
// launch per mode left the last round of blocks of each partly empty), and
// the row tiles of a column of tiles go to one XCD one after the other: its
// L2 then holds the columns of B that they share, and A, which all of its
// blocks share.  Against a launch per mode: FP64 256 x 64, M = 1, both
// transforms 26.7 -> 15 us (4 launches to 2), 1024 x 128 11.3 -> 8 us each,
// 2048 x 256 178 -> 168 us; mixed 2048 x 256, M = 1, 69 -> 62 us.
template <int TM, int TN>
__device__ __forceinline__ bool gemm_tile(const GemmBatch &gb, int &item, int &n0, int &m0) {
  const int mt = (gb.M + TM - 1) / TM, i = (int)(blockIdx.x >> 3);
  const int g = (i / mt) * 8 + (int)(blockIdx.x & 7);
  if (g >= gb.nt[gb.nitems]) return false;
  item = 0;
  while (g >= gb.nt[item + 1]) item++;
  n0 = (g - gb.nt[item]) * TN;
  m0 = (i % mt) * TM;
  return true;
}
// fills nt for tiles of TN columns; the number of blocks of the launch
static unsigned gemm_blocks(GemmBatch &gb, int tm, int tn) {
  gb.nt[0] = 0;
  for (int i = 0; i < gb.nitems; i++) gb.nt[i + 1] = gb.nt[i] + (gb.it[i].N + tn - 1) / tn;
  return (unsigned)((gb.nt[gb.nitems] + 7) / 8 * 8) * (unsigned)((gb.M + tm - 1) / tm);
}

// ---------------------------------------------------------------- B loader
// A thread's source of B elements: columns n and n + 1 (n even) of rows k.
// BMODE 0: a real field with an even number of columns (one aligned
// 2-element load); 1: alpha X + beta Y of complex fields, one complex element
// of each, either through the m = -1 map; 2: a real field with an odd number
// of columns.  Everything of the item that the loop needs is taken out of
// the kernel's arguments here, once, and the loads have no branches: rows
// past K read row K - 1 and count as zero, columns past N read the last ones
// and are never stored.
template <typename T> struct BSrc {
  const T *x, *y;
  int64_t ld;
  int K, n1;
  T ax, ay, bx, by;
  bool rx, ry;
};
template <typename T, int BMODE>
__device__ __forceinline__ BSrc<T> b_source(const GemmBatch &gb, const GemmItem &it, int n) {
  BSrc<T> s = {};
  s.K = gb.K;
  if constexpr (BMODE == 1) {
    const int Nx = gb.Nx, c = n < it.N ? n >> 1 : 0;
    s.ld = 2 * Nx;
    s.x = (const T *)it.X + 2 * (it.remapX ? (Nx - c) % Nx : c);
    s.y = it.Y ? (const T *)it.Y + 2 * (it.remapY ? (Nx - c) % Nx : c) : nullptr;
    s.ax = (T)it.alpha.x;
    s.ay = (T)it.alpha.y;
    s.bx = (T)it.beta.x;
    s.by = (T)it.beta.y;
    s.rx = it.remapX;
    s.ry = it.remapY;
  } else {
    const int c = n < it.N ? n : (BMODE == 0 ? it.N - 2 : it.N - 1);
    s.ld = it.N;
    s.x = (const T *)it.X + c;
    s.n1 = c + 1 < it.N ? 1 : 0;
  }
  return s;
}
// The loaded elements stay raw (load_b) and become B values only where they
// are stored to LDS (b_value): a block issues the next K-step's loads,
// multiplies the current one, and only then computes, so the loads stay in
// flight across the MFMAs (with the complex products formed right after the
// loads, each K-step waited for them: the mixed rot product took 597 us per
// step instead of 360 on the 4096 x 512 step).
template <typename T, int BMODE> struct BRaw { T x0, x1; };
template <typename T> struct BRaw<T, 1> { T x0, x1, y0, y1; };

template <typename T, int BMODE>
__device__ __forceinline__ BRaw<T, BMODE> load_b(const BSrc<T> &s, int k) {
  typedef T t2 __attribute__((ext_vector_type(2)));
  const int64_t o = (int64_t)(k < s.K ? k : s.K - 1) * s.ld;
  BRaw<T, BMODE> r;
  if constexpr (BMODE == 2) {
    r.x0 = s.x[o];
    r.x1 = s.x[o + s.n1];
  } else {
    const t2 v = *(const t2 *)(s.x + o);
    r.x0 = v.x;
    r.x1 = v.y;
  }
  if constexpr (BMODE == 1) {
    r.y0 = r.y1 = (T)0;
    if (s.y) {
      const t2 w = *(const t2 *)(s.y + o);
      r.y0 = w.x;
      r.y1 = w.y;
    }
  }
  return r;
}
template <typename T> struct pair_t { T a, b; };
// (k: the row that v was loaded for)
template <typename T, int BMODE>
__device__ __forceinline__ pair_t<T> b_value(const BSrc<T> &s, const BRaw<T, BMODE> &v, int k) {
  pair_t<T> r = {(T)0, (T)0};
  if constexpr (BMODE == 1) {
    if (k >= s.K) return r;
    {
      const T a = s.rx ? -v.x0 : v.x0, b = v.x1;  // -conj(F(-kx)): (-re, +im)
      r.a = s.ax * a - s.ay * b;
      r.b = s.ax * b + s.ay * a;
    }
    if (s.y) {
      const T a = s.ry ? -v.y0 : v.y0, b = v.y1;
      r.a += s.bx * a - s.by * b;
      r.b += s.bx * b + s.by * a;
    }
  } else {
    r.a = k < s.K ? v.x0 : (T)0;
    r.b = k < s.K ? v.x1 : (T)0;
  }
  return r;
}

// ---------------------------------------------------------------- f64 / f32
// (registers held to 5 waves per SIMD: the accumulators stay in VGPRs)
template <typename T, int BMODE>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(5))) k_gemm(GemmBatch gb) {
  constexpr int BK = 16;
  constexpr int AP = (sizeof(T) == 8) ? 8 : 16;  // row pad: stride = 128 B mod 256 B
  __shared__ T As[BK][BM + AP];
  __shared__ T Bs[BK][BN + AP];
  int item, n0, m0;
  if (!gemm_tile<BM, BN>(gb, item, n0, m0)) return;
  const GemmItem &it = gb.it[item];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wr = wave >> 1, wc = wave & 1;
  const T *A = (const T *)it.A;
  // A: thread loads row ar, k = ak..ak+3 (padded table, no checks)
  const int ar = tid >> 2, ak = (tid & 3) * 4;
  // B: thread owns columns 2*bp, 2*bp+1 and rows bk, bk+8
  const int bp = tid & 31, bk = tid >> 5;
  T ra[4];
  BRaw<T, BMODE> rb[2];
  const BSrc<T> bs = b_source<T, BMODE>(gb, it, n0 + 2 * bp);
  auto gload = [&](int k0) {
    const T *pa = A + (int64_t)(m0 + ar) * gb.lda + k0 + ak;
#pragma unroll
    for (int q = 0; q < 4; q++) ra[q] = pa[q];
#pragma unroll
    for (int q = 0; q < 2; q++) rb[q] = load_b<T, BMODE>(bs, k0 + bk + 8 * q);
  };
  typedef typename std::conditional<sizeof(T) == 8, d4, f4>::type acc_t;
  acc_t acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++) acc[i][j] = (acc_t){0, 0, 0, 0};
  gload(0);
  for (int k0 = 0; k0 < gb.K; k0 += BK) {
#pragma unroll
    for (int q = 0; q < 4; q++) As[ak + q][ar] = ra[q];
#pragma unroll
    for (int q = 0; q < 2; q++) {
      const pair_t<T> b = b_value<T, BMODE>(bs, rb[q], k0 + bk + 8 * q);
      Bs[bk + 8 * q][2 * bp] = b.a;
      Bs[bk + 8 * q][2 * bp + 1] = b.b;
    }
    __syncthreads();
    if (k0 + BK < gb.K) gload(k0 + BK);
#pragma unroll
    for (int kk = 0; kk < BK; kk += 4) {
      T a[2], b[2];
#pragma unroll
      for (int i = 0; i < 2; i++) a[i] = As[kk + (lane >> 4)][32 * wr + 16 * i + (lane & 15)];
#pragma unroll
      for (int j = 0; j < 2; j++) b[j] = Bs[kk + (lane >> 4)][32 * wc + 16 * j + (lane & 15)];
#pragma unroll
      for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) {
          if constexpr (sizeof(T) == 8)
            acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i], b[j], acc[i][j], 0, 0, 0);
          else
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b[j], acc[i][j], 0, 0, 0);
        }
    }
    __syncthreads();
  }
  T *C = (T *)it.C;
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        // f64 16x16x4: row = l/16 + 4r ; f32 16x16x4: row = 4*(l/16) + r
        int rloc = (sizeof(T) == 8) ? ((lane >> 4) + 4 * r) : (4 * (lane >> 4) + r);
        int row = m0 + 32 * wr + 16 * i + rloc;
        int col = n0 + 32 * wc + 16 * j + (lane & 15);
        if (row < gb.M && col < it.N) C[(int64_t)row * it.N + col] = acc[i][j][r];
      }
}

// ---------------------------------------------------------------- split-BF16
__device__ __forceinline__ void split_bf16(float v, unsigned short &hi, unsigned short &lo) {
  __bf16 h = (__bf16)v;
  __bf16 l = (__bf16)(v - (float)h);
  hi = __builtin_bit_cast(unsigned short, h);
  lo = __builtin_bit_cast(unsigned short, l);
}

template <int BK, int BMODE>
__global__ void __launch_bounds__(256) k_gemm_bf16x3(GemmBatch gb) {
  constexpr int KP = BK + 8;  // row stride 16-byte aligned, staggers banks
  constexpr int NA = BK / 32;  // 16-byte A vectors per thread (hi and lo)
  constexpr int NB = BK / 8;   // B column pairs per thread
  // operands stored k-contiguous so each lane reads 8 bf16 (16 B) at once
  __shared__ __attribute__((aligned(16))) unsigned short Ah[BM][KP], Al[BM][KP];
  __shared__ __attribute__((aligned(16))) unsigned short Bh[BN][KP], Bl[BN][KP];
  int item, n0, m0;
  if (!gemm_tile<BM, BN>(gb, item, n0, m0)) return;
  const GemmItem &it = gb.it[item];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wr = wave >> 1, wc = wave & 1;
  const unsigned short *Ahg = (const unsigned short *)it.A, *Alg = (const unsigned short *)it.A_lo;
  // A: thread loads row ar, k = ak .. ak + 8*NA - 1 (hi and lo)
  const int ar = tid >> 2, ak = (tid & 3) * 8 * NA;
  // B: thread owns columns 2*bp, 2*bp+1 and k = bk .. bk + NB - 1
  const int bp = tid & 31, bk = (tid >> 5) * NB;
  us8 rah[NA], ral[NA];
  BRaw<float, BMODE> rb[NB];
  const BSrc<float> bs = b_source<float, BMODE>(gb, it, n0 + 2 * bp);
  auto gload = [&](int k0) {
    const int64_t o = (int64_t)(m0 + ar) * gb.lda + k0 + ak;
#pragma unroll
    for (int v = 0; v < NA; v++) {
      rah[v] = *(const us8 *)(Ahg + o + 8 * v);
      ral[v] = *(const us8 *)(Alg + o + 8 * v);
    }
#pragma unroll
    for (int q = 0; q < NB; q++) rb[q] = load_b<float, BMODE>(bs, k0 + bk + q);
  };
  f4 acc[2][2], cor[2][2];
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++) acc[i][j] = cor[i][j] = (f4){0, 0, 0, 0};
  gload(0);
  for (int k0 = 0; k0 < gb.K; k0 += BK) {
#pragma unroll
    for (int v = 0; v < NA; v++) {
      *(us8 *)&Ah[ar][ak + 8 * v] = rah[v];
      *(us8 *)&Al[ar][ak + 8 * v] = ral[v];
    }
#pragma unroll
    for (int q0 = 0; q0 < NB; q0 += 4) {
      us4 bh0, bl0, bh1, bl1;
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const pair_t<float> b = b_value<float, BMODE>(bs, rb[q0 + q], k0 + bk + q0 + q);
        unsigned short h, l;
        split_bf16(b.a, h, l);
        bh0[q] = h;
        bl0[q] = l;
        split_bf16(b.b, h, l);
        bh1[q] = h;
        bl1[q] = l;
      }
      *(us4 *)&Bh[2 * bp][bk + q0] = bh0;
      *(us4 *)&Bl[2 * bp][bk + q0] = bl0;
      *(us4 *)&Bh[2 * bp + 1][bk + q0] = bh1;
      *(us4 *)&Bl[2 * bp + 1][bk + q0] = bl1;
    }
    __syncthreads();
    if (k0 + BK < gb.K) gload(k0 + BK);
#pragma unroll
    for (int ks = 0; ks < BK; ks += 32) {
      bf8 ah[2], al[2], bhv[2], blv[2];
#pragma unroll
      for (int i = 0; i < 2; i++) {
        const int row = 32 * wr + 16 * i + (lane & 15), k = ks + 8 * (lane >> 4);
        ah[i] = __builtin_bit_cast(bf8, *(const us8 *)&Ah[row][k]);
        al[i] = __builtin_bit_cast(bf8, *(const us8 *)&Al[row][k]);
      }
#pragma unroll
      for (int j = 0; j < 2; j++) {
        const int col = 32 * wc + 16 * j + (lane & 15), k = ks + 8 * (lane >> 4);
        bhv[j] = __builtin_bit_cast(bf8, *(const us8 *)&Bh[col][k]);
        blv[j] = __builtin_bit_cast(bf8, *(const us8 *)&Bl[col][k]);
      }
#pragma unroll
      for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) {
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[i], bhv[j], acc[i][j], 0, 0, 0);
          cor[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[i], blv[j], cor[i][j], 0, 0, 0);
          cor[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al[i], bhv[j], cor[i][j], 0, 0, 0);
        }
    }
    __syncthreads();
  }
  float *C = (float *)it.C;
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        int row = m0 + 32 * wr + 16 * i + 4 * (lane >> 4) + r;
        int col = n0 + 32 * wc + 16 * j + (lane & 15);
        if (row < gb.M && col < it.N) C[(int64_t)row * it.N + col] = acc[i][j][r] + cor[i][j][r];
      }
}

// ---------------------------------------------------------------- 128 x 128 tiles
// The split-BF16 product with a 128 x 128 output tile per block (each wave a
// 64 x 64 quadrant of 4 x 4 MFMA tiles), for launches with enough tiles to
// fill the GPU: four times the matrix-core work per LDS round trip and
// barrier, and half the operand loads per flop.  Two LDS buffers: while one
// K-step is multiplied the next is split into the other buffer and the one
// after it is on its way from memory.  Bound by what does not overlap at two
// waves per SIMD: both transforms of 4096 x 512, M = 2 take 512 us, 355
// without the operand loads, 280 without the split too, of which 85 are the
// LDS reads and 82 the stores of C.
template <int BMODE>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) k_gemm128_bf16x3(GemmBatch gb) {
  constexpr int TM = 128, TN = 128, BK = 32, KP = BK + 8;
  typedef unsigned short Tile[TM][KP];
  __shared__ __attribute__((aligned(16))) Tile Ah[2], Al[2], Bh[2], Bl[2];
  int item, n0, m0;
  if (!gemm_tile<TM, TN>(gb, item, n0, m0)) return;
  const GemmItem &it = gb.it[item];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wr = wave >> 1, wc = wave & 1;
  const unsigned short *Ahg = (const unsigned short *)it.A, *Alg = (const unsigned short *)it.A_lo;
  // A: thread loads rows ar and ar + 64, k = ak .. ak + 7 (hi and lo), four
  // lanes a 64-byte piece of a row; rows beyond the 64-row padding of the
  // table are not read
  const int ar = tid >> 2, ak = (tid & 3) * 8;
  const bool arow = m0 + 64 < ((gb.M + 63) & ~63);
  // B: thread owns columns 2*bp, 2*bp+1 and k = bk .. bk + 7
  const int bp = tid & 63, bk = (tid >> 6) * 8;
  us8 rah[2], ral[2];
  BRaw<float, BMODE> rb[8];
  const BSrc<float> bs = b_source<float, BMODE>(gb, it, n0 + 2 * bp);
  auto gload = [&](int k0) {
    const int64_t o = (int64_t)(m0 + ar) * gb.lda + k0 + ak;
#pragma unroll
    for (int v = 0; v < 2; v++) {
      rah[v] = v == 0 || arow ? *(const us8 *)(Ahg + o + 64 * v * gb.lda) : (us8){0, 0, 0, 0, 0, 0, 0, 0};
      ral[v] = v == 0 || arow ? *(const us8 *)(Alg + o + 64 * v * gb.lda) : (us8){0, 0, 0, 0, 0, 0, 0, 0};
    }
#pragma unroll
    for (int q = 0; q < 8; q++) rb[q] = load_b<float, BMODE>(bs, k0 + bk + q);
  };
  auto put = [&](int buf, int k0) {
#pragma unroll
    for (int v = 0; v < 2; v++) {
      *(us8 *)&Ah[buf][ar + 64 * v][ak] = rah[v];
      *(us8 *)&Al[buf][ar + 64 * v][ak] = ral[v];
    }
    us8 bh0, bl0, bh1, bl1;
#pragma unroll
    for (int q = 0; q < 8; q++) {
      const pair_t<float> b = b_value<float, BMODE>(bs, rb[q], k0 + bk + q);
      unsigned short h, l;
      split_bf16(b.a, h, l);
      bh0[q] = h;
      bl0[q] = l;
      split_bf16(b.b, h, l);
      bh1[q] = h;
      bl1[q] = l;
    }
    *(us8 *)&Bh[buf][2 * bp][bk] = bh0;
    *(us8 *)&Bl[buf][2 * bp][bk] = bl0;
    *(us8 *)&Bh[buf][2 * bp + 1][bk] = bh1;
    *(us8 *)&Bl[buf][2 * bp + 1][bk] = bl1;
  };
  f4 acc[4][4], cor[4][4];
#pragma unroll
  for (int i = 0; i < 4; i++)
#pragma unroll
    for (int j = 0; j < 4; j++) acc[i][j] = cor[i][j] = (f4){0, 0, 0, 0};
  gload(0);
  put(0, 0);
  if (BK < gb.K) gload(BK);
  __syncthreads();
  for (int k0 = 0, buf = 0; k0 < gb.K; k0 += BK, buf ^= 1) {
    if (k0 + BK < gb.K) put(buf ^ 1, k0 + BK);
    if (k0 + 2 * BK < gb.K) gload(k0 + 2 * BK);
    const int kq = 8 * (lane >> 4);
    bf8 bhv[4], blv[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int col = 64 * wc + 16 * j + (lane & 15);
      bhv[j] = __builtin_bit_cast(bf8, *(const us8 *)&Bh[buf][col][kq]);
      blv[j] = __builtin_bit_cast(bf8, *(const us8 *)&Bl[buf][col][kq]);
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int row = 64 * wr + 16 * i + (lane & 15);
      const bf8 ah = __builtin_bit_cast(bf8, *(const us8 *)&Ah[buf][row][kq]);
      const bf8 al = __builtin_bit_cast(bf8, *(const us8 *)&Al[buf][row][kq]);
#pragma unroll
      for (int j = 0; j < 4; j++) {
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bhv[j], acc[i][j], 0, 0, 0);
        cor[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, blv[j], cor[i][j], 0, 0, 0);
        cor[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al, bhv[j], cor[i][j], 0, 0, 0);
      }
    }
    __syncthreads();
  }
  float *C = (float *)it.C;
#pragma unroll
  for (int i = 0; i < 4; i++)
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        int row = m0 + 64 * wr + 16 * i + 4 * (lane >> 4) + r;
        int col = n0 + 64 * wc + 16 * j + (lane & 15);
        if (row < gb.M && col < it.N) C[(int64_t)row * it.N + col] = acc[i][j][r] + cor[i][j][r];
      }
}

#ifndef CHM_BF16_BK
#define CHM_BF16_BK 32
#endif

// ---------------------------------------------------------------- launch timing
// Measurement aid: while enabled (chm_dht_timing(1)), every product launch
// on a stream that is not being captured is bracketed by two HIP events
// recorded on its own stream, kept with the launch's algorithmic flops
// (2 M K N per item: real FP32-equivalent work for the split-BF16 form).
struct TimedLaunch {
  hipEvent_t a, b;
  double flops;
  int kind;
};
static std::mutex t_mu;
static bool t_on = false;
static std::vector<TimedLaunch> t_launches;

static void t_clear() {
  for (auto &t : t_launches) {
    hipEventDestroy(t.a);
    hipEventDestroy(t.b);
  }
  t_launches.clear();
}

extern "C" int chm_dht_timing(int32_t enable) {
  std::lock_guard<std::mutex> lock(t_mu);
  t_clear();
  t_on = enable != 0;
  return CHM_OK;
}

extern "C" int64_t chm_dht_timing_collect(double *ms, double *flops, int32_t *kind, int64_t max) {
  std::lock_guard<std::mutex> lock(t_mu);
  int64_t n = 0;
  for (auto &t : t_launches) {
    if (n >= max) break;
    if (hipEventSynchronize(t.b) != hipSuccess) return -1;
    float v = 0.f;
    if (hipEventElapsedTime(&v, t.a, t.b) != hipSuccess) return -1;
    if (ms) ms[n] = v;
    if (flops) flops[n] = t.flops;
    if (kind) kind[n] = t.kind;
    n++;
  }
  t_clear();
  return n;
}

static bool t_begin(hipStream_t st, TimedLaunch *t) {
  std::lock_guard<std::mutex> lock(t_mu);
  if (!t_on) return false;
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(st, &cs) != hipSuccess || cs != hipStreamCaptureStatusNone) return false;
  if (hipEventCreate(&t->a) != hipSuccess) return false;
  if (hipEventCreate(&t->b) != hipSuccess) {
    hipEventDestroy(t->a);
    return false;
  }
  hipEventRecord(t->a, st);
  return true;
}

static void t_end(hipStream_t st, TimedLaunch *t) {
  hipEventRecord(t->b, st);
  std::lock_guard<std::mutex> lock(t_mu);
  t_launches.push_back(*t);
}

int chm_gemm_launch(const GemmBatch &gb_in, int nitems, int kind, hipStream_t st) {
  if (nitems <= 0) return CHM_OK;
  if (nitems > GEMM_MAXB || gb_in.M <= 0 || gb_in.K <= 0) return CHM_EINVAL;
  if (gb_in.lda < gemm_lda(gb_in.K)) return CHM_EINVAL;
  GemmBatch gb = gb_in;
  gb.nitems = nitems;
  // A complex B operand taken as it is (alpha = 1, no second operand, no
  // m = -1 map) is a real [K][2 Nx] matrix: read it directly.
  bool plain = gb.bmode == 1;
  double cols = 0;
  for (int i = 0; i < nitems; i++) {
    const GemmItem &it = gb.it[i];
    if (it.N <= 0 || (gb.bmode == 1 && it.N != 2 * gb.Nx)) return CHM_EINVAL;
    plain = plain && it.alpha.x == 1.0 && it.alpha.y == 0.0 && !it.Y && !it.remapX;
    cols += it.N;
  }
  if (plain) gb.bmode = 0;
  // split-BF16: 128 x 128 tiles when they fill the GPU's rounds of 512 blocks
  // (two per CU) to two thirds at least: K = 511, 512 blocks 76 us against 86
  // with 64 x 64 tiles (with the row FFT of the transform), 2560 362 against
  // 437; K = 255, 512 blocks 57 against 62, but 576 blocks 39 against 34.5
  // (product alone), 640 78 against 76 and 256 38.8 against 38.0.  The FP64 /
  // FP32 products keep 64 x 64 tiles: the larger tile measured slower there
  // (3.11 -> 3.65 ms per step at 4096 x 512), its 64 accumulators per lane
  // allow only two waves per SIMD against seven.
  const int64_t big = gemm_blocks(gb, 128, 128), rounds = (big + 511) / 512;
  const bool use128 = kind == GEMM_BF16X3 && big >= 512 && 3 * big >= 2 * 512 * rounds;
  const unsigned grid = use128 ? gemm_blocks(gb, 128, 128) : gemm_blocks(gb, BM, BN);
  bool odd = false;
  for (int i = 0; i < nitems; i++) odd = odd || (gb.it[i].N & 1);
  if (odd && kind != GEMM_F64) return CHM_EUNSUPPORTED;
  TimedLaunch tl;
  const bool timed = t_begin(st, &tl);
  const bool cplx = gb.bmode == 1;
  if (kind == GEMM_F64) {
    if (cplx) k_gemm<double, 1><<<grid, 256, 0, st>>>(gb);
    else if (odd) k_gemm<double, 2><<<grid, 256, 0, st>>>(gb);
    else k_gemm<double, 0><<<grid, 256, 0, st>>>(gb);
  } else if (kind == GEMM_F32) {
    if (cplx) k_gemm<float, 1><<<grid, 256, 0, st>>>(gb);
    else k_gemm<float, 0><<<grid, 256, 0, st>>>(gb);
  } else if (use128) {
    if (cplx) k_gemm128_bf16x3<1><<<grid, 256, 0, st>>>(gb);
    else k_gemm128_bf16x3<0><<<grid, 256, 0, st>>>(gb);
  } else {
    if (cplx) k_gemm_bf16x3<CHM_BF16_BK, 1><<<grid, 256, 0, st>>>(gb);
    else k_gemm_bf16x3<CHM_BF16_BK, 0><<<grid, 256, 0, st>>>(gb);
  }
  if (timed) {
    tl.flops = 2.0 * gb.M * (double)gb.K * cols;
    tl.kind = kind;
    t_end(st, &tl);
  }
  CHM_CHECK_LAUNCH();
  return CHM_OK;
}

// Zero-padded copy of a row-major [M][K] double matrix into the layout the
// products read: [round_up(M, 64)][gemm_lda(K)] as double, float or split BF16.
__global__ void k_pad_table(const double *__restrict__ src, int M, int K, int Mp, int lda, double *d64,
                            float *f32, unsigned short *hi, unsigned short *lo) {
  int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= (int64_t)Mp * lda) return;
  int i = (int)(e / lda), k = (int)(e % lda);
  double v = (i < M && k < K) ? src[(int64_t)i * K + k] : 0.0;
  if (d64) d64[e] = v;
  if (f32) f32[e] = (float)v;
  if (hi) {
    __bf16 h = (__bf16)(float)v;
    __bf16 l = (__bf16)(float)(v - (double)(float)h);
    hi[e] = __builtin_bit_cast(unsigned short, h);
    lo[e] = __builtin_bit_cast(unsigned short, l);
  }
}

extern "C" size_t chm_dht_table_elems(int32_t M, int32_t K) {
  return (size_t)((M + BM - 1) / BM * BM) * gemm_lda(K);
}

extern "C" int chm_pad_table(const double *src, int32_t M, int32_t K, double *d64, float *f32,
                             uint16_t *bf16_hi, uint16_t *bf16_lo, void *stream) {
  if (!src || M <= 0 || K <= 0 || ((bf16_hi == nullptr) != (bf16_lo == nullptr))) return CHM_EINVAL;
  int Mp = (M + BM - 1) / BM * BM, lda = gemm_lda(K);
  int64_t n = (int64_t)Mp * lda;
  k_pad_table<<<chm_blocks(n, 256), 256, 0, (hipStream_t)stream>>>(src, M, K, Mp, lda, d64, f32,
                                                                   (unsigned short *)bf16_hi,
                                                                   (unsigned short *)bf16_lo);
  CHM_CHECK_LAUNCH();
  return CHM_OK;
}

// Plain real product for table construction and tests:
// C[M x N] = A[M x K] @ B[K x N]; A padded as chm_pad_table writes it
// ([round_up(M,64)][round_up(K,64)]), B and C row-major, contiguous.
extern "C" int chm_gemm_f64(const double *A, const double *B, double *C, int32_t M, int32_t K,
                            int32_t N, void *stream) {
  GemmBatch gb = {};
  gb.M = M;
  gb.K = K;
  gb.lda = gemm_lda(K);
  gb.bmode = 0;
  gb.it[0].A = A;
  gb.it[0].X = B;
  gb.it[0].C = C;
  gb.it[0].N = N;
  return chm_gemm_launch(gb, 1, GEMM_F64, (hipStream_t)stream);
}
