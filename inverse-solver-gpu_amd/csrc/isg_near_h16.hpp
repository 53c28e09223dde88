// isg_near_h16.hpp -- near field + L2P (k_near_h16) and P2M (k_p2m_h16) of the
// FP32 operator on gfx950's FP16 matrix cores with split operands
// (v_mfma_f32_16x16x32_f16).
//
// Every FP32 operand x is carried as two FP16 numbers, hi = rne16(2^e x) and
// lo = rne16(2^e x - hi), with a power-of-two scale 2^e chosen so that
// |2^e x| < 2^14 -- per table, and for the data per workgroup and right-hand side
// (the leaf level's M2M: per box; k_down_h16: per parent).  hi + lo holds x to 2^-22
// relative (elements below 2^-16 of the largest one, whose lo is subnormal, to 2^-38
// of the largest, absolutely; the largest one's field reaches every output of the
// workgroup, so that does not show: with amplitudes over 30 and 40 octaves and with
// point sources 2^24 above the rest, the error of each leaf box relative to its own
// field is that of the FP32 kernels or less, 1 to 15 right-hand sides, 64 to 2048
// px).  A product x a is formed
// as hi.hi + hi.lo + lo.hi in FP32 accumulators (the dropped lo.lo term is
// below 2^-22 relative): three FP16 MFMAs, each 16 times the FP32 rate, for
// one FP32 MFMA's worth of products.  Complex products take the four-product
// form (cr += dr ar - di ai, ci += dr ai + di ar): 12 MFMAs per 16 x 16 x 32
// block.  The scales are exact powers of two and are divided out of the FP32
// accumulators at the end.
//
// The near field and L2P run in the mirror-symmetric basis of a leaf box
// (isg_near_sym.hpp: a quarter of the multiplications): the data operand is
// the folded quarter window, formed in FP32 and then split.
//
// Reference counterpart: the near-field and L2P stages of matvec_gpu.cu
// (kernels.cu:32-81, :292-319); the results equal the FP32 kernels' to the
// split's 2^-22.
#pragma once

#include "isg_kernels.hpp"
#include "isg_near_sym.hpp"

namespace isg {

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));

// Tuning values of the near and P2M stages that select the split kernels
// (FP32 operator); the near stage has one kernel for both.
constexpr int kNearSplit = 128;
constexpr int kNearSplitWide = 256;

// Power-of-two exponent e with |2^e m| < 2^14 for the largest magnitude m
// (0 for m = 0 or m not finite: Inf / NaN then propagate as in FP32).
__host__ __device__ inline int h16_scale_exp(float m) {
  if (!(m > 0.f) || !(m <= 3.0e38f)) return 0;
  int e;
  (void)frexpf(m, &e);  // m = f 2^e, f in [0.5, 1)
  e = 14 - e;
  return e > 126 ? 126 : (e < -126 ? -126 : e);
}

// element e of hi and lo: the split of v
__device__ __forceinline__ void h16_split(float v, v8h& hi, v8h& lo, int e) {
  const _Float16 h = (_Float16)v;
  hi[e] = h;
  lo[e] = (_Float16)(v - (float)h);  // exact difference: at most 13 significant bits
}

__device__ __forceinline__ float h16_absmax(float4 v) {
  return fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w)));
}

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
  return v;
}

// Workgroup maxima of N values; every thread gets all of them.
template <int N>
__device__ __forceinline__ void block_max(float (&m)[N], float (*red)[kBlock / 64]) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int q = 0; q < N; q++) m[q] = wave_max(m[q]);
  if (lane == 0)
#pragma unroll
    for (int q = 0; q < N; q++) red[q][w] = m[q];
  __syncthreads();
#pragma unroll
  for (int q = 0; q < N; q++) {
    float v = red[q][0];
#pragma unroll
    for (int i = 1; i < kBlock / 64; i++) v = fmaxf(v, red[q][i]);
    m[q] = v;
  }
}

// 16-byte load from a caller's vector: complex FP32 elements, aligned to 8 bytes
// only (the loads are the same instructions, which take any such address).
typedef float v4f_8 __attribute__((ext_vector_type(4), aligned(8)));
__device__ __forceinline__ float4 h16_load(const zf* p, int i) {  // elements 2 i, 2 i + 1
  const v4f_8 v = reinterpret_cast<const v4f_8*>(p)[i];
  return make_float4(v.x, v.y, v.z, v.w);
}

// a[q] for a runtime q without indexing a private array (which would live in scratch)
template <typename T>
__device__ __forceinline__ T sel2(const T (&a)[2], int q) {
  return q ? a[1] : a[0];
}

__device__ __forceinline__ v8h h16_neg(v8h v) {
  return __builtin_bit_cast(v8h, __builtin_bit_cast(v4u, v) ^ 0x80008000u);
}

// cr + i ci += (a0 + a1 + i (a2 + a3)) (b0 + b1 + i (b2 + b3)) without the
// lo.lo terms; a = data parts (re hi, re lo, im hi, im lo), b = table parts,
// nb = -b2, -b3.  The two accumulators alternate so that consecutive MFMAs
// are independent.
__device__ __forceinline__ void h16_cmac(const v8h (&a)[4], const v8h (&b)[4], const v8h (&nb)[2], v4f& cr,
                                         v4f& ci) {
  cr = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[0], b[0], cr, 0, 0, 0);
  ci = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[0], b[2], ci, 0, 0, 0);
  cr = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[0], b[1], cr, 0, 0, 0);
  ci = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[0], b[3], ci, 0, 0, 0);
  cr = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[1], b[0], cr, 0, 0, 0);
  ci = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[1], b[2], ci, 0, 0, 0);
  cr = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[2], nb[0], cr, 0, 0, 0);
  ci = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[2], b[0], ci, 0, 0, 0);
  cr = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[2], nb[1], cr, 0, 0, 0);
  ci = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[2], b[1], ci, 0, 0, 0);
  cr = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[3], nb[0], cr, 0, 0, 0);
  ci = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[3], b[0], ci, 0, 0, 0);
}

// Split-FP16 table: out[b][part][g][m] (m < ncolp) = 8 FP16 parts of
// 2^ex src[(b / per) bstride + k srow + m], k = 32 (b % per) + 8 g + e,
// e = 0..7 (zero for k >= kmax or m >= ncol); one thread per (b, g, m).
static __global__ void __launch_bounds__(256) k_split16(const zf* __restrict__ src, int per, long bstride, int kmax,
                                                        int srow, int ncol, int ncolp, int ex, int nblk,
                                                        v8h* __restrict__ out) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= nblk * 4 * ncolp) return;
  const int m = t % ncolp, g = (t / ncolp) & 3, b = t / (4 * ncolp);
  const float s = ldexpf(1.f, ex);
  v8h ph[4];
#pragma unroll
  for (int e = 0; e < 8; e++) {
    const int k = 32 * (b % per) + 8 * g + e;
    const zf v = (k < kmax && m < ncol) ? src[(long)(b / per) * bstride + (long)k * srow + m] : mkc<float>(0.f, 0.f);
    h16_split(v.x * s, ph[0], ph[1], e);
    h16_split(v.y * s, ph[2], ph[3], e);
  }
#pragma unroll
  for (int P = 0; P < 4; P++) out[((long)(b * 4 + P) * 4 + g) * ncolp + m] = ph[P];
}

// Split tables of k_near_h16, from the FP32 symmetric ones: chunk b of 32
// k-slots, out[b][c][part][lk][col] = 8 FP16 parts (slots 8 lk .. +7).
//   near (tn, 5 chunks): slot (b, lk, e) is quarter-window pixel (i, j): b < 3:
//     (4 + e, 4 b + lk), eight pixels of a neighbour box's row; then
//     (e % 4, 2 (4 (b - 3) + lk) + e / 4), two rows of the box's own half; zero past 144
//   l2p (tl, 1 chunk): slot (lk, e) is direction orbit 8 lk + e, zero past nrep
constexpr int kS16Chunks = 5;
static __global__ void __launch_bounds__(256) k_split16_sym(const zf* __restrict__ tn, int et,
                                                            const zf* __restrict__ tl, int nrep, int eb,
                                                            v8h* __restrict__ out) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (kS16Chunks + 1) * 4 * 4 * 16) return;
  const int col = t & 15, lk = (t >> 4) & 3, c = (t >> 6) & 3, b = t >> 8;
  const float s = ldexpf(1.f, b < kS16Chunks ? et : eb);
  v8h ph[4];
#pragma unroll
  for (int e = 0; e < 8; e++) {
    zf v = mkc<float>(0.f, 0.f);
    if (b < kS16Chunks) {
      const int i = b < 3 ? 4 + e : e & 3, j = b < 3 ? 4 * b + lk : 2 * (4 * (b - 3) + lk) + (e >> 2);
      if (j < 12) v = tn[(c * kSymK + 12 * j + i) * 16 + col];
    } else if (8 * lk + e < nrep) {
      v = tl[(c * nrep + 8 * lk + e) * 16 + col];
    }
    h16_split(v.x * s, ph[0], ph[1], e);
    h16_split(v.y * s, ph[2], ph[3], e);
  }
#pragma unroll
  for (int P = 0; P < 4; P++) out[(((b * 4 + c) * 4 + P) * 4 + lk) * 16 + col] = ph[P];
}

// Near field + L2P of the FP32 operator, split FP16, symmetric classes.
// Workgroup: 64 Morton-consecutive boxes (8 x 8) of one right-hand side.  The
// 10 x 10-box halo is loaded once into registers, its largest component sets
// the data scale (two bits of headroom: a folded value sums four), and the
// scaled FP32 pixels are staged in LDS.  Wave w owns row
// blocks 2 (w / 2), +1 (16 boxes each) and the classes odd or even in y by
// w % 2, even and odd in x: a table fragment then serves two row blocks and a
// halo pixel is read by two waves.  Per chunk and row block a lane reads the
// four mirror images of its 8 slots (16-byte reads; the 16 boxes of a block
// fall in distinct banks), folds them (4 FP32 operations per operand) and
// splits them (about as many), for 24 MFMAs.
// What bounds it (1024^2 x 64 right-hand sides, 498 us; the dense split kernel took
// 900): vector work 320 us, MFMA 123, memory 1.65 GB = 350 us; three workgroups per
// CU instead of two were worth 572 -> 498 us, hence the 664-element pitch and the
// 168-register limit.
constexpr int kS16Box = 66, kS16Row = 664;  // halo layout: 16-byte reads need box / 2 odd, row / 2 = 4 mod 8
constexpr int kS16Rows = 10 * kS16Row;       // LDS elements of the halo: with the static part 53.7 KB, three workgroups per CU
// LDS bytes for S leaf directions; the kernel takes S <= 124 (one L2P chunk)
__host__ __device__ inline size_t s16_lds(int S) {
  const int l2p = 64 * (S + 1), out = 64 * 64;
  const int m = l2p > out ? l2p : out;
  return (size_t)(kS16Rows > m ? kS16Rows : m) * sizeof(zf);
}
constexpr int kS16MaxS = 124;

typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef float v2f __attribute__((ext_vector_type(2)));

// v - hi, exact, as one mixed-precision multiply-add per element (the compiler
// would convert hi back and subtract)
__device__ __forceinline__ v2f h16_rest(v2f v, v2h hi) {
  v2f r;
  asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[0,0,0] op_sel_hi:[1,0,0]" : "=v"(r.x) : "v"(hi), "v"(v.x));
  asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r.y) : "v"(hi), "v"(v.y));
  return r;
}

// elements e, e + 1 of the four parts of a pair of complex values
__device__ __forceinline__ void h16_split_pair(v2f re, v2f im, v8h (&a)[4], int e) {
  const v2h rh = __builtin_convertvector(re, v2h), mh = __builtin_convertvector(im, v2h);
  const v2h rl = __builtin_convertvector(h16_rest(re, rh), v2h), ml = __builtin_convertvector(h16_rest(im, mh), v2h);
  a[0][e] = rh.x;
  a[0][e + 1] = rh.y;
  a[1][e] = rl.x;
  a[1][e + 1] = rl.y;
  a[2][e] = mh.x;
  a[2][e + 1] = mh.y;
  a[3][e] = ml.x;
  a[3][e + 1] = ml.y;
}

template <int POST>
__global__ void __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(3)))
k_near_h16(const zf* __restrict__ y, long ys, const zf* __restrict__ loc, long ls, zf* __restrict__ r, long rs,
           const v8h* __restrict__ tab, int et, int eb, int S, int nbs, const int* __restrict__ act,
           NearPost<float> post) {
  constexpr int BS = kS16Box, RS = kS16Row;
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  zf* tile = reinterpret_cast<zf*>(smem_raw);
  __shared__ int hoff[100];
  __shared__ float red[2][kBlock / 64];
  const int rhs = blockIdx.y;
  if (rhs_off(act, rhs)) return;
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, lk = lane >> 4;
  const int oy = w & 1, rb0 = 2 * (w >> 1);
  const float sy = oy ? -1.f : 1.f;
  const long b0 = (long)xcd_block() * 64;
  const int X0 = (int)compact2((unsigned)b0), Y0 = (int)compact2((unsigned)b0 >> 1);
  if (tid < 100) {
    const int hx = tid % 10, hy = tid / 10, sxb = X0 - 1 + hx, syb = Y0 - 1 + hy;
    hoff[tid] = (sxb >= 0 && syb >= 0 && sxb < nbs && syb < nbs) ? (int)morton2(sxb, syb) * 64 : -1;
  }
  __syncthreads();
  // table fragments of this wave's two classes (2 oy, 2 oy + 1)
  const v8h* tl = tab + (2 * oy * 4 * 4 + lk) * 16 + li;  // + chunk * 1024 + class * 256 + part * 64
  auto load_b = [&](v8h (&b)[2][4], int chunk) {
#pragma unroll
    for (int c = 0; c < 2; c++)
#pragma unroll
      for (int P = 0; P < 4; P++) b[c][P] = tl[chunk * 1024 + c * 256 + P * 64];
  };
  v8h bt[2][2][4];
  load_b(bt[0], 0);
  int es;
  {
    constexpr int NU = 13;  // 100 boxes x 32 float4
    const zf* yq = y + (long)rhs * ys;
    float4 v[NU];
    float m[1] = {0.f};
#pragma unroll
    for (int u = 0; u < NU; u++) {
      const int e = tid + u * kBlock, ec = e < 3200 ? e : 3199;
      const int off = hoff[ec >> 5];
      v[u] = h16_load(yq, ((off < 0 ? 0 : off) >> 1) + (ec & 31));
      if (off < 0) v[u] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
#pragma unroll
    for (int u = 0; u < NU; u++) m[0] = fmaxf(m[0], h16_absmax(v[u]));  // clamped repeats change no maximum
    block_max<1>(m, red);
    es = h16_scale_exp(m[0]) - 2;
    const float s = ldexpf(1.f, es);
#pragma unroll
    for (int u = 0; u < NU; u++) {
      const int e = tid + u * kBlock;
      const int h = e >> 5;
      if (e < 3200)
        *reinterpret_cast<float4*>(&tile[h * BS + h / 10 * (RS - 10 * BS) + 2 * (e & 31)]) =
            make_float4(v[u].x * s, v[u].y * s, v[u].z * s, v[u].w * s);
    }
  }
  v4f cr[2][2], cn[2][2], ci[2][2];  // [row block][class]: real part cr - cn, imaginary part ci
#pragma unroll
  for (int j = 0; j < 2; j++)
#pragma unroll
    for (int c = 0; c < 2; c++) {
      cr[j][c] = v4f{0, 0, 0, 0};
      cn[j][c] = v4f{0, 0, 0, 0};
      ci[j][c] = v4f{0, 0, 0, 0};
    }
  int base[2];  // window corner (upper left neighbour) of box 16 (rb0 + j) + li
#pragma unroll
  for (int j = 0; j < 2; j++) {
    const unsigned c = (unsigned)(16 * (rb0 + j) + li);
    base[j] = (int)compact2(c >> 1) * RS + (int)compact2(c) * BS;
  }
  // a pair of slots folded: rows first (sign sy), then both column parities
  auto fold2 = [&](float4 pp, float4 mp, float4 pm, float4 mm, v8h (&a)[2][4], int e) {
    // (pp, pm: columns ascending; mp, mm: descending)
    const float ex0 = fmaf(sy, pm.x, pp.x), ey0 = fmaf(sy, pm.y, pp.y), ex1 = fmaf(sy, pm.z, pp.z),
                ey1 = fmaf(sy, pm.w, pp.w);
    const float fx0 = fmaf(sy, mm.z, mp.z), fy0 = fmaf(sy, mm.w, mp.w), fx1 = fmaf(sy, mm.x, mp.x),
                fy1 = fmaf(sy, mm.y, mp.y);
    h16_split_pair(v2f{ex0 + fx0, ex1 + fx1}, v2f{ey0 + fy0, ey1 + fy1}, a[0], e);
    h16_split_pair(v2f{ex0 - fx0, ex1 - fx1}, v2f{ey0 - fy0, ey1 - fy1}, a[1], e);
  };
  // both classes' chains interleaved: six independent accumulators
  auto mac = [&](const v8h (&a)[2][4], const v8h (&b)[2][4], int j) {
#define ISG_S16(ACC, P, Q)                \
  _Pragma("unroll") for (int c = 0; c < 2; c++) ACC[j][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[c][P], b[c][Q], ACC[j][c], 0, 0, 0);
    ISG_S16(cr, 0, 0)
    ISG_S16(ci, 0, 2)
    ISG_S16(cn, 2, 2)
    ISG_S16(cr, 0, 1)
    ISG_S16(ci, 0, 3)
    ISG_S16(cn, 2, 3)
    ISG_S16(cr, 1, 0)
    ISG_S16(ci, 1, 2)
    ISG_S16(cn, 3, 2)
    ISG_S16(ci, 2, 0)
    ISG_S16(ci, 2, 1)
    ISG_S16(ci, 3, 0)
#undef ISG_S16
  };
  __syncthreads();
#pragma unroll
  for (int b = 0; b < kS16Chunks; b++) {
    load_b(bt[(b + 1) & 1], b + 1);  // (the last one is the L2P's)
#pragma unroll
    for (int j = 0; j < 2; j++) {
      v8h a[2][4];
      if (b < 3) {
        // rows 12 + 4 b + lk and 11 - 4 b - lk of the window, eight columns of the right and left neighbours
        const zf* p = tile + base[j] + 8 * lk + (b == 0 ? RS + 32 : (b == 1 ? 2 * RS : 2 * RS + 32));
        const zf* q = tile + base[j] + 8 * (3 - lk) + (b == 0 ? RS : (b == 1 ? 32 : 0));
#pragma unroll
        for (int t = 0; t < 4; t++) {
          auto at = [&](const zf* s, int o) { return *reinterpret_cast<const float4*>(s + o); };
          fold2(at(p, 2 * BS + 2 * t), at(p, 6 - 2 * t), at(q, 2 * BS + 2 * t), at(q, 6 - 2 * t), a, 2 * t);
        }
      } else {
        // the box's own columns: quarter-window rows j0, j0 + 1 (two slots' worth of lanes idle in the last chunk)
        const int j0 = b == 3 ? 2 * lk : 8 + 2 * (lk & 1);
        const zf* p = tile + base[j] + BS + (j0 < 4 ? RS + (4 + j0) * 8 : 2 * RS + (j0 - 4) * 8);
        const zf* q = tile + base[j] + BS + (j0 < 4 ? RS + (3 - j0) * 8 : (11 - j0) * 8);
#pragma unroll
        for (int t = 0; t < 4; t++) {
          auto at = [&](const zf* s, int o) { return *reinterpret_cast<const float4*>(s + o); };
          const int up = (t >> 1) * 8, e = 2 * (t & 1);  // second row; column pair
          fold2(at(p, up + 4 + e), at(p, up + 2 - e), at(q, 4 + e - up), at(q, 2 - e - up), a, 2 * t);
        }
      }
      mac(a, bt[b & 1], j);
    }
  }
  // ---- L2P: the tile's locals staged raw, rows of S + 1; orbits m = 8 lk + e
  __syncthreads();
  int el;
  {
    float m[1] = {0.f};
    const int n4 = 32 * S;  // 64 boxes x S locals in float4 (S even)
    constexpr int U = 9;
    const float4* lq = reinterpret_cast<const float4*>(loc + (long)rhs * ls + b0 * S);
    const int hs = S >> 1, db = kBlock / hs, dk = kBlock - db * hs;  // box and pair of element e, stepped
    int bx = tid / hs, kp = tid - bx * hs;
    for (int e0 = tid; e0 < n4; e0 += U * kBlock) {
      float4 t[U];
      int at[U];
#pragma unroll
      for (int u = 0; u < U; u++) {
        const int e = e0 + u * kBlock;
        t[u] = lq[e < n4 ? e : n4 - 1];
        at[u] = bx * (S + 1) + 2 * kp;
        bx += db;
        kp += dk;
        if (kp >= hs) {
          kp -= hs;
          bx++;
        }
      }
#pragma unroll
      for (int u = 0; u < U; u++) {
        m[0] = fmaxf(m[0], h16_absmax(t[u]));  // clamped repeats change no maximum
        if (e0 + u * kBlock < n4) {
          tile[at[u]] = mkc<float>(t[u].x, t[u].y);
          tile[at[u] + 1] = mkc<float>(t[u].z, t[u].w);
        }
      }
    }
    block_max<1>(m, red + 1);  // (its barrier also covers the staging)
    el = h16_scale_exp(m[0]) - 2;
  }
  {
    // near accumulators carry 2^(es + et); bring them to the L2P's 2^(el + eb)
    const int n = (el + eb) - (es + et);
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int c = 0; c < 2; c++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
          cr[j][c][i] = ldexpf(cr[j][c][i] - cn[j][c][i], n);
          cn[j][c][i] = 0.f;
          ci[j][c][i] = ldexpf(ci[j][c][i], n);
        }
  }
  const float sl = ldexpf(1.f, el);
#pragma unroll
  for (int j = 0; j < 2; j++) {
    const zf* t = tile + (16 * (rb0 + j) + li) * (S + 1);
    v8h a[2][4];
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
      zf g[2], h[2];
#pragma unroll
      for (int u = 0; u < 2; u++) {
        const int m = min(8 * lk + e + u, S >> 2);  // (past S / 4 the table is zero)
        const zf v0 = t[m], v1 = t[(S >> 1) - m], v2 = t[m ? S - m : 0], v3 = t[(S >> 1) + m];
        g[u] = mkc<float>(fmaf(sy, v2.x, v0.x) * sl, fmaf(sy, v2.y, v0.y) * sl);
        h[u] = mkc<float>(fmaf(sy, v3.x, v1.x) * sl, fmaf(sy, v3.y, v1.y) * sl);
      }
      h16_split_pair(v2f{g[0].x + h[0].x, g[1].x + h[1].x}, v2f{g[0].y + h[0].y, g[1].y + h[1].y}, a[0], e);
      h16_split_pair(v2f{g[0].x - h[0].x, g[1].x - h[1].x}, v2f{g[0].y - h[0].y, g[1].y - h[1].y}, a[1], e);
    }
    mac(a, bt[kS16Chunks & 1], j);
  }
  // ---- back to pixels through LDS (as k_near_mfma)
  __syncthreads();
  {
    const int n = -(el + eb), p = li & 3, q = li >> 2;
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int c = 0; c < 2; c++) {
        const int px = (oy ? 3 - q : 4 + q) * 8 + (c ? 3 - p : 4 + p);
#pragma unroll
        for (int i = 0; i < 4; i++)
          tile[(16 * (rb0 + j) + 4 * lk + i) * 64 + px] = mkc<float>(ldexpf(cr[j][c][i] - cn[j][c][i], n), ldexpf(ci[j][c][i], n));
      }
  }
  __syncthreads();
  sym_unfold<float, 64>(tile);
  __syncthreads();
  near_epilogue<float, float, 64, POST>(tile, r, rs, b0, rhs, post);
}

// Maximum of non-negative values over the 16 lanes of a row.
__device__ __forceinline__ float row_max(float v) {
  unsigned m = __builtin_bit_cast(unsigned, v);  // ordered as the floats are (a NaN above all)
  m = max(m, (unsigned)__builtin_amdgcn_update_dpp(0, (int)m, 0x128, 0xf, 0xf, false));  // row_ror:8, 4, 2, 1
  m = max(m, (unsigned)__builtin_amdgcn_update_dpp(0, (int)m, 0x124, 0xf, 0xf, false));
  m = max(m, (unsigned)__builtin_amdgcn_update_dpp(0, (int)m, 0x122, 0xf, 0xf, false));
  m = max(m, (unsigned)__builtin_amdgcn_update_dpp(0, (int)m, 0x121, 0xf, 0xf, false));
  return __builtin_bit_cast(float, m);
}

// P2M of the FP32 operator on split FP16: agm[box][s] = sum_n coeffT[n][s]
// y[box 64 + n] for 32 Morton-consecutive boxes of two right-hand sides.
// The workgroup's input (2 x 32 boxes x 64 pixels) is loaded once into
// registers, whole lines per instruction (8 pixels per thread and 64-byte stride
// between lanes, with three to five arrays in flight, ran from L2: 697 -> 557 us
// for STEP 2 at 1024 px x 64), its largest component per
// right-hand side sets the data scale, and it is staged split in LDS as
// [rhs][part][pixel group 8][box 32] x 8 FP16 (boxes XOR 2 (g mod 4) against
// bank conflicts).  Wave w owns right-hand side w / 2, row block w % 2 (16
// boxes) and all ceil(S / 16) column blocks (samples); K = 64 pixels in two
// MFMA chunks of 32.  The coefficient table coef[kc][part][g][s] (s padded to
// 16 ceil(S / 16), zero beyond S) carries its own scale 2^ec.  Results go
// straight from the accumulators to HBM: lane li stores sample 16 cb + li of
// box 16 j + 4 (lane / 16) + i, 16 consecutive samples per row.
// Grid (B / 32, ceil(nrhs / 2)), kBlock threads.
//
// UP: the interpolation to the parents (M2M of the leaf level) follows in the
// same workgroup, from the multipoles in registers (P2mUp).  They are scaled by
// their box's largest component, split again and staged in LDS, real parts
// first, then imaginary parts, with the first samples repeated past the end so
// that a window never wraps.  Rows of the matrix product are boxes, 16 of them
// the children of four parents, columns 16 parent samples, K the window of child
// samples (<= kUpWin, from a multiple of 8, padded to 64 by zeros of the table);
// wave w takes the parent samples 16 w + 64 u of all four row blocks.  A lane
// ends with the four children of one parent: shifted and summed in registers.
// HBM bounds both: alone, P2M wrote the multipoles in 239 us and M2M, on FP32
// matrix products, read them again in 289 us (1024 px x 64); together 361 us, and
// with STEP 2 or 3 620 and 566 instead of 557 + 289 and 485 + 289.
constexpr int kP2mH16MaxCB = 6;  // column blocks held per wave (S <= 96)
constexpr int kUpWin = 48, kUpPitch = 120, kUpRounds = 2, kUpCB = 5;
// kUpCB column blocks exactly; a window from any 8 j < S ends inside what is staged
constexpr int kUpMinS = 16 * kUpCB - 15, kUpMaxS = kUpPitch - kUpWin;
struct P2mUp {
  zf* par = nullptr;  // parents, ps between systems, Sp samples
  long ps = 0;
  const v8h* tab = nullptr;  // [sample block 16][k chunk 32][hi, lo][lane], scale 2^ec
  const int* s0 = nullptr;   // window start of each sample block
  const zf* shift = nullptr;  // [4][Sp]
  int Sp = 0, ec = 0;
};
// (at least 4 waves per SIMD: unbounded, the compiler hoists every
// coefficient fragment of both K chunks and takes 256 registers)
template <int STEP, bool UP>
__global__ void __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(4)))
k_p2m_h16(const zf* __restrict__ y, long ys, zf* __restrict__ agm, long as, const v8h* __restrict__ coef, int ec, int S,
          int nrhs, const int* __restrict__ act, P2mStep<float> step, P2mUp up) {
  __shared__ v8h hal[2 * 4 * 8 * 32];
  __shared__ float red[4][kBlock / 64];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int li = lane & 15, lk = lane >> 4;
  const int rw = w >> 1, j = w & 1;
  const int rhs[2] = {2 * (int)blockIdx.y, 2 * (int)blockIdx.y + 1};
  bool on[2];
#pragma unroll
  for (int q = 0; q < 2; q++) on[q] = rhs[q] < nrhs && !rhs_off(act, rhs[q]);
  if (!on[0] && !on[1]) return;
  const bool mine = sel2(on, rw);
  const int rv[2] = {on[0] ? rhs[0] : rhs[1], on[1] ? rhs[1] : rhs[0]};
  const long b0 = (long)xcd_block() * 32;
  const int ncb = UP ? kUpCB : (S + 15) / 16, ncolp = 16 * ncb;
  // load c of this thread: pixels 2 pr and 2 pr + 1 of group g8 of box bx + 8 c, so
  // that a wave's load and store instructions cover whole lines
  const int bx = tid >> 5, g8 = (tid >> 2) & 7, pr = tid & 3;
  float4 v[2][4];
#pragma unroll
  for (int q = 0; q < 2; q++) {
    const long o = (long)sel2(rv, q) * ys + b0 * 64 + 2 * tid;  // + 512 c
    if constexpr (STEP == 0) {
#pragma unroll
      for (int c = 0; c < 4; c++) v[q][c] = h16_load(y + o + 512 * c, 0);
    } else {
      // (a switched-off system's vectors stay as they are)
      if (!sel2(on, q)) {
#pragma unroll
        for (int c = 0; c < 4; c++) v[q][c] = make_float4(0.f, 0.f, 0.f, 0.f);
        continue;
      }
      const StepCoef cf = step_coef<STEP>(step, rhs[q], hal);  // (hal is filled behind block_max's barrier)
      const zd* g = step.g + rhs[q] * step.gs + b0 * 64 + 2 * tid;
      StepIn<float> in[8];
      auto ld = [&](const zf* a, zf StepIn<float>::*f) {
#pragma unroll
        for (int c = 0; c < 4; c++) {
          const float4 x = *reinterpret_cast<const float4*>(a + o + 512 * c);
          in[2 * c].*f = mkc<float>(x.x, x.y);
          in[2 * c + 1].*f = mkc<float>(x.z, x.w);
        }
      };
      ld(step.r, &StepIn<float>::r);
      if (STEP == 3 || !cf.first) ld(step.v, &StepIn<float>::v);
      if (STEP == 2 && !cf.first) ld(step.p, &StepIn<float>::p);
      if (!step.herm) {
#pragma unroll
        for (int c = 0; c < 4; c++) {
          in[2 * c].g = g[512 * c];
          in[2 * c + 1].g = g[512 * c + 1];
        }
      }
      float4 pv[4];
#pragma unroll
      for (int c = 0; c < 4; c++) {
        zf p0, p1;
        const zf y0 = step_value<STEP>(step, cf, in[2 * c], p0), y1 = step_value<STEP>(step, cf, in[2 * c + 1], p1);
        pv[c] = make_float4(p0.x, p0.y, p1.x, p1.y);
        v[q][c] = make_float4(y0.x, y0.y, y1.x, y1.y);
      }
#pragma unroll
      for (int c = 0; c < 4; c++) {
        *reinterpret_cast<float4*>(step.p + o + 512 * c) = pv[c];
        *reinterpret_cast<float4*>(step.y + o + 512 * c) = v[q][c];
      }
    }
  }
  int es[2];
  {
    float m[2];
#pragma unroll
    for (int q = 0; q < 2; q++) {
      m[q] = 0.f;
      if (sel2(on, q))
#pragma unroll
        for (int c = 0; c < 4; c++) m[q] = fmaxf(m[q], h16_absmax(v[q][c]));
    }
    block_max<2>(m, red);
    es[0] = h16_scale_exp(m[0]);
    es[1] = h16_scale_exp(m[1]);
  }
#pragma unroll
  for (int q = 0; q < 2; q++) {
    const float s = sel2(on, q) ? ldexpf(1.f, sel2(es, q)) : 0.f;
#pragma unroll
    for (int c = 0; c < 4; c++) {
      const v2f re = v2f{v[q][c].x * s, v[q][c].z * s}, im = v2f{v[q][c].y * s, v[q][c].w * s};
      const v2h rh = __builtin_convertvector(re, v2h), mh = __builtin_convertvector(im, v2h);
      const v2h part[4] = {rh, __builtin_convertvector(h16_rest(re, rh), v2h), mh,
                           __builtin_convertvector(h16_rest(im, mh), v2h)};
#pragma unroll
      for (int P = 0; P < 4; P++)
        reinterpret_cast<v2h*>(hal + ((q * 4 + P) * 8 + g8) * 32 + ((bx + 8 * c) ^ (2 * (g8 & 3))))[pr] = part[P];
    }
  }
  __syncthreads();
  if (!UP && !mine) return;  // no barrier follows
  v4f cr[kP2mH16MaxCB], ci[kP2mH16MaxCB];
#pragma unroll
  for (int c = 0; c < kP2mH16MaxCB; c++) {
    cr[c] = v4f{0, 0, 0, 0};
    ci[c] = v4f{0, 0, 0, 0};
  }
  const v8h* tl = coef + lk * ncolp + li;  // + (kc * 4 + P) * 4 * ncolp + 16 cb
#pragma unroll
  for (int kc = 0; kc < 2; kc++) {
    v8h a[4];
#pragma unroll
    for (int P = 0; P < 4; P++) a[P] = hal[((rw * 4 + P) * 8 + 4 * kc + lk) * 32 + ((16 * j + li) ^ (2 * lk))];
#pragma unroll
    for (int cb = 0; cb < kP2mH16MaxCB; cb++) {
      if (cb < ncb) {
        if constexpr (UP) __builtin_amdgcn_sched_barrier(0);
        v8h b[4], nb[2];
#pragma unroll
        for (int P = 0; P < 4; P++) b[P] = tl[(long)(kc * 4 + P) * 4 * ncolp + 16 * cb];
        nb[0] = h16_neg(b[2]);
        nb[1] = h16_neg(b[3]);
        h16_cmac(a, b, nb, cr[cb], ci[cb]);
      }
    }
  }
  const int n = -(sel2(es, rw) + ec);
  zf* out = agm + (long)sel2(rhs, rw) * as + (b0 + 16 * j + 4 * lk) * S;
#pragma unroll
  for (int cb = 0; cb < kP2mH16MaxCB; cb++) {
    const int sm = 16 * cb + li;
    if (mine && cb < ncb && sm < S) {
#pragma unroll
      for (int i = 0; i < 4; i++) out[(long)i * S + sm] = mkc<float>(ldexpf(cr[cb][i], n), ldexpf(ci[cb][i], n));
    }
  }
  if constexpr (UP) {
    // ---- M2M: row block w of the workgroup is this wave's 16 boxes
    __shared__ int exs[64];
    _Float16* hl = reinterpret_cast<_Float16*>(hal);  // [row block 4][hi, lo][box 16][kUpPitch]
    float sc[4];
    int ex[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      float m = 0.f;
#pragma unroll
      for (int cb = 0; cb < kUpCB; cb++) m = fmaxf(m, fmaxf(fabsf(cr[cb][i]), fabsf(ci[cb][i])));
      ex[i] = h16_scale_exp(row_max(m));
      sc[i] = ldexpf(1.f, ex[i]);
    }
    auto put = [&](const v4f (&c)[kP2mH16MaxCB]) {
#pragma unroll
      for (int cb = 0; cb < kUpCB; cb++) {
        const int k = 16 * cb + li;
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const float x = c[cb][i] * sc[i];
          const _Float16 hi = (_Float16)x, lo = (_Float16)(x - (float)hi);
          _Float16* d = hl + (w * 32 + 4 * lk + i) * kUpPitch + k;
          if (k < S) {
            d[0] = hi;
            d[16 * kUpPitch] = lo;
            if (k + S < kUpPitch) {
              d[S] = hi;
              d[S + 16 * kUpPitch] = lo;
            }
          }
        }
      }
    };
    const int nck = (up.Sp + 15) / 16;
    // products of sample block ck with the staged parts of all row blocks
    auto band = [&](int ck, v4f (&acc)[4]) {
      const v8h* tb = up.tab + ck * 256 + lane;
      v8h b[2][2];
#pragma unroll
      for (int kc = 0; kc < 2; kc++)
#pragma unroll
        for (int P = 0; P < 2; P++) b[kc][P] = tb[(kc * 2 + P) * 64];
      const int s0 = up.s0[ck];
#pragma unroll
      for (int rb = 0; rb < 4; rb++) {
        acc[rb] = v4f{0, 0, 0, 0};
        const _Float16* d = hl + (rb * 32 + li) * kUpPitch + s0;
#pragma unroll
        for (int kc = 0; kc < 2; kc++) {
          // (past the window the table is zero; any staged value will do)
          const int k = kc == 0 ? 8 * lk : 32 + 8 * (lk & 1);
          const v8h hi = *reinterpret_cast<const v8h*>(d + k), lo = *reinterpret_cast<const v8h*>(d + 16 * kUpPitch + k);
          acc[rb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(hi, b[kc][0], acc[rb], 0, 0, 0);
          acc[rb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(hi, b[kc][1], acc[rb], 0, 0, 0);
          acc[rb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(lo, b[kc][0], acc[rb], 0, 0, 0);
        }
      }
    };
    __syncthreads();  // the input is no longer read
    __builtin_amdgcn_sched_barrier(0);
    if (li == 0)
#pragma unroll
      for (int i = 0; i < 4; i++) exs[16 * w + 4 * lk + i] = ex[i];
    put(cr);
    __syncthreads();
    v4f re[kUpRounds][4];
#pragma unroll
    for (int u = 0; u < kUpRounds; u++) {
      if (w + 4 * u < nck) band(w + 4 * u, re[u]);
      __builtin_amdgcn_sched_barrier(0);  // (rounds interleaved would not fit the registers)
    }
    __syncthreads();
    put(ci);
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kUpRounds; u++) {
      const int ck = w + 4 * u, col = 16 * ck + li;
      if (ck < nck) {
        v4f im[4];
        band(ck, im);
        __builtin_amdgcn_sched_barrier(0);
        zf sh[4];
#pragma unroll
        for (int i = 0; i < 4; i++) sh[i] = up.shift[i * up.Sp + min(col, up.Sp - 1)];
#pragma unroll
        for (int rb = 0; rb < 4; rb++) {
          const int n0 = -(es[rb >> 1] + ec + up.ec);
          zf o = mkc<float>(0.f, 0.f);
#pragma unroll
          for (int i = 0; i < 4; i++) {
            const int e = n0 - exs[16 * rb + 4 * lk + i];
            o = cfma(sh[i], mkc<float>(ldexpf(re[u][rb][i], e), ldexpf(im[rb][i], e)), o);
          }
          if (on[rb >> 1] && col < up.Sp)
            up.par[(long)rhs[rb >> 1] * up.ps + ((b0 >> 2) + 4 * (rb & 1) + lk) * up.Sp + col] = o;
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
  }
}

}  // namespace isg
