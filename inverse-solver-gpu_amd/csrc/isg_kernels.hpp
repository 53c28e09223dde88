// isg_kernels.hpp -- HIP kernels of the MLFMA operator and the BiCGSTAB
// vector algebra, written for gfx950 (64-lane wavefronts, 256-thread blocks).
//
// Operator stages (reference counterparts in parentheses):
//   k_p2m_mfma, k_p2m_sym (isg_p2m_sym.hpp), k_p2m_h16 (isg_near_h16.hpp)
//                leaf radiation patterns on the matrix cores (kernels.cu:6-30)
//   k_interp_band, k_m2m_chunk, k_m2m   child -> parent interpolate+shift (kernels.cu:83-136)
//   k_m2l_par, k_m2l_tile, k_m2l_reg    diagonal translation (kernels.cu:239-266)
//   k_interp_band, k_l2l_chunk, k_l2l   parent -> child shift+anterpolate (kernels.cu:137-238)
//   k_down_h16, k_down64 (isg_down.hpp) translation and anterpolation of a level in one
//   k_near_mfma (isg_near_sym.hpp)  near field + leaf receiving patterns on the
//                matrix cores                     (kernels.cu:32-81, :292-319)
//   k_rx_*    receiver interpolation / anterpolation (matvec_gpu.cu:351-361, :395-401)
// Grids are (work items / 256, right-hand sides); blockIdx.y selects the
// right-hand side and an optional `act` mask skips converged ones.
#pragma once

#include "isg_device.hpp"

namespace isg {

constexpr int kBlock = 256;

__device__ __forceinline__ bool rhs_off(const int* act, int rhs) { return act != nullptr && act[rhs] == 0; }

// XCD-aware workgroup order.  Workgroups are dealt to the 8 XCDs (each with
// its own L2) round-robin by linear id, so consecutive blockIdx.x run on
// different L2s.  When gridDim.x is a multiple of 8 (then x mod 8 is the
// XCD for every blockIdx.y), this bijection gives each XCD a contiguous
// range of logical ids: neighbouring tiles and the sample chunks of one tile,
// which read the same cache lines, then share one L2.
__device__ __forceinline__ int xcd_block() {
  const int x = blockIdx.x, n = gridDim.x;
  return (n & 7) ? x : (x & 7) * (n >> 3) + (x >> 3);
}

// Strided staging of n elements (element e = tid, tid + kBlock, ...): the
// loads of U consecutive strides, ld(e), are issued before any of them is
// stored with st(e, v), so each thread has U memory requests in flight
// instead of waiting for every load in turn before the next one issues.
// ld should only load (arithmetic on the loaded values belongs in st, or the
// compiler waits for each load before issuing the next).
template <typename T>
struct CPair {
  cplx<T> a, b;
};

template <int U, typename V, typename Ld, typename St>
__device__ __forceinline__ void stage(int n, Ld ld, St st) {
  for (int e0 = threadIdx.x; e0 < n; e0 += U * kBlock) {
    V v[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int e = e0 + u * kBlock;
      if (e < n) v[u] = ld(e);
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int e = e0 + u * kBlock;
      if (e < n) st(e, v[u]);
    }
  }
}

// Direct-from-cache interpolation kernels, one thread per target sample; used
// for root levels whose LDS staging would exceed 64 KB.
// parent[p][k] = sum_c shift[c][k] * sum_t w[t][k] child[4p+c][(i0[k]+t) mod Sc]
template <typename T>
__global__ void __launch_bounds__(kBlock) k_m2m(const cplx<T>* __restrict__ child, long cs, cplx<T>* __restrict__ par,
                                                long ps, const T* __restrict__ wT, const int* __restrict__ i0,
                                                const cplx<T>* __restrict__ shift, int Sp, int Sc, int np, int ntap,
                                                const int* __restrict__ act) {
  int rhs = blockIdx.y;
  if (rhs_off(act, rhs)) return;
  long idx = (long)blockIdx.x * kBlock + threadIdx.x;
  if (idx >= (long)np * Sp) return;
  int p = (int)(idx / Sp), k = (int)(idx - (long)p * Sp);
  int j0 = i0[k];
  cplx<T> acc = mkc<T>(0, 0);
  for (int c = 0; c < 4; c++) {
    const cplx<T>* ch = child + rhs * cs + (long)(4 * p + c) * Sc;
    cplx<T> red = mkc<T>(0, 0);
    int j = j0;
    for (int t = 0; t < ntap; t++) {
      T w = wT[t * Sp + k];
      cplx<T> v = ch[j];
      red.x += w * v.x;
      red.y += w * v.y;
      j = (j + 1 == Sc) ? 0 : j + 1;
    }
    acc = cfma(red, shift[c * Sp + k], acc);
  }
  par[rhs * ps + idx] = acc;
}

// child[c][k] (+)= sum_t a[t][k] * shiftL[c%4][j] * par[c/4][j], j = (j0[k]+t) mod Sp
template <typename T>
__global__ void __launch_bounds__(kBlock) k_l2l(const cplx<T>* __restrict__ par, long ps, cplx<T>* __restrict__ child,
                                                long cs, const T* __restrict__ aT, const int* __restrict__ j0s,
                                                const cplx<T>* __restrict__ shift, int Sp, int Sc, int np, int ntap,
                                                int accumulate, const int* __restrict__ act) {
  int rhs = blockIdx.y;
  if (rhs_off(act, rhs)) return;
  long idx = (long)blockIdx.x * kBlock + threadIdx.x;
  if (idx >= (long)4 * np * Sc) return;
  int c = (int)(idx / Sc), k = (int)(idx - (long)c * Sc);
  int p = c >> 2, cm = c & 3;
  const cplx<T>* pv = par + rhs * ps + (long)p * Sp;
  const cplx<T>* sh = shift + cm * Sp;
  cplx<T> acc = mkc<T>(0, 0);
  int j = j0s[k];
  for (int t = 0; t < ntap; t++) {
    T w = aT[t * Sc + k];
    cplx<T> v = cmul(sh[j], pv[j]);
    acc.x += w * v.x;
    acc.y += w * v.y;
    j = (j + 1 == Sp) ? 0 : j + 1;
  }
  cplx<T>* dst = child + rhs * cs + idx;
  *dst = accumulate ? cadd(*dst, acc) : acc;
}

// ---------------------------------------------------------------------------
// Matrix-core products.  Operand
// layout of the 16x16x4 instructions (checked on gfx950): A[i][k] in lane
// i + 16k, B[k][j] in lane j + 16k; the 16x16 result D[i][j] is in lane
// j + 16(i/4), register i%4 for f32 and in lane j + 16(i%4), register i/4
// for f64 -- Mfma<T>::row gives the row of (lane group g, register q).
// Every kernel puts the data vectors (boxes, clusters) in the A operand and
// the operator table in the B operand, so the 16 lanes of a group hold 16
// consecutive samples / pixels of the result and stores coalesce.
template <typename T>
struct Mfma;
template <>
struct Mfma<double> {
  typedef double v4 __attribute__((ext_vector_type(4)));
  static constexpr bool kRowsAcrossLanes = true;  // rows g + 4q: siblings across lane groups
  static __device__ __forceinline__ v4 mac(double a, double b, v4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int g, int q) { return g + 4 * q; }
  // cr + i ci += d * a   (d data, A operand; a table, B operand; nai = -a.y)
  // three-product form (Gauss): p1 += dr ar, p2 += di ai, p3 += (dr + di)(ar + ai)
  // with asum = ar + ai; then d a = (p1 - p2) + i (p3 - p1 - p2)
  static __device__ __forceinline__ void cmac3(cplx<double> d, cplx<double> a, double asum, v4& p1, v4& p2, v4& p3) {
    p1 = mac(d.x, a.x, p1);
    p2 = mac(d.y, a.y, p2);
    p3 = mac(d.x + d.y, asum, p3);
  }
};
template <>
struct Mfma<float> {
  typedef float v4 __attribute__((ext_vector_type(4)));
  static constexpr bool kRowsAcrossLanes = false;  // rows 4g + q: siblings in one lane
  static __device__ __forceinline__ v4 mac(float a, float b, v4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int g, int q) { return 4 * g + q; }
  static __device__ __forceinline__ void cmac3(cplx<float> d, cplx<float> a, float asum, v4& p1, v4& p2, v4& p3) {
    p1 = mac(d.x, a.x, p1);
    p2 = mac(d.y, a.y, p2);
    p3 = mac(d.x + d.y, asum, p3);
  }
};

// ---- BiCGSTAB helpers shared by the vector kernels and the near-field epilogue
constexpr int kSlots = 3;

// The contrast weight g[i] enters prep only in the forward product and post
// only in the adjoint one; it is loaded only there (herm is uniform per launch).
__device__ __forceinline__ zd prep_val(zd x, const zd* g, long i, bool herm) { return herm ? cconj(x) : cmul(x, g[i]); }
__device__ __forceinline__ zd post_val(zd x, zd gy, const zd* g, long i, bool herm) {
  return herm ? csub(x, cconj(cmul(g[i], gy))) : csub(x, gy);
}

// Block-level sum of up to 3 complex partials; thread 0 writes part[slot].
template <int NS>
__device__ __forceinline__ void block_store(zd (&v)[NS], double2* part, int nblk, int blk) {
  __shared__ double sh[NS * 2][kBlock / 64];
  int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int s = 0; s < NS; s++) {
    double a = wave_sum(v[s].x), b = wave_sum(v[s].y);
    if (lane == 0) {
      sh[2 * s][w] = a;
      sh[2 * s + 1][w] = b;
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int s = 0; s < NS; s++) {
      double a = 0, b = 0;
      for (int i = 0; i < kBlock / 64; i++) {
        a += sh[2 * s][i];
        b += sh[2 * s + 1][i];
      }
      part[s * nblk + blk] = make_double2(a, b);
    }
  }
}

#define ISG_VEC_LOOP(N) for (long i = (long)blockIdx.x * kBlock + threadIdx.x; i < (N); i += (long)gridDim.x * kBlock)

// Vector kernels are templated on the storage type V of the work vectors
// (double, or float for the mixed-precision solver); arithmetic and the dot
// product partials are FP64 either way, the solution x and the right-hand
// side b are always FP64.
template <typename V>
__device__ __forceinline__ zd ldv(const cplx<V>* a, long i) { return ccast<double>(a[i]); }
template <typename V>
__device__ __forceinline__ zd stv(cplx<V>* a, long i, zd v) {
  cplx<V> w = ccast<V>(v);
  a[i] = w;
  return ccast<double>(w);  // the value as stored
}

// Sum over blocks of one system's partials, slots 0 .. NS - 1, in a fixed order;
// every thread gets it.  sh: LDS, reusable after the caller's next barrier.
template <int NS>
__device__ __forceinline__ void part_sum(const double2* __restrict__ pr, int nblk, zd (&tot)[NS],
                                         double (*sh)[kBlock / 64]) {
  double v[2 * NS];
#pragma unroll
  for (int s = 0; s < NS; s++) {
    v[2 * s] = v[2 * s + 1] = 0;
    for (int j = threadIdx.x; j < nblk; j += kBlock) {
      const double2 q = pr[s * nblk + j];
      v[2 * s] += q.x;
      v[2 * s + 1] += q.y;
    }
  }
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  __syncthreads();  // an earlier call's sums have been read
#pragma unroll
  for (int s = 0; s < 2 * NS; s++) {
    const double a = wave_sum(v[s]);
    if (lane == 0) sh[s][w] = a;
  }
  __syncthreads();
#pragma unroll
  for (int s = 0; s < NS; s++) {
    tot[s] = mkc<double>(0, 0);
    for (int i = 0; i < kBlock / 64; i++) {
      tot[s].x += sh[2 * s][i];
      tot[s].y += sh[2 * s + 1][i];
    }
  }
}

// The vector step of P2mStep, element by element (o: the system's offset,
// element i of it; load only loads, so that a group's loads are in flight
// together).  Every element belongs to one workgroup.  alpha is summed by each
// workgroup from the near field's partials (a kernel of one workgroup per system
// between the two products costs 5 us of latency; where the workgroups are too
// many for that, k_bi_reduce has left one partial per system); the first stores it.
template <typename V>
struct StepIn {
  cplx<V> r, p, v;
  zd g;
};
struct StepCoef {
  zd a, b;
  bool first;
};
template <int STEP, typename V>
__device__ __forceinline__ StepCoef step_coef(const P2mStep<V>& q, int rhs, void* lds) {
  StepCoef c;
  c.first = false;
  if constexpr (STEP == 2) {
    const BiState& S = q.st[rhs];
    c.a = S.beta;
    c.b = mkc<double>(-S.omega.x, -S.omega.y);
    c.first = S.first != 0;
  } else if constexpr (STEP == 3) {
    zd t[1];
    part_sum<1>(q.part + rhs * q.pstride, q.nblk, t, static_cast<double(*)[kBlock / 64]>(lds));
    const zd al = zdiv(q.st[rhs].rho, t[0]);
    if (blockIdx.x == 0 && threadIdx.x == 0) q.st[rhs].alpha = al;
    c.a = mkc<double>(-al.x, -al.y);
  }
  return c;
}
template <int STEP, typename V>
__device__ __forceinline__ StepIn<V> step_load(const P2mStep<V>& q, const StepCoef& c, long o, long go, long i) {
  StepIn<V> in;
  in.r = q.r[o + i];
  if constexpr (STEP == 2) {
    if (!c.first) {
      in.p = q.p[o + i];
      in.v = q.v[o + i];
    }
  }
  if constexpr (STEP == 3) in.v = q.v[o + i];
  if (!q.herm) in.g = q.g[go + i];
  return in;
}
template <int STEP, typename V>
__device__ __forceinline__ cplx<V> step_value(const P2mStep<V>& q, const StepCoef& c, const StepIn<V>& in, cplx<V>& pv) {
  zd x = ccast<double>(in.r);
  if constexpr (STEP == 2)
    if (!c.first) x = cfma(c.a, cfma(c.b, ccast<double>(in.v), ccast<double>(in.p)), x);
  if constexpr (STEP == 3) x = cfma(c.a, ccast<double>(in.v), x);
  pv = ccast<V>(x);
  x = ccast<double>(pv);  // the value as stored
  return ccast<V>(q.herm ? cconj(x) : cmul(x, in.g));
}

// Output of a near-field kernel whose NB x 64 products are in LDS: stored, or
// the BiCGSTAB post step / residual check of NearPost.
template <typename T, typename TI, int NB, int POST>
__device__ __forceinline__ void near_epilogue(const cplx<T>* tile, cplx<TI>* __restrict__ r, long rs, long b0, int rhs,
                                              const NearPost<TI>& post) {
  const int tid = threadIdx.x;
  if constexpr (POST == 0) {
    cplx<TI>* out = r + rhs * rs + b0 * 64;
#pragma unroll 4
    for (int e = tid; e < NB * 64; e += kBlock) out[e] = ccast<TI>(tile[e]);
  } else {
  // BiCGSTAB post step (modes 1, 2) or residual check (mode 3, FP64) on the
  // operator output, rounded to the vector type TI first, as a separate pass
  // reading the stored product back would see it.
  const long o = rhs * rs + b0 * 64;
  const zd* gr = post.g + rhs * post.gs + b0 * 64;
  zd acc[2] = {mkc<double>(0, 0), mkc<double>(0, 0)};
  struct In {
    cplx<TI> x, aux;  // aux: r~ (mode 1) or b (mode 3)
    zd g;
  };
  const bool herm = post.herm != 0;
  stage<2, In>(
      NB * 64,
      [&](int e) {
        In v;
        v.x = post.x[o + e];
        if (POST == 1) v.aux = post.rt[o + e];
        if (POST == 3) v.aux = post.b[o + e];
        if (herm) v.g = gr[e];  // the forward post step does not use g
        return v;
      },
      [&](int e, In v) {
        const cplx<T> gt = tile[e];
        const zd gy = mkc<double>((double)(TI)gt.x, (double)(TI)gt.y);
        const zd xv = ccast<double>(v.x);
        const zd px = herm ? csub(xv, cconj(cmul(v.g, gy))) : csub(xv, gy);
        if constexpr (POST == 3) {
          r[o + e] = ccast<TI>(gt);  // the product itself, as the plain kernel stores it
          const zd bv = ccast<double>(v.aux), rv = csub(bv, px);
          acc[0].x += bv.x * bv.x + bv.y * bv.y;
          acc[1].x += rv.x * rv.x + rv.y * rv.y;
        } else {
          const zd res = stv(r, o + e, px);
          if (POST == 1) {
            const zd a = ccast<double>(v.aux);
            acc[0].x += a.x * res.x + a.y * res.y;
            acc[0].y += a.x * res.y - a.y * res.x;
          } else {
            acc[0].x += res.x * xv.x + res.y * xv.y;
            acc[0].y += res.x * xv.y - res.y * xv.x;
            acc[1].x += res.x * res.x + res.y * res.y;
          }
        }
      });
    block_store<2>(acc, post.part + (long)rhs * kSlots * gridDim.x, gridDim.x, blockIdx.x);
  }
}

// ---------------------------------------------------------------------------
// Sample-chunked LDS interpolation (upper levels: few clusters, many samples).
// A workgroup owns one parent (or G small parents) and a chunk of <= 256
// target samples.  Taps of consecutive targets advance monotonically (mod the
// source count), so the chunk needs one contiguous window of each source
// vector: window start = first[k0], offset of target k = (first[k] -
// first[k0]) mod Ssrc.  All four windows (children, or shifted parent copies)
// go to LDS once; each thread then forms one target from LDS.

// The upper levels have little work (16 parents of 1036 samples at 1024^2) and
// these kernels were bound by the latency of their serial tap loop, each tap
// waiting for its weight from L2: the weights, shifts and first-tap indices of a
// thread are now loaded into registers before the staging (NT taps, compiled in for
// the default 30 and 60; 0: any count, loaded along the way), and the staging steps its indices instead of
// dividing.  Per launch at 512^2 x 15 right-hand sides (FP32): M2M 14.5 -> 8.5 us,
// L2L 19.6 -> 17.4 us.

// Window staging: the calling wave loads elements j0, j0 + 1, .. of n (mod K),
// lane by lane, all loads (up to 4 x 64) issued before the first store.
template <typename Ld, typename St>
__device__ __forceinline__ void stage_window(int n, int j0, int K, Ld ld, St st) {
  const int lane = threadIdx.x & 63;
  for (int t0 = lane; t0 < n; t0 += 256) {
    decltype(ld(0)) v[4];
#pragma unroll
    for (int u = 0; u < 4; u++) {
      int j = j0 + min(t0 + 64 * u, n - 1);
      while (j >= K) j -= K;
      v[u] = ld(j);
    }
#pragma unroll
    for (int u = 0; u < 4; u++)
      if (t0 + 64 * u < n) st(t0 + 64 * u, v[u]);
  }
}

// M2M: parent[p][k] = sum_c shiftM[c][k] sum_t w[t][k] child[4p+c][first[k]+t]
template <typename T, int NT>
__global__ void __launch_bounds__(kBlock) k_m2m_chunk(const cplx<T>* __restrict__ child, long cs,
                                                      cplx<T>* __restrict__ par, long ps, const T* __restrict__ wT,
                                                      const int* __restrict__ i0, const cplx<T>* __restrict__ shift,
                                                      int Sp, int Sc, int G, int kch, int nch, int ntap,
                                                      const int* __restrict__ act) {
  extern __shared__ char smem_raw[];
  cplx<T>* lds = reinterpret_cast<cplx<T>*>(smem_raw);
  const int rhs = blockIdx.y;
  if (rhs_off(act, rhs)) return;
  const int pg = blockIdx.x / nch, ch = blockIdx.x - pg * nch;
  const long p0 = (long)pg * G;
  const int k0 = ch * kch, kn = min(kch, Sp - k0);
  const int base = i0[k0];
  int W = i0[k0 + kn - 1] - base;
  if (W < 0) W += Sc;
  W += ntap;
  const int o = min((int)threadIdx.x, G * kn - 1);
  const int g = o / kn, k = k0 + (o - g * kn);
  const int ik = i0[k];
  T w[NT ? NT : 1];
  cplx<T> sh[4];
  if constexpr (NT > 0) {
#pragma unroll
    for (int t = 0; t < NT; t++) w[t] = wT[t * Sp + k];
  }
#pragma unroll
  for (int c = 0; c < 4; c++) sh[c] = shift[c * Sp + k];
  const cplx<T>* cr = child + rhs * cs + 4 * p0 * Sc;
  for (int v = threadIdx.x >> 6; v < 4 * G; v += kBlock / 64)  // v = 4 g + c (consecutive children)
    stage_window(
        W, base, Sc, [&](int j) { return cr[(long)v * Sc + j]; }, [&](int t, cplx<T> x) { lds[v * W + t] = x; });
  __syncthreads();
  if ((int)threadIdx.x >= G * kn) return;
  int d = ik - base;
  if (d < 0) d += Sc;
  cplx<T> acc = mkc<T>(0, 0);
  if constexpr (NT > 0) {
#pragma unroll
    for (int c = 0; c < 4; c++) {
      const cplx<T>* src = lds + (4 * g + c) * W + d;
      cplx<T> red = mkc<T>(0, 0);
#pragma unroll
      for (int t = 0; t < NT; t++) {
        red.x += w[t] * src[t].x;
        red.y += w[t] * src[t].y;
      }
      acc = cfma(red, sh[c], acc);
    }
  } else {
    // a weight is loaded once for the four children, several in flight (M2M above the
    // leaf at 512 px x 2, 28 taps: child by child FP64 59 us and FP32 43, with two taps
    // in flight 45 and 41, with four 34 and 47)
    constexpr int U = sizeof(T) == 8 ? 4 : 2;
    const cplx<T>* src = lds + 4 * g * W + d;
    cplx<T> red[4];
#pragma unroll
    for (int c = 0; c < 4; c++) red[c] = mkc<T>(0, 0);
#pragma unroll U
    for (int t = 0; t < ntap; t++) {
      const T wt = wT[t * Sp + k];
#pragma unroll
      for (int c = 0; c < 4; c++) {
        red[c].x += wt * src[c * W + t].x;
        red[c].y += wt * src[c * W + t].y;
      }
    }
#pragma unroll
    for (int c = 0; c < 4; c++) acc = cfma(red[c], sh[c], acc);
  }
  par[rhs * ps + (p0 + g) * Sp + k] = acc;
}

// L2L: child[4p+c][k] (+)= sum_t a[t][k] (shiftL[c] o par[p])[first[k]+t];
// wave c forms child c's window and its kch <= 64 samples
template <typename T, int NT>
__global__ void __launch_bounds__(kBlock) k_l2l_chunk(const cplx<T>* __restrict__ par, long ps,
                                                      cplx<T>* __restrict__ child, long cs, const T* __restrict__ aT,
                                                      const int* __restrict__ j0s, const cplx<T>* __restrict__ shift,
                                                      int Sp, int Sc, int kch, int nch, int ntap, int accumulate,
                                                      const int* __restrict__ act) {
  extern __shared__ char smem_raw[];
  cplx<T>* lds = reinterpret_cast<cplx<T>*>(smem_raw);
  const int rhs = blockIdx.y;
  if (rhs_off(act, rhs)) return;
  const int p = blockIdx.x / nch, ch = blockIdx.x - p * nch;
  const int k0 = ch * kch, kn = min(kch, Sc - k0);
  const int base = j0s[k0];
  int W = j0s[k0 + kn - 1] - base;
  if (W < 0) W += Sp;
  W += ntap;
  const int lane = threadIdx.x & 63, c = threadIdx.x >> 6;
  const int k = k0 + min(lane, kn - 1);
  const int jk = j0s[k];
  T w[NT ? NT : 1];
  if constexpr (NT > 0) {
#pragma unroll
    for (int t = 0; t < NT; t++) w[t] = aT[t * Sc + k];
  }
  cplx<T>* dst = child + rhs * cs + (4L * p + c) * Sc + k;
  cplx<T> old = mkc<T>(0, 0);
  if (accumulate) old = *dst;
  const cplx<T>* pv = par + rhs * ps + (long)p * Sp;
  cplx<T>* win = lds + c * W;
  stage_window(
      W, base, Sp, [&](int j) { return CPair<T>{shift[c * Sp + j], pv[j]}; },
      [&](int t, CPair<T> x) { win[t] = cmul(x.a, x.b); });
  __syncthreads();
  if (lane >= kn) return;
  int d = jk - base;
  if (d < 0) d += Sp;
  const cplx<T>* src = win + d;
  cplx<T> red = mkc<T>(0, 0);
  if constexpr (NT > 0) {
#pragma unroll
    for (int t = 0; t < NT; t++) {
      red.x += w[t] * src[t].x;
      red.y += w[t] * src[t].y;
    }
  } else {
    for (int t = 0; t < ntap; t++) {
      const T wt = aT[t * Sc + k];
      red.x += wt * src[t].x;
      red.y += wt * src[t].y;
    }
  }
  *dst = accumulate ? cadd(old, red) : red;
}

// Interpolation (M2M) and anterpolation (L2L) on the matrix cores, for the
// levels with many clusters.  Out[k][col] = sum_j A[k][j] In[j][col], A the
// real interpolator (30 taps per row, M2M) or anterpolator (60 taps, L2L),
// columns = the child vectors (4 per parent) of NC/4 consecutive parents.
// A is banded: the taps of 16 consecutive rows k all fall in one window of
// KB <= K inputs starting at s0[rb] (modulo K), so each 16-row block is a
// 16 x KB dense block ("band block"), stored K-major as AB[rb][kk][16].
//   M2M (MODE 0): In = children (contiguous); the epilogue multiplies by
//                 shiftM[c][k] and sums the 4 sibling columns, then writes
//                 parent[p][k].
//   L2L (MODE 1): In = shiftL[c] o parent, staged per column; Out is added to
//                 (or assigned to) child[4p+c][k].
// The KB/4 table fragments of a block are loaded into registers before its
// MFMA chain; the data columns come from LDS (one padding element per column).
template <typename T, int MODE, int NCB, int KQ>
__global__ void __launch_bounds__(kBlock) k_interp_band(const cplx<T>* __restrict__ src, long ss,
                                                        cplx<T>* __restrict__ dst, long ds, const T* __restrict__ AB,
                                                        const int* __restrict__ s0v, int KB,
                                                        const cplx<T>* __restrict__ shift, int Mrows, int K,
                                                        int accumulate, const int* __restrict__ act) {
  typedef typename Mfma<T>::v4 v4;
  constexpr int NC = 16 * NCB;
  extern __shared__ char smem_raw[];
  cplx<T>* tile = reinterpret_cast<cplx<T>*>(smem_raw);
  const int rhs = blockIdx.y;
  if (rhs_off(act, rhs)) return;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int li = lane & 15, lk = lane >> 4;
  const int row = K + 1;
  const long p0 = (long)xcd_block() * (NC / 4);
  // M2M: element e = col * K + j of the NC x K block of children goes to
  // tile[col * (K + 1) + j] = tile[e + col].  L2L: element e = p * K + j of the
  // NC/4 parents is loaded once and gives the 4 children's columns
  // tile[(4 p + c) * (K + 1) + j] = shiftL[c][j] parent[p][j].  Each thread
  // starts at e = tid and advances by kBlock; (col, j) are stepped rather than
  // divided out of e, and the loads of U strides are issued before the first
  // store.
  if constexpr (MODE == 0) {
    constexpr int U = sizeof(T) == 4 ? 8 : 4;
    const int n = NC * K, dcol = kBlock / K, dj = kBlock - dcol * K;
    int col = tid / K, j = tid - col * K;
    const cplx<T>* s = src + rhs * ss + 4 * p0 * K;
    for (int e0 = tid; e0 < n; e0 += U * kBlock) {
      cplx<T> a[U];
      int cu[U];
#pragma unroll
      for (int u = 0; u < U; u++) {
        const int e = e0 + u * kBlock;
        cu[u] = col;
        a[u] = s[e < n ? e : n - 1];  // NC consecutive children of length K (clamped load)
        j += dj;
        col += dcol;
        if (j >= K) {
          j -= K;
          col++;
        }
      }
#pragma unroll
      for (int u = 0; u < U; u++) {
        const int e = e0 + u * kBlock;
        if (e < n) tile[e + cu[u]] = a[u];
      }
    }
  } else {
    constexpr int U = 4;
    const int n = (NC / 4) * K, dp = kBlock / K, dj = kBlock - dp * K;
    int pp = tid / K, j = tid - pp * K;
    const cplx<T>* s = src + rhs * ss + p0 * K;
    for (int e0 = tid; e0 < n; e0 += U * kBlock) {
      cplx<T> a[U];
      int pu[U], ju[U];
#pragma unroll
      for (int u = 0; u < U; u++) {
        const int e = e0 + u * kBlock;
        pu[u] = pp;
        ju[u] = j;
        a[u] = s[e < n ? e : n - 1];  // NC/4 consecutive parents of length K (clamped load)
        j += dj;
        pp += dp;
        if (j >= K) {
          j -= K;
          pp++;
        }
      }
#pragma unroll
      for (int u = 0; u < U; u++) {
        const int e = e0 + u * kBlock;
        if (e < n) {
          cplx<T>* t = tile + 4 * pu[u] * row + ju[u];
#pragma unroll
          for (int c = 0; c < 4; c++) t[c * row] = cmul(shift[c * K + ju[u]], a[u]);
        }
      }
    }
  }
  __syncthreads();
  const int nrb = (Mrows + 15) / 16;
  const int nkq = KB >> 2;
  // (row block, column block) items spread evenly over the 4 waves; the M2M
  // with two column blocks takes both of a row block in one item, so that its
  // band rows and sibling shifts (which do not depend on the column) are
  // loaded once for both
  constexpr bool RB_ITEMS = MODE == 0 && NCB == 2;
  constexpr int CPI = RB_ITEMS ? NCB : 1;  // column blocks per item
  for (int item = w; item < nrb * NCB / CPI; item += 4) {
    const int rb = RB_ITEMS ? item : item / NCB, cb0 = RB_ITEMS ? 0 : item - rb * NCB;
    const T* ab = AB + (long)rb * KB * 16;
    T a[KQ];
#pragma unroll
    for (int q = 0; q < KQ; q++) a[q] = (q < nkq) ? ab[(4 * q + lk) * 16 + li] : (T)0;
    const int s0 = s0v[rb];
    // the epilogue's operands (M2M: sibling shifts; L2L: the child locals it
    // adds to) are loaded here, so their latency overlaps the MFMA chain
    const int k = 16 * rb + li;
    cplx<T> pre[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
      pre[q] = mkc<T>(0, 0);
      if (k < Mrows) {
        if (MODE == 0) {
          pre[q] = shift[q * Mrows + k];
        } else if (accumulate) {
          pre[q] = dst[rhs * ds + (4 * p0 + 16 * cb0 + Mfma<T>::row(lk, q)) * (long)Mrows + k];
        }
      }
    }
#pragma unroll
    for (int cc = 0; cc < CPI; cc++) {
      const int cb = cb0 + cc;
      // M2M: columns in the order that leaves the 4 siblings of parent 4 cb + lk to a lane
      const int ci = MODE == 0 && Mfma<T>::kRowsAcrossLanes ? 4 * (li & 3) + (li >> 2) : li;
      const cplx<T>* tcol = tile + (16 * cb + ci) * row;
      v4 cr0 = v4{0, 0, 0, 0}, ci0 = v4{0, 0, 0, 0};
#pragma unroll
      for (int q = 0; q < KQ; q++) {
        if (q < nkq) {
          int j = s0 + 4 * q + lk;
          if (j >= K) j -= K;
          const cplx<T> bv = tcol[j];
          cr0 = Mfma<T>::mac(bv.x, a[q], cr0);
          ci0 = Mfma<T>::mac(bv.y, a[q], ci0);
        }
      }
      // D[col][k]: lane li holds target sample k = 16 rb + li; col = 16 cb + row(lk, q)
      if (MODE == 0) {
        // parent = sum over the 4 sibling columns of shiftM[c][k] * D[col][k]
        T xr = 0, xi = 0;
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const cplx<T> sq = pre[q];
          const T vr = cr0[q], vi = ci0[q];
          xr += vr * sq.x - vi * sq.y;
          xi += vr * sq.y + vi * sq.x;
        }
        if (k < Mrows) dst[rhs * ds + (p0 + 4 * cb + lk) * Mrows + k] = mkc<T>(xr, xi);
      } else if (k < Mrows) {
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const int col = 16 * cb + Mfma<T>::row(lk, q);
          cplx<T>* o = dst + rhs * ds + (4 * p0 + col) * (long)Mrows + k;
          cplx<T> v = mkc<T>(cr0[q], ci0[q]);
          *o = accumulate ? cadd(pre[q], v) : v;
        }
      }
    }
  }
}

// M2L staging for a TS x TS tile of target boxes at corner (X0, Y0) and
// samples k0 .. k0+KC-1: the multipoles of the (TS+4)^2 boxes around it
// (zero outside the level or past S) and the 49 translation operators.
template <typename T, int TS, int KC>
__device__ __forceinline__ void m2l_stage(cplx<T> (*src)[KC], cplx<T> (*tr)[KC], const cplx<T>* a,
                                          const cplx<T>* trans, int X0, int Y0, int k0, int nb, int S) {
  constexpr int SB = TS + 4, NS = SB * SB * KC;
  constexpr int US = NS / kBlock < 9 ? (NS + kBlock - 1) / kBlock : 9;
  // offset of each halo box's multipole (Morton index * S), -1 outside the
  // level: one Morton conversion per box instead of one per element
  __shared__ int boff[SB * SB];
  for (int b = threadIdx.x; b < SB * SB; b += kBlock) {
    const int sx = X0 - 2 + b % SB, sy = Y0 - 2 + b / SB;
    boff[b] = (sx >= 0 && sy >= 0 && sx < nb && sy < nb) ? (int)morton2(sx, sy) * S : -1;
  }
  __syncthreads();
  // kBlock is a multiple of KC: each thread keeps one sample kk
  const int kk = threadIdx.x % KC;
  const bool kin = k0 + kk < S;
  stage<US, cplx<T>>(
      NS,
      [&](int e) {
        const int off = boff[e / KC];
        cplx<T> v = mkc<T>(0, 0);
        if (off >= 0 && kin) v = a[(long)off + k0 + kk];
        return v;
      },
      [&](int e, cplx<T> v) { src[e / KC][kk] = v; });
  stage<(49 * KC + kBlock - 1) / kBlock, cplx<T>>(
      49 * KC, [&](int e) { return kin ? trans[(long)(e / KC) * S + k0 + kk] : mkc<T>(0, 0); },
      [&](int e, cplx<T> v) { tr[e / KC][kk] = v; });
}

// Tiled M2L.  A workgroup owns a TS x TS block of target boxes (Morton
// consecutive) and KC consecutive samples.  The interaction lists of the
// block lie in the (TS+4)^2 block of boxes around it; those multipoles and
// the 49 translation operators for the KC samples are staged in LDS once, so
// each multipole sample is read from memory (TS+4)^2/TS^2 times instead of
// once per interaction (<= 27).
template <typename T, int TS, int KC>
__global__ void __launch_bounds__(kBlock) k_m2l_tile(const cplx<T>* __restrict__ agm, cplx<T>* __restrict__ agl,
                                                     long st, const cplx<T>* __restrict__ trans, int lev, int S,
                                                     const int* __restrict__ act) {
  constexpr int SB = TS + 4;
  __shared__ cplx<T> src[SB * SB][KC];
  __shared__ cplx<T> tr[49][KC];
  const int rhs = blockIdx.y;
  if (rhs_off(act, rhs)) return;
  const int nb = 1 << lev;
  const int nchunk = (S + KC - 1) / KC;
  const int lb = xcd_block();
  const int tile = lb / nchunk, chunk = lb - tile * nchunk;
  const int k0 = chunk * KC;
  const unsigned m0 = (unsigned)tile * TS * TS;
  const int X0 = (int)compact2(m0), Y0 = (int)compact2(m0 >> 1);
  m2l_stage<T, TS, KC>(src, tr, agm + rhs * st, trans, X0, Y0, k0, nb, S);
  __syncthreads();
  for (int o = threadIdx.x; o < TS * TS * KC; o += kBlock) {
    int tl = o / KC, kk = o - tl * KC;
    if (k0 + kk >= S) continue;
    unsigned m = m0 + tl;
    int X = (int)compact2(m), Y = (int)compact2(m >> 1);
    int bx = (X >> 1) * 2 - 2, by = (Y >> 1) * 2 - 2;
    cplx<T> acc = mkc<T>(0, 0);
    for (int sy = by; sy < by + 6; sy++) {
      if (sy < 0 || sy >= nb) continue;
      int dy = sy - Y;
      for (int sx = bx; sx < bx + 6; sx++) {
        if (sx < 0 || sx >= nb) continue;
        int dx = sx - X;
        if (dx >= -1 && dx <= 1 && dy >= -1 && dy <= 1) continue;
        acc = cfma(tr[7 * (dy + 3) + dx + 3][kk], src[(sy - Y0 + 2) * SB + (sx - X0 + 2)][kk], acc);
      }
    }
    agl[rhs * st + (long)m * S + k0 + kk] = acc;
  }
}

// M2L with the translation operators in registers.  Staging as k_m2l_tile
// (8x8 target boxes, their 12x12 source halo, KC samples).  A target box's
// far list depends only on its position class (X & 1, Y & 1): the 27 boxes
// of the parent's 6x6 neighbourhood outside its own 3x3, at offsets fixed
// per class.  Each thread owns one sample kk and one class, loads that
// class's 27 operators once and sweeps 64 / (256 / KC) targets of the class
// with compile-time LDS offsets; source boxes outside the domain are staged
// as zeros, so no bounds tests remain.
template <typename T, int PX, int PY, int KC, int NT>
__device__ __forceinline__ void m2l_class(const cplx<T> (*src)[KC], const cplx<T> (*tr)[KC], int kk, int part,
                                          cplx<T>* __restrict__ out, unsigned m0, int S, int k0) {
  constexpr int SB = 12;
  cplx<T> t[27];
  {
    int j = 0;
#pragma unroll
    for (int dy = -2 - PY; dy <= 3 - PY; dy++)
#pragma unroll
      for (int dx = -2 - PX; dx <= 3 - PX; dx++)
        if (dx < -1 || dx > 1 || dy < -1 || dy > 1) t[j++] = tr[7 * (dy + 3) + dx + 3][kk];
  }
  // the class's 16 targets (2i + PX, 2j + PY), i, j = 0..3, numbered 4j + i;
  // this thread takes numbers part * NT .. part * NT + NT - 1
#pragma unroll 1
  for (int q = 0; q < NT; q++) {
    const int tt = part * NT + q;
    const int i = tt & 3, jj = tt >> 2;
    const int lx = 2 * i + PX, ly = 2 * jj + PY;
    const int base = (ly + 2) * SB + lx + 2;
    cplx<T> acc = mkc<T>(0, 0);
    int j = 0;
#pragma unroll
    for (int dy = -2 - PY; dy <= 3 - PY; dy++)
#pragma unroll
      for (int dx = -2 - PX; dx <= 3 - PX; dx++)
        if (dx < -1 || dx > 1 || dy < -1 || dy > 1) acc = cfma(t[j++], src[base + dy * SB + dx][kk], acc);
    if (k0 + kk < S) out[(long)(m0 + morton2((unsigned)lx, (unsigned)ly)) * S + k0 + kk] = acc;
  }
}

template <typename T, int KC>
__global__ void __launch_bounds__(kBlock) k_m2l_reg(const cplx<T>* __restrict__ agm, cplx<T>* __restrict__ agl,
                                                    long st, const cplx<T>* __restrict__ trans, int lev, int S,
                                                    const int* __restrict__ act) {
  constexpr int TS = 8, SB = TS + 4;
  constexpr int G = kBlock / KC;      // thread groups: 4 classes x G/4 parts
  constexpr int NT = 16 / (G / 4);    // targets per thread (16 per class per tile)
  static_assert(G % 4 == 0 && NT >= 1 && 16 % (G / 4) == 0, "KC must divide the tile");
  __shared__ cplx<T> src[SB * SB][KC];
  __shared__ cplx<T> tr[49][KC];
  const int rhs = blockIdx.y;
  if (rhs_off(act, rhs)) return;
  const int nb = 1 << lev;
  const int nchunk = (S + KC - 1) / KC;
  const int lb = xcd_block();
  const int tile = lb / nchunk, chunk = lb - tile * nchunk;
  const int k0 = chunk * KC;
  const unsigned m0 = (unsigned)tile * TS * TS;
  const int X0 = (int)compact2(m0), Y0 = (int)compact2(m0 >> 1);
  m2l_stage<T, TS, KC>(src, tr, agm + rhs * st, trans, X0, Y0, k0, nb, S);
  __syncthreads();
  const int kk = threadIdx.x % KC, grp = threadIdx.x / KC;
  const int cls = grp & 3, part = grp >> 2;
  cplx<T>* out = agl + rhs * st;
  switch (cls) {
    case 0: m2l_class<T, 0, 0, KC, NT>(src, tr, kk, part, out, m0, S, k0); break;
    case 1: m2l_class<T, 1, 0, KC, NT>(src, tr, kk, part, out, m0, S, k0); break;
    case 2: m2l_class<T, 0, 1, KC, NT>(src, tr, kk, part, out, m0, S, k0); break;
    default: m2l_class<T, 1, 1, KC, NT>(src, tr, kk, part, out, m0, S, k0); break;
  }
}

// M2L per parent: a workgroup owns 4x4 parents (8x8 target boxes) and 16
// samples; a thread owns one parent and one sample.  The far lists of the
// four children all lie in the parent's 6x6 neighbourhood of child-level
// boxes: the thread loads those 36 sources into registers once, then walks
// the 49 translation offsets, reading each operator once and applying it to
// every child for which that offset is a far interaction (27 per child).
// LDS reads per thread: 36 + 49 for 108 complex multiply-adds.
constexpr int kParTS = 8, kParSB = kParTS + 4, kParKC = 16;

// Workgroup coordinates of k_m2l_par: 8x8 boxes starting at Morton index m0 (corner X0, Y0), samples k0 .. k0+15.
struct ParBlock {
  int chunk, k0, X0, Y0;
  unsigned m0;
  __device__ __forceinline__ ParBlock(int S, int lb) {
    const int nchunk = (S + kParKC - 1) / kParKC;
    const int tile = lb / nchunk;
    chunk = lb - tile * nchunk;
    k0 = chunk * kParKC;
    m0 = (unsigned)tile * kParTS * kParTS;
    X0 = (int)compact2(m0);
    Y0 = (int)compact2(m0 >> 1);
  }
};

// the parent's 6x6 source neighbourhood (first child at tile position lx0, ly0)
template <typename T>
__device__ __forceinline__ void par_load(const cplx<T> (*src)[kParKC], int lx0, int ly0, int kk, cplx<T> (&sv)[6][6]) {
#pragma unroll
  for (int dy = 0; dy < 6; dy++)
#pragma unroll
    for (int dx = 0; dx < 6; dx++) sv[dy][dx] = src[(ly0 + dy) * kParSB + lx0 + dx][kk];
}

// acc[c] = sum over the 27 far offsets of child c of T_offset * source
template <typename T>
__device__ __forceinline__ void par_translate(const cplx<T> (*tr)[kParKC], int kk, const cplx<T> (&sv)[6][6],
                                              cplx<T> (&acc)[4]) {
#pragma unroll
  for (int c = 0; c < 4; c++) acc[c] = mkc<T>(0, 0);
#pragma unroll
  for (int ey = -3; ey <= 3; ey++)
#pragma unroll
    for (int ex = -3; ex <= 3; ex++) {
      const cplx<T> t = tr[7 * (ey + 3) + ex + 3][kk];
      if (ex >= -1 && ex <= 1 && ey >= -1 && ey <= 1) continue;  // near offsets
#pragma unroll
      for (int c = 0; c < 4; c++) {
        const int sx = (c & 1) + ex, sy = (c >> 1) + ey;  // source, relative to the first child
        if (sx >= -2 && sx <= 3 && sy >= -2 && sy <= 3) acc[c] = cfma(t, sv[sy + 2][sx + 2], acc[c]);
      }
    }
}

// The same sums source by source: each of the 36 sources is read once and
// added into every child it is a far-field source of, with that offset's
// operator (read from LDS per use): registers for 4 accumulators instead of
// the 36-source neighbourhood.
template <typename T>
__device__ __forceinline__ void par_translate_stream(const cplx<T> (*src)[kParKC], const cplx<T> (*tr)[kParKC],
                                                     int lx0, int ly0, int kk, cplx<T> (&acc)[4]) {
#pragma unroll
  for (int c = 0; c < 4; c++) acc[c] = mkc<T>(0, 0);
#pragma unroll
  for (int sy = -2; sy <= 3; sy++)
#pragma unroll
    for (int sx = -2; sx <= 3; sx++) {
      const cplx<T> v = src[(ly0 + sy + 2) * kParSB + lx0 + sx + 2][kk];
#pragma unroll
      for (int c = 0; c < 4; c++) {
        const int ex = sx - (c & 1), ey = sy - (c >> 1);  // offset of the source from child c
        if (ex < -3 || ex > 3 || ey < -3 || ey > 3) continue;
        if (ex >= -1 && ex <= 1 && ey >= -1 && ey <= 1) continue;  // near offsets
        acc[c] = cfma(tr[7 * (ey + 3) + ex + 3][kk], v, acc[c]);
      }
    }
}

// One level of a merged M2L launch: its multipoles, locals, operators and
// first workgroup (per right-hand side).
template <typename T>
struct M2LLevel {
  const cplx<T>* m;
  cplx<T>* l;
  const cplx<T>* trans;
  long st;
  int first, lev, S;
};
constexpr int kM2LMaxLevels = 10;
template <typename T>
struct M2LSet {
  M2LLevel<T> lv[kM2LMaxLevels];
  int n;
};

// M2L of several levels in one launch (they are independent once the
// multipoles are there): workgroups first[q] .. of the grid belong to set
// entry q.  A level of 4 x 4 boxes fills a quarter of its one tile.
// (at least 2 waves per SIMD: the FP64 instantiation otherwise takes 256+ registers
// and runs one wave per SIMD; measured 2.00 -> 1.52 ms per FP64 launch set)
template <typename T>
__global__ void __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(2)))
k_m2l_par(M2LSet<T> set, const int* __restrict__ act) {
  __shared__ cplx<T> src[kParSB * kParSB][kParKC];
  __shared__ cplx<T> tr[49][kParKC];
  const int rhs = blockIdx.y;
  if (rhs_off(act, rhs)) return;
  const int lb = xcd_block();
  M2LLevel<T> L = set.lv[0];
  for (int q = 1; q < set.n; q++)
    if (lb >= set.lv[q].first) L = set.lv[q];
  const int S = L.S, nb = 1 << L.lev;
  const ParBlock B(S, lb - L.first);
  m2l_stage<T, kParTS, kParKC>(src, tr, L.m + rhs * L.st, L.trans, B.X0, B.Y0, B.k0, nb, S);
  __syncthreads();
  const int kk = threadIdx.x % kParKC, pp = threadIdx.x / kParKC;
  const int lx0 = 2 * (pp & 3), ly0 = 2 * (pp >> 2);  // first child of the parent, tile coordinates
  if (lx0 >= nb || ly0 >= nb || B.k0 + kk >= S) return;
  cplx<T> acc[4];
  if constexpr (sizeof(T) == 8) {
    par_translate_stream<T>(src, tr, lx0, ly0, kk, acc);
  } else {
    cplx<T> sv[6][6];
    par_load<T>(src, lx0, ly0, kk, sv);
    par_translate<T>(tr, kk, sv, acc);
  }
  cplx<T>* out = L.l + rhs * L.st + (long)(B.m0 + 4 * morton2((unsigned)(pp & 3), (unsigned)(pp >> 2))) * S;
#pragma unroll
  for (int c = 0; c < 4; c++) out[(long)c * S + B.k0 + kk] = acc[c];
}

// Input of P2M: the NB x 64 pixels of boxes b0 .. of system rhs to tile[box][65],
// or the vector step of P2mStep, which forms them (y is unused then).  Loads are
// issued in groups ahead of their LDS stores.
template <typename T, typename TI, int NB, int STEP>
__device__ __forceinline__ void p2m_stage(cplx<T>* tile, const cplx<TI>* __restrict__ y, long ys, long b0, int rhs,
                                          const P2mStep<TI>& step) {
  const cplx<TI>* yr = y + rhs * ys + b0 * 64;
  if constexpr (STEP == 0) {
    stage<sizeof(T) == 4 ? 8 : 4, cplx<TI>>(
        NB * 64, [&](int idx) { return yr[idx]; },
        [&](int idx, cplx<TI> v) { tile[(idx >> 6) * 65 + (idx & 63)] = ccast<T>(v); });
  } else {
    const long o = rhs * ys + b0 * 64, go = rhs * step.gs + b0 * 64;
    const StepCoef c = step_coef<STEP>(step, rhs, tile);
    if constexpr (STEP == 3) __syncthreads();
    stage<4, StepIn<TI>>(
        NB * 64, [&](int idx) { return step_load<STEP>(step, c, o, go, idx); },
        [&](int idx, const StepIn<TI>& in) {
          cplx<TI> pv;
          const cplx<TI> yv = step_value<STEP>(step, c, in, pv);
          if constexpr (STEP > 1) {
            step.p[o + idx] = pv;
            step.y[o + idx] = yv;
          }
          tile[(idx >> 6) * 65 + (idx & 63)] = ccast<T>(yv);
        });
  }
}

// P2M on the matrix cores: agm[box][k] = sum_n coeffT[n][k] y[box*64+n] for a
// tile of NB boxes.  The work is cut into units of 16 rows k x 16 boxes, dealt
// round-robin to the 4 waves: with S = 68 (5 row blocks) and 64-box tiles
// every wave gets 5 units (whole row blocks per wave would leave three waves
// idle half the time).  STEP: the vector step of P2mStep while loading; y is
// unused then.  FP64 up to kP2mSymS samples goes to k_p2m_sym.
// With S <= kP2mRows (at most 5 row blocks) the units' results stay in
// registers until every wave is done, then go through LDS so that the tile's
// contiguous output range [b0 S, (b0 + NB) S) is written with whole,
// coalesced lines (stored from the MFMA layout, a box's row blocks came from
// different waves and partial lines reached HBM separately).
constexpr int kP2mRows = 80;
template <typename T, typename TI, int NB, int STEP = 0>
__global__ void __launch_bounds__(kBlock) k_p2m_mfma(const cplx<TI>* __restrict__ y, long ys,
                                                     cplx<T>* __restrict__ agm, long as,
                                                     const cplx<T>* __restrict__ coeffT, int S,
                                                     const int* __restrict__ act, P2mStep<TI> step) {
  typedef typename Mfma<T>::v4 v4;
  constexpr int NN = NB / 16;
  constexpr int MAXU = (5 * NN + 3) / 4;  // units per wave with 5 row blocks
  __shared__ cplx<T> tile[NB * kP2mRows];  // input rows of 65, later the output rows of S
  const int rhs = blockIdx.y;
  if (rhs_off(act, rhs)) return;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int li = lane & 15, lk = lane >> 4;
  const long b0 = (long)xcd_block() * NB;
  p2m_stage<T, TI, NB, STEP>(tile, y, ys, b0, rhs, step);
  __syncthreads();
  const int nrb = (S + 15) / 16, nunit = nrb * NN;
  const bool staged = S <= kP2mRows;
  cplx<T>* out = agm + rhs * as;
  cplx<T> res[MAXU][4];
  // one unit: rows 16 rb .. +15 of the 16 boxes 16 j .. +15
  auto unit = [&](int u, cplx<T>(&o)[4]) {
    const int rb = u / NN, j = u - rb * NN;
    v4 p1 = v4{0, 0, 0, 0}, p2 = v4{0, 0, 0, 0}, p3 = v4{0, 0, 0, 0};
    const int krow = 16 * rb + li;
    const cplx<T>* trow = tile + (16 * j + li) * 65;
    // the coefficients of PRE k-steps are loaded together ahead of their MFMAs
    constexpr int PRE = sizeof(T) == 4 ? 8 : 4;
#pragma unroll 1
    for (int k0 = 0; k0 < 16; k0 += PRE) {
      cplx<T> a[PRE];
#pragma unroll
      for (int v = 0; v < PRE; v++) a[v] = (krow < S) ? coeffT[(4 * (k0 + v) + lk) * S + krow] : mkc<T>(0, 0);
#pragma unroll
      for (int v = 0; v < PRE; v++) {
        const T asum = a[v].x + a[v].y;
        Mfma<T>::cmac3(trow[4 * (k0 + v) + lk], a[v], asum, p1, p2, p3);
      }
    }
#pragma unroll
    for (int q = 0; q < 4; q++) o[q] = mkc<T>(p1[q] - p2[q], p3[q] - p1[q] - p2[q]);
  };
  if (staged) {
    // the wave's units as one software pipeline over (unit, k-batch) steps:
    // the coefficients of the next step are loaded while the current step's
    // MFMAs run (coeffT comes from L2; one step waiting for its own loads per
    // batch was the kernel's critical path)
    constexpr int PRE = sizeof(T) == 4 ? 8 : 4;
    constexpr int NBAT = 16 / PRE;  // k-batches per unit
    cplx<T> ab[2][PRE];
    auto load_step = [&](int c, int b, cplx<T>(&a)[PRE]) {
      const int u = w + 4 * c, krow = 16 * (u / NN) + li;
#pragma unroll
      for (int v = 0; v < PRE; v++)
        a[v] = (u < nunit && krow < S) ? coeffT[(4 * (b * PRE + v) + lk) * S + krow] : mkc<T>(0, 0);
    };
    load_step(0, 0, ab[0]);
#pragma unroll
    for (int c = 0; c < MAXU; c++) {
      const int u = w + 4 * c;
      const int j = u - (u / NN) * NN;
      const cplx<T>* trow = tile + (16 * j + li) * 65;
      v4 p1 = v4{0, 0, 0, 0}, p2 = v4{0, 0, 0, 0}, p3 = v4{0, 0, 0, 0};
#pragma unroll
      for (int b = 0; b < NBAT; b++) {
        const int i = c * NBAT + b;
        if (i + 1 < MAXU * NBAT) load_step((i + 1) / NBAT, (i + 1) % NBAT, ab[(i + 1) & 1]);
        if (u < nunit) {
#pragma unroll
          for (int v = 0; v < PRE; v++) {
            const cplx<T> a = ab[i & 1][v];
            Mfma<T>::cmac3(trow[4 * (b * PRE + v) + lk], a, a.x + a.y, p1, p2, p3);
          }
        }
      }
#pragma unroll
      for (int q = 0; q < 4; q++) res[c][q] = mkc<T>(p1[q] - p2[q], p3[q] - p1[q] - p2[q]);
    }
    __syncthreads();  // the input tile is no longer read: it takes the output
#pragma unroll
    for (int c = 0; c < MAXU; c++) {
      const int u = w + 4 * c;
      const int rb = u / NN, j = u - rb * NN, krow = 16 * rb + li;
      if (u < nunit && krow < S) {
#pragma unroll
        for (int q = 0; q < 4; q++) tile[(16 * j + Mfma<T>::row(lk, q)) * S + krow] = res[c][q];
      }
    }
    __syncthreads();
    cplx<T>* ob = out + b0 * S;
    for (int e = tid; e < NB * S; e += kBlock) ob[e] = tile[e];
  } else {
    for (int u = w; u < nunit; u += 4) {
      cplx<T> o[4];
      unit(u, o);
      const int rb = u / NN, j = u - rb * NN, krow = 16 * rb + li;
      if (krow < S) {
#pragma unroll
        for (int q = 0; q < 4; q++) out[(b0 + 16 * j + Mfma<T>::row(lk, q)) * S + krow] = o[q];
      }
    }
  }
}

// Sum of the four waves' partial values of 64 outputs, wave 0 gets it.
__device__ __forceinline__ zd rx_sum(zd v) {
  __shared__ zd sh[3][64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (w) sh[w - 1][lane] = v;
  __syncthreads();
  if (!w)
    for (int i = 0; i < 3; i++) v = cadd(v, sh[i][lane]);
  return v;
}

// Receiver interpolation.  Both directions are short sums of gathered values and
// were bound by the latency of one tap after the other (1000 outputs, 33 and 14
// us): a workgroup owns 64 outputs, its waves a quarter of the taps each, several
// of them in flight (512 px x 16: 33 -> 5.3 us, 14.5 -> 4.4 us).
// Grid (ceil(outputs / 64), right-hand sides).

// receiver values: out[m] = sum_t wT[t][m] agm0[(i0[m]+t) mod S0]
template <typename T>
__global__ void __launch_bounds__(kBlock) k_rx_interp(const cplx<T>* __restrict__ agm0, long as, zd* __restrict__ out,
                                                      long os, const T* __restrict__ wT, const int* __restrict__ i0,
                                                      int S0, int R, int ntap) {
  const int rhs = blockIdx.y, m = blockIdx.x * 64 + (threadIdx.x & 63), w = threadIdx.x >> 6;
  const int q = (ntap + 3) / 4, t1 = min(q * (w + 1), ntap);
  zd acc = mkc<double>(0, 0);
  if (m < R) {
    const cplx<T>* a = agm0 + rhs * as;
    const int j0 = i0[m];
#pragma unroll 4
    for (int t = q * w; t < t1; t++) {
      const zd v = ccast<double>(a[(j0 + t) % S0]);
      const double x = (double)wT[t * R + m];
      acc.x += x * v.x;
      acc.y += x * v.y;
    }
  }
  acc = rx_sum(acc);
  if (w == 0 && m < R) out[rhs * os + m] = acc;
}

// root locals from receiver values: agl0[k] = (sum_t aT[t][k] in[aI[t][k]]) * (-4i) * sc
template <typename T>
__global__ void __launch_bounds__(kBlock) k_rx_anterp(const zd* __restrict__ in, long is, cplx<T>* __restrict__ agl0,
                                                      long as, const T* __restrict__ aT, const int* __restrict__ aI,
                                                      int S0, int ntap, double sc) {
  const int rhs = blockIdx.y, k = blockIdx.x * 64 + (threadIdx.x & 63), w = threadIdx.x >> 6;
  const int q = (ntap + 3) / 4, t1 = min(q * (w + 1), ntap);
  zd acc = mkc<double>(0, 0);
  if (k < S0) {
    const zd* v = in + rhs * is;
#pragma unroll 5
    for (int t = q * w; t < t1; t++) {
      const double x = (double)aT[t * S0 + k];
      const zd u = v[aI[t * S0 + k]];
      acc.x += x * u.x;
      acc.y += x * u.y;
    }
  }
  acc = rx_sum(acc);
  if (w == 0 && k < S0) {
    const zd r = cmul(acc, mkc<double>(0.0, -4.0));
    agl0[rhs * as + k] = ccast<T>(mkc<double>(r.x * sc, r.y * sc));
  }
}

}  // namespace isg
