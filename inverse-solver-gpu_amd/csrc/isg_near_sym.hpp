// isg_near_sym.hpp -- near field + leaf receiving patterns (L2P) on the matrix
// cores in the mirror-symmetric basis of a leaf box.
//
// The kernel h(dx, dy) of the near field depends on |dx| and |dy| only, and the
// leaf directions are equispaced (S a multiple of 4), so both stages commute
// with the two reflections of a leaf box about its centre lines.  With
//   X_c(i, j) = sum over signs of chi_c x(+-i, +-j)     (i, j = 0..11: a quarter
//                of the 24 x 24 pixel window of the box and its neighbours)
//   Y_c(p, q) likewise for the 8 x 8 outputs            (p, q = 0..3)
// for the four classes c = (even / odd in x, even / odd in y) the product
// splits into four independent ones, Y_c = T_c X_c with T_c 144 x 16 instead
// of one 576 x 64: a quarter of the multiplications.  L2P splits the same way
// over the orbits of the directions: 4 x (S / 4 + 1) x 16 instead of S x 64.
// The transforms are sums of 4 values; forming the operand costs 6 additions
// per matrix-core operand (3 products of 16 x 16 x 4), and the outputs are
// transformed back in LDS.
//
// What bounds it: in FP64 and FP32 the matrix cores and the vector ALUs do not
// overlap (4 waves per SIMD, FP64 512^2 x 16 right-hand sides: 53 us of MFMA and
// 23 of vector work in 100 us, 205 MB of memory traffic 43 us).  Per launch, dense
// blocks / this kernel: FP64 1024^2 x 1 77 / 31 us, 512^2 x 16 280 / 100 us,
// 1024^2 x 64 4600 / 1530 us.  16-box tiles (2.25 x the tile's pixels staged, from
// L2, but 4 workgroups per CU) beat 32-box ones everywhere: 100 / 120 us.
#pragma once

#include "isg_kernels.hpp"

namespace isg {

constexpr int kSymK = 144;  // quarter-window pixels

// orbits of the S leaf directions under the reflections, rounded up to a k-step of 4
__host__ __device__ inline int sym_reps(int S) { return (S / 4 + 1 + 3) / 4 * 4; }

// Halo layout of the tile: element (box (hx, hy), pixel) at hy RS + hx BS + pixel.
// A wave reads, for 16 boxes (4 x 4) and 4 neighbouring pixels, one element per
// lane; BS and RS make the lanes of one LDS pass hit different banks (16-byte
// elements: 8 lanes, BS odd and RS = 4 mod 8; 8-byte ones: 32 lanes, BS = 2 and
// RS = 8 mod 32).
template <typename T>
struct SymTile {
  static constexpr int kBox = sizeof(T) == 8 ? 65 : 66;
  static constexpr int row(int hx) {
    constexpr int m = sizeof(T) == 8 ? 8 : 32, want = sizeof(T) == 8 ? 4 : 8;
    const int r = hx * kBox;
    return r + (want + m - r % m) % m;
  }
};

// LDS elements of k_near_mfma<NB>: the halo, later NB rows of S + 1 locals, later NB x 64 outputs.
template <typename T>
__host__ __device__ inline int near_sym_elems(int NB, int S, bool with_near) {
  const int tx = (NB == 16) ? 4 : 8, ty = NB / tx;
  const int halo = with_near ? (ty + 2) * SymTile<T>::row(tx + 2) : 0;
  const int l2p = NB * (S + 1) > NB * 64 ? NB * (S + 1) : NB * 64;
  return halo > l2p ? halo : l2p;
}

// Tables, rounded from FP64: near[c][12 j + i][4 q + p] and l2p[c][m][4 q + p]
// (m < sym_reps(S), zero for m > S / 4), c = 2 (odd in y) + (odd in x); (p, q)
// the column and row distance from the box centre, output pixel (4 + q, 4 + p).
// A direction on an axis (m = 0, S / 4) appears twice in its orbit sum: weight 1/2.
template <typename T>
__global__ void __launch_bounds__(256) k_sym_tables(const zd* __restrict__ near, const zd* __restrict__ basisT, int S,
                                                    cplx<T>* __restrict__ tn, cplx<T>* __restrict__ tl) {
  const int nrep = sym_reps(S), nn = 4 * kSymK * 16, nl = 4 * nrep * 16;
  for (int e = blockIdx.x * 256 + threadIdx.x; e < nn + nl; e += gridDim.x * 256) {
    const bool is_near = e < nn;
    const int f = is_near ? e : e - nn, K = is_near ? kSymK : nrep;
    const int c = f / (K * 16), k = f / 16 % K, pq = f & 15;
    const int m = (4 + (pq >> 2)) * 8 + 4 + (pq & 3);
    zd s = mkc<double>(0, 0);
    double wgt = 0.25;
    for (int g = 0; g < 4; g++) {  // g = 2 (row mirrored) + (column mirrored)
      const bool neg = (((g & 1) & c) ^ ((g >> 1) & (c >> 1))) != 0;
      zd v = mkc<double>(0, 0);
      if (is_near) {
        const int i = k % 12, j = k / 12;
        const int wc = (g & 1) ? 11 - i : 12 + i, wr = (g & 2) ? 11 - j : 12 + j;
        v = near[((long)(3 * (wr >> 3) + (wc >> 3)) * 64 + (wr & 7) * 8 + (wc & 7)) * 64 + m];
      } else if (k <= S / 4) {
        const int d = g == 0 ? k : (g == 1 ? S / 2 - k : (g == 2 ? (k ? S - k : 0) : S / 2 + k));
        v = basisT[(long)d * 64 + m];
        if (k == 0 || k == S / 4) wgt = 0.125;
      }
      s = neg ? csub(s, v) : mkc<double>(s.x + v.x, s.y + v.y);
    }
    (is_near ? tn : tl)[f] = mkc<T>((T)(wgt * s.x), (T)(wgt * s.y));
  }
}

// Class values to pixels, in place: tile[box][64] holds class c's value of
// (p, q) in the place of the pixel in quadrant c.
template <typename T, int NB>
__device__ __forceinline__ void sym_unfold(cplx<T>* tile) {
#pragma unroll
  for (int u = 0; u < NB / 16; u++) {
    const int e = threadIdx.x + u * kBlock, p = e & 3, q = (e >> 2) & 3;
    cplx<T>* t = tile + (e >> 4) * 64;
    cplx<T>*t0 = t + (4 + q) * 8 + 4 + p, *t1 = t + (4 + q) * 8 + 3 - p, *t2 = t + (3 - q) * 8 + 4 + p,
           *t3 = t + (3 - q) * 8 + 3 - p;
    const cplx<T> a = cadd(*t0, *t1), b = csub(*t0, *t1), c = cadd(*t2, *t3), d = csub(*t2, *t3);
    *t0 = cadd(a, c);
    *t1 = cadd(b, d);
    *t2 = csub(a, c);
    *t3 = csub(b, d);
  }
}

// Workgroup: NB Morton-consecutive boxes of one right-hand side, wave w = class w.
// Data operand (A): lane li + 16 lk holds element k = 4 kk + lk of box li of a
// 16-box block, formed from four LDS reads; table (B): column li = output (p, q).
// Complex products in the three-product form.  Epilogues (POST) as NearPost.
template <typename T, typename TI, int NB, int POST>
__global__ void __launch_bounds__(kBlock) k_near_mfma(const cplx<TI>* __restrict__ y, long ys,
                                                     const cplx<T>* __restrict__ loc, long ls,
                                                     cplx<TI>* __restrict__ r, long rs, const cplx<T>* __restrict__ tn,
                                                     const cplx<T>* __restrict__ tl, int S, int nbs, int with_near,
                                                     const int* __restrict__ act, NearPost<TI> post) {
  typedef typename Mfma<T>::v4 v4;
  constexpr int NN = NB / 16;
  constexpr int TX = (NB == 16) ? 4 : 8, TY = NB / TX, HX = TX + 2, HY = TY + 2;
  constexpr int BS = SymTile<T>::kBox, RS = SymTile<T>::row(HX);
  constexpr int PRE = 6;  // k-steps (two quarter-window rows) whose table values are loaded ahead
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  cplx<T>* tile = reinterpret_cast<cplx<T>*>(smem_raw);
  const int rhs = blockIdx.y;
  if (rhs_off(act, rhs)) return;
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, lk = lane >> 4;
  const long b0 = (long)xcd_block() * NB;
  const T sx = (w & 1) ? (T)-1 : (T)1, sy = (w & 2) ? (T)-1 : (T)1;
  v4 p1[NN], p2[NN], p3[NN];
#pragma unroll
  for (int j = 0; j < NN; j++) {
    p1[j] = v4{0, 0, 0, 0};
    p2[j] = v4{0, 0, 0, 0};
    p3[j] = v4{0, 0, 0, 0};
  }
  // class w's combination of the four mirror images (column, row)
  auto fold = [&](cplx<T> pp, cplx<T> mp, cplx<T> pm, cplx<T> mm) {
    const T ax = fma(sx, mp.x, pp.x), ay = fma(sx, mp.y, pp.y);
    const T bx = fma(sx, mm.x, pm.x), by = fma(sx, mm.y, pm.y);
    return mkc<T>(fma(sy, bx, ax), fma(sy, by, ay));
  };
  const cplx<TI>* yr = y + rhs * ys;
  const int nlk = sym_reps(S) / 4;
  const cplx<T>* tln = tl + ((long)w * 4 * nlk + lk) * 16 + li;
  cplx<T> tb[2][PRE];
  if (with_near) {
    const cplx<T>* tnn = tn + ((long)w * kSymK + lk) * 16 + li;
#pragma unroll
    for (int u = 0; u < PRE; u++) tb[0][u] = tnn[u * 64];
    const int X0 = (int)compact2((unsigned)b0), Y0 = (int)compact2((unsigned)b0 >> 1);
    // pixel offset of each halo box (Morton index * 64), -1 outside the grid, and its place in LDS
    __shared__ int hoff[HX * HY], hpos[HX * HY];
    for (int h = tid; h < HX * HY; h += kBlock) {
      const int sxb = X0 - 1 + h % HX, syb = Y0 - 1 + h / HX;
      hoff[h] = (sxb >= 0 && syb >= 0 && sxb < nbs && syb < nbs) ? (int)morton2(sxb, syb) * 64 : -1;
      hpos[h] = (h / HX) * RS + (h % HX) * BS;
    }
    __syncthreads();
    stage<sizeof(T) == 4 ? 8 : 4, cplx<TI>>(
        HX * HY * 64,
        [&](int idx) {
          const int off = hoff[idx >> 6];
          cplx<TI> v = mkc<TI>(0, 0);
          if (off >= 0) {
            v = yr[(long)off + (idx & 63)];
            // residual check: the input is the iterate x, contrast-weighted here
            if constexpr (POST == 3) v = prep_val(v, post.g, rhs * post.gs + off + (idx & 63), post.herm != 0);
          }
          return v;
        },
        [&](int idx, cplx<TI> v) { tile[hpos[idx >> 6] + (idx & 63)] = ccast<T>(v); });
    // window corner (upper left neighbour) of box 16 j + li, plus and minus side of this lane's column
    const cplx<T>*wp[NN], *wm[NN];
#pragma unroll
    for (int j = 0; j < NN; j++) {
      const unsigned c = (unsigned)(16 * j + li);
      const int base = (int)compact2(c >> 1) * RS + (int)compact2(c) * BS;
      wp[j] = tile + base + lk;
      wm[j] = tile + base + 3 - lk;
    }
    __syncthreads();
#pragma unroll
    for (int bt = 0; bt < 6; bt++) {
      if (bt + 1 < 6) {
#pragma unroll
        for (int u = 0; u < PRE; u++) tb[(bt + 1) & 1][u] = tnn[((bt + 1) * PRE + u) * 64];
      }
#pragma unroll
      for (int u = 0; u < PRE; u++) {
        const int jr = 2 * bt + u / 3, q = u % 3;  // k = 12 jr + 4 q + lk
        // offsets from the window corner: rows 12 + jr and 11 - jr, columns 12 + 4 q + lk and 11 - 4 q - lk
        const int rp = jr < 4 ? RS + (4 + jr) * 8 : 2 * RS + (jr - 4) * 8;
        const int rm = jr < 4 ? RS + (3 - jr) * 8 : (11 - jr) * 8;
        const int cp = q == 0 ? BS + 4 : 2 * BS + (q - 1) * 4;
        const int cm = q == 0 ? BS : (2 - q) * 4;
        const cplx<T> a = tb[bt & 1][u];
        const T asum = a.x + a.y;
#pragma unroll
        for (int j = 0; j < NN; j++) {
          const cplx<T> d = fold(wp[j][rp + cp], wm[j][rp + cm], wp[j][rm + cp], wm[j][rm + cm]);
          Mfma<T>::cmac3(d, a, asum, p1[j], p2[j], p3[j]);
        }
      }
    }
  }
  // ---- L2P over the direction orbits m = 4 kk + lk <= S / 4 (rows of S + 1 locals in LDS)
#pragma unroll
  for (int u = 0; u < PRE; u++) tb[0][u] = tln[(u < nlk ? u : nlk - 1) * 64];
  __syncthreads();
  const cplx<T>* lr = loc + rhs * ls + b0 * S;
  {
    // element idx = j * S + k goes to tile[j * (S + 1) + k] = tile[idx + j];
    // j is stepped rather than divided out of idx
    constexpr int U = sizeof(T) == 4 ? 8 : 4;
    const int n = NB * S, dj = kBlock / S, dk = kBlock - dj * S;
    int jb = tid / S, kq = tid - jb * S;
    for (int e0 = tid; e0 < n; e0 += U * kBlock) {
      cplx<T> v[U];
      int ju[U];
#pragma unroll
      for (int u = 0; u < U; u++) {
        const int e = e0 + u * kBlock;
        ju[u] = jb;
        v[u] = lr[e < n ? e : n - 1];  // unconditional (clamped) load: the array stays in registers
        kq += dk;
        jb += dj;
        if (kq >= S) {
          kq -= S;
          jb++;
        }
      }
#pragma unroll
      for (int u = 0; u < U; u++) {
        const int e = e0 + u * kBlock;
        if (e < n) tile[e + ju[u]] = v[u];
      }
    }
  }
  __syncthreads();
#pragma unroll 1
  for (int k0 = 0; k0 < nlk; k0 += PRE) {
    if (k0 > 0) {
#pragma unroll
      for (int u = 0; u < PRE; u++) tb[0][u] = tln[(k0 + u < nlk ? k0 + u : nlk - 1) * 64];
    }
#pragma unroll
    for (int u = 0; u < PRE; u++) {
      if (k0 + u < nlk) {
        const int m = min(4 * (k0 + u) + lk, S >> 2);  // (past S / 4 the table is zero)
        const int d1 = (S >> 1) - m, d2 = m ? S - m : 0, d3 = (S >> 1) + m;
        const cplx<T> a = tb[0][u];
        const T asum = a.x + a.y;
#pragma unroll
        for (int j = 0; j < NN; j++) {
          const cplx<T>* t = tile + (16 * j + li) * (S + 1);
          const cplx<T> d = fold(t[m], t[d1], t[d2], t[d3]);
          Mfma<T>::cmac3(d, a, asum, p1[j], p2[j], p3[j]);
        }
      }
    }
  }
  // ---- back to pixels: class w's value of (p, q) takes the place of the
  // pixel in quadrant w, then each thread transforms its quadruples in place
  __syncthreads();
#pragma unroll
  for (int j = 0; j < NN; j++) {
    const int p = li & 3, q = li >> 2;
    const int px = ((w & 2) ? 3 - q : 4 + q) * 8 + ((w & 1) ? 3 - p : 4 + p);
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const T re = p1[j][i] - p2[j][i], im = p3[j][i] - p1[j][i] - p2[j][i];
      tile[(16 * j + Mfma<T>::row(lk, i)) * 64 + px] = mkc<T>(re, im);
    }
  }
  __syncthreads();
  sym_unfold<T, NB>(tile);
  __syncthreads();
  near_epilogue<T, TI, NB, POST>(tile, r, rs, b0, rhs, post);
}

}  // namespace isg
