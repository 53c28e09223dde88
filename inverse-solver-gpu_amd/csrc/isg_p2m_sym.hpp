// isg_p2m_sym.hpp -- leaf radiation patterns (P2M) in the mirror-symmetric basis
// of a leaf box, with the interpolation to the parents (M2M of the leaf level)
// in the same workgroup.
//
// A plane wave exp(-i k.d) is a product of one factor in x and one in y, so with
// the classes c = (even / odd in x, even / odd in y) of isg_near_sym.hpp
//   F_c(p, q)  = sum over the four mirror images g of chi_c(g) y(g (p, q))
//   Z_c(m)     = i^[c = 1, 2] sum_pq tau_c(p, q; m) F_c(p, q),   m = 0 .. S / 4
//   M(g m)     = sum_c chi_c(g) Z_c(m)
// with real tables tau: 4 x 16 x (S / 4 + 1) real-by-complex products instead of
// 64 x S complex ones, 2 matrix products where the dense form took 3 and a
// quarter of the rows (S = 68: 18 of 32, in two blocks): a sixth of the
// matrix work, which was most of the dense kernel's time.
// The multipoles are then in LDS, where the band of the parents' interpolator is
// applied to them: as a kernel of its own M2M read them back from memory.
// P2M + leaf M2M, dense P2M and band M2M / this kernel: 256 px x 1 9.6 + 8.2 / 11.1
// us, 1024 px x 1 18.5 + 13 / 20.2, 512 px x 16 51 + 37 / 55 (170 MB: 36 us at the
// rate of a large copy), 1024 px x 64 739 + 530 / 870.
// FP64 only: FP32 has the split-FP16 kernel for large batches.
#pragma once

#include "isg_kernels.hpp"

namespace isg {

constexpr int kP2mSymS = 124;  // directions: S / 4 + 1 <= 32 orbits, two column blocks
constexpr int kSymBand = 48;   // longest band window

// tau[c][4 q + p][m], m < 32 (zero past S / 4); (p, q) the column and row distance
// from the box centre.
__global__ void __launch_bounds__(256) k_sym_p2m_table(const zd* __restrict__ coeffT, int S, double* __restrict__ tau) {
  const int e = blockIdx.x * 256 + threadIdx.x;
  if (e >= 4 * 16 * 32) return;
  const int m = e & 31, p = (e >> 5) & 3, q = (e >> 7) & 3, c = e >> 9;
  double v = 0;
  if (m <= S / 4)
    for (int g = 0; g < 4; g++) {  // g = 2 (row mirrored) + (column mirrored)
      const int n = ((g & 2) ? 3 - q : 4 + q) * 8 + ((g & 1) ? 3 - p : 4 + p);
      const zd a = coeffT[(long)n * S + m];
      const double x = (c == 0 || c == 3) ? a.x : a.y;
      v += (((g & 1) & c) ^ ((g >> 1) & (c >> 1))) ? -x : x;
    }
  tau[e] = 0.25 * v;
}

// M2M of the leaf level (UP): band blocks ab[sample block 16][kb][16] of the
// interpolator with window starts s0, child shifts [4][Sp].
struct SymUp {
  zd* par = nullptr;
  long ps = 0;
  const double* ab = nullptr;
  const int* s0 = nullptr;
  const zd* shift = nullptr;
  int Sp = 0, kb = 0;
};

__host__ __device__ inline size_t p2m_sym_lds(int NB, int S) {
  return (size_t)NB * (S + 1 > 65 ? S + 1 : 65) * sizeof(zd);
}

// Workgroup: NB Morton-consecutive boxes of one right-hand side; wave w = class w,
// then sample blocks w, w + 4, .. of the parents.  S a multiple of 4.
// Dynamic LDS p2m_sym_lds: the pixels [box][65], later the multipoles [box][S + 1].
template <int NB, int STEP, bool UP>
__global__ void __launch_bounds__(kBlock) k_p2m_sym(const zd* __restrict__ y, long ys, zd* __restrict__ agm, long as,
                                                    const double* __restrict__ tau, int S,
                                                    const int* __restrict__ act, P2mStep<double> step, SymUp up) {
  typedef Mfma<double>::v4 v4;
  constexpr int NN = NB / 16;
  extern __shared__ __attribute__((aligned(16))) char smem_raw[];
  zd* tile = reinterpret_cast<zd*>(smem_raw);
  const int rhs = blockIdx.y;
  if (rhs_off(act, rhs)) return;
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, lk = lane >> 4;
  const long b0 = (long)xcd_block() * NB;
  double b[4][2];
#pragma unroll
  for (int q = 0; q < 4; q++)
#pragma unroll
    for (int rb = 0; rb < 2; rb++) b[q][rb] = tau[(w * 16 + 4 * q + lk) * 32 + 16 * rb + li];
  p2m_stage<double, double, NB, STEP>(tile, y, ys, b0, rhs, step);
  __syncthreads();
  // ---- Z_w: rows boxes, columns orbits, K = the quarter's pixels (q, p = lk)
  const double sx = (w & 1) ? -1.0 : 1.0, sy = (w & 2) ? -1.0 : 1.0;
  v4 re[NN][2], im[NN][2];
#pragma unroll
  for (int j = 0; j < NN; j++) {
#pragma unroll
    for (int rb = 0; rb < 2; rb++) re[j][rb] = im[j][rb] = v4{0, 0, 0, 0};
    const zd* t = tile + (16 * j + li) * 65;
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const zd t0 = t[(4 + q) * 8 + 4 + lk], t1 = t[(4 + q) * 8 + 3 - lk], t2 = t[(3 - q) * 8 + 4 + lk],
                    t3 = t[(3 - q) * 8 + 3 - lk];
      const double fx = (t0.x + sx * t1.x) + sy * (t2.x + sx * t3.x), fy = (t0.y + sx * t1.y) + sy * (t2.y + sx * t3.y);
#pragma unroll
      for (int rb = 0; rb < 2; rb++) {
        re[j][rb] = Mfma<double>::mac(fx, b[q][rb], re[j][rb]);
        im[j][rb] = Mfma<double>::mac(fy, b[q][rb], im[j][rb]);
      }
    }
  }
  __syncthreads();
  // class w's value of an orbit goes to the place of its w-th direction (on the
  // axes, m = 0 and S / 4, two classes vanish and two directions coincide)
  const int P = S + 1, q4 = S / 4;
  const bool turn = w == 1 || w == 2;  // factor i
#pragma unroll
  for (int rb = 0; rb < 2; rb++) {
    const int m = 16 * rb + li;
    const int d = w == 0 ? m : (w == 1 ? S / 2 - m : (w == 2 ? S - m : S / 2 + m));
    if (m > q4 || (m == 0 && (w & 2)) || (m == q4 && (w & 1))) continue;
#pragma unroll
    for (int j = 0; j < NN; j++)
#pragma unroll
      for (int i = 0; i < 4; i++)
        tile[(16 * j + Mfma<double>::row(lk, i)) * P + d] =
            turn ? mkc<double>(-im[j][rb][i], re[j][rb][i]) : mkc<double>(re[j][rb][i], im[j][rb][i]);
  }
  __syncthreads();
  // ---- classes to directions, in place
  for (int e = tid; e < NB * 32; e += kBlock) {
    const int m = e & 31;
    if (m > q4) continue;
    zd* t = tile + (e >> 5) * P;
    if (m == 0 || m == q4) {
      zd*t0 = t + m, *t1 = t + (m == 0 ? S / 2 : S - m);
      const zd a = *t0, c = *t1;
      *t0 = cadd(a, c);
      *t1 = csub(a, c);
    } else {
      zd*t0 = t + m, *t1 = t + S / 2 - m, *t2 = t + S - m, *t3 = t + S / 2 + m;
      const zd a = cadd(*t0, *t1), c = csub(*t0, *t1), d = cadd(*t2, *t3), f = csub(*t2, *t3);
      *t0 = cadd(a, d);  // chi(identity): + + + +
      *t1 = cadd(c, f);  // column mirrored: + - + -
      *t2 = csub(a, d);  // row mirrored: + + - -
      *t3 = csub(c, f);  // both: + - - +
    }
  }
  __syncthreads();
  zd* ob = agm + rhs * as + b0 * S;
  for (int e = tid; e < NB * S; e += kBlock) {
    const int bx = e / S;
    ob[e] = tile[e + bx];
  }
  if constexpr (UP) {
    // ---- M2M: rows boxes, permuted so that a lane ends with the four children of
    // one parent, columns 16 parent samples, K the window of child samples
    constexpr int NQ = kSymBand / 4;
    const int br = 4 * (li & 3) + (li >> 2), nck = (up.Sp + 15) / 16;
    for (int ck = w; ck < nck; ck += 4) {
      double a[NQ];
#pragma unroll
      for (int q = 0; q < NQ; q++) a[q] = 4 * q < up.kb ? up.ab[(ck * up.kb + 4 * q + lk) * 16 + li] : 0.0;
      const int s0 = up.s0[ck], col = 16 * ck + li;
      zd sh[4];
#pragma unroll
      for (int i = 0; i < 4; i++) sh[i] = up.shift[i * up.Sp + min(col, up.Sp - 1)];
#pragma unroll
      for (int j = 0; j < NN; j++) {
        v4 cr = v4{0, 0, 0, 0}, ci = v4{0, 0, 0, 0};
        const zd* row = tile + (16 * j + br) * P;
#pragma unroll
        for (int q = 0; q < NQ; q++) {
          if (4 * q >= up.kb) break;
          int k = s0 + 4 * q + lk;
          k -= k >= S ? S : 0;
          const zd v = row[k];
          cr = Mfma<double>::mac(v.x, a[q], cr);
          ci = Mfma<double>::mac(v.y, a[q], ci);
        }
        zd o = mkc<double>(0, 0);
#pragma unroll
        for (int i = 0; i < 4; i++) o = cfma(sh[i], mkc<double>(cr[i], ci[i]), o);
        if (col < up.Sp) up.par[rhs * up.ps + ((b0 >> 2) + 4 * j + lk) * up.Sp + col] = o;
      }
    }
  }
}

}  // namespace isg
