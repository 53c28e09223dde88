// isg_down.hpp -- downward pass of one level: its translations (M2L) and the
// interpolation of the parents' locals (L2L) in one kernel.  k_down_h16: the FP32
// operator, interpolating on the FP16 matrix cores with split operands; k_down64:
// the FP64 operator, on the FP64 ones.
//
// local_i[box][k] = sum over the 27 far boxes of T[k] multipole_i[box'][k]
//                 + sum_j A[k][j] shiftL[c][j] local_{i-1}[parent][j]
// Reference counterpart: kernels.cu:239-266 and :137-238.
//
// FP32: the shift of child position c is folded into the anterpolator (a complex
// table per child position), so that the operand is the parents' locals
// themselves: 16 parents x the window of 16 samples, split once into FP16 hi +
// lo (isg_near_h16.hpp) under one power-of-two scale per parent, for four child
// positions.  The separate kernels shifted every parent four times and ran the
// real product on v_mfma_f32_16x16x4, which shares the vector ALUs' time.
#pragma once

#include "isg_near_h16.hpp"

namespace isg {

constexpr int kDownTS = 8, kDownSB = kDownTS + 4, kDownKC = 16;
constexpr int kDownK = 96;                // window slots (three MFMA chunks)
constexpr int kDownG = kDownK / 8;        // groups of 8 slots
constexpr int kDownFrag = 4 * kDownG * 16;  // v8h fragments of a window: [part][group][parent]
constexpr int kDownPer = 16;  // most right-hand sides of a workgroup (bits of `live`)
constexpr int kDownFar = 27;

// Table of one level: out[rb][c][part][g][col] = 8 FP16 parts of
// 2^ec AB[rb][8 g + e][col] shiftL[c][(s0[rb] + 8 g + e) mod Sp], zero past KB.
static __global__ void __launch_bounds__(256) k_split_l2l(const double* __restrict__ AB, const int* __restrict__ s0v,
                                                          int KB, const zd* __restrict__ shift, int Sp, int nrb, int ec,
                                                          v8h* __restrict__ out) {
  const int t = blockIdx.x * 256 + threadIdx.x;
  if (t >= nrb * 4 * kDownG * 16) return;
  const int col = t & 15, g = (t >> 4) % kDownG, c = (t >> 4) / kDownG & 3, rb = (t >> 4) / (kDownG * 4);
  const double s = ldexp(1.0, ec);
  v8h ph[4];
#pragma unroll
  for (int e = 0; e < 8; e++) {
    const int kk = 8 * g + e;
    float x = 0.f, y = 0.f;
    if (kk < KB) {
      int j = s0v[rb] + kk;
      if (j >= Sp) j -= Sp;
      const zd h = shift[c * Sp + j];
      const double a = AB[((long)rb * KB + kk) * 16 + col] * s;
      x = (float)(a * h.x);
      y = (float)(a * h.y);
    }
    h16_split(x, ph[0], ph[1], e);
    h16_split(y, ph[2], ph[3], e);
  }
#pragma unroll
  for (int P = 0; P < 4; P++) out[(((long)(rb * 4 + c) * 4 + P) * kDownG + g) * 16 + col] = ph[P];
}

// max(m, |a|, |b|)
__device__ __forceinline__ float max3_abs(float m, float a, float b) {
  float r;
  asm("v_max3_f32 %0, %1, |%2|, |%3|" : "=v"(r) : "v"(m), "v"(a), "v"(b));
  return r;
}

// Buffer descriptor of `bytes` bytes at p (raw, 32-bit offsets; a load past the
// end returns 0) and an 8-byte load through it.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t down_rsrc(const void* p, unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ zf down_load(__amdgpu_buffer_rsrc_t rs, unsigned off) {
  return __builtin_bit_cast(zf, __builtin_amdgcn_raw_buffer_load_b64(rs, (int)off, 0, 0));
}

// The 27 translation operators of child position (CX, CY) at one sample.
template <int CX, int CY, typename T>
__device__ __forceinline__ void down_load_t(const cplx<T>* __restrict__ trans, int S, int k, cplx<T> (&t)[kDownFar]) {
  int j = 0;
#pragma unroll
  for (int dy = -2 - CY; dy <= 3 - CY; dy++)
#pragma unroll
    for (int dx = -2 - CX; dx <= 3 - CX; dx++)
      if (dx < -1 || dx > 1 || dy < -1 || dy > 1) t[j++] = trans[(long)(7 * (dy + 3) + dx + 3) * S + k];
}

// acc[i] += sum over far offsets of T * source for child position (CX, CY) of the
// four parents i of a 2 x 2 block: their sources lie in 8 x 8 boxes, each read
// once (s points at this lane's sample of box (-2, -2) from the block's corner).
// W sources of a row are read while the previous ones are multiplied (left to
// itself the compiler reads two at a time and waits for them); first holds the
// first W.
template <int CX, int CY, int W, typename T>
__device__ __forceinline__ void down_m2l(const cplx<T>* __restrict__ s, const cplx<T> (&t)[kDownFar],
                                         const cplx<T> (&first)[W], cplx<T> (&acc)[4]) {
  constexpr int H = 8 / W;  // groups per row
  cplx<T> grp[2][W];
#pragma unroll
  for (int x = 0; x < W; x++) grp[0][x] = first[x];
#pragma unroll
  for (int h = 0; h < 8 * H; h++) {  // sources (sx, sy) = (x0 + x - 2, y - 2)
    const int y = h / H, x0 = W * (h % H);
    if (h + 1 < 8 * H) {
#pragma unroll
      for (int x = 0; x < W; x++)
        grp[(h + 1) & 1][x] = s[((h + 1) / H * kDownSB + W * ((h + 1) % H) + x) * kDownKC];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int x = 0; x < W; x++) {
      const cplx<T> v = grp[h & 1][x];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int ax = x0 + x - 2 - 2 * (i & 1), ay = y - 2 - 2 * (i >> 1);  // from the parent's first child
        if (ax < -2 || ax > 3 || ay < -2 || ay > 3) continue;
        const int dx = ax - CX, dy = ay - CY;
        if (dx >= -1 && dx <= 1 && dy >= -1 && dy <= 1) continue;  // near
        // position among the far offsets, row by row: rows above the near
        // block are whole (6), its rows lack 3
        const int far_row = ay + 2, near0 = CY + 1;  // near rows near0 .. near0 + 2
        const int before = 6 * far_row - 3 * (far_row <= near0 ? 0 : (far_row >= near0 + 3 ? 3 : far_row - near0));
        const int in_row = (far_row >= near0 && far_row < near0 + 3 && dx > 1) ? ax + 2 - 3 : ax + 2;
        acc[i] = cfma(t[before + in_row], v, acc[i]);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  }
}

// Workgroup: 8 x 8 boxes (16 parents) and 16 samples, for `per` right-hand sides
// one after another: operators, table fragments and staging offsets are loaded
// once.  Per right-hand side the 12 x 12 source boxes go to LDS and the parents'
// windows are split into it (thread = parent x group of 8 slots; the parent's
// scale from its 16 lanes), double-buffered: one barrier, and the next
// right-hand side's loads run during the products.  Wave w owns child position
// w; lane li + 16 lk holds sample li and, as the matrix cores return it, parents
// 4 lk .. +3, a 2 x 2 block, for which it also sums the translations (64 source
// reads for 108 multiply-adds, the 27 operators in registers): results go
// straight to memory.
// What bounds it (1024^2 x 64 right-hand sides, leaf level, 569 us; the fused
// kernel with the FP32 interpolation took 803, and levels 3 .. 7 together 1018
// instead of about 1500): vector work 345 us at two waves per SIMD (232-245
// registers, 60 KB of LDS), memory 1.57 GB = 330 us; the last of the 5 chunks of
// S = 68 has 4 samples.  Reading sources a row ahead was worth 644 -> 569 us.
// Grid (tiles * ceil(S / 16), ceil(nrhs / per)); level >= 3.
__global__ void __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(2)))
k_down_h16(const zf* __restrict__ agm, zf* __restrict__ agl, long st, const zf* __restrict__ trans, int lev, int S,
           const zf* __restrict__ par, long ps, int Sp, const v8h* __restrict__ tab, const int* __restrict__ s0v,
           int KB, int ec, int nrhs, int per, const int* __restrict__ act) {
  constexpr int NB = kDownSB * kDownSB;  // staged boxes, 9 per thread
  __shared__ zf src[2][NB * kDownKC];
  __shared__ v8h win[2][kDownFrag];
  __shared__ int ex[2][16];
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, lk = lane >> 4;
  // active right-hand sides of the group, as bits
  const int rg = blockIdx.y * per;
  unsigned live = 0;
  for (int q = 0; q < per && rg + q < nrhs; q++) live |= (rhs_off(act, rg + q) ? 0u : 1u) << q;
  live = __builtin_amdgcn_readfirstlane(live);
  if (!live) return;
  auto next = [&]() {
    const int q = __builtin_ctz(live);
    live &= live - 1;
    return rg + q;
  };
  int r = next();
  const int nb = 1 << lev, nchunk = (S + kDownKC - 1) / kDownKC;
  const int lb = xcd_block(), tile = lb / nchunk, chunk = lb - tile * nchunk;
  const int k0 = chunk * kDownKC;
  const unsigned m0 = (unsigned)tile * kDownTS * kDownTS;
  const int X0 = (int)compact2(m0), Y0 = (int)compact2(m0 >> 1);
  // ---- once per workgroup
  const int ks = min(k0 + (tid & 15), S - 1);  // (samples past S are computed and not stored)
  unsigned soff[9];  // byte offsets; past the end (zeros) for boxes outside the grid
#pragma unroll
  for (int u = 0; u < 9; u++) {
    const int b = (tid >> 4) + 16 * u, bx = X0 - 2 + b % kDownSB, by = Y0 - 2 + b / kDownSB;
    const bool ok = bx >= 0 && by >= 0 && bx < nb && by < nb;
    soff[u] = ok ? (morton2(bx, by) * S + ks) * (unsigned)sizeof(zf) : 0xffffff00u;
  }
  const int wp = tid >> 4, wg = tid & 15;  // window: parent, group of 8 slots
  unsigned woff[8];
  {
    const int s0 = s0v[chunk];
#pragma unroll
    for (int e = 0; e < 8; e++) {
      int j = s0 + min(8 * min(wg, kDownG - 1) + e, KB - 1);  // (slots past KB: a valid value, zero in the table)
      if (j >= Sp) j -= Sp;
      woff[e] = (((m0 >> 2) + wp) * Sp + j) * (unsigned)sizeof(zf);
    }
  }
  v8h b[3][4];
#pragma unroll
  for (int c = 0; c < 3; c++)
#pragma unroll
    for (int P = 0; P < 4; P++) b[c][P] = tab[(((long)(chunk * 4 + w) * 4 + P) * kDownG + 4 * c + lk) * 16 + li];
  zf t[kDownFar];
  const int kt = min(k0 + li, S - 1);
  switch (w) {
    case 0: down_load_t<0, 0>(trans, S, kt, t); break;
    case 1: down_load_t<1, 0>(trans, S, kt, t); break;
    case 2: down_load_t<0, 1>(trans, S, kt, t); break;
    default: down_load_t<1, 1>(trans, S, kt, t); break;
  }
  zf sv[9], wv[8];
  const unsigned mbytes = (unsigned)nb * nb * S * (unsigned)sizeof(zf), pbytes = (unsigned)nb * nb / 4 * Sp * (unsigned)sizeof(zf);
  auto load = [&](int q) {
    // one level of one right-hand side is below 4 GiB (host check): 32-bit offsets, no address arithmetic
    const __amdgpu_buffer_rsrc_t a = down_rsrc(agm + (long)q * st, mbytes), p = down_rsrc(par + (long)q * ps, pbytes);
#pragma unroll
    for (int u = 0; u < 9; u++) sv[u] = down_load(a, soff[u]);
#pragma unroll
    for (int e = 0; e < 8; e++) wv[e] = down_load(p, woff[e]);
  };
  load(r);
  const unsigned ooff = ((m0 + 16 * lk + w) * S + k0 + li) * (unsigned)sizeof(zf), ostep = 4 * S * (unsigned)sizeof(zf);
  const bool store = k0 + li < S;
  for (int buf = 0;; buf ^= 1) {
    // ---- staging
#pragma unroll
    for (int u = 0; u < 9; u++) src[buf][tid + kBlock * u] = sv[u];
    {
      float m = 0.f;
#pragma unroll
      for (int e = 0; e < 8; e++) m = max3_abs(m, wv[e].x, wv[e].y);
      m = row_max(m);  // the 16 lanes of a parent (groups past the window hold valid values of it)
      const int es = h16_scale_exp(m);
      const float s = ldexpf(1.f, es);
      v8h ph[4];
#pragma unroll
      for (int e = 0; e < 8; e += 2)
        h16_split_pair(v2f{wv[e].x * s, wv[e + 1].x * s}, v2f{wv[e].y * s, wv[e + 1].y * s}, ph, e);
      if (wg < kDownG) {
#pragma unroll
        for (int P = 0; P < 4; P++) win[buf][(P * kDownG + wg) * 16 + (wp ^ (wg & 7))] = ph[P];
      }
      if (wg == 0) ex[buf][wp] = es;
    }
    __syncthreads();
    const bool more = live != 0;
    const int rn = more ? next() : r;
    if (more) load(rn);
    // ---- interpolation: rows = parents 4 lk + i, columns = samples; the
    // fragments of a chunk are read during the previous chunk's products, the
    // translations' first sources during the last one's
    v4f cr = v4f{0, 0, 0, 0}, cn = v4f{0, 0, 0, 0}, ci = v4f{0, 0, 0, 0};
    v8h a[2][4];
    auto frags = [&](int c) {
#pragma unroll
      for (int P = 0; P < 4; P++) a[c & 1][P] = win[buf][(P * kDownG + 4 * c + lk) * 16 + (li ^ ((4 * c + lk) & 7))];
    };
    const zf* s = src[buf] + (4 * (lk >> 1) * kDownSB + 4 * (lk & 1)) * kDownKC + li;
    zf first[8];
    frags(0);
#pragma unroll
    for (int c = 0; c < 3; c++) {
      if (c < 2) {
        frags(c + 1);
      } else {
#pragma unroll
        for (int x = 0; x < 8; x++) first[x] = s[x * kDownKC];
      }
      __builtin_amdgcn_sched_barrier(0);
      const v8h(&f)[4] = a[c & 1];
      cr = __builtin_amdgcn_mfma_f32_16x16x32_f16(f[0], b[c][0], cr, 0, 0, 0);
      ci = __builtin_amdgcn_mfma_f32_16x16x32_f16(f[0], b[c][2], ci, 0, 0, 0);
      cn = __builtin_amdgcn_mfma_f32_16x16x32_f16(f[2], b[c][2], cn, 0, 0, 0);
      cr = __builtin_amdgcn_mfma_f32_16x16x32_f16(f[0], b[c][1], cr, 0, 0, 0);
      ci = __builtin_amdgcn_mfma_f32_16x16x32_f16(f[0], b[c][3], ci, 0, 0, 0);
      cn = __builtin_amdgcn_mfma_f32_16x16x32_f16(f[2], b[c][3], cn, 0, 0, 0);
      cr = __builtin_amdgcn_mfma_f32_16x16x32_f16(f[1], b[c][0], cr, 0, 0, 0);
      ci = __builtin_amdgcn_mfma_f32_16x16x32_f16(f[1], b[c][2], ci, 0, 0, 0);
      cn = __builtin_amdgcn_mfma_f32_16x16x32_f16(f[3], b[c][2], cn, 0, 0, 0);
      ci = __builtin_amdgcn_mfma_f32_16x16x32_f16(f[2], b[c][0], ci, 0, 0, 0);
      ci = __builtin_amdgcn_mfma_f32_16x16x32_f16(f[2], b[c][1], ci, 0, 0, 0);
      ci = __builtin_amdgcn_mfma_f32_16x16x32_f16(f[3], b[c][0], ci, 0, 0, 0);
    }
    // ---- translations
    zf acc[4];
#pragma unroll
    for (int i = 0; i < 4; i++) acc[i] = mkc<float>(0.f, 0.f);
    switch (w) {
      case 0: down_m2l<0, 0, 8>(s, t, first, acc); break;
      case 1: down_m2l<1, 0, 8>(s, t, first, acc); break;
      case 2: down_m2l<0, 1, 8>(s, t, first, acc); break;
      default: down_m2l<1, 1, 8>(s, t, first, acc); break;
    }
    if (store) {
      char* o = reinterpret_cast<char*>(agl + (long)r * st);
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int n = -(ex[buf][4 * lk + i] + ec);
        *reinterpret_cast<zf*>(o + (ooff + i * ostep)) =
            mkc<float>(acc[i].x + ldexpf(cr[i] - cn[i], n), acc[i].y + ldexpf(ci[i], n));
      }
    }
    if (!more) break;
    r = rn;
  }
}

// ---------------------------------------------------------------------------
// The same downward step in FP64: interpolation on v_mfma_f64_16x16x4 with the
// real band block and the parents shifted as they are read (a complex table
// would take half as many matrix products again, and FP64 products share the
// vector ALUs' time).  Per workgroup the band block, the child shifts and, in
// registers, the 27 operators are loaded once; per right-hand side the source
// boxes and the parents' windows go to LDS.  Wave w owns child position w; the
// rows of the matrix product are permuted so that a lane (li, lk) receives
// parents 4 lk .. +3, a 2 x 2 block, as in k_down_h16.  FAR = false: the
// interpolation alone (the transposed receiver product has no translations;
// levels 3 .. 6 at 512 px x 16, 149 us as band and chunked kernels, 100 here).
// FP64 work bounds it (an FP64 product of this chip's vector or matrix units
// either way): 1024 px x 64 right-hand sides, M2L and L2L of levels 2 .. 7, 3140
// us as separate kernels (M2L 1100, L2L 2040), 1890 here, of which about 1000 is
// arithmetic at the rate of a large matrix product; 512 px x 16, 195 -> 150 us.
// Grid (tiles * ceil(S / 16), ceil(nrhs / per)); level >= 3; KB <= kDownK.
template <bool FAR>
__global__ void __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(2)))
k_down64(const zd* __restrict__ agm, zd* __restrict__ agl, long st, const zd* __restrict__ trans, int lev, int S,
         const zd* __restrict__ par, long ps, int Sp, const double* __restrict__ AB, const int* __restrict__ s0v, int KB,
         const zd* __restrict__ shift, int nrhs, int per, const int* __restrict__ act) {
  typedef Mfma<double>::v4 v4;
  constexpr int NS = FAR ? kDownSB * kDownSB * kDownKC : 1, NW = 16 * kDownK / kBlock, WP = kDownK + 1;
  __shared__ zd src[NS], win[16 * WP], sh[4 * kDownK];  // win[parent][window]
  __shared__ double ab[kDownK * 16];
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, lk = lane >> 4;
  // active right-hand sides of the group, as bits
  const int rg = blockIdx.y * per;
  unsigned live = 0;
  for (int q = 0; q < per && rg + q < nrhs; q++) live |= (rhs_off(act, rg + q) ? 0u : 1u) << q;
  live = __builtin_amdgcn_readfirstlane(live);
  if (!live) return;
  const int nb = 1 << lev, nchunk = (S + kDownKC - 1) / kDownKC;
  const int lb = xcd_block(), tile = lb / nchunk, chunk = lb - tile * nchunk;
  const int k0 = chunk * kDownKC;
  const unsigned m0 = (unsigned)tile * kDownTS * kDownTS;
  const int X0 = (int)compact2(m0), Y0 = (int)compact2(m0 >> 1);
  // ---- once per workgroup
  const int ks = min(k0 + (tid & 15), S - 1);  // (samples past S are computed and not stored)
  unsigned soff[9];  // byte offsets; past the end (zeros) for boxes outside the grid
#pragma unroll
  for (int u = 0; FAR && u < 9; u++) {
    const int b = (tid >> 4) + 16 * u, bx = X0 - 2 + b % kDownSB, by = Y0 - 2 + b / kDownSB;
    const bool ok = bx >= 0 && by >= 0 && bx < nb && by < nb;
    soff[u] = ok ? (morton2(bx, by) * S + ks) * (unsigned)sizeof(zd) : 0xffffff00u;
  }
  const int s0 = s0v[chunk];
  unsigned woff[NW], wdst[NW];  // window element e = p KB + jj of parent p
#pragma unroll
  for (int u = 0; u < NW; u++) {
    const int e = min(tid + kBlock * u, 16 * KB - 1), p = e / KB, jj = e - p * KB;
    int j = s0 + jj;
    if (j >= Sp) j -= Sp;
    woff[u] = (((m0 >> 2) + p) * Sp + j) * (unsigned)sizeof(zd);
    wdst[u] = p * WP + jj;
  }
  const unsigned mbytes = (unsigned)nb * nb * S * (unsigned)sizeof(zd), pbytes = (unsigned)nb * nb / 4 * Sp * (unsigned)sizeof(zd);
  zd wv[NW];
  auto load_window = [&](int r) {
    const __amdgpu_buffer_rsrc_t p = down_rsrc(par + (long)r * ps, pbytes);
#pragma unroll
    for (int u = 0; u < NW; u++)
      wv[u] = __builtin_bit_cast(zd, __builtin_amdgcn_raw_buffer_load_b128(p, (int)woff[u], 0, 0));
  };
  int r = rg + __builtin_ctz(live);
  load_window(r);
  // (the tables' loads are all issued before the first is stored: as loops of load
  // and store they were six waits in a row, half of a small level's time)
  constexpr int NA = 16 * kDownK / kBlock, NH = (4 * kDownK + kBlock - 1) / kBlock;
  double av[NA];
  zd hv[NH];
#pragma unroll
  for (int u = 0; u < NH; u++) {
    const int e = min(tid + kBlock * u, 4 * KB - 1), c = e / KB;
    int j = s0 + e - c * KB;
    if (j >= Sp) j -= Sp;
    hv[u] = shift[c * Sp + j];
  }
#pragma unroll
  for (int u = 0; u < NA; u++) av[u] = AB[(long)chunk * KB * 16 + min(tid + kBlock * u, 16 * KB - 1)];
  zd t[kDownFar];
  if constexpr (FAR) {
    const int kt = min(k0 + li, S - 1);
    switch (w) {
      case 0: down_load_t<0, 0>(trans, S, kt, t); break;
      case 1: down_load_t<1, 0>(trans, S, kt, t); break;
      case 2: down_load_t<0, 1>(trans, S, kt, t); break;
      default: down_load_t<1, 1>(trans, S, kt, t); break;
    }
  }
#pragma unroll
  for (int u = 0; u < NH; u++) sh[min(tid + kBlock * u, 4 * KB - 1)] = hv[u];
#pragma unroll
  for (int u = 0; u < NA; u++) ab[min(tid + kBlock * u, 16 * KB - 1)] = av[u];
  const unsigned ooff = ((m0 + 16 * lk + w) * S + k0 + li) * (unsigned)sizeof(zd), ostep = 4 * S * (unsigned)sizeof(zd);
  const bool store = k0 + li < S;
  const zd* wrow = win + (4 * (li & 3) + (li >> 2)) * WP + lk;  // this lane's row of the product
  const zd* srow = sh + w * KB + lk;
  const double* arow = ab + lk * 16 + li;
  const int nkq = KB >> 2;
  // The sources of a right-hand side and the next one's windows are in flight
  // during the interpolation.
#pragma unroll
  for (int u = 0; u < NW; u++) win[wdst[u]] = wv[u];  // (the clamped last ones repeat one element)
  __syncthreads();
  for (;;) {
    live &= live - 1;
    const bool more = live != 0;
    const int rn = more ? rg + __builtin_ctz(live) : r;
    zd sv[9];
    if constexpr (FAR) {
      const __amdgpu_buffer_rsrc_t a = down_rsrc(agm + (long)r * st, mbytes);
#pragma unroll
      for (int u = 0; u < 9; u++)
        sv[u] = __builtin_bit_cast(zd, __builtin_amdgcn_raw_buffer_load_b128(a, (int)soff[u], 0, 0));
    }
    if (more) load_window(rn);
    // ---- interpolation: rows = parents, columns = samples
    v4 cr = v4{0, 0, 0, 0}, ci = v4{0, 0, 0, 0};
#pragma unroll 4
    for (int q = 0; q < nkq; q++) {
      const zd v = cmul(srow[4 * q], wrow[4 * q]);
      const double a = arow[64 * q];
      cr = Mfma<double>::mac(v.x, a, cr);
      ci = Mfma<double>::mac(v.y, a, ci);
    }
    if (FAR || more) __syncthreads();  // windows and the previous right-hand side's sources are no longer read
    if constexpr (FAR) {
#pragma unroll
      for (int u = 0; u < 9; u++) src[tid + kBlock * u] = sv[u];
    }
    if (more) {
#pragma unroll
      for (int u = 0; u < NW; u++) win[wdst[u]] = wv[u];
    }
    if (FAR || more) __syncthreads();
    // ---- translations
    zd acc[4];
#pragma unroll
    for (int i = 0; i < 4; i++) acc[i] = mkc<double>(cr[i], ci[i]);
    if constexpr (FAR) {
      zd first[4];
      const zd* s = src + (4 * (lk >> 1) * kDownSB + 4 * (lk & 1)) * kDownKC + li;
#pragma unroll
      for (int x = 0; x < 4; x++) first[x] = s[x * kDownKC];
      switch (w) {
        case 0: down_m2l<0, 0, 4>(s, t, first, acc); break;
        case 1: down_m2l<1, 0, 4>(s, t, first, acc); break;
        case 2: down_m2l<0, 1, 4>(s, t, first, acc); break;
        default: down_m2l<1, 1, 4>(s, t, first, acc); break;
      }
    }
    if (store) {
      char* o = reinterpret_cast<char*>(agl + (long)r * st);
#pragma unroll
      for (int i = 0; i < 4; i++) *reinterpret_cast<zd*>(o + (ooff + i * ostep)) = acc[i];
    }
    if (!more) break;
    r = rn;
  }
}

}  // namespace isg
