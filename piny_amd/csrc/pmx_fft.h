// The 3-D FFT of the PME grids in LDS with the fold of the spread's halo
// boxes and the influence-function convolution (internal; instantiated for
// FP32 grids by pmx_fft32.hip and for FP64 ones by pmx_fft64.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "pmx_device.h"

namespace pmx {

// Complex type of a grid scalar T (double2 for FP64, float2 for the mixed
// precision's FP32 grids).
template <typename T>
struct Cx;
template <>
struct Cx<double> {
  using C = double2;
  __device__ static C make(double x, double y) { return make_double2(x, y); }
};
template <>
struct Cx<float> {
  using C = float2;
  __device__ static C make(float x, float y) { return make_float2(x, y); }
};

// --- FFT --------------------------------------------------------------------------

// Batched 1D complex FFTs held in LDS, cooperative over the workgroup:
// mixed-radix Stockham passes (radix 2, 3, 4, 5 — the radices of FFTPACK,
// fft_generic.f:14-84 — and 8), unnormalised, sign -1 for exp(-i) (DCFFTF) and +1 for
// exp(+i) (DCFFTB).  Line l element e lives at buf[l*dist + e*stride].  A
// pass reads every butterfly's inputs into registers, waits, then writes the
// outputs in place, so no permutation pass is needed.  Lanes run along the
// contiguous direction (lines when stride > 1), which keeps LDS accesses
// free of bank conflicts.  nlines * K <= MAXP and blockDim.x == NT (the
// plane classes of launch_fft_t).
template <int R, typename T>
__device__ __forceinline__ void dft_small(typename Cx<T>::C (&v)[R], int sign) {
  using C = typename Cx<T>::C;
  if constexpr (R == 2) {
    const C a = v[0], b = v[1];
    v[0] = Cx<T>::make(a.x + b.x, a.y + b.y);
    v[1] = Cx<T>::make(a.x - b.x, a.y - b.y);
  } else if constexpr (R == 4) {
    const C a0 = Cx<T>::make(v[0].x + v[2].x, v[0].y + v[2].y);
    const C a1 = Cx<T>::make(v[0].x - v[2].x, v[0].y - v[2].y);
    const C b0 = Cx<T>::make(v[1].x + v[3].x, v[1].y + v[3].y);
    const C b1 = Cx<T>::make(v[1].x - v[3].x, v[1].y - v[3].y);
    // b1 * (sign * i)
    const C c1 = sign < 0 ? Cx<T>::make(b1.y, -b1.x) : Cx<T>::make(-b1.y, b1.x);
    v[0] = Cx<T>::make(a0.x + b0.x, a0.y + b0.y);
    v[2] = Cx<T>::make(a0.x - b0.x, a0.y - b0.y);
    v[1] = Cx<T>::make(a1.x + c1.x, a1.y + c1.y);
    v[3] = Cx<T>::make(a1.x - c1.x, a1.y - c1.y);
  } else if constexpr (R == 8) {
    // two 4-point DFTs of the even and odd inputs, combined with the
    // eighth roots w^k = exp(sign 2 pi i k / 8): X[k] = E[k] + w^k O[k],
    // X[k + 4] = E[k] - w^k O[k]
    C e[4] = {v[0], v[2], v[4], v[6]}, o[4] = {v[1], v[3], v[5], v[7]};
    dft_small<4, T>(e, sign);
    dft_small<4, T>(o, sign);
    const T h = (T)0.70710678118654752440, sg = (T)sign;
    const C w1 = Cx<T>::make(h * (o[1].x - sg * o[1].y), h * (o[1].y + sg * o[1].x));    // (1 + sign i) h
    const C w2 = Cx<T>::make(-sg * o[2].y, sg * o[2].x);                                // sign i
    const C w3 = Cx<T>::make(-h * (o[3].x + sg * o[3].y), h * (sg * o[3].x - o[3].y));  // (-1 + sign i) h
    v[0] = Cx<T>::make(e[0].x + o[0].x, e[0].y + o[0].y);
    v[4] = Cx<T>::make(e[0].x - o[0].x, e[0].y - o[0].y);
    v[1] = Cx<T>::make(e[1].x + w1.x, e[1].y + w1.y);
    v[5] = Cx<T>::make(e[1].x - w1.x, e[1].y - w1.y);
    v[2] = Cx<T>::make(e[2].x + w2.x, e[2].y + w2.y);
    v[6] = Cx<T>::make(e[2].x - w2.x, e[2].y - w2.y);
    v[3] = Cx<T>::make(e[3].x + w3.x, e[3].y + w3.y);
    v[7] = Cx<T>::make(e[3].x - w3.x, e[3].y - w3.y);
  } else if constexpr (R == 3) {
    const C t = Cx<T>::make(v[1].x + v[2].x, v[1].y + v[2].y);
    const T h = (T)0.86602540378443864676 * (T)sign;
    const C m = Cx<T>::make(v[0].x - (T)0.5 * t.x, v[0].y - (T)0.5 * t.y);
    const C d = Cx<T>::make(h * (v[1].x - v[2].x), h * (v[1].y - v[2].y));
    v[0] = Cx<T>::make(v[0].x + t.x, v[0].y + t.y);
    v[1] = Cx<T>::make(m.x - d.y, m.y + d.x);
    v[2] = Cx<T>::make(m.x + d.y, m.y - d.x);
  } else if constexpr (R == 6) {
    // two 3-point DFTs of the even and odd inputs, combined with the sixth
    // roots w^k = exp(sign 2 pi i k / 6): X[k] = E[k] + w^k O[k], X[k + 3] =
    // E[k] - w^k O[k]
    C e[3] = {v[0], v[2], v[4]}, o[3] = {v[1], v[3], v[5]};
    dft_small<3, T>(e, sign);
    dft_small<3, T>(o, sign);
    const T h = (T)0.86602540378443864676 * (T)sign;
    const C w1 = Cx<T>::make((T)0.5 * o[1].x - h * o[1].y, (T)0.5 * o[1].y + h * o[1].x);
    const C w2 = Cx<T>::make((T)-0.5 * o[2].x - h * o[2].y, (T)-0.5 * o[2].y + h * o[2].x);
    v[0] = Cx<T>::make(e[0].x + o[0].x, e[0].y + o[0].y);
    v[3] = Cx<T>::make(e[0].x - o[0].x, e[0].y - o[0].y);
    v[1] = Cx<T>::make(e[1].x + w1.x, e[1].y + w1.y);
    v[4] = Cx<T>::make(e[1].x - w1.x, e[1].y - w1.y);
    v[2] = Cx<T>::make(e[2].x + w2.x, e[2].y + w2.y);
    v[5] = Cx<T>::make(e[2].x - w2.x, e[2].y - w2.y);
  } else {
    // direct DFT: out[k] = sum_m v[m] exp(sign 2 pi i k m / R)
    constexpr double c5[5] = {1.0, 0.30901699437494742410, -0.80901699437494742410, -0.80901699437494742410,
                              0.30901699437494742410};
    constexpr double s5[5] = {0.0, 0.95105651629515357212, 0.58778525229247312917, -0.58778525229247312917,
                              -0.95105651629515357212};
    C out[R];
#pragma unroll
    for (int k = 0; k < R; k++) {
      T re = (T)0, im = (T)0;
#pragma unroll
      for (int m = 0; m < R; m++) {
        const int km = (k * m) % R;
        const T cr = (T)c5[km];
        const T ci = (T)(s5[km] * (double)sign);
        re += v[m].x * cr - v[m].y * ci;
        im += v[m].x * ci + v[m].y * cr;
      }
      out[k] = Cx<T>::make(re, im);
    }
#pragma unroll
    for (int k = 0; k < R; k++) v[k] = out[k];
  }
}

// k / d for 0 <= k, k * d < 2^32 as a multiply-high by m = floor(2^32 / d) + 1,
// m formed once per divisor (2^32 / d is at least 1/d from an integer unless
// exact, so its double quotient floors exactly); d = 1, whose m does not fit
// 32 bits, is taken apart.
struct FastDiv {
  unsigned m;
  int d;
  __device__ explicit FastDiv(int d_)
      : m(d_ > 1 ? (unsigned)(unsigned long long)(4294967296.0 / (double)d_) + 1u : 0u), d(d_) {}
  __device__ int q(int k) const { return d > 1 ? (int)__umulhi((unsigned)k, m) : k; }
};

// Division by D where it is known (a grid of a compile-time size), else by FastDiv.
template <int D>
struct IndexDiv {
  __device__ explicit IndexDiv(int) {}
  __device__ int q(int k) const { return k / D; }
};
template <>
struct IndexDiv<0> : FastDiv {
  using FastDiv::FastDiv;
};

template <int R, typename T, int NT, int MAXP>
__device__ void stockham_pass(typename Cx<T>::C *buf, int K, int nlines, int stride, int dist, int Ns, int sign,
                              const typename Cx<T>::C *__restrict__ tw) {
  using C = typename Cx<T>::C;
  constexpr int MAXB = (MAXP / R + NT - 1) / NT;
  const int tid = threadIdx.x, nt = blockDim.x;
  const int KR = K / R, nb = nlines * KR;
  const bool lines_fast = stride != 1;
  // butterfly bi -> (line l, index j): lines run fastest when stride > 1
  const FastDiv dl(lines_fast ? nlines : KR), dn(Ns);
  auto line_index = [&](int bi, int &l, int &j) {
    const int qt = dl.q(bi), rm = bi - qt * dl.d;
    l = lines_fast ? rm : qt;
    j = lines_fast ? qt : rm;
  };
  // element offsets: the k-th input of a butterfly sits k * KR * stride
  // after its first, the k-th output k * Ns * stride (uniform steps, so the
  // per-lane index work is one multiply-add per butterfly and side)
  const int kin = KR * stride, kout = Ns * stride;
  C v[MAXB][R];
  int lq[MAXB], jqv[MAXB];
#pragma unroll
  for (int q = 0; q < MAXB; q++) {
    const int bi = tid + q * nt;
    if (bi < nb) {
      int l, j;
      line_index(bi, l, j);
      lq[q] = l;
      jqv[q] = j;
      const C *p = buf + (l * dist + j * stride);
#pragma unroll
      for (int k = 0; k < R; k++) v[q][k] = p[k * kin];
    }
  }
  __syncthreads();
  const int tstep = K / (Ns * R);
#pragma unroll
  for (int q = 0; q < MAXB; q++) {
    const int bi = tid + q * nt;
    if (bi < nb) {
      const int l = lq[q], j = jqv[q];
      const int jq = dn.q(j), jm = j - jq * Ns;
      const int jt = jm * tstep;
      int ti = 0;
#pragma unroll
      for (int k = 1; k < R; k++) {  // twiddle exp(sign 2 pi i jm k / (Ns R))
        ti += jt;
        const C t = tw[ti];  // (cos, -sin) of 2 pi m / K, m = jm k tstep
        const T wr = t.x, wi = sign < 0 ? t.y : -t.y;
        const C a = v[q][k];
        v[q][k] = Cx<T>::make(a.x * wr - a.y * wi, a.x * wi + a.y * wr);
      }
      dft_small<R, T>(v[q], sign);
      C *p = buf + (l * dist + (jq * Ns * R + jm) * stride);
#pragma unroll
      for (int k = 0; k < R; k++) p[k * kout] = v[q][k];
    }
  }
  __syncthreads();
}

template <typename T, int NT, int MAXP>
__device__ void lds_fft(typename Cx<T>::C *buf, int K, int nlines, int stride, int dist, int sign,
                        const typename Cx<T>::C *tw, int npass, const int *radix) {
  int Ns = 1;
  for (int s = 0; s < npass; s++) {
    switch (radix[s]) {
      case 8:  // FP32 only (the host plans radix 8 for FP32 grids)
        if constexpr (sizeof(T) == 4) stockham_pass<8, T, NT, MAXP>(buf, K, nlines, stride, dist, Ns, sign, tw);
        break;
      case 2: stockham_pass<2, T, NT, MAXP>(buf, K, nlines, stride, dist, Ns, sign, tw); break;
      case 3: stockham_pass<3, T, NT, MAXP>(buf, K, nlines, stride, dist, Ns, sign, tw); break;
      case 4: stockham_pass<4, T, NT, MAXP>(buf, K, nlines, stride, dist, Ns, sign, tw); break;
      default: stockham_pass<5, T, NT, MAXP>(buf, K, nlines, stride, dist, Ns, sign, tw); break;
    }
    Ns *= radix[s];
  }
}

// stockham_pass with every size a compile-time constant (transform length
// K, NL lines, element stride ST, line distance DS, sub-transform length NS,
// NT lanes): the same loads, twiddles, butterflies and stores in the same
// order, with the index arithmetic folded to shifts and constants.  NS = 1
// multiplies by no twiddle (all of them are 1 there, also in stockham_pass,
// exactly).
template <int R, typename T, int NT, int K, int NL, int ST, int DS, int NS>
__device__ __forceinline__ void stockham_pass_c(typename Cx<T>::C *buf, int sign,
                                                const typename Cx<T>::C *__restrict__ tw) {
  using C = typename Cx<T>::C;
  constexpr int KR = K / R, NB = NL * KR, MAXB = (NB + NT - 1) / NT;
  constexpr bool LINES_FAST = ST != 1;
  constexpr int KIN = KR * ST, KOUT = NS * ST, TSTEP = K / (NS * R);
  const int tid = threadIdx.x;
  C v[MAXB][R];
#pragma unroll
  for (int q = 0; q < MAXB; q++) {
    const int bi = tid + q * NT;
    if (NB % NT == 0 || bi < NB) {
      const int l = LINES_FAST ? bi % NL : bi / KR, j = LINES_FAST ? bi / NL : bi % KR;
      const C *p = buf + (l * DS + j * ST);
#pragma unroll
      for (int k = 0; k < R; k++) v[q][k] = p[k * KIN];
    }
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < MAXB; q++) {
    const int bi = tid + q * NT;
    if (NB % NT == 0 || bi < NB) {
      const int l = LINES_FAST ? bi % NL : bi / KR, j = LINES_FAST ? bi / NL : bi % KR;
      const int jq = j / NS, jm = j % NS;
      if (NS > 1) {
        const int jt = jm * TSTEP;
#pragma unroll
        for (int k = 1; k < R; k++) {  // twiddle exp(sign 2 pi i jm k / (NS R))
          const C t = tw[jt * k];
          const T wr = t.x, wi = sign < 0 ? t.y : -t.y;
          const C a = v[q][k];
          v[q][k] = Cx<T>::make(a.x * wr - a.y * wi, a.x * wi + a.y * wr);
        }
      }
      dft_small<R, T>(v[q], sign);
      C *p = buf + (l * DS + (jq * NS * R + jm) * ST);
#pragma unroll
      for (int k = 0; k < R; k++) p[k * KOUT] = v[q][k];
    }
  }
  __syncthreads();
}

// Radix of the pass that follows sub-transforms of length NS in a plan of
// length K with every size a compile-time constant: 6 for the last 6 or 36,
// then 8 (FP32 grids only: in FP64 its butterflies need more than 128 VGPRs),
// 4, 6, 2, 3, 5.
constexpr int fft_radix(int K, int NS, bool f32) {
  const int rem = K / NS;
  if (rem == 6 || rem == 36) return 6;
  if (rem == 16) return 4;
  if (f32 && rem % 8 == 0) return 8;
  if (rem % 4 == 0) return 4;
  if (rem % 6 == 0) return 6;
  if (rem % 2 == 0) return 2;
  return rem % 3 == 0 ? 3 : 5;
}

// NL lines of length K, passes and their sizes unrolled at compile time.
template <typename T, int NT, int K, int NL, int ST, int DS, int NS = 1>
__device__ __forceinline__ void lds_fft_c(typename Cx<T>::C *buf, int sign, const typename Cx<T>::C *tw) {
  if constexpr (NS < K) {
    constexpr int R = fft_radix(K, NS, sizeof(T) == 4);
    stockham_pass_c<R, T, NT, K, NL, ST, DS, NS>(buf, sign, tw);
    lds_fft_c<T, NT, K, NL, ST, DS, NS * R>(buf, sign, tw);
  }
}

template <typename T>
__device__ __forceinline__ const typename Cx<T>::C *twiddles(const FftArgs &a, int d) {
  if constexpr (sizeof(T) == 8)
    return a.tw[d];
  else
    return a.twf[d];
}

// The K[d] twiddles of axis d copied into LDS at dst: the passes read them at
// lane-varying indices, which LDS serves without a vector-memory round trip.
template <typename T>
__device__ __forceinline__ void stage_twiddles(const FftArgs &a, int d, typename Cx<T>::C *dst) {
  const typename Cx<T>::C *src = twiddles<T>(a, d);
  for (int k = threadIdx.x; k < a.K[d]; k += blockDim.x) dst[k] = src[k];
}

// Plane c of bead b's spread charge into LDS as complex values, folded from
// the halo boxes: along each axis, point l of tile t is held by the box of
// tile t - o (periodically) at l + o*T for every o with l + o*T < H.  Tiles
// divide the grid, so the offset is exact also across the periodic boundary.
// With at most two boxes per axis (T >= n - 1) every point makes the same 8
// loads, the absent overlaps re-reading its own element and adding zero, so
// the loads of 4 points per lane are in flight together; smaller tiles take
// the loop over all overlaps.  Sums run in the order (c, b, a) of the boxes.
template <typename T, int KC>
__device__ __forceinline__ void fold_plane(const FftArgs &a, int c, int b, typename Cx<T>::C *sm) {
  const int Ka = KC > 0 ? KC : a.K[0], npt = Ka * (KC > 0 ? KC : a.K[1]);
  const int T0 = a.T[0], T1 = a.T[1], T2 = a.T[2];
  const int H0 = a.H[0], H1 = a.H[1], H2 = a.H[2], H01 = H0 * H1;
  const int nt0 = a.nt[0], nt1 = a.nt[1], nt2 = a.nt[2];
  const int hv = (int)a.hvol;
  const T *hb = (const T *)a.hbuf + (size_t)b * a.ntile * a.hvol;
  const int tc = c / T2, lc = c - tc * T2;
  if (a.nbr[0] <= 2 && a.nbr[1] <= 2 && a.nbr[2] <= 2) {
    const bool ec = lc + T2 < H2;
    const int rc0 = tc * nt1, rc1 = ec ? (tc ? tc - 1 : nt2 - 1) * nt1 : rc0;
    const int oc0 = lc * H01, oc1 = ec ? (lc + T2) * H01 : oc0;
    for (int w0 = threadIdx.x; w0 < npt; w0 += 4 * blockDim.x) {
      T v[4][8];
      unsigned m[4];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int w = min(w0 + u * (int)blockDim.x, npt - 1);
        const int gb = KC > 0 ? w / Ka : (int)__umulhi((unsigned)w, a.mKa), ga = w - gb * Ka;
        const int ta = (int)__umulhi((unsigned)ga, a.mT0), la = ga - ta * T0;
        const int tb = (int)__umulhi((unsigned)gb, a.mT1), lb = gb - tb * T1;
        const bool ea = la + T0 < H0, eb = lb + T1 < H1;
        const int sa1 = ea ? (ta ? ta - 1 : nt0 - 1) : ta, sb1 = eb ? (tb ? tb - 1 : nt1 - 1) : tb;
        const int xa = ea ? T0 : 0, xb = eb ? T1 * H0 : 0, e = lb * H0 + la;
        m[u] = (ea ? 1u : 0u) | (eb ? 2u : 0u);
        v[u][0] = hb[((rc0 + tb) * nt0 + ta) * hv + oc0 + e];
        v[u][1] = hb[((rc0 + tb) * nt0 + sa1) * hv + oc0 + e + xa];
        v[u][2] = hb[((rc0 + sb1) * nt0 + ta) * hv + oc0 + e + xb];
        v[u][3] = hb[((rc0 + sb1) * nt0 + sa1) * hv + oc0 + e + xa + xb];
        v[u][4] = hb[((rc1 + tb) * nt0 + ta) * hv + oc1 + e];
        v[u][5] = hb[((rc1 + tb) * nt0 + sa1) * hv + oc1 + e + xa];
        v[u][6] = hb[((rc1 + sb1) * nt0 + ta) * hv + oc1 + e + xb];
        v[u][7] = hb[((rc1 + sb1) * nt0 + sa1) * hv + oc1 + e + xa + xb];
      }
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int w = w0 + u * (int)blockDim.x;
        const bool ea = m[u] & 1u, eb = m[u] & 2u;
        T s = v[u][0];
        s += ea ? v[u][1] : (T)0;
        s += eb ? v[u][2] : (T)0;
        s += (ea && eb) ? v[u][3] : (T)0;
        s += ec ? v[u][4] : (T)0;
        s += (ec && ea) ? v[u][5] : (T)0;
        s += (ec && eb) ? v[u][6] : (T)0;
        s += (ec && ea && eb) ? v[u][7] : (T)0;
        if (w < npt) sm[w] = Cx<T>::make(s, (T)0);
      }
    }
    return;
  }
  for (int w = threadIdx.x; w < npt; w += blockDim.x) {
    const int gb = w / Ka, ga = w - gb * Ka;
    const int ta = ga / T0, la = ga - ta * T0, tb = gb / T1, lb = gb - tb * T1;
    T s = (T)0;
    for (int oc = 0; oc < a.nbr[2] && lc + oc * T2 < H2; oc++) {
      const int sc = (tc - oc % nt2 + nt2) % nt2;
      for (int ob = 0; ob < a.nbr[1] && lb + ob * T1 < H1; ob++) {
        const int sb = (tb - ob % nt1 + nt1) % nt1;
        for (int oa = 0; oa < a.nbr[0] && la + oa * T0 < H0; oa++) {
          const int sa = (ta - oa % nt0 + nt0) % nt0;
          s += hb[((sc * nt1 + sb) * nt0 + sa) * hv + (lc + oc * T2) * H01 + (lb + ob * T1) * H0 + la + oa * T0];
        }
      }
    }
    sm[w] = Cx<T>::make(s, (T)0);
  }
}

// forward transform of one c-plane of one bead: the folded charge plane,
// real along a, then b.  LDS holds the plane as Kb lines of Ka complex
// values; only a' = 0..Ka/2 is kept (Hermitian half).  spec layout:
// [bead][c][b][a'] complex.
template <typename T, int NT, int MAXP, int KC>
__global__ void __launch_bounds__(NT) k_fft_fwd_ab(FftArgs a) {
  using C = typename Cx<T>::C;
  extern __shared__ __align__(16) unsigned char lds_raw[];
  C *sm = (C *)lds_raw;
  int c, b;
  xcd_unit_bead(a.K[2], a.P, c, b);
  const int Ka = KC > 0 ? KC : a.K[0], Kb = KC > 0 ? KC : a.K[1], Ha = Ka / 2 + 1;
  C *twa = sm + Ka * Kb, *twb = twa + Ka;  // twiddles after the plane
  stage_twiddles<T>(a, 0, twa);
  stage_twiddles<T>(a, 1, twb);
  fold_plane<T, KC>(a, c, b, sm);
  __syncthreads();
  if constexpr (KC > 0) {
    lds_fft_c<T, NT, KC, KC, 1, KC>(sm, -1, twa);
    lds_fft_c<T, NT, KC, KC / 2 + 1, KC, 1>(sm, -1, twb);
  } else {
    lds_fft<T, NT, MAXP>(sm, Ka, Kb, 1, Ka, -1, twa, a.npass[0], a.radix[0]);
    lds_fft<T, NT, MAXP>(sm, Kb, Ha, Ka, 1, -1, twb, a.npass[1], a.radix[1]);
  }
  C *sp = (C *)a.spec + (size_t)b * a.sstride + (size_t)c * Kb * Ha;
  const IndexDiv<(KC > 0 ? KC / 2 + 1 : 0)> dh(Ha);
  for (int w = threadIdx.x; w < Kb * Ha; w += blockDim.x) {
    const int bb = dh.q(w), aa = w - bb * Ha;
    sp[w] = sm[bb * Ka + aa];
  }
}

// along c for one (bead, b) row: forward FFT, influence function over the
// half-space sphere list (ewald3d_pme.c:367-430): energy, virial, and the
// product with preg*bweight, then the inverse FFT.  Energy and virial are
// summed in FP64 into one partial row per (b row, bead).
template <typename T, int NT, int MAXP, int KC>
__global__ void __launch_bounds__(NT) k_fft_c_conv(FftArgs a) {
  using C = typename Cx<T>::C;
  extern __shared__ __align__(16) unsigned char lds_raw[];
  C *sm = (C *)lds_raw;
  int bb, b;
  xcd_unit_bead(a.K[1], a.P, bb, b);
  const int Ka = KC > 0 ? KC : a.K[0], Kb = KC > 0 ? KC : a.K[1], Kc = KC > 0 ? KC : a.K[2], Ha = Ka / 2 + 1;
  C *twc = sm + Kc * Ha;  // twiddles after the lines
  stage_twiddles<T>(a, 2, twc);
  C *sp = (C *)a.spec + (size_t)b * a.sstride;
  const IndexDiv<(KC > 0 ? KC / 2 + 1 : 0)> dh(Ha);
  for (int w0 = threadIdx.x; w0 < Kc * Ha; w0 += 8 * blockDim.x) {
    C v[8];
#pragma unroll
    for (int u = 0; u < 8; u++) {
      const int w = w0 + u * blockDim.x;
      const int cc = dh.q(w);
      // a select, not a conditional store: the latter put v on the stack in FP64
      v[u] = w < Kc * Ha ? sp[((size_t)cc * Kb + bb) * Ha + (w - cc * Ha)] : Cx<T>::make((T)0, (T)0);
    }
#pragma unroll
    for (int u = 0; u < 8; u++) {
      const int w = w0 + u * blockDim.x;
      if (w < Kc * Ha) sm[w] = v[u];
    }
  }
  __syncthreads();
  if constexpr (KC > 0) lds_fft_c<T, NT, KC, KC / 2 + 1, KC / 2 + 1, 1>(sm, -1, twc);
  else lds_fft<T, NT, MAXP>(sm, Kc, Ha, Ha, 1, -1, twc, a.npass[2], a.radix[2]);
  const double *hi = a.cell.hi;
  const double tpi = 2.0 * M_PI, falp2 = a.falp2;
  const int kb = bb <= Kb / 2 ? bb : bb - Kb;
  double e = 0.0, v11 = 0.0, v22 = 0.0, v33 = 0.0, v12 = 0.0, v13 = 0.0, v23 = 0.0;
  for (int w = threadIdx.x; w < Kc * Ha; w += blockDim.x) {
    const int cc = dh.q(w), aa = w - cc * Ha;
    const double W = a.infl[((size_t)cc * Kb + bb) * Ha + aa];
    const C s = sm[w];
    if (W != 0.0) {
      const int kc = cc <= Kc / 2 ? cc : cc - Kc;
      const double ga = tpi * (double)aa, gb = tpi * (double)kb, gc = tpi * (double)kc;
      const double xk = (ga * hi[0] + gb * hi[1] + gc * hi[2]);
      const double yk = (ga * hi[3] + gb * hi[4] + gc * hi[5]);
      const double zk = (ga * hi[6] + gb * hi[7] + gc * hi[8]);
      const double g2 = xk * xk + yk * yk + zk * zk;
      const double wsum = (aa == 0) ? 0.5 : 1.0;  // a' = 0 holds both +k and -k
      const double sx = (double)s.x, sy = (double)s.y;
      const double sm2 = (sx * sx + sy * sy) * wsum;
      e += W * sm2;
      const double prep = -2.0 * W * ((g2 / falp2) + 1.0) / g2 * sm2;
      v11 += prep * xk * xk;
      v22 += prep * yk * yk;
      v33 += prep * zk * zk;
      v12 += prep * xk * yk;
      v13 += prep * xk * zk;
      v23 += prep * yk * zk;
    }
    sm[w] = Cx<T>::make((T)(s.x * W), (T)(s.y * W));
  }
  {
    // the k-space pressure also carries the energy on its diagonal
    // (ewald3d_pme.c:412-414); reduced before the inverse transform so the
    // sums are not held in registers through it
    const double vals[FFT_NV] = {e, v11 + e, v22 + e, v33 + e, v12, v13, v23};
    block_partials<FFT_NV>(vals, 1, b, a.P, a.part, bb, a.K[1]);
  }
  __syncthreads();
  if constexpr (KC > 0) lds_fft_c<T, NT, KC, KC / 2 + 1, KC / 2 + 1, 1>(sm, +1, twc);
  else lds_fft<T, NT, MAXP>(sm, Kc, Ha, Ha, 1, +1, twc, a.npass[2], a.radix[2]);
  for (int w = threadIdx.x; w < Kc * Ha; w += blockDim.x) {
    const int cc = dh.q(w), aa = w - cc * Ha;
    sp[((size_t)cc * Kb + bb) * Ha + aa] = sm[w];
  }
}

// inverse transform of one c-plane: along b, then complex-to-real along a.
template <typename T, int NT, int MAXP, int KC>
__global__ void __launch_bounds__(NT) k_fft_inv_ba(FftArgs a) {
  using C = typename Cx<T>::C;
  extern __shared__ __align__(16) unsigned char lds_raw[];
  C *sm = (C *)lds_raw;
  int c, b;
  xcd_unit_bead(a.K[2], a.P, c, b);
  const int Ka = KC > 0 ? KC : a.K[0], Kb = KC > 0 ? KC : a.K[1], Ha = Ka / 2 + 1;
  C *twa = sm + Ka * Kb, *twb = twa + Ka;  // twiddles after the plane
  stage_twiddles<T>(a, 0, twa);
  stage_twiddles<T>(a, 1, twb);
  const C *sp = (const C *)a.spec + (size_t)b * a.sstride + (size_t)c * Kb * Ha;
  const IndexDiv<KC> dka(Ka);
  for (int w0 = threadIdx.x; w0 < Kb * Ka; w0 += 8 * blockDim.x) {
    C v[8];
#pragma unroll
    for (int u = 0; u < 8; u++) {
      const int w = w0 + u * blockDim.x;
      const int bb = dka.q(w), aa = w - bb * Ka;
      v[u] = (w < Kb * Ka && aa < Ha) ? sp[bb * Ha + aa] : Cx<T>::make((T)0, (T)0);
    }
#pragma unroll
    for (int u = 0; u < 8; u++) {
      const int w = w0 + u * blockDim.x;
      if (w < Kb * Ka) sm[w] = v[u];
    }
  }
  __syncthreads();
  if constexpr (KC > 0) lds_fft_c<T, NT, KC, KC / 2 + 1, KC, 1>(sm, +1, twb);
  else lds_fft<T, NT, MAXP>(sm, Kb, Ha, Ka, 1, +1, twb, a.npass[1], a.radix[1]);
  // Hermitian completion along a: X[Ka - a'] = conj(X[a'])
  for (int w = threadIdx.x; w < Kb * Ka; w += blockDim.x) {
    const int bb = dka.q(w), aa = w - bb * Ka;
    if (aa >= Ha) {
      const C v = sm[bb * Ka + (Ka - aa)];
      sm[w] = Cx<T>::make(v.x, -v.y);
    }
  }
  __syncthreads();
  if constexpr (KC > 0) lds_fft_c<T, NT, KC, KC, 1, KC>(sm, +1, twa);
  else lds_fft<T, NT, MAXP>(sm, Ka, Kb, 1, Ka, +1, twa, a.npass[0], a.radix[0]);
  T *g = (T *)a.grid + (size_t)b * a.gstride + (size_t)c * Ka * Kb;
  for (int w = threadIdx.x; w < Ka * Kb; w += blockDim.x) g[w] = sm[w].x;
}

template <typename T, int NT, int NTC, int MAXP, int KC>
hipError_t launch_fft_class(const FftArgs &f, hipStream_t st) {
  using C = typename Cx<T>::C;
  const int Ka = f.K[0], Kb = f.K[1], Kc = f.K[2], Ha = Ka / 2 + 1;
  // the plane (or the lines) and the twiddles of the axes it transforms
  const size_t lab = ((size_t)Ka * Kb + Ka + Kb) * sizeof(C), lch = ((size_t)Kc * Ha + Kc) * sizeof(C);
  if (lab > FFT_LDS_DYN || lch > FFT_LDS_DYN) return hipErrorInvalidValue;  // refused at setup already
  if (lab > 65536 || lch > 65536) {  // beyond 64 KB the kernels ask for the larger LDS
    hipError_t e;
    if ((e = hipFuncSetAttribute((const void *)k_fft_fwd_ab<T, NT, MAXP, KC>,
                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lab)) != hipSuccess)
      return e;
    if ((e = hipFuncSetAttribute((const void *)k_fft_c_conv<T, NTC, MAXP, KC>,
                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lch)) != hipSuccess)
      return e;
    if ((e = hipFuncSetAttribute((const void *)k_fft_inv_ba<T, NT, MAXP, KC>,
                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lab)) != hipSuccess)
      return e;
  }
  hipLaunchKernelGGL(HIP_KERNEL_NAME(k_fft_fwd_ab<T, NT, MAXP, KC>), dim3(xcd_grid(Kc, f.P)), dim3(NT), lab, st, f);
  hipLaunchKernelGGL(HIP_KERNEL_NAME(k_fft_c_conv<T, NTC, MAXP, KC>), dim3(xcd_grid(Kb, f.P)), dim3(NTC), lch, st, f);
  hipLaunchKernelGGL(HIP_KERNEL_NAME(k_fft_inv_ba<T, NT, MAXP, KC>), dim3(xcd_grid(Kc, f.P)), dim3(NT), lab, st, f);
  return hipGetLastError();
}

// Cubic grids of the sizes PINY's radix table gives up to 96 points take
// kernels built for the size: passes, strides and index divisions fold to
// constants, radix 6 saves a pass where 6 or 36 is left (48 = 8 x 6), and the
// lanes of a workgroup are what its passes' butterflies divide into with the
// fewest idle (planes: NT, lines along c: NTC), with room for several
// workgroups' LDS on a CU.  The run-time form rounds its lanes up to a plane
// class and keeps registers for the class's largest plane: at 72 points one
// workgroup of 1024 lanes a CU, with 20 % of its butterfly slots in use.  The
// three kernels, run-time form -> this: 48^3 x 32 beads FP32 99 -> 56 us, FP64
// 128 -> 83; 72^3 x 16 beads FP32 260 -> 101; 48^3, one bead, FP64 45 -> 32;
// 12^3 24 -> 14.
template <typename T>
hipError_t launch_fft_cubic(const FftArgs &f, hipStream_t st) {
  constexpr bool F = sizeof(T) == 4;
  switch (f.K[0]) {
    case 12: return launch_fft_class<T, 64, 64, 0, 12>(f, st);
    case 16: return launch_fft_class<T, 64, 64, 0, 16>(f, st);
    case 20: return launch_fft_class<T, 128, 64, 0, 20>(f, st);
    case 24: return launch_fft_class<T, 192, 128, 0, 24>(f, st);
    case 32: return launch_fft_class<T, F ? 128 : 256, 192, 0, 32>(f, st);
    case 36: return launch_fft_class<T, 256, 128, 0, 36>(f, st);
    case 40: return launch_fft_class<T, F ? 192 : 448, 192, 0, 40>(f, st);
    case 48: return launch_fft_class<T, F ? 192 : 256, F ? 256 : 320, 0, 48>(f, st);
    case 60: return launch_fft_class<T, F ? 256 : 512, 320, 0, 60>(f, st);
    case 64: return launch_fft_class<T, F ? 256 : 512, F ? 320 : 576, 0, 64>(f, st);
    case 72: return launch_fft_class<T, F ? 384 : 896, 448, 0, 72>(f, st);
    case 80: return launch_fft_class<T, F ? 320 : 832, 448, 0, 80>(f, st);
    case 96: return launch_fft_class<T, F ? 384 : 768, 640, 0, 96>(f, st);
    default: return hipErrorNotSupported;
  }
}

// Other grids: two plane classes, planes of up to FFT_MAX_PLANE points with
// 256 lanes, larger ones (up to FFT_LDS_MAX bytes, the LDS a workgroup may
// hold on MI355X) with 1024 lanes, so the registers that stage a Stockham
// pass stay few in both.
template <typename T>
hipError_t launch_fft_t(const FftArgs &f, hipStream_t st) {
  using C = typename Cx<T>::C;
  const int Ka = f.K[0], Kb = f.K[1], Kc = f.K[2], Ha = Ka / 2 + 1;
  if (Ka == Kb && Kb == Kc) {
    const hipError_t e = launch_fft_cubic<T>(f, st);
    if (e != hipErrorNotSupported) return e;
  }
  if ((size_t)Ka * Kb <= FFT_MAX_PLANE && (size_t)Kc * Ha <= FFT_MAX_PLANE)
    return launch_fft_class<T, 256, 256, FFT_MAX_PLANE, 0>(f, st);
  return launch_fft_class<T, 1024, 1024, (int)(FFT_LDS_MAX / sizeof(C)), 0>(f, st);
}

}  // namespace pmx
