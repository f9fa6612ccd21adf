// Particle-mesh Ewald on gfx950: charge binning, tiled spread and gather,
// and the 3-D FFT with the influence-function convolution.
//
// Arithmetic restates ewald3d_pme.c (PINY): fractional coordinates and
// B-spline weights (:241-337), charge stuffing (:342-356), the k-space sum
// over the half-space sphere list (:367-430) and the force gather (:500-560).
// The MI355X layout differs from the reference's loop order:
//  - every (charge, bead) is binned by the grid tile holding the first point
//    of its support, and within the tile by that point's plane (a counting
//    sort: k_pme_count, k_pme_scan, k_pme_place, or k_pme_sort alone);
//  - the spread is a contraction: per plane of a tile, outer products of the
//    charges' weights along a and b, summed on the FP64 matrix cores into a
//    16 x 16 patch held in registers (k_pme_spread_mm), written out once (no
//    atomics, no grid clear).  Orders above 8, and grids without a fitting
//    tile, take LDS atomics into a halo box instead (k_pme_spread);
//  - the forward FFT sums, as it loads each grid plane, every point's own
//    box and the overhang of the boxes below it (the fold into the periodic
//    grid never goes through memory);
//  - the gather loads the tile's halo box of (T + n - 1)^3 potential values
//    into LDS and each lane reduces one charge's n^3 products in registers.
#include <hip/hip_runtime.h>

#include "pmx_device.h"

namespace pmx {

namespace {

constexpr int PME_BLOCK = 128;  // lanes per (tile, bead) workgroup: about one per charge
// lanes per charge in the spread (measured: with FP32 weights 90, 80 and 74
// us for 1, 2 and 4 lanes; with FP64 weights, whose registers allow fewer
// wavefronts, more lanes did not help)
template <typename T>
constexpr int spread_lanes() {
  return sizeof(T) == 4 ? 4 : 1;
}

// B-spline weights M_n(frac + j - 1), j = 1..NI, by the recursion of
// ewald3d_pme.c:296-337; dmn (order NI-1 differences, :516-530) if DERIV.
template <int NI, bool DERIV, typename T>
__device__ __forceinline__ void bspline(T frac, T (&mn)[NI + 1], T (&dmn)[NI + 1]) {
  T u[NI + 1];
#pragma unroll
  for (int j = 1; j <= NI; j++) u[j] = frac + (T)(j - 1);
  mn[1] = (T)1 - fabs(u[1] - (T)1);
  mn[2] = (T)1 - fabs(u[2] - (T)1);
#pragma unroll
  for (int j = 3; j <= NI; j++) mn[j] = (T)0;
#pragma unroll
  for (int o = 3; o <= NI; o++) {
    const T rn = (T)o, rn1 = (T)1 / ((T)(o - 1));
#pragma unroll
    for (int j = o; j >= 2; j--) mn[j] = (u[j] * mn[j] + (rn - u[j]) * mn[j - 1]) * rn1;
    mn[1] = u[1] * mn[1] * rn1;
    if (DERIV && o == NI - 1) {
      dmn[1] = mn[1];
#pragma unroll
      for (int j = 2; j <= NI; j++) dmn[j] = mn[j] - mn[j - 1];
    }
  }
}

__device__ __forceinline__ void tile_origin(const PmeArgs &a, int tl, int &o0, int &o1, int &o2) {
  const int ta = tl % a.nt[0], tb = (tl / a.nt[0]) % a.nt[1], tc = tl / (a.nt[0] * a.nt[1]);
  o0 = ta * a.T[0];
  o1 = tb * a.T[1];
  o2 = tc * a.T[2];
}

}  // namespace

// --- binning -----------------------------------------------------------------

// a (charge, bead) item: fractional grid offset per axis and the charge
template <typename T>
struct Rec;
template <>
struct Rec<double> {
  using V = double4;
};
template <>
struct Rec<float> {
  using V = float4;
};

// Item (charge ic, bead b): the fractional grid coordinates
// (ewald3d_pme.c:241-262, 270-276), formed in FP64; the first support point
// per axis relative to its tile (below PME_TILE_MAX on a grid axis of any
// length), 10 bits each, with the charge's index; and the item's bin: its tile
// and, with zb > 1, its plane within the tile.  The fused operations are written
// out and no others formed: k_pme_count and k_pme_place form the same item, and
// both must round alike for the bin that the one counted to be the other's.
// (Without them k_pme_count takes 33 VGPRs and no longer fits beside the mixed
// pair kernel's four wavefronts of 120: 12001 SPC/Fw, P = 16, 689 -> 705 us.)
template <typename T>
__device__ __forceinline__ int pme_item(const PmeArgs &a, int ic, int b, typename Rec<T>::V &f, int2 &si) {
#pragma clang fp contract(off)
  const size_t ib = (size_t)a.ichrg[ic] * a.P + b;
  const double x = a.x[ib], y = a.y[ib], z = a.z[ib];
  const double *hi = a.cell.hi;
  double s[3], fr[3];
  s[0] = fma(z, hi[6], fma(y, hi[3], x * hi[0]));
  s[1] = fma(z, hi[7], fma(y, hi[4], x * hi[1]));
  s[2] = fma(z, hi[8], fma(y, hi[5], x * hi[2]));
  int tile[3], l[3];  // the tile along each axis, and the first support point in it
#pragma unroll
  for (int d = 0; d < 3; d++) {
    const int K = a.K[d];
    const double t = s[d] - nint_d((s[d] - 0.5));
    const double sc = t * (double)K;
    int ig = (int)(sc);
    fr[d] = fma(t, (double)K, -(double)ig);
    // support points (0-based) ig - n + 1 .. ig, periodic; ig = K (a
    // coordinate rounding onto the upper face) is the same set as ig = 0
    ig = ((ig % K) + K) % K;
    const int g = ig - a.n + 1, s0 = ((g % K) + K) % K;
    tile[d] = s0 / a.T[d];
    l[d] = s0 - tile[d] * a.T[d];
  }
  f.x = (T)fr[0];
  f.y = (T)fr[1];
  f.z = (T)fr[2];
  f.w = (T)a.q[a.ichrg[ic]];
  si = make_int2(l[0] | (l[1] << 10) | (l[2] << 20), ic);
  const int tl = (tile[2] * a.nt[1] + tile[1]) * a.nt[0] + tile[0];
  return a.zb > 1 ? tl * a.zb + l[2] : tl;
}

// The counting sort of the items by bin.  k_pme_count: one thread per (charge,
// bead) in the positions' own order; an atomic on the item's bin (some
// charges to a bin, so the addresses differ) hands out its place there.
// k_pme_scan: the bins' first places, one workgroup a bead, which leaves the
// counts zero for the next call.  k_pme_place: every item formed again and
// written to its place (its 24 bytes cost more to keep than to form).
template <typename T>
__global__ void __launch_bounds__(256) k_pme_count(PmeArgs a) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= a.nchrg * a.P) return;
  const int c = t / a.P, b = t - c * a.P;
  typename Rec<T>::V f;
  int2 si;
  const int key = pme_item<T>(a, c, b, f, si);
  a.kp[t] = make_int2(key, atomicAdd(a.cnt + (size_t)b * a.nbin + key, 1));
}

// exclusive scan over the workgroup's threads of each one's value
__device__ __forceinline__ int block_scan(int v, int *wsum) {
  const int tid = threadIdx.x, lane = tid & 63;
  int inc = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int u = __shfl_up(inc, off, 64);
    inc += lane >= off ? u : 0;
  }
  if (lane == 63) wsum[tid >> 6] = inc;
  __syncthreads();
  int run = inc - v;
  for (int w = 0; w < (tid >> 6); w++) run += wsum[w];
  return run;
}

constexpr int SCAN_PER = 4;  // bins a thread takes per round of k_pme_scan
__global__ void __launch_bounds__(1024) k_pme_scan(PmeArgs a) {
  __shared__ int wsum[16];
  __shared__ int total;
  const int b = blockIdx.x, nbin = a.nbin, tid = threadIdx.x;
  int *cnt = a.cnt + (size_t)b * nbin, *off = a.off + (size_t)b * (nbin + 1);
  int base = 0;
  for (int k0 = 0; k0 < nbin; k0 += 1024 * SCAN_PER) {
    const int k = k0 + tid * SCAN_PER;
    int v[SCAN_PER], sum = 0;
#pragma unroll
    for (int u = 0; u < SCAN_PER; u++) {
      v[u] = k + u < nbin ? cnt[k + u] : 0;
      sum += v[u];
    }
    int run = base + block_scan(sum, wsum);
    if (tid == 1023) total = run + sum;
#pragma unroll
    for (int u = 0; u < SCAN_PER; u++)
      if (k + u < nbin) {
        off[k + u] = run;
        cnt[k + u] = 0;
        run += v[u];
      }
    __syncthreads();
    base = total;
    __syncthreads();
  }
  if (tid == 0) off[nbin] = base;
}

template <typename T>
__global__ void __launch_bounds__(256) k_pme_place(PmeArgs a) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= a.nchrg * a.P) return;
  const int c = t / a.P, b = t - c * a.P;
  typename Rec<T>::V f;
  int2 si;
  (void)pme_item<T>(a, c, b, f, si);
  const int2 kp = a.kp[t];
  const size_t o = (size_t)b * a.nchrg + a.off[(size_t)b * (a.nbin + 1) + kp.x] + kp.y;
  ((typename Rec<T>::V *)a.rfs)[o] = f;
  a.ris[o] = si;
}

// The same sort of a small box (up to SORT_ITEMS charges and SORT_BINS bins) in
// one launch, one workgroup a bead: the items stay in registers, the counts
// in LDS.
constexpr int SORT_PER = 2, SORT_ITEMS = 1024 * SORT_PER, SORT_BINS = 8192;
template <typename T>
__global__ void __launch_bounds__(1024) k_pme_sort(PmeArgs a) {
  using V = typename Rec<T>::V;
  extern __shared__ int hist[];  // [nbin]
  __shared__ int wsum[16];
  const int b = blockIdx.x, tid = threadIdx.x, n = a.nchrg, nbin = a.nbin;
  for (int k = tid; k < nbin; k += 1024) hist[k] = 0;
  __syncthreads();
  V f[SORT_PER];
  int2 si[SORT_PER];
  int key[SORT_PER], pos[SORT_PER];
#pragma unroll
  for (int u = 0; u < SORT_PER; u++) {
    const int c = tid + u * 1024;
    if (c < n) {
      key[u] = pme_item<T>(a, c, b, f[u], si[u]);
      pos[u] = atomicAdd(hist + key[u], 1);
    }
  }
  __syncthreads();
  const int per = (nbin + 1023) / 1024, lo = min(nbin, tid * per), hi = min(nbin, lo + per);
  int sum = 0;
  for (int k = lo; k < hi; k++) sum += hist[k];
  int run = block_scan(sum, wsum);
  int *off = a.off + (size_t)b * (nbin + 1);
  for (int k = lo; k < hi; k++) {
    const int v = hist[k];
    hist[k] = run;
    off[k] = run;
    run += v;
  }
  if (tid == 0) off[nbin] = n;
  __syncthreads();
#pragma unroll
  for (int u = 0; u < SORT_PER; u++) {
    const int c = tid + u * 1024;
    if (c < n) {
      const size_t o = (size_t)b * n + hist[key[u]] + pos[u];
      ((V *)a.rfs)[o] = f[u];
      a.ris[o] = si[u];
    }
  }
}

template <typename T>
hipError_t launch_bin_t(const PmeArgs &a, hipStream_t st) {
  // one launch while a workgroup holds a bead's items; with more a single
  // workgroup's time shows (15009 charges, P = 1: 44 us, against 14 in three)
  if (a.nchrg <= SORT_ITEMS && a.nbin <= SORT_BINS) {
    hipLaunchKernelGGL(HIP_KERNEL_NAME(k_pme_sort<T>), dim3(a.P), dim3(1024), (size_t)a.nbin * sizeof(int), st, a);
    return hipGetLastError();
  }
  const dim3 grid((unsigned)(((size_t)a.nchrg * a.P + 255) / 256)), block(256);
  hipLaunchKernelGGL(HIP_KERNEL_NAME(k_pme_count<T>), grid, block, 0, st, a);
  hipLaunchKernelGGL(k_pme_scan, dim3(a.P), dim3(1024), 0, st, a);
  hipLaunchKernelGGL(HIP_KERNEL_NAME(k_pme_place<T>), grid, block, 0, st, a);
  return hipGetLastError();
}

hipError_t launch_pme_bin(const PmeArgs &a, hipStream_t st) {
  return a.f32 ? launch_bin_t<float>(a, st) : launch_bin_t<double>(a, st);
}

// --- spread --------------------------------------------------------------------

// the items of bead b's tile tl: [lo, hi) of the bead's sorted items
__device__ __forceinline__ void tile_items(const PmeArgs &a, int tl, int b, int &lo, int &hi) {
  const int *off = a.off + (size_t)b * (a.nbin + 1) + (size_t)tl * a.zb;
  lo = off[0];
  hi = off[a.zb];
}

// Weights of one item along the three axes: w[d][m] is the weight of support
// point s_d + m (M_n index j = n - m); l[d] is s_d relative to the tile origin.
template <int NI, bool DERIV, typename T>
__device__ __forceinline__ void item_weights(const typename Rec<T>::V &f, int s, T (&w)[3][NI], T (&dw)[3][NI],
                                             int (&l)[3]) {
  const T fr[3] = {f.x, f.y, f.z};
#pragma unroll
  for (int d = 0; d < 3; d++) {
    T mn[NI + 1], dmn[NI + 1];
    bspline<NI, DERIV, T>(fr[d], mn, dmn);
    l[d] = (s >> (10 * d)) & (PME_TILE_MAX - 1);
#pragma unroll
    for (int m = 0; m < NI; m++) {
      w[d][m] = mn[NI - m];
      if (DERIV) dw[d][m] = dmn[NI - m];
    }
  }
}

// The spread as a contraction, one wavefront per (tile, bead).  A charge adds
// q w_c[m] w_b w_a^T to planes s_c + m of its tile's halo box, so plane by
// plane four charges with the same s_c (the tile's items come sorted by it)
// are one rank-4 update of the plane's b x a patch:
// v_mfma_f64_16x16x4 with A[b][k] = q w_c[m] w_b of charge k and B[k][a] = w_a,
// zero outside the support.  The n planes that open charges reach live in
// registers, n rolling accumulators of 16 x 16 (T + n - 1 <= 16); each is
// stored, rounded to the grid type once, when its last charge has passed.
// Weights are formed for 16 charges at a time (48 lanes, one axis each) and
// read back from LDS.
//
// The LDS atomics of the form below (216 of FP64 per charge at order 6) took
// 64 us on the same tiles of 4096 q-TIP4P/F at P = 32 (a 48^3 grid) and 77 us
// on their 16 x 16 x 8 ones; the matrix cores' part here is 20 us and the
// vector instructions beside it 17: 53 us.
typedef double mm_acc __attribute__((ext_vector_type(4)));
template <int NI, typename T>
__global__ void __launch_bounds__(64) k_pme_spread_mm(PmeArgs a) {
  constexpr int NB = 16;
  __shared__ double sw[NB][3][NI];
  __shared__ int sl[NB][2];
  int tl, b;
  xcd_unit_bead(a.ntile, a.P, tl, b);
  const int lane = threadIdx.x, row = lane & 15, kq = lane >> 4;
  const int Tz = a.T[2], H0 = a.H[0], H1 = a.H[1], H01 = H0 * H1;
  const int *off = a.off + (size_t)b * (a.nbin + 1) + (size_t)tl * Tz;
  const int offl = off[min(lane, Tz)];  // lane z holds the start of plane z's items (Tz < 64)
  const int lo = __builtin_amdgcn_readlane(offl, 0), hi = __builtin_amdgcn_readlane(offl, Tz);
  const typename Rec<T>::V *rf = (const typename Rec<T>::V *)a.rfs + (size_t)b * a.nchrg;
  const int2 *ri = a.ris + (size_t)b * a.nchrg;
  T *dst = (T *)a.hbuf + ((size_t)b * a.ntile + tl) * a.hvol;
  mm_acc acc[NI];
#pragma unroll
  for (int m = 0; m < NI; m++) acc[m] = mm_acc{0.0, 0.0, 0.0, 0.0};
  // this lane's entries of a plane, as byte offsets from the plane
  unsigned po[4];
  bool in[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    in[i] = row < H0 && kq + 4 * i < H1;
    po[i] = (unsigned)((kq + 4 * i) * H0 + row) * (unsigned)sizeof(T);
  }
  int pb = lo - NB, p = lo;  // batch in LDS: items pb .. pb + NB - 1
  // the next batch's items, loaded while the current one is summed
  typename Rec<T>::V fn{};
  int sn = 0;
  auto next = [&](int from) {
    if (hi > lo) {  // uniform
      const int c = min(from + row, hi - 1);
      fn = rf[c];
      sn = ri[c].x;
    }
  };
  next(lo);
  for (int z0 = 0; z0 < Tz + NI - 1; z0 += NI) {
#pragma unroll
    for (int u = 0; u < NI; u++) {
      const int z = z0 + u;
      if (z < Tz + NI - 1) {
        const int e = z < Tz ? __builtin_amdgcn_readlane(offl, z + 1) : p;
        while (p < e) {
          if (p >= pb + NB) {
            pb = p;
            __builtin_amdgcn_wave_barrier();
            if (kq < 3) {
              T mn[NI + 1], dmn[NI + 1];
              bspline<NI, false, T>(kq == 0 ? fn.x : kq == 1 ? fn.y : fn.z, mn, dmn);
              const double q = kq == 2 ? (double)fn.w : 1.0;
#pragma unroll
              for (int m = 0; m < NI; m++) sw[row][kq][m] = (double)mn[NI - m] * q;
            } else {
              sl[row][0] = sn & (PME_TILE_MAX - 1);
              sl[row][1] = (sn >> 10) & (PME_TILE_MAX - 1);
            }
            next(pb + NB);
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
          }
          const int n = min(4, min(e, pb + NB) - p), c = min(p - pb + kq, NB - 1);
          const bool on = kq < n;
          const int ta = row - sl[c][0], tb = row - sl[c][1];
          const double wa = sw[c][0][min(max(ta, 0), NI - 1)], wb = sw[c][1][min(max(tb, 0), NI - 1)];
          const double B = on && (unsigned)ta < (unsigned)NI ? wa : 0.0;
          const bool bon = on && (unsigned)tb < (unsigned)NI;
#pragma unroll
          for (int m = 0; m < NI; m++) {
            const double A = bon ? wb * sw[c][2][m] : 0.0;
            acc[(u + m) % NI] = __builtin_amdgcn_mfma_f64_16x16x4f64(A, B, acc[(u + m) % NI], 0, 0, 0);
          }
          p += n;
        }
        // plane z is complete: lane (row, kq) holds b rows kq + 4 i of column a = row
        char *plane = (char *)(dst + z * H01);
#pragma unroll
        for (int i = 0; i < 4; i++)
          if (in[i]) *(T *)(plane + po[i]) = (T)acc[u][i];
        acc[u] = mm_acc{0.0, 0.0, 0.0, 0.0};
      }
    }
  }
}

// one workgroup per (tile, bead), one lane per charge of the bin; the
// charge's n^3 products go into the LDS halo box with LDS atomics.  The box
// accumulates in FP64 for both grid types: the weights are formed in T, and
// the FP32 path rounds the box once when it is stored (FP32 LDS atomics
// measured 5x slower than FP64 ones on MI355X for this access pattern).
template <int NI, typename T>
__global__ void __launch_bounds__(spread_lanes<T>() * PME_BLOCK) k_pme_spread(PmeArgs a) {
  extern __shared__ __align__(16) unsigned char lds_raw[];
  double *box = (double *)lds_raw;
  const int hvol = (int)a.hvol;
  int tl, b;
  xcd_unit_bead(a.ntile, a.P, tl, b);
  const int tid = threadIdx.x;
  for (int k = tid; k < hvol; k += blockDim.x) box[k] = 0.0;
  const size_t bin = (size_t)b * a.ntile + tl;
  int lo, hi;
  tile_items(a, tl, b, lo, hi);
  const typename Rec<T>::V *rf = (const typename Rec<T>::V *)a.rfs + (size_t)b * a.nchrg;
  const int2 *ri = a.ris + (size_t)b * a.nchrg;
  const int H0 = a.H[0], H01 = a.H[0] * a.H[1];
  __syncthreads();
  // L lanes per charge, each adding every L-th row (mc, mb) of the support
  // (more wavefronts in flight for the LDS atomics)
  constexpr int L = spread_lanes<T>();
  const int part = tid % L;
  for (int c = lo + tid / L; c < hi; c += blockDim.x / L) {
    const typename Rec<T>::V f = rf[c];
    const T q = f.w;
    T w[3][NI], dw[3][NI];
    int l[3];
    item_weights<NI, false, T>(f, ri[c].x, w, dw, l);
#pragma unroll
    for (int m = 0; m < NI; m++) w[0][m] *= q;
    for (int rw = part; rw < NI * NI; rw += L) {
      const int mc = rw / NI, mb = rw - mc * NI;
      const T wbc = w[1][mb] * w[2][mc];
      double *row = box + (l[2] + mc) * H01 + (l[1] + mb) * H0 + l[0];
#pragma unroll
      for (int ma = 0; ma < NI; ma++) atomicAdd(row + ma, (double)(w[0][ma] * wbc));
    }
  }
  __syncthreads();
  T *dst = (T *)a.hbuf + bin * a.hvol;
  for (int k = tid; k < hvol; k += blockDim.x) dst[k] = (T)box[k];
}

// --- gather ---------------------------------------------------------------------

// The potential on the halo box of tile origin org, bead b, into LDS, with
// batches of 8 loads in flight per lane.
template <typename T>
__device__ __forceinline__ void load_halo(const PmeArgs &a, int b, const int (&org)[3], T *box) {
  const int hvol = (int)a.hvol;
  const int Ka = a.K[0], Kb = a.K[1], Kc = a.K[2];
  const int H0 = a.H[0], H1 = a.H[1], H01 = H0 * H1;
  const T *g = (const T *)a.grid + (size_t)b * a.gstride;
  for (int k0 = threadIdx.x; k0 < hvol; k0 += 8 * blockDim.x) {
    T v[8];
#pragma unroll
    for (int u = 0; u < 8; u++) {
      const int k = k0 + u * blockDim.x;
      v[u] = (T)0;
      if (k < hvol) {
        const int q0 = (int)__umulhi((unsigned)k, a.mH0), lc = (int)__umulhi((unsigned)q0, a.mH1);
        const int la = k - q0 * H0, lb = q0 - lc * H1;
        // org < K and l < H <= K + n - 1, so org + l < 3 K (n - 1 <= K on
        // every grid): two conditional subtractions wrap it into the grid
        int ga = org[0] + la, gb = org[1] + lb, gc = org[2] + lc;
        ga -= ga >= Ka ? Ka : 0;
        gb -= gb >= Kb ? Kb : 0;
        gc -= gc >= Kc ? Kc : 0;
        ga -= ga >= Ka ? Ka : 0;
        gb -= gb >= Kb ? Kb : 0;
        gc -= gc >= Kc ? Kc : 0;
        v[u] = g[((size_t)gc * Kb + gb) * Ka + ga];
      }
    }
#pragma unroll
    for (int u = 0; u < 8; u++) {
      const int k = k0 + u * blockDim.x;
      if (k < hvol) box[k] = v[u];
    }
  }
}

// The same box by rows of 16 points, V of them a lane (8 or 16 bytes), for
// tiles whose first point is V-aligned in the grid (T[0] a multiple of V, so
// the grid's rows are too) and whose rows are at most 16 wide: the lane's
// column, its wrap included, is fixed, and only the row is divided into (b, c)
// and wrapped.  One point a lane took some 22 instructions each, half of the
// gather's.  The points past the row's end are read (they lie in the grid) and
// stored in the row's padding; rows are box_stride apart, which keeps the
// vector stores aligned and lets neighbouring rows start on other banks (at a
// stride of 16 the gather's reads met on them: FP64 68 us).
template <typename T>
__host__ __device__ constexpr int box_stride() {
  return sizeof(T) == 4 ? 20 : 18;
}
template <typename T, int V>
__device__ __forceinline__ void load_halo_rows(const PmeArgs &a, int b, const int (&org)[3], T *box) {
  typedef T vec __attribute__((ext_vector_type(V)));
  constexpr int LR = 16 / V;  // lanes per row
  const int Ka = a.K[0], Kb = a.K[1], Kc = a.K[2], H1 = a.H[1], rows = H1 * a.H[2];
  const T *g = (const T *)a.grid + (size_t)b * a.gstride;
  const int q = threadIdx.x % LR, step = blockDim.x / LR;
  int ga = org[0] + q * V;
  while (ga >= Ka) ga -= Ka;
  for (int r0 = threadIdx.x / LR; r0 < rows; r0 += 4 * step) {
    vec v[4];
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const int r = min(r0 + u * step, rows - 1), lc = (int)__umulhi((unsigned)r, a.mH1), lb = r - lc * H1;
      // n - 1 <= K on every grid: two conditional subtractions wrap
      int gb = org[1] + lb, gc = org[2] + lc;
      gb -= gb >= Kb ? Kb : 0;
      gc -= gc >= Kc ? Kc : 0;
      gb -= gb >= Kb ? Kb : 0;
      gc -= gc >= Kc ? Kc : 0;
      v[u] = *(const vec *)(g + (gc * Kb + gb) * Ka + ga);
    }
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const int r = r0 + u * step;
      if (r < rows) *(vec *)(box + r * box_stride<T>() + q * V) = v[u];
    }
  }
}

// One workgroup per (tile, bead): the potential on the halo box into LDS,
// then two lanes per charge (ewald3d_pme.c:534-560); lane part sums the planes
// mc = part * NI / 2 ... and the pair adds its sums.  Row sums in T; their
// products with the other axes' weights and the sums over rows in FP64.  V:
// points a lane loads (load_halo_rows), 0 for tiles it does not take.
// 4096 q-TIP4P/F at P = 32, mixed 35 -> 26 us, FP64 47 -> 40 us (LDS busy 59 %
// of the cycles, half of that bank conflicts of the charges' random places;
// vector units 49 %).
template <int NI, typename T, int V>
__global__ void __launch_bounds__(256) k_pme_gather(PmeArgs a) {
  extern __shared__ __align__(16) unsigned char lds_raw[];
  T *box = (T *)lds_raw;
  int tl, b;
  xcd_unit_bead(a.ntile, a.P, tl, b);
  const int tid = threadIdx.x;
  int lo, hi_;
  tile_items(a, tl, b, lo, hi_);
  if (lo == hi_) return;  // uniform over the workgroup
  const typename Rec<T>::V *rf = (const typename Rec<T>::V *)a.rfs + (size_t)b * a.nchrg;
  const int2 *ri = a.ris + (size_t)b * a.nchrg;
  int org[3];
  tile_origin(a, tl, org[0], org[1], org[2]);
  const int Ka = a.K[0], Kb = a.K[1], Kc = a.K[2];
  const int H0 = V > 0 ? box_stride<T>() : a.H[0], H01 = H0 * a.H[1];
  if constexpr (V > 0) load_halo_rows<T, V>(a, b, org, box);
  else load_halo<T>(a, b, org, box);
  __syncthreads();
  const double *hi = a.cell.hi;
  constexpr int HP = NI / 2;   // planes of lane 0
  constexpr int KP = NI - HP;  // planes per lane (lane 0 pads odd orders with zero weights)
  const int part = tid & 1;
  for (int c = lo + tid / 2; c < hi_; c += blockDim.x / 2) {
    const int2 si = ri[c];
    const typename Rec<T>::V f = rf[c];
    const int i = a.ichrg[si.y];
    T w[3][NI], dw[3][NI];
    int l[3];
    item_weights<NI, true, T>(f, si.x, w, dw, l);
    double wb[NI], dwb[NI];
#pragma unroll
    for (int m = 0; m < NI; m++) {
      wb[m] = (double)w[1][m];
      dwb[m] = (double)dw[1][m];
    }
    const T *base = box + (l[2] + part * HP) * H01 + l[1] * H0 + l[0];
    double da = 0.0, db = 0.0, dc = 0.0;
#pragma unroll
    for (int k = 0; k < KP; k++) {
      // lane 0 has HP planes: with an odd order its last is lane 1's first,
      // with weight zero
      const T a0 = k < HP ? w[2][k] : (T)0, d0 = k < HP ? dw[2][k] : (T)0;
      const double wc = (double)(part ? w[2][HP + k] : a0), dwc = (double)(part ? dw[2][HP + k] : d0);
      double pa = 0.0, pb = 0.0, pc = 0.0;
#pragma unroll
      for (int mb = 0; mb < NI; mb++) {
        const T *row = base + mb * H0;
        T r0 = (T)0, r1 = (T)0;
#pragma unroll
        for (int ma = 0; ma < NI; ma++) {
          const T phi = row[ma];
          r0 += dw[0][ma] * phi;
          r1 += w[0][ma] * phi;
        }
        pa += (double)r0 * wb[mb];
        pb += (double)r1 * dwb[mb];
        pc += (double)r1 * wb[mb];
      }
      da += pa * wc;
      db += pb * wc;
      dc += pc * dwc;
      base += H01;
    }
    // the pair's lanes hold the same charge
    da = dpp_rotate_add<0xB1>(da);  // quad_perm 1, 0, 3, 2
    db = dpp_rotate_add<0xB1>(db);
    dc = dpp_rotate_add<0xB1>(dc);
    if (part == 0) {
      const double q = a.q[i];
      da *= (double)Ka * q;
      db *= (double)Kb * q;
      dc *= (double)Kc * q;
      // bead-major, so the lines of one bead are written from its own XCD
      const size_t ib = (size_t)b * a.N + i;
      a.rx[ib] = -(da * hi[0] + db * hi[1] + dc * hi[2]);
      a.ry[ib] = -(da * hi[3] + db * hi[4] + dc * hi[5]);
      a.rz[ib] = -(da * hi[6] + db * hi[7] + dc * hi[8]);
    }
  }
}

// The k-space part of dE_b/dq_i: the convolved grid (the derivative of the
// k-space energy with respect to the grid charges) interpolated at the charge
// with the B-spline weights themselves (the gather's weights without the
// derivative).  One workgroup per (tile, bead), one lane per charge.
template <int NI, typename T>
__global__ void __launch_bounds__(PME_BLOCK) k_pme_phi(PmeArgs a) {
  extern __shared__ __align__(16) unsigned char lds_raw[];
  T *box = (T *)lds_raw;
  int tl, b;
  xcd_unit_bead(a.ntile, a.P, tl, b);
  const int tid = threadIdx.x;
  int lo, hi_;
  tile_items(a, tl, b, lo, hi_);
  if (lo == hi_) return;  // uniform over the workgroup
  const typename Rec<T>::V *rf = (const typename Rec<T>::V *)a.rfs + (size_t)b * a.nchrg;
  const int2 *ri = a.ris + (size_t)b * a.nchrg;
  int org[3];
  tile_origin(a, tl, org[0], org[1], org[2]);
  const int H0 = a.H[0], H01 = H0 * a.H[1];
  load_halo<T>(a, b, org, box);
  __syncthreads();
  for (int c = lo + tid; c < hi_; c += blockDim.x) {
    const int2 si = ri[c];
    const int i = a.ichrg[si.y];
    T w[3][NI], dw[3][NI];
    int l[3];
    item_weights<NI, false, T>(rf[c], si.x, w, dw, l);
    double v = 0.0;
    for (int mc = 0; mc < NI; mc++) {
#pragma unroll
      for (int mb = 0; mb < NI; mb++) {
        const T *row = box + (l[2] + mc) * H01 + (l[1] + mb) * H0 + l[0];
        T r = (T)0;
#pragma unroll
        for (int ma = 0; ma < NI; ma++) r += w[0][ma] * row[ma];
        v += (double)(r * (w[1][mb] * w[2][mc]));
      }
    }
    a.phi[(size_t)i * a.P + b] += v;
  }
}

// LDS of the gather (the halo box in the grid type) and of the spread (the
// halo box in FP64)
size_t pme_lds_bytes(const PmeArgs &a, bool gather) {
  return a.hvol * (gather && a.f32 ? sizeof(float) : sizeof(double));
}

#define PMX_PME_CASES(X) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(11) X(12)

template <typename T>
hipError_t launch_spread_t(const PmeArgs &a, hipStream_t st) {
  if (a.mm) {
    const dim3 g(xcd_grid(a.ntile, a.P));
    switch (a.n) {
      case 4: hipLaunchKernelGGL(HIP_KERNEL_NAME(k_pme_spread_mm<4, T>), g, dim3(64), 0, st, a); break;
      case 5: hipLaunchKernelGGL(HIP_KERNEL_NAME(k_pme_spread_mm<5, T>), g, dim3(64), 0, st, a); break;
      case 6: hipLaunchKernelGGL(HIP_KERNEL_NAME(k_pme_spread_mm<6, T>), g, dim3(64), 0, st, a); break;
      case 7: hipLaunchKernelGGL(HIP_KERNEL_NAME(k_pme_spread_mm<7, T>), g, dim3(64), 0, st, a); break;
      case 8: hipLaunchKernelGGL(HIP_KERNEL_NAME(k_pme_spread_mm<8, T>), g, dim3(64), 0, st, a); break;
      default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
  }
  const dim3 grid(xcd_grid(a.ntile, a.P)), block(spread_lanes<T>() * PME_BLOCK);
  const size_t lds = pme_lds_bytes(a, false);
  switch (a.n) {
#define X(NI) \
  case NI:                                                                                                  \
    if (lds > 65536)                                                                                          \
      (void)hipFuncSetAttribute((const void *)k_pme_spread<NI, T>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds); \
    hipLaunchKernelGGL(HIP_KERNEL_NAME(k_pme_spread<NI, T>), grid, block, lds, st, a);                                \
    break;
    PMX_PME_CASES(X)
#undef X
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

template <int NI, typename T, int V>
void launch_gather_v(const PmeArgs &a, hipStream_t st) {
  const size_t lds = V > 0 ? (size_t)box_stride<T>() * a.H[1] * a.H[2] * sizeof(T) : pme_lds_bytes(a, true);
  if (lds > 65536)
    (void)hipFuncSetAttribute((const void *)k_pme_gather<NI, T, V>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  // two lanes per charge: 256 lanes when a tile holds over 64 charges on average
  const int lanes = (long)a.nchrg > 64l * a.ntile ? 256 : 128;
  hipLaunchKernelGGL(HIP_KERNEL_NAME(k_pme_gather<NI, T, V>), dim3(xcd_grid(a.ntile, a.P)), dim3(lanes), lds, st, a);
}

template <typename T>
hipError_t launch_gather_t(const PmeArgs &a, hipStream_t st) {
  constexpr int V2 = 16 / (int)sizeof(T), V1 = V2 / 2;  // points of a 16 and an 8 byte load
  // rows of up to 16 points; their padding must fit the LDS where the box does
  const bool rows = a.H[0] <= 16 && (size_t)box_stride<T>() * a.H[1] * a.H[2] * sizeof(T) <= FFT_LDS_MAX;
  const int v = !rows ? 0 : a.T[0] % V2 == 0 ? V2 : a.T[0] % V1 == 0 ? V1 : 0;
  switch (a.n) {
#define X(NI)                                                    \
  case NI:                                                       \
    if (v == V2) launch_gather_v<NI, T, V2>(a, st);              \
    else if (v == V1) launch_gather_v<NI, T, V1>(a, st);         \
    else launch_gather_v<NI, T, 0>(a, st);                       \
    break;
    PMX_PME_CASES(X)
#undef X
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

// spread into halo boxes (the forward FFT folds them into the grid)
hipError_t launch_pme_spread(const PmeArgs &a, hipStream_t st) {
  return a.f32 ? launch_spread_t<float>(a, st) : launch_spread_t<double>(a, st);
}

template <typename T>
hipError_t launch_phi_t(const PmeArgs &a, hipStream_t st) {
  const dim3 grid(xcd_grid(a.ntile, a.P)), block(PME_BLOCK);
  const size_t lds = pme_lds_bytes(a, true);
  switch (a.n) {
#define X(NI) \
  case NI:                                                                                                  \
    if (lds > 65536)                                                                                          \
      (void)hipFuncSetAttribute((const void *)k_pme_phi<NI, T>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds); \
    hipLaunchKernelGGL(HIP_KERNEL_NAME(k_pme_phi<NI, T>), grid, block, lds, st, a);                                \
    break;
    PMX_PME_CASES(X)
#undef X
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_pme_phi(const PmeArgs &a, hipStream_t st) {
  return a.f32 ? launch_phi_t<float>(a, st) : launch_phi_t<double>(a, st);
}

// --- standard Ewald ---------------------------------------------------------------

// Structure factors, ewald3d_recip (ewald3d.c:27-373) with direct phases:
// one thread per (k, bead) sums q cos and q sin of 2 pi k.s over LDS tiles
// of the charges' fractional coordinates s = h^-1 r, then the k term's
// energy preg |S|^2 and pressure tensor go into block partial rows (the
// energy also on the diagonal, as the PME convolution writes them).
__global__ void __launch_bounds__(EWALD_BLOCK) k_ewald_sk(EwaldArgs a) {
  __shared__ double4 sq[EWALD_BLOCK];
  const int tid = threadIdx.x, b = blockIdx.y;
  const int k = blockIdx.x * EWALD_BLOCK + tid;
  const bool on = k < a.nk;
  const double4 kv = on ? a.kv[k] : make_double4(0, 0, 0, 0);
  const double *hi = a.cell.hi;
  double sr = 0.0, si = 0.0;
  for (int c0 = 0; c0 < a.nchrg; c0 += EWALD_BLOCK) {
    __syncthreads();
    if (c0 + tid < a.nchrg) {
      const int i = a.ichrg[c0 + tid];
      const size_t ib = (size_t)i * a.P + b;
      const double x = a.x[ib], y = a.y[ib], z = a.z[ib];
      sq[tid] = make_double4(x * hi[0] + y * hi[3] + z * hi[6], x * hi[1] + y * hi[4] + z * hi[7],
                             x * hi[2] + y * hi[5] + z * hi[8], a.q[i]);
    }
    __syncthreads();
    const int n = min(EWALD_BLOCK, a.nchrg - c0);
    for (int m = 0; m < n; m++) {
      const double4 c = sq[m];
      double sn, cs;
      sincos(kv.x * c.x + kv.y * c.y + kv.z * c.z, &sn, &cs);
      sr += cs * c.w;
      si += sn * c.w;
    }
  }
  double vals[FFT_NV] = {0, 0, 0, 0, 0, 0, 0};
  if (on) {
    const double4 kg = a.kg[k];
    const double smag = sr * sr + si * si;
    const double e = smag * kv.w, pr = kg.w * smag;
    vals[0] = e;
    vals[1] = pr * kg.x * kg.x + e;
    vals[2] = pr * kg.y * kg.y + e;
    vals[3] = pr * kg.z * kg.z + e;
    vals[4] = pr * kg.x * kg.y;
    vals[5] = pr * kg.x * kg.z;
    vals[6] = pr * kg.y * kg.z;
    a.sk[(size_t)b * a.nk + k] = make_double2(2.0 * kv.w * sr, 2.0 * kv.w * si);
  }
  block_partials<FFT_NV>(vals, 1, b, a.P, a.part, blockIdx.x, gridDim.x);
}

// Forces: one thread per (charge, bead) sums, over LDS tiles of the k list
// in ascending order, k (sin(k.r) 2 preg Re S - cos(k.r) 2 preg Im S), and
// adds q times it to the force (each (charge, bead) is one thread's).
__global__ void __launch_bounds__(EWALD_BLOCK) k_ewald_force(EwaldArgs a) {
  __shared__ double4 skv[EWALD_BLOCK], skg[EWALD_BLOCK];
  __shared__ double2 ssk[EWALD_BLOCK];
  const int tid = threadIdx.x, b = blockIdx.y;
  const int c = blockIdx.x * EWALD_BLOCK + tid;
  const bool on = c < a.nchrg;
  const double *hi = a.cell.hi;
  int i = 0;
  double s0 = 0.0, s1 = 0.0, s2 = 0.0;
  if (on) {
    i = a.ichrg[c];
    const size_t ib = (size_t)i * a.P + b;
    const double x = a.x[ib], y = a.y[ib], z = a.z[ib];
    s0 = x * hi[0] + y * hi[3] + z * hi[6];
    s1 = x * hi[1] + y * hi[4] + z * hi[7];
    s2 = x * hi[2] + y * hi[5] + z * hi[8];
  }
  double fx = 0.0, fy = 0.0, fz = 0.0;
  for (int k0 = 0; k0 < a.nk; k0 += EWALD_BLOCK) {
    __syncthreads();
    if (k0 + tid < a.nk) {
      skv[tid] = a.kv[k0 + tid];
      skg[tid] = a.kg[k0 + tid];
      ssk[tid] = a.sk[(size_t)b * a.nk + k0 + tid];
    }
    __syncthreads();
    const int n = min(EWALD_BLOCK, a.nk - k0);
    for (int m = 0; m < n; m++) {
      double sn, cs;
      sincos(skv[m].x * s0 + skv[m].y * s1 + skv[m].z * s2, &sn, &cs);
      const double fd = sn * ssk[m].x - cs * ssk[m].y;
      fx += skg[m].x * fd;
      fy += skg[m].y * fd;
      fz += skg[m].z * fd;
    }
  }
  if (on) {  // bead-major, added to the other forces after the pair kernel
    const size_t ib = (size_t)b * a.N + i;
    const double q = a.q[i];
    a.rx[ib] = fx * q;
    a.ry[ib] = fy * q;
    a.rz[ib] = fz * q;
  }
}

hipError_t launch_ewald(const EwaldArgs &a, hipStream_t st) {
  hipLaunchKernelGGL(k_ewald_sk, dim3((a.nk + EWALD_BLOCK - 1) / EWALD_BLOCK, a.P), dim3(EWALD_BLOCK), 0, st, a);
  hipLaunchKernelGGL(k_ewald_force, dim3((a.nchrg + EWALD_BLOCK - 1) / EWALD_BLOCK, a.P), dim3(EWALD_BLOCK), 0, st,
                     a);
  return hipGetLastError();
}

hipError_t launch_pme_gather(const PmeArgs &a, hipStream_t st) {
  return a.f32 ? launch_gather_t<float>(a, st) : launch_gather_t<double>(a, st);
}

}  // namespace pmx
