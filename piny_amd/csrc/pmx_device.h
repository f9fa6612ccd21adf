// Device helpers shared by the kernel files (internal).
#pragma once

#include <hip/hip_runtime.h>

#include "pmx_kernels.h"

namespace pmx {

__device__ __forceinline__ int nint_piny(double x) {
  // NINT with SIMP_NINT, defines.h:96-97
  return (int)((x) >= 0.0 ? ((x) + 0.5) : ((x)-0.5));
}

// The same rounding (half away from zero) as a double, without the round
// trip through an integer register: trunc(x + copysign(0.5, x)) equals
// (int)(x >= 0 ? x + 0.5 : x - 0.5) for every |x| < 2^31, up to the sign of
// a zero result.
__device__ __forceinline__ double nint_d(double x) { return trunc(x + copysign(0.5, x)); }

__device__ __forceinline__ void atomic_add(double *p, double v) { unsafeAtomicAdd(p, v); }

// v summed over the lanes whose index agrees modulo nb (nb a power of two up
// to 64), in every lane: exchanges across the wavefront's halves and rows
// (v_permlane32_swap, v_permlane16_swap), then DPP rotations within a row of
// 16, which need no LDS round trip (a shuffle of a double is two
// ds_bpermute).  A rotation by 8, 4, 2 or 1 serves as the exchange of that
// distance because the values already repeat with twice that period.
template <int CTRL>
__device__ __forceinline__ double dpp_rotate_add(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, false);
  return v + __hiloint2double(hi, lo);
}
__device__ __forceinline__ double wave_sum_mod(double v, int nb) {
  if (nb <= 32) {
    const auto lo = __builtin_amdgcn_permlane32_swap(__double2loint(v), __double2loint(v), false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap(__double2hiint(v), __double2hiint(v), false, false);
    v = __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
  }
  if (nb <= 16) {
    const auto lo = __builtin_amdgcn_permlane16_swap(__double2loint(v), __double2loint(v), false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap(__double2hiint(v), __double2hiint(v), false, false);
    v = __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
  }
  if (nb <= 8) v = dpp_rotate_add<0x128>(v);  // row_ror:8
  if (nb <= 4) v = dpp_rotate_add<0x124>(v);
  if (nb <= 2) v = dpp_rotate_add<0x122>(v);
  if (nb <= 1) v = dpp_rotate_add<0x121>(v);
  return v;
}

// Per-bead sums of NV values over the threads of one workgroup: thread t
// holds bead slot t % nb, and store(k, bead slot, sum) is called once for
// every value k and slot.  The order of the sums is fixed, so the result
// does not depend on scheduling.  Every thread of the block must call it;
// lds holds cap doubles (at least blockDim.x), free when it is called and
// again when it returns.
//
// The values go through LDS in batches as large as cap allows, two barriers
// a batch (one value at a time, with a barrier pair and a chain of LDS
// shuffles for each, took 23 of the 29 us that k_intra_mol's 31 values cost
// a box of 64 molecules).  nb a divisor of 64: each wavefront sums by lane
// exchanges first and LDS holds one entry per (value, wavefront, slot).
// Other nb: LDS holds every thread's value, and up to blockDim / nb threads
// a slot sum a run of them each before the last sum.
template <int NV, class Store>
__device__ __forceinline__ void block_sums(double (&v)[NV], int nb, double *lds, int cap, Store store) {
  const int tid = threadIdx.x, lane = tid & 63, bs = blockDim.x;
  if ((64 % nb) == 0 && (bs & 63) == 0) {
#pragma unroll
    for (int k = 0; k < NV; k++) v[k] = wave_sum_mod(v[k], nb);
    const int nw = bs >> 6, row = nw * nb, per = cap / row;
    for (int k0 = 0; k0 < NV; k0 += per) {
      const int n = min(per, NV - k0);
#pragma unroll
      for (int k = 0; k < NV; k++)
        if (k >= k0 && k < k0 + n && lane < nb) lds[(k - k0) * row + (tid >> 6) * nb + lane] = v[k];
      __syncthreads();
      for (int u = tid; u < n * nb; u += bs) {
        const int k = u / nb, b = u - k * nb;
        double t = 0.0;
        for (int w = 0; w < nw; w++) t += lds[k * row + w * nb + b];
        store(k0 + k, b, t);
      }
      __syncthreads();
    }
    return;
  }
  const int per = cap / bs, rows = bs / nb;  // blockDim.x is a multiple of nb
  for (int k0 = 0; k0 < NV; k0 += per) {
    const int n = min(per, NV - k0);
#pragma unroll
    for (int k = 0; k < NV; k++)
      if (k >= k0 && k < k0 + n) lds[(k - k0) * bs + tid] = v[k];
    __syncthreads();
    // seg threads per (value, slot), each the sum of a run of len rows into
    // its first row
    const int seg = max(1, min(rows, rows / n)), len = (rows + seg - 1) / seg;
    const int k = tid / (seg * nb), rem = tid - k * (seg * nb), g = rem / nb, b = rem - g * nb;
    if (k < n && seg > 1) {
      double t = 0.0;
      for (int r = g * len; r < min(rows, (g + 1) * len); r++) t += lds[k * bs + r * nb + b];
      if (g * len < rows) lds[k * bs + g * len * nb + b] = t;
    }
    __syncthreads();
    for (int u = tid; u < n * nb; u += bs) {
      const int kk = u / nb, bb = u - kk * nb, step = seg > 1 ? len : 1;
      double t = 0.0;
      for (int r = 0; r < rows; r += step) t += lds[kk * bs + r * nb + bb];
      store(k0 + kk, bb, t);
    }
    __syncthreads();
  }
}

// Those sums as a stage's partial row, part[(v*P + bead0 + k)*G + blk] for
// k < nb (the G blocks of one (value, bead) slot are contiguous, so the
// reduction reads them coalesced).
template <int NV>
__device__ __forceinline__ void block_partials(const double (&v)[NV], int nb, int bead0, int P, double *part,
                                               size_t blk, size_t G) {
  __shared__ double red[256];
  double s[NV];
#pragma unroll
  for (int k = 0; k < NV; k++) s[k] = v[k];
  block_sums<NV>(s, nb, red, 256, [&](int k, int b, double t) {
    if (bead0 + b < P) part[((size_t)k * P + bead0 + b) * G + blk] = t;
  });
}

// Workgroups are dispatched to the 8 XCDs of an MI355X in turn (workgroup
// id modulo 8), each XCD with its own L2.  Kernels whose work is (unit,
// bead) with units sharing a bead's data (PME tiles, FFT planes) launch
// units * P workgroups in one dimension.  Every group of 8 beads puts one
// bead on each XCD, so a bead's data stays in one L2.  The P % 8 beads left
// over are dealt to all XCDs, beads fastest: one XCD a bead would leave the
// others idle (a box of one bead ran its k space on 32 of the 256 CUs; 5003
// SPC/Fw, P = 1: 329 -> 309 us a force call).
__device__ __forceinline__ void xcd_unit_bead(int units, int P, int &unit, int &bead) {
  const int L = blockIdx.x, full = P & ~7, nfull = units * full;
  if (L < nfull) {
    const int r = L >> 3;
    bead = (L & 7) + 8 * (r / units);
    unit = r % units;
  } else {
    const int r = L - nfull, rem = P - full;
    bead = full + r % rem;
    unit = r / rem;
  }
}

inline unsigned xcd_grid(int units, int P) { return (unsigned)units * (unsigned)P; }

}  // namespace pmx
