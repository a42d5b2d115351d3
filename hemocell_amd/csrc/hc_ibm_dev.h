// hc_ibm_dev.h -- device helpers of the immersed-boundary coupling, shared by the
// IBM kernels and the fused per-cell step kernel.
#pragma once
#include <cmath>
#include <type_traits>

#include "hc_d3q19.h"
#include "hc_launch.h"
#include "hc_wrap.h"

namespace hcg {
namespace {

__device__ __forceinline__ int64_t wrap_mod(int64_t c, int n) {
  int64_t m = c % n;
  return m < 0 ? m + n : m;
}

// phi2 support of position p.  phi2(d) = max(1 - |d|, 0) is non-zero only on
// the nodes floor(p) and floor(p) + 1 of each axis, so the reference's 3x3x3
// candidates around the nearest node reduce to this 2x2x2 block, visited in the
// same x -> y -> z order.  Each of the 8 slots keeps its weight (0 when the
// node lies outside a non-periodic domain, has zero weight or is a wall node);
// adding the zero weights to the total changes nothing, so the normalised
// weights are those of immersedBoundaryMethod.h:62-138.  Fixed slots keep
// everything in registers.  W = double evaluates the weights in FP64 as the
// reference does; W = float (the FP32-shifted form's cell kernels) takes the
// fractional offsets p - floor(p) in FP64 and the weights from them in FP32,
// where 1 - d and d are the two hat values of an axis.
template <typename W>
struct SupportT {
  uint32_t idx[8];
  W w[8];
  int lo[3];  // unwrapped coordinates of the slot-0 node
};
using Support = SupportT<double>;

// Node indices and normalised weights from the low corner n0 and the hat values
// q of each axis.  A support inside the domain (all but the vertices at a domain
// face) is one index and three strides; otherwise the axes that leave it are
// wrapped or, closed, lose the hat value beyond the face: `fl(a)` gives the low
// corner as a double there (positions far outside do not fit an int).
template <typename W, typename FL>
__device__ __forceinline__ void finish_support(const int (&n0)[3], W (&q)[3][2], bool finite, FL fl,
                                               const LatticeDev& L, const uint8_t* __restrict__ type, SupportT<W>& s) {
  const int dims[3] = {L.nx, L.ny, L.nz};
  int w0[3], step[3];
  bool inside = finite;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    s.lo[a] = w0[a] = n0[a];
    step[a] = 1;
    inside = inside && (unsigned)n0[a] < (unsigned)(dims[a] - 1);
  }
  if (!inside) {
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      int w[2];
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const double node = finite ? fl(a) + (double)k : -1.0;
        if (node >= 0.0 && node < (double)dims[a]) {
          w[k] = (int)node;
        } else if (finite && L.periodic[a]) {
          w[k] = wrap_node(node, dims[a]);
        } else {
          w[k] = 0;
          q[a][k] = W(0);
        }
      }
      w0[a] = w[0];
      step[a] = w[1] - w[0];
    }
  }
  const uint32_t dz = (uint32_t)step[2], dy = (uint32_t)step[1] * (uint32_t)L.nz,
                 dx = (uint32_t)step[0] * (uint32_t)(L.ny * L.nz);
  const uint32_t n = (uint32_t)w0[2] + (uint32_t)L.nz * ((uint32_t)w0[1] + (uint32_t)L.ny * (uint32_t)w0[0]);
  W total = W(0);
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    s.idx[k] = n + ((k & 4) ? dx : 0u) + ((k & 2) ? dy : 0u) + ((k & 1) ? dz : 0u);
    s.w[k] = q[0][k >> 2] * q[1][(k >> 1) & 1] * q[2][k & 1];
  }
  if (type) {
    uint8_t t[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) t[k] = type[s.idx[k]];
#pragma unroll
    for (int k = 0; k < 8; ++k)
      if (t[k] != HC_NODE_FLUID) s.w[k] = W(0);
  }
#pragma unroll
  for (int k = 0; k < 8; ++k) total += s.w[k];
  const W coeff = W(1) / total;
#pragma unroll
  for (int k = 0; k < 8; ++k) s.w[k] = s.w[k] != W(0) ? s.w[k] * coeff : W(0);
}

template <typename W>
__device__ __forceinline__ void ibm_support(double p0, double p1, double p2, const LatticeDev& L,
                                            const uint8_t* __restrict__ type, SupportT<W>& s) {
  const double p[3] = {p0, p1, p2};
  W q[3][2];
  int n0[3];
  bool finite = true;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    finite = finite && fabs(p[a]) < 1.0e15;
    const double fl = floor(p[a]);
    n0[a] = (int)fl;
    if (std::is_same<W, float>::value) {
      const W d = (W)(p[a] - fl);  // in [0, 1)
      q[a][0] = W(1) - d;
      q[a][1] = d;
    } else {
      q[a][0] = (W)fmax(1.0 - fabs(p[a] - fl), 0.0);
      q[a][1] = (W)fmax(1.0 - fabs(p[a] - (fl + 1.0)), 0.0);
    }
  }
  finish_support(n0, q, finite, [&](int a) { return floor(p[a]); }, L, type, s);
}

// One force contribution to the spread: rounded to a multiple of L.spread_q when
// the exact spread is on.  spread_q is a power of two, so both scalings are
// exact and rint is the only rounding; the sums of such multiples stay exact
// (hence independent of the order of the adds) while they are below 2^53
// spread_q in magnitude.
template <typename R>
__device__ __forceinline__ double spread_term(double v, const LatticeDev& L) {
  if (std::is_same<R, float>::value) return v;  // FP64 only
  return L.spread_q > 0.0 ? rint(v * L.spread_inv_q) * L.spread_q : v;
}

// Minimum / maximum over a full wavefront by cross-lane moves within rows of 16
// and broadcasts between them; the result is in lane 63.  Every lane is active.
template <int CTRL>
__device__ __forceinline__ int dpp_move(int v) {
  return __builtin_amdgcn_update_dpp(v, v, CTRL, 0xf, 0xf, false);  // lanes without a source keep v
}
__device__ __forceinline__ int wave_min63(int v) {
  v = min(v, dpp_move<0x111>(v));  // row_shr:1, 2, 4, 8
  v = min(v, dpp_move<0x112>(v));
  v = min(v, dpp_move<0x114>(v));
  v = min(v, dpp_move<0x118>(v));
  v = min(v, dpp_move<0x142>(v));  // row_bcast:15, 31
  return min(v, dpp_move<0x143>(v));
}
__device__ __forceinline__ int wave_max63(int v) {
  v = max(v, dpp_move<0x111>(v));
  v = max(v, dpp_move<0x112>(v));
  v = max(v, dpp_move<0x114>(v));
  v = max(v, dpp_move<0x118>(v));
  v = max(v, dpp_move<0x142>(v));
  return max(v, dpp_move<0x143>(v));
}
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_moved(double v) {  // 0 in lanes without a source and rows not in ROWS
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, ROWS, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, ROWS, 0xf, false);
  return __hiloint2double(hi, lo);
}
// lane 63 gets the wavefront's sum, always added in the same order
__device__ __forceinline__ double wave_sum63(double v) {
  v += dpp_moved<0x111, 0xf>(v);
  v += dpp_moved<0x112, 0xf>(v);
  v += dpp_moved<0x114, 0xf>(v);
  v += dpp_moved<0x118, 0xf>(v);
  v += dpp_moved<0x142, 0xa>(v);
  return v + dpp_moved<0x143, 0xc>(v);
}
// The workgroup's bounds from its threads' bounds, in LDS: reduced over each
// wavefront first, then one LDS atomic per wavefront and bound.  With an atomic
// per thread the lanes of a wavefront queue at one LDS word: 35000 of the 158000
// cycles of a lone 642-vertex cell at 1024 threads (its step 84.6 -> 73.5 us), and
// the 15.5k-RBC suspension's FP32 step 3.35 -> 3.23 ms.
__device__ __forceinline__ void block_bounds(const int (&lmin)[3], const int (&lmax)[3], int* bmin, int* bmax) {
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const int lo = wave_min63(lmin[a]), hi = wave_max63(lmax[a]);
    if ((threadIdx.x & 63) == 63) {
      atomicMin(&bmin[a], lo);
      atomicMax(&bmax[a], hi);
    }
  }
}

// one thread's note of a cell's support box (VertexDev::box)
__device__ __forceinline__ void write_box(int* box, const int* bmin, const int* bmax, bool bad) {
  if (!box) return;
  for (int a = 0; a < 3; ++a) {
    box[a] = bmin[a];
    box[3 + a] = bad || bmax[a] < bmin[a] ? -1 : bmax[a] - bmin[a] + 2;
  }
}

__device__ __forceinline__ void atomic_add(float* p, float v) { unsafeAtomicAdd(p, v); }
__device__ __forceinline__ void atomic_add(double* p, double v) { unsafeAtomicAdd(p, v); }

__device__ __forceinline__ void lds_add(float* p, float v) { atomicAdd(p, v); }
__device__ __forceinline__ void lds_add(double* p, double v) { atomicAdd(p, v); }

}  // namespace
}  // namespace hcg
