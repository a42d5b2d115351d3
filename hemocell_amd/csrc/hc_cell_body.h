// hc_cell_body.h -- the vertex half of the IB-LBM step, fused per cell.
//
// One workgroup per cell runs, in the order of HemoCell::iterate()
// (core/hemoCell.cpp:299-376):
//   1. interpolateFluidVelocity + advanceParticles of step t
//      (core/hemoCellParticleField.cpp:566-588, :819-839): the cell's vertices
//      read the fluid velocity of their phi2 support, move, and land in LDS;
//   2. applyConstitutiveModel of step t (:633-675 and the model's
//      ParticleMechanics) on the positions in LDS;
//   3. spreadParticleForce of step t+1 (:841-863): the forces just computed (plus
//      any extra force, capped to f_limit in place) are spread from the same
//      positions into the force buffer of the next step, through one sum in LDS
//      per support node of the cell and one global atomic per non-zero sum.
//      The sums are doubles in both precisions: LDS double atomic adds run
//      several times faster than float ones on this chip.
// Step t+1's spread needs exactly x_t and F(x_t), which steps 1-2 produce, so
// doing it here saves reloading the cell.  Positions stay in LDS for the whole
// kernel; per-vertex bending forces and velocities too when they fit.
//
// Instantiated by hc_cell_f64.hip (FP64, compiled without contracting
// multiply-adds, so that every layout and launch rounds alike; its red and white
// cells sum around a vertex's ring, not in the oracle's order) and hc_cell_f32.hip
// (the FP32-shifted form, which may fuse them).
#pragma once
#include <algorithm>
#include <type_traits>

#include "hc_ibm_dev.h"
#include "hc_lds_plan.h"
#include "hc_mech_dev.h"

namespace hcg {
namespace {

enum { CELL_INTERP = 1, CELL_MECH = 2, CELL_SPREAD = 4 };
// 64-triangle chunks of a mesh whose volume is summed in an order independent of
// the block size (meshes up to 8192 triangles)
constexpr int kVolChunks = 128;

// Scalar type of the positions in LDS and of the membrane mechanics: the FP32-
// shifted form's staged kernels keep float offsets from the cell's first vertex
// (the mechanics only takes differences of positions; the volume stays FP64);
// everything else keeps absolute double positions.
template <typename R, bool STAGED, bool GPOS>
using MechT = typename std::conditional<std::is_same<R, float>::value && STAGED && !GPOS, float, double>::type;

// STAGED: positions, velocities and bending forces in LDS.  Otherwise positions
// in LDS and the rest in global memory, or (GPOS) the positions too: then the
// workgroup needs LDS only for the spread box and fits beside the many small
// workgroups of another cell type running at the same time.
template <typename R, int MODEL, int BS, bool STAGED, bool GPOS>
__device__ __forceinline__ void cell_step_body(const VertexDev& V, const TypeDev& T, const int64_t base, int* cell_box,
                                               const R* __restrict__ uf, const uint8_t* __restrict__ type,
                                               const LatticeDev& L, R* __restrict__ Fnext,
                                               const double* __restrict__ extra, double* __restrict__ scratch,
                                               double f_limit, int flags, int box_nodes,
                                               unsigned long long* wall_hits) {
  using P = MechT<R, STAGED, GPOS>;
  constexpr bool REL = !std::is_same<P, double>::value;  // LDS holds offsets from the cell origin
  // scalar of the support weights, the interpolated velocity and the spread's
  // contributions: FP32 in the FP32-shifted form (whose velocity field and
  // force field are FP32), FP64 otherwise
  using SW = typename std::conditional<std::is_same<R, float>::value, float, double>::type;
  extern __shared__ __align__(16) double sm[];
  __shared__ double red[kVolChunks];
  __shared__ double vforce_sh;
  __shared__ int bmin[3], bmax[3], bad, farpk;
  __shared__ int wsum[BS / 64];
  const int tid = threadIdx.x;
  const int nv = T.nv;
  const int64_t vs = V.vs;
  const bool visc = (MODEL != HC_MODEL_RBC) || (T.eta_m != 0.0);
  // the spread's support box bounds, first used after the barrier ending phase 1
  if (tid == 0) {
    for (int a = 0; a < 3; ++a) {
      bmin[a] = 0x7fffffff;
      bmax[a] = -0x7fffffff;
    }
    bad = 0;
    farpk = 0;
  }
  // origin of the offsets: the first vertex before this step's advance, read by
  // every thread before any thread moves it (its advanced position is stored
  // only after the barrier that ends phase 1)
  double org0 = 0.0, org1 = 0.0, org2 = 0.0;
  if (REL) {
    org0 = V.x[base];
    org1 = V.x[vs + base];
    org2 = V.x[2 * vs + base];
  }
  __shared__ double held_sh[3];  // REL: vertex 0's advanced position until then
  bool held = false;
  // LDS: positions, then (STAGED) velocities, then a region shared by the bending
  // forces (phase 2) and the spread box (phase 3)
  P* const sp_ = reinterpret_cast<P*>(sm);
  P* px = GPOS ? reinterpret_cast<P*>(V.x + base) : sp_;
  P* py = GPOS ? reinterpret_cast<P*>(V.x + vs + base) : sp_ + nv;
  P* pz = GPOS ? reinterpret_cast<P*>(V.x + 2 * vs + base) : sp_ + 2 * nv;
  P *vx, *vy, *vz, *bx, *by, *bz;
  // the region (bending forces, then the box) after the fixed part (hc_lds_plan.h)
  double* const region =
      reinterpret_cast<double*>(reinterpret_cast<char*>(sm) + cell_fixed_bytes(nv, visc, sizeof(P), STAGED, GPOS));
  if (STAGED) {
    vx = sp_ + 3 * nv;
    vy = sp_ + 4 * nv;
    vz = sp_ + 5 * nv;
    bx = reinterpret_cast<P*>(region);
    by = bx + nv;
    bz = bx + 2 * nv;
  } else {
    vx = reinterpret_cast<P*>(V.v + base);
    vy = reinterpret_cast<P*>(V.v + vs + base);
    vz = reinterpret_cast<P*>(V.v + 2 * vs + base);
    bx = reinterpret_cast<P*>(scratch + base);
    by = reinterpret_cast<P*>(scratch + vs + base);
    bz = reinterpret_cast<P*>(scratch + 2 * vs + base);
  }
  // Absolute position of vertex k for the spread: LDS (double), or with float
  // offsets in LDS (REL) a packed copy that phase 3 writes over the offsets once
  // the mechanics is done: per axis the node floor(x) relative to the origin's
  // node (8 bits) and x - floor(x) in 24-bit fixed point, which rebuilds floor(x)
  // exactly and the fraction to 2^-24 (a float's resolution near 1) without
  // rereading the vertex planes; the planes when a cell spans more than 127 nodes.
  bool use_pk = false;
  const uint32_t* const pk = reinterpret_cast<const uint32_t*>(sp_);
  const double fo0 = floor(org0), fo1 = floor(org1), fo2 = floor(org2);
  auto unpack = [&](double fo, uint32_t w) -> double {
    return fo + (double)((int)(w >> 24) - 128) + (double)(w & 0xFFFFFFu) * (1.0 / 16777216.0);
  };
  auto pos_x = [&](int k) -> double {
    return REL ? (use_pk ? unpack(fo0, pk[k]) : V.x[base + k]) : (double)px[k];
  };
  auto pos_y = [&](int k) -> double {
    return REL ? (use_pk ? unpack(fo1, pk[nv + k]) : V.x[vs + base + k]) : (double)py[k];
  };
  auto pos_z = [&](int k) -> double {
    return REL ? (use_pk ? unpack(fo2, pk[2 * nv + k]) : V.x[2 * vs + base + k]) : (double)pz[k];
  };
  // low corner and support of vertex k for the spread; from a packed position
  // without double arithmetic
  const int foi[3] = {(int)fo0, (int)fo1, (int)fo2};
  auto low_node = [&](int k, int (&n0)[3]) {
    if (REL && use_pk) {
#pragma unroll
      for (int a = 0; a < 3; ++a) n0[a] = foi[a] + (int)(pk[a * nv + k] >> 24) - 128;
    } else {
      n0[0] = (int)floor(pos_x(k));
      n0[1] = (int)floor(pos_y(k));
      n0[2] = (int)floor(pos_z(k));
    }
  };
  auto support_of = [&](int k, SupportT<SW>& sp) {
    if (REL && use_pk) {
      int n0[3];
      SW q[3][2];
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        const uint32_t w = pk[a * nv + k];
        n0[a] = foi[a] + (int)(w >> 24) - 128;
        q[a][1] = (SW)(w & 0xFFFFFFu) * SW(1.0 / 16777216.0);
        q[a][0] = SW(1) - q[a][1];
      }
      finish_support(n0, q, true, [&](int a) { return (double)n0[a]; }, L, type, sp);
    } else {
      ibm_support(pos_x(k), pos_y(k), pos_z(k), L, type, sp);
    }
  };
  // the spread's scratch: the region and the list bytes after it
  const int scratch_bytes = 24 * box_nodes + (int)cell_list_bytes(nv);

  // ---- 1. interpolation and advance ------------------------------------------
  // A thread takes up to U of its vertices at once, so their position loads are in
  // flight together.
  // A vertex removed by wall contact (flag) stays where it is and spreads
  // nothing; its cell is incomplete from then on (hemoCellParticleField.cpp:
  // 566-588 removes it; applyConstitutiveModel, :633-675, skips cells with a
  // vertex missing and zeroes the rest's forces).
  constexpr int U = 3;
  bool lrem = false, lfar = false;
  // the vertex is on a node that is not fluid: a wall hit
  auto wall_contact = [&](int64_t i, const int (&wc)[3]) {
    if (type[(uint32_t)wc[2] + (uint32_t)L.nz * ((uint32_t)wc[1] + (uint32_t)L.ny * (uint32_t)wc[0])] == HC_NODE_FLUID)
      return;
    atomicAdd(wall_hits, 1ull);
    if (V.flag) V.flag[i] = VFLAG_REMOVED;
    lrem = true;
  };
  for (int k0 = tid; k0 < nv; k0 += U * BS) {
    double xa[U][3];
    bool gone[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = k0 + u * BS;
      if (k >= nv) continue;
      const int64_t i = base + k;
      xa[u][0] = V.x[i];
      xa[u][1] = V.x[vs + i];
      xa[u][2] = V.x[2 * vs + i];
      gone[u] = V.flag && (V.flag[i] & VFLAG_REMOVED);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = k0 + u * BS;
      if (k >= nv) continue;
      const int64_t i = base + k;
      if (gone[u]) {
        lrem = true;
        if (!GPOS) {
          px[k] = (P)(xa[u][0] - org0);
          py[k] = (P)(xa[u][1] - org1);
          pz[k] = (P)(xa[u][2] - org2);
        }
        if (STAGED && visc) vx[k] = vy[k] = vz[k] = P(0);
        continue;
      }
      double v0, v1, v2;
      if (flags & CELL_INTERP) {
        SupportT<SW> sp;
        ibm_support(xa[u][0], xa[u][1], xa[u][2], L, type, sp);
        // four nodes at a time, the ones without weight too, so that their reads are
        // in flight together (behind a test per node each was waited for alone;
        // eight at a time take the registers of a wavefront per SIMD)
        SW w0 = SW(0), w1 = SW(0), w2 = SW(0);
#pragma unroll
        for (int h = 0; h < 8; h += 4) {
          R un[4][3];
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const R* at = uf + 3 * (uint64_t)sp.idx[h + q];
            un[q][0] = at[0];
            un[q][1] = at[1];
            un[q][2] = at[2];
          }
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const bool on = sp.w[h + q] != SW(0);
            w0 += (on ? (SW)un[q][0] : SW(0)) * sp.w[h + q];
            w1 += (on ? (SW)un[q][1] : SW(0)) * sp.w[h + q];
            w2 += (on ? (SW)un[q][2] : SW(0)) * sp.w[h + q];
          }
          __builtin_amdgcn_sched_barrier(0);
        }
        V.v[i] = v0 = (double)w0;
        V.v[vs + i] = v1 = (double)w1;
        V.v[2 * vs + i] = v2 = (double)w2;
      } else {
        v0 = V.v[i];
        v1 = V.v[vs + i];
        v2 = V.v[2 * vs + i];
      }
      const double x0 = xa[u][0] + v0, x1 = xa[u][1] + v1, x2 = xa[u][2] + v2;
      if (REL && k == 0) {
        held = true;
        held_sh[0] = x0;
        held_sh[1] = x1;
        held_sh[2] = x2;
      } else {
        V.x[i] = x0;
        V.x[vs + i] = x1;
        V.x[2 * vs + i] = x2;
      }
      if (!GPOS) {
        px[k] = (P)(x0 - org0);
        py[k] = (P)(x1 - org1);
        pz[k] = (P)(x2 - org2);
      }
      if (STAGED && visc) {
        vx[k] = (P)v0;
        vy[k] = (P)v1;
        vz[k] = (P)v2;
      }
      if (type && isfinite(x0) && isfinite(x1) && isfinite(x2)) {
        const double p[3] = {x0, x1, x2};
        const int dims[3] = {L.nx, L.ny, L.nz};
        int wc[3];
        bool out = false;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          const double fl = floor(p[a] + 0.5);
          if (fl >= 0.0 && fl < (double)dims[a]) wc[a] = (int)fl;
          else if (!(fabs(fl) < kNearNodes)) lfar = out = true;
          else if (L.periodic[a]) wc[a] = wrap_node(fl, dims[a]);
          else out = true;
        }
        if (!out) wall_contact(i, wc);
      }
    }
  }
  // A vertex flung so far that its node takes an exact remainder: by itself, since the
  // remainder's loop in the one above held up every vertex (743 RBC in FP64 130 -> 132 us
  // per launch, the platelets beside them 44 -> 50).
  if (lfar) {
#pragma unroll 1
    for (int k = tid; k < nv; k += BS) {
      const int64_t i = base + k;
      if (V.flag && (V.flag[i] & VFLAG_REMOVED)) continue;
      const bool kept = REL && k == 0;  // held back
      const double p[3] = {kept ? held_sh[0] : V.x[i], kept ? held_sh[1] : V.x[vs + i],
                           kept ? held_sh[2] : V.x[2 * vs + i]};
      const int dims[3] = {L.nx, L.ny, L.nz};
      int wc[3];
      bool out = !(isfinite(p[0]) && isfinite(p[1]) && isfinite(p[2])), far = false;
      for (int a = 0; a < 3; ++a) {
        const double fl = floor(p[a] + 0.5);
        far = far || !(fabs(fl) < kNearNodes);
        if (out) continue;
        if (L.periodic[a]) wc[a] = wrap_far(fl, dims[a]);
        else if (fl >= 0.0 && fl < (double)dims[a]) wc[a] = (int)fl;
        else out = true;
      }
      if (far && !out) wall_contact(i, wc);
    }
  }
  const bool incomplete = __syncthreads_or(lrem) != 0;
  if (held) {
    V.x[base] = held_sh[0];
    V.x[vs + base] = held_sh[1];
    V.x[2 * vs + base] = held_sh[2];
  }
  const CellViewT<P> c{px, py, pz};

  // The force a vertex spreads: its force plus any extra force, capped to f_limit
  // (hemoCellParticleField.cpp:846-852).  Applied where the mechanics stores the
  // force when it ran on this cell, else by the spread.
  auto cap_force = [&](int64_t i, double& f0, double& f1, double& f2) -> bool {
    bool changed = false;
    if (extra) {
      f0 += extra[i];
      f1 += extra[vs + i];
      f2 += extra[2 * vs + i];
      changed = true;
    }
    const double fm = sqrt(f0 * f0 + f1 * f1 + f2 * f2);
    if (fm > f_limit) {
      const double sc = f_limit / fm;
      f0 *= sc;
      f1 *= sc;
      f2 *= sc;
      changed = true;
    }
    return changed;
  };
  const bool capped = (flags & CELL_MECH) && !incomplete;

  // ---- 2. mechanics ------------------------------------------------------------
  if ((flags & CELL_MECH) && incomplete) {
    for (int k = tid; k < nv; k += BS) {
      const int64_t i = base + k;
      V.f[i] = 0.0;
      V.f[vs + i] = 0.0;
      V.f[2 * vs + i] = 0.0;
    }
    __syncthreads();
  } else if (flags & CELL_MECH) {
    // FP64: roots and quotients once per triangle and edge (hc_mech_dev.h).  Region
    // left beside the bending forces for both lists of factors: everything is
    // evaluated at once, then gathered; otherwise one after the other, with the
    // vertices' sums in V.f between.  The sums are the same either way.  One
    // RBC 57 -> 52 us per step; 120 x 136 x 250 nodes with 1886 RBC 765 -> 743.
    constexpr bool kFactors = MODEL != HC_MODEL_PLT && std::is_same<R, double>::value;
    constexpr bool kOnce = kFactors && STAGED;
    const bool once = kOnce && T.rid;  // at most 2 nv triangles and 3 nv edges
    const bool apart = 3 * nv + T.nt + T.ne <= 3 * box_nodes;
    P* const tri_f = reinterpret_cast<P*>(region) + (apart ? 3 * nv : 0);
    // the volume: triangle t is lane t % 64 of chunk t / 64; a wavefront sums a
    // chunk over its lanes (by moves between registers: through LDS the six steps
    // cost a fifth of the mechanics) and the chunks are added in order, so the sum
    // is the same at every block size (batched, mixed and alone launches agree bit
    // for bit); larger meshes sum per thread, then per wavefront
    const int nchunk = (T.nt + 63) >> 6;
    int nred = nchunk;
    if (nchunk <= kVolChunks) {
      const V3T<P> rm = c.pos(0);
      const D3 r = {(double)rm.x, (double)rm.y, (double)rm.z};
      for (int ch = tid >> 6; ch < nchunk; ch += BS / 64) {
        const int t = (ch << 6) | (tid & 63);
        const double part = wave_sum63(volume_term(c, T, t, r));
        if ((tid & 63) == 63) red[ch] = part;
        if (kOnce && once && t < T.nt) tri_f[t] = triangle_factor(c, T, t);
      }
    } else {
      const double part = wave_sum63(volume_partial<BS>(c, T, tid));
      if ((tid & 63) == 63) red[tid >> 6] = part;
      nred = BS / 64;
      if (kOnce && once)
        for (int t = tid; t < T.nt; t += BS) tri_f[t] = triangle_factor(c, T, t);
    }
    auto volume_force = [&]() {
      double vsum = red[0];
      for (int w = 1; w < nred; ++w) vsum += red[w];
      const double volume = vsum * (1.0 / 6.0);
      const double vf = (volume - T.volume_eq) / T.volume_eq;
      return -T.k_volume * vf / fabs(MaxCellVolumetricChange - vf * vf);
    };
    if constexpr (kOnce) {
      if (once) {
        P* const edge_f = reinterpret_cast<P*>(region) + (apart ? 3 * nv + T.nt : 0);
        auto edges = [&]() {
          for (int e = tid; e < T.ne; e += BS) edge_f[e] = edge_factor(c, T, e, vx, vy, vz, visc);
        };
        auto bending = [&]() {
          for (int k = tid; k < nv; k += BS) {
            const RingOf ring(T, k);
            const V3T<P> b = bending_of_ring<P>(c, T, k, ring.R, ring.nr);
            bx[k] = b.x;
            by[k] = b.y;
            bz[k] = b.z;
          }
        };
        // each of steps 1 (triangles), 2 (bending) and 4 (edges, inner links, cap)
        // adds to the vertices' sums
        auto gather = [&](int steps, P vforce) {
          for (int k = tid; k < nv; k += BS) {
            const int64_t i = base + k;
            const RingOf ring(T, k);
            P f0 = P(0), f1 = P(0), f2 = P(0);
            if (steps & 1) {
              gather_triangles<P>(c, T, ring, k, tri_f, vforce, f0, f1, f2);
            } else {
              f0 = V.f[i];
              f1 = V.f[vs + i];
              f2 = V.f[2 * vs + i];
            }
            if (steps & 2) gather_bending<P>(ring, k, bx, by, bz, f0, f1, f2);
            if (steps & 4) {
              gather_edges<P>(c, T, ring, k, edge_f, f0, f1, f2);
              inner_forces<MODEL, P>(c, T, k, f0, f1, f2);
              if (flags & CELL_SPREAD) cap_force(i, f0, f1, f2);
            }
            V.f[i] = f0;
            V.f[vs + i] = f1;
            V.f[2 * vs + i] = f2;
          }
        };
        if (apart) {
          bending();
          edges();
        }
        __syncthreads();  // the factors, and the volume's partial sums
        const P vforce = (P)volume_force();
        if (apart) {
          gather(7, vforce);
        } else {
          gather(1, vforce);
          __syncthreads();
          bending();
          __syncthreads();
          gather(2, P(0));
          __syncthreads();
          edges();
          __syncthreads();
          gather(4, P(0));
        }
      }
    }
    if (!once) {
      __syncthreads();
      if (tid == 0) vforce_sh = volume_force();
      // FP32 RBC and WBC: the ring-ordered tables, else the compact per-slot ones
      // (both built beside the padded tables, whose entries lie 112 bytes apart: a
      // 642-vertex WBC's forces took 22 of 77 kcycles with them, 13 with the rings)
      constexpr bool kCompact = MODEL != HC_MODEL_PLT && std::is_same<P, float>::value;
      const bool compact = kCompact && T.cring != nullptr;
      if (MODEL != HC_MODEL_PLT) {
        for (int k = tid; k < nv; k += BS) {
          V3T<P> b;
          if constexpr (kCompact) b = compact ? bending_force_c(c, T, k) : bending_force(c, T, k);
          else b = bending_force(c, T, k);
          bx[k] = b.x;
          by[k] = b.y;
          bz[k] = b.z;
        }
      }
      // A platelet's edges once each, for the vertices to gather: by vertex, every
      // edge was evaluated four times and a vertex's twelve one after another
      // (24 platelets in FP64: this kernel 51 -> 37 us).
      P* edge_f = nullptr;
      if constexpr (MODEL == HC_MODEL_PLT && STAGED) {
        if (6 * (size_t)T.ne * sizeof(P) <= platelet_edge_bytes(nv, sizeof(P))) {
          edge_f = reinterpret_cast<P*>(region);
          for (int e = tid; e < T.ne; e += BS) platelet_edge(c, T, e, vx, vy, vz, edge_f + e, T.ne);
        }
      }
      __syncthreads();
      const P vforce = (P)vforce_sh;
      for (int k = tid; k < nv; k += BS) {
        V3T<P> F;
        if constexpr (kFactors && !STAGED) {
          if (T.rid) F = vertex_force_factors<MODEL, P>(c, T, k, vforce, bx, by, bz, vx, vy, vz, visc);
          else F = vertex_force<MODEL, TERM_ALL, P>(c, T, k, vforce, bx, by, bz, vx, vy, vz, visc);
        } else if constexpr (kCompact) {
          if (T.rpar) F = vertex_force_ring(c, T, k, vforce, bx, by, bz, vx, vy, vz, visc);
          else if (compact) F = vertex_force_compact(c, T, k, vforce, bx, by, bz, vx, vy, vz, visc);
          else F = vertex_force<MODEL, TERM_ALL & ~TERM_INNER, P>(c, T, k, vforce, bx, by, bz, vx, vy, vz, visc);
          inner_forces<MODEL, P>(c, T, k, F.x, F.y, F.z);
        } else F = vertex_force<MODEL, TERM_ALL, P>(c, T, k, vforce, bx, by, bz, vx, vy, vz, visc, edge_f);
        const int64_t i = base + k;
        double f0 = (double)F.x, f1 = (double)F.y, f2 = (double)F.z;
        if (flags & CELL_SPREAD) cap_force(i, f0, f1, f2);
        V.f[i] = f0;
        V.f[vs + i] = f1;
        V.f[2 * vs + i] = f2;
      }
    }
    __syncthreads();  // forces visible to the whole workgroup; the region is free again
  }
  if (!(flags & CELL_SPREAD)) return;

  // ---- 3. spread of the next step ---------------------------------------------
  // the force each vertex spreads: its force plus any extra force, capped to
  // f_limit and written back in place when that changed it
  // (hemoCellParticleField.cpp:846-852; done by the mechanics above when it ran
  // on this cell); with repulsion the spread is a pass of its own.  The packed
  // positions below overwrite the offsets: the mechanics ended with a barrier.
  {
    int lmin[3] = {0x7fffffff, 0x7fffffff, 0x7fffffff}, lmax[3] = {-0x7fffffff, -0x7fffffff, -0x7fffffff};
    bool lbad = false, lfar = false;
    uint32_t* const pkw = reinterpret_cast<uint32_t*>(sp_);
    const double fo[3] = {fo0, fo1, fo2};
    for (int k = tid; k < nv; k += BS) {
      const double p[3] = {pos_x(k), pos_y(k), pos_z(k)};  // use_pk is still false here
      for (int a = 0; a < 3; ++a) {
        if (!(fabs(p[a]) < 1.0e9)) {
          lbad = true;
          continue;
        }
        const double fl = floor(p[a]);
        const int cc = (int)fl;
        lmin[a] = min(lmin[a], cc);
        lmax[a] = max(lmax[a], cc);
        if (REL) {
          const double rel = fl - fo[a];
          if (!(rel >= -128.0 && rel <= 127.0)) lfar = true;
          const uint32_t f24 = min((uint32_t)((p[a] - fl) * 16777216.0), 0xFFFFFFu);
          pkw[a * nv + k] = ((uint32_t)((int)rel + 128) << 24) | f24;
        }
      }
      const int64_t i = base + k;
      if (capped || (incomplete && (V.flag[i] & VFLAG_REMOVED))) continue;
      double f0 = V.f[i], f1 = V.f[vs + i], f2 = V.f[2 * vs + i];
      if (cap_force(i, f0, f1, f2)) {
        V.f[i] = f0;
        V.f[vs + i] = f1;
        V.f[2 * vs + i] = f2;
      }
    }
    block_bounds(lmin, lmax, bmin, bmax);
    if (lbad) bad = 1;
    if (lfar) farpk = 1;
    // the spread's scratch starts at zero: the row masks and the node sums
    for (int e = tid; e < scratch_bytes / 8; e += BS) region[e] = 0.0;
  }
  __syncthreads();
  use_pk = REL && !bad && !farpk;
  if (tid == 0) write_box(cell_box, bmin, bmax, bad != 0);
  const int o0 = bmin[0], o1 = bmin[1], o2 = bmin[2];
  const int s0 = bmax[0] - bmin[0] + 2, s1 = bmax[1] - bmin[1] + 2, s2 = bmax[2] - bmin[2] + 2;
  // Only the nodes in some vertex's support get a sum: a mask of 64 z-nodes per
  // (x, y) row of the box says which, and a node's place is the number of marked
  // nodes before it.  An RBC's surface touches ~1290 of the up to 5832 nodes of
  // its box and fits in two passes of ~680 sums (a WBC's 2210 in four), where
  // slabs of the whole box took one pass per x-plane (18 passes of ~70 vertices
  // on 256 threads, two barriers each).  With the supports' short forms above:
  // the 15.5k-RBC suspension's step 3.23 -> 2.99 ms in FP32 and 2.88 -> 2.85 ms
  // (half the box) in FP64, a lone RBC 73 -> 58 us with everything in one pass.
  const int zw = (s2 + 63) >> 6;
  const bool sane = !bad && s0 > 0 && s0 <= 4096 && s1 <= 4096 && s2 <= 65536;
  const int64_t nrows = sane ? (int64_t)s0 * s1 * zw : 0;
  // per row a 64-bit mask and a first place, per sum 3 doubles and its node
  const bool direct = !sane || 12 * nrows + 28 * 64 > scratch_bytes;
  const int64_t S = L.stride;
  auto spread_force = [&](int64_t i, double& f0, double& f1, double& f2) {
    if (incomplete && (V.flag[i] & VFLAG_REMOVED)) {
      f0 = f1 = f2 = 0.0;
      return;
    }
    f0 = V.f[i];
    f1 = V.f[vs + i];
    f2 = V.f[2 * vs + i];
  };
  if (direct) {
    for (int k = tid; k < nv; k += BS) {
      const int64_t i = base + k;
      double f0, f1, f2;
      spread_force(i, f0, f1, f2);
      const SW g0 = (SW)f0, g1 = (SW)f1, g2 = (SW)f2;
      SupportT<SW> sp;
      support_of(k, sp);
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        if (sp.w[q] == SW(0)) continue;
        const int64_t n = sp.idx[q];
        atomic_add(&Fnext[n], (R)spread_term<R>((double)(g0 * sp.w[q]), L));
        atomic_add(&Fnext[S + n], (R)spread_term<R>((double)(g1 * sp.w[q]), L));
        atomic_add(&Fnext[2 * S + n], (R)spread_term<R>((double)(g2 * sp.w[q]), L));
      }
    }
    return;
  }
  const int rows = (int)nrows;
  const int cap = (scratch_bytes - 12 * rows) / 28;
  unsigned long long* const mask = reinterpret_cast<unsigned long long*>(region);
  double* const box = region + rows;
  uint32_t* const place = reinterpret_cast<uint32_t*>(box + 3 * cap);
  uint32_t* const node = place + rows;
  // lanes of one wavefront take vertices ~nv/64 apart (fewer LDS same-address operations)
  const int per = (nv + 63) / 64;
  for (int k = tid; k < 64 * per; k += BS) {
    const int vtx = (k & 63) * per + (k >> 6);
    if (vtx >= nv) continue;
    int n0[3];
    low_node(vtx, n0);
    const int lz = n0[2] - o2;
    const int r = (n0[1] - o1 + s1 * (n0[0] - o0)) * zw + (lz >> 6), bit = lz & 63;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int rq = r + ((q >> 1) * s1 + (q & 1)) * zw;
      atomicOr(&mask[rq], 3ull << bit);
      if (bit == 63) atomicOr(&mask[rq + 1], 1ull);
    }
  }
  __syncthreads();
  // each row's first place: an exclusive prefix sum of the rows' node counts
  int total = 0;
  for (int r0 = 0; r0 < rows; r0 += BS) {
    const int r = r0 + tid;
    const int c = r < rows ? __popcll(mask[r]) : 0;
    int inc = c;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_up(inc, o);
      if ((tid & 63) >= o) inc += y;
    }
    if ((tid & 63) == 63) wsum[tid >> 6] = inc;
    __syncthreads();
    int before = total;
#pragma unroll
    for (int w = 0; w < BS / 64; ++w) {
      if (w < (tid >> 6)) before += wsum[w];
      total += wsum[w];
    }
    if (r < rows) place[r] = (uint32_t)(before + inc - c);
    if (r0 + BS < rows) __syncthreads();
  }
  const int dims[3] = {L.nx, L.ny, L.nz};
  auto wrapped = [&](int a, int c) -> uint32_t { return (c >= 0 && c < dims[a]) ? (uint32_t)c : (uint32_t)wrap_node((double)c, dims[a]); };
  for (int p0 = 0; p0 < total; p0 += cap) {
    const int count = min(cap, total - p0);
    // the nodes of this pass's places (a thread's rows are those whose place it wrote)
    for (int r = tid; r < rows; r += BS) {
      unsigned long long m = mask[r];
      int j = (int)place[r] - p0;
      if (j >= count || j + __popcll(m) <= 0) continue;
      const unsigned xy = zw == 1 ? (unsigned)r : (unsigned)r / (unsigned)zw;
      const unsigned lx = xy / (unsigned)s1, ly = xy - lx * (unsigned)s1;
      const int z = o2 + 64 * (r - (int)xy * zw);
      const uint32_t at = (uint32_t)L.nz * (wrapped(1, o1 + (int)ly) + (uint32_t)L.ny * wrapped(0, o0 + (int)lx));
      for (; m; m &= m - 1, ++j)
        if (j >= 0 && j < count) node[j] = at + wrapped(2, z + __builtin_ctzll(m));
    }
    __syncthreads();
    for (int k = tid; k < 64 * per; k += BS) {
      const int vtx = (k & 63) * per + (k >> 6);
      if (vtx >= nv) continue;
      SupportT<SW> sp;
      support_of(vtx, sp);
      const int lz = sp.lo[2] - o2, bit = lz & 63;
      const int r = (sp.lo[1] - o1 + s1 * (sp.lo[0] - o0)) * zw + (lz >> 6);
      double f0, f1, f2;
      spread_force(base + vtx, f0, f1, f2);
      const SW g0 = (SW)f0, g1 = (SW)f1, g2 = (SW)f2;
#pragma unroll
      for (int q = 0; q < 8; q += 2) {
        const int rq = r + ((q >> 2) * s1 + ((q >> 1) & 1)) * zw;
        // the node at z and the next place, z + 1
        const int e = (int)place[rq] - p0 + __popcll(mask[rq] & ((1ull << bit) - 1ull));
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          if ((unsigned)(e + h) >= (unsigned)count || sp.w[q + h] == SW(0)) continue;
          lds_add(&box[e + h], spread_term<R>((double)(g0 * sp.w[q + h]), L));
          lds_add(&box[cap + e + h], spread_term<R>((double)(g1 * sp.w[q + h]), L));
          lds_add(&box[2 * cap + e + h], spread_term<R>((double)(g2 * sp.w[q + h]), L));
        }
      }
    }
    __syncthreads();
    for (int j = tid; j < count; j += BS) {
      const double a = box[j], b = box[cap + j], c = box[2 * cap + j];
      box[j] = 0.0;  // zero for the next pass
      box[cap + j] = 0.0;
      box[2 * cap + j] = 0.0;
      const int64_t n = node[j];
      if (a != 0.0) atomic_add(&Fnext[n], (R)a);
      if (b != 0.0) atomic_add(&Fnext[S + n], (R)b);
      if (c != 0.0) atomic_add(&Fnext[2 * S + n], (R)c);
    }
    if (p0 + cap < total) __syncthreads();  // the sums are zero and the nodes free again
  }
}

template <typename R, int MODEL, int BS, bool STAGED, bool GPOS>
__global__ __launch_bounds__(BS) void k_cell_step(VertexDev V, TypeDev T, const int32_t* __restrict__ cells,
                                                  const int64_t* __restrict__ cell_base, const R* __restrict__ uf,
                                                  const uint8_t* __restrict__ type, LatticeDev L, R* __restrict__ Fnext,
                                                  const double* __restrict__ extra, double* __restrict__ scratch,
                                                  double f_limit, int flags, int box_nodes,
                                                  unsigned long long* wall_hits) {
  cell_step_body<R, MODEL, BS, STAGED, GPOS>(V, T, cell_base[cells[blockIdx.x]],
                                             V.box ? V.box + kBoxInts * (int64_t)cells[blockIdx.x] : nullptr, uf, type, L, Fnext, extra, scratch,
                                             f_limit, flags, box_nodes, wall_hits);
}

// cells of several independent cases in one launch, one workgroup per cell
template <typename R, int MODEL, int BS, bool STAGED, bool GPOS>
__global__ __launch_bounds__(BS) void k_cell_step_multi(const CellCase* __restrict__ cs, int box_nodes) {
  const CellCase& c = cs[blockIdx.x];
  cell_step_body<R, MODEL, BS, STAGED, GPOS>(c.V, c.T, c.base, c.box, (const R*)c.uf, c.type, c.L, (R*)c.Fnext, c.extra,
                                             c.scratch, c.f_limit, c.flags, box_nodes, c.wall_hits);
}

// Cells of several cases and meshes in one launch, one workgroup per cell, when
// there are no more of them than compute units: they run at the same time in any
// case, and three launches side by side cost the fork to two more streams and the
// join, 25 us of a step (three served cases 82 -> 62 us, 24 cases 361 -> 346).
// With more cells the largest mesh's LDS would keep the small ones' workgroups
// waiting.
template <typename R>
__global__ __launch_bounds__((all_block<R>())) void k_cell_step_all(const CellCase* __restrict__ cs) {
  const CellCase& c = cs[blockIdx.x];
  if (c.T.model == HC_MODEL_RBC)
    cell_step_body<R, HC_MODEL_RBC, all_block<R>(), true, false>(c.V, c.T, c.base, c.box, (const R*)c.uf, c.type, c.L,
                                                            (R*)c.Fnext, c.extra, c.scratch, c.f_limit, c.flags,
                                                            c.box_nodes, c.wall_hits);
  else if (c.T.model == HC_MODEL_PLT)
    cell_step_body<R, HC_MODEL_PLT, all_block<R>(), true, false>(c.V, c.T, c.base, c.box, (const R*)c.uf, c.type, c.L,
                                                            (R*)c.Fnext, c.extra, c.scratch, c.f_limit, c.flags,
                                                            c.box_nodes, c.wall_hits);
  else
    cell_step_body<R, HC_MODEL_WBC, all_block<R>(), true, false>(c.V, c.T, c.base, c.box, (const R*)c.uf, c.type, c.L,
                                                            (R*)c.Fnext, c.extra, c.scratch, c.f_limit, c.flags,
                                                            c.box_nodes, c.wall_hits);
}

// Cells of every type in one persistent launch: each workgroup takes the next
// entry of the queue (cell, type index; the types with the most vertices first)
// until the queue is empty.  RBC and platelet cells run the staged body, WBCs
// the one with positions in global memory; all share the launch's dynamic LDS.
template <typename R>
__global__ __launch_bounds__(kMixedBlock) void k_cell_step_mixed(
    VertexDev V, const TypeDev* __restrict__ types, MixedArgs A, const int2* __restrict__ queue, int nqueue,
    unsigned int* __restrict__ head, const int64_t* __restrict__ cell_base, const R* __restrict__ uf,
    const uint8_t* __restrict__ type, LatticeDev L, R* __restrict__ Fnext, const double* __restrict__ extra,
    double* __restrict__ scratch, double f_limit, unsigned long long* wall_hits) {
  __shared__ int slot;
  for (;;) {
    if (threadIdx.x == 0) slot = (int)atomicAdd(head, 1u);
    __syncthreads();
    const int q = slot;
    __syncthreads();  // every thread has read the slot before thread 0 takes the next one
    if (q >= nqueue) break;
    const int2 e = queue[q];
    const TypeDev& T = types[e.y];
    const int64_t base = cell_base[e.x];
    int* const box = V.box ? V.box + kBoxInts * (int64_t)e.x : nullptr;
    if (T.model == HC_MODEL_RBC)
      cell_step_body<R, HC_MODEL_RBC, kMixedBlock, true, false>(V, T, base, box, uf, type, L, Fnext, extra, scratch,
                                                                 f_limit, A.flags[e.y], A.box_nodes[e.y], wall_hits);
    else if (T.model == HC_MODEL_PLT)
      cell_step_body<R, HC_MODEL_PLT, kMixedBlock, true, false>(V, T, base, box, uf, type, L, Fnext, extra, scratch,
                                                                 f_limit, A.flags[e.y], A.box_nodes[e.y], wall_hits);
    else
      cell_step_body<R, HC_MODEL_WBC, kMixedBlock, false, true>(V, T, base, box, uf, type, L, Fnext, extra, scratch,
                                                                 f_limit, A.flags[e.y], A.box_nodes[e.y], wall_hits);
    __syncthreads();  // the next cell reuses the LDS
  }
}

}  // namespace

// Static LDS of one kernel instantiation (the reduction array grows with the block).
template <typename K>
static size_t static_lds(K kernel) {
  hipFuncAttributes a{};
  if (hipFuncGetAttributes(&a, reinterpret_cast<const void*>(kernel)) != hipSuccess) return 32768;
  return a.sharedSizeBytes;
}

// Lay out the dynamic LDS of one cell type for block size B and launch: staged
// (positions, velocities and a region shared by the mechanics and the spread's
// scratch) when it fits beside the kernel's static LDS, else positions plus as much
// scratch as fits; with positions in global memory only the scratch.
template <typename R, int M, int B>
static hipError_t launch_cell(hipStream_t s, const VertexDev& V, const TypeDev& T, const int32_t* cells, int ncells,
                              const int64_t* cell_base, const R* uf, const uint8_t* type, const LatticeDev& L, R* Fnext,
                              const double* extra, double* scratch, double f_limit, int flags, int box_bytes,
                              int lds_device, unsigned long long* wall_hits, CellPositions pos,
                              const CellCase* multi = nullptr) {
  static const size_t st_staged = std::max(static_lds(k_cell_step<R, M, B, true, false>),
                                           static_lds(k_cell_step_multi<R, M, B, true, false>));
  static const size_t st_plain = std::max(static_lds(k_cell_step<R, M, B, false, false>),
                                          static_lds(k_cell_step_multi<R, M, B, false, false>));
  // positions in global memory: 256 threads at most
  constexpr bool kGlobal = B <= 256;
  static const size_t st_gpos = kGlobal ? static_lds(k_cell_step<R, M, kGlobal ? B : 256, false, true>) : 0;
  if (pos == POS_GLOBAL && !kGlobal) return hipErrorInvalidConfiguration;
  const bool visc = (T.model != HC_MODEL_RBC) || (T.eta_m != 0.0);
  // the staged kernel's position scalar: float offsets in the FP32-shifted form
  const CellLdsPlan plan = cell_lds_layout(T.model, T.nv, visc, sizeof(MechT<R, true, false>), (size_t)box_bytes,
                                           (size_t)lds_device, st_staged, st_plain, st_gpos, pos);
  if (!plan.ok) return hipErrorInvalidConfiguration;
  const bool gpos = pos == POS_GLOBAL;
  const bool staged = plan.staged;
  const int box_nodes = plan.box_nodes;
  const size_t dyn = plan.dyn;
  if (multi) {
    if (gpos) return hipErrorInvalidValue;
    if (staged)
      hipLaunchKernelGGL((k_cell_step_multi<R, M, B, true, false>), dim3((unsigned)ncells), dim3(B), dyn, s, multi,
                         box_nodes);
    else
      hipLaunchKernelGGL((k_cell_step_multi<R, M, B, false, false>), dim3((unsigned)ncells), dim3(B), dyn, s, multi,
                         box_nodes);
    return hipGetLastError();
  }
  if (staged)
    hipLaunchKernelGGL((k_cell_step<R, M, B, true, false>), dim3((unsigned)ncells), dim3(B), dyn, s, V, T, cells,
                       cell_base, uf, type, L, Fnext, extra, scratch, f_limit, flags, box_nodes, wall_hits);
  else if (gpos)
    hipLaunchKernelGGL((k_cell_step<R, M, kGlobal ? B : 256, false, true>), dim3((unsigned)ncells), dim3(B), dyn, s, V,
                       T, cells, cell_base, uf, type, L, Fnext, extra, scratch, f_limit, flags, box_nodes, wall_hits);
  else
    hipLaunchKernelGGL((k_cell_step<R, M, B, false, false>), dim3((unsigned)ncells), dim3(B), dyn, s, V, T, cells,
                       cell_base, uf, type, L, Fnext, extra, scratch, f_limit, flags, box_nodes, wall_hits);
  return hipGetLastError();
}

template <typename R>
hipError_t launch_cell_step(hipStream_t s, const VertexDev& V, const TypeDev& T, const int32_t* cells, int ncells,
                            const int64_t* cell_base, const R* uf, const uint8_t* type, const LatticeDev& L,
                            R* Fnext, const double* extra, double* scratch, double f_limit, int flags, int box_bytes,
                            int lds_device, unsigned long long* wall_hits, int block, CellPositions pos) {
  if (ncells <= 0) return hipSuccess;
  // threads per cell for the RBC and WBC meshes: 256, 512 or 1024; a block whose
  // static LDS leaves too little room for the cell falls back to a smaller one
  hipError_t e = hipErrorInvalidConfiguration;
#define HC_CELL(M, B)                                                                                                \
  if (e == hipErrorInvalidConfiguration)                                                                             \
    e = launch_cell<R, M, B>(s, V, T, cells, ncells, cell_base, uf, type, L, Fnext, extra, scratch, f_limit, flags, \
                             box_bytes, lds_device, wall_hits, pos);
  switch (T.model) {
    case HC_MODEL_RBC:
      if (block >= 1024) HC_CELL(HC_MODEL_RBC, 1024)
      if (block >= 512) HC_CELL(HC_MODEL_RBC, 512)
      HC_CELL(HC_MODEL_RBC, 256)
      break;
    case HC_MODEL_PLT:
      if (block >= 256) HC_CELL(HC_MODEL_PLT, 256)
      HC_CELL(HC_MODEL_PLT, 64)
      break;
    case HC_MODEL_WBC:
      if (block >= 1024) HC_CELL(HC_MODEL_WBC, 1024)
      if (block >= 512) HC_CELL(HC_MODEL_WBC, 512)
      HC_CELL(HC_MODEL_WBC, 256)
      break;
    default:
      return hipErrorInvalidValue;
  }
#undef HC_CELL
  // a mesh whose positions do not fit the workgroup's LDS at any block (a
  // 2562-vertex WBC on a 64 KB device) keeps them in global memory
  if (e == hipErrorInvalidConfiguration && pos != POS_GLOBAL)
    return launch_cell_step<R>(s, V, T, cells, ncells, cell_base, uf, type, L, Fnext, extra, scratch, f_limit, flags,
                               box_bytes, lds_device, wall_hits, 256, POS_GLOBAL);
  return e;
}

// The persistent mixed launch: dynamic LDS for the largest need of the types
// present (staged RBC and platelet cells, WBCs with positions in global memory),
// each type's box filling what its layout leaves; `grid` workgroups.
template <typename R>
hipError_t launch_cell_step_mixed(hipStream_t s, const VertexDev& V, const TypeDev* d_types, const TypeDev* h_types,
                                  int ntypes, const int* flags, const int2* queue, int nqueue, unsigned int* head,
                                  int grid, const int64_t* cell_base, const R* uf, const uint8_t* type,
                                  const LatticeDev& L, R* Fnext, const double* extra, double* scratch, double f_limit,
                                  int box_bytes, int lds_device, unsigned long long* wall_hits) {
  if (nqueue <= 0) return hipSuccess;
  if (ntypes > kMaxMixedTypes || grid <= 0) return hipErrorInvalidValue;
  static const size_t st = static_lds(k_cell_step_mixed<R>);
  int model[kMaxMixedTypes], nv[kMaxMixedTypes];
  bool visc[kMaxMixedTypes];
  for (int t = 0; t < ntypes; ++t) {
    model[t] = h_types[t].model;
    nv[t] = h_types[t].nv;
    visc[t] = (h_types[t].model != HC_MODEL_RBC) || (h_types[t].eta_m != 0.0);
  }
  MixedArgs A{};
  size_t dyn = 0;
  for (size_t box : {(size_t)box_bytes, std::min((size_t)box_bytes, kLeastBox)})
    if (dyn == 0)
      dyn = mixed_lds_plan(ntypes, model, nv, visc, sizeof(MechT<R, true, false>), box, (size_t)lds_device, st,
                           A.box_nodes);
  if (dyn == 0) return hipErrorInvalidConfiguration;
  for (int t = 0; t < ntypes; ++t) A.flags[t] = flags[t];
  hipError_t e = launch_fill_zero<float>(s, reinterpret_cast<float*>(head), 1);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((k_cell_step_mixed<R>), dim3((unsigned)std::min(grid, nqueue)), dim3(kMixedBlock), dyn, s, V,
                     d_types, A, queue, nqueue, head, cell_base, uf, type, L, Fnext, extra, scratch, f_limit,
                     wall_hits);
  return hipGetLastError();
}

// Room for one mesh in the launch of all cells: its spread nodes, and the dynamic
// LDS it needs; false when it has to be launched by itself.
template <typename R>
bool cell_step_all_plan(const TypeDev& T, int box_bytes, int lds_device, int* box_nodes, size_t* dyn) {
  static const size_t st = static_lds(k_cell_step_all<R>);
  const bool visc = (T.model != HC_MODEL_RBC) || (T.eta_m != 0.0);
  const CellLdsPlan p = cell_lds_layout(T.model, T.nv, visc, sizeof(MechT<R, true, false>), (size_t)box_bytes,
                                        (size_t)lds_device, st, st, st, POS_LDS);
  if (!p.ok || !p.staged) return false;
  *box_nodes = p.box_nodes;
  *dyn = std::max(*dyn, p.dyn);
  return true;
}

template <typename R>
hipError_t launch_cell_step_all(hipStream_t s, const CellCase* cases, int ncells, size_t dyn) {
  if (ncells <= 0) return hipSuccess;
  hipLaunchKernelGGL((k_cell_step_all<R>), dim3((unsigned)ncells), dim3(all_block<R>()), dyn, s, cases);
  return hipGetLastError();
}

template <typename R>
hipError_t launch_cell_step_multi(hipStream_t s, const TypeDev& T, const CellCase* cases, int ncells, int box_bytes,
                                  int lds_device, int block) {
  if (ncells <= 0) return hipSuccess;
  const VertexDev V{};
  const LatticeDev L{};
  hipError_t e = hipErrorInvalidConfiguration;
#define HC_CELL(M, B)                                                                                             \
  if (e == hipErrorInvalidConfiguration)                                                                          \
    e = launch_cell<R, M, B>(s, V, T, nullptr, ncells, nullptr, nullptr, nullptr, L, nullptr, nullptr, nullptr, 0.0, \
                             0, box_bytes, lds_device, nullptr, POS_LDS, cases);
  switch (T.model) {
    case HC_MODEL_RBC:
      if (block >= 1024) HC_CELL(HC_MODEL_RBC, 1024)
      if (block >= 512) HC_CELL(HC_MODEL_RBC, 512)
      HC_CELL(HC_MODEL_RBC, 256)
      return e;
    case HC_MODEL_PLT:
      if (block >= 256) HC_CELL(HC_MODEL_PLT, 256)
      HC_CELL(HC_MODEL_PLT, 64)
      return e;
    case HC_MODEL_WBC:
      if (block >= 1024) HC_CELL(HC_MODEL_WBC, 1024)
      if (block >= 512) HC_CELL(HC_MODEL_WBC, 512)
      HC_CELL(HC_MODEL_WBC, 256)
      return e;
    default:
      return hipErrorInvalidValue;
  }
#undef HC_CELL
}

}  // namespace hcg
