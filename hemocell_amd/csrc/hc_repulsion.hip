// hc_repulsion.hip -- vertex binning and cell-cell repulsion on MI355X.
//
// Replaces (reference paths relative to the HemoCell tree):
//   HemoCellParticleField::update_pg           core/hemoCellParticleField.cpp:137-168
//   HemoCellParticleField::applyRepulsionForce core/hemoCellParticleField.cpp:677-743
//   populateBoundaryParticles / applyBoundaryRepulsionForce  :865-918
//
// Binning: every vertex gets the key of its nearest node, floor(x + 0.5) per
// axis (wrapped on periodic axes; vertices outside a non-periodic axis get the
// key N and no bin).  A node's vertices are counted with atomics, the first of
// them reserves a run of entries, every vertex copies its position, cell and id
// there, and each run is put into ascending vertex order, the order in which
// update_pg appends them.  The runs themselves lie in no particular order.  A
// final pass clears exactly the touched nodes again, so no per-step pass over
// all N nodes is needed.  Unlike the reference's fixed 10 slots per node, bins
// have no capacity limit.  (A radix sort of key and id before: eight merge
// launches of 6 us for 157k vertices, and the vertices' data gathered by id.)
//
// Forces: the reference walks every node l with itself and 13 forward
// neighbours m (a half stencil) and, for each ordered pair (i in bin l, j in
// bin m) of vertices of different cells closer than the cut-off, adds
// F = k (r_c / r) r_hat to i and subtracts it from j.  Here each vertex v
// gathers its own terms: it enumerates the nodes l whose half stencil reaches
// its node, in ascending node order, and within each (l, offset) visits the
// pairs in the reference's loop order.  The separation of the reversed pair is
// the exact negation of the forward one (IEEE subtraction, minimum image
// included), so the FP64 sum per vertex is formed from the same terms in the
// same order, without atomics.
#include "hc_launch.h"

namespace hcg {
namespace {

// the 14-offset half stencil of applyRepulsionForce, in its visiting order
__constant__ int kOff[14][3] = {{0, 0, 0}, {0, 0, 1}, {0, 1, 0}, {0, 1, 1},   {1, -1, -1}, {1, -1, 0}, {1, -1, 1},
                                {1, 0, -1}, {1, 0, 0}, {1, 0, 1}, {1, 1, -1}, {1, 1, 0},   {1, 1, 1},  {0, 1, -1}};

// node coordinate along an axis of size n: wrapped when periodic, -1 outside
__device__ __forceinline__ int wrap_axis(int64_t c, int n, int periodic) {
  if (c >= 0 && c < n) return (int)c;
  if (!periodic) return -1;
  int64_t m = c % n;
  if (m < 0) m += n;
  return (int)m;
}

__device__ __forceinline__ int64_t node_index(int x, int y, int z, const LatticeDev& L) {
  return (int64_t)z + (int64_t)L.nz * ((int64_t)y + (int64_t)L.ny * x);
}

// nearest-node key of vertex i (N when it is outside the domain or was removed by
// wall contact: such a vertex is in no bin and repels nothing)
__device__ __forceinline__ uint32_t vertex_key(const VertexDev& V, int64_t i, const LatticeDev& L, int c[3]) {
  const int dims[3] = {L.nx, L.ny, L.nz};
  bool inside = !(V.flag && (V.flag[i] & VFLAG_REMOVED));
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const double p = V.x[a * V.vs + i];
    if (!(fabs(p) < 1.0e15)) {
      inside = false;
      c[a] = -1;
      continue;
    }
    c[a] = wrap_axis((int64_t)floor(p + 0.5), dims[a], L.periodic[a]);
    inside &= c[a] >= 0;
  }
  return inside ? (uint32_t)node_index(c[0], c[1], c[2], L) : (uint32_t)L.N;
}

// the key of every vertex and its rank of arrival in its node's bin (counted in
// bins[key].y, zero between launches)
__global__ __launch_bounds__(256) void k_bin_count(VertexDev V, LatticeDev L, uint32_t* __restrict__ keys,
                                                   int32_t* __restrict__ ranks, int2* __restrict__ bins) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= V.n) return;
  int c[3];
  const uint32_t k = vertex_key(V, i, L, c);
  keys[i] = k;
  ranks[i] = k < (uint32_t)L.N ? atomicAdd(&bins[k].y, 1) : 0;
}

// [start, end) of every occupied node: its first vertex reserves the run, one
// atomic per workgroup (one per wavefront queued at the counter: 32 us for 157k
// vertices)
__global__ __launch_bounds__(256) void k_bin_reserve(const uint32_t* __restrict__ keys,
                                                     const int32_t* __restrict__ ranks, int64_t n, uint32_t N,
                                                     int2* __restrict__ bins, int* __restrict__ used) {
  __shared__ int sums[4];
  __shared__ int first_of_block;
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t k = p < n ? keys[p] : N;
  const bool first = k < N && ranks[p] == 0;
  const int count = first ? bins[k].y : 0;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int inc = count;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int y = __shfl_up(inc, o);
    if (lane >= o) inc += y;
  }
  if (lane == 63) sums[wave] = inc;
  __syncthreads();
  if (threadIdx.x == 0) {
    const int total = sums[0] + sums[1] + sums[2] + sums[3];
    first_of_block = total > 0 ? atomicAdd(used, total) : 0;
  }
  __syncthreads();
  int start = first_of_block + inc - count;
  for (int w = 0; w < wave; ++w) start += sums[w];
  if (first) bins[k] = make_int2(start, start + count);
}

__global__ __launch_bounds__(256) void k_bin_fill(VertexDev V, const uint32_t* __restrict__ keys,
                                                  const int32_t* __restrict__ ranks, uint32_t N,
                                                  const int32_t* __restrict__ vcell, const int2* __restrict__ bins,
                                                  BinEntry* __restrict__ entries) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= V.n) return;
  const uint32_t k = keys[i];
  if (k >= N) return;
  entries[bins[k].x + ranks[i]] = BinEntry{V.x[i], V.x[V.vs + i], V.x[2 * V.vs + i], (int32_t)i, vcell[i]};
}

// each run into ascending vertex order, by the thread of its first vertex: by
// insertion, long runs (collapsed cells) by heap sort.  A run whose vertices all
// belong to one cell is marked: its end is stored complemented.
__device__ void sift_down(BinEntry* e, int i, int n) {
  const BinEntry x = e[i];
  for (int k; (k = 2 * i + 1) < n; i = k) {
    if (k + 1 < n && e[k + 1].id > e[k].id) ++k;
    if (e[k].id <= x.id) break;
    e[i] = e[k];
  }
  e[i] = x;
}
__global__ __launch_bounds__(256) void k_bin_order(const uint32_t* __restrict__ keys, const int32_t* __restrict__ ranks,
                                                   int64_t n, uint32_t N, int2* __restrict__ bins,
                                                   BinEntry* __restrict__ entries) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n || ranks[p] != 0) return;
  const uint32_t k = keys[p];
  if (k >= N) return;
  const int2 b = bins[k];
  BinEntry* const e = entries + b.x;
  const int count = b.y - b.x;
  bool one = true;
  for (int i = 1; i < count; ++i) one = one && e[i].cell == e[0].cell;
  if (one) bins[k].y = ~b.y;
  if (count <= 16) {
    for (int i = 1; i < count; ++i) {
      const BinEntry x = e[i];
      int j = i;
      for (; j > 0 && e[j - 1].id > x.id; --j) e[j] = e[j - 1];
      if (j != i) e[j] = x;
    }
  } else {
    for (int i = count / 2 - 1; i >= 0; --i) sift_down(e, i, count);
    for (int i = count - 1; i > 0; --i) {
      const BinEntry x = e[0];
      e[0] = e[i];
      e[i] = x;
      sift_down(e, 0, i);
    }
  }
}

// the touched nodes empty again; vertices in no bin (outside the domain, removed,
// without a finite position) feel nothing
__global__ __launch_bounds__(256) void k_bin_clear(VertexDev V, const uint32_t* __restrict__ keys, uint32_t N,
                                                   int2* __restrict__ bins, int* __restrict__ used) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p == 0) *used = 0;
  if (p >= V.n) return;
  const uint32_t k = keys[p];
  if (k < N) {
    bins[k] = make_int2(0, 0);
  } else {
    V.frep[p] = 0.0;
    V.frep[V.vs + p] = 0.0;
    V.frep[2 * V.vs + p] = 0.0;
  }
}

// Boundary particles (populateBoundaryParticles, hemoCellParticleField.cpp:865-887):
// bounce-back nodes with a node that is not bounce-back among their 26
// neighbours; neighbours wrap on periodic axes and end at non-periodic faces.
__global__ void k_boundary_flags(const uint8_t* __restrict__ type, LatticeDev L, uint8_t* __restrict__ flags) {
  const int64_t n = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= L.N) return;
  uint8_t flag = 0;
  if (type && type[n] == HC_NODE_BOUNCEBACK) {
    const int z = (int)(n % L.nz);
    const int64_t t = n / L.nz;
    const int y = (int)(t % L.ny), x = (int)(t / L.ny);
    for (int dx = -1; dx <= 1 && !flag; ++dx) {
      const int xx = wrap_axis(x + dx, L.nx, L.periodic[0]);
      if (xx < 0) continue;
      for (int dy = -1; dy <= 1 && !flag; ++dy) {
        const int yy = wrap_axis(y + dy, L.ny, L.periodic[1]);
        if (yy < 0) continue;
        for (int dz = -1; dz <= 1 && !flag; ++dz) {
          const int zz = wrap_axis(z + dz, L.nz, L.periodic[2]);
          if (zz < 0) continue;
          if (type[node_index(xx, yy, zz, L)] != HC_NODE_BOUNCEBACK) flag = 1;
        }
      }
    }
  }
  flags[n] = flag;
}

// Wall repulsion (applyBoundaryRepulsionForce, hemoCellParticleField.cpp:889-918):
// every boundary particle b adds k (r_c / r) r_hat, r = x - b, to each vertex of
// the bins in its 3x3x3 neighbourhood closer than r_c.  Gathered per vertex: the
// boundary particles in the 3x3x3 neighbourhood of the vertex's own bin, in
// ascending x, y, z (the reference's order of boundary particles), the separation
// taken to the unwrapped node, i.e. the minimum image.  Overwrites fbr.
__global__ void k_boundary_repulsion(VertexDev V, LatticeDev L, const uint8_t* __restrict__ flags, double k_rep,
                                     double r_c) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= V.n) return;
  const int64_t vs = V.vs;
  const double p[3] = {V.x[i], V.x[vs + i], V.x[2 * vs + i]};
  double F0 = 0.0, F1 = 0.0, F2 = 0.0;
  const bool removed = V.flag && (V.flag[i] & VFLAG_REMOVED);
  if (!removed && fabs(p[0]) < 1.0e9 && fabs(p[1]) < 1.0e9 && fabs(p[2]) < 1.0e9) {
    const int64_t c0 = (int64_t)floor(p[0] + 0.5), c1 = (int64_t)floor(p[1] + 0.5), c2 = (int64_t)floor(p[2] + 0.5);
    for (int dx = -1; dx <= 1; ++dx) {
      const int xx = wrap_axis(c0 + dx, L.nx, L.periodic[0]);
      if (xx < 0) continue;
      for (int dy = -1; dy <= 1; ++dy) {
        const int yy = wrap_axis(c1 + dy, L.ny, L.periodic[1]);
        if (yy < 0) continue;
        for (int dz = -1; dz <= 1; ++dz) {
          const int zz = wrap_axis(c2 + dz, L.nz, L.periodic[2]);
          if (zz < 0 || !flags[node_index(xx, yy, zz, L)]) continue;
          const double d0 = p[0] - (double)(c0 + dx), d1 = p[1] - (double)(c1 + dy), d2 = p[2] - (double)(c2 + dz);
          const double dist = sqrt(d0 * d0 + d1 * d1 + d2 * d2);
          if (dist < r_c) {
            const double s = k_rep * (1 / (dist / r_c));
            F0 = F0 + s * (d0 / dist);
            F1 = F1 + s * (d1 / dist);
            F2 = F2 + s * (d2 / dist);
          }
        }
      }
    }
  }
  V.fbr[i] = F0;
  V.fbr[vs + i] = F1;
  V.fbr[2 * vs + i] = F2;
}

__global__ void k_vertex_bins(const VertexDev V, LatticeDev L, int64_t* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= V.n) return;
  int c[3];
  const uint32_t k = vertex_key(V, i, L, c);
  out[i] = k >= (uint32_t)L.N ? -1 : (int64_t)k;
}

struct Pos {
  double x, y, z;
};

// the minimum image of a separation along a periodic axis of size n: d - n
// floor(d / n + 1/2), which is d itself well inside half the axis
__device__ __forceinline__ double min_image(double d, double n) {
  return fabs(d) < 0.25 * n ? d : d - n * floor(d / n + 0.5);
}

// the repulsion term of vertex v from partner w (F on v), zero when excluded
__device__ __forceinline__ void pair_term(const Pos& pv, int cv, int v, const BinEntry& w, const LatticeDev& L,
                                          double k_rep, double r_c, double& a0, double& a1, double& a2) {
  if (w.id == v || w.cell == cv) return;
  double d0 = pv.x - w.x, d1 = pv.y - w.y, d2 = pv.z - w.z;
  if (L.periodic[0]) d0 = min_image(d0, (double)L.nx);
  if (L.periodic[1]) d1 = min_image(d1, (double)L.ny);
  if (L.periodic[2]) d2 = min_image(d2, (double)L.nz);
  const double dist = sqrt(d0 * d0 + d1 * d1 + d2 * d2);
  if (dist < r_c) {
    const double s = k_rep * (1 / (dist / r_c));
    a0 += s * (d0 / dist);
    a1 += s * (d1 / dist);
    a2 += s * (d2 / dist);
  }
}

// A vertex's terms come from the 27 nodes around its own: its own bin and the 13
// its half stencil reaches, and the 13 nodes l = c - off whose half stencil reaches
// its node, each once and in ascending node index.  Where no periodic axis has
// fewer than three nodes these 27 differ, and off is in the half stencil when
// (off.x, off.y, off.z) is lexicographically positive; ascending l is then
// ascending wrapped coordinates per axis, a rotation of the order inside the
// domain.  ANY_SIZE: also periodic axes of one or two nodes, by a sorted list.  It
// served every vertex beside a face before, and with the wavefronts it held up took
// 270 us for 157k vertices at 30% on 64 x 64 x 128 nodes (now 99 us).
// One thread per bin entry: neighbouring threads visit the same runs.
template <bool ANY_SIZE>
__global__ __launch_bounds__(256) void k_repulsion(VertexDev V, LatticeDev L, const int* __restrict__ used,
                                                   const int2* __restrict__ bins, const BinEntry* __restrict__ entries,
                                                   double k_rep, double r_c) {
  const int64_t p0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p0 >= (int64_t)*used) return;
  const BinEntry self = entries[p0];
  const int v = self.id, cv = self.cell;
  const Pos pv{self.x, self.y, self.z};
  const int dims[3] = {L.nx, L.ny, L.nz};
  const double px[3] = {self.x, self.y, self.z};
  int c[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) c[a] = wrap_axis((int64_t)floor(px[a] + 0.5), dims[a], L.periodic[a]);
  const int64_t key = node_index(c[0], c[1], c[2], L);
  double a0 = 0.0, a1 = 0.0, a2 = 0.0;
  auto visit = [&](const int2 b) {
    const int end = b.y < 0 ? ~b.y : b.y;
    for (int p = b.x; p < end; ++p) pair_term(pv, cv, v, entries[p], L, k_rep, r_c, a0, a1, a2);
  };
  // both ends in the vertex's own bin: for i in bin, for j in bin
  auto own = [&](const int2 b) {
    if (b.y < 0) return;  // no other cell
    for (int p = b.x; p < b.y; ++p) {
      if (entries[p].id == v) visit(b);
      else pair_term(pv, cv, v, entries[p], L, k_rep, r_c, a0, a1, a2);
    }
  };
  if constexpr (!ANY_SIZE) {
    // the nodes of the neighbours c - 1, c, c + 1 per axis, -1 outside the domain
    int side[3][3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const int n = dims[a], wrap = L.periodic[a] ? 0 : -1;
      side[a][0] = c[a] > 0 ? c[a] - 1 : (wrap < 0 ? -1 : n - 1);
      side[a][1] = c[a];
      side[a][2] = c[a] < n - 1 ? c[a] + 1 : wrap;
    }
    auto at = [&](int x, int y, int z) {
      const bool ok = (x | y | z) >= 0;
      return ok ? bins[node_index(x, y, z, L)] : make_int2(0, 0);
    };
    // Nearly every vertex around is of the vertex's own cell: a run marked as one
    // cell's is judged by its first entry's cell, read for all runs at once.
    auto visit_all = [&](auto& b) {
      constexpr int n = sizeof(b) / sizeof(int2);
      int cell[n];
#pragma unroll
      for (int o = 0; o < n; ++o) cell[o] = entries[b[o].y < 0 ? b[o].x : p0].cell;
#pragma unroll
      for (int o = 0; o < n; ++o)
        if (b[o].x != b[o].y && !(b[o].y < 0 && cell[o] == cv)) visit(b[o]);
    };
    // places of the ascending order: i of the x plane, j and k of y and z
    const int rx = c[0] == 0 && L.periodic[0];
    int yo[3], zo[3];
    const int ry = !L.periodic[1] ? 0 : c[1] == 0 ? 1 : c[1] == dims[1] - 1 ? 2 : 0;
    const int rz = !L.periodic[2] ? 0 : c[2] == 0 ? 1 : c[2] == dims[2] - 1 ? 2 : 0;
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      yo[j] = j + ry < 3 ? j + ry : j + ry - 3;
      zo[j] = j + rz < 3 ? j + rz : j + rz - 3;
    }
    auto pick = [](const int (&v)[3], int j) { return j == 0 ? v[0] : j == 1 ? v[1] : v[2]; };
    // the nodes l of the plane l.x = side[0][xi], those below the vertex's node or
    // those above it
    auto plane = [&](int xi, bool above) {
      int2 b[9];
#pragma unroll
      for (int j = 0; j < 3; ++j)
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          const int yi = yo[j], zi = zo[k];
          const int x = xi ? side[0][1] : side[0][0], y = pick(side[1], yi), z = pick(side[2], zi);
          // off = c - l positive; l against c in node order
          const bool reaches = xi == 0 || yi == 0 || (yi == 1 && zi == 0);
          const bool up = x != c[0] ? x > c[0] : y != c[1] ? y > c[1] : z > c[2];
          b[3 * j + k] = reaches && up == above ? at(x, y, z) : make_int2(0, 0);
        }
      visit_all(b);
    };
    const bool first_is_up = rx != 0;  // the plane c.x - 1 is the domain's last
    // below: the plane c.x - 1 (unless wrapped), then the vertex's own
    if (!first_is_up) plane(0, false);
    plane(1, false);
    const int2 self_bin = bins[key];
    const int x1 = side[0][2], y0 = side[1][0], y1 = side[1][2], z0 = side[2][0], z1 = side[2][2];
    int2 f[13] = {at(c[0], c[1], z1), at(c[0], y1, c[2]), at(c[0], y1, z1), at(x1, y0, z0),   at(x1, y0, c[2]),
                  at(x1, y0, z1),     at(x1, c[1], z0),   at(x1, c[1], c[2]), at(x1, c[1], z1), at(x1, y1, z0),
                  at(x1, y1, c[2]),   at(x1, y1, z1),     at(c[0], y1, z0)};
    own(self_bin);
    visit_all(f);
    if (ry || rz) plane(1, true);
    if (first_is_up) plane(0, true);
  } else {
    // the nodes l whose half stencil reaches this node, ascending and each once, and for each every offset that joins it with this node
    int64_t cand[14];
    int nc = 0;
    for (int o = 0; o < 14; ++o) {
      int l3[3];
      bool ok = true;
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        l3[a] = wrap_axis((int64_t)c[a] - kOff[o][a], dims[a], L.periodic[a]);
        ok &= l3[a] >= 0;
      }
      if (!ok) continue;
      const int64_t l = node_index(l3[0], l3[1], l3[2], L);
      bool dup = false;
      for (int q = 0; q < nc; ++q) dup |= cand[q] == l;
      if (dup) continue;
      // insertion into the ascending list
      int q = nc++;
      while (q > 0 && cand[q - 1] > l) {
        cand[q] = cand[q - 1];
        --q;
      }
      cand[q] = l;
    }
    for (int q = 0; q < nc; ++q) {
      const int64_t l = cand[q];
      const int2 bl = bins[l];
      if (bl.x == bl.y) continue;
      const int lx = (int)(l / ((int64_t)L.ny * L.nz));
      const int ly = (int)((l / L.nz) % L.ny);
      const int lz = (int)(l % L.nz);
      for (int o = 0; o < 14; ++o) {
        const int mx = wrap_axis((int64_t)lx + kOff[o][0], L.nx, L.periodic[0]);
        const int my = wrap_axis((int64_t)ly + kOff[o][1], L.ny, L.periodic[1]);
        const int mz = wrap_axis((int64_t)lz + kOff[o][2], L.nz, L.periodic[2]);
        if (mx < 0 || my < 0 || mz < 0) continue;
        const int64_t m = node_index(mx, my, mz, L);
        if (l == key && m == key) own(bl);
        else if (l == key) visit(bins[m]);
        else if (m == key) visit(bl);
      }
    }
  }
  V.frep[v] = a0;
  V.frep[V.vs + v] = a1;
  V.frep[2 * V.vs + v] = a2;
}

}  // namespace

hipError_t launch_repulsion(hipStream_t s, const VertexDev& V, const LatticeDev& L, const RepulsionBufs& B,
                            double k_rep, double r_c) {
  if (V.n <= 0) return hipSuccess;
  if (V.n > INT32_MAX || L.N >= (int64_t)UINT32_MAX) return hipErrorInvalidValue;
  const dim3 grid((unsigned)((V.n + 255) / 256)), block(256);
  const uint32_t N = (uint32_t)L.N;
  hipLaunchKernelGGL(k_bin_count, grid, block, 0, s, V, L, B.keys, B.ranks, B.bins);
  hipLaunchKernelGGL(k_bin_reserve, grid, block, 0, s, B.keys, B.ranks, V.n, N, B.bins, B.used);
  hipLaunchKernelGGL(k_bin_fill, grid, block, 0, s, V, B.keys, B.ranks, N, B.vcell, B.bins, B.entries);
  hipLaunchKernelGGL(k_bin_order, grid, block, 0, s, B.keys, B.ranks, V.n, N, B.bins, B.entries);
  const bool distinct =
      (!L.periodic[0] || L.nx > 2) && (!L.periodic[1] || L.ny > 2) && (!L.periodic[2] || L.nz > 2);
  hipLaunchKernelGGL(distinct ? k_repulsion<false> : k_repulsion<true>, grid, block, 0, s, V, L, B.used, B.bins,
                     B.entries, k_rep, r_c);
  hipLaunchKernelGGL(k_bin_clear, grid, block, 0, s, V, B.keys, N, B.bins, B.used);
  return hipGetLastError();
}

hipError_t launch_boundary_flags(hipStream_t s, const uint8_t* type, const LatticeDev& L, uint8_t* flags) {
  if (L.N <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_boundary_flags, dim3((unsigned)((L.N + 255) / 256)), dim3(256), 0, s, type, L, flags);
  return hipGetLastError();
}

hipError_t launch_boundary_repulsion(hipStream_t s, const VertexDev& V, const LatticeDev& L, const uint8_t* flags,
                                     double k, double r_c) {
  if (V.n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_boundary_repulsion, dim3((unsigned)((V.n + 255) / 256)), dim3(256), 0, s, V, L, flags, k, r_c);
  return hipGetLastError();
}

hipError_t launch_vertex_bins(hipStream_t s, const VertexDev& V, const LatticeDev& L, int64_t* out) {
  if (V.n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_vertex_bins, dim3((unsigned)((V.n + 255) / 256)), dim3(256), 0, s, V, L, out);
  return hipGetLastError();
}

}  // namespace hcg
