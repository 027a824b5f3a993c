// fem.hip — Newton gradient, energies and strain of the cloth step (FP64).
#include "elements.h"

namespace cloth {

// One thread per vertex: evalInternal gradient at the vertex (membrane in
// triangle order, then bending in hinge order), plus inertia
// M (x - yHat) / h^2 (newton.ts:116-120), plus the contact gradient when
// present (:122-124), pins zeroed (:126); grid-reduces sum g^2 (:127).
__global__ void __launch_bounds__(kBlock) k_gradient(DMesh me, DMat mat, const double* __restrict__ x,
                                                     const double* __restrict__ yhat, double inv_h2,
                                                     const double* __restrict__ ceg, double* __restrict__ g,
                                                     jsm::dd* partials) {
  jsm::dd acc2 = jsm::dd_zero();
  for (uint32_t v = blockIdx.x * blockDim.x + threadIdx.x; v < me.n; v += gridDim.x * blockDim.x) {
    double acc[3];
    internal_grad_vertex(me, mat, x, v, acc);
    const double m = me.mass[v];
    const bool pinned = me.pinmask[v] != 0;
#pragma unroll
    for (int k = 0; k < 3; k++) {
      const size_t i = (size_t)v * 3 + k;
      double gi = m * (x[i] - yhat[i]) * inv_h2 + acc[k];
      if (ceg) gi += ceg[i];
      if (pinned) gi = 0;
      g[i] = gi;
      jsm::dd_add_prod(acc2, gi, gi);
    }
  }
  block_partial_dd<kBlock>(acc2, partials);
}

// The same gradient with 16 lanes per vertex: the lanes evaluate the vertex's
// triangle corners, then the components of its hinges' gradients (two dihedral
// energies each), and lane i < 3 adds component i in triangle and hinge order.
// One thread evaluates 72 dihedrals of an interior vertex one after the other,
// 84 us whatever the mesh's size up to 65,536 vertices (95 us there; 250 us for
// 262,144, where the FP64 units are full); here the chain is 6 dihedrals, 17 us
// for 91 as for 2,000 vertices, but lanes idle at the ends of the rounds: 116 us
// for 65,536.  The two meet near 45,000 vertices.
constexpr uint32_t kGradLanes = 16;
constexpr uint32_t kGradWideMax = 32768;

__global__ void __launch_bounds__(kBlock) k_gradient_wide(DMesh me, DMat mat, const double* __restrict__ x,
                                                          const double* __restrict__ yhat, double inv_h2,
                                                          const double* __restrict__ ceg, double* __restrict__ g,
                                                          jsm::dd* partials) {
  constexpr uint32_t kVerts = kBlock / kGradLanes;
  jsm::dd acc2 = jsm::dd_zero();
  const uint32_t sub = threadIdx.x % kGradLanes;
  const int base = (int)(threadIdx.x % kWave - sub);
  // uniform trip count; the groups past the last vertex take part idle
  for (uint32_t v0 = blockIdx.x * kVerts; v0 < me.n; v0 += gridDim.x * kVerts) {
    const uint32_t v = v0 + threadIdx.x / kGradLanes;
    const bool valid = v < me.n;
    double acc = 0;  // component `sub`
    const uint32_t tb = valid ? me.vt_off[v] : 0, te = valid ? me.vt_off[v + 1] : 0;
    for (uint32_t r = tb; r < te; r += kGradLanes) {
      double gc[3] = {0, 0, 0};
      if (r + sub < te) {
        const uint32_t rec = me.vt_rec[r + sub];
        const uint32_t t = rec >> 2;
        double x0[3], x1[3], x2[3];
        ld3(x, me.idx[(size_t)t * 3], x0);
        ld3(x, me.idx[(size_t)t * 3 + 1], x1);
        ld3(x, me.idx[(size_t)t * 3 + 2], x2);
        tri_grad_corner(tri_state(x0, x1, x2, me.inv_dm + (size_t)t * 4), me.area[t], mat, rec & 3, gc);
      }
      const uint32_t cnt = min(kGradLanes, te - r);
      for (uint32_t q = 0; q < cnt; q++) {
        const double c0 = __shfl(gc[0], base + (int)q, kWave), c1 = __shfl(gc[1], base + (int)q, kWave),
                     c2 = __shfl(gc[2], base + (int)q, kWave);
        acc += sub == 0 ? c0 : sub == 1 ? c1 : c2;
      }
    }
    if (mat.kb > 0) {
      const uint32_t hb = valid ? me.vh_off[v] : 0, tasks = valid ? (me.vh_off[v + 1] - hb) * 3 : 0;
      for (uint32_t r = 0; r < tasks; r += kGradLanes) {
        double d = 0;
        if (r + sub < tasks) {
          const uint32_t hh = me.vh_rec[hb + (r + sub) / 3] >> 2;
          const int i = (int)((r + sub) % 3);
          uint32_t vs[4];
          double P[4][3];
#pragma unroll
          for (int s = 0; s < 4; s++) {
            vs[s] = me.hv[(size_t)hh * 4 + s];
            ld3(x, vs[s], P[s]);
          }
          d = hinge_fd(vs, P, v, i, x[(size_t)v * 3 + i], me.hrest[hh], me.hlen[hh], me.hasum[hh], mat.kb);
        }
        const uint32_t cnt = min(kGradLanes, tasks - r);
        for (uint32_t q = 0; q < cnt; q++) {
          const double t = __shfl(d, base + (int)q, kWave);
          if ((r + q) % 3 == sub) acc += t;
        }
      }
    }
    if (valid && sub < 3) {
      const size_t i = (size_t)v * 3 + sub;
      const double m = me.mass[v];
      double gi = m * (x[i] - yhat[i]) * inv_h2 + acc;
      if (ceg) gi += ceg[i];
      if (me.pinmask[v] != 0) gi = 0;
      g[i] = gi;
      jsm::dd_add_prod(acc2, gi, gi);
    }
  }
  block_partial_dd<kBlock>(acc2, partials);
}

void launch_gradient(hipStream_t st, const DMesh& me, const DMat& mat, const double* x, const double* yhat,
                     double inv_h2, const double* ceg, double* g, jsm::dd* partials, double* out_sumsq) {
  const bool wide = me.n <= kGradWideMax;
  const unsigned grid = wide ? red_grid((size_t)me.n * kGradLanes) : red_grid(me.n);
  hipLaunchKernelGGL(wide ? k_gradient_wide : k_gradient, dim3(grid), dim3(kBlock), 0, st, me, mat, x, yhat, inv_h2,
                     ceg, g, partials);
  CS_LAUNCH_CHECK();
  FinishJobs f{};
  f.j[0] = FinishJob{partials, grid, FIN_DD, 0, out_sumsq};
  launch_finish(st, f, 1);
}

// totalEnergy (newton.ts:76-88) minus the contact merit term: inertia sum
// over DOFs and internalEnergyOnly (fem.ts:56-75) over triangles then hinges,
// each returned correctly rounded.
__global__ void __launch_bounds__(kBlock) k_energy(DMesh me, DMat mat, const double* __restrict__ x,
                                                   const double* __restrict__ yhat, double h,
                                                   jsm::dd* partials) {
  jsm::dd ein = jsm::dd_zero(), eint = jsm::dd_zero();
  const size_t n3 = (size_t)me.n * 3;
  const size_t nh = mat.kb > 0 ? me.nh : 0;
  const size_t total = n3 + me.m + nh;
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < total; i += (size_t)gridDim.x * blockDim.x) {
    if (i < n3) {
      const double m = me.mass[i / 3];
      const double d = x[i] - yhat[i];
      jsm::dd_add(ein, 0.5 * m * d * d / (h * h));
    } else if (i < n3 + me.m) {
      const size_t t = i - n3;
      double x0[3], x1[3], x2[3];
      ld3(x, me.idx[t * 3], x0);
      ld3(x, me.idx[t * 3 + 1], x1);
      ld3(x, me.idx[t * 3 + 2], x2);
      const TriState s = tri_state(x0, x1, x2, me.inv_dm + t * 4);
      jsm::dd_add(eint, tri_energy(s, me.area[t], mat));
    } else {
      const size_t hh = i - n3 - me.m;
      double P[4][3];
      for (int s = 0; s < 4; s++) ld3(x, me.hv[hh * 4 + s], P[s]);
      jsm::dd_add(eint, hinge_energy4(P, me.hrest[hh], me.hlen[hh], me.hasum[hh], mat.kb));
    }
  }
  block_partial_dd<kBlock>(ein, partials);
  block_partial_dd<kBlock>(eint, partials + kMaxRedBlocks);
}

void launch_energy(hipStream_t st, const DMesh& me, const DMat& mat, const double* x, const double* yhat,
                   double h, jsm::dd* partials, double* out2) {
  const size_t total = (size_t)me.n * 3 + me.m + me.nh;
  const unsigned grid = red_grid(total);
  hipLaunchKernelGGL(k_energy, dim3(grid), dim3(kBlock), 0, st, me, mat, x, yhat, h, partials);
  CS_LAUNCH_CHECK();
  FinishJobs f{};
  f.j[0] = FinishJob{partials, grid, FIN_DD, 0, out2};
  f.j[1] = FinishJob{partials + kMaxRedBlocks, grid, FIN_DD, 0, out2 + 1};
  launch_finish(st, f, 2);
}

// maxStrain (fem.ts:37): Math.max over |E00|, |E11|, |E01| of every triangle.
__global__ void __launch_bounds__(kBlock) k_max_strain(DMesh me, const double* __restrict__ x, double* partials) {
  double mx = 0;
  for (uint32_t t = blockIdx.x * blockDim.x + threadIdx.x; t < me.m; t += gridDim.x * blockDim.x) {
    double x0[3], x1[3], x2[3];
    ld3(x, me.idx[(size_t)t * 3], x0);
    ld3(x, me.idx[(size_t)t * 3 + 1], x1);
    ld3(x, me.idx[(size_t)t * 3 + 2], x2);
    const TriState s = tri_state(x0, x1, x2, me.inv_dm + (size_t)t * 4);
    mx = jsm::jmax(jsm::jmax(jsm::jmax(mx, jsm::fabs_(s.E00)), jsm::fabs_(s.E11)), jsm::fabs_(s.E01));
  }
  block_partial_ext<kBlock, JsMax>(mx, partials);
}

void launch_max_strain(hipStream_t st, const DMesh& me, const double* x, double* partials, double* out) {
  const unsigned grid = red_grid(me.m);
  hipLaunchKernelGGL(k_max_strain, dim3(grid), dim3(kBlock), 0, st, me, x, partials);
  CS_LAUNCH_CHECK();
  FinishJobs f{};
  f.j[0] = FinishJob{partials, grid, FIN_JSMAX, 1, out};
  launch_finish(st, f, 1);
}

}  // namespace cloth
