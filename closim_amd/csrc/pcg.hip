// pcg.hip — device-resident PCG of the Newton step (pcg.ts:11-95) in FP64.
//
// Per iteration three kernels; each writes block partials of its dot
// products and the next kernel merges them (fixed order, every block the
// same bits), so no scalar ever makes a host round trip or needs a fence:
//   k_hvp     [merge |p|^2 -> FD step h] Ap = hvpFull(p) (newton.ts:135-146),
//             pins zeroed; partials of p.Ap
//   k_update  [merge p.Ap -> breakdown test, alpha] x += alpha p,
//             r -= alpha Ap, z = M^-1 r; partials of r.r and r.z
//   k_dir     [merge r.r -> residual test; r.z -> beta] p = z + beta p;
//             partials of p.p
// A `done` latch turns the remaining launches of a converged solve into
// no-ops, which is exactly the reference's early return.  Block 0 records
// decisions; every block takes them from the same merged values.
#include "coop.h"
#include "elements.h"
#include "pcg.h"
#include "schwarz.h"
#include "vsum.h"

namespace cloth {

enum { PART_BB = 0, PART_RR = 1, PART_RZ = 2, PART_PP = 3, PART_PAP = 4 };

__device__ __forceinline__ jsm::dd* part(const PcgArgs& a, int which) {
  return a.partials + (size_t)which * kMaxRedBlocks;
}

// dd_c = kappa max(b'', 0) (J_c . p) of active contact c (distJvp,
// contact-assembly.ts:395-414, scaled as in applyHvp :376-386).
__device__ __forceinline__ double contact_dd(const DContactHvp& H, uint32_t ci, const double* p) {
  if (!H.inr[ci]) return 0.0;
  const Frozen& c = H.act[ci];
  double j;
  if (c.kind == 2) {
    j = p[(size_t)c.p * 3 + 1];
  } else if (c.kind == 0) {
    const size_t q = c.p;
    j = c.nx * p[q * 3] + c.ny * p[q * 3 + 1] + c.nz * p[q * 3 + 2];
    const double ws[3] = {c.w0, c.w1, c.w2};
    const int vs[3] = {c.a, c.b, c.c};
    for (int k = 0; k < 3; k++) {
      if (vs[k] < 0) continue;
      const size_t r = vs[k];
      j -= ws[k] * (c.nx * p[r * 3] + c.ny * p[r * 3 + 1] + c.nz * p[r * 3 + 2]);
    }
  } else {
    const double ws[4] = {c.w0, c.w1, c.w2, c.w3};
    const int vs[4] = {c.a, c.b, c.c, c.d};
    j = 0;
    for (int k = 0; k < 4; k++) {
      if (vs[k] < 0) continue;
      const size_t r = vs[k];
      j += ws[k] * (c.nx * p[r * 3] + c.ny * p[r * 3 + 1] + c.nz * p[r * 3 + 2]);
    }
  }
  return H.coeff[ci] * j;
}

__global__ void k_dot(const double* __restrict__ a, const double* __restrict__ b, size_t n, jsm::dd* partials);

// One incident triangle corner: what does not change during a solve.
struct HvpCorner {
  uint32_t i0, i1, i2;
  int corner;
  double x0[3], x1[3], x2[3], area;
  float inv[4];
};
__device__ __forceinline__ void load_corner(const PcgArgs& a, uint4 cr, HvpCorner& c) {
  const uint32_t t = cr.w >> 2;
  c.corner = cr.w & 3;
  c.i0 = cr.x;
  c.i1 = cr.y;
  c.i2 = cr.z;
  ld3(a.x, c.i0, c.x0); ld3(a.x, c.i1, c.x1); ld3(a.x, c.i2, c.x2);
  const float* inv = a.me.inv_dm + (size_t)t * 4;
  c.inv[0] = inv[0]; c.inv[1] = inv[1]; c.inv[2] = inv[2]; c.inv[3] = inv[3];
  c.area = a.me.area[t];
}

// Contribution of one incident triangle corner to the membrane HVP at the
// vertex: analytic, or the two gradient corners of the FD operator.
__device__ __forceinline__ void hvp_corner(const PcgArgs& a, const HvpCorner& c, const double* p, double h, double* g0,
                                           double* g1) {
  double p0[3], p1[3], p2[3];
  ld3(p, c.i0, p0); ld3(p, c.i1, p1); ld3(p, c.i2, p2);
  const double *x0 = c.x0, *x1 = c.x1, *x2 = c.x2;
  if (a.hvp_mode == HVP_FD) {
    // membraneHvp (fem.ts:108-130): gradients at x + h p and x - h p
    double xp0[3], xp1[3], xp2[3], xm0[3], xm1[3], xm2[3];
#pragma unroll
    for (int i = 0; i < 3; i++) {
      xp0[i] = x0[i] + h * p0[i]; xm0[i] = x0[i] - h * p0[i];
      xp1[i] = x1[i] + h * p1[i]; xm1[i] = x1[i] - h * p1[i];
      xp2[i] = x2[i] + h * p2[i]; xm2[i] = x2[i] - h * p2[i];
    }
    const TriState sp = tri_state(xp0, xp1, xp2, c.inv);
    tri_grad_corner(sp, c.area, a.mat, c.corner, g0);
    const TriState sm = tri_state(xm0, xm1, xm2, c.inv);
    tri_grad_corner(sm, c.area, a.mat, c.corner, g1);
  } else {
    const TriState s = tri_state(x0, x1, x2, c.inv);
    tri_hvp_corner(s, p0, p1, p2, c.area, a.mat, c.corner, g0, a.psd != 0);
    g1[0] = g1[1] = g1[2] = 0;
  }
}

// One contact incidence entry's term at the vertex (applyHvp's addDistGrad),
// g = the contact's dd_c.
__device__ __forceinline__ bool contact_term(const DContactHvp& H, uint32_t ent, double g, double* c) {
  const uint32_t ci = ent >> 3;
  const int slot = ent & 7;
  if (g == 0) return false;
  const Frozen& f = H.act[ci];
  if (f.kind == 2) {
    c[0] = 0; c[1] = g; c[2] = 0;
  } else if (f.kind == 0) {
    if (slot == 0) {
      c[0] = g * f.nx; c[1] = g * f.ny; c[2] = g * f.nz;
    } else {
      const double w = slot == 1 ? f.w0 : slot == 2 ? f.w1 : f.w2;
      c[0] = -g * w * f.nx; c[1] = -g * w * f.ny; c[2] = -g * w * f.nz;
    }
  } else {
    const double w = slot == 0 ? f.w0 : slot == 1 ? f.w1 : slot == 2 ? f.w2 : f.w3;
    c[0] = g * w * f.nx; c[1] = g * w * f.ny; c[2] = g * w * f.nz;
  }
  return true;
}

constexpr int kLanesPerVertex = 8;
constexpr int kVertsPerBlock = kBlock / kLanesPerVertex;

// hvpFull at vertex v: M p / h^2 + H_membrane p (+ contact), unfiltered.
// The 8 lanes of a vertex group evaluate up to 8 incident corners at once; lane 0 of the group adds them in list order, so
// the sums are the reference's element-order sums bit for bit.
__device__ __forceinline__ void hvp_vertex8(const PcgArgs& a, uint32_t v, bool valid, const double* __restrict__ p,
                                            double h, double* out) {
  const DMesh& me = a.me;
  const int sub = threadIdx.x % kLanesPerVertex;
  const int base = (threadIdx.x % kWave) - sub;
  double acc0[3] = {0, 0, 0}, acc1[3] = {0, 0, 0};
  const uint32_t b = valid ? me.vt_off[v] : 0, e = valid ? me.vt_off[v + 1] : 0;
  // rounds of 8 corners; the round count is uniform within the group
  for (uint32_t r0 = b; r0 < e; r0 += kLanesPerVertex) {
    double g0[3] = {0, 0, 0}, g1[3] = {0, 0, 0};
    const uint32_t q = r0 + sub;
    if (q < e) {
      HvpCorner c;
      load_corner(a, me.vt_corner[q], c);
      hvp_corner(a, c, p, h, g0, g1);
    }
    const uint32_t cnt = min((uint32_t)kLanesPerVertex, e - r0);
    for (uint32_t j = 0; j < cnt; j++) {
#pragma unroll
      for (int i = 0; i < 3; i++) {
        acc0[i] += __shfl(g0[i], base + (int)j, kWave);
        acc1[i] += __shfl(g1[i], base + (int)j, kWave);
      }
    }
  }
  double Hp[3];
  if (a.hvp_mode == HVP_FD) {
#pragma unroll
    for (int i = 0; i < 3; i++) Hp[i] = (acc0[i] - acc1[i]) / (2 * h);
  } else {
    Hp[0] = acc0[0]; Hp[1] = acc0[1]; Hp[2] = acc0[2];
  }
  const double m = valid ? (double)me.mass[v] : 0.0;
#pragma unroll
  for (int i = 0; i < 3; i++) out[i] = m * (valid ? p[(size_t)v * 3 + i] : 0.0) * a.inv_h2 + Hp[i];
  if (a.contact.act && a.contact.nv && valid) {
    // applyHvp (contact-assembly.ts:371-392): cHp summed per vertex in list
    // order by k_contact_vsum, then out += cHp (vsum holds the sums of this
    // HVP only while the active set has incidence entries: nv > 0)
    out[0] += a.contact.vsum[(size_t)v * 3];
    out[1] += a.contact.vsum[(size_t)v * 3 + 1];
    out[2] += a.contact.vsum[(size_t)v * 3 + 2];
  }
}

// applyHvp's contact part (out.fill(0), then addDistGrad per active contact
// in list order, skipping dd == 0) in two passes: every incidence entry's
// term in parallel (a skipped entry stores +0, which leaves a sum that
// started at +0 unchanged), then one thread per contact vertex and component
// adds its entries in list order.
__global__ void __launch_bounds__(kBlock) k_contact_terms(DContactHvp H, const double* __restrict__ p,
                                                          const int32_t* done) {
  if (block_latched(done)) return;
  const uint32_t e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= H.E) return;
  double t[3] = {0, 0, 0};
  const uint32_t ent = H.v_ent[e];
  if (!contact_term(H, ent, contact_dd(H, ent >> 3, p), t)) t[0] = t[1] = t[2] = 0;
  H.term[(size_t)e * 3] = t[0];
  H.term[(size_t)e * 3 + 1] = t[1];
  H.term[(size_t)e * 3 + 2] = t[2];
}

__global__ void __launch_bounds__(kBlock) k_contact_vsum(DContactHvp H, const int32_t* done) {
  if (block_latched(done)) return;
  const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= H.nv * 3) return;
  const uint32_t v = H.cverts[t / 3];
  const int q = t % 3;
  H.vsum[(size_t)v * 3 + q] = ordered_sum<3, 0>(H.term + q, H.v_off[v], H.v_off[v + 1], 0.0);
}

// The same where vertices have many entries (use_vertex_groups): dd_c once
// per contact, then k_vertex_sums.
__global__ void __launch_bounds__(kBlock) k_contact_dd(DContactHvp H, const double* __restrict__ p,
                                                       const int32_t* done) {
  if (block_latched(done)) return;
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < H.C) H.dd[i] = contact_dd(H, i, p);
}

struct HvpSums {
  static constexpr bool kPair = false;
  DContactHvp H;
  const int32_t* done;
  __device__ bool skip() const { return block_latched(done); }
  __device__ double init(uint32_t, int) const { return 0.0; }
  __device__ void term(uint32_t e, double* t) const {
    const uint32_t ent = H.v_ent[e];
    if (!contact_term(H, ent, H.dd[ent >> 3], t)) t[0] = t[1] = t[2] = 0;
  }
  __device__ void store(uint32_t v, int q, double s) const { H.vsum[(size_t)v * 3 + q] = s; }
};

// z = M^-1 r at vertex v (Jacobi with the diag > 1e-12 guard, or 3x3 block).
__device__ __forceinline__ void precond_vertex(const PcgArgs& a, uint32_t v, const double* r3, double* z3) {
  if (a.precond == PRE_BLOCK) {
    const double* f = a.binv + (size_t)v * 9;
    z3[0] = f[0] * r3[0] + f[1] * r3[1] + f[2] * r3[2];
    z3[1] = f[3] * r3[0] + f[4] * r3[1] + f[5] * r3[2];
    z3[2] = f[6] * r3[0] + f[7] * r3[1] + f[8] * r3[2];
  } else {
#pragma unroll
    for (int i = 0; i < 3; i++) {
      const double d = a.diag[(size_t)v * 3 + i];
      z3[i] = d > 1e-12 ? r3[i] / d : r3[i];
    }
  }
}

__global__ void __launch_bounds__(kBlock) k_pcg_init(PcgArgs a) {
  jsm::dd rz = jsm::dd_zero(), bb = jsm::dd_zero(), rr = jsm::dd_zero(), pp = jsm::dd_zero();
  for (uint32_t v = blockIdx.x * blockDim.x + threadIdx.x; v < a.me.n; v += gridDim.x * blockDim.x) {
    const bool pinned = a.me.pinmask[v] != 0;
    double r3[3], z3[3];
#pragma unroll
    for (int i = 0; i < 3; i++) {
      const size_t j = (size_t)v * 3 + i;
      const double bi = a.b[j];
      jsm::dd_add_prod(bb, bi, bi);
      r3[i] = pinned ? 0.0 : bi;
      a.sol[j] = 0.0;
      a.r[j] = r3[i];
    }
    if (a.precond != PRE_SCHWARZ) {
      precond_vertex(a, v, r3, z3);
#pragma unroll
      for (int i = 0; i < 3; i++) {
        const size_t j = (size_t)v * 3 + i;
        if (pinned) z3[i] = 0.0;
        a.z[j] = z3[i];
        a.p[j] = z3[i];
        jsm::dd_add_prod(rz, r3[i], z3[i]);
        jsm::dd_add_prod(pp, z3[i], z3[i]);
      }
    }
#pragma unroll
    for (int i = 0; i < 3; i++) jsm::dd_add_prod(rr, r3[i], r3[i]);
  }
  block_partial_dd<kBlock>(bb, part(a, PART_BB));
  block_partial_dd<kBlock>(rr, part(a, PART_RR));
  if (a.precond != PRE_SCHWARZ) {
    block_partial_dd<kBlock>(rz, part(a, PART_RZ));
    block_partial_dd<kBlock>(pp, part(a, PART_PP));
  }
}

// External preconditioner (Schwarz): z was written by the apply; the pin
// filter on z (pcg.ts:46, :84), then p = z (init only), r.z and p.p partials.
__global__ void __launch_bounds__(kBlock) k_pcg_ext_z(PcgArgs a, int init) {
  if (!init && block_latched(&a.s->done)) return;
  jsm::dd rz = jsm::dd_zero(), pp = jsm::dd_zero();
  for (uint32_t v = blockIdx.x * blockDim.x + threadIdx.x; v < a.me.n; v += gridDim.x * blockDim.x) {
    const bool pinned = a.me.pinmask[v] != 0;
#pragma unroll
    for (int i = 0; i < 3; i++) {
      const size_t j = (size_t)v * 3 + i;
      const double zi = pinned ? 0.0 : a.z[j];
      a.z[j] = zi;
      jsm::dd_add_prod(rz, a.r[j], zi);
      if (init) {
        a.p[j] = zi;
        jsm::dd_add_prod(pp, zi, zi);
      }
    }
  }
  block_partial_dd<kBlock>(rz, part(a, PART_RZ));
  if (init) block_partial_dd<kBlock>(pp, part(a, PART_PP));
}

// After init, one block: tolerance, initial residual and rz, early return.
__global__ void __launch_bounds__(kBlock) k_pcg_init_decide(PcgArgs a, unsigned count) {
  const double bb = jsm::dd_value(merge_partials_dd<kBlock>(part(a, PART_BB), count));
  const double rr = jsm::dd_value(merge_partials_dd<kBlock>(part(a, PART_RR), count));
  const double rz = jsm::dd_value(merge_partials_dd<kBlock>(part(a, PART_RZ), count));
  if (threadIdx.x == 0) {
    PcgScalars* s = a.s;
    s->bnorm = jsm::sqrt_(bb);
    s->abs_tol = jsm::jmax(a.tol * jsm::jmax(s->bnorm, 1e-12), 1e-12);
    s->residual = jsm::sqrt_(rr);
    s->rz[0] = rz;
    s->iters = 0;
    s->done = (s->residual < s->abs_tol) ? 2 : 0;  // 2 converged, 1 (k_pcg_update) breakdown
  }
}

__global__ void __launch_bounds__(kBlock) k_pcg_hvp(PcgArgs a, int k, unsigned pp_count) {
  PcgScalars* s = a.s;
  if (block_latched(&s->done)) return;
  double h = 0;
  if (a.hvp_mode == HVP_FD)
    h = 1e-8 * (1 + jsm::sqrt_(jsm::dd_value(merge_partials_dd<kBlock>(part(a, PART_PP), pp_count))));
  jsm::dd pap = jsm::dd_zero();
  const int sub = threadIdx.x % kLanesPerVertex;
  const uint32_t stride = gridDim.x * kVertsPerBlock;
  // the loop count is uniform per vertex group (all 8 lanes share v)
  for (uint32_t v0 = blockIdx.x * kVertsPerBlock; v0 < a.me.n; v0 += stride) {
    const uint32_t v = v0 + threadIdx.x / kLanesPerVertex;
    const bool valid = v < a.me.n;
    double o[3];
    hvp_vertex8(a, v, valid, a.p, h, o);
    if (valid && sub == 0) {
      const bool pinned = a.me.pinmask[v] != 0;
#pragma unroll
      for (int i = 0; i < 3; i++) {
        const size_t j = (size_t)v * 3 + i;
        const double ap = pinned ? 0.0 : o[i];
        a.Ap[j] = ap;
        jsm::dd_add_prod(pap, a.p[j], ap);
      }
    }
  }
  block_partial_dd<kBlock>(pap, part(a, PART_PAP));
}

// ---- the step adjoint's PCG -------------------------------------------------
// Three kernels an iteration beside the hinge terms: the product with the
// bending sums and the partial sums of p.Ap; sol, r and the preconditioner with
// those of r.r and r.z; the stop and the next direction.  As separate products,
// dots, finishes and vector kernels an iteration was 13 launches, 49 us of
// them on the 128x128 sheet; now four, 33 us (the adjoint of a step 93 -> 52 ms).
__global__ void __launch_bounds__(kBlock) k_adj_product(PcgArgs a, const double* __restrict__ term,
                                                        const int32_t* done) {
  if (block_latched(done)) return;
  const int sub = threadIdx.x % kLanesPerVertex;
  const int base = (threadIdx.x % kWave) - sub;
  const uint32_t stride = gridDim.x * kVertsPerBlock;
  jsm::dd pap = jsm::dd_zero();
  for (uint32_t v0 = blockIdx.x * kVertsPerBlock; v0 < a.me.n; v0 += stride) {
    const uint32_t v = v0 + threadIdx.x / kLanesPerVertex;
    const bool valid = v < a.me.n;
    double o[3], s[3] = {0, 0, 0};
    hvp_vertex8(a, v, valid, a.p, 0.0, o);
    if (term) {
      // the vertex's hinge terms, 8 loaded at a time, added in hinge order
      const uint32_t hb = valid ? a.me.vh_off[v] : 0, he = valid ? a.me.vh_off[v + 1] : 0;
      for (uint32_t r0 = hb; r0 < he; r0 += kLanesPerVertex) {
        double t[3] = {0, 0, 0};
        if (r0 + sub < he) {
          const uint32_t rec = a.me.vh_rec[r0 + sub];
          ld3(term, (rec >> 2) * 4 + (rec & 3), t);
        }
        const uint32_t cnt = min((uint32_t)kLanesPerVertex, he - r0);
        for (uint32_t q = 0; q < cnt; q++)
#pragma unroll
          for (int i = 0; i < 3; i++) s[i] += __shfl(t[i], base + (int)q, kWave);
      }
    }
    if (valid && sub == 0) {
      const bool pinned = a.me.pinmask[v] != 0;
#pragma unroll
      for (int i = 0; i < 3; i++) {
        const size_t j = (size_t)v * 3 + i;
        const double ap = pinned ? 0.0 : term ? o[i] + s[i] : o[i];
        a.Ap[j] = ap;
        jsm::dd_add_prod(pap, a.p[j], ap);
      }
    }
  }
  block_partial_dd<kBlock>(pap, part(a, PART_PAP));
}

__global__ void __launch_bounds__(kBlock) k_adj_update(PcgArgs a, AdjPcg* s, int cur, unsigned pap_count) {
  if (block_latched(&s->done)) return;
  const double pap = jsm::dd_value(merge_partials_dd<kBlock>(part(a, PART_PAP), pap_count));
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    s->pap = pap;
    if (!(pap > 0)) s->done = 1;
  }
  if (!(pap > 0)) return;
  const double alpha = s->rz[cur] / pap;
  jsm::dd rr = jsm::dd_zero(), rz = jsm::dd_zero();
  for (uint32_t v = blockIdx.x * blockDim.x + threadIdx.x; v < a.me.n; v += gridDim.x * blockDim.x) {
    double r3[3], z3[3];
#pragma unroll
    for (int i = 0; i < 3; i++) {
      const size_t j = (size_t)v * 3 + i;
      a.sol[j] += alpha * a.p[j];
      r3[i] = a.r[j] - alpha * a.Ap[j];
      a.r[j] = r3[i];
      jsm::dd_add_prod(rr, r3[i], r3[i]);
    }
    const bool pinned = a.me.pinmask[v] != 0;
    const double* f = a.binv + (size_t)v * 9;
#pragma unroll
    for (int i = 0; i < 3; i++) {
      z3[i] = pinned ? 0.0 : f[3 * i] * r3[0] + f[3 * i + 1] * r3[1] + f[3 * i + 2] * r3[2];
      a.z[(size_t)v * 3 + i] = z3[i];
      jsm::dd_add_prod(rz, r3[i], z3[i]);
    }
  }
  block_partial_dd<kBlock>(rr, part(a, PART_RR));
  block_partial_dd<kBlock>(rz, part(a, PART_RZ));
}

__global__ void __launch_bounds__(kBlock) k_adj_dir(PcgArgs a, AdjPcg* s, int cur) {
  if (block_latched(&s->done)) return;
  const double rr = jsm::dd_value(merge_partials_dd<kBlock>(part(a, PART_RR), gridDim.x));
  const double rz = jsm::dd_value(merge_partials_dd<kBlock>(part(a, PART_RZ), gridDim.x));
  const double rel = sqrt(rr / s->bnorm2);
  const bool stop = rel <= s->tol;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    s->rr = rr;
    s->rz[cur ^ 1] = rz;
    s->rel = rel;
    s->it++;
    if (stop) s->done = 2;
  }
  if (stop) return;
  const double beta = rz / s->rz[cur];
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < (size_t)a.me.n * 3;
       i += (size_t)gridDim.x * blockDim.x)
    a.p[i] = a.z[i] + beta * a.p[i];
}

unsigned adj_product(hipStream_t st, const PcgArgs& a, const double* bend_term, const AdjPcg* s) {
  const unsigned g = (unsigned)std::min<size_t>(kMaxHvpBlocks, ((size_t)a.me.n + kVertsPerBlock - 1) / kVertsPerBlock);
  hipLaunchKernelGGL(k_adj_product, dim3(g), dim3(kBlock), 0, st, a, bend_term, &s->done);
  CS_LAUNCH_CHECK();
  return g;
}

unsigned adj_product_dot(hipStream_t st, const PcgArgs& a) {
  const size_t n3 = (size_t)a.me.n * 3;
  hipLaunchKernelGGL(k_dot, dim3(red_grid(n3)), dim3(kBlock), 0, st, a.p, a.Ap, n3,
                     a.partials + (size_t)PART_PAP * kMaxRedBlocks);
  CS_LAUNCH_CHECK();
  return red_grid(n3);
}

void adj_advance(hipStream_t st, const PcgArgs& a, AdjPcg* s, int cur, unsigned pap_count) {
  const dim3 g(red_grid(a.me.n)), b(kBlock);
  hipLaunchKernelGGL(k_adj_update, g, b, 0, st, a, s, cur, pap_count);
  hipLaunchKernelGGL(k_adj_dir, g, b, 0, st, a, s, cur);
  CS_LAUNCH_CHECK();
}

__global__ void __launch_bounds__(kBlock) k_pcg_update(PcgArgs a, int k, unsigned count) {
  PcgScalars* s = a.s;
  if (block_latched(&s->done)) return;
  const double pAp = jsm::dd_value(merge_partials_dd<kBlock>(part(a, PART_PAP), count));
  if (!(pAp > 1e-30)) {
    // non-positive curvature: stop with the current x (pcg.ts:65-68)
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      s->pAp = pAp;
      s->done = 1;
      s->iters = k;
    }
    return;
  }
  const double alpha = s->rz[k & 1] / pAp;
  jsm::dd rr = jsm::dd_zero(), rz = jsm::dd_zero();
  for (uint32_t v = blockIdx.x * blockDim.x + threadIdx.x; v < a.me.n; v += gridDim.x * blockDim.x) {
    const bool pinned = a.me.pinmask[v] != 0;
    double r3[3], z3[3];
#pragma unroll
    for (int i = 0; i < 3; i++) {
      const size_t j = (size_t)v * 3 + i;
      double xi = a.sol[j] + alpha * a.p[j];
      double ri = a.r[j] - alpha * a.Ap[j];
      if (pinned) { xi = 0.0; ri = 0.0; }
      a.sol[j] = xi;
      a.r[j] = ri;
      r3[i] = ri;
      jsm::dd_add_prod(rr, ri, ri);
    }
    if (a.precond != PRE_SCHWARZ) {
      precond_vertex(a, v, r3, z3);
#pragma unroll
      for (int i = 0; i < 3; i++) {
        if (pinned) z3[i] = 0.0;
        a.z[(size_t)v * 3 + i] = z3[i];
        jsm::dd_add_prod(rz, r3[i], z3[i]);
      }
    }
  }
  block_partial_dd<kBlock>(rr, part(a, PART_RR));
  if (a.precond != PRE_SCHWARZ) block_partial_dd<kBlock>(rz, part(a, PART_RZ));
}

__global__ void __launch_bounds__(kBlock) k_pcg_dir(PcgArgs a, int k) {
  PcgScalars* s = a.s;
  if (block_latched(&s->done)) return;
  const double residual = jsm::sqrt_(jsm::dd_value(merge_partials_dd<kBlock>(part(a, PART_RR), gridDim.x)));
  if (residual < s->abs_tol) {
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      s->residual = residual;
      s->done = 2;  // converged in this iteration
      s->iters = k + 1;
    }
    return;
  }
  const double rzNew = jsm::dd_value(merge_partials_dd<kBlock>(part(a, PART_RZ), gridDim.x));
  const double beta = rzNew / s->rz[k & 1];
  jsm::dd pp = jsm::dd_zero();
  for (uint32_t v = blockIdx.x * blockDim.x + threadIdx.x; v < a.me.n; v += gridDim.x * blockDim.x) {
    const bool pinned = a.me.pinmask[v] != 0;
#pragma unroll
    for (int i = 0; i < 3; i++) {
      const size_t j = (size_t)v * 3 + i;
      const double pi = pinned ? 0.0 : a.z[j] + beta * a.p[j];
      a.p[j] = pi;
      jsm::dd_add_prod(pp, pi, pi);
    }
  }
  block_partial_dd<kBlock>(pp, part(a, PART_PP));
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    s->rz[(k + 1) & 1] = rzNew;
    s->residual = residual;
  }
}

// ---- the whole solve in one launch (small meshes) ---------------------------
//
// Below a few thousand vertices an iteration of the three kernels above is
// launches, kernel boundaries and the latency of merging partials: 25 us in
// all (16 us of kernels) for 91 vertices as for 2,000.  Here each 8-lane group
// keeps its vertex for the whole solve, lane i < 3 component i of r, z, p, Ap
// and the solution in registers with the vertex's corners; only p and the
// work-groups' sums are exchanged, three exchanges an iteration.  The
// arithmetic is that of the kernels above; their reductions carry about twice
// the precision of the double they return, as does Sum2 here, so both return
// the same double unless the exact sum lies within 2^-100 or so of the middle
// between two.  Bound by the latency of three reductions
// with their exchanges (about 2 us each) and of the FD product.  Measured per
// iteration: 9.1 us for 91 vertices (2 work-groups), 12.6 us for 2,000 (32); a
// step of the 13x7 strip 11.7 -> 6.1 ms, of the 20x100 strip 10.8 -> 5.0 ms.
constexpr int kSmallBlock = 512, kSmallWaves = kSmallBlock / kWave;
constexpr int kSmallVerts = kSmallBlock / kLanesPerVertex;  // vertices per work-group

// A sum with the rounding errors of its additions summed beside it: the next
// addition waits for s alone, one operation, where a renormalised merge
// (jsm::dd) waits for eleven.  The errors are summed in plain FP64, without
// renormalising; over trees of 64 to 8,192 products (positive, of mixed sign,
// cancelling to 1e-12) s + e was within 2.7 * 2^-106 of the exact sum, relative
// to the sum of magnitudes, and jsm::dd within 1.4 * 2^-106; both rounded to
// the exact sum's double in all of 180 sums.
struct Sum2 {
  double s, e;
};
__device__ __forceinline__ Sum2 sum2_prod(double a, double b) {
  Sum2 r;
  jsm::two_prod(a, b, r.s, r.e);
  return r;
}
__device__ __forceinline__ Sum2 sum2_merge(Sum2 a, Sum2 b) {
  Sum2 r;
  double e;
  jsm::two_sum(a.s, b.s, r.s, e);
  r.e = (a.e + b.e) + e;
  return r;
}
template <int kCtrl>
__device__ __forceinline__ double dpp_f64(double x) {
  const unsigned long long u = __builtin_bit_cast(unsigned long long, x);
  const unsigned lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)u, kCtrl, 0xf, 0xf, false);
  const unsigned hi = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(u >> 32), kCtrl, 0xf, 0xf, false);
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}
// every lane's value plus its rotations within the row of 16 lanes
template <int kRot>
__device__ __forceinline__ Sum2 sum2_ror(Sum2 v) {
  return sum2_merge(v, Sum2{dpp_f64<0x120 + kRot>(v.s), dpp_f64<0x120 + kRot>(v.e)});
}
__device__ __forceinline__ Sum2 sum2_xor(Sum2 v, int m) {
  return sum2_merge(v, Sum2{__shfl_xor(v.s, m, kWave), __shfl_xor(v.e, m, kWave)});
}
template <int NQ>
__device__ __forceinline__ void sum2_wave(Sum2 (&v)[NQ]) {
#pragma unroll
  for (int q = 0; q < NQ; q++) v[q] = sum2_ror<8>(v[q]);
#pragma unroll
  for (int q = 0; q < NQ; q++) v[q] = sum2_ror<4>(v[q]);
#pragma unroll
  for (int q = 0; q < NQ; q++) v[q] = sum2_ror<2>(v[q]);
#pragma unroll
  for (int q = 0; q < NQ; q++) v[q] = sum2_ror<1>(v[q]);
#pragma unroll
  for (int q = 0; q < NQ; q++) v[q] = sum2_xor(v[q], 16);
#pragma unroll
  for (int q = 0; q < NQ; q++) v[q] = sum2_xor(v[q], 32);
}

// Sums NQ values over all work-groups; every thread gets the totals.  A grid
// barrier; with `publish`, vectors written with coop_store before it may be
// read with plain loads after it.  False when an exchange gave up.
template <int NQ>
__device__ __forceinline__ bool small_sums(const CoopExchange& ex, uint32_t& turn, Sum2 (&v)[NQ], double (&tot)[NQ],
                                           bool publish) {
  __shared__ Sum2 s_wave[NQ][kSmallWaves];
  __shared__ double s_tot[NQ];
  __shared__ int s_ok;
  static_assert(kSmallWaves == 8, "the waves' sums repeat twice in a row of 16 lanes");
  const int lane = threadIdx.x % kWave, wid = threadIdx.x / kWave;
  sum2_wave(v);
  if (lane == 0)
#pragma unroll
    for (int q = 0; q < NQ; q++) s_wave[q][wid] = v[q];
  if (publish) coop_drain();
  __syncthreads();
  if (wid == 0) {
#pragma unroll
    for (int q = 0; q < NQ; q++) {
      v[q] = s_wave[q][lane % kSmallWaves];
      v[q] = sum2_ror<1>(sum2_ror<2>(sum2_ror<4>(v[q])));
    }
    uint64_t mine[2 * NQ], got[2 * NQ];
#pragma unroll
    for (int q = 0; q < NQ; q++) {
      mine[2 * q] = coop_word(v[q].s);
      mine[2 * q + 1] = coop_word(v[q].e);
    }
    const bool ok = coop_exchange<2 * NQ>(ex, turn, mine, got);
#pragma unroll
    for (int q = 0; q < NQ; q++)
      v[q] = Sum2{__builtin_bit_cast(double, got[2 * q]), __builtin_bit_cast(double, got[2 * q + 1])};
    sum2_wave(v);
    if (lane == 0) {
#pragma unroll
      for (int q = 0; q < NQ; q++) s_tot[q] = v[q].s + v[q].e;
      s_ok = ok ? 1 : 0;
    }
    if (publish) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < NQ; q++) tot[q] = s_tot[q];
  return s_ok != 0;
}

__global__ void __launch_bounds__(kSmallBlock) k_pcg_small(PcgArgs a, CoopExchange ex, int max_iters) {
  const int sub = threadIdx.x % kLanesPerVertex;
  const int base = (threadIdx.x % kWave) - sub;
  const uint32_t v = blockIdx.x * kSmallVerts + threadIdx.x / kLanesPerVertex;
  const bool valid = v < a.me.n, own = valid && sub < 3;
  const size_t j = (size_t)v * 3 + sub;
  const bool pinned = valid && a.me.pinmask[v] != 0;
  const bool fd = a.hvp_mode == HVP_FD;
  // the vertex's corners, 8 to a round: those of the first round stay in
  // registers (the exchanges invalidate the caches)
  __shared__ double s_corner[kSmallBlock][7];
  const uint32_t cb = valid ? a.me.vt_off[v] : 0, ce = valid ? a.me.vt_off[v + 1] : 0;
  HvpCorner first{};
  if (cb + sub < ce) load_corner(a, a.me.vt_corner[cb + sub], first);
  const double mass = valid ? (double)a.me.mass[v] : 0.0;
  uint32_t turn = 0;
  // M^-1 of the group's residual, this lane's component
  double pre[3] = {0, 0, 0};
  if (own) {
    if (a.precond == PRE_BLOCK)
      for (int i = 0; i < 3; i++) pre[i] = a.binv[(size_t)v * 9 + sub * 3 + i];
    else
      pre[0] = a.diag[j];
  }
  auto precond = [&](double r) {
    const double r0 = __shfl(r, base, kWave), r1 = __shfl(r, base + 1, kWave), r2 = __shfl(r, base + 2, kWave);
    if (!own || pinned) return 0.0;
    if (a.precond == PRE_BLOCK) return pre[0] * r0 + pre[1] * r1 + pre[2] * r2;
    return pre[0] > 1e-12 ? r / pre[0] : r;
  };
  const double b = own ? a.b[j] : 0.0;
  double r = own && !pinned ? b : 0.0, sol = 0.0;
  double z = precond(r), p = z;
  if (own) coop_store(&a.p[j], p);
  double rz, pp, abs_tol, residual, bnorm, pAp = 0;
  int done = 0, iters = 0;
  bool ok;
  {
    Sum2 s4[4] = {sum2_prod(b, b), sum2_prod(r, r), sum2_prod(r, z), sum2_prod(z, z)};
    double t[4];
    ok = small_sums<4>(ex, turn, s4, t, true);
    bnorm = jsm::sqrt_(t[0]);
    abs_tol = jsm::jmax(a.tol * jsm::jmax(bnorm, 1e-12), 1e-12);
    residual = jsm::sqrt_(t[1]);
    rz = t[2];
    pp = t[3];
    done = residual < abs_tol ? 2 : 0;
  }
  for (int k = 0; ok && !done && k < max_iters; k++) {
    const double h = fd ? 1e-8 * (1 + jsm::sqrt_(pp)) : 0.0;
    // as hvp_vertex8; the corners' parts go through LDS, where lane i < 3
    // adds component i in list order
    double acc0 = 0, acc1 = 0;
    for (uint32_t r0 = cb; r0 < ce; r0 += kLanesPerVertex) {
      double g0[3] = {0, 0, 0}, g1[3] = {0, 0, 0};
      if (r0 + sub < ce) {
        if (r0 == cb) {
          hvp_corner(a, first, a.p, h, g0, g1);
        } else {
          HvpCorner c;
          load_corner(a, a.me.vt_corner[r0 + sub], c);
          hvp_corner(a, c, a.p, h, g0, g1);
        }
      }
#pragma unroll
      for (int i = 0; i < 3; i++) {
        s_corner[threadIdx.x][i] = g0[i];
        s_corner[threadIdx.x][3 + i] = g1[i];
      }
      __builtin_amdgcn_wave_barrier();
      if (sub < 3) {
        const uint32_t cnt = min((uint32_t)kLanesPerVertex, ce - r0);
        const double* g = &s_corner[threadIdx.x - sub][sub];
        double t0[kLanesPerVertex], t1[kLanesPerVertex];
#pragma unroll
        for (int q = 0; q < kLanesPerVertex; q++) {
          t0[q] = g[q * 7];
          t1[q] = g[q * 7 + 3];
        }
#pragma unroll
        for (uint32_t q = 0; q < kLanesPerVertex; q++)
          if (q < cnt) {
            acc0 += t0[q];
            acc1 += t1[q];
          }
      }
      __builtin_amdgcn_wave_barrier();
    }
    double ap = mass * p * a.inv_h2 + (fd ? (acc0 - acc1) / (2 * h) : acc0);
    if (a.contact.act && a.contact.nv) {
      // applyHvp per vertex: the group's lanes form 8 entries' terms at a
      // time, added in list order
      double cs[3] = {0, 0, 0};
      const uint32_t eb = valid ? a.contact.v_off[v] : 0, ee = valid ? a.contact.v_off[v + 1] : 0;
      for (uint32_t e0 = eb; e0 < ee; e0 += kLanesPerVertex) {
        double t[3] = {0, 0, 0};
        if (e0 + sub < ee) {
          const uint32_t ent = a.contact.v_ent[e0 + sub];
          if (!contact_term(a.contact, ent, contact_dd(a.contact, ent >> 3, a.p), t)) t[0] = t[1] = t[2] = 0;
        }
        const uint32_t cnt = min((uint32_t)kLanesPerVertex, ee - e0);
        for (uint32_t q = 0; q < cnt; q++)
#pragma unroll
          for (int i = 0; i < 3; i++) cs[i] += __shfl(t[i], base + (int)q, kWave);
      }
      ap += sub == 0 ? cs[0] : sub == 1 ? cs[1] : cs[2];
    }
    if (!own || pinned) ap = 0.0;
    {
      Sum2 s1[1] = {sum2_prod(p, ap)};
      double t[1];
      ok = small_sums<1>(ex, turn, s1, t, false);
      pAp = t[0];
    }
    if (!ok) break;
    if (!(pAp > 1e-30)) {
      done = 1;  // non-positive curvature: stop with the current x (pcg.ts:65-68)
      iters = k;
      break;
    }
    const double alpha = rz / pAp;
    if (own && !pinned) {
      sol = sol + alpha * p;
      r = r - alpha * ap;
    }
    z = precond(r);
    double rz_new;
    {
      Sum2 s2[2] = {sum2_prod(r, r), sum2_prod(r, z)};
      double t[2];
      ok = small_sums<2>(ex, turn, s2, t, false);
      residual = jsm::sqrt_(t[0]);
      rz_new = t[1];
    }
    if (!ok) break;
    if (residual < abs_tol) {
      done = 2;
      iters = k + 1;
      break;
    }
    const double beta = rz_new / rz;
    rz = rz_new;
    p = own && !pinned ? z + beta * p : 0.0;
    if (own) coop_store(&a.p[j], p);
    {
      Sum2 s1[1] = {sum2_prod(p, p)};
      double t[1];
      ok = small_sums<1>(ex, turn, s1, t, true);
      pp = t[0];
    }
  }
  if (own) a.sol[j] = sol;
  // the p.p partials of the last p, for a later HVP launch on these operands
  if (blockIdx.x == 0)
    for (uint32_t i = threadIdx.x; i < (a.me.n + kBlock - 1) / kBlock; i += blockDim.x)
      part(a, PART_PP)[i] = i ? jsm::dd_zero() : jsm::dd{pp, 0.0};
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    PcgScalars* s = a.s;
    s->rz[0] = s->rz[1] = rz;
    s->pAp = pAp;
    s->residual = residual;
    s->abs_tol = abs_tol;
    s->bnorm = bnorm;
    s->done = done;
    s->iters = iters;
  }
}

unsigned pcg_grid(const PcgArgs& a) { return red_grid(a.me.n); }
unsigned pcg_hvp_grid(const PcgArgs& a) {
  return (unsigned)std::min<size_t>(kMaxHvpBlocks, ((size_t)a.me.n + kVertsPerBlock - 1) / kVertsPerBlock);
}

void pcg_init(hipStream_t st, const PcgArgs& a) {
  hipLaunchKernelGGL(k_pcg_init, dim3(pcg_grid(a)), dim3(kBlock), 0, st, a);
  CS_LAUNCH_CHECK();
  if (a.precond == PRE_SCHWARZ) {
    a.sw->apply64(a.r, a.z, nullptr);
    hipLaunchKernelGGL(k_pcg_ext_z, dim3(pcg_grid(a)), dim3(kBlock), 0, st, a, 1);
    CS_LAUNCH_CHECK();
  }
  hipLaunchKernelGGL(k_pcg_init_decide, dim3(1), dim3(kBlock), 0, st, a, pcg_grid(a));
  CS_LAUNCH_CHECK();
}

// Solves the system in one launch where that is the faster way: up to
// kCoopMaxBlocks work-groups of 64 vertices, no Schwarz, and no vertex with
// many contacts.  A vertex's entries are summed by its 8 lanes, 8 at a time, and
// every work-group waits for the longest sum: a step's time per iteration
// grows by 0.26 us an entry of that vertex.  40x40 sheets on a floor with a
// finer and finer static grid under one vertex, here / with the separate
// kernels: 46 / 52 us at 53 entries, 100 / 56 at 273, 195 / 68 at 609, 954 / 157
// at 3,573 (20x20 and 62x62 sheets alike); the lines meet near 85.  False
// when it was not done (another path solves it, from the same inputs); *out
// holds the scalars otherwise.
constexpr uint32_t kSmallMaxEntries = 64;
bool pcg_solve_small(hipStream_t st, const PcgArgs& a, int max_iters, CoopState& coop, PcgScalars* out) {
  const unsigned blocks = (a.me.n + kSmallVerts - 1) / kSmallVerts;
  if (a.precond == PRE_SCHWARZ || blocks > kCoopMaxBlocks || blocks < 1) return false;
  if (a.contact.act && a.contact.nv && a.contact.most > kSmallMaxEntries) return false;
  if (coop.gave_up) return false;
  CoopTicket ticket(coop.device, blocks, coop.cus);
  if (!ticket) return false;
  coop.slots.alloc(1);
  CoopSlots* ex = coop.slots.ptr;
  CS_HIP(hipMemsetAsync(ex, 0xff, sizeof(CoopSlots), st));
  hipLaunchKernelGGL(k_pcg_small, dim3(blocks), dim3(kSmallBlock), 0, st, a, CoopExchange{ex, coop.polls}, max_iters);
  CS_LAUNCH_CHECK();
  uint64_t gave_up;
  CS_HIP(hipMemcpyAsync(&gave_up, &ex->gave_up, sizeof(gave_up), hipMemcpyDeviceToHost, st));
  CS_HIP(hipMemcpyAsync(out, a.s, sizeof(*out), hipMemcpyDeviceToHost, st));
  CS_HIP(hipStreamSynchronize(st));
  coop.gave_up = gave_up != kCoopEmpty;
  return !coop.gave_up;
}

// Back-to-back HVP launches on the operands of the last solve (Ap and the
// p.Ap partials are overwritten; the latch is cleared for the run and set after).
double pcg_time_hvp(hipStream_t st, const PcgArgs& a, int reps) {
  if (reps < 1) return 0.0;
  CS_HIP(hipMemsetAsync(&a.s->done, 0, sizeof(int32_t), st));
  hipEvent_t e0, e1;
  CS_HIP(hipEventCreate(&e0));
  CS_HIP(hipEventCreate(&e1));
  const dim3 g(pcg_hvp_grid(a)), b(kBlock);
  hipLaunchKernelGGL(k_pcg_hvp, g, b, 0, st, a, 0, pcg_grid(a));
  CS_HIP(hipEventRecord(e0, st));
  for (int i = 0; i < reps; i++) hipLaunchKernelGGL(k_pcg_hvp, g, b, 0, st, a, 0, pcg_grid(a));
  CS_HIP(hipEventRecord(e1, st));
  CS_HIP(hipEventSynchronize(e1));
  float ms = 0;
  CS_HIP(hipEventElapsedTime(&ms, e0, e1));
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  const int32_t one = 1;
  CS_HIP(hipMemcpyAsync(&a.s->done, &one, sizeof(one), hipMemcpyHostToDevice, st));
  CS_HIP(hipStreamSynchronize(st));
  return (double)ms / reps;
}

void pcg_iteration(hipStream_t st, const PcgArgs& a, int k) {
  pcg_iteration_hvp(st, a, k);
  pcg_iteration_rest(st, a, k);
}

// The HVP grid differs from the vector grid; its partial count is passed on.
void pcg_iteration_hvp(hipStream_t st, const PcgArgs& a, int k) {
  if (a.contact.act && a.contact.nv && use_vertex_groups(a.contact.E, a.contact.nv)) {
    hipLaunchKernelGGL(k_contact_dd, dim3(grid_for(a.contact.C)), dim3(kBlock), 0, st, a.contact, a.p, &a.s->done);
    launch_vertex_sums(st, HvpSums{a.contact, &a.s->done}, a.contact.nv, a.contact.cverts, a.contact.v_off);
  } else if (a.contact.act && a.contact.nv) {
    hipLaunchKernelGGL(k_contact_terms, dim3(grid_for(a.contact.E)), dim3(kBlock), 0, st, a.contact, a.p, &a.s->done);
    hipLaunchKernelGGL(k_contact_vsum, dim3(grid_for((size_t)a.contact.nv * 3)), dim3(kBlock), 0, st, a.contact,
                       &a.s->done);
  }
  hipLaunchKernelGGL(k_pcg_hvp, dim3(pcg_hvp_grid(a)), dim3(kBlock), 0, st, a, k, pcg_grid(a));
  CS_LAUNCH_CHECK();
}

void pcg_iteration_rest(hipStream_t st, const PcgArgs& a, int k) {
  const dim3 g(pcg_grid(a)), b(kBlock);
  hipLaunchKernelGGL(k_pcg_update, g, b, 0, st, a, k, pcg_hvp_grid(a));
  if (a.precond == PRE_SCHWARZ) {
    a.sw->apply64(a.r, a.z, &a.s->done);
    hipLaunchKernelGGL(k_pcg_ext_z, g, b, 0, st, a, 0);
  }
  hipLaunchKernelGGL(k_pcg_dir, g, b, 0, st, a, k);
  CS_LAUNCH_CHECK();
}

// ---- block-Jacobi factors ---------------------------------------------------

// Diagonal 3x3 block (corner vc) of triangleHessian9 (membrane-blocks.ts:21-98),
// same loop nest and accumulation order as the reference for those entries.
__device__ void tri_hessian_block(const double* x0, const double* x1, const double* x2, const float* inv,
                                  double area, const DMat& mat, int vc, double* hb) {
  const double a = inv[0], b = inv[1], c = inv[2], d = inv[3];
  const double* X[3] = {x0, x1, x2};
  const double K[3][2] = {{-(a + c), -(b + d)}, {a, b}, {c, d}};
  double F[3][2] = {{0, 0}, {0, 0}, {0, 0}};
  for (int i = 0; i < 3; i++)
    for (int j = 0; j < 2; j++)
      for (int v = 0; v < 3; v++) F[i][j] += K[v][j] * X[v][i];
  double Cm[2][2] = {{0, 0}, {0, 0}};
  for (int l = 0; l < 2; l++)
    for (int m = 0; m < 2; m++)
      for (int i = 0; i < 3; i++) Cm[l][m] += F[i][l] * F[i][m];
  const double E00 = 0.5 * (Cm[0][0] - 1), E11 = 0.5 * (Cm[1][1] - 1), E01 = 0.5 * Cm[0][1];
  const double S00 = mat.c00 * E00 + mat.c01 * E11;
  const double S11 = mat.c11 * E11 + mat.c01 * E00;
  const double S01 = 2 * mat.g * E01;
  const double S[2][2] = {{S00, S01}, {S01, S11}};
  double D[2][2][2][2];
  for (int q = 0; q < 16; q++) (&D[0][0][0][0])[q] = 0;
  D[0][0][0][0] = mat.c00;
  D[1][1][1][1] = mat.c11;
  D[0][0][1][1] = mat.c01; D[1][1][0][0] = mat.c01;
  D[0][1][0][1] = mat.g; D[0][1][1][0] = mat.g; D[1][0][0][1] = mat.g; D[1][0][1][0] = mat.g;
  const double s = mat.thick * area;
  // M[A][i][j] = (i == A % 3) ? K[A / 3][j] : 0
  for (int ra = 0; ra < 3; ra++) {
    for (int rb = 0; rb < 3; rb++) {
      const int A = vc * 3 + ra, B = vc * 3 + rb;
      const int av = A / 3, ai = A % 3, bv = B / 3, bi = B % 3;
      double sum = 0;
      for (int i = 0; i < 3; i++) {
        for (int j = 0; j < 2; j++) {
          const double mA = (i == ai) ? K[av][j] : 0.0;
          if (mA == 0) continue;
          double dP = 0;
          for (int k = 0; k < 2; k++) {
            const double mBik = (i == bi) ? K[bv][k] : 0.0;
            dP += mBik * S[k][j];
            double dE = 0;
            for (int l = 0; l < 2; l++) {
              for (int m2 = 0; m2 < 2; m2++) {
                const double dd = D[k][j][l][m2];
                if (dd == 0) continue;
                double dElm = 0;
                for (int p = 0; p < 3; p++) {
                  const double mBpl = (p == bi) ? K[bv][l] : 0.0;
                  const double mBpm = (p == bi) ? K[bv][m2] : 0.0;
                  dElm += mBpl * F[p][m2] + F[p][l] * mBpm;
                }
                dE += dd * 0.5 * dElm;
              }
            }
            dP += F[i][k] * dE;
          }
          sum += mA * dP;
        }
      }
      hb[ra * 3 + rb] = s * sum;
    }
  }
}

// buildBlockFactors (block-jacobi.ts:30-87), one thread per vertex.
__global__ void __launch_bounds__(kBlock) k_block_factors(DMesh me, DMat mat, const double* __restrict__ x,
                                                          const double* __restrict__ diag, double* binv,
                                                          uint8_t* flag) {
  const uint32_t v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= me.n) return;
  double bl[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0}, hb[9];
  for (uint32_t k = me.vt_off[v]; k < me.vt_off[v + 1]; k++) {
    const uint32_t rec = me.vt_rec[k];
    const uint32_t t = rec >> 2;
    const int corner = rec & 3;
    double x0[3], x1[3], x2[3];
    ld3(x, me.idx[(size_t)t * 3], x0);
    ld3(x, me.idx[(size_t)t * 3 + 1], x1);
    ld3(x, me.idx[(size_t)t * 3 + 2], x2);
    tri_hessian_block(x0, x1, x2, me.inv_dm + (size_t)t * 4, me.area[t], mat, corner, hb);
    for (int q = 0; q < 9; q++) bl[q] += hb[q];
  }
  const double d0 = diag[(size_t)v * 3], d1 = diag[(size_t)v * 3 + 1], d2 = diag[(size_t)v * 3 + 2];
  const double B00 = bl[0] + d0, B11 = bl[4] + d1, B22 = bl[8] + d2;
  const double B01 = 0.5 * (bl[1] + bl[3]);
  const double B02 = 0.5 * (bl[2] + bl[6]);
  const double B12 = 0.5 * (bl[5] + bl[7]);
  const double tr = jsm::fabs_(B00) + jsm::fabs_(B11) + jsm::fabs_(B22);
  const double tiny = 1e-20 * (1 + tr);
  bool ok = true;
  if (!(B00 > tiny)) ok = false;
  if (ok && !(B00 * B11 - B01 * B01 > tiny * (1 + jsm::fabs_(B00) + jsm::fabs_(B11)))) ok = false;
  const double det = B00 * (B11 * B22 - B12 * B12) - B01 * (B01 * B22 - B12 * B02) + B02 * (B01 * B12 - B11 * B02);
  if (ok && !(det > tiny * (1 + tr) * (1 + tr))) ok = false;
  double* o = binv + (size_t)v * 9;
  if (ok) {
    const double s = 1 / det;
    o[0] = (B11 * B22 - B12 * B12) * s;
    o[1] = (B02 * B12 - B01 * B22) * s;
    o[2] = (B01 * B12 - B11 * B02) * s;
    o[3] = (B02 * B12 - B01 * B22) * s;
    o[4] = (B00 * B22 - B02 * B02) * s;
    o[5] = (B01 * B02 - B00 * B12) * s;
    o[6] = (B01 * B12 - B11 * B02) * s;
    o[7] = (B01 * B02 - B00 * B12) * s;
    o[8] = (B00 * B11 - B01 * B01) * s;
    if (flag) flag[v] = 1;
  } else {
    const double i0 = d0 > 1e-12 ? 1 / d0 : 0;
    const double i1 = d1 > 1e-12 ? 1 / d1 : 0;
    const double i2 = d2 > 1e-12 ? 1 / d2 : 0;
    o[0] = i0; o[1] = 0; o[2] = 0;
    o[3] = 0; o[4] = i1; o[5] = 0;
    o[6] = 0; o[7] = 0; o[8] = i2;
    if (flag) flag[v] = 0;
  }
}

void launch_block_factors(hipStream_t st, const DMesh& me, const DMat& mat, const double* x, const double* diag,
                          double* binv, uint8_t* flag) {
  hipLaunchKernelGGL(k_block_factors, dim3(grid_for(me.n)), dim3(kBlock), 0, st, me, mat, x, diag, binv, flag);
  CS_LAUNCH_CHECK();
}

// ---- vector helpers ---------------------------------------------------------

__global__ void __launch_bounds__(kBlock) k_dot(const double* __restrict__ a, const double* __restrict__ b,
                                                size_t n, jsm::dd* partials) {
  jsm::dd acc = jsm::dd_zero();
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    jsm::dd_add_prod(acc, a[i], b[i]);
  block_partial_dd<kBlock>(acc, partials);
}

void launch_dot(hipStream_t st, const double* a, const double* b, size_t n, jsm::dd* partials, double* out) {
  const unsigned grid = red_grid(n);
  hipLaunchKernelGGL(k_dot, dim3(grid), dim3(kBlock), 0, st, a, b, n, partials);
  CS_LAUNCH_CHECK();
  FinishJobs f{};
  f.j[0] = FinishJob{partials, grid, FIN_DD, 0, out};
  launch_finish(st, f, 1);
}

__global__ void __launch_bounds__(kBlock) k_max_abs(const double* __restrict__ a, size_t n, double* partials) {
  double m = 0;
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
    const double v = jsm::fabs_(a[i]);
    if (v > m) m = v;
  }
  block_partial_ext<kBlock, GtMax>(m, partials);
}

void launch_max_abs(hipStream_t st, const double* a, size_t n, double* partials, double* out) {
  const unsigned grid = red_grid(n);
  hipLaunchKernelGGL(k_max_abs, dim3(grid), dim3(kBlock), 0, st, a, n, partials);
  CS_LAUNCH_CHECK();
  FinishJobs f{};
  f.j[0] = FinishJob{partials, grid, FIN_GTMAX, 1, out};
  launch_finish(st, f, 1);
}

__global__ void k_fallback_dir(const double* __restrict__ g, const double* __restrict__ diag, double* dx, size_t n) {
  const size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (i < n) dx[i] = -g[i] / diag[i];
}
void launch_fallback_dir(hipStream_t st, const double* g, const double* diag, double* dx, size_t n) {
  hipLaunchKernelGGL(k_fallback_dir, dim3(grid_for(n)), dim3(kBlock), 0, st, g, diag, dx, n);
  CS_LAUNCH_CHECK();
}

__global__ void k_scale(double* v, double s, size_t n) {
  const size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (i < n) v[i] *= s;
}
void launch_scale(hipStream_t st, double* v, double s, size_t n) {
  hipLaunchKernelGGL(k_scale, dim3(grid_for(n)), dim3(kBlock), 0, st, v, s, n);
  CS_LAUNCH_CHECK();
}

__global__ void k_trial(const double* __restrict__ x, const double* __restrict__ dx, double alpha, double* xt,
                        size_t n) {
  const size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (i < n) xt[i] = x[i] + alpha * dx[i];
}
void launch_trial(hipStream_t st, const double* x, const double* dx, double alpha, double* xt, size_t n) {
  hipLaunchKernelGGL(k_trial, dim3(grid_for(n)), dim3(kBlock), 0, st, x, dx, alpha, xt, n);
  CS_LAUNCH_CHECK();
}

__global__ void k_neg(const double* __restrict__ g, double* b, size_t n) {
  const size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (i < n) b[i] = -g[i];
}
void launch_neg(hipStream_t st, const double* g, double* b, size_t n) {
  hipLaunchKernelGGL(k_neg, dim3(grid_for(n)), dim3(kBlock), 0, st, g, b, n);
  CS_LAUNCH_CHECK();
}

}  // namespace cloth
