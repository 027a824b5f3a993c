// vsum.h — per-vertex sums over the contact incidence, in list order.
#pragma once

#include "common.h"

namespace cloth {

// out[v] = init(v) + the terms of v's incidence entries, added in list order
// (two values per entry and component, a then b, when Op::kPair), for the nv
// vertices that have entries.  One work-group per vertex: its threads form
// 256 entries' terms at once in LDS, then three lanes, one per component, add
// them in order.
//
// Bound by the gathers of the terms and the chain of dependent additions
// (about 10 cycles each).  The form it stands beside (terms of all entries
// into memory, then one thread per vertex and component adding with strided
// loads) leaves the chip idle where few vertices have many contacts: two
// 33x33 sheets on each other (2,178 vertices, 256 entries each) took 30 + 27 us
// per Hessian product, now 7 + 20 us; the 256x256 drape on its sphere (134
// vertices, up to 566 entries) 4 + 21 us, now 4 + 9 us.  Where a vertex has
// one or two entries (a sheet lying on the floor) a work-group each is waste:
// see use_vertex_groups.
template <class Op>
__global__ void __launch_bounds__(kBlock) k_vertex_sums(Op op, uint32_t nv, const uint32_t* __restrict__ cverts,
                                                        const uint32_t* __restrict__ v_off) {
  constexpr int N = Op::kPair ? 6 : 3;
  __shared__ double buf[kBlock * N];
  if (op.skip()) return;
  for (uint32_t i = blockIdx.x; i < nv; i += gridDim.x) {
    const uint32_t v = cverts[i], b = v_off[v], e = v_off[v + 1];
    double acc = threadIdx.x < 3 ? op.init(v, threadIdx.x) : 0.0;
    for (uint32_t base = b; base < e; base += kBlock) {
      if (base + threadIdx.x < e) {
        double t[N];
        op.term(base + threadIdx.x, t);
#pragma unroll
        for (int q = 0; q < N; q++) buf[threadIdx.x * N + q] = t[q];
      }
      __syncthreads();
      if (threadIdx.x < 3) {
        const uint32_t cnt = min((uint32_t)kBlock, e - base);
        const double* s = buf + threadIdx.x;
        uint32_t j = 0;
        for (; j + 8 <= cnt; j += 8) {
          double a[8], c[8];
#pragma unroll
          for (int k = 0; k < 8; k++) {
            a[k] = s[(j + k) * N];
            if (Op::kPair) c[k] = s[(j + k) * N + 3];
          }
#pragma unroll
          for (int k = 0; k < 8; k++) {
            acc += a[k];
            if (Op::kPair) acc += c[k];
          }
        }
        for (; j < cnt; j++) {
          acc += s[j * N];
          if (Op::kPair) acc += s[j * N + 3];
        }
      }
      __syncthreads();
    }
    if (threadIdx.x < 3) op.store(v, threadIdx.x, acc);
  }
}

template <class Op>
inline void launch_vertex_sums(hipStream_t st, const Op& op, uint32_t nv, const uint32_t* cverts,
                               const uint32_t* v_off) {
  hipLaunchKernelGGL(HIP_KERNEL_NAME(k_vertex_sums<Op>), dim3(nv < 8192u ? nv : 8192u), dim3(kBlock), 0, st, op, nv,
                     cverts, v_off);
  CS_LAUNCH_CHECK();
}

// Whether the E entries of nv vertices are summed by a work-group per vertex.
// Measured per PCG iteration of a step, the older form / this one: one entry a
// vertex, 16,641 vertices 94 / 102 us, 65,536 vertices 175 / 223 us (a
// work-group each is waste); 58 to 77 entries, 112 to 6,733 vertices, 195 / 180
// to 1,695 / 1,660 us; 349 to 396 entries, 882 to 33,282 vertices, 173 / 150 to
// 7,936 / 7,633 us.  Between 1 and 58 the line is a choice: where one vertex
// has many more than the rest the two differ little up to 16,641 vertices
// (3,969 vertices of 1.1 entries, 273 on one: 62 / 60 us).
inline bool use_vertex_groups(uint32_t E, uint32_t nv) { return E >= 16u * nv; }

}  // namespace cloth
