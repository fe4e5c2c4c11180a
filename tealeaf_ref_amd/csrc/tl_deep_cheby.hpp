// Chebyshev iterations, many per pass (tl_deep.hpp).  One iteration
// (kernels/tea_leaf_cheby_kernel.f90:111-200) is
//   w = A u;  r = u0 - w;  p' = alpha p + beta r;  u' = u + p'
// so a stage keeps two rows of u and one of p in registers, and the ring holds
// u0 beside the faces and the diagonal.  u and p are read from one buffer and
// written to the other.
#pragma once

#include "tl_deep.hpp"
#include "tl_loopk.hpp"

namespace tl {

// Fields of the ring: kx, ky (times rx, ry), u0 and the diagonal.
constexpr int DEEP_CHEBY_FIELDS = 4;

struct DeepCheby {
  const double *u, *p, *u0, *Kx, *Ky;
  double *u_out, *p_out;
  double *w, *r;             // of the last iteration, in a last pass
  double rx, ry;
  double *part_rr;
};

namespace {

// LAST: the last pass of a run also stores w and r and the partials of r.r.
// At 4096^2 ten iterations take 207 us in one pass (268 with w and r), against 166
// us for every two before: 20.7 us an iteration instead of 83.  Bound, as
// k_deep_ppcg, by the instructions of its one wave per SIMD, with memory close
// behind (1.05 GB at 5.1 TB/s).  The ring of ten stages takes the CU's 160 KB: 10
// rows x 4 fields x 1 KB for each of four waves.
template <int STAGES, int LAST>
__global__ __launch_bounds__(BLOCK) void k_deep_cheby(DeepGeo g, DeepCoef<double> co,
                                                      DeepCheby a) {
  constexpr int V = 2, NF = DEEP_CHEBY_FIELDS;
  typedef double T;
  typedef typename dev::Vec<T, V>::type VT;
  extern __shared__ char dyn[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int nb = g.blocks;
  const int b = blockIdx.x;
  const int lb = nb % NUM_XCD == 0 ? (b % NUM_XCD) * (nb / NUM_XCD) + b / NUM_XCD : b;
  const dev::DeepStrip<T, V, STAGES> t(g, lb * (BLOCK / WAVE) + wave);
  VT *ring = (VT *)dyn + (long)wave * STAGES * NF * WAVE + t.lane;
  auto at = [&](int slot, int f) -> VT & { return ring[(slot * NF + f) * WAVE]; };
  double acc = 0.0;
  struct In {
    VT kx, ky, u, p, u0;
  };
  int yl = t.first;
  long row_l = (long)yl * t.pitch;
  auto load = [&]() {
    In i;
    const bool is = yl < t.ny;
    i.kx = t.load(a.Kx, row_l, is);
    i.ky = t.load(a.Ky, row_l, is && yl > 0);
    i.u = t.load(a.u, row_l, is);
    i.p = t.load(a.p, row_l, is);
    i.u0 = t.load(a.u0, row_l, is);
    yl += 1;
    row_l += t.pitch;
    return i;
  };
  dev::LaneCoef<T> cs(co);
  if (t.live) {
    // rows of u before stage s + 1: behind[s], centre[s]; p of iteration s on
    // the row stage s + 1 takes next
    VT behind[STAGES], centre[STAGES], ps[STAGES];
#pragma unroll
    for (int s = 0; s < STAGES; ++s) behind[s] = centre[s] = ps[s] = VT(0);
    VT kx1 = VT(0), ky1 = VT(0), u01 = VT(0);
    for (int i = 0; i < STAGES * NF; ++i) ring[i * WAVE] = VT(0);
    constexpr int AHEAD = dev::DEEP_AHEAD;
    In q[AHEAD];
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) q[i] = load();
    long row_o = ((long)t.first - STAGES) * t.pitch;
    struct Faces {
      VT kx, ky, di, u0;
    };
    auto step = [&](int y, In &qi, const int slot) {
      In in = qi;
      // no readlane and no multiple of the pitch leaves the row to wait for it
      // in a register
      asm volatile("" : "+v"(cs.a), "+v"(cs.b), "+s"(row_l), "+s"(row_o));
      const int yo = y - STAGES;
      qi = load();
      in.kx = t.faces_x(in.kx) * a.rx;
      in.ky = in.ky * a.ry;
      VT kyu = in.ky;
      Faces f = {kx1, ky1, VT(0), u01};
      T kxr = dev::from_above(f.kx[0]);
#pragma unroll
      for (int e = 0; e < V; ++e)
        f.di[e] = T(1) + (kyu[e] + f.ky[e]) + (dev::vec_right<T, V>(f.kx, e, kxr) + f.kx[e]);
      at(slot, 0) = f.kx;
      at(slot, 1) = f.ky;
      at(slot, 2) = f.u0;
      at(slot, 3) = f.di;
      VT ahead = in.u, p = ps[0], w = VT(0), r = VT(0);
      ps[0] = in.p;
#pragma unroll
      for (int s = 0; s < STAGES; ++s) {
        // the next stage's fields (row y - 2 - s) on their way during this one
        Faces nf = f;
        if (s + 1 < STAGES) {
          const int o = (slot - s - 1 + STAGES) % STAGES;
          nf = {at(o, 0), at(o, 1), at(o, 3), at(o, 2)};
        }
        __builtin_amdgcn_sched_barrier(0);
        const VT c = centre[s];
        const T lo = dev::from_below(c[V - 1]), hi = dev::from_above(c[0]);
        if (s > 0) kxr = dev::from_above(f.kx[0]);
#pragma unroll
        for (int e = 0; e < V; ++e) {
          const T l = dev::vec_left<T, V>(c, e, lo), rr = dev::vec_right<T, V>(c, e, hi);
          const T kr = dev::vec_right<T, V>(f.kx, e, kxr);
          if (LAST && s + 1 == STAGES) {
            w[e] = f.di[e] * c[e] - kr * rr - f.kx[e] * l - f.ky[e] * behind[s][e] -
                   kyu[e] * ahead[e];
            r[e] = f.u0[e] - w[e];
          } else {
            r[e] = f.u0[e] - f.di[e] * c[e] + kr * rr + f.kx[e] * l + f.ky[e] * behind[s][e] +
                   kyu[e] * ahead[e];
          }
        }
        const VT pn = cs.alpha(s) * p + cs.beta(s) * r;
        const VT un = c + pn;
        behind[s] = c;
        centre[s] = ahead;
        ahead = un;
        if (s + 1 < STAGES) {
          p = ps[s + 1];
          ps[s + 1] = pn;
        } else {
          p = pn;
        }
        kyu = f.ky;
        f = nf;
      }
      kx1 = in.kx;
      ky1 = in.ky;
      u01 = in.u0;
      const bool ok = yo >= t.y0 && yo < t.y1;
      t.store(a.u_out, row_o, ahead, ok);
      t.store(a.p_out, row_o, p, ok);
      if (LAST) {
        t.store(a.w, row_o, w, ok);
        t.store(a.r, row_o, r, ok);
        r = t.only_if(r, ok);
#pragma unroll
        for (int e = 0; e < V; ++e) acc += r[e] * r[e];
      }
      row_o += t.pitch;
    };
    // steps past the last row store nothing
    for (int y = t.first; y <= t.last; y += STAGES) {
#pragma unroll
      for (int j = 0; j < STAGES; ++j) step(y + j, q[j % AHEAD], j);
    }
    // carry the halo ring of u to the new buffer: the columns beside the mesh
    // a row per lane, the rows beyond it a column per lane
    if (t.left_edge || t.right_edge)
      for (int y = t.y0 + t.lane; y < t.y1; y += WAVE) {
        const long i = (long)y * t.pitch;
        if (t.left_edge) a.u_out[i - 1] = a.u[i - 1];
        if (t.right_edge) a.u_out[i + t.nx] = a.u[i + t.nx];
      }
    for (int side = 0; side < 2; ++side) {
      if (side ? t.y1 != t.ny : t.y0 != 0) continue;
      const long hr = side ? (long)t.ny * t.pitch : -t.pitch;
      if (t.mine)
        for (int e = 0; e < V; ++e)
          if (t.c + e < t.nx) a.u_out[hr + t.c + e] = a.u[hr + t.c + e];
    }
  }
  if (LAST) {
    // cells outside the mesh have u0 = A u = 0; ghosts are not the lane's
    if (!t.mine) acc = 0.0;
    __syncthreads();
    acc = dev::block_sum(acc, (double *)dyn);
    if (threadIdx.x == 0) a.part_rr[blockIdx.x] = acc;
  }
}

constexpr size_t deep_cheby_lds(int stages) {
  return (size_t)(BLOCK / WAVE) * stages * DEEP_CHEBY_FIELDS * WAVE * 16;
}

template <int STAGES>
int deep_cheby_launch(const double *alphas, const double *betas, const DeepCheby &a, bool last,
                      int *nparts) {
  DeepCoef<double> co;
  for (int s = 0; s < DEEP_MAX; ++s) {
    co.a[s] = s < STAGES ? alphas[s] : 0.0;
    co.b[s] = s < STAGES ? betas[s] : 0.0;
  }
  const size_t lds = deep_cheby_lds(STAGES);
  // what the registers (and from six stages on the rings) let a CU hold
  const DeepGeo g = deep_geo<double, 2>(STAGES, S().pitch, STAGES <= 2 ? 3 : STAGES <= 4 ? 2 : 1);
  hipEvent_t ev;
  prof_arm(3, &ev);
  klaunch_lds(last ? &k_deep_cheby<STAGES, 1> : &k_deep_cheby<STAGES, 0>, dim3(g.blocks),
              dim3(BLOCK), lds, g, co, a);
  prof_end(3, ev);
  *nparts = g.blocks;
  if (hipGetLastError() != hipSuccess) return fail(TL_ERR_HIP, "Chebyshev pass launch");
  return TL_OK;
}

inline int deep_cheby(int stages, const double *alphas, const double *betas, const DeepCheby &a,
                      bool last, int *nparts) {
  switch (stages) {
    case 2: return deep_cheby_launch<2>(alphas, betas, a, last, nparts);
    case 4: return deep_cheby_launch<4>(alphas, betas, a, last, nparts);
    case 6: return deep_cheby_launch<6>(alphas, betas, a, last, nparts);
    case 8: return deep_cheby_launch<8>(alphas, betas, a, last, nparts);
    default: return deep_cheby_launch<DEEP_MAX>(alphas, betas, a, last, nparts);
  }
}

}  // namespace
}  // namespace tl
