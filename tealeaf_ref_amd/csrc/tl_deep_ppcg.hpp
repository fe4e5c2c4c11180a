// PPCG's inner steps, many per pass (tl_deep.hpp).  Included by tl_loopk.hpp.
#pragma once

#include "tl_deep.hpp"

namespace tl {

template <typename T>
struct DeepPpcg {
  const T *r, *r_store, *Kx, *Ky;
  const T *sd_in, *rt_in, *ut_in;   // not in a first pass
  T *sd_out, *rt_out, *ut_out;      // not in a last pass
  T *z;
  T rx, ry, theta_r;
  double *part_rrn, *part_zr;
  const Ctl *ctl;
};

namespace {

// What bounds it: the instructions of one wave per SIMD (the LDS holds no
// more rings).  About 590 for a row of ten sweeps of 128 FP64 columns, of
// which 240 are the FP64 arithmetic, issue in 1.2 us a row; memory would allow
// 110 us for the 40 bytes a cell.  Ten sweeps at 4096^2: 216 us in one pass
// against 880 us in five passes of two (FP32, 256 columns a wave: 158 against
// 446).  What it took, from 341 us: the rows unrolled by the ring's length, so
// that no register moves and no ring address is computed (309); the faces of
// the next stage read from the LDS while the current one is computed, the
// output row's loads issued before the prefetched row's, and the coefficients
// in lanes instead of spilled scalar registers (211).  More rows in flight
// (four or five instead of two) spill, and gain nothing where they do not.
template <typename T, int V, int STAGES, int FIRST, int LAST>
__global__ __launch_bounds__(BLOCK) void k_deep_ppcg(DeepGeo g, DeepCoef<T> co,
                                                     DeepPpcg<T> a) {
  typedef typename dev::Vec<T, V>::type VT;
  constexpr bool DIFF = diff_form<T>();
  constexpr int NF = DIFF ? 2 : 3;     // ring fields: kx, ky and, in the Di form, Di
  extern __shared__ char dyn[];
  if (a.ctl && a.ctl->stop) return;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int nb = g.blocks;
  const int b = blockIdx.x;
  const int lb = nb % NUM_XCD == 0 ? (b % NUM_XCD) * (nb / NUM_XCD) + b / NUM_XCD : b;
  const dev::DeepStrip<T, V, STAGES> t(g, lb * (BLOCK / WAVE) + wave);
  VT *ring = (VT *)dyn + (long)wave * STAGES * NF * WAVE + t.lane;
  auto at = [&](int slot, int f) -> VT & { return ring[(slot * NF + f) * WAVE]; };
  double arrn = 0.0, azr = 0.0;
  struct In {
    VT kx, ky, sd, rt;
  };
  // rows are loaded in order, from one past the last on the last row again
  // (what lies beyond the mesh is masked)
  int yl = t.first;
  long row_l = (long)yl * t.pitch;
  auto load = [&]() {
    In i;
    i.kx = t.load(a.Kx, row_l);
    i.ky = t.load(a.Ky, row_l);
    if (FIRST) {
      i.rt = t.load(a.r, row_l);
      i.sd = VT(0);
    } else {
      i.rt = t.load(a.rt_in, row_l);
      i.sd = t.load(a.sd_in, row_l);
    }
    yl += 1;
    row_l += yl < t.ny ? t.pitch : 0;
    return i;
  };
  dev::LaneCoef<T> cs(co);
  if (t.live) {
    // rows of sd before stage s + 1: behind[s], centre[s]; rtemp and utemp of
    // sweep s on the row stage s + 1 takes next
    VT behind[STAGES], centre[STAGES], rts[STAGES], uts[STAGES];
#pragma unroll
    for (int s = 0; s < STAGES; ++s) behind[s] = centre[s] = rts[s] = uts[s] = VT(0);
    VT kx1 = VT(0), ky1 = VT(0);
    // rows below the first one loaded are rows of zeros without faces
    for (int i = 0; i < STAGES * NF; ++i) ring[i * WAVE] = VT(0);
    constexpr int AHEAD = dev::deep_ahead(STAGES);
    In q[AHEAD];
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) q[i] = load();
    // what an output row needs besides the stages' results, loaded a step
    // ahead: r and r_store, and utemp of the passes before, which is added
    // there, where only its own cell reads it
    struct Out {
      VT rv, rs, u0;
    };
    Out o1 = {VT(0), VT(0), VT(0)};
    long row_o = (long)t.y0 * t.pitch;  // row of the next output
    auto load_out = [&](long row) {
      Out o = {VT(0), VT(0), VT(0)};
      if (LAST) o.rv = t.load(a.r, row);
      if (LAST) o.rs = t.load(a.r_store, row);
      if (!FIRST && (t.out || t.part)) o.u0 = t.load(a.ut_in, row);
      return o;
    };
    struct Faces {
      VT kx, ky, di;
    };
    // one row; `slot` is the ring slot of row y - 1, a constant in the unrolled
    // loop, as every ring address and register of the stages then is
    auto step = [&](int y, In &qi, const int slot) {
      In in = qi;
      asm volatile("" : "+v"(cs.a), "+v"(cs.b));  // no readlane leaves the row
      const int yo = y - STAGES;
      // the next output row's loads before the row's after next, so that
      // waiting for the first does not wait for the second
      const Out out = o1;
      const bool ok = yo >= t.y0 && yo < t.y1;
      o1 = load_out(row_o + (ok && yo + 1 < t.y1 ? t.pitch : 0));
      qi = load();
      in.kx = t.faces_x(in.kx, y);
      in.ky = t.faces_y(in.ky, y);
      in.rt = t.cells(in.rt, y);
      if (!FIRST) in.sd = t.cells(in.sd, y);
      VT in_ut = VT(0);
      if (FIRST) in.sd = in_ut = in.rt * a.theta_r;
      // faces and diagonal of row y - 1 into the ring
      VT kyu = in.ky;
      Faces f = {kx1, ky1, VT(0)};
      T kxr = dev::from_above(f.kx[0]);
      if (!DIFF) {
#pragma unroll
        for (int e = 0; e < V; ++e)
          f.di[e] = T(1) + a.ry * (kyu[e] + f.ky[e]) +
                    a.rx * (dev::vec_right<T, V>(f.kx, e, kxr) + f.kx[e]);
        at(slot, 2) = f.di;
      }
      at(slot, 0) = f.kx;
      at(slot, 1) = f.ky;
      VT ahead = in.sd, rt = rts[0], ut = uts[0];
      rts[0] = in.rt;
      uts[0] = in_ut;
#pragma unroll
      for (int s = 0; s < STAGES; ++s) {
        // the next stage's faces (row y - 2 - s) on their way during this one
        Faces nf = f;
        if (s + 1 < STAGES) {
          const int o = (slot - s - 1 + STAGES) % STAGES;
          nf.kx = at(o, 0);
          nf.ky = at(o, 1);
          if (!DIFF) nf.di = at(o, 2);
        }
        __builtin_amdgcn_sched_barrier(0);
        const VT c = centre[s];
        const T lo = dev::from_below(c[V - 1]), hi = dev::from_above(c[0]);
        if (s > 0) kxr = dev::from_above(f.kx[0]);
        VT w;
#pragma unroll
        for (int e = 0; e < V; ++e) {
          const T l = dev::vec_left<T, V>(c, e, lo), r = dev::vec_right<T, V>(c, e, hi);
          const T kr = dev::vec_right<T, V>(f.kx, e, kxr);
          if (DIFF)
            w[e] = dev::apply_diff<T>(c[e], l, r, behind[s][e], ahead[e], f.kx[e], kr, f.ky[e],
                                      kyu[e], a.rx, a.ry);
          else
            w[e] = f.di[e] * c[e] - a.ry * (kyu[e] * ahead[e] + f.ky[e] * behind[s][e]) -
                   a.rx * (kr * r + f.kx[e] * l);
        }
        const VT rn = rt - w;
        const VT sn = cs.alpha(s) * c + cs.beta(s) * rn;
        const VT un = ut + sn;
        behind[s] = c;
        centre[s] = ahead;
        ahead = sn;
        if (s + 1 < STAGES) {
          rt = rts[s + 1];
          rts[s + 1] = rn;
          ut = uts[s + 1];
          uts[s + 1] = un;
        } else {
          rt = rn;
          ut = un;
        }
        kyu = f.ky;
        f = nf;
      }
      kx1 = in.kx;
      ky1 = in.ky;
      if (!FIRST) ut = out.u0 + ut;
      if (LAST) {
        t.store(a.z, row_o, ut, ok);
        const VT rv = t.cells_if(out.rv, ok), rs = t.cells_if(out.rs, ok);
        ut = t.cells_if(ut, ok);
#pragma unroll
        for (int e = 0; e < V; ++e) {
          arrn += ((double)rv[e] - (double)rs[e]) * (double)ut[e];
          azr += (double)ut[e] * (double)rv[e];
        }
      } else {
        t.store(a.sd_out, row_o, ahead, ok);
        t.store(a.rt_out, row_o, rt, ok);
        t.store(a.ut_out, row_o, ut, ok);
      }
      row_o += ok ? t.pitch : 0;
    };
    // steps past the last row store nothing
    for (int y = t.first; y <= t.last; y += STAGES) {
#pragma unroll
      for (int j = 0; j < STAGES; ++j) step(y + j, q[j % AHEAD], j);
    }
  }
  if (LAST) {
    // what the lanes of ghost columns have added up is not theirs
    if (!t.out && !t.part) arrn = azr = 0.0;
    // the ring's memory serves the block's sums
    __syncthreads();
    double *lds = (double *)dyn;
    arrn = dev::block_sum(arrn, lds);
    azr = dev::block_sum(azr, lds);
    if (threadIdx.x == 0) {
      a.part_rrn[blockIdx.x] = arrn;
      a.part_zr[blockIdx.x] = azr;
    }
  }
}

// LDS of a block: four waves' rings
template <typename T>
constexpr size_t deep_lds(int stages) {
  return (size_t)(BLOCK / WAVE) * stages * (diff_form<T>() ? 2 : 3) * WAVE * 16;
}

template <typename T, int V, int STAGES, int FIRST, int LAST>
int deep_launch(const DeepGeo &g, const double *alphas, const double *betas, const DeepPpcg<T> &a) {
  DeepCoef<T> co;
  for (int s = 0; s < DEEP_MAX; ++s) {
    co.a[s] = s < STAGES ? (T)alphas[s] : T(0);
    co.b[s] = s < STAGES ? (T)betas[s] : T(0);
  }
  hipEvent_t ev;
  prof_arm(2, &ev);
  klaunch_lds(&k_deep_ppcg<T, V, STAGES, FIRST, LAST>, dim3(g.blocks), dim3(BLOCK),
              deep_lds<T>(STAGES), g, co, a);
  prof_end(2, ev);
  TL_HIP(hipGetLastError());
  return TL_OK;
}

// The passes of `inner` sweeps: an even count of at most DEEP_MAX in each, as
// alike as they can be, after a single sweep where `inner` is odd.
inline int deep_passes(int inner) { return (inner / 2 * 2 + DEEP_MAX - 1) / DEEP_MAX; }
// sweeps of the next pass, of `left` (even) sweeps in `passes` passes
inline int deep_next(int left, int passes) { return (left / 2 + passes - 1) / passes * 2; }
inline int deep_last(int inner) {
  int left = inner / 2 * 2, n = 0;
  for (int p = deep_passes(inner); p > 0; --p) left -= n = deep_next(left, p);
  return n;
}
inline bool deep_on() {
  const char *e = getenv("TL_DEEP");
  return !e || atoi(e) != 0;
}
// Not on meshes so wide that their strips alone would leave more partial sums
// than the slots hold (MAX_GRID blocks of four strips of at least 84 columns).
inline bool deep_fits() {
  return S().nx <= MAX_GRID * 4 * 84 && sweep_pairs() && deep_on();
}
// Whether the deep passes take these sweeps: not with a preconditioner (one
// or two sweeps per pass there), and not fewer than 4.
inline bool deep_takes(int inner, int diag, int block) {
  return !diag && !block && inner >= 4 && deep_fits();
}

// Strips and tiles of a pass whose blocks a CU holds `per_cu` of.
template <typename T, int V>
DeepGeo deep_geo(int stages, long pitch, int per_cu) {
  const State &s = S();
  DeepGeo g;
  g.nx = s.nx;
  g.ny = s.ny;
  g.pitch = pitch;
  const int strip = dev::deep_strip(stages, V);
  g.strips = (s.nx + strip - 1) / strip;
  // one round of waves: what the CUs hold at once
  const int waves = (s.cus > 0 ? s.cus : 256) * per_cu * (BLOCK / WAVE);
  int tiles = waves / g.strips;
  if (tiles < 1) tiles = 1;
  g.rows = (s.ny + tiles - 1) / tiles;
  // whole turns of the ring: a strip is walked in steps of `stages` rows
  g.rows = (g.rows + stages - 1) / stages * stages;
  g.tiles = (s.ny + g.rows - 1) / g.rows;
  const int w = BLOCK / WAVE;
  g.blocks = (int)(((long)g.strips * g.tiles + w - 1) / w);
  if (g.blocks >= NUM_XCD) g.blocks = (g.blocks + NUM_XCD - 1) / NUM_XCD * NUM_XCD;
  return g;
}

// PPCG's passes: four stages take under 256 registers, so a CU holds two
// blocks; with more the registers or the rings allow one.
template <typename T, int V>
DeepGeo deep_ppcg_geo(int stages, long pitch) {
  return deep_geo<T, V>(stages, pitch, stages <= 4 ? 2 : 1);
}

// Partial sums the last pass leaves.
template <typename T, int V>
int deep_parts(int inner, long pitch) {
  return deep_ppcg_geo<T, V>(deep_last(inner), pitch).blocks;
}

template <typename T, int V, int FIRST, int LAST>
int deep_dispatch(int stages, long pitch, const double *alphas, const double *betas,
                  const DeepPpcg<T> &a) {
  const DeepGeo g = deep_ppcg_geo<T, V>(stages, pitch);
  // 4 sweeps: alone, or after the single sweep of an odd count
  if constexpr (LAST)
    if (stages == 4) return deep_launch<T, V, 4, FIRST, LAST>(g, alphas, betas, a);
  if (stages == 6) return deep_launch<T, V, 6, FIRST, LAST>(g, alphas, betas, a);
  if (stages == 8) return deep_launch<T, V, 8, FIRST, LAST>(g, alphas, betas, a);
  return deep_launch<T, V, DEEP_MAX, FIRST, LAST>(g, alphas, betas, a);
}

}  // namespace
}  // namespace tl
