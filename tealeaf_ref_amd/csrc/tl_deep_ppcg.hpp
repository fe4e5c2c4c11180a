// PPCG's inner steps, many per pass (tl_deep.hpp).  Included by tl_loopk.hpp.
#pragma once

#include "tl_deep.hpp"

namespace tl {

template <typename T>
struct DeepPpcg {
  const T *r, *r_store, *Kx, *Ky;
  const T *z_in, *zp_in;   // z and z one sweep before; not in a first pass
  T *z_out, *zp_out;       // ... of the next pass; not in a last pass
  T *z;
  T rx, ry, theta_r;
  double *part_rrn, *part_zr;
  Ctl *ctl;
  // FIRST 2, the first pass of an outer iteration n with its update of r
  // (tea_solve.f90:300-309): rro = z.r, from the partials that the sweeps
  // before left or rro_in, alpha = rro / p.w, r_out = r - alpha w.  r is left
  // as it is and serves as r_store: the two change places every iteration.
  const T *w;
  T *r_out;
  int n, first, npw, nzr;
  double rro_in;
  const double *part_pw, *zr_in;
  double *hrro, *halpha;
};

namespace {

// Ring fields of a pass: kx, ky (times rx, ry), r and, in the Di form, Di.
template <typename T>
constexpr int deep_fields() {
  return diff_form<T>() ? 3 : 4;
}

// The sweeps are done on z itself,
//   z' = z + alpha (z - z'') + beta (r - A z),   z'' one sweep before z,
// which is the recurrence of rtemp, sd and utemp
// (kernels/tea_leaf_ppcg_kernel.f90:288-306) with rtemp = r - A z and sd = z -
// z''.  z'' is what the stage before holds as its row below, so a stage keeps two
// rows of one field.
//
// At 4096^2 ten sweeps of FP64 and the update of r take 194 us (FP32, 256
// columns a wave: 129): 883 MB at 4.6 TB/s, and 0.8 of the 1.1 us a row are
// taken also where the mesh lies in the caches.  The instructions of one wave
// per SIMD (the LDS holds no more rings) are 345 a row, 180 of them FP64.  With
// rtemp, sd and utemp in four rows of registers a stage, masks by bits, row
// addresses per lane and faces not yet multiplied by rx and ry they were 540,
// and the pass took 211 us without the update of r, which took another 141.
// Finishing a stage while the next one's other terms are formed gained nothing
// (193 us), nor did five rows in flight instead of two.
template <typename T, int V, int STAGES, int FIRST, int LAST>
__global__ __launch_bounds__(BLOCK) void k_deep_ppcg(DeepGeo g, DeepCoef<T> co,
                                                     DeepPpcg<T> a) {
  typedef typename dev::Vec<T, V>::type VT;
  constexpr bool DIFF = diff_form<T>();
  constexpr int NF = deep_fields<T>();  // ring fields: kx, ky, r and, in the Di form, Di
  constexpr bool UPD = FIRST == 2;
  extern __shared__ char dyn[];
  if (a.ctl && a.ctl->stop) return;
  T ca = T(0);
  if constexpr (UPD) {
    double *lds = (double *)dyn;
    const double pw = dev::sum_partials(a.part_pw, a.npw, lds);
    const double rro = a.first ? a.rro_in : dev::sum_partials(a.zr_in, a.nzr, lds);
    if (nonfinite_stop(a.n, pw, rro, a.ctl)) return;
    const double alpha = rro / pw;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      a.hrro[a.n] = rro;
      a.halpha[a.n] = alpha;
    }
    ca = (T)alpha;
    __syncthreads();  // the ring takes the sums' place
  }
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int nb = g.blocks;
  const int b = blockIdx.x;
  const int lb = nb % NUM_XCD == 0 ? (b % NUM_XCD) * (nb / NUM_XCD) + b / NUM_XCD : b;
  const dev::DeepStrip<T, V, STAGES> t(g, lb * (BLOCK / WAVE) + wave);
  VT *ring = (VT *)dyn + (long)wave * STAGES * NF * WAVE + t.lane;
  auto at = [&](int slot, int f) -> VT & { return ring[(slot * NF + f) * WAVE]; };
  double arrn = 0.0, azr = 0.0;
  // a row as loaded: z is w where r is updated
  struct In {
    VT kx, ky, r, z, zp;
  };
  // rows are loaded in order; without faces below the mesh's first row
  int yl = t.first;
  long row_l = (long)yl * t.pitch;
  auto load = [&]() {
    In i;
    const bool is = yl < t.ny;
    i.kx = t.load(a.Kx, row_l, is);
    i.ky = t.load(a.Ky, row_l, is && yl > 0);
    i.r = t.load(a.r, row_l, is);
    i.z = i.zp = VT(0);
    if (UPD) i.z = t.load(a.w, row_l, is);
    if (!FIRST) {
      i.z = t.load(a.z_in, row_l, is);
      i.zp = t.load(a.zp_in, row_l, is);
    }
    yl += 1;
    row_l += t.pitch;
    return i;
  };
  T vrx = a.rx, vry = a.ry, vth = a.theta_r, vca = ca;
  asm volatile("" : "+v"(vrx), "+v"(vry), "+v"(vth), "+v"(vca));
  if (t.live) {
    // rows of z before stage s + 1: behind[s], centre[s]
    VT behind[STAGES], centre[STAGES];
#pragma unroll
    for (int s = 0; s < STAGES; ++s) behind[s] = centre[s] = VT(0);
    // the row loaded last
    VT kx1 = VT(0), ky1 = VT(0), r1 = VT(0), zp1 = VT(0);
    // rows below the first one loaded are rows of zeros without faces
    for (int i = 0; i < STAGES * NF; ++i) ring[i * WAVE] = VT(0);
    constexpr int AHEAD = dev::DEEP_AHEAD;
    In q[AHEAD];
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) q[i] = load();
    // r_store of the output row: in a single pass r as it was loaded, kept
    // since then (read again it came from memory: 757 MB read at 4096^2 instead of
    // 613), else loaded a step ahead
    constexpr bool RRN = LAST && FIRST != 1;
    VT rs1 = VT(0), r_was[UPD && LAST ? STAGES : 1];
#pragma unroll
    for (int s = 0; UPD && LAST && s < STAGES; ++s) r_was[s] = VT(0);
    long row_o = ((long)t.first - STAGES) * t.pitch;  // row of the output
    struct Row {
      VT kx, ky, r, di;
    };
    // one row; `slot` is the ring slot of row y - 1, a constant in the unrolled
    // loop, as every ring address and register of the stages then is
    auto step = [&](int y, In &qi, const int slot) {
      In in = qi;
      // no readlane and no multiple of the pitch leaves the row to wait for it
      // in a register
      asm volatile("" : "+s"(row_l), "+s"(row_o));
      const int yo = y - STAGES;
      // the next output row's loads before the row's after next, so that
      // waiting for the first does not wait for the second
      VT rs = rs1;
      const bool ok = yo >= t.y0 && yo < t.y1;
      if (RRN && !UPD)
        rs1 = t.load(a.r_store, row_o + t.pitch, yo + 1 >= t.y0 && yo + 1 < t.y1);
      qi = load();
      in.kx = t.faces_x(in.kx) * vrx;
      in.ky = in.ky * vry;
      if (UPD && LAST) {
        rs = r_was[slot];  // of row y - STAGES
        r_was[slot] = in.r;
      }
      if (UPD) in.r = in.r - vca * in.z;
      if (FIRST) in.z = in.r * vth;
      // row y - 1 into the ring
      VT kyu = in.ky;
      Row f = {kx1, ky1, r1, VT(0)};
      T kxr = dev::from_above(f.kx[0]);
      if (!DIFF) {
#pragma unroll
        for (int e = 0; e < V; ++e)
          f.di[e] = T(1) + (kyu[e] + f.ky[e]) + (dev::vec_right<T, V>(f.kx, e, kxr) + f.kx[e]);
        at(slot, 3) = f.di;
      }
      at(slot, 0) = f.kx;
      at(slot, 1) = f.ky;
      at(slot, 2) = f.r;
      VT ahead = in.z, before = zp1, out_r = VT(0), out_zp = VT(0);
#pragma unroll
      for (int s = 0; s < STAGES; ++s) {
        // the next stage's row y - 2 - s on its way during this one
        Row nf = f;
        if (s + 1 < STAGES) {
          const int o = (slot - s - 1 + STAGES) % STAGES;
          nf.kx = at(o, 0);
          nf.ky = at(o, 1);
          nf.r = at(o, 2);
          if (!DIFF) nf.di = at(o, 3);
        }
        __builtin_amdgcn_sched_barrier(0);
        const VT c = centre[s];
        const T lo = dev::from_below(c[V - 1]), hi = dev::from_above(c[0]);
        if (s > 0) kxr = dev::from_above(f.kx[0]);
        VT zn;
#pragma unroll
        for (int e = 0; e < V; ++e) {
          const T l = dev::vec_left<T, V>(c, e, lo), r = dev::vec_right<T, V>(c, e, hi);
          const T kr = dev::vec_right<T, V>(f.kx, e, kxr);
          T res;  // r - A z
          if (DIFF)
            res = f.r[e] - c[e] + f.kx[e] * (l - c[e]) + kr * (r - c[e]) +
                  f.ky[e] * (behind[s][e] - c[e]) + kyu[e] * (ahead[e] - c[e]);
          else
            res = f.r[e] - f.di[e] * c[e] + f.kx[e] * l + kr * r + f.ky[e] * behind[s][e] +
                  kyu[e] * ahead[e];
          const T d = (FIRST && s == 0) ? c[e] : c[e] - before[e];
          zn[e] = c[e] + co.a[s] * d + co.b[s] * res;
        }
        before = behind[s];
        behind[s] = c;
        centre[s] = ahead;
        ahead = zn;
        if (s + 1 == STAGES) {
          out_r = f.r;
          out_zp = c;
        }
        kyu = f.ky;
        f = nf;
      }
      kx1 = in.kx;
      ky1 = in.ky;
      r1 = in.r;
      if (!FIRST) zp1 = in.zp;
      if (UPD) t.store(a.r_out, row_o, out_r, ok);
      if (LAST) {
        t.store(a.z, row_o, ahead, ok);
        const VT z = t.only_if(ahead, ok);
#pragma unroll
        for (int e = 0; e < V; ++e) {
          if (RRN) arrn += ((double)out_r[e] - (double)rs[e]) * (double)z[e];
          azr += (double)z[e] * (double)out_r[e];
        }
      } else {
        t.store(a.z_out, row_o, ahead, ok);
        t.store(a.zp_out, row_o, out_zp, ok);
      }
      row_o += t.pitch;
    };
    // steps past the last row store nothing
    for (int y = t.first; y <= t.last; y += STAGES) {
#pragma unroll
      for (int j = 0; j < STAGES; ++j) step(y + j, q[j % AHEAD], j);
    }
  }
  if (LAST) {
    // what the lanes of ghost columns have added up is not theirs
    if (!t.mine) arrn = azr = 0.0;
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
  return (size_t)(BLOCK / WAVE) * stages * deep_fields<T>() * WAVE * 16;
}

// `count` sweeps in STAGES stages; a stage without a sweep (an odd count's
// last) hands z on as it is.
template <typename T, int V, int STAGES, int FIRST, int LAST>
int deep_launch(const DeepGeo &g, int count, const double *alphas, const double *betas,
                const DeepPpcg<T> &a) {
  DeepCoef<T> co;
  for (int s = 0; s < DEEP_MAX; ++s) {
    co.a[s] = s < count ? (T)alphas[s] : T(0);
    co.b[s] = s < count ? (T)betas[s] : T(0);
  }
  hipEvent_t ev;
  prof_arm(2, &ev);
  klaunch_lds(&k_deep_ppcg<T, V, STAGES, FIRST, LAST>, dim3(g.blocks), dim3(BLOCK),
              deep_lds<T>(STAGES), g, co, a);
  prof_end(2, ev);
  TL_HIP(hipGetLastError());
  return TL_OK;
}

// The passes of `inner` sweeps: an even number of stages, at most DEEP_MAX, in
// each, as alike as they can be.
inline int deep_stages(int inner) { return (inner + 1) / 2 * 2; }
inline int deep_passes(int inner) { return (deep_stages(inner) + DEEP_MAX - 1) / DEEP_MAX; }
// stages of the next pass, of `left` (even) stages in `passes` passes
inline int deep_next(int left, int passes) { return (left / 2 + passes - 1) / passes * 2; }
inline int deep_last(int inner) {
  int left = deep_stages(inner), n = 0;
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
int deep_dispatch(int stages, int count, long pitch, const double *alphas, const double *betas,
                  const DeepPpcg<T> &a) {
  const DeepGeo g = deep_ppcg_geo<T, V>(stages, pitch);
  // four sweeps fill a pass only on their own
  if constexpr (FIRST && LAST)
    if (stages == 4) return deep_launch<T, V, 4, FIRST, LAST>(g, count, alphas, betas, a);
  if (stages == 6) return deep_launch<T, V, 6, FIRST, LAST>(g, count, alphas, betas, a);
  if (stages == 8) return deep_launch<T, V, 8, FIRST, LAST>(g, count, alphas, betas, a);
  return deep_launch<T, V, DEEP_MAX, FIRST, LAST>(g, count, alphas, betas, a);
}
// first: 0 no, 1 yes, 2 with the update of r
template <typename T, int V>
int deep_pass(int first, bool last, int stages, int count, long pitch, const double *alphas,
              const double *betas, const DeepPpcg<T> &a) {
  auto f = first == 2   ? (last ? &deep_dispatch<T, V, 2, 1> : &deep_dispatch<T, V, 2, 0>)
           : first == 1 ? (last ? &deep_dispatch<T, V, 1, 1> : &deep_dispatch<T, V, 1, 0>)
                        : (last ? &deep_dispatch<T, V, 0, 1> : &deep_dispatch<T, V, 0, 0>);
  return f(stages, count, pitch, alphas, betas, a);
}

}  // namespace
}  // namespace tl
