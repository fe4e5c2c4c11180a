// Kernels and launches of the on-chip solver loops (tl_resident.hpp).
#include <cstring>

#include "tl_resident.hpp"

using namespace tl;

namespace {

using dev::ResFaces;
using dev::ResGhost;
using dev::ResShared;
using dev::ResTile;

// A field a lane keeps for the whole loop: in registers, or in the block's
// dynamic LDS where the registers are needed for others.
template <typename T, int R, bool LDS>
struct Kept {
  typedef typename dev::Vec<T, 2>::type VT;
  VT v[R];
  __device__ Kept(char *, int) {}
  __device__ VT get(int j) const { return v[j]; }
  __device__ void set(int j, VT x) { v[j] = x; }
};
template <typename T, int R>
struct Kept<T, R, true> {
  typedef typename dev::Vec<T, 2>::type VT;
  VT *v;
  __device__ Kept(char *lds, int slot) : v((VT *)lds + (long)slot * R * RES_THREADS + threadIdx.x) {}
  __device__ VT get(int j) const { return v[j * RES_THREADS]; }
  __device__ void set(int j, VT x) { v[j * RES_THREADS] = x; }
};

// The ghosts of a field in memory, for the first iteration.
template <typename T, int R>
__device__ inline ResGhost<T> load_ghosts(const ResTile<T, R> &t, const ResGeo &g, const T *f) {
  ResGhost<T> o;
  o.dn = t.load(f, g, t.y0 - 1);
  o.up = t.load(f, g, t.y0 + R);
  o.side = T(0);
  if (t.lane < 2 * R) {
    const bool lft = t.lane < R;
    const int y = t.y0 + (lft ? t.lane : t.lane - R);
    if (y < g.ny && (lft ? t.left : t.right))
      o.side = *t.at(f, g, lft ? t.bx * RES_COLS - 1 : (t.bx + 1) * RES_COLS, y);
  }
  return o;
}

// ---------------------------------------------------------------------------
// CG: iterations n_first.. of run_cg_loop in one launch
// ---------------------------------------------------------------------------
// Where a lane's fields live at R rows: it has 256 registers, of which r, p,
// w (or z) and kx take four fields.  Larger tiles move u and ky to LDS (160 KB
// per CU); the preconditioner's fields are then read again in every
// iteration, from the L2.  The splits are those at which the kernel spills no
// vector register, and it must not: the compiler may place a spill inside a
// region that only some lanes run, where it misses the others.  The build
// fails where one does (spills.awk).
//
// What bounds it: the two exchanges of an iteration.  Of a wave's time they take
// 0.81 at 512^2 (64 blocks of four rows, 5.0 us an iteration), 0.86 at 777x1031
// with jac_diag (231 blocks of four rows, 6.8 us), and with eight rows a lane,
// where the arithmetic counts, 0.71 at 1024^2 (7.0 us) and 0.68 at 1500x997 with
// jac_block (8.9 us).  Against the pass kernels: 512^2 step 5.7 -> 2.4 ms, 777x1031
// with jac_diag 23.0 -> 4.8 ms, 1500x997 with jac_block 87.5 -> 20.3 ms, the 1024^2
// adjoint's CG solves 155 -> 41 ms.
enum Where { REGS, MEMORY };
template <typename T, int R, int PREC>
struct CgPlan {
  static constexpr int SIZE = (int)sizeof(T) / 4 * 2 * R;  // registers of one field
  static constexpr bool U_LDS = SIZE >= 24;
  static constexpr bool KY_LDS = SIZE >= (PREC == TL_PREC_NONE ? 32 : 24);
  static constexpr Where M = PREC == TL_PREC_NONE  ? REGS
                             : PREC == TL_PREC_JAC_BLOCK ? MEMORY
                             : SIZE >= 24  ? MEMORY
                                           : REGS;
  static constexpr int SLOTS = (U_LDS ? 1 : 0) + (KY_LDS ? 1 : 0);
  static constexpr size_t BYTES = (size_t)SLOTS * R * RES_THREADS * 2 * sizeof(T);
};

template <typename T, int R, int PREC>
__global__ __launch_bounds__(RES_THREADS) void k_res_cg(ResGeo g, ResCg<T> a) {
  typedef typename dev::Vec<T, 2>::type VT;
  typedef CgPlan<T, R, PREC> Plan;
  extern __shared__ char dyn[];
  __shared__ ResShared<T, R, 1> sh;
  if (threadIdx.x < 2) sh.dead[threadIdx.x] = 0;
  const ResTile<T, R> t(g);
  ResFaces<T, R, Plan::KY_LDS> k;
  k.load(t, g, a.Kx, a.Ky, sh.kxr[t.wave],
         (VT *)dyn + (long)(Plan::U_LDS ? 1 : 0) * R * RES_THREADS + threadIdx.x);
  VT r[R], p[R];
  constexpr bool HAS_Z = PREC != TL_PREC_NONE;
  VT z[HAS_Z ? R : 1];
  Kept<T, R, Plan::U_LDS> u(dyn, 0);
  // Mi of the diagonal preconditioner, where it is kept
  Kept<T, Plan::M == MEMORY || !HAS_Z ? 1 : R, false> m(dyn, 0);
  // what goes to LDS first, while there are registers to pass through
  if (Plan::KY_LDS) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int j = 0; j < R; ++j) u.set(j, t.load(a.u, g, t.y0 + j));
  if (Plan::U_LDS) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int j = 0; j < R; ++j) {
    const int y = t.y0 + j;
    r[j] = t.load(a.r, g, y);
    p[j] = t.load(a.pin, g, y);
    if constexpr (HAS_Z && Plan::M != MEMORY) m.set(j, t.load(a.Mi, g, y));
  }
  ResGhost<T> pg = load_ghosts<T, R>(t, g, a.pin);
  const bool lead = t.blk == 0 && threadIdx.x == 0;
  double rro = a.rro, err = 0.0, rrn = 0.0;
  int reason = 0, n_end = 0;
  bool dead = false, update = false;
  T be = T(0);
  ResGhost<T> gh;
  ResOrder<true> o;
  if (lead) a.hrro[a.n_first] = rro;
  __syncthreads();
  // body(j, w) of row j of w = A p
  auto apply_p = [&](auto body) {
    if (t.lane < 2 * R) sh.side[t.wave][t.lane] = pg.side;
    __builtin_amdgcn_wave_barrier();
    dev::res_apply<diff_form<T>()>(t, k, p, pg.dn, pg.up, sh.side[t.wave], sh.kxr[t.wave], a.rx,
                                   a.ry, body);
  };
  for (int n = a.n_first;; ++n) {
    VT w[R];
    // ---- w = A p, p.w
    double acc = 0.0;
    apply_p([&](int j, VT wv) {
      w[j] = wv;
      acc += (double)wv.x * (double)p[j].x;
      acc += (double)wv.y * (double)p[j].y;
    });
    double pw;
    if (!dev::res_exchange<false, true>(t, g, sh, o, acc, &pw, (const VT(*)[R]) nullptr,
                                        (ResGhost<T> *)nullptr)) {
      dead = true;
      break;
    }
    if (!isfinite(pw)) {
      reason = TL_LOOP_NONFINITE;
      n_end = n;
      err = pw;
      break;
    }
    const double alpha = rro / pw;
    if (lead) a.halpha[n] = alpha;
    // ---- u += alpha p, r -= alpha w, z = M^-1 r, r.r or r.z
    const T al = (T)alpha;
    acc = 0.0;
#pragma unroll
    for (int j = 0; j < R; ++j) {
      u.set(j, u.get(j) + al * p[j]);
      r[j] = r[j] - al * w[j];
    }
    bool ok;
    const int yn = t.row_anew();
    if constexpr (PREC == TL_PREC_NONE) {
#pragma unroll
      for (int j = 0; j < R; ++j) {
        acc += (double)r[j].x * (double)r[j].x;
        acc += (double)r[j].y * (double)r[j].y;
      }
      ok = dev::res_exchange<true, true>(t, g, sh, o, acc, &rrn, &r, &gh);
    } else {
      if constexpr (PREC == TL_PREC_JAC_DIAG) {
#pragma unroll
        for (int j = 0; j < R; ++j) {
          if constexpr (Plan::M == MEMORY) z[j] = t.load(a.Mi, g, yn + j) * r[j];
          else z[j] = m.get(j) * r[j];
        }
      } else {
        // 4-row Thomas solve (tea_block_solve, kernels/tea_leaf_common_kernel.f90:
        // 378-468); cells outside the mesh have r = 0, bfp = 0 and Di = 1.  cp
        // above the first row is formed as k_block_init forms it.
#pragma unroll
        for (int b = 0; b < R; b += 4) {
          __builtin_amdgcn_sched_barrier(0);  // one group's loads at a time
          VT di = t.load(a.Di, g, yn + b), bf[3];
          const VT c0 = t.load(a.cp, g, yn + b);
#pragma unroll
          for (int q = 1; q < 4; ++q) bf[q - 1] = t.load(a.bfp, g, yn + b + q);
          if (!t.okx || b >= t.rows) di.x = T(1);
          if (!t.oky || b >= t.rows) di.y = T(1);
          z[b] = r[b] / di;
#pragma unroll
          for (int q = 1; q < 4; ++q)
            z[b + q] = (r[b + q] - (-k.ky(b + q) * a.ry) * z[b + q - 1]) * bf[q - 1];
          // back substitution; the last row of a short block has no row above
#pragma unroll
          for (int q = 2; q >= 0; --q) {
            const VT c = q > 0 ? (-k.ky(b + q + 1) * a.ry) * bf[q > 0 ? q - 1 : 0] : c0;
            z[b + q] = b + q + 1 < t.rows ? z[b + q] - c * z[b + q + 1] : z[b + q];
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
#pragma unroll
      for (int j = 0; j < R; ++j) {
        acc += (double)r[j].x * (double)z[j].x;
        acc += (double)r[j].y * (double)z[j].y;
      }
      ok = dev::res_exchange<true, true>(t, g, sh, o, acc, &rrn, &z, &gh);
    }
    if (!ok) {
      dead = true;
      break;
    }
    // ---- head of iteration n + 1 (loop_head)
    const double beta = rrn / rro;
    err = sqrt(fabs(rrn));
    const bool bad = !isfinite(rrn), conv = !bad && fabs(err) < a.lp.eps_abs;
    const bool tail = n == a.n_last, pause = n == a.n_pause;
    const bool sw = !bad && !conv && !tail && a.lp.check_switch && fabs(err) <= a.lp.epslim &&
                    n + 1 >= a.lp.presteps;
    if (lead) {
      a.hbeta[n] = beta;
      a.herr[n] = err;
    }
    be = (T)beta;
    if (bad || conv || sw || tail || pause) {
      reason = bad    ? TL_LOOP_NONFINITE
               : conv ? TL_LOOP_CONVERGED
               : sw   ? TL_LOOP_SWITCH
               : tail ? TL_LOOP_MAXITERS
                      : RES_PAUSED;
      n_end = sw ? n + 1 : n;
      update = true;
      break;
    }
#pragma unroll
    for (int j = 0; j < R; ++j) {
      if constexpr (HAS_Z) p[j] = z[j] + be * p[j];
      else p[j] = r[j] + be * p[j];
    }
    pg.dn = gh.dn + be * pg.dn;
    pg.up = gh.up + be * pg.up;
    pg.side = gh.side + be * pg.side;
    if (lead) a.hrro[n + 1] = rrn;
    rro = rrn;
  }
  if (dead) {
    if (threadIdx.x == 0) *g.abort_flag = 1;
    return;
  }
  // the fields as the loop leaves them; w = A p of the last iteration is
  // formed again rather than held through it
  const int col = t.col_anew(), row = t.row_anew();
  apply_p([&](int j, VT wv) { t.store(a.w, g, col, row + j, wv); });
#pragma unroll
  for (int j = 0; j < R; ++j) {
    const int y = row + j;
    t.store(a.u, g, col, y, u.get(j));
    t.store(a.r, g, col, y, r[j]);
    VT pj = p[j];
    if (update) {
      if constexpr (HAS_Z) pj = z[j] + be * pj;
      else pj = r[j] + be * pj;
      if constexpr (HAS_Z) t.store(a.z, g, col, y, z[j]);
    }
    t.store(a.p, g, col, y, pj);
  }
  if (lead) {
    a.ctl->stop = 1;
    a.ctl->reason = reason;
    a.ctl->n_end = n_end;
    a.ctl->error = err;
    a.ctl->old_error = err;
    a.ctl->rro = rrn;
  }
  if (a.hist && t.blk == 0) {
    __syncthreads();  // the leading lane has written them
    const int last = a.n_base + HHIST - 1 < n_end ? a.n_base + HHIST - 1 : n_end;
    for (int i = a.n_first + threadIdx.x; i <= last; i += RES_THREADS) {
      a.hist[i - a.n_base] = a.halpha[i];
      a.hist[HHIST + i - a.n_base] = a.hbeta[i];
    }
  }
}

// ---------------------------------------------------------------------------
// Jacobi: iterations n_first.. of tl_jacobi_loop in one launch
// ---------------------------------------------------------------------------
// One exchange per iteration carries the halos of the new u and the sum of
// |u - un|, so that the exit test of an iteration is settled before the next
// one begins.  Cells outside the mesh are zero: with external faces whose
// coefficients are zero nothing crosses them, and reflective faces, whose
// coefficients are not, are to read zero there (as k_jl_v, ZE); what is held
// for them is 1 / Di = 0.  Every operation is rounded as the reference's, so that
// the iterates are the reference's to the bit and an exit at a fixed point of
// the rounding comes at its iteration: no products are fused, and the quotient
// by Di is the product with the rounded 1 / Di, corrected by its remainder
// (Markstein 1990), the division's own result in three operations for about ten.
//
// What bounds it: the exchange, 0.81 of a wave's time with 225 blocks of five rows
// (1100x1000: 3.9 us an iteration).  Steps of 1000 iterations by passes and on the
// chip: 1100x1000 11.1 and 4.0 ms, 1400^2 14.2 and 5.0, 512^2 5.5 and 2.9, 100^2 4.4
// and 2.3.
// tea_leaf_jacobi_kernel.f90:60-66
__device__ inline double jacobi_num(double s0, double l, double r, double d, double u, double kxl,
                                    double kxr, double kyd, double kyu, double rx, double ry) {
#pragma clang fp contract(off)
  return s0 + rx * (kxr * r + kxl * l) + ry * (kyu * u + kyd * d);
}
__device__ inline double jacobi_den(double kxl, double kxr, double kyd, double kyu, double rx,
                                    double ry) {
#pragma clang fp contract(off)
  return 1.0 + rx * (kxl + kxr) + ry * (kyd + kyu);
}

template <int R>
struct JacobiPlan {
  // of 256 registers a field takes 4 a row
  static constexpr bool KY_LDS = R >= 8, U0_LDS = R >= 8;
  static constexpr size_t BYTES = KY_LDS ? (size_t)2 * R * RES_THREADS * 2 * sizeof(double) : 0;
};

template <int R>
__global__ __launch_bounds__(RES_THREADS) void k_res_jacobi(ResGeo g, ResJacobi a) {
  typedef double T;
  typedef typename dev::Vec<T, 2>::type VT;
  extern __shared__ char dyn[];
  __shared__ ResShared<T, R, 1> sh;
  if (threadIdx.x < 2) sh.dead[threadIdx.x] = 0;
  const ResTile<T, R> t(g);
  VT u[R], rdi[R], kx[R], ky_top = VT(0);
  Kept<T, R, JacobiPlan<R>::U0_LDS> u0(dyn, 1);
  Kept<T, R, JacobiPlan<R>::KY_LDS> ky_in(dyn, 0);
  T *kxr = sh.kxr[t.wave];
  // the faces, which the row above and the column right of the mesh have too
#pragma unroll
  for (int j = 0; j <= R; ++j) {
    const int y = t.y0 + j;
    VT v = VT(0);
    if (t.okx && y <= g.ny) {
      v = *(const VT *)t.at(a.Ky, g, t.c, y);
      if (!t.oky) v.y = T(0);
    }
    if (j < R) ky_in.set(j < R ? j : 0, v);
    else ky_top = v;
  }
  if (JacobiPlan<R>::KY_LDS) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int j = 0; j < R; ++j) {
    const int y = t.y0 + j;
    kx[j] = VT(0);
    if (t.c <= g.nx && y < g.ny) {
      kx[j] = *(const VT *)t.at(a.Kx, g, t.c, y);
      if (t.c == g.nx) kx[j].y = T(0);
    }
    if (t.lane == WAVE - 1)
      kxr[j] = (y < g.ny && t.c + 2 <= g.nx) ? *t.at(a.Kx, g, t.c + 2, y) : T(0);
  }
  auto ky = [&](int j) { return j < R ? ky_in.get(j < R ? j : 0) : ky_top; };
  __builtin_amdgcn_wave_barrier();
  auto right_face = [&](int j) {
    const T kr = dev::lane_above(kx[j].x), gk = kxr[j];
    return t.lane == WAVE - 1 ? gk : kr;
  };
  auto diagonal = [&](int j, T kr, VT kd, VT ku) {
    VT d;
    d.x = jacobi_den(kx[j].x, kx[j].y, kd.x, ku.x, a.rx, a.ry);
    d.y = jacobi_den(kx[j].y, kr, kd.y, ku.y, a.rx, a.ry);
    return d;
  };
#pragma unroll
  for (int j = 0; j < R; ++j) {
    const VT d = diagonal(j, right_face(j), ky(j), ky(j + 1));
    const bool in = t.y0 + j < g.ny;
    rdi[j].x = in && t.okx ? T(1) / d.x : T(0);
    rdi[j].y = in && t.oky ? T(1) / d.y : T(0);
  }
#pragma unroll
  for (int j = 0; j < R; ++j) {
    u[j] = t.load(a.u, g, t.y0 + j);
    u0.set(j, t.load(a.u0, g, t.y0 + j));
  }
  ResGhost<T> gh = load_ghosts<T, R>(t, g, a.u);
  const bool lead = t.blk == 0 && threadIdx.x == 0;
  T *side = sh.side[t.wave];
  double err = 0.0;
  int reason = 0, n = a.n_first;
  bool dead = false;
  ResOrder<true> o;
  __syncthreads();
  for (;; ++n) {
    if (t.lane < 2 * R) side[t.lane] = gh.side;
    __builtin_amdgcn_wave_barrier();
    double acc = 0.0;
    VT dn = gh.dn, kd = ky(0);
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const VT c = u[j];
      // taller tiles form the diagonal anew: no registers to hold it
      if (R >= 6) {
        asm volatile("" : "+v"(kx[j].x));
        __builtin_amdgcn_sched_barrier(0);
      }
      T l = dev::lane_below(c.y), r = dev::lane_above(c.x);
      const T gl = side[j], gr = side[R + j], kr = right_face(j);
      l = t.lane == 0 ? gl : l;
      r = t.lane == WAVE - 1 ? gr : r;
      const VT up = j + 1 < R ? u[j + 1 < R ? j + 1 : j] : gh.up;
      const VT ku = ky(j + 1);
      const VT s0 = u0.get(j);
      VT b;
      b.x = jacobi_num(s0.x, l, c.y, dn.x, up.x, kx[j].x, kx[j].y, kd.x, ku.x, a.rx, a.ry);
      b.y = jacobi_num(s0.y, c.x, r, dn.y, up.y, kx[j].y, kr, kd.y, ku.y, a.rx, a.ry);
      const VT q = b * rdi[j], di = diagonal(j, kr, kd, ku);
      VT v;
      v.x = fma(fma(-di.x, q.x, b.x), rdi[j].x, q.x);
      v.y = fma(fma(-di.y, q.y, b.y), rdi[j].y, q.y);
      acc += fabs(v.x - c.x) + fabs(v.y - c.y);
      // ... and finish a row before the next, or all rows' operands wait together
      if (R >= 6) asm volatile("" : "+v"(v.x), "+v"(v.y), "+v"(acc));
      dn = c;
      kd = ku;
      u[j] = v;
    }
    double sum;
    if (!dev::res_exchange<true, true>(t, g, sh, o, acc, &sum, &u, &gh)) {
      dead = true;
      break;
    }
    // with other blocks the exchange ends with a barrier, after which the waves'
    // edge rows in LDS may be written again
    if (g.tx * g.ty == 1) __syncthreads();
    err = sqrt(fabs(sum));
    if (lead) a.herr[n] = err;
    const bool conv = err < a.eps_abs, bad = !isfinite(err);
    if (conv || bad || n == a.n_last || n == a.n_pause) {
      reason = conv               ? TL_LOOP_CONVERGED
               : bad              ? TL_LOOP_NONFINITE
               : n == a.n_last    ? TL_LOOP_MAXITERS
                                  : RES_PAUSED;
      break;
    }
  }
  if (dead) {
    if (threadIdx.x == 0) *g.abort_flag = 1;
    return;
  }
  const int col = t.col_anew(), row = t.row_anew();
#pragma unroll
  for (int j = 0; j < R; ++j) t.store(a.u, g, col, row + j, u[j]);
  if (lead) {
    a.ctl->stop = 1;
    a.ctl->reason = reason;
    a.ctl->n_end = n;
    a.ctl->error = err;
  }
}

// ---------------------------------------------------------------------------
// Chebyshev: iterations of tl_cheby_run, up to RES_CHEBY_STEPS in one launch
// ---------------------------------------------------------------------------
// An iteration (kernels/tea_leaf_cheby_kernel.f90:111-200) needs the halos of u
// alone, so its exchange is with the neighbouring blocks only; the sum r.r is
// formed once, at the end of a run.
//
// What bounds it: the exchange with the neighbours, 0.9 us of 1.4 (256^2, one row
// a lane), and from four rows on the arithmetic.  A step of 25 CG and 975
// Chebyshev iterations against passes of ten: 256^2 3.3 -> 2.0 ms, 512^2 3.5 ->
// 2.2, 1024^2 4.6 -> 2.8, 1400^2 5.2 -> 4.0.
constexpr int RES_CHEBY_STEPS = 128;  // coefficients that go along as arguments
struct ChebyArgs {
  ResCheby f;
  int count;
  bool last;               // of the run: w, r and r.r are wanted
  double *norm;            // host memory
  double a[RES_CHEBY_STEPS], b[RES_CHEBY_STEPS];
};
template <int R>
struct ChebyPlan {
  static constexpr bool KY_LDS = R >= 8;  // of 256 registers a field takes 4 a row
  static constexpr size_t BYTES = KY_LDS ? (size_t)R * RES_THREADS * 2 * sizeof(double) : 0;
};

template <int R>
__global__ __launch_bounds__(RES_THREADS) void k_res_cheby(ResGeo g, ChebyArgs a) {
  typedef double T;
  typedef typename dev::Vec<T, 2>::type VT;
  extern __shared__ char dyn[];
  __shared__ ResShared<T, R, 2> sh;
  if (threadIdx.x < 2) sh.dead[threadIdx.x] = 0;
  const ResTile<T, R> t(g);
  ResFaces<T, R, ChebyPlan<R>::KY_LDS> k;
  T *kxr = sh.kxr[t.wave], *side = sh.side[t.wave];
  k.load(t, g, a.f.Kx, a.f.Ky, kxr, (VT *)dyn + threadIdx.x);
  if (ChebyPlan<R>::KY_LDS) __builtin_amdgcn_sched_barrier(0);
  VT u[R], p[R], u0[R];
#pragma unroll
  for (int j = 0; j < R; ++j) {
    u[j] = t.load(a.f.u, g, t.y0 + j);
    p[j] = t.load(a.f.p, g, t.y0 + j);
    u0[j] = t.load(a.f.u0, g, t.y0 + j);
  }
  ResGhost<T> gh = load_ghosts<T, R>(t, g, a.f.u);
  __syncthreads();
  double acc = 0.0;
  const int col = t.col_anew();
  ResOrder<false> o;
  for (int n = 0;; ++n) {
    const bool end = n + 1 == a.count, out = end && a.last;
    const T al = a.a[n], be = a.b[n];
    if (t.lane < 2 * R) side[t.lane] = gh.side;
    __builtin_amdgcn_wave_barrier();
    const int row = t.row_anew();
    VT dn = gh.dn, kd = k.ky(0);
#pragma unroll
    for (int j = 0; j < R; ++j) {
      if (R >= 6) __builtin_amdgcn_sched_barrier(0);
      const VT c = u[j];
      T l = dev::lane_below(c.y), r = dev::lane_above(c.x), kr = dev::lane_above(k.kx[j].x);
      const T gl = side[j], gr = side[R + j], gk = kxr[j];
      l = t.lane == 0 ? gl : l;
      r = t.lane == WAVE - 1 ? gr : r;
      kr = t.lane == WAVE - 1 ? gk : kr;
      const VT up = j + 1 < R ? u[j + 1 < R ? j + 1 : j] : gh.up, ku = k.ky(j + 1);
      VT w;
      w.x = dev::op_cell<false>(c.x, l, c.y, dn.x, up.x, k.kx[j].x, k.kx[j].y, kd.x, ku.x, a.f.rx,
                           a.f.ry);
      w.y = dev::op_cell<false>(c.y, c.x, r, dn.y, up.y, k.kx[j].y, kr, kd.y, ku.y, a.f.rx, a.f.ry);
      const VT res = u0[j] - w;
      if (out) {
        t.store(a.f.w, g, col, row + j, w);
        t.store(a.f.r, g, col, row + j, res);
        acc += res.x * res.x + res.y * res.y;
      }
      p[j] = al * p[j] + be * res;
      u[j] = c + p[j];
      dn = c;
      kd = ku;
    }
    if (end) break;
    if (!dev::res_exchange<true, false>(t, g, sh, o, 0.0, (double *)nullptr, &u, &gh)) {
      if (threadIdx.x == 0) *g.abort_flag = 1;
      return;
    }
  }
  const int row = t.row_anew();
#pragma unroll
  for (int j = 0; j < R; ++j) {
    t.store(a.f.u, g, col, row + j, u[j]);
    t.store(a.f.p, g, col, row + j, p[j]);
  }
  if (!a.last) {
    // a wait that ran out in the last exchange: there is none after it to tell
    __syncthreads();
    if (threadIdx.x == 0 && (sh.dead[0] || sh.dead[1])) *g.abort_flag = 1;
  } else {
    double rr;
    if (!dev::res_exchange<false, true>(t, g, sh, o, acc, &rr,
                                        (const VT(*)[R]) nullptr, (ResGhost<T> *)nullptr)) {
      if (threadIdx.x == 0) *g.abort_flag = 1;
      return;
    }
    if (t.blk == 0 && threadIdx.x == 0) *a.norm = rr;
  }
}

// ---------------------------------------------------------------------------
// PPCG: outer iterations of run_ppcg_loop with their inner steps in one launch
// ---------------------------------------------------------------------------
// The inner steps work on z and z one step before, as k_deep_ppcg's do, and
// need z's halos alone; two sums end an outer iteration (z.r and (r -
// r_store).z) and one its first half.  With a preconditioner M the steps start
// from M^-1 r / theta and add beta M^-1 (r - A z).
//
// What bounds it: with ten inner steps the exchanges, ten of 0.9 us and two of 1.4
// to 2.1, and from four rows a lane on the arithmetic.  Whole steps against the
// passes: 256^2 1.48 -> 0.88 ms, 512^2 2.27 -> 1.38, 1024^2 5.4 -> 2.8; FP32 inside the
// refined solver 256^2 2.4 -> 1.2, 1024^2 6.5 -> 3.1.
constexpr int RES_PPCG_STEPS = 64;  // inner steps whose coefficients go along as arguments
template <typename T>
struct PpcgArgs {
  ResPpcg<T> f;
  T a[RES_PPCG_STEPS], b[RES_PPCG_STEPS];
};
template <typename T, int R>
struct PpcgPlan {
  static constexpr int SIZE = (int)sizeof(T) / 4 * 2 * R;  // registers of one field
  // u, p and r_store are idle during the inner steps: in LDS, of which the
  // tallest tiles have no more than u and p fill
  static constexpr bool LDS = SIZE >= 16, RS_MEMORY = SIZE >= 24;
  static constexpr size_t BYTES =
      LDS ? (size_t)(RS_MEMORY ? 2 : 3) * R * RES_THREADS * 2 * sizeof(T) : 0;
  static_assert(BYTES + sizeof(ResShared<T, R, 2>) <= 160 * 1024, "LDS of a CU");
};

template <typename T, int R, int PREC>
__global__ __launch_bounds__(RES_THREADS) void k_res_ppcg(ResGeo g, PpcgArgs<T> args) {
  typedef typename dev::Vec<T, 2>::type VT;
  constexpr bool DIAG = PREC == TL_PREC_JAC_DIAG, BLK = PREC == TL_PREC_JAC_BLOCK;
  constexpr bool M_REGS = DIAG && R * sizeof(T) < 48;  // else read again in every step
  constexpr bool LDS = PpcgPlan<T, R>::LDS, RS_MEMORY = PpcgPlan<T, R>::RS_MEMORY;
  const ResPpcg<T> &a = args.f;
  extern __shared__ char dyn[];
  __shared__ ResShared<T, R, 2> sh;
  if (threadIdx.x < 2) sh.dead[threadIdx.x] = 0;
  const ResTile<T, R> t(g);
  ResFaces<T, R, false> k;
  T *kxr = sh.kxr[t.wave], *side = sh.side[t.wave];
  Kept<T, R, LDS> u(dyn, 0), p(dyn, 1);
  Kept<T, RS_MEMORY ? 1 : R, LDS && !RS_MEMORY> rs(dyn, 2);
#pragma unroll
  for (int j = 0; j < R; ++j) {
    u.set(j, t.load(a.u, g, t.y0 + j));
    p.set(j, t.load(a.pin, g, t.y0 + j));
  }
  if (LDS) __builtin_amdgcn_sched_barrier(0);
  k.load(t, g, a.Kx, a.Ky, kxr, (VT *)nullptr);
  VT r[R], z[R], zp[R];
#pragma unroll
  for (int j = 0; j < R; ++j) {
    r[j] = t.load(a.r, g, t.y0 + j);
    z[j] = zp[j] = VT(0);
  }
  // Mi; and of the block preconditioner's groups of four rows Di and cp of the
  // first and bfp of the others (cells outside the mesh have bfp = cp = 0, Di = 1)
  VT m[M_REGS ? R : 1], di[BLK ? R / 4 : 1], c0[BLK ? R / 4 : 1], bf[BLK ? R : 1];
  if constexpr (M_REGS)
#pragma unroll
    for (int j = 0; j < R; ++j) m[j] = t.load(a.Mi, g, t.y0 + j);
  if constexpr (BLK)
#pragma unroll
    for (int b = 0; b < R; b += 4) {
      di[b / 4] = t.load(a.Di, g, t.y0 + b);
      c0[b / 4] = t.load(a.cp, g, t.y0 + b);
      if (!t.okx || b >= t.rows) di[b / 4].x = T(1);
      if (!t.oky || b >= t.rows) di[b / 4].y = T(1);
#pragma unroll
      for (int q = 1; q < 4; ++q) bf[b + q] = t.load(a.bfp, g, t.y0 + b + q);
    }
  // M^-1 of a row, or of all rows (tea_block_solve, as in k_res_cg)
  auto mul = [&](int j, VT x, int row) {
    if constexpr (M_REGS) return m[j] * x;
    else if constexpr (DIAG) return t.load(a.Mi, g, row + j) * x;
    else return x;
  };
  auto solve = [&](VT (&x)[R]) {
#pragma unroll
    for (int b = 0; b < R; b += 4) {
      x[b] = x[b] / di[b / 4];
#pragma unroll
      for (int q = 1; q < 4; ++q)
        x[b + q] = (x[b + q] - (-k.ky(b + q) * a.ry) * x[b + q - 1]) * bf[b + q];
#pragma unroll
      for (int q = 2; q >= 0; --q) {
        const VT c = q > 0 ? (-k.ky(b + q + 1) * a.ry) * bf[b + (q > 0 ? q : 1)] : c0[b / 4];
        x[b + q] = b + q + 1 < t.rows ? x[b + q] - c * x[b + q + 1] : x[b + q];
      }
    }
  };
  ResGhost<T> pg = load_ghosts<T, R>(t, g, a.pin), gh;
  const bool lead = t.blk == 0 && threadIdx.x == 0;
  double rro = a.rro, err = 0.0, sums[2] = {0.0, 0.0};
  int reason = 0, n_end = 0;
  bool dead = false, update = false;
  T be = T(0);
  ResOrder<false> o;
  __syncthreads();
  for (int n = a.n_first;; ++n) {
    // ---- w = A p (in z), p.w
    double acc = 0.0;
    {
      VT v[R];
#pragma unroll
      for (int j = 0; j < R; ++j) v[j] = p.get(j);
      if (t.lane < 2 * R) side[t.lane] = pg.side;
      __builtin_amdgcn_wave_barrier();
      dev::res_apply<diff_form<T>()>(t, k, v, pg.dn, pg.up, side, kxr, a.rx, a.ry,
                                     [&](int j, VT w) {
        z[j] = w;
        acc += (double)w.x * (double)v[j].x;
        acc += (double)w.y * (double)v[j].y;
      });
    }
    double pw;
    if (!dev::res_exchange<false, 1>(t, g, sh, o, acc, &pw, (const VT(*)[R]) nullptr,
                                     (ResGhost<T> *)nullptr)) {
      dead = true;
      break;
    }
    if (!isfinite(pw) || !isfinite(rro)) {
      reason = TL_LOOP_NONFINITE;
      n_end = n;
      err = isfinite(pw) ? rro : pw;
      break;
    }
    const T al = (T)(rro / pw);
    const int row = t.row_anew();
#pragma unroll
    for (int j = 0; j < R; ++j) {
      u.set(j, u.get(j) + al * p.get(j));
      if constexpr (RS_MEMORY) t.store(a.r_store, g, t.c, row + j, r[j]);
      else rs.set(j, r[j]);
      r[j] = r[j] - al * z[j];
      z[j] = BLK ? r[j] : mul(j, r[j], row) * a.theta_r;
      zp[j] = VT(0);
    }
    if constexpr (BLK) {
      solve(z);
#pragma unroll
      for (int j = 0; j < R; ++j) z[j] = z[j] * a.theta_r;
    }
    // ---- the inner steps
    for (int i = 0; i < a.inner; ++i) {
      if (!dev::res_exchange<true, 0>(t, g, sh, o, 0.0, (double *)nullptr, &z, &gh)) {
        dead = true;
        break;
      }
      const T ca = args.a[i], cb = args.b[i];
      if (t.lane < 2 * R) side[t.lane] = gh.side;
      __builtin_amdgcn_wave_barrier();
      VT dn = gh.dn, kd = k.ky(0);
      VT d[BLK ? R : 1];
      const int at = t.row_anew();
#pragma unroll
      for (int j = 0; j < R; ++j) {
        if (R * sizeof(T) >= 48) __builtin_amdgcn_sched_barrier(0);
        const VT c = z[j];
        T l = dev::lane_below(c.y), rt = dev::lane_above(c.x), kr = dev::lane_above(k.kx[j].x);
        const T gl = side[j], gr = side[R + j], gk = kxr[j];
        l = t.lane == 0 ? gl : l;
        rt = t.lane == WAVE - 1 ? gr : rt;
        kr = t.lane == WAVE - 1 ? gk : kr;
        const VT up = j + 1 < R ? z[j + 1 < R ? j + 1 : j] : gh.up, ku = k.ky(j + 1);
        VT w;
        w.x = dev::op_cell<diff_form<T>()>(c.x, l, c.y, dn.x, up.x, k.kx[j].x, k.kx[j].y, kd.x,
                                           ku.x, a.rx, a.ry);
        w.y = dev::op_cell<diff_form<T>()>(c.y, c.x, rt, dn.y, up.y, k.kx[j].y, kr, kd.y, ku.y,
                                           a.rx, a.ry);
        if constexpr (BLK) {
          d[j] = r[j] - w;
          dn = c;
          kd = ku;
          continue;
        }
        VT zn = c + ca * (c - zp[j]) + cb * mul(j, r[j] - w, at);
        // a row is finished before the next, or all rows' operands wait together
        if (R * sizeof(T) >= 48) asm volatile("" : "+v"(zn.x), "+v"(zn.y));
        zp[j] = c;
        z[j] = zn;
        dn = c;
        kd = ku;
      }
      if constexpr (BLK) {
        solve(d);
#pragma unroll
        for (int j = 0; j < R; ++j) {
          const VT c = z[j];
          z[j] = c + ca * (c - zp[j]) + cb * d[j];
          zp[j] = c;
        }
      }
    }
    if (dead) break;
    double a0 = 0.0, a1 = 0.0;
    const int back = t.row_anew();
#pragma unroll
    for (int j = 0; j < R; ++j) {
      VT ro;
      if constexpr (RS_MEMORY) ro = t.load(a.r_store, g, back + j);
      else ro = rs.get(j);
      a0 += ((double)r[j].x - (double)ro.x) * (double)z[j].x;
      a0 += ((double)r[j].y - (double)ro.y) * (double)z[j].y;
      a1 += (double)z[j].x * (double)r[j].x;
      a1 += (double)z[j].y * (double)r[j].y;
    }
    if (!dev::res_exchange<true, 2>(t, g, sh, o, a0, sums, &z, &gh, a1)) {
      dead = true;
      break;
    }
    // ---- head of iteration n + 1 (loop_head)
    const double rrn = sums[0], beta = rrn / rro;
    err = sqrt(fabs(rrn));
    const bool bad = !isfinite(rrn), conv = !bad && fabs(err) < a.eps_abs;
    const bool tail = n == a.n_last, pause = n == a.n_pause;
    if (lead) a.herr[n] = err;
    be = (T)beta;
    if (bad || conv || tail || pause) {
      reason = bad    ? TL_LOOP_NONFINITE
               : conv ? TL_LOOP_CONVERGED
               : tail ? TL_LOOP_MAXITERS
                      : RES_PAUSED;
      n_end = n;
      update = true;
      break;
    }
#pragma unroll
    for (int j = 0; j < R; ++j) p.set(j, z[j] + be * p.get(j));
    pg.dn = gh.dn + be * pg.dn;
    pg.up = gh.up + be * pg.up;
    pg.side = gh.side + be * pg.side;
    rro = sums[1];
  }
  if (dead) {
    if (threadIdx.x == 0) *g.abort_flag = 1;
    return;
  }
  const int col = t.col_anew(), row = t.row_anew();
#pragma unroll
  for (int j = 0; j < R; ++j) {
    const int y = row + j;
    t.store(a.u, g, col, y, u.get(j));
    t.store(a.r, g, col, y, r[j]);
    VT pj = p.get(j);
    if (update) {
      pj = z[j] + be * pj;
      t.store(a.z, g, col, y, z[j]);
      if constexpr (!RS_MEMORY) t.store(a.r_store, g, col, y, rs.get(j));
    }
    t.store(a.p, g, col, y, pj);
  }
  if (lead) {
    a.ctl->stop = 1;
    a.ctl->reason = reason;
    a.ctl->n_end = n_end;
    a.ctl->error = err;
    a.ctl->old_error = sums[1];
    a.ctl->rro = sums[0];
  }
}

}  // namespace

namespace tl {

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
namespace {

int env_int(const char *name, int dflt) {
  const char *e = getenv(name);
  return e ? atoi(e) : dflt;
}

__global__ void k_res_clear(u64 *__restrict__ p, long n) {
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n;
       i += (long)gridDim.x * blockDim.x)
    p[i] = 0;
}

constexpr long RES_WORDS = (long)(RES_PARTS + RES_HALOS);

// What a launch tells the host, in the pinned memory of the loops' control
// block copies (drive uses the first three): the kernel writes it there itself,
// and the host needs to wait for the stream only.
struct ResHost {
  Ctl *ctl;
  int *abort_flag;
  double *norm;
};
ResHost res_host() {
  Ctl *hc = (Ctl *)S().hctl;
  static_assert(3 * sizeof(Ctl) + 16 <= 256, "pinned memory of the control block");
  return {&hc[2], (int *)(hc + 3), (double *)(hc + 3) + 1};
}

// What a tiling costs an iteration, in us: `block` for every block, which all
// others wait for, `row` for every row a lane holds, `memory` more where
// preconditioner fields are read again (from `from` rows on).  Fitted to steps
// of 400 CG iterations: 512^2 with 128, 88, 64, 44 and 32 blocks of 2, 3, 4, 6
// and 8 rows 2.16, 2.05, 2.04, 2.29 and 2.54 ms; 640^2 with 200, 100 and 50
// blocks of 2, 4 and 8 rows 2.62, 2.12 and 2.59; 777^2 with jac_diag and 175,
// 119 and 91 blocks of 4, 6 and 8 rows 2.61, 2.86 and 3.00; and of 1000 Jacobi
// iterations: 512^2 with 256, 128, 64 and 44 blocks of 1, 2, 4 and 6 rows 3.21,
// 2.92, 3.11 and 3.63 ms, 1100^2 with 252 and 207 blocks of 5 and 6 rows 4.02 and
// 4.30.  Chebyshev's blocks wait for their neighbours only: 1000 iterations at
// 256^2 with 1, 2, 4 and 8 rows 1.54, 1.70, 1.96 and 3.12.  A single block waits
// for none, and up to 8, one on each XCD, wait 0.2 us less in an exchange (1.2 for
// 1.4 us).
struct ResCost {
  double block, row, memory;
  int from;
};
constexpr ResCost CG_COST = {0.019, 0.42, 0.0, 0}, CG_PREC_COST = {0.019, 0.42, 1.0, 6},
                  JACOBI_COST = {0.0035, 0.2, 0.0, 0}, CHEBY_COST = {0.0, 0.2, 0.0, 0};

// Rows per lane for an nx x ny mesh, of the counts in `rows` (ascending): 0
// when no tiling has at most one block per CU.
int res_rows(int nx, int ny, const int *rows, int nrows, const ResCost &c) {
  const State &s = S();
  const int forced = env_int("TL_RES_ROWS", 0);
  const int cap = s.cus < RES_MAX_BLOCKS ? s.cus : RES_MAX_BLOCKS;
  const long tx = (nx + RES_COLS - 1) / RES_COLS;
  int best = 0;
  double best_cost = 0.0;
  for (int i = 0; i < nrows; ++i) {
    const int R = rows[i];
    const long ty = (ny + (long)RES_WAVES * R - 1) / ((long)RES_WAVES * R), nb = tx * ty;
    if (nb > cap) continue;
    if (forced == R) return R;
    const double wait = nb == 1 ? 0.0 : (nb <= NUM_XCD ? 1.1 : 1.5);
    const double cost = wait + c.block * nb + c.row * R +
                        (c.memory > 0.0 && R >= c.from ? c.memory : 0.0);
    if (!best || cost < best_cost) {
      best = R;
      best_cost = cost;
    }
  }
  return best;
}

constexpr int ROWS64[] = {1, 2, 3, 4, 6, 8}, ROWS64_BLK[] = {4, 8};
constexpr int ROWS32[] = {1, 2, 3, 4, 6, 8, 12, 16};

template <typename T>
int rows_for(int nx, int ny, int prec) {
  if (sizeof(T) == 4) return res_rows(nx, ny, ROWS32, 8, CG_COST);
  const ResCost &c = prec == TL_PREC_NONE ? CG_COST : CG_PREC_COST;
  return prec == TL_PREC_JAC_BLOCK ? res_rows(nx, ny, ROWS64_BLK, 2, c)
                                   : res_rows(nx, ny, ROWS64, 6, c);
}

constexpr int RES_REFUSED = -1;

// One launch of a kernel over a's mesh: cooperatively, so that every block is
// resident when the first one waits (a single block waits for none).  The
// runtime refuses cooperative launches while another process holds the
// device's; the chunk's loops then run the pass kernels from there on, also in the
// middle of a loop, whose launches leave the fields as the passes do.
// `launch`: its number in the loop (TL_RES_REFUSE takes that one as refused).
template <typename A>
int res_launch(int launch, void (*k)(ResGeo, A), ResGeo g, A a, size_t lds) {
  State &s = S();
  const int nb = g.tx * g.ty;
  if (nb == 1) {
    hipLaunchKernelGGL(k, dim3(1), dim3(RES_THREADS), lds, s.stream, g, a);
    TL_HIP(hipGetLastError());
    return TL_OK;
  }
  void *args[] = {&g, &a};
  if (launch != env_int("TL_RES_REFUSE", -1) &&
      hipLaunchCooperativeKernel((const void *)k, dim3(nb), dim3(RES_THREADS), args,
                                 (unsigned)lds, s.stream) == hipSuccess)
    return TL_OK;
  (void)hipGetLastError();
  s.res_refused = true;
  return RES_REFUSED;
}

ResGeo res_geo(int R, long pitch) {
  State &s = S();
  ResGeo g;
  g.nx = s.nx;
  g.ny = s.ny;
  g.pitch = (unsigned)pitch;
  g.tx = (s.nx + RES_COLS - 1) / RES_COLS;
  g.ty = (s.ny + RES_WAVES * R - 1) / (RES_WAVES * R);
  g.part = s.res_mem;
  g.halo = s.res_mem + RES_PARTS;
  g.abort_flag = res_host().abort_flag;
  g.limit = 2000000000LL;  // 20 s
  if (const char *e = getenv("TL_RES_LIMIT")) g.limit = atoll(e);
  return g;
}

// Tags for `exchanges` exchanges; before they run out the buffers start over.
int res_tags(long exchanges, unsigned *epoch) {
  State &s = S();
  if ((u64)s.res_epoch + (u64)exchanges > 0xfffffff0ull) {
    hipLaunchKernelGGL(k_res_clear, dim3(1024), dim3(BLOCK), 0, s.stream, s.res_mem, RES_WORDS);
    TL_HIP(hipGetLastError());
    s.res_epoch = 1;
  }
  *epoch = s.res_epoch;
  s.res_epoch += (unsigned)exchanges;
  return TL_OK;
}

// Wait for a launch; whether a wait of a block ran out.
int res_wait() {
  int *flag = res_host().abort_flag;
  TL_HIP(hipStreamSynchronize(S().stream));
  if (!*flag) return TL_OK;
  *flag = 0;
  return fail(TL_ERR_HIP, "solver loop: a block waited too long for the others");
}

// iterations of one launch: long loops come back to the host in between
int res_chunk() {
  const int c = env_int("TL_RES_CHUNK", 1 << 16);
  return c < 1 ? 1 : (c > 1 << 20 ? 1 << 20 : c);
}

template <typename T, int R, int PREC>
int cg_launch(int launch, const ResGeo &g, const ResCg<T> &a) {
  return res_launch(launch, &k_res_cg<T, R, PREC>, g, a, CgPlan<T, R, PREC>::BYTES);
}

template <typename T>
int cg_dispatch(int launch, int R, int prec, const ResGeo &g, const ResCg<T> &a) {
#define CASE(RR, PP)   if (R == RR && prec == PP) return cg_launch<T, RR, PP>(launch, g, a)
  CASE(1, TL_PREC_NONE);
  CASE(2, TL_PREC_NONE);
  CASE(3, TL_PREC_NONE);
  CASE(4, TL_PREC_NONE);
  CASE(6, TL_PREC_NONE);
  CASE(8, TL_PREC_NONE);
  if constexpr (sizeof(T) == 4) {
    CASE(12, TL_PREC_NONE);
    CASE(16, TL_PREC_NONE);
  } else {
    CASE(1, TL_PREC_JAC_DIAG);
    CASE(2, TL_PREC_JAC_DIAG);
    CASE(3, TL_PREC_JAC_DIAG);
    CASE(4, TL_PREC_JAC_DIAG);
    CASE(6, TL_PREC_JAC_DIAG);
    CASE(8, TL_PREC_JAC_DIAG);
    CASE(4, TL_PREC_JAC_BLOCK);
    CASE(8, TL_PREC_JAC_BLOCK);
  }
#undef CASE
  return fail(TL_ERR_STATE, "solver loop: no kernel for this tiling");
}

}  // namespace

// Kernel timing counts the launches of the pass kernels: while it is on, the
// loops run them.  TL_RESIDENT=0 (read on every call) switches to them too.
static bool resident_on() {
  const State &s = S();
  return s.res_mem && !s.res_refused && !s.prof && !s.passes && env_int("TL_RESIDENT", 1);
}

long resident_words(int nx, int ny) {
  return (rows_for<double>(nx, ny, TL_PREC_NONE) || rows_for<float>(nx, ny, TL_PREC_NONE))
             ? RES_WORDS
             : 0;
}

template <typename T>
int resident_cg(ResCg<T> &a, int prec, long pitch, Ctl *out) {
  State &s = S();
  if (!resident_on()) return 0;
  const int R = rows_for<T>(s.nx, s.ny, prec);
  if (!R) return 0;
  ResGeo g = res_geo(R, pitch);
  a.ctl = res_host().ctl;
  const int chunk = res_chunk();
  for (int k = 0;; ++k) {
    const long left = (long)a.n_last - a.n_first + 1;
    const long run = left < chunk ? left : chunk;
    a.n_pause = (int)(a.n_first + run - 1);
    int rc;
    if ((rc = res_tags(2 * run, &g.epoch))) return -rc;
    rc = cg_dispatch<T>(k, R, prec, g, a);
    if (rc == RES_REFUSED) return 0;
    if (rc || (rc = res_wait())) return -rc;
    *out = *a.ctl;
    if (out->reason != RES_PAUSED) return 1;
    // p has been updated: the next launch starts as a first iteration does
    a.n_first = out->n_end + 1;
    a.rro = out->rro;
    a.pin = a.p;
  }
}
template int resident_cg<double>(ResCg<double> &, int, long, Ctl *);
template int resident_cg<float>(ResCg<float> &, int, long, Ctl *);

int resident_jacobi(ResJacobi &a, long pitch, Ctl *out) {
  State &s = S();
  if (!resident_on()) return 0;
  static constexpr int ROWS[] = {1, 2, 3, 4, 5, 6, 8};
  const int R = res_rows(s.nx, s.ny, ROWS, 7, JACOBI_COST);
  if (!R) return 0;
  ResGeo g = res_geo(R, pitch);
  a.ctl = res_host().ctl;
  const int chunk = res_chunk();
  for (int k = 0;; ++k) {
    const long left = (long)a.n_last - a.n_first + 1;
    const long run = left < chunk ? left : chunk;
    a.n_pause = (int)(a.n_first + run - 1);
    int rc;
    if ((rc = res_tags(run, &g.epoch))) return -rc;
#define CASE(RR) R == RR ? res_launch(k, &k_res_jacobi<RR>, g, a, JacobiPlan<RR>::BYTES)
    rc = CASE(1) : CASE(2) : CASE(3) : CASE(4) : CASE(5) : CASE(6)
         : res_launch(k, &k_res_jacobi<8>, g, a, JacobiPlan<8>::BYTES);
#undef CASE
    if (rc == RES_REFUSED) return 0;
    if (rc || (rc = res_wait())) return -rc;
    *out = *a.ctl;
    if (out->reason != RES_PAUSED) return 1;
    a.n_first = out->n_end + 1;
  }
}

// Runs too short for a launch of more than one block, cooperative and 8 us
// dearer for it: under nine iterations, which the passes do sooner (us without the
// norm, on the chip and by passes: 130^2 2 its 30 and 20, 6 its 36 and 28, 8 its 38
// and 34; 512^2 31 and 22, 38 and 29, 41 and 35; 1400^2 4 its 58 and 45, 8 its 70
// and 49), but for three and five on meshes of a million cells and more, where the
// odd iteration takes a pass of its own (1024^2 42 and 42, 45 and 45; 1400^2 55
// and 59, 62 and 64).  A row count asked for by TL_RES_ROWS is taken for any run.
static bool cheby_short(int count, int blocks) {
  const State &s = S();
  if (blocks == 1 || count >= 9 || env_int("TL_RES_ROWS", 0) > 0) return false;
  const bool large = (double)s.nx * (double)s.ny >= 1e6;
  return !(large && (count == 3 || count == 5));
}

int resident_cheby(const ResCheby &f, const double *alphas, const double *betas, int count,
                   long pitch, bool want_norm, double *norm, int *ran) {
  State &s = S();
  *ran = 0;
  if (!resident_on()) return 0;
  const int R = res_rows(s.nx, s.ny, ROWS64, 6, CHEBY_COST);
  if (!R) return 0;
  ResGeo g = res_geo(R, pitch);
  if (cheby_short(count, g.tx * g.ty)) return 0;
  ChebyArgs a;
  a.f = f;
  a.norm = res_host().norm;
  int rc;
  for (int done = 0, k = 0; done < count; done += a.count, ++k) {
    a.count = count - done < RES_CHEBY_STEPS ? count - done : RES_CHEBY_STEPS;
    a.last = done + a.count == count;
    memcpy(a.a, alphas + done, sizeof(double) * a.count);
    memcpy(a.b, betas + done, sizeof(double) * a.count);
    if ((rc = res_tags(a.count + 1, &g.epoch))) return -rc;
#define CASE(RR) R == RR ? res_launch(k, &k_res_cheby<RR>, g, a, ChebyPlan<RR>::BYTES)
    rc = CASE(1) : CASE(2) : CASE(3) : CASE(4) : CASE(6)
         : res_launch(k, &k_res_cheby<8>, g, a, ChebyPlan<8>::BYTES);
#undef CASE
    if (rc == RES_REFUSED) {
      *ran = done;
      if (done && (rc = res_wait())) return -rc;
      return 0;
    }
    if (rc) return -rc;
  }
  // waited for without the norm too: a wait of a block that ran out is this
  // call's error, and u must not pass on as its result
  if ((rc = res_wait())) return -rc;
  if (want_norm) *norm = *a.norm;
  return 1;
}

template <typename T>
int resident_ppcg(ResPpcg<T> &f, int prec, const double *alphas, const double *betas, long pitch,
                  Ctl *out) {
  State &s = S();
  if (!resident_on() || f.inner < 1 || f.inner > RES_PPCG_STEPS) return 0;
  static constexpr int R64[] = {1, 2, 3, 4, 6}, R32[] = {1, 2, 3, 4, 6, 8, 12}, RBLK[] = {4};
  const ResCost cost = {0.019, 0.2 * (f.inner + 2), 0.0, 0};
  const int R = sizeof(T) == 4                 ? res_rows(s.nx, s.ny, R32, 7, cost)
                : prec == TL_PREC_JAC_BLOCK ? res_rows(s.nx, s.ny, RBLK, 1, cost)
                                            : res_rows(s.nx, s.ny, R64, 5, cost);
  if (!R) return 0;
  ResGeo g = res_geo(R, pitch);
  PpcgArgs<T> a;
  a.f = f;
  a.f.ctl = res_host().ctl;
  for (int i = 0; i < RES_PPCG_STEPS; ++i) {
    a.a[i] = i < f.inner ? (T)alphas[i] : T(0);
    a.b[i] = i < f.inner ? (T)betas[i] : T(0);
  }
  const int chunk = res_chunk();
  for (int k = 0;; ++k) {
    const long left = (long)f.n_last - a.f.n_first + 1;
    const long run = left < chunk ? left : chunk;
    a.f.n_pause = (int)(a.f.n_first + run - 1);
    int rc;
    if ((rc = res_tags((f.inner + 2L) * run, &g.epoch))) return -rc;
#define RUN(RR, PP) res_launch(k, &k_res_ppcg<T, RR, PP>, g, a, PpcgPlan<T, RR>::BYTES)
#define CASE(RR, PP) R == RR ? RUN(RR, PP)
    constexpr int NONE = TL_PREC_NONE, DIAG = TL_PREC_JAC_DIAG, BLK = TL_PREC_JAC_BLOCK;
    if constexpr (sizeof(T) == 4)
      rc = CASE(1, NONE) : CASE(2, NONE) : CASE(3, NONE) : CASE(4, NONE) : CASE(6, NONE)
           : CASE(8, NONE) : RUN(12, NONE);
    else if (prec == BLK)
      rc = RUN(4, BLK);
    else if (prec == DIAG)
      rc = CASE(1, DIAG) : CASE(2, DIAG) : CASE(3, DIAG) : CASE(4, DIAG) : RUN(6, DIAG);
    else
      rc = CASE(1, NONE) : CASE(2, NONE) : CASE(3, NONE) : CASE(4, NONE) : RUN(6, NONE);
#undef CASE
#undef RUN
    if (rc == RES_REFUSED) {
      f = a.f;
      return 0;
    }
    if (rc || (rc = res_wait())) return -rc;
    *out = *a.f.ctl;
    // the sum z.r enters the next iteration; the control block has no other
    // place for it
    const double zr = out->old_error;
    out->old_error = out->error;
    if (out->reason != RES_PAUSED) return 1;
    // p has been updated: the next launch starts as a first iteration does
    a.f.n_first = out->n_end + 1;
    a.f.rro = zr;
    a.f.pin = a.f.p;
  }
}
template int resident_ppcg<double>(ResPpcg<double> &, int, const double *, const double *, long,
                                   Ctl *);
template int resident_ppcg<float>(ResPpcg<float> &, int, const double *, const double *, long,
                                  Ctl *);

}  // namespace tl
