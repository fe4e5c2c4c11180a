// Solver loops that keep the whole mesh on the chip: one block per CU holds a
// tile of every field in its registers and LDS for the whole loop, and the
// blocks exchange halos and partial sums through device memory while the
// kernel runs.
//
// Why: on meshes of up to about two million cells a pass of the
// kernel-per-pass loops (tl_loopk.hpp) is bound by latency, not by bytes:
// launch, the sum of the previous pass's partials, the dependent loads, the
// block reduction (512^2: 12.5 us per CG iteration for 25 MB).  256 CUs hold
// 128 MB of registers and 40 MB of LDS, and an all-to-all sum of one double
// per block takes 1.4 us at 128 blocks and 2.1 us at 256 (0.9 us for an
// exchange with the neighbours alone), against about 6 us per pass.
//
// Exchange.  Every value crosses as 64-bit words of 32 payload bits and a
// 32-bit tag, written and read with relaxed atomics of agent scope: a reader
// that finds the tag of the current exchange has the payload, so neither
// fences nor flags are needed, and a word is never read half written.  Tags
// count up over the life of the chunk, and the buffers start as zeros.  There
// are two copies of them, so that no word is written again before its readers
// have it (tl_res_order.hpp).
//
// The grid never exceeds one block per CU and is launched cooperatively, so
// that all blocks are resident; a wait that lasts longer than `limit` ticks of
// the 100 MHz clock sets the abort word and every block leaves the kernel.
#pragma once

#include "tl_loopk.hpp"
#include "tl_res_order.hpp"

namespace tl {

typedef unsigned long long u64;

constexpr int RES_WAVES = 8;                 // waves per block, stacked in y
constexpr int RES_THREADS = RES_WAVES * WAVE;
constexpr int RES_COLS = 2 * WAVE;           // two columns per lane
constexpr int RES_MAX_BLOCKS = 256;
constexpr int RES_MAX_ROWS = 16;             // rows per lane at most
constexpr int RES_PART_WORDS = 16;           // words between two blocks' partials: a 128-byte line each
// words of one block's halo: two rows of 128 and two sides of 8 x 16 values
constexpr int RES_HALO_WORDS = 2 * (2 * RES_COLS + 2 * RES_WAVES * RES_MAX_ROWS);
constexpr size_t RES_PARTS = 2 * (size_t)RES_MAX_BLOCKS * RES_PART_WORDS;
constexpr size_t RES_HALOS = 2 * (size_t)RES_MAX_BLOCKS * RES_HALO_WORDS;

struct ResGeo {
  int nx, ny;
  unsigned pitch;          // in elements of the field type
  int tx, ty;              // tiles across and up: block b has tile (b % tx, b / tx)
  unsigned epoch;          // tag of the first exchange
  u64 *part, *halo;
  int *abort_flag;
  long long limit;         // ticks of the 100 MHz clock a wait may last
};

namespace dev {

// ---- sums over a wave with DPP (every lane returns the total) ------------------
template <int CTRL, int ROWS>
__device__ inline double dpp_add(double v) {
  const u64 b = __builtin_bit_cast(u64, v);
  const unsigned lo =
      (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)b, CTRL, ROWS, 0xF, true);
  const unsigned hi =
      (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)(b >> 32), CTRL, ROWS, 0xF, true);
  return v + __builtin_bit_cast(double, (u64)lo | ((u64)hi << 32));
}
// The shuffles of wave_sum go through the LDS crossbar (6 dependent steps of
// about 100 cycles); row shifts and broadcasts stay in the VALU.
__device__ inline double wave_total(double v) {
  v = dpp_add<0x111, 0xF>(v);  // row_shr:1
  v = dpp_add<0x112, 0xF>(v);  // row_shr:2
  v = dpp_add<0x114, 0xF>(v);  // row_shr:4
  v = dpp_add<0x118, 0xF>(v);  // row_shr:8: lane 15 of each row has its sum
  v = dpp_add<0x142, 0xA>(v);  // row_bcast:15 into rows 1 and 3
  v = dpp_add<0x143, 0xC>(v);  // row_bcast:31 into rows 2 and 3: lane 63 has the total
  const u64 b = __builtin_bit_cast(u64, v);
  const unsigned lo = __builtin_amdgcn_readlane((int)(unsigned)b, WAVE - 1);
  const unsigned hi = __builtin_amdgcn_readlane((int)(unsigned)(b >> 32), WAVE - 1);
  return __builtin_bit_cast(double, (u64)lo | ((u64)hi << 32));
}
// neighbouring lanes' values (lane 0 / lane 63 get their own)
template <typename T>
__device__ inline T lane_below(T v) { return dpp_shift<0x138>(v); }  // wave_shr:1
template <typename T>
__device__ inline T lane_above(T v) { return dpp_shift<0x130>(v); }  // wave_shl:1

// ---- tagged words -------------------------------------------------------------------
// Word i of a buffer, its byte offset in 32 bits: one register per address
// instead of two.
__device__ inline u64 *word(u64 *base, unsigned i) { return (u64 *)((char *)base + 8u * i); }
__device__ inline void put(u64 *base, unsigned i, unsigned payload, unsigned tag) {
  __hip_atomic_store(word(base, i), ((u64)payload << 32) | tag, __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline u64 get(u64 *base, unsigned i) {
  return __hip_atomic_load(word(base, i), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// words per value: a double takes two
template <typename T>
constexpr int res_words() { return sizeof(T) == 8 ? 2 : 1; }
// store a value at word i of a run of n values (word planes of n, so lanes
// write consecutive words)
template <typename T>
__device__ inline void put_value(u64 *base, int n, unsigned i, T v, unsigned tag) {
  if constexpr (sizeof(T) == 8) {
    const u64 b = __builtin_bit_cast(u64, v);
    put(base, i, (unsigned)b, tag);
    put(base, i + n, (unsigned)(b >> 32), tag);
  } else {
    put(base, i, __builtin_bit_cast(unsigned, v), tag);
  }
}
template <typename T>
struct Words {
  u64 w[res_words<T>()];
};
template <typename T>
__device__ inline Words<T> get_words(u64 *base, int n, unsigned i) {
  Words<T> o;
  o.w[0] = get(base, i);
  if constexpr (sizeof(T) == 8) o.w[1] = get(base, i + n);
  return o;
}
template <typename T>
__device__ inline bool tagged(const Words<T> &o, unsigned tag) {
  bool ok = (unsigned)o.w[0] == tag;
  if constexpr (sizeof(T) == 8) ok = ok && (unsigned)o.w[1] == tag;
  return ok;
}
template <typename T>
__device__ inline T value_of(const Words<T> &o) {
  if constexpr (sizeof(T) == 8)
    return __builtin_bit_cast(double, (o.w[0] >> 32) | (o.w[1] & 0xffffffff00000000ull));
  else
    return __builtin_bit_cast(T, (unsigned)(o.w[0] >> 32));
}

// One block's LDS besides the fields it keeps there.  What one wave writes for
// others is indexed by the exchange's or the sum's parity (EB = 1 for the edge
// rows where every second exchange has none): a wave that is an exchange ahead never
// writes what another still reads.
template <typename T, int R, int EB>
struct ResShared {
  typedef typename Vec<T, 2>::type VT;
  double red[2][2][RES_WAVES], tot[2][2][RES_WAVES];  // [parity][sum][wave]
  int dead[2];                       // a wait of this block has run out
  VT bottom[EB][RES_WAVES][WAVE], top[EB][RES_WAVES][WAVE];  // edge rows of every wave
  T side[RES_WAVES][2 * R];          // ghost columns: left rows, then right rows
  T kxr[RES_WAVES][R];               // Kx right of the tile
};

// What one lane needs to know of the tile it holds.
template <typename T, int R>
struct ResTile {
  typedef typename Vec<T, 2>::type VT;
  int lane, wave, blk, bx, by;
  int c, y0, rows;                   // first column; first row and rows inside the mesh
  bool okx, oky;                     // the lane's two columns lie in the mesh
  bool left, right, below, above;    // neighbouring tiles exist

  __device__ explicit ResTile(const ResGeo &g) {
    lane = threadIdx.x & (WAVE - 1);
    // uniform in the wave, which keeps the row tests in scalar registers
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    blk = blockIdx.x;
    bx = blk % g.tx;
    by = blk / g.tx;
    c = bx * RES_COLS + 2 * lane;
    y0 = (by * RES_WAVES + wave) * R;
    rows = g.ny - y0;
    rows = rows < 0 ? 0 : (rows > R ? R : rows);
    okx = c < g.nx;
    oky = c + 1 < g.nx;
    left = bx > 0;
    right = bx + 1 < g.tx;
    below = by > 0;
    above = by + 1 < g.ty;
  }
  // Cell (col, y) of a field: the row is the same for the whole wave, so its
  // address stays in scalar registers and a lane's part takes one register.
  __device__ static const T *at(const T *f, const ResGeo &g, int col, int y) {
    const char *row = (const char *)f + (unsigned)y * g.pitch * (unsigned)sizeof(T);
    return (const T *)(row + (unsigned)col * (unsigned)sizeof(T));
  }
  // Row y of a field through a buffer descriptor whose length is the mesh's
  // width, or 0 for a row that is none: what is read outside the mesh is zero
  // and what is written there is dropped, in the hardware.
  __device__ static __amdgpu_buffer_rsrc_t desc(const T *f, const ResGeo &g, int y) {
    return __builtin_amdgcn_make_buffer_rsrc((void *)at(f, g, 0, y), 0,
                                             y >= 0 && y < g.ny ? g.nx * (int)sizeof(T) : 0,
                                             0x00027000);
  }
  __device__ VT load(const T *f, const ResGeo &g, int y) const {
    const int off = c * (int)sizeof(T);
    if constexpr (sizeof(T) == 8)
      return __builtin_bit_cast(VT, __builtin_amdgcn_raw_buffer_load_b128(desc(f, g, y), off, 0, 0));
    else
      return __builtin_bit_cast(VT, __builtin_amdgcn_raw_buffer_load_b64(desc(f, g, y), off, 0, 0));
  }
  // column `col` is c, handed in anew after the loop so that no address of
  // the first loads is kept in registers for the stores
  __device__ void store(T *f, const ResGeo &g, int col, int y, VT v) const {
    typedef unsigned U __attribute__((ext_vector_type(sizeof(VT) / 4)));
    const int off = col * (int)sizeof(T);
    if constexpr (sizeof(T) == 8)
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(U, v), desc(f, g, y), off, 0, 0);
    else
      __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(U, v), desc(f, g, y), off, 0, 0);
  }
  // the first row, anew for the same reason (and no row's address in scalar ones)
  __device__ int row_anew() const {
    int y = y0;
    asm volatile("" : "+s"(y));
    return y;
  }
  __device__ int col_anew() const {
    int col = c;
    asm volatile("" : "+v"(col));
    return col;
  }
};

// The face coefficients of a lane's cells: kx[j] left of its two columns
// (the face right of the second is the next lane's, and in lane 63 in LDS),
// ky below row j (row R: above the last), in registers or, with KY_LDS, in the
// block's dynamic LDS.  Faces on the mesh's edge are taken as zero: with
// reflective faces the mirrored cell has the cell's own value, so their two
// terms cancel; cells outside the mesh then have no face at all.
template <typename T, int R, bool KY_LDS>
struct ResFaces {
  typedef typename Vec<T, 2>::type VT;
  VT kx[R], ky_top;
  VT ky_r[KY_LDS ? 1 : R];
  VT *ky_l;

  __device__ void load(const ResTile<T, R> &t, const ResGeo &g, const T *Kx, const T *Ky,
                       T *kxr, VT *lds) {
    ky_l = lds;
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const int y = t.y0 + j;
      kx[j] = t.load(Kx, g, y);
      if (t.c == 0) kx[j].x = T(0);
      if (t.lane == WAVE - 1) kxr[j] = (y < g.ny && t.c + 2 < g.nx) ? *t.at(Kx, g, t.c + 2, y) : T(0);
      const VT v = y > 0 ? t.load(Ky, g, y) : VT(0);
      if constexpr (KY_LDS) ky_l[j * RES_THREADS] = v;
      else ky_r[j] = v;
    }
    ky_top = t.load(Ky, g, t.y0 + R);
  }
  __device__ VT ky(int j) const {
    if constexpr (KY_LDS) return j < R ? ky_l[j * RES_THREADS] : ky_top;
    else return j < R ? ky_r[j < R ? j : 0] : ky_top;
  }
};

// A applied to a lane's cells: v[0..R-1] with the rows `dn` and `up` beyond
// them and the ghost columns in `side` (left rows, then right rows).
// body(j, w) takes row j's result, which is 0 in cells outside the mesh.
template <bool DIFF, typename T, int R, bool KY_LDS, typename BODY>
__device__ inline void res_apply(const ResTile<T, R> &t, const ResFaces<T, R, KY_LDS> &k,
                                 const typename Vec<T, 2>::type (&v)[R],
                                 typename Vec<T, 2>::type dn, typename Vec<T, 2>::type up,
                                 const T *side, const T *kxr, T rx, T ry, BODY body) {
  typedef typename Vec<T, 2>::type VT;
  VT kd = k.ky(0);
#pragma unroll
  for (int j = 0; j < R; ++j) {
    T l = lane_below(v[j].y), r = lane_above(v[j].x), kr = lane_above(k.kx[j].x);
    // every lane reads the same word: no divergence, no bank conflict
    const T gl = side[j], gr = side[R + j], gk = kxr[j];
    l = t.lane == 0 ? gl : l;
    r = t.lane == WAVE - 1 ? gr : r;
    kr = t.lane == WAVE - 1 ? gk : kr;
    const VT d = j > 0 ? v[j > 0 ? j - 1 : 0] : dn;
    const VT u = j + 1 < R ? v[j + 1 < R ? j + 1 : j] : up;
    const VT ku = k.ky(j + 1);
    VT w;
    w.x = op_cell<DIFF>(v[j].x, l, v[j].y, d.x, u.x, k.kx[j].x, k.kx[j].y, kd.x, ku.x, rx, ry);
    w.y = op_cell<DIFF>(v[j].y, v[j].x, r, d.y, u.y, k.kx[j].y, kr, kd.y, ku.y, rx, ry);
    kd = ku;
    body(j, w);
  }
}

// The ghosts of a lane: the rows beyond its wave's, and (in lanes 0..2R-1)
// one cell each of the ghost columns.
template <typename T>
struct ResGhost {
  typedef typename Vec<T, 2>::type VT;
  VT dn, up;
  T side;
};

// The loop's next exchange, number o.s.  HALO: the
// edges of `v` go to the neighbours and their edges come back in `gh`.  SUM:
// returns one or two sums of `part` (and `part2`) over the lanes of all blocks,
// added in one fixed order everywhere, so every block has the same bits.  Returns false in
// every wave of a block when a wait of the block has run out (in a wave that
// waits for halos alone, one exchange later).
template <bool HALO, int SUM, typename T, int R, int EB, typename ORDER>
__device__ inline bool res_exchange(const ResTile<T, R> &t, const ResGeo &g,
                                    ResShared<T, R, EB> &sh, ORDER &o, double part, double *total,
                                    const typename Vec<T, 2>::type (*v)[R], ResGhost<T> *gh,
                                    double part2 = 0.0) {
  typedef typename Vec<T, 2>::type VT;
  static_assert(SUM > 0 || !ORDER::every_sums, "the loop's order");
  const int buf = o.halos(), sb = o.sums();  // the exchange's parity, and the sum's
  const int eb = EB > 1 ? buf : 0;
  constexpr int SIDE = RES_WAVES * R;        // values of one side
  const unsigned tag = o.tag(g.epoch);
  o.next(SUM > 0);
  const int nb = g.tx * g.ty;
  // the tallest tiles form their addresses anew in every exchange: no registers
  // to hold them through the loop
  int lane = t.lane;
  if (R * sizeof(T) >= 64) asm volatile("" : "+v"(lane));
  u64 *parts = g.part + sb * (RES_MAX_BLOCKS * RES_PART_WORDS);
  u64 *halos = g.halo + buf * (RES_MAX_BLOCKS * RES_HALO_WORDS);
  constexpr int W = res_words<T>();
  // runs of a block's halo: bottom row, top row, left side, right side
  constexpr int RUN_B = 0, RUN_T = W * RES_COLS, RUN_L = 2 * W * RES_COLS,
                RUN_R = RUN_L + W * SIDE;
  if constexpr (HALO) {
    const VT vb = (*v)[0], vt = (*v)[R - 1];
    sh.bottom[eb][t.wave][lane] = vb;
    sh.top[eb][t.wave][lane] = vt;
    u64 *mine = halos + t.blk * RES_HALO_WORDS;
    if (t.wave == 0 && t.below) {
      put_value<T>(mine, RES_COLS, RUN_B + lane, vb.x, tag);
      put_value<T>(mine, RES_COLS, RUN_B + WAVE + lane, vb.y, tag);
    }
    if (t.wave == RES_WAVES - 1 && t.above) {
      put_value<T>(mine, RES_COLS, RUN_T + lane, vt.x, tag);
      put_value<T>(mine, RES_COLS, RUN_T + WAVE + lane, vt.y, tag);
    }
    // the wave's edge columns, moved to lanes 0..2R-1
    T *sd = sh.side[t.wave];
    if (lane == 0 || lane == WAVE - 1) {
      const int off = lane == 0 ? 0 : R;
#pragma unroll
      for (int j = 0; j < R; ++j) sd[off + j] = lane == 0 ? (*v)[j].x : (*v)[j].y;
    }
    __builtin_amdgcn_wave_barrier();
    if (lane < 2 * R) {
      const T e = sd[lane];
      const bool lft = lane < R;
      const int i = t.wave * R + (lft ? lane : lane - R);
      if (lft ? t.left : t.right) put_value<T>(mine, SIDE, (lft ? RUN_L : RUN_R) + i, e, tag);
    }
  }
  if constexpr (SUM > 0) {
    part = wave_total(part);
    if (SUM > 1) part2 = wave_total(part2);
    if (lane == 0) {
      sh.red[sb][0][t.wave] = part;
      if (SUM > 1) sh.red[sb][1][t.wave] = part2;
    }
  }
  __syncthreads();
  double own[2] = {0.0, 0.0};
  if constexpr (SUM > 0) {
#pragma unroll
    for (int m = 0; m < SUM; ++m)
#pragma unroll
      for (int i = 0; i < RES_WAVES; ++i) own[m] += sh.red[sb][m][i];
    if (nb > 1 && t.wave == 0 && lane < 2 * SUM) {
      const u64 b = __builtin_bit_cast(u64, SUM > 1 && lane >= 2 ? own[1] : own[0]);
      put(parts, t.blk * RES_PART_WORDS + lane, lane & 1 ? (unsigned)(b >> 32) : (unsigned)b, tag);
    }
  }
  // ---- wait for the others: lanes of waves 1.. take one block's partial each
  // (waves 0 and 7 are busy with the rows), lanes 0..2R-1 of every wave one
  // ghost cell of the sides
  if constexpr (HALO) {
    gh->dn = t.wave > 0 ? sh.top[eb][t.wave > 0 ? t.wave - 1 : 0][lane] : VT(0);
    gh->up = t.wave < RES_WAVES - 1
                 ? sh.bottom[eb][t.wave < RES_WAVES - 1 ? t.wave + 1 : 0][lane]
                 : VT(0);
    gh->side = T(0);
  }
  const int from = (int)threadIdx.x - WAVE;  // the block this lane takes a partial of
  const bool want_p = SUM > 0 && nb > 1 && from >= 0 && from < nb;
  const bool want_b = HALO && t.wave == 0 && t.below;
  const bool want_t = HALO && t.wave == RES_WAVES - 1 && t.above;
  const bool lft = lane < R;
  const bool want_s = HALO && lane < 2 * R && (lft ? t.left : t.right);
  double q[2] = {0.0, 0.0};
  if (want_p || want_b || want_t || want_s) {
    const unsigned pp = (want_p ? from : 0) * RES_PART_WORDS;
    unsigned pr = 0, ps = 0;
    if constexpr (HALO) {
      if (want_b) pr = (t.blk - g.tx) * RES_HALO_WORDS + RUN_T + lane;
      if (want_t) pr = (t.blk + g.tx) * RES_HALO_WORDS + RUN_B + lane;
      if (want_s)
        ps = (lft ? t.blk - 1 : t.blk + 1) * RES_HALO_WORDS + (lft ? RUN_R : RUN_L) + t.wave * R +
             (lft ? lane : lane - R);
    }
    Words<double> a[2] = {};
    Words<T> r0 = {}, r1 = {}, sw = {};
    int spins = 0;
    long long t_start = 0;
    for (;;) {
      if (want_p)
#pragma unroll
        for (int m = 0; m < SUM; ++m) {
          a[m].w[0] = get(parts, pp + 2 * m);
          a[m].w[1] = get(parts, pp + 2 * m + 1);
        }
      if constexpr (HALO) {
        if (want_b || want_t) {
          r0 = get_words<T>(halos, RES_COLS, pr);
          r1 = get_words<T>(halos, RES_COLS, pr + WAVE);
        }
        if (want_s) sw = get_words<T>(halos, SIDE, ps);
      }
      bool ok = !want_p || (tagged<double>(a[0], tag) && (SUM < 2 || tagged<double>(a[1], tag)));
      if constexpr (HALO) {
        if (want_b || want_t) ok = ok && tagged<T>(r0, tag) && tagged<T>(r1, tag);
        if (want_s) ok = ok && tagged<T>(sw, tag);
      }
      if (ok && g.limit >= 0) break;  // a negative limit lets every wait run out
      if ((++spins & 1023) == 0) {
        const long long now = wall_clock64();
        if (t_start == 0) t_start = now;
        if (now - t_start > g.limit) {
          sh.dead[buf] = 1;
          break;
        }
      }
    }
    if (want_p)
#pragma unroll
      for (int m = 0; m < SUM; ++m) q[m] = value_of<double>(a[m]);
    if constexpr (HALO) {
      VT row;
      row.x = value_of<T>(r0);
      row.y = value_of<T>(r1);
      if (want_b) gh->dn = row;
      if (want_t) gh->up = row;
      if (want_s) gh->side = value_of<T>(sw);
    }
  }
  if constexpr (SUM > 0) {
    if (nb > 1) {
      const int waves = (nb + WAVE - 1) / WAVE;  // waves 1..waves hold partials
      if (t.wave >= 1 && t.wave <= waves)
#pragma unroll
        for (int m = 0; m < SUM; ++m) {
          q[m] = wave_total(q[m]);
          if (lane == 0) sh.tot[sb][m][t.wave - 1] = q[m];
        }
      __syncthreads();
#pragma unroll
      for (int m = 0; m < SUM; ++m) {
        own[m] = 0.0;
        for (int i = 0; i < waves; ++i) own[m] += sh.tot[sb][m][i];
      }
      if (sh.dead[0] || sh.dead[1]) return false;  // this one, or one for halos alone before
    }
#pragma unroll
    for (int m = 0; m < SUM; ++m) total[m] = own[m];
    return true;
  }
  // no second barrier: what the exchange before found is settled
  return !sh.dead[buf ^ 1];
}

}  // namespace dev
}  // namespace tl
