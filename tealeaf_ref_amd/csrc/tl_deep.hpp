// Many sweeps of a stencil recurrence in one pass over the mesh (temporal
// blocking), for PPCG's inner steps (k_deep_ppcg): `steps` sweeps
//   rtemp -= A sd;  sd' = alpha sd + beta rtemp;  utemp += sd'
// read r and the faces once and write z once, 40 bytes per cell in FP64
// instead of 64 for every two sweeps.
//
// A wave walks a strip of 64 V columns upwards on its own, with no barrier.
// Sweep s ("stage s") runs s rows behind the row being loaded: at the step that
// loads row y, stage s turns sd of sweep s - 1 on rows y-s-1, y-s, y-s+1 into
// sd of sweep s on row y-s, the last of the three coming from stage s - 1 in
// the same step.  Every stage keeps two rows of sd and one of rtemp and utemp
// in registers; the faces and the diagonal of the last STAGES rows, which all
// stages need in turn, lie in a ring in the wave's own LDS.  The outermost
// columns and the first and last STAGES rows of a strip are ghosts: each
// stage's results are wrong one column and row further in, so STAGES on every
// side (rounded up to whole vectors) are walked and thrown away.  Faces on
// the mesh's edge are taken as zero (a mirrored neighbour's two terms
// cancel), and cells outside the mesh as zero with zero faces, so that the
// mesh's edge needs no code in the stages.
#pragma once

#include "tl_stencilv.hpp"

namespace tl {

// Most stages of one kernel: 10 rows x 3 fields x 1 KB of ring per wave are
// 120 KB of the CU's 160 KB for four waves.
constexpr int DEEP_MAX = 10;

template <typename T>
struct DeepCoef {
  T a[DEEP_MAX], b[DEEP_MAX];
};

struct DeepGeo {
  int nx, ny;
  long pitch;
  int strips, tiles, rows;   // strips across; tiles up, of `rows` rows
  int blocks;                // of four waves; wave g: strip g % strips, tile g / strips
};

namespace dev {

// The coefficients of the sweeps, sweep s's in lane s of vector registers: as
// scalars over the whole unrolled loop they would be spilled.
template <typename T>
struct LaneCoef {
  T a, b;
  __device__ explicit LaneCoef(const DeepCoef<T> &co) : a(0), b(0) {
    const int lane = threadIdx.x & (WAVE - 1);
#pragma unroll
    for (int s = 0; s < DEEP_MAX; ++s)
      if (lane == s) {
        a = co.a[s];
        b = co.b[s];
      }
    // from here on only readlane knows what the lanes hold
    asm volatile("" : "+v"(a), "+v"(b));
  }
  static __device__ T pick(T v, int s) {
    if constexpr (sizeof(T) == 8) {
      const unsigned long long q = __builtin_bit_cast(unsigned long long, v);
      const unsigned lo = __builtin_amdgcn_readlane((int)(unsigned)q, s);
      const unsigned hi = __builtin_amdgcn_readlane((int)(unsigned)(q >> 32), s);
      return __builtin_bit_cast(T, (unsigned long long)lo | ((unsigned long long)hi << 32));
    } else {
      return __builtin_bit_cast(T, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), s));
    }
  }
  __device__ T alpha(int s) const { return pick(a, s); }
  __device__ T beta(int s) const { return pick(b, s); }
};

// Rows in flight: loads run this far ahead of the stages.  A divisor of the
// ring's length, so that the unrolled rows use fixed registers.
constexpr int deep_ahead(int stages) {
  (void)stages;
  return 2;
}

constexpr int deep_ghost(int stages, int V) { return (stages + V - 1) / V * V; }
constexpr int deep_strip(int stages, int V) { return WAVE * V - 2 * deep_ghost(stages, V); }

// The neighbouring lanes' values; lane 0 and lane 63 get 0.  Unlike
// dpp_shift, whose lane without a source keeps its own value, this needs no
// copy before the move.
template <int CTRL, typename T>
__device__ inline T dpp_zero(T v) {
  if constexpr (sizeof(T) == 8) {
    const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo =
        (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)b, CTRL, 0xF, 0xF, true);
    const unsigned hi =
        (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)(b >> 32), CTRL, 0xF, 0xF, true);
    return __builtin_bit_cast(T, (unsigned long long)lo | ((unsigned long long)hi << 32));
  } else {
    return __builtin_bit_cast(
        T, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
  }
}
template <typename T>
__device__ inline T from_below(T v) { return dpp_zero<0x138>(v); }  // wave_shr:1
template <typename T>
__device__ inline T from_above(T v) { return dpp_zero<0x130>(v); }  // wave_shl:1

template <typename T, int V>
__device__ inline T vec_left(const typename Vec<T, V>::type &v, int e, T below) {
  return e == 0 ? below : v[e > 0 ? e - 1 : 0];
}
template <typename T, int V>
__device__ inline T vec_right(const typename Vec<T, V>::type &v, int e, T above) {
  return e + 1 < V ? v[e + 1 < V ? e + 1 : e] : above;
}

// Bits of a value kept where the mask is set.
template <typename T>
__device__ inline T keep(T v, unsigned m) {
  if constexpr (sizeof(T) == 8) {
    const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = (unsigned)b & m, hi = (unsigned)(b >> 32) & m;
    return __builtin_bit_cast(T, (unsigned long long)lo | ((unsigned long long)hi << 32));
  } else {
    return __builtin_bit_cast(T, __builtin_bit_cast(unsigned, v) & m);
  }
}

// What a wave holds of its strip.
template <typename T, int V, int STAGES>
struct DeepStrip {
  typedef typename Vec<T, V>::type VT;
  int lane, c;               // first column of the lane
  unsigned off;              // bytes from the row to it, clamped into the row
  int y0, y1;                // rows this wave stores
  int first, last;           // rows it loads
  bool live;                 // a tile exists
  bool left_edge, right_edge;  // it has the mesh's first / last column
  bool out, part;            // the lane's columns are stored; only some of them
  bool any_part;             // ... in some lane of the wave
  unsigned in[V], face[V];   // the lane's cells in the mesh; with a face on the left
  int nx, ny;
  long pitch;

  __device__ DeepStrip(const DeepGeo &g, int wave_id) {
    lane = threadIdx.x & (WAVE - 1);
    const int strip = wave_id % g.strips, tile = wave_id / g.strips;
    live = tile < g.tiles;
    constexpr int G = deep_ghost(STAGES, V), S = deep_strip(STAGES, V);
    const int x0 = strip * S - G;
    c = x0 + V * lane;
    nx = g.nx;
    ny = g.ny;
    pitch = g.pitch;
    const int top = (nx / V) * V;
    off = (unsigned)(c < 0 ? 0 : (c > top ? top : c)) * (unsigned)sizeof(T);
    y0 = tile * g.rows;
    y1 = y0 + g.rows < ny ? y0 + g.rows : ny;
    first = y0 - STAGES > 0 ? y0 - STAGES : 0;
    last = y1 - 1 + STAGES;
    out = c >= strip * S && c < (strip + 1) * S && c < nx;
    part = out && c + V > nx;
    left_edge = strip == 0;
    right_edge = strip == g.strips - 1;
    any_part = __any(part);
    out = out && !part;
#pragma unroll
    for (int e = 0; e < V; ++e) {
      in[e] = c + e >= 0 && c + e < nx ? ~0u : 0u;
      face[e] = c + e > 0 && c + e < nx ? ~0u : 0u;
    }
  }
  // the lane's cells of a row that starts at element `row` of a field
  __device__ VT load(const T *__restrict__ f, long row) const {
    return *(const VT *)((const char *)(f + row) + off);
  }
  // zero where the mesh is not: by bits and not by compares, whose masks
  // would fill the scalar registers over the unrolled rows
  __device__ static VT masked(VT v, const unsigned (&m)[V], bool row) {
    const unsigned r = row ? ~0u : 0u;
#pragma unroll
    for (int e = 0; e < V; ++e) v[e] = keep(v[e], m[e] & r);
    return v;
  }
  __device__ VT cells(VT v, int y) const { return masked(v, in, y < ny); }
  __device__ VT cells_if(VT v, bool row) const { return masked(v, in, row); }
  __device__ VT faces_x(VT v, int y) const { return masked(v, face, y < ny); }
  __device__ VT faces_y(VT v, int y) const { return masked(v, in, y > 0 && y < ny); }
  // Rows that are not stored (ok false) pass through the same instructions with
  // no lane on: a branch around the store would leave the compiler unsure how
  // many are in flight, and it would then wait for them with the loads.
  __device__ void store(T *f, long row, VT v, bool ok) const {
    if (out & ok) *(VT *)((char *)(f + row) + off) = v;
    if (any_part) {
      if (part & ok) stv<false, T, V>(f + row, c, nx, v);
    }
  }
};

}  // namespace dev
}  // namespace tl
