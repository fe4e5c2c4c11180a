// Many steps of a stencil recurrence in one pass over the mesh (temporal
// blocking): PPCG's inner sweeps (k_deep_ppcg) and Chebyshev iterations
// (k_deep_cheby).  The fields are read and written once for all the steps.
//
// A wave walks a strip of 64 V columns upwards on its own, with no barrier.
// Step s ("stage s") runs s rows behind the row being loaded: when row y is
// loaded, stage s turns the field after s steps on rows y-s-2, y-s-1, y-s into
// the field after s + 1 steps on row y-s-1, the last of the three coming from
// stage s - 1 in the same turn.  A stage keeps two rows of the field in
// registers; what the rows hold for all stages in turn (faces, diagonal, right
// hand side) lies for the last STAGES rows in a ring in the wave's own LDS.
// The outermost columns and the first and last STAGES rows of a strip are
// ghosts: each stage's results are wrong one column and row further in, so
// STAGES on every side (rounded up to whole vectors) are walked and thrown
// away.  Faces on the mesh's edge are taken as zero (a mirrored neighbour's two
// terms cancel), and cells outside the mesh as zero with zero faces, so that
// the mesh's edge needs no code in the stages.
#pragma once

#include "tl_stencilv.hpp"

namespace tl {

// Most stages of one kernel: 10 rows x 4 fields x 1 KB of ring per wave are
// the CU's 160 KB for four waves.
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

// The coefficients of the steps, step s's in lane s of vector registers: as
// scalars over the whole unrolled loop they are spilled where the kernel has
// many other scalars (Chebyshev's pass).
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
// ring's length, so that the unrolled rows use fixed registers.  Five rows
// instead of two gained nothing at 4096^2 (PPCG FP64 204 us for 206, FP32 136 for
// 130, Chebyshev 211 for 208).
constexpr int DEEP_AHEAD = 2;

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

// What a wave holds of its strip.  Rows are read and written through buffer
// descriptors of their own, whose length is the mesh's width, or 0 for a row
// that is none: what is read outside is zero and what is written there is
// dropped, in the hardware, so that no lane is masked and no branch splits the
// unrolled rows.  (Masks by bits, a row address per lane and stores behind a
// branch took 60 of the 540 instructions of a row of ten sweeps, and registers
// that the stages' rows then lacked.)
template <typename T, int V, int STAGES>
struct DeepStrip {
  typedef typename Vec<T, V>::type VT;
  typedef unsigned U4 __attribute__((ext_vector_type(4)));
  static_assert(sizeof(VT) == 16, "a lane's columns are one 16-byte access");
  int lane, c;               // first column of the lane
  int y0, y1;                // rows this wave stores
  int first, last;           // rows it loads
  bool live;                 // a tile exists
  bool left_edge, right_edge;  // it has the mesh's first / last column
  bool mine;                 // the lane's columns are the strip's own, and in the mesh
  unsigned off_in, off_out;  // bytes from the row to them; where they are not mine, beyond it
  unsigned face0;            // bits of the lane's first left face: none on the mesh's edge
  int nx, ny;
  long pitch;

  __device__ DeepStrip(const DeepGeo &g, int wave_id) {
    lane = threadIdx.x & (WAVE - 1);
    const int strip = wave_id % g.strips, tile = wave_id / g.strips;
    live = tile < g.tiles;
    constexpr int G = deep_ghost(STAGES, V), S = deep_strip(STAGES, V);
    c = strip * S - G + V * lane;
    nx = g.nx;
    ny = g.ny;
    pitch = g.pitch;
    y0 = tile * g.rows;
    y1 = y0 + g.rows < ny ? y0 + g.rows : ny;
    first = y0 - STAGES > 0 ? y0 - STAGES : 0;
    last = y1 - 1 + STAGES;
    mine = c >= strip * S && c < (strip + 1) * S && c < nx;
    left_edge = strip == 0;
    right_edge = strip == g.strips - 1;
    constexpr unsigned NOWHERE = ~0u - 15u;
    off_in = c < 0 ? NOWHERE : (unsigned)c * (unsigned)sizeof(T);
    off_out = mine ? off_in : NOWHERE;
    face0 = c == 0 ? 0u : ~0u;
  }
  // the row that starts at element `row` of a field; none if !is
  __device__ __amdgpu_buffer_rsrc_t desc(const T *f, long row, bool is) const {
    return __builtin_amdgcn_make_buffer_rsrc((void *)(f + row), 0,
                                             is ? nx * (int)sizeof(T) : 0, 0x00027000);
  }
  __device__ VT load(const T *f, long row, bool is) const {
    return __builtin_bit_cast(
        VT, __builtin_amdgcn_raw_buffer_load_b128(desc(f, row, is), (int)off_in, 0, 0));
  }
  __device__ void store(T *f, long row, VT v, bool is) const {
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(U4, v), desc(f, row, is),
                                           (int)off_out, 0, 0);
  }
  // faces on the left: none on the mesh's edge
  __device__ VT faces_x(VT v) const {
    v[0] = keep(v[0], face0);
    return v;
  }
  // zero unless `row`: by bits and not by a compare per element
  __device__ static VT only_if(VT v, bool row) {
#pragma unroll
    for (int e = 0; e < V; ++e) v[e] = keep(v[e], row ? ~0u : 0u);
    return v;
  }
};

}  // namespace dev
}  // namespace tl
