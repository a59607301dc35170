// Temporal-blocked Gauss-Seidel/SOR pressure solve for gfx950, bit-identical to the
// reference's serial in-place sweeps (pressureJacobiIteration, fluid.go:188-234).
//
// Cell (i,j) of sweep k needs (i-1,j,k), (i,j-1,k), (i+1,j,k-1), (i,j+1,k-1) and (i,j,k-1).
// With skewed rows i' = i + k these become forward dependences in (i', k), plus a
// j-lag of at most one column. A tile is 64 skewed rows (the lanes a) by TK = W x S sweeps;
// a wave holds S of them in registers and marches along j: at step s it updates, for each of
// its sweeps b, the cells (i = i0 + a - b, j = s - a - b) of sweep k0 + b. Every face then
// travels as follows:
//   U right face, after the update, -> (a+1, b)   at s+1   (DPP wave_shr:1)
//   U left face                     -> (a, b+1)   at s+1   (register; LDS to the next wave)
//   V bottom face and p             -> (a+1, b+1) at s+1   (DPP wave_shr:1; p is used at s+2)
//   V top face                      -> (a, b) itself       (register)
// Within a step the sweeps run from the last to the first, so each takes what its predecessor
// left in registers at the step before, and the S updates of a step are independent: a wave
// needs no barrier and no LDS round trip between its sweeps. Only a wave's first sweep (from the
// wave before it) and its lane 0 (from the tile one row-tile up) read LDS, two steps ahead.
//
// The solve is a wavefront over a chain of dependent steps, so its time is steps times the time
// of a step, not memory or arithmetic rate; and a step is the issue of one wave's instructions: a
// lone wave issues an independent vector instruction every 4.7 cycles, a dependent one after 8,
// a 16-byte LDS write takes 28 and a 4-byte one 16 (measured). So a step is about 18 vector
// instructions per sweep and the few LDS accesses around them: 160 cycles for one sweep to a
// wave, 270 for two, and 60 more for its share of the block's loads, checks and barrier; one
// sweep a wave with a barrier a step took 640.
//
// The waves of a workgroup run one block of B steps apart, with one barrier per block: wave
// w runs block n while wave w-1 runs block n+1 into the other half of their LDS buffer. Between
// tiles the boundary goes through global memory: per step the three faces and p of lane 63 of
// each sweep (the G stream, for the tile one row-tile up) and the last wave's 64 lanes (the K
// stream, for the next TK sweeps). Each cell's values are one 16-byte word with a tag, the number
// of the solve, in each half, and the consumer loads the words until they carry the tag of this
// solve. So a handoff costs one trip of the data: no wait for stores, no progress counters, no
// polls beside the loads themselves. A block's words are loaded while the block before it runs.
// The compiler has to know how many stores were issued since a load to wait for the load alone, so
// every path of a block issues the same loads and stores, under branches that it sees are uniform
// (with a wait for the stores 256^2 took 0.180 ms a solve, 512^2 0.540). Tiles run as a persistent
// kernel in ticket order (a topological order of the tile graph), so whatever a workgroup waits for was
// taken earlier by a workgroup that runs, or (queue_of_tiles) will be by one that has started.
// k_gs_skew lays the initial state out as K-stream words and k_gs_unskew takes the last sweep's back,
// so tiles read and write nothing but words, whole lines at a time.
//
// What a solve with these two kernels measured (events around it), one sweep a wave with a barrier a
// step -> now: 256^2 40 sweeps 0.49 -> 0.140 ms, 300x251 8 sweeps 0.42 -> 0.097, 512^2 200 sweeps 1.32 ->
// 0.451, 4096^2 200 sweeps 10.5 -> 4.97 (k_gs_wave alone 0.122, 0.078, 0.437, 4.73). At 4096^2 the two
// waves of a SIMD are bound by their issue: 53 issue slots of 4 cycles a step of two sweeps, 40 of them
// vector instructions (34 the shifts and updates).
//
// Cells outside the interior or solid pass their faces through unchanged, exactly like
// the skipped cells of the serial loop. Faces no interior cell touches keep their input
// values. The result (U, V and p) goes to separate output buffers, so the early exit (stop after the
// first sweep with max|div| < 1e-5, fluid.go:175-177) is a re-run of fewer sweeps from
// the untouched input, decided on the device.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <type_traits>
#include <vector>

#include "fl_internal.h"

namespace fl {

static constexpr int LANES = 64;
// Bounded wait, in tries of a microsecond or more (several seconds); then error and continue. A wait is
// short where a tile's producers were handed out before it; with a queue to an XCD it can last as long as the
// tiles before its producer's take an XCD that other work holds all but a workgroup of (up to 0.1 s at 4096^2).
static constexpr int SPIN_LIMIT = 1 << 22;

// Tiles whose K streams stay in one XCD's L2 (queue_of_tiles).
__host__ __device__ constexpr bool near_tiles(int tk) { return tk == 16; }
static constexpr int MAXQ = 16;  // queues of tiles, one per XCD
// Blocks after which a tile's buffers begin anew (even: the waves take two blocks a turn). Beginning them anew for
// every block cost 0.5% to 1% on small grids (a step of 256^2 0.1516 -> 0.1523 ms, 300x251 0.1140 -> 0.1152).
static constexpr int SEGMENT = 1 << 16;
__host__ __device__ constexpr int segment_rows(int blk) { return SEGMENT * blk + 4 * LANES; }  // with those read ahead
// The counters of one launch (main run or re-run), zero before it.
struct GsCounters {
  int32_t ticket[MAXQ + 1];  // of each XCD's queue, and of all tiles in one
  int32_t here;              // XCDs of which a workgroup has started, a bit each
  int32_t mode;              // how the launch hands out its tiles (MODE_NEAR, MODE_FAR), 0 before it is known
};
// A solve's state on the device: the counters of its two launches; whether some simulation asks for
// the re-run; the number of the solve, from which its tags are made (kept from solve to solve).
struct GsState {
  GsCounters run[2];
  int32_t rerun, solve;
};
enum { MODE_NEAR = 1, MODE_FAR = 2 };

// One launch of the solve (main run or early-exit re-run).
struct GsRun {
  const SolveTile* tiles;  // each queue's tiles in ticket order, then all of them
  const int* first;   // [nq + 2] where each queue's tiles begin, then all tiles, and the end
  int nq;             // 0: all tiles from one queue
  int mode;           // 0, or MODE_FAR asked for by a test
  int which;          // 0 main run (K sweeps), 1 re-run (ctrl[1] sweeps of each simulation)
  int K;
  GsCounters* count;
  const int32_t* rerun;  // a batch's re-run launch only: nonzero when some simulation asked for one
  const int32_t* solve;
  const float* omega;
  float damping;
};

__device__ __forceinline__ bool tile_empty(int g, int kb, int K, int TK, int NX) {
  int k0 = kb * TK;
  if (k0 >= K) return true;
  int kmax = min(k0 + TK, K) - 1;
  int rmin = LANES * g - kmax, rmax = LANES * g + LANES - 1 - k0;
  return rmax < 0 || rmin > NX - 1;
}

// A handoff word: a left or right U face, a bottom V face and p with the solve's tag, 16 bytes.
// Each 8-byte half carries the tag's 16 bits (and half of V), so a consumer that loads the word
// while it is being written sees for each half whether it is this solve's; only the 8-byte halves
// have to arrive whole. Words are written once per solve, so the tag they hold before is that of one of the
// last solves. Device-coherent accesses (sc1), so that neither side needs a cache writeback or
// invalidate. The intrinsics' offsets are 32 bits and a tile's K rows 1 KB each, so a buffer begins
// at the rows of a stretch of SEGMENT blocks (or of a layout item), and its offsets stay within those.
typedef uint32_t word4 __attribute__((ext_vector_type(4)));
static constexpr int CACHED = 0, SC1 = 16, VOLATILE_OP = (int)0x80000000;  // cache policy of the buffer intrinsics
__device__ __forceinline__ __amdgpu_buffer_rsrc_t word_buffer(const void* p) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, 0xffffffff, 0x00027000);
}
__device__ __forceinline__ word4 ld_word(__amdgpu_buffer_rsrc_t b, uint32_t byte) {
  return __builtin_amdgcn_raw_buffer_load_b128(b, byte, 0, SC1 | VOLATILE_OP);
}
template <int POLICY>
__device__ __forceinline__ void st_word(__amdgpu_buffer_rsrc_t b, uint32_t byte, float u, float v, float p, uint32_t tag) {
  word4 w;
  w.x = __float_as_uint(u);
  w.y = (__float_as_uint(v) & 0xffffu) | (tag << 16);
  w.z = __float_as_uint(p);
  w.w = __builtin_amdgcn_alignbit(tag, __float_as_uint(v), 16);
  __builtin_amdgcn_raw_buffer_store_b128(w, b, byte, 0, POLICY);
}
// Zero in the upper 16 bits when both halves carry the tag.
__device__ __forceinline__ uint32_t word_tag(word4 w, uint32_t tag) { return (w.y ^ (tag << 16)) | (w.w ^ (tag << 16)); }
__device__ __forceinline__ float word_u(word4 w) { return __uint_as_float(w.x); }
__device__ __forceinline__ float word_v(word4 w) { return __uint_as_float(__builtin_amdgcn_perm(w.w, w.y, 0x05040100u)); }
__device__ __forceinline__ float word_p(word4 w) { return __uint_as_float(w.z); }
__device__ __forceinline__ int ld_err(const int32_t* p) {
  return __hip_atomic_load(const_cast<int32_t*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ const SimDesc& sim_desc(const OneSim& m, int) { return m.d; }
__device__ __forceinline__ const SimDesc& sim_desc(const ManySims& m, int e) { return m.sims[e]; }

// Early exit of solveSingleGrid (fluid.go:175-177): the sweeps to re-run of a main run of N, up to
// the first whose max |div| is below 1e-5, or 0 if that is the last or none. By one wave: lane l scans
// sweeps l, l+64, ...; the wave's minimum is the first such sweep.
__device__ __forceinline__ int sweeps_to_rerun(const SimDesc& D, int N) {
  int first = N;
  if (D.early_exit)
    for (int k = threadIdx.x & (LANES - 1); k < N; k += LANES)
      if (__uint_as_float(D.maxdiv[k]) < 1e-5f) {
        first = k;
        break;
      }
  for (int o = LANES / 2; o > 0; o >>= 1) first = min(first, __shfl_xor(first, o, LANES));
  return first + 1 < N ? first + 1 : 0;
}

// Lane a takes lane a-1's v; lane 0 takes its own `first`.
__device__ __forceinline__ float from_lane_below(float first, float v) {
  return __int_as_float(
      __builtin_amdgcn_update_dpp(__float_as_int(first), __float_as_int(v), 0x138, 0xF, 0xF, false));
}
// Lane a takes lane a+1's v; lane 63 takes its own `last`.
__device__ __forceinline__ float from_lane_above(float last, float v) {
  return __int_as_float(
      __builtin_amdgcn_update_dpp(__float_as_int(last), __float_as_int(v), 0x130, 0xF, 0xF, false));
}
__device__ __forceinline__ bool every_lane(bool v) { return __builtin_amdgcn_ballot_w64(!v) == 0; }
__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }
template <class T> __device__ __forceinline__ T* uniform(T* p) {
  const uint64_t v = reinterpret_cast<uint64_t>(p);
  const uint32_t lo = uniform((int)v), hi = uniform((int)(v >> 32));
  return reinterpret_cast<T*>((uint64_t)hi << 32 | lo);
}
__device__ __forceinline__ float uniform(float v) { return __int_as_float(uniform(__float_as_int(v))); }

typedef float float4_any __attribute__((ext_vector_type(4), aligned(4)));  // four floats at any word address

// S sweeps of a wave, in registers. What each sweep left at the step before: UrO the right U
// face, UlO, VbO, pO the left U face, bottom V face and p; Vt the top V face (the next column's
// bottom face); pn the p of the next column.
template <int S> struct Sweeps {
  float UrO[S], UlO[S], VbO[S], pO[S], Vt[S], pn[S], md[S], om[S];
  float rn[S];  // coarse solve: the right-hand side of the next column
};

// What a sweep solves: the pressure projection (SOLVE_GS), or the multigrid's coarse correction
// (SOLVE_COARSE, fluid.go:686-716: its cell needs p of the same five cells and the right-hand side,
// which travels where V does; its words hold p for U).
enum { SOLVE_GS, SOLVE_COARSE };

// The weights of a cell by the mask of its fluid neighbours (the index, 0 for a cell that no
// sweep updates), in LDS: what the update multiplies its faces by, 1/s, s, and a mask for div.
// An inactive cell has q = -0 and weights +0, and x + (+0 * -0) is x to the bit.
struct CellW {
  float4 w;  // -sx0, sx1, -sy0, sy1
  float4 d;  // 1/s, s, bits: all ones where updated, unused
};
__device__ __forceinline__ CellW cell_weights(int mask) {
  const float x0 = (mask & 1) ? 1.0f : 0.0f, x1 = (mask & 2) ? 1.0f : 0.0f, y0 = (mask & 4) ? 1.0f : 0.0f,
              y1 = (mask & 8) ? 1.0f : 0.0f;
  const float s = x0 + x1 + y0 + y1;
  CellW c;
  c.w = mask ? make_float4(-x0, x1, -y0, y1) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  c.d = make_float4(mask ? 1.0f / s : 1.0f, mask ? s : 1.0f, __uint_as_float(mask ? 0xffffffffu : 0u), 0.0f);
  return c;
}

// One step's cells of a wave's S sweeps: their faces, p and cells before and after the update. The
// operations are written sweep by sweep inside each line of the update, so that consecutive
// instructions are independent (a dependent one issues 8 cycles after its source, an independent
// one after 4 to 5).
template <int S> struct Cells {
  float Ul[S], Ur[S], Vb[S], Vt[S], p[S];
};
#define FL_EACH _Pragma("unroll") for (int c = 0; c < S; c++)

// The reference cell update (fluid.go:196-229) where every cell of the wave is a fluid interior
// cell with four fluid neighbours: s = 4 and all weights are 1, so (-div)/4 is the exact product
// with 0.25 and the face updates are plain adds. Damping is 1 (q * 1 is q).
template <int S>
__device__ __forceinline__ void update_plain(Cells<S>& x, float (&md)[S], const float (&om)[S], float cp) {
  float d[S], q[S], t[S];
  FL_EACH d[c] = x.Ur[c] - x.Ul[c];
  FL_EACH d[c] += x.Vt[c];
  FL_EACH d[c] -= x.Vb[c];
  FL_EACH q[c] = -d[c] * 0.25f;
  FL_EACH md[c] = fmaxf(md[c], fabsf(d[c]));
  FL_EACH q[c] *= om[c];
  FL_EACH t[c] = cp * q[c];
  FL_EACH x.Ur[c] += q[c];
  FL_EACH x.Vb[c] -= q[c];
  FL_EACH x.Vt[c] += q[c];
  FL_EACH x.Ul[c] -= q[c];
  FL_EACH x.p[c] += t[c];
}
// The update of any cell. The weights are 0 or 1, so each fma rounds once what the reference's
// multiply (exact) and add round. -div / s: the product with the rounded 1/s and one correction
// step is the correctly rounded quotient for every float and s in 1..4 (compared with the
// division over all 2^32 floats); v_div_fixup gives infinities and NaN the division's results.
// FULL: any damping, relaxation and cp (also negative or not finite): the inactive cells' faces
// are selected instead of left to the signs of their zeros.
template <int S, bool FULL>
__device__ __forceinline__ void update_any(Cells<S>& x, float (&md)[S], const float (&om)[S], float damping, float cp,
                                           const CellW (&w)[S]) {
  float d[S], q[S], e[S], t[S];
  FL_EACH d[c] = x.Ur[c] - x.Ul[c];
  FL_EACH d[c] += x.Vt[c];
  FL_EACH d[c] -= x.Vb[c];
  FL_EACH d[c] = __uint_as_float(__float_as_uint(d[c]) & __float_as_uint(w[c].d.z));
  FL_EACH q[c] = -d[c] * w[c].d.x;
  FL_EACH md[c] = fmaxf(md[c], fabsf(d[c]));
  FL_EACH e[c] = __builtin_fmaf(q[c], w[c].d.y, d[c]);
  FL_EACH q[c] = __builtin_fmaf(e[c], -w[c].d.x, q[c]);
  FL_EACH q[c] = __builtin_amdgcn_div_fixupf(q[c], w[c].d.y, -d[c]);
  FL_EACH q[c] *= om[c];
  if constexpr (FULL) {
    FL_EACH q[c] *= damping;
    FL_EACH {
      const bool on = __float_as_uint(w[c].d.z) != 0u;
      const float p = x.p[c] + cp * q[c], ul = __builtin_fmaf(w[c].w.x, q[c], x.Ul[c]),
                  ur = __builtin_fmaf(w[c].w.y, q[c], x.Ur[c]), vb = __builtin_fmaf(w[c].w.z, q[c], x.Vb[c]),
                  vt = __builtin_fmaf(w[c].w.w, q[c], x.Vt[c]);
      x.p[c] = on ? p : x.p[c];
      x.Ul[c] = on ? ul : x.Ul[c];
      x.Ur[c] = on ? ur : x.Ur[c];
      x.Vb[c] = on ? vb : x.Vb[c];
      x.Vt[c] = on ? vt : x.Vt[c];
    }
  } else {
    FL_EACH t[c] = cp * q[c];
    FL_EACH x.Ur[c] = __builtin_fmaf(w[c].w.y, q[c], x.Ur[c]);
    FL_EACH x.Vb[c] = __builtin_fmaf(w[c].w.z, q[c], x.Vb[c]);
    FL_EACH x.Vt[c] = __builtin_fmaf(w[c].w.w, q[c], x.Vt[c]);
    FL_EACH x.Ul[c] = __builtin_fmaf(w[c].w.x, q[c], x.Ul[c]);
    FL_EACH x.p[c] += t[c];
  }
}

// The masks of a block's cells of a sweep in a row, four bits each; loaded from any byte.
typedef uint32_t mask8_any __attribute__((aligned(1)));
typedef uint16_t mask4_any __attribute__((aligned(1)));

template <int S, int W, int B> struct GsShared {
  static constexpr int GP = (3 * S + 3 + 3) / 4 * 4;  // pitch of a Gi row, one float before and two after it
  float4 K[W > 1 ? W - 1 : 1][2][B][W > 1 ? LANES : 1];  // K[w - 1]: the rows (U, V, p) wave w's first sweep reads
  float Gi[W][B + 1][GP];      // boundary below lane 0: V, p of the sweep before, U of this one
  float4 tabw[16], tabd[16];   // CellW by mask
  int tile, far;
};

// The coarse update (fluid.go:699-711) of S sweeps' cells: p of the neighbours (i - 1, j), (i + 1, j),
// (i, j - 1), (i, j + 1) and of the cell, and its right-hand side. As in the updates above.
template <int S> struct CoarseCells {
  float n[S], s[S], w[S], e[S], p[S], rhs[S];
};
static constexpr float COARSE_RELAX = 1.6f;
template <int S> __device__ __forceinline__ void coarse_plain(CoarseCells<S>& x) {
  float a[S], b[S];
  FL_EACH a[c] = x.n[c] - x.p[c];
  FL_EACH b[c] = x.s[c] - x.p[c];
  FL_EACH a[c] += b[c];
  FL_EACH b[c] = x.w[c] - x.p[c];
  FL_EACH a[c] += b[c];
  FL_EACH b[c] = x.e[c] - x.p[c];
  FL_EACH a[c] += b[c];
  FL_EACH a[c] = x.rhs[c] - a[c];
  FL_EACH a[c] *= -0.25f;
  FL_EACH a[c] *= COARSE_RELAX;
  FL_EACH x.p[c] += a[c];
}
template <int S> __device__ __forceinline__ void coarse_any(CoarseCells<S>& x, const CellW (&w)[S]) {
  float a[S], b[S], q[S], e[S];
  FL_EACH a[c] = -w[c].w.x * (x.n[c] - x.p[c]);
  FL_EACH a[c] = __builtin_fmaf(w[c].w.y, x.s[c] - x.p[c], a[c]);
  FL_EACH a[c] = __builtin_fmaf(-w[c].w.z, x.w[c] - x.p[c], a[c]);
  FL_EACH a[c] = __builtin_fmaf(w[c].w.w, x.e[c] - x.p[c], a[c]);
  FL_EACH a[c] = x.rhs[c] - a[c];
  FL_EACH q[c] = -a[c] * w[c].d.x;
  FL_EACH e[c] = __builtin_fmaf(q[c], w[c].d.y, a[c]);
  FL_EACH q[c] = __builtin_fmaf(e[c], -w[c].d.x, q[c]);
  FL_EACH q[c] = __builtin_amdgcn_div_fixupf(q[c], w[c].d.y, -a[c]);
  FL_EACH q[c] *= COARSE_RELAX;
  FL_EACH b[c] = x.p[c] + q[c];
  FL_EACH x.p[c] = __float_as_uint(w[c].d.z) != 0u ? b[c] : x.p[c];
}

// How a block's cells are updated: all plain; with weights looked up once (along a wall, say: every
// lane's cells of a sweep have the same mask); or with weights looked up per cell.
enum { BLOCK_PLAIN, BLOCK_SAME, BLOCK_ANY };
// Where a wave's rows go: to the next wave's LDS rows, or to memory as handoff words, written through
// to where every XCD reads them or (OUT_CACHED) left in this XCD's L2.
enum { OUT_LDS, OUT_WORDS, OUT_CACHED };

// One block of B steps of a wave. gi, Kin: this block's boundary rows in LDS (Kin, Kout at this
// lane); k: the first step's K row; mk: the masks. A FIRST wave's rows are the words kw instead,
// row u for step u. Each step
// first takes what it needs from its neighbours (the loads of the step before have arrived),
// then stores what the step before left, loads for the next step, and updates: so no step waits
// for its own LDS traffic. The code of a block is straight, a copy for each mode and output.
// go: lane 63's U, V, p of each sweep after step u, at lane 64 - B + u: every step shifts them down
// a lane and lets lane 63 in, one instruction a value into the register that the value leaves (a
// store of lane 63 to LDS took two exec changes and two writes, 44 cycles a step for one sweep).
// ROW63: without the last sweep's V and p, which the caller takes from the LDS rows.
template <int SOLVE, int S, int B, int GP, int MODE, bool FIRST, int OUT, bool FULL, bool ROW63>
__device__ __forceinline__ void run_block(Sweeps<S>& Q, const word4 (&kw)[FIRST ? B : 1], float (&k)[3],
                                          const uint32_t (&mk)[S], const float* gi, const float4* Kin, float4* Kout,
                                          float (&go)[S][3], const char* tab, __amdgpu_buffer_rsrc_t kbuf,
                                          uint32_t kbyte, uint32_t tag, float damping, float cp) {
  constexpr int GN = (3 * S + 3) / 4 * 4;
  float g[2][GN], kr[2][3];  // the boundary and K rows of this step and the next, in turn
  CellW cw[S], cn[S];
  auto load_gi = [&](int u) {
    float(&d)[GN] = g[u % 2];
#pragma unroll
    for (int x = 0; x < 3 * S; x += 4) {
      if (x + 2 < 3 * S) {
        *reinterpret_cast<float4*>(&d[x]) = *reinterpret_cast<const float4*>(gi + u * GP + x);
      } else {
        *reinterpret_cast<float2*>(&d[x]) = *reinterpret_cast<const float2*>(gi + u * GP + x);
      }
    }
  };
  auto load_k = [&](int u) {  // what step u reads
    if constexpr (FIRST) return;
    const float4 v = Kin[(u - 1) * LANES];
    kr[u % 2][0] = v.x;
    kr[u % 2][1] = v.y;
    kr[u % 2][2] = v.z;
  };
  auto load_cw = [&](int u, CellW (&d)[S]) {
#pragma unroll
    for (int c = 0; c < S; c++) {
      const char* at = tab + ((u == 0 ? mk[c] << 4 : mk[c] >> (4 * u - 4)) & 0xF0u);
      d[c].w = *reinterpret_cast<const float4*>(at);
      d[c].d = *reinterpret_cast<const float4*>(at + 256);
    }
  };
  auto put = [&](int u) {
    const float ul = SOLVE == SOLVE_GS ? Q.UlO[S - 1] : Q.pO[S - 1];
    if constexpr (OUT == OUT_LDS)
      Kout[u * LANES] = make_float4(ul, Q.VbO[S - 1], Q.pO[S - 1], 0.0f);
    else
      st_word<OUT == OUT_CACHED ? CACHED : SC1>(kbuf, kbyte + u * (LANES * 16), ul, Q.VbO[S - 1], Q.pO[S - 1], tag);
#pragma unroll
    for (int c = 0; c < S; c++) {
      if (SOLVE == SOLVE_GS) go[c][0] = from_lane_above(Q.UrO[c], go[c][0]);
      if (ROW63 && c == S - 1) continue;
      go[c][1] = from_lane_above(Q.VbO[c], go[c][1]);
      go[c][2] = from_lane_above(Q.pO[c], go[c][2]);
    }
  };
  load_gi(0);
  load_gi(1);
  load_k(1);
  if constexpr (!FIRST) {
#pragma unroll
    for (int f = 0; f < 3; f++) kr[0][f] = k[f];
  }
#pragma unroll
  for (int c = 0; c < S; c++) go[c][0] = go[c][1] = go[c][2] = 0.0f;
  if constexpr (MODE != BLOCK_PLAIN) load_cw(0, cw);
#pragma unroll
  for (int u = 0; u < B; u++) {
    Cells<S> x;
    CoarseCells<S> y;
    float pnext[S];
    if constexpr (FIRST) {
      kr[u % 2][0] = word_u(kw[u]);
      kr[u % 2][1] = word_v(kw[u]);
      kr[u % 2][2] = word_p(kw[u]);
    }
#pragma unroll
    for (int c = 0; c < S; c++) {
      const float vnext = from_lane_below(g[u % 2][3 * c], c ? Q.VbO[c - 1] : kr[u % 2][1]);
      pnext[c] = from_lane_below(g[u % 2][3 * c + 1], c ? Q.pO[c - 1] : kr[u % 2][2]);
      if constexpr (SOLVE == SOLVE_GS) {
        x.Ul[c] = from_lane_below(g[u % 2][3 * c + 2], Q.UrO[c]);
        x.Vt[c] = vnext;
        x.Ur[c] = c ? Q.UlO[c - 1] : kr[u % 2][0];
        x.Vb[c] = Q.Vt[c];
        x.p[c] = Q.pn[c];
      } else {
        y.n[c] = from_lane_below(g[u % 2][3 * c + 2], Q.pO[c]);
        y.s[c] = c ? Q.pO[c - 1] : kr[u % 2][0];
        y.w[c] = Q.Vt[c];
        y.e[c] = pnext[c];
        y.p[c] = Q.pn[c];
        y.rhs[c] = Q.rn[c];
        Q.rn[c] = vnext;
      }
      Q.pn[c] = pnext[c];
    }
    __builtin_amdgcn_sched_barrier(0);
    if (u > 0) put(u - 1);
    if (u + 2 < B) load_gi(u + 2);
    if (u + 2 <= B) load_k(u + 2);
    if constexpr (MODE == BLOCK_ANY)
      if (u + 1 < B) load_cw(u + 1, cn);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (SOLVE == SOLVE_GS && MODE == BLOCK_PLAIN)
      update_plain<S>(x, Q.md, Q.om, cp);
    else if constexpr (SOLVE == SOLVE_GS)
      update_any<S, FULL>(x, Q.md, Q.om, damping, cp, cw);
    else if constexpr (MODE == BLOCK_PLAIN)
      coarse_plain<S>(y);
    else
      coarse_any<S>(y, cw);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < S; c++) {
      if constexpr (SOLVE == SOLVE_GS) {
        Q.UrO[c] = x.Ur[c];
        Q.Vt[c] = x.Vt[c];
        Q.UlO[c] = x.Ul[c];
        Q.VbO[c] = x.Vb[c];
        Q.pO[c] = x.p[c];
      } else {
        Q.Vt[c] = y.p[c];
        Q.VbO[c] = y.rhs[c];
        Q.pO[c] = y.p[c];
      }
    }
    if (MODE == BLOCK_ANY && u + 1 < B) {
#pragma unroll
      for (int c = 0; c < S; c++) cw[c] = cn[c];
    }
  }
  put(B - 1);
  if constexpr (!FIRST) {
#pragma unroll
    for (int f = 0; f < 3; f++) k[f] = kr[0][f];
  }
}

// The queue a workgroup takes its tiles from (called by one thread of it). A row-tile's tiles are
// all in the queue of one XCD, so that their K streams, one 1 KB row a step each, stay in that XCD's
// L2 (OUT_CACHED; written through to memory the 4096^2 solve of 200 sweeps takes 5.74 ms against 4.97,
// 2048^2 2.04 against 1.70). Only for tiles of 16 sweeps, which make more rows than XCDs: on small
// grids whole rows divide unevenly (512^2 0.530 ms against 0.475). A workgroup serves the XCD that it
// runs on. Each queue needs a workgroup, or tiles would wait for ever for those of a queue without
// one, so the first workgroups wait until one has started on every XCD (a few microseconds). If that
// fails (an XCD that is busy with something else, or kept from this stream) the launch takes all
// tiles from one queue instead and writes its K streams through. Solves on two streams at once do
// so now and then: two of 4096^2 4.7 ms a step each, of 2048^2 1.42 (with the L2 written back after
// every block instead 6.2 and 1.43, and 22 ms a step where a solve alone took that way).
static __device__ int queue_of_tiles(const GsRun& R) {
  if (R.mode == MODE_FAR) return R.nq;
  const int q = __builtin_amdgcn_s_getreg(20 | (3 << 11)) % R.nq;  // HW_REG_XCC_ID, 4 bits
  GsCounters* C = R.count;
  int seen = atomicOr(&C->here, 1 << q) | 1 << q;
  const int all = (1 << R.nq) - 1;
  int mode = 0;
  for (int it = 0; seen != all && it < 256 && !mode; it++) {
    __builtin_amdgcn_s_sleep(4);
    seen = ld_err(&C->here);
    mode = ld_err(&C->mode);
  }
  if (!mode) {
    const int want = seen == all ? MODE_NEAR : MODE_FAR, was = atomicCAS(&C->mode, 0, want);
    mode = was ? was : want;
  }
  return mode == MODE_NEAR ? q : R.nq;
}

typedef __attribute__((address_space(3))) float lds_float;  // a pointer that lanes compute stays an LDS one

// S sweeps per wave, W waves per workgroup (TK = S W sweeps per tile), B columns per block.
template <int SOLVE, int S, int W, int B, bool FULL, class M>
__global__ __launch_bounds__(W* LANES, W > 4 ? 2 : 1) void k_gs_wave(M m, GsRun R) {
  constexpr int TK = S * W, GP = GsShared<S, W, B>::GP;
  constexpr bool NEAR = near_tiles(TK);
  constexpr uint32_t BITS = B == 4 ? 0xFFFFu : 0xFFFFFFFFu;  // of a word of masks that a block uses
  constexpr uint32_t KROW = 16 * LANES, GROW = 16 * TK;      // bytes of a row of words
  static_assert(B * (S + 1) <= LANES, "a lane loads one G word per block");
  __shared__ GsShared<S, W, B> sh;
  const int lane = threadIdx.x & (LANES - 1);
  // wave-uniform, and held in a scalar register so every test on it is a scalar branch
  const int w = uniform((int)(threadIdx.x / LANES));
  // a re-run launch with nothing to re-run ends here, in every workgroup alike. A single
  // simulation's decides it here, in every wave (by a launch of its own, 4.5 us a solve).
  int again = 0;
  if constexpr (std::is_same<M, OneSim>::value) {
    if (R.which) {
      again = uniform(sweeps_to_rerun(m.d, R.K));
      if (blockIdx.x == 0 && threadIdx.x == 0) m.d.ctrl[1] = again;
      if (!again) return;
    }
  } else {
    if (R.rerun && *R.rerun == 0) return;
  }
  if (threadIdx.x < 16) {
    const CellW c = cell_weights(threadIdx.x);
    sh.tabw[threadIdx.x] = c.w;
    sh.tabd[threadIdx.x] = c.d;
  }
  const int queue = NEAR && threadIdx.x == 0 ? queue_of_tiles(R) : 0;
  const uint32_t tag0 = 2u * (uint32_t)uniform(*R.solve) & 0xffffu, tag = (tag0 + (uint32_t)R.which) & 0xffffu;
  int vzero = 0;  // a zero the compiler keeps in a vector register: LDS addresses built on it stay there too
  asm volatile("" : "+v"(vzero));
  const float* gi = &sh.Gi[w][1][0] + vzero;
  const char* tab = reinterpret_cast<const char*>(sh.tabw);

  for (;;) {
    if (threadIdx.x == 0) {
      const int t = R.first[queue] + atomicAdd(&R.count->ticket[queue], 1);
      sh.tile = t < R.first[queue + 1] ? t : -1;
      sh.far = NEAR && queue == R.nq;
    }
    __syncthreads();
    const int t = uniform(sh.tile), far = uniform(sh.far);
    __syncthreads();
    if (t < 0) break;
    const SolveTile te = R.tiles[t];
    const int sim = te.sim, g = te.g, kb = te.kb;
    const SimDesc& D = sim_desc(m, sim);
    const int NX = D.g.NX, NY = D.g.NY, rows = D.rows;
    const int nblk = rows / B;
    int32_t* err = D.ctrl + 3;
    const int K = !R.which ? R.K : std::is_same<M, OneSim>::value ? again : D.ctrl[1];
    const int Kp = (K + S - 1) / S * S;  // with the sweeps that only fill the last wave
    if (tile_empty(g, kb, Kp, TK, NX)) continue;
    const float cp = D.cp, damping = R.damping;
    const int k0 = kb * TK;
    const int i0 = LANES * g - k0;     // row of (lane 0, sweep 0)
    const int b0 = w * S;              // this wave's first sweep in the tile
    const bool wave_on = k0 + b0 < K;
    const bool words = w == W - 1 || k0 + b0 + S >= K;  // its rows go to the next sweeps' tile, or are the result
    const bool g_wave = g + 1 < D.G;                    // lane 63's faces go to the next row-tile
    // Producers: G stream (g-1,kb), K stream (g,kb-1), corner (g-1,kb-1); the first sweeps take the
    // K stream's place from the initial state's rows (k_gs_skew).
    const bool hG = g > 0 && !tile_empty(g - 1, kb, Kp, TK, NX);
    const bool hK = kb == 0 || !tile_empty(g, kb - 1, Kp, TK, NX);
    const bool hC = g > 0 && (kb == 0 || !tile_empty(g - 1, kb - 1, Kp, TK, NX));
    const size_t gtile = (size_t)rows * GROW;
    const uint32_t ktag = kb ? tag : tag0;
    const int kfirst = kb ? TK - 1 : 0, klast = kb ? rows - 1 : rows;  // row of step 0, last row

    Sweeps<S> Q;
    uint32_t mk[S], mkeep[S];
    const uint8_t* mrow[S];
    int mcol[S];
    const uint32_t mpitch = mask_pitch(NY);
#pragma unroll
    for (int c = 0; c < S; c++) {
      // read once into a scalar register: a vector-loaded value used in the step would make
      // every step wait for the wave's memory operations
      Q.om[c] = uniform(SOLVE == SOLVE_GS && k0 + b0 + c < K ? R.omega[min(k0 + b0 + c, K - 1)] : 1.0f);
      Q.rn[c] = 0.0f;
      Q.UrO[c] = Q.UlO[c] = Q.VbO[c] = Q.pO[c] = Q.Vt[c] = Q.pn[c] = Q.md[c] = 0.0f;
      mkeep[c] = k0 + b0 + c < K ? BITS : 0u;  // past the solve's last sweep the cells pass their faces on
      // rows 0 and NX - 1 are all 0; the copy in which this lane's columns start a byte (an odd
      // first column j: byte (j + 1) / 2 of the odd copy)
      mrow[c] = D.masks + (((lane + b0 + c) & 1) ? (size_t)NX * mpitch : 0) +
                (size_t)min(max(i0 + lane - b0 - c, 0), NX - 1) * mpitch + MASK_PAD / 2;
      mcol[c] = (1 - lane - b0 - c) >> 1;
    }
    const int mlast = (NY + 2) >> 1;
    float k[3] = {0.0f, 0.0f, 0.0f};

    // The G words of a block this lane loads: word (u, x) is what sweep b0 - 1 + x of the tile
    // below left at lane 63 for this wave's step u; a tile's first sweep (w = 0, x = 0) takes the
    // last sweep of the corner tile instead. need: all ones in the lanes that wait for a producer.
    const int gu = lane / (S + 1), gx = lane - gu * (S + 1);
    const bool gcorner = w == 0 && gx == 0, gstage = gu < B;
    const uint32_t gat = gcorner ? 16 * (TK - 1) : (uint32_t)gtile + 16 * (b0 - 1 + gx);  // (words_fit)
    const uint32_t goff = gat + (gcorner ? gu + LANES + kfirst : gu + LANES - 1) * GROW;
    const uint32_t gtag = gcorner ? ktag : tag, gneed = gstage && (gcorner ? hC : hG) ? ~0u : 0u, kneed = hK ? ~0u : 0u;
    lds_float* const gdst = (lds_float*)&sh.Gi[w][min(gu, B - 1) + 1][3 * gx];
    const bool gout = g_wave && lane >= LANES - B;  // stores lane 63's words of step lane - (64 - B)
    const uint32_t goword = max(lane - (LANES - B), 0) * GROW + 16 * b0;
    // Ends a wait for words that all carry this solve's tag. Bounded: after SPIN_LIMIT tries, or
    // once another wait of this simulation has expired (err set), err is set and the solve goes
    // on, so one whose producers stall ends within seconds with FL_ERR_INTERNAL.
    auto expired = [&](int it) __attribute__((always_inline)) {
      if (it > SPIN_LIMIT || ((it & 255) == 255 && ld_err(err) != 0)) {
        if (lane == 0) atomicOr(err, 1);
        return true;
      }
      __builtin_amdgcn_s_sleep(2);
      return false;
    };
    // One wave's part of the tile: FIRST, whether it is the tile's first wave and loads K words; OUT,
    // where its rows go. A copy of the code for each, so that none carries another's registers. Wave w
    // stages its first block in phase w - 1 and runs block n in phase w + n; a phase ends in a barrier.
    auto run_wave = [&](auto first_c, auto out_c) __attribute__((always_inline)) {
      constexpr bool FIRST = decltype(first_c)::value;
      constexpr int OUT = decltype(out_c)::value;
      // The words and masks of a block. The loads are issued without a condition, at addresses that
      // are always valid, so that the compiler can count them and none waits for another.
      struct Block {
        uint32_t mw[S];
        word4 gw, kw[FIRST ? B : 1];
      };
      // The buffers of a stretch of blocks that begins with block `from`. Below, n counts from there. (The
      // tile is looked up again, so that no base takes scalar registers from the blocks: they spilled, 256^2
      // 0.1516 -> 0.1535 ms. In a batch the addresses come from vector loads: uniform() spares a loop over the lanes
      // at every access, a step of 6 grids 0.329 -> 0.246 ms, of 48 2.92 -> 2.58.)
      // The G stream has a column of tiles before the first for the initial state (k_gs_skew), so the
      // corner's words lie a tile before the G stream's.
      __amdgpu_buffer_rsrc_t kmine, gmine, gprod, kprod;
      int nleft, klastn;  // blocks from there to the tile's end, last K row
      uint32_t glast;
      auto begin_at = [&](int from) __attribute__((always_inline)) {
        const SolveTile te = R.tiles[uniform(sh.tile)];
        const SimDesc& D = sim_desc(m, te.sim);
        const int KB = D.KB, g = te.g, kb = te.kb, row = from * B;
        const size_t ktile = (size_t)rows * KROW, itile = (size_t)(rows + 1) * KROW;
        const uint8_t* ksrc = kb ? D.kout + (size_t)(kb - 1) * ktile : D.kinit;  // of row-tile 0
        const size_t kstep = kb ? KB * ktile : itile;                            // to the next row-tile
        kmine = word_buffer(uniform(D.kout + (size_t)(g * KB + kb) * ktile + (size_t)row * KROW));
        gmine = word_buffer(uniform(D.gout + (size_t)(g * (KB + 1) + kb + 1) * gtile + (size_t)row * GROW));
        gprod = word_buffer(uniform(D.gout + (size_t)(max(g - 1, 0) * (KB + 1) + (g > 0 ? kb : 0)) * gtile + (size_t)row * GROW));
        kprod = word_buffer(uniform(ksrc + g * kstep + (size_t)row * KROW));
        nleft = nblk - from;
        klastn = min(klast - row, segment_rows(B));
        glast = gat + min(rows - 1 - row, segment_rows(B)) * GROW;
      };
      auto load_g = [&](Block& x, int n) __attribute__((always_inline)) {
        x.gw = ld_word(gprod, min(goff + n * (B * GROW), glast));
      };
      auto load_k = [&](Block& x, int n, int u) __attribute__((always_inline)) {
        x.kw[u] = __builtin_amdgcn_raw_buffer_load_b128(kprod, 16 * lane, min(n * B + u + kfirst, klastn) * KROW,
                                                        SC1 | VOLATILE_OP);
      };
      auto load = [&](Block& x, int n) __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < S; c++) {
          const uint8_t* at = mrow[c] + min(max(n * (B / 2) + mcol[c], -(MASK_PAD / 2)), mlast);
          if constexpr (B == 8)
            x.mw[c] = *reinterpret_cast<const mask8_any*>(at);
          else
            x.mw[c] = *reinterpret_cast<const mask4_any*>(at);
        }
        load_g(x, n);
        if constexpr (FIRST) {
#pragma unroll
          for (int u = 0; u < B; u++) load_k(x, n, u);
        }
      };
      auto stage = [&](Block& x, int n) __attribute__((always_inline)) {
        auto arrived = [&]() __attribute__((always_inline)) {
          uint32_t d = word_tag(x.gw, gtag) & gneed;
          if constexpr (FIRST) {
            uint32_t e = 0;
#pragma unroll
            for (int u = 0; u < B; u++) e |= word_tag(x.kw[u], ktag);
            d |= e & kneed;
          }
          return every_lane(d < 0x10000u);
        };
        // The first check stands before the loop: at the loop's head it would have to wait for every
        // store issued since. A wait polls with the G words and the block's last K row only: 256 CUs
        // that reload whole blocks would take the bandwidth their producers need.
        if (!arrived()) {
          for (int it = 0; !expired(it); it++) {
            load_g(x, n);
            if constexpr (FIRST) {
              load_k(x, n, B - 1);
              if (every_lane(word_tag(x.kw[B - 1], ktag) < 0x10000u)) {
#pragma unroll
                for (int u = 0; u < B - 1; u++) load_k(x, n, u);
              }
            }
            if (arrived()) break;
          }
        }
        // (a producer that does not exist leaves arbitrary values to lane 0, or to lanes off the
        // grid, whose cells lie outside the interior in every sweep)
        if (gstage) {
          gdst[-1] = word_u(x.gw);
          gdst[0] = word_v(x.gw);
          gdst[1] = word_p(x.gw);
        }
#pragma unroll
        for (int c = 0; c < S; c++) {
          mk[c] = x.mw[c] & mkeep[c];
          asm volatile("" : "+v"(mk[c]));  // now: the scheduler would wait for the masks after the next stores
        }
      };
      float go[S][3];
      // The last sweep's V and p of lane 63 are in the rows that the wave left in LDS: the last B lanes
      // read them there after the block, two shifts a step less (256^2 the kernel 123 -> 120 us, 512^2 200
      // sweeps 444 -> 436, 2048x1024 861 -> 842). Not in tiles of 16 sweeps, which lose (4096^2 4.74 ->
      // 4.79 ms).
      constexpr bool ROW63 = OUT == OUT_LDS && !NEAR;
      const float4* krow63[2] = {};
      if constexpr (ROW63) {
        krow63[0] = &sh.K[w][0][max(lane - (LANES - B), 0)][LANES - 1];
        krow63[1] = &sh.K[w][1][max(lane - (LANES - B), 0)][LANES - 1];
      }
      auto run = [&](const Block& x, int n) __attribute__((always_inline)) {
        const float4* Kin = FIRST ? nullptr : &sh.K[w - 1][n & 1][0][lane];
        float4* Kout = OUT != OUT_LDS ? nullptr : &sh.K[w][n & 1][0][lane];
        const uint32_t kbyte = (uint32_t)n * (B * KROW) + 16 * lane;
        bool plain = true, same = true;
#pragma unroll
        for (int c = 0; c < S; c++) {
          plain = plain && mk[c] == BITS;
          same = same && mk[c] == (mk[c] & 0xFu) * (BITS / 0xFu);
        }
#define FL_RUN(MODE) \
  run_block<SOLVE, S, B, GP, MODE, FIRST, OUT, FULL, ROW63>(Q, x.kw, k, mk, gi, Kin, Kout, go, tab, kmine, kbyte, tag, damping, cp)
        if (!FULL && every_lane(plain)) {
          FL_RUN(BLOCK_PLAIN);
        } else if (every_lane(same)) {
          FL_RUN(BLOCK_SAME);
        } else {
          FL_RUN(BLOCK_ANY);
        }
#undef FL_RUN
        if constexpr (ROW63) {
          const float4 v = *krow63[n & 1];
          go[S - 1][1] = v.y;
          go[S - 1][2] = v.z;
        }
      };
      for (int p = 0; p < w; p++) __syncthreads();
      // Block n runs while the words of block n + 1 are on their way (the last block's once more
      // after the end). They are waited for before the stores of lane 63's words are issued: vector
      // memory operations complete in order, and a wait behind a store would last as long as the
      // store's way to memory.
      auto phase = [&](const Block& x, Block& next, int n) __attribute__((always_inline)) {
        const int n1 = min(n + 1, nleft - 1);
        load(next, n1);
        run(x, n);
        stage(next, n1);
        if (gout) {
#pragma unroll
          for (int c = 0; c < S; c++)
            st_word<SC1>(gmine, goword + n * (B * GROW) + 16 * c, go[c][SOLVE == SOLVE_GS ? 0 : 2], go[c][1], go[c][2], tag);
        }
        __syncthreads();
      };
      Block x, y;
      begin_at(0);
      load(x, 0);
      stage(x, 0);
      __syncthreads();
      for (int from = 0;;) {
        const int end = min(nleft, SEGMENT);
        if constexpr (FIRST) {  // two blocks to a turn, so that their words stay where they were loaded
          for (int n = 0;;) {
            phase(x, y, n);
            if (++n == end) break;
            phase(y, x, n);
            if (++n == end) break;
          }
        } else {
          for (int n = 0; n < end; n++) phase(x, x, n);
        }
        if ((from += SEGMENT) >= nblk) break;
        begin_at(from);
#pragma unroll
        for (int c = 0; c < S; c++) mcol[c] += SEGMENT * B / 2;
      }
      for (int p = w + 1; p < W; p++) __syncthreads();
    };
    using first_t = std::true_type;
    using later_t = std::false_type;
    using lds_t = std::integral_constant<int, OUT_LDS>;
    using words_t = std::integral_constant<int, OUT_WORDS>;
    using cached_t = std::integral_constant<int, OUT_CACHED>;
    auto run_words = [&](auto first_c) __attribute__((always_inline)) {
      if constexpr (NEAR) {
        if (!far) return run_wave(first_c, cached_t{});
      }
      run_wave(first_c, words_t{});
    };
    if (!wave_on) {
      for (int p = 0; p < nblk + W; p++) __syncthreads();
    } else if (w == 0) {
      if (words)
        run_words(first_t{});
      else if constexpr (W > 1)
        run_wave(first_t{}, lds_t{});
    } else if constexpr (W > 1) {
      if (words)
        run_words(later_t{});
      else
        run_wave(later_t{}, lds_t{});
    }
    if (SOLVE != SOLVE_GS) continue;
    // per-sweep max |div|
#pragma unroll
    for (int c = 0; c < S; c++) {
      float mv = Q.md[c];
      for (int o = 32; o > 0; o >>= 1) mv = fmaxf(mv, __shfl_xor(mv, o, 64));
      if (lane == 0 && k0 + b0 + c < K && mv > 0.0f)
        atomicMax(&D.maxdiv[R.which * D.nmax + k0 + b0 + c], __float_as_uint(mv));
    }
  }
}

// The initial state in the solve's layout, and the result out of it. An item is 64 rows of words of
// one row-tile; each of a workgroup's SKEW_WAVES waves moves SKEW_ROWS of the tile's 64 grid rows, 64
// columns each, through LDS, so that both sides read and write whole lines. Bound by the latency of
// its loads on small grids (30 items at 256^2) and by memory on large ones, so a wave has all of its
// loads in flight at once: with 4, 8 and 16 waves k_gs_skew took 13.4, 8.4 and 6.3 us at 256^2, 277,
// 199 and 166 us on an ensemble of 18.6 M cells, 165, 114 and 100 us (4.7 TB/s) at 4096^2; k_gs_unskew
// 8.4, 6.4 and 5.2 us, 168, 135 and 133 us, 103 us.
static constexpr int SKEW_WAVES = 16, SKEW_ROWS = LANES / SKEW_WAVES;
__device__ __forceinline__ void skew_item(const OneSim& m, const SkewItem*, int item, const SimDesc*& D, int& g, int& t0) {
  D = &m.d;
  const int nt = (D->rows + 1 + LANES - 1) / LANES;
  g = item / nt;
  t0 = (item % nt) * LANES;
}
__device__ __forceinline__ void skew_item(const ManySims& m, const SkewItem* items, int item, const SimDesc*& D, int& g,
                                          int& t0) {
  const SkewItem it = items[item];
  D = &m.sims[it.sim];
  g = it.g;
  t0 = it.t0;
}

// Faces and cells no interior cell touches keep their input values: U with i = 0 or
// j in {0, NY-1}; V with i in {0, NX-1} or j = 0; p on the ring. All lie on the ring.
__device__ __forceinline__ void ring_copy(const SimDesc& D, int i, int j, int rPin, int rPout) {
  const int NX = D.g.NX, NY = D.g.NY;
  const size_t c = (size_t)i * NY + j;
  if (!(i >= 1 && j >= 1 && j <= NY - 2)) D.buf[B_U2][c] = D.buf[B_U][c];
  if (!(i >= 1 && i <= NX - 2 && j >= 1)) D.buf[B_V2][c] = D.buf[B_V][c];
  D.buf[rPout][c] = rPin >= 0 ? D.buf[rPin][c] : 0.0f;
}
// Ring item `item` of 256 cells of each side, by thread t of 256.
__device__ __forceinline__ void ring_desc(const OneSim& m, int item, const SimDesc*& D, int& t) {
  D = &m.d;
  t += item * 256;
}
__device__ __forceinline__ void ring_desc(const ManySims& m, int item, const SimDesc*& D, int& t) {
  const RingItem it = m.rings[item];
  D = &m.sims[it.sim];
  t += it.blk * 256;
}
// What precedes a solve besides its layout: the ring, and the per-sweep maxima and re-run sweeps of
// every simulation set to zero. It only has to come before the solve, so it takes the first
// workgroups of the layout's launch (a launch of its own took 4.7 us, two in a batch).
struct GsPrep {
  int groups, rings;  // workgroups, ring items
  int rPout;
  uint32_t* maxdiv;
  int nmd;
  int32_t* ctrl;
  int nsim;
};
static constexpr int RINGS_PER_GROUP = SKEW_WAVES * LANES / 256;
static int prep_groups(int rings) { return (rings + RINGS_PER_GROUP - 1) / RINGS_PER_GROUP; }
template <class M> __device__ __forceinline__ void prepare_solve(const M& m, const GsPrep& P, int rPin) {
  const int item = blockIdx.x * RINGS_PER_GROUP + threadIdx.x / 256;
  if (item < P.rings) {
    const SimDesc* D;
    int t = threadIdx.x % 256;
    ring_desc(m, item, D, t);
    const int NX = D->g.NX, NY = D->g.NY;
    if (t < NX) {
      ring_copy(*D, t, 0, rPin, P.rPout);
      ring_copy(*D, t, NY - 1, rPin, P.rPout);
    }
    if (t < NY) {
      ring_copy(*D, 0, t, rPin, P.rPout);
      ring_copy(*D, NX - 1, t, rPin, P.rPout);
    }
  }
  const int t0 = blockIdx.x * blockDim.x + threadIdx.x, stride = P.groups * blockDim.x;
  for (int t = t0; t < P.nmd; t += stride) P.maxdiv[t] = 0u;
  for (int t = t0; t < P.nsim; t += stride) P.ctrl[4 * t] = P.ctrl[4 * t + 1] = 0;
}

// Row t (stored at t + 1) of row-tile g holds, at lane a, U, V and p of cell (64 g + a + 1, t - a + 1):
// what lane a of a sweep before the first would have left at step t.
template <class M>
__global__ __launch_bounds__(SKEW_WAVES * LANES) void k_gs_skew(M m, const SkewItem* items, const int32_t* solve, int tk, int rPin,
                                                                 GsPrep P) {
  __shared__ float sh[3][LANES][LANES + 1];
  if (blockIdx.x < (unsigned)P.groups) return prepare_solve(m, P, rPin);
  const SimDesc* D;
  int g, t0;
  skew_item(m, items, blockIdx.x - P.groups, D, g, t0);
  const int lane = threadIdx.x & 63, w = threadIdx.x / 64, NX = D->g.NX, NY = D->g.NY;
  const float* src[3] = {D->buf[B_U],  // (a coarse solve has none)
                         D->buf[B_V], rPin >= 0 ? D->buf[rPin] : nullptr};
#pragma unroll
  for (int x = 0; x < SKEW_ROWS; x++) {
    const int a = SKEW_ROWS * w + x, r = LANES * g + a + 1, j = t0 - a + lane;
    const bool in = r < NX && j >= 0 && j < NY;
#pragma unroll
    for (int f = 0; f < 3; f++) sh[f][a][lane] = in && src[f] ? src[f][(size_t)r * NY + j] : 0.0f;
  }
  __syncthreads();
  const uint32_t tag = 2u * (uint32_t)*solve & 0xffffu;
  const __amdgpu_buffer_rsrc_t dst = word_buffer(D->kinit + ((size_t)g * (D->rows + 1) + t0) * (16 * LANES));
  // lane 63's also as the last sweep's of the G stream's first column
  const __amdgpu_buffer_rsrc_t gdst = word_buffer(D->gout + ((size_t)g * (D->KB + 1) * D->rows + t0) * (16 * tk));
#pragma unroll
  for (int x = 0; x < SKEW_ROWS; x++) {
    const int u = SKEW_ROWS * w + x;
    if (t0 + u <= D->rows)
      st_word<CACHED>(dst, (uint32_t)u * (16 * LANES) + 16 * lane, sh[0][lane][u], sh[1][lane][u], sh[2][lane][u], tag);
    if (lane == LANES - 1 && t0 + u < D->rows)
      st_word<CACHED>(gdst, (uint32_t)u * (16 * tk) + 16 * (tk - 1), sh[0][lane][u], sh[1][lane][u], sh[2][lane][u], tag);
  }
}

// The number of the next solve and its counters (one workgroup of the solve's last kernel).
__device__ __forceinline__ void next_solve(GsState* S) {
  int32_t* c = reinterpret_cast<int32_t*>(S->run);
  for (int t = threadIdx.x; t < (int)(sizeof(S->run) / sizeof(int32_t)); t += blockDim.x) c[t] = 0;
  if (threadIdx.x == 0) {
    S->rerun = 0;
    ++S->solve;
  }
}

// The rows of the last sweep's wave (its last sweep b, padded to the wave's S) to U2, V2 and role
// rPout: row t of row-tile g holds cell (64 g + a - k0 - b, t - a - b) at lane a. An early exit
// (ctrl[1] sweeps) takes the re-run's. A coarse solve has p alone. turb: the turbulence that follows
// the solve (strength times dt; 0: none). Also numbers the next solve and zeroes its counters.
template <class M>
__global__ __launch_bounds__(SKEW_WAVES * LANES) void k_gs_unskew(M m, const SkewItem* items, GsState* state, int N, int tk, int S,
                                                   int rPout, bool coarse, float turb) {
  __shared__ float sh[3][LANES][LANES + 1];
  const SimDesc* D;
  int g, t0;
  skew_item(m, items, blockIdx.x, D, g, t0);
  if (blockIdx.x == 0) next_solve(state);
  const int lane = threadIdx.x & 63, w = threadIdx.x / 64, NX = D->g.NX, NY = D->g.NY, rows = D->rows;
  const int kept = D->early_exit ? D->ctrl[1] : 0, K = kept > 0 ? kept : N;
  const int kb = (K - 1) / tk, k0 = kb * tk, b = (K - 1 - k0) / S * S + S - 1;
  const int r0 = LANES * g - k0 - b;  // row of lane 0
  if (r0 > NX - 1 || r0 + LANES - 1 < 1) return;
  const int first = min(t0, rows - 1);  // (the item past the last row of words has no cells)
  const __amdgpu_buffer_rsrc_t src = word_buffer(D->kout + ((size_t)(g * D->KB + kb) * rows + first) * (16 * LANES));
#pragma unroll
  for (int x = 0; x < SKEW_ROWS; x++) {
    const int u = SKEW_ROWS * w + x;
    const word4 v = ld_word(src, (uint32_t)min(u, rows - 1 - first) * (16 * LANES) + 16 * lane);
    sh[0][lane][u] = word_u(v);
    sh[1][lane][u] = word_v(v);
    sh[2][lane][u] = word_p(v);
  }
  uint32_t fluid[SKEW_ROWS] = {};  // the cells that take turbulence, loaded with the words
#pragma unroll
  for (int x = 0; x < SKEW_ROWS; x++) {
    const int r = r0 + SKEW_ROWS * w + x, j = t0 + lane - SKEW_ROWS * w - x - b;
    if (turb != 0.0f && r >= 1 && r <= NX - 2 && j >= 1 && j <= NY - 2) fluid[x] = D->flags[(size_t)r * NY + j] & CF_FLUID;
  }
  __syncthreads();
  float* const dst[3] = {D->buf[B_U2], D->buf[B_V2], D->buf[rPout]};
#pragma unroll
  for (int x = 0; x < SKEW_ROWS; x++) {
    const int a = SKEW_ROWS * w + x, r = r0 + a, j = t0 + lane - a - b;
    if (r < 1 || r > NX - 1 || j < 1 || j > NY - 1 || t0 + lane >= rows) continue;
    const size_t c = (size_t)r * NY + j;
    float u = sh[0][a][lane], v = sh[1][a][lane];
    if (fluid[x]) add_turbulence(u, v, r, j, turb);
    if (!coarse && j <= NY - 2) dst[0][c] = u;
    if (!coarse && r <= NX - 2) dst[1][c] = v;
    if (r <= NX - 2 && j <= NY - 2) dst[2][c] = sh[2][a][lane];
  }
}

// Every member's early exit, one wave each: the sweeps to re-run to ctrl[1], and whether the re-run
// launch has any. (A single simulation's re-run launch decides for itself.)
__global__ void k_gs_decide(ManySims m, int nsim, int N, int32_t* rerun) {
  const int e = blockIdx.x * (blockDim.x / LANES) + threadIdx.x / LANES;
  if (e >= nsim) return;
  const SimDesc& D = m.sims[e];
  const int again = sweeps_to_rerun(D, N);
  if ((threadIdx.x & (LANES - 1)) == 0) {
    D.ctrl[1] = again;
    if (again) atomicOr(rerun, 1);
  }
}

static bool tile_empty_h(int g, int kb, int K, int TK, int NX) {
  int k0 = kb * TK;
  if (k0 >= K) return true;
  int kmax = std::min(k0 + TK, K) - 1;
  int rmin = LANES * g - kmax, rmax = LANES * g + LANES - 1 - k0;
  return rmax < 0 || rmin > NX - 1;
}

// Waves per workgroup of a tile of tk sweeps: two sweeps to a wave; one in the small tiles, whose
// few waves leave the CU's issue slots free (measured before the layout kernels were shortened: 4
// sweeps, 256^2 jet 0.154 ms a solve against 0.175 with two waves of two; 300x251 0.110 against
// 0.136). Four to a wave lost everywhere (2048^2 2.35 ms against 1.72 at 16 sweeps, 2048x1024 1.55
// against 1.09 at 8).
static int tile_waves(int tk) { return tk <= 4 ? tk : tk / 2; }
static int tile_sweeps(int tk) { return tk / tile_waves(tk); }  // sweeps per wave
// N sweeps with those that only fill the last wave: their cells pass their faces on.
static int padded(int N, int tk) {
  const int s = tile_sweeps(tk);
  return (N + s - 1) / s * s;
}

// Tile geometry of one simulation for N sweeps with tk sweeps per tile and blk columns per
// block.
struct TileGeom {
  int G, KB, rows;
};
static TileGeom geom(int NX, int NY, int N, int tk, int blk) {
  TileGeom t;
  t.G = (NX + padded(N, tk) - 1 + LANES - 1) / LANES;
  t.KB = (N + tk - 1) / tk;
  const int steps = NY + LANES - 1 + tk - 1;
  t.rows = (steps + blk - 1) / blk * blk;
  return t;
}
// A wave loads its G words from its producer's tile and the corner tile before it in one instruction,
// so their offsets span one tile of `rows` rows and a stretch of SEGMENT blocks, and have to stay
// below 2^32. With one row-tile the words are not used.
static bool words_fit(const TileGeom& t, int tk, int blk) {
  return t.G == 1 || ((uint64_t)t.rows + segment_rows(blk)) * (16 * tk) < (uint64_t)1 << 32;
}
// The depth to use where tiles of tk sweeps are too long for that (16.2 million columns with 16):
// shallower ones, whose G rows are smaller.
static int shallow_enough(int NX, int NY, int N, int tk, int blk) {
  while (tk > 2 && !words_fit(geom(NX, NY, N, tk, blk), tk, blk)) tk /= 2;
  return tk;
}
// Tiles are handed out in the order their producers let them start: a consumer loads a block
// ahead, so it runs 64 + 2 BLK columns behind the tile one row-tile up, and TK + 2 BLK plus the
// (W - 1) blocks between the first and the last wave behind the tile one sweep block back; the
// key is that estimate of its start. Producers always get smaller keys (a topological order, which
// the persistent kernel needs: a workgroup never waits on a tile no workgroup has taken).
struct GsTile {
  long long key;
  int row;  // of all simulations' row-tiles
  SolveTile t;
};
static void append_tiles(std::vector<GsTile>& out, int sim, int row0, int NX, int N, int tk, int blk, const TileGeom& t) {
  for (int g = 0; g < t.G; g++)
    for (int kb = 0; kb < t.KB; kb++)
      if (!tile_empty_h(g, kb, padded(N, tk), tk, NX)) {
        const long long start = (long long)(LANES + 2 * blk) * g + (long long)(tk + (tile_waves(tk) + 1) * blk) * kb;
        out.push_back({(start << 32) | ((long long)sim << 12) | kb, row0 + g, SolveTile{sim, g, kb, 0}});
      }
}
// The tiles of nq queues, each in ticket order, then all in ticket order; first[q]: where they begin.
// Row-tiles go to the queue that has the fewest steps so far, in the order of their first tiles.
// Returns the tiles of the longest queue.
static int queue_tiles(std::vector<GsTile>& tiles, const std::vector<int>& row_steps, int nq, std::vector<SolveTile>& out,
                       std::vector<int>& first) {
  std::sort(tiles.begin(), tiles.end(), [](const GsTile& a, const GsTile& b) { return a.key < b.key; });
  std::vector<long long> load(row_steps.size(), 0), total(nq, 0);
  std::vector<int> queue(row_steps.size(), -1);
  for (const GsTile& t : tiles) load[t.row] += row_steps[t.row];
  std::vector<std::vector<SolveTile>> lists(nq);
  for (const GsTile& t : tiles) {
    int& q = queue[t.row];
    if (q < 0 && nq > 0) {
      q = (int)(std::min_element(total.begin(), total.end()) - total.begin());
      total[q] += load[t.row];
    }
    if (nq > 0) lists[q].push_back(t.t);
  }
  size_t longest = 0;
  for (auto& l : lists) {
    first.push_back((int)out.size());
    out.insert(out.end(), l.begin(), l.end());
    longest = std::max(longest, l.size());
  }
  first.push_back((int)out.size());
  for (const GsTile& t : tiles) out.push_back(t.t);
  first.push_back((int)out.size());
  return (int)longest;
}
// One queue per XCD of 32 CUs.
static int device_queues(int dev, int tk) {
  int cus = 0;
  if (!near_tiles(tk)) return 0;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) cus = 256;
  return std::min(MAXQ, std::max(1, cus / 32));
}

// Tiles of tk sweeps that a solve has in flight at once: the row-tiles that start (80 steps one
// after the other) before the first ends, by the blocks of sweeps.
static long long tiles_in_flight(int NX, int NY, int N, int tk) {
  const long long rows = std::min((NX + N - 1 + LANES - 1) / LANES, (NY + LANES + 79) / 80);
  return rows * ((N + tk - 1) / tk);
}
// Sweeps per tile for the number of tiles in flight by their depth: the smallest tile of which
// there is no more than one per CU. Small tiles spread a small grid over the CUs and
// step faster; once there are more of them than CUs, large ones hand over less and take fewer
// turns. Solve times in ms with 4, 8, 16 sweeps: 300x251 8 sweeps 0.097 0.127 0.132; 256^2 40 sweeps
// 0.140 0.158 0.207; 777x391 33 sweeps 0.224 0.285 0.389; 1024^2 40 sweeps (140 in flight with 4)
// 0.363 0.444 0.615; 1024^2 100 sweeps (350 with 4, 182 with 8) 0.618 0.599 0.717; 512^2 200 sweeps
// (400, 200) 0.474 0.451 0.598; 2048x1024 100 sweeps (350, 182) 1.010 0.945 1.033; 4096^2 40 sweeps
// (265 with 8) 3.20 2.77 2.43; 2048^2 200 sweeps (675) 2.79 2.05 1.68; 4096^2 200 sweeps 10.2 6.5 5.0.
// Two sweeps (the knob takes them) gain at most 0.004 ms on 4 and lose from 1024^2 on: 300x251 0.093, 256^2
// 0.142, 777x391 0.218, 1024^2 40 sweeps 0.432.
template <class F> static int depth_for(F in_flight) { return in_flight(4) <= 256 ? 4 : in_flight(8) <= 256 ? 8 : 16; }
static bool tk_knob(const fl_params& P) {
  return P.block_sweeps == 2 || P.block_sweeps == 4 || P.block_sweeps == 8 || P.block_sweeps == 16;
}
int pick_tk(const fl_params& P, int NX, int NY, int N) {
  const int tk = tk_knob(P) ? P.block_sweeps : depth_for([&](int tk) { return tiles_in_flight(NX, NY, N, tk); });
  return shallow_enough(NX, NY, N, tk, pick_blk(P));
}
// Columns per block: 4 with the knob, else 8, which won at every size (4096^2 200 sweeps 5.0 ms
// against 7.0, 256^2 0.140 against 0.151). 16, which the knob also takes, would not fit in LDS.
int pick_blk(const fl_params& P) { return P.block_cols == 4 ? 4 : 8; }
// The update that leaves inactive cells alone by the signs of zeros needs these; any other
// parameters take the FULL kernels.
static bool regular(const fl_params& P, float cp) {
  return P.pressure_damping == 1.0f && cp > 0.0f && std::isfinite(cp) && P.relaxation > 0.0f &&
         std::isfinite(P.relaxation);
}

// The kernel of one tile shape and launch map, and its persistent grid for `ntiles` tiles: as
// many workgroups as fit on the device at once (and no more than there are tiles).
template <class M> struct GsKernels {
  using Fn = void (*)(M, GsRun);
  static Fn get(int tk, int blk, bool full) {
#define FL_GS_CASE(S, W, B) \
  if (tk == S * W && blk == B) return full ? k_gs_wave<SOLVE_GS, S, W, B, true, M> : k_gs_wave<SOLVE_GS, S, W, B, false, M>;
    FL_GS_CASE(1, 2, 4) FL_GS_CASE(1, 2, 8)
    FL_GS_CASE(1, 4, 4) FL_GS_CASE(1, 4, 8)
    FL_GS_CASE(2, 4, 4) FL_GS_CASE(2, 4, 8)
    FL_GS_CASE(2, 8, 4) FL_GS_CASE(2, 8, 8)
#undef FL_GS_CASE
    return nullptr;
  }
};
template <class M> static int occupancy_grid(int dev, int tk, int blk, int ntiles) {  // ntiles: as if all queues were the longest
  int per_cu = 0;
  hipDeviceProp_t prop;
  if (hipGetDeviceProperties(&prop, dev) != hipSuccess) return 1;
  (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, GsKernels<M>::get(tk, blk, false), tile_waves(tk) * LANES, 0);
  return std::max(1, std::min(ntiles, std::max(1, per_cu) * prop.multiProcessorCount));
}
template <class M>
static int launch_gs(int tk, int blk, int grid, hipStream_t stream, const M& m, const GsRun& R, bool full) {
  auto fn = GsKernels<M>::get(tk, blk, full);
  if (!fn) {
    set_error("no Gauss-Seidel kernel for " + std::to_string(tk) + " sweeps x " + std::to_string(blk) + " columns");
    return FL_ERR_INTERNAL;
  }
  hipLaunchKernelGGL(fn, dim3(grid), dim3(tile_waves(tk) * LANES), 0, stream, m, R);
  FL_HIP(hipGetLastError());
  return FL_OK;
}

static void free_work(GsWork& W) {
  for (void* p : {(void*)W.d_tile, (void*)W.d_first, (void*)W.d_state, (void*)W.d_kout, (void*)W.d_gout, (void*)W.d_kinit})
    if (p) (void)hipFree(p);
  (void)hipGetLastError();  // of a failed allocation: the next launch's check is not to report it
  W = GsWork{};
}
static int plan(GsWork& W, Ctx* c, int NX, int NY, int N, int tk, int blk) {
  const TileGeom t = geom(NX, NY, N, tk, blk);
  W.tk = tk;
  W.blk = blk;
  W.G = t.G;
  W.KB = t.KB;
  W.rows = t.rows;
  std::vector<GsTile> order;
  append_tiles(order, 0, 0, NX, N, tk, blk, t);
  std::vector<SolveTile> tiles;
  std::vector<int> first;
  W.nq = device_queues(c->dev, tk);
  const int longest = queue_tiles(order, std::vector<int>(t.G, t.rows), W.nq, tiles, first);
  W.ntiles = (int)order.size();
  const size_t nt = (size_t)W.G * W.KB;
  const size_t kbytes = 16 * nt * W.rows * LANES, gbytes = 16 * (nt + W.G) * W.rows * tk;
  FL_HIP(hipMalloc(&W.d_tile, sizeof(SolveTile) * std::max<size_t>(1, tiles.size())));
  FL_HIP(hipMalloc(&W.d_first, sizeof(int) * first.size()));
  FL_HIP(hipMalloc(&W.d_kout, kbytes));
  FL_HIP(hipMalloc(&W.d_gout, gbytes));
  FL_HIP(hipMalloc(&W.d_kinit, (size_t)16 * W.G * (W.rows + 1) * LANES));
  FL_HIP(hipMalloc(&W.d_state, sizeof(GsState)));
  // no word may carry a tag before a solve writes it: the words start at tag 0, the solves at 1
  FL_HIP(hipMemsetAsync(W.d_kout, 0, kbytes, c->stream));
  FL_HIP(hipMemsetAsync(W.d_gout, 0, gbytes, c->stream));
  GsState state{};
  state.solve = 1;
  FL_HIP(hipMemcpy(W.d_state, &state, sizeof(state), hipMemcpyHostToDevice));
  FL_HIP(hipMemcpy(W.d_tile, tiles.data(), sizeof(SolveTile) * tiles.size(), hipMemcpyHostToDevice));
  FL_HIP(hipMemcpy(W.d_first, first.data(), sizeof(int) * first.size(), hipMemcpyHostToDevice));
  W.grid = occupancy_grid<OneSim>(c->dev, tk, blk, std::max(W.ntiles, W.nq * longest));
  return FL_OK;
}
// The layout for N sweeps in tiles of tk, or of up to `deepest` if the words of those do not fit the
// device: deeper tiles hand over less (a column of 40 sweeps takes 12 KB a row-tile in tiles of 4, 7 of
// 8, 5 of 16).
static int layout(GsWork& W, Ctx* c, int NX, int NY, int N, int tk, int deepest, int blk) {
  if (W.n_alloc == N && W.asked == tk && W.blk == blk) return FL_OK;
  FL_HIP(hipStreamSynchronize(c->stream));  // earlier solves may still use the old layout
  int rc = FL_OK;
  for (int t = tk; t == tk || (t <= deepest && words_fit(geom(NX, NY, N, t, blk), t, blk)); t *= 2) {
    free_work(W);
    if ((rc = plan(W, c, NX, NY, N, t, blk)) == FL_OK) {
      W.n_alloc = N;
      W.asked = tk;
      return FL_OK;
    }
  }
  free_work(W);  // a layout is whole or none: the next solve plans again
  return rc;
}

bool gs_wave_supported(Ctx* c, int numIters) { return numIters >= 1 && c->NX >= 3 && c->NY >= 3; }

static int enqueue_solve(Ctx* c, int N, float cp) {
  GsWork& W = c->gs;
  int rc = layout(W, c, c->NX, c->NY, N, pick_tk(c->prm, c->NX, c->NY, N), tk_knob(c->prm) ? 0 : 16, pick_blk(c->prm));
  if (rc) return rc;
  if (c->flags_dirty && (rc = launch_flags(c))) return rc;
  SimDesc d = c->desc();
  d.cp = cp;
  OneSim m{d};
  const int mr = std::max(c->NX, c->NY);
  // Simulate's fill(p, 0) left to this solve: the initial p is zero and is not read
  const int rPin = c->gs_p_zero ? -1 : (int)B_P;
  c->gs_p_zero = false;
  const int nskew = W.G * ((W.rows + 1 + LANES - 1) / LANES);
  const int rings = (mr + 255) / 256;
  const GsPrep P{prep_groups(rings), rings, (int)B_T3, c->d_maxdiv, 2 * c->nmax, c->d_ctrl, 1};
  hipLaunchKernelGGL(k_gs_skew<OneSim>, dim3(P.groups + nskew), dim3(SKEW_WAVES * LANES), 0, c->stream, m, nullptr,
                     &W.d_state->solve, W.tk, rPin, P);
  FL_HIP(hipGetLastError());
  GsRun R{};
  R.tiles = W.d_tile;
  R.first = W.d_first;
  R.nq = W.nq;
  R.mode = c->gs_far ? MODE_FAR : 0;
  R.K = N;
  R.solve = &W.d_state->solve;
  R.omega = c->d_omega;
  R.damping = c->prm.pressure_damping;
  W.lag = c->prm.handoff_lag >= 1 && c->prm.handoff_lag <= 3 ? c->prm.handoff_lag : 1;
  const bool full = !regular(c->prm, cp);
  // without the early exit no re-run can be requested: it is skipped
  const int runs = c->prm.early_exit ? 2 : 1;
  for (int which = 0; which < runs; which++) {
    R.which = which;
    R.count = &W.d_state->run[which];
    if ((rc = launch_gs(W.tk, W.blk, W.grid, c->stream, m, R, full))) return rc;
  }
  hipLaunchKernelGGL(k_gs_unskew<OneSim>, dim3(nskew), dim3(SKEW_WAVES * LANES), 0, c->stream, m, nullptr, W.d_state, N, W.tk,
                     tile_sweeps(W.tk), (int)B_T3, false, c->gs_turb);
  FL_HIP(hipGetLastError());
  std::swap(c->U, c->U2);
  std::swap(c->V, c->V2);
  std::swap(c->p, c->T3);
  c->host_sweeps = -1;
  return FL_OK;
}
// A solve's last kernel resets the counters for the next, so one that was not enqueued whole leaves
// a layout that must not be used again.
int gs_wave_solve(Ctx* c, int N, float cp) {
  const int rc = enqueue_solve(c, N, cp);
  if (rc) c->gs.n_alloc = -1;
  return rc;
}

int pressure_free(Ctx* c) {
  free_work(c->gs);
  free_work(c->mg_gs);
  return FL_OK;
}

// solveCoarseGrid's sweeps (fluid.go:686-716) from p = 0 by the same tiles. It
// replaces one launch per diagonal of 32 x 64 tiles and sweep, 89 launches of 24 us at 257^2:
// 2.16 ms -> 0.16.
static int enqueue_coarse_solve(Ctx* c, int cNX, int cNY, int N, const float* rhs, float* p, uint8_t* masks) {
  GsWork& W = c->mg_gs;
  const int blk = 8;
  int rc = layout(W, c, cNX, cNY, N, std::min(8, pick_tk(fl_params{}, cNX, cNY, N)), 8, blk);
  if (rc) return rc;
  SimDesc d = c->desc();
  d.g.NX = cNX;
  d.g.NY = cNY;
  d.buf[B_U] = nullptr;
  d.buf[B_V] = const_cast<float*>(rhs);
  d.buf[B_T3] = p;
  d.masks = masks;
  d.kout = W.d_kout;
  d.gout = W.d_gout;
  d.kinit = W.d_kinit;
  d.G = W.G;
  d.KB = W.KB;
  d.rows = W.rows;
  d.early_exit = 0;
  OneSim m{d};
  const int nskew = W.G * ((W.rows + 1 + LANES - 1) / LANES);
  hipLaunchKernelGGL(k_gs_skew<OneSim>, dim3(nskew), dim3(SKEW_WAVES * LANES), 0, c->stream, m, nullptr,
                     &W.d_state->solve, W.tk, -1, GsPrep{});
  FL_HIP(hipGetLastError());
  GsRun R{};
  R.tiles = W.d_tile;
  R.first = W.d_first;
  R.nq = W.nq;
  R.K = N;
  R.solve = &W.d_state->solve;
  R.count = &W.d_state->run[0];
  auto fn = W.tk == 4 ? k_gs_wave<SOLVE_COARSE, 1, 4, 8, false, OneSim> : k_gs_wave<SOLVE_COARSE, 2, 4, 8, false, OneSim>;
  hipLaunchKernelGGL(fn, dim3(W.grid), dim3(tile_waves(W.tk) * LANES), 0, c->stream, m, R);
  FL_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_gs_unskew<OneSim>, dim3(nskew), dim3(SKEW_WAVES * LANES), 0, c->stream, m, nullptr, W.d_state, N, W.tk,
                     tile_sweeps(W.tk), (int)B_T3, true, 0.0f);
  FL_HIP(hipGetLastError());
  return FL_OK;
}
int gs_coarse_solve(Ctx* c, int cNX, int cNY, int N, const float* rhs, float* p, uint8_t* masks) {
  const int rc = enqueue_coarse_solve(c, cNX, cNY, N, rhs, p, masks);
  if (rc) c->mg_gs.n_alloc = -1;
  return rc;
}

// ---- batched solve ------------------------------------------------------------------------
// All members' tiles in one ticket list, merged by hyperplane start; one persistent launch
// drains it (and one more for the members that early-exit). The initial p is read from role
// rPin (rPin < 0: all zero, Simulate's fill(p, 0)), the solve's p written to rPout, the
// velocity to U2, V2.
// A batch's sweeps per tile: as for one grid, by the tiles of all members.
static int batch_tk(const fl_params& P, const std::vector<SimDesc>& descs, int N) {
  int tk = P.block_sweeps;
  if (!tk_knob(P))
    tk = depth_for([&](int tk) {
      long long n = 0;
      for (const SimDesc& d : descs) n += tiles_in_flight(d.g.NX, d.g.NY, N, tk);
      return n;
    });
  for (const SimDesc& d : descs) tk = shallow_enough(d.g.NX, d.g.NY, N, tk, pick_blk(P));
  return tk;
}
static void batch_free_layout(Batch* B) {
  for (void* p : {(void*)B->d_tiles, (void*)B->d_first, (void*)B->kout, (void*)B->gout, (void*)B->kinit, (void*)B->d_skews,
                  (void*)B->state})
    if (p) (void)hipFree(p);
  (void)hipGetLastError();  // as in free_work
  B->d_tiles = nullptr;
  B->d_first = nullptr;
  B->kout = B->gout = B->kinit = nullptr;
  B->d_skews = nullptr;
  B->state = nullptr;
  B->gs_fields.clear();
  B->gs_n = -1;
}
static int batch_plan(Batch* B, int N, int tk, int blk, const std::vector<SimDesc>& descs) {
  std::vector<GsTile> order;
  std::vector<int> row_steps;
  size_t kbytes = 0, gbytes = 0, ibytes = 0;
  std::vector<SkewItem> skews;
  std::vector<TileGeom> tg(descs.size());
  for (size_t e = 0; e < descs.size(); e++) {
    tg[e] = geom(descs[e].g.NX, descs[e].g.NY, N, tk, blk);
    append_tiles(order, (int)e, (int)row_steps.size(), descs[e].g.NX, N, tk, blk, tg[e]);
    row_steps.insert(row_steps.end(), tg[e].G, tg[e].rows);
    const size_t nt = (size_t)tg[e].G * tg[e].KB;
    kbytes += 16 * nt * tg[e].rows * LANES;
    gbytes += 16 * (nt + tg[e].G) * tg[e].rows * tk;
    ibytes += (size_t)16 * tg[e].G * (tg[e].rows + 1) * LANES;
    for (int g = 0; g < tg[e].G; g++)
      for (int t0 = 0; t0 <= tg[e].rows; t0 += LANES) skews.push_back(SkewItem{(int)e, g, t0, 0});
  }
  std::vector<SolveTile> tiles;
  std::vector<int> first;
  B->nq = device_queues(B->dev, tk);
  const int longest = queue_tiles(order, row_steps, B->nq, tiles, first);
  B->ntiles = (int)order.size();
  FL_HIP(hipMalloc(&B->d_tiles, sizeof(SolveTile) * std::max<size_t>(1, tiles.size())));
  FL_HIP(hipMalloc(&B->d_first, sizeof(int) * first.size()));
  FL_HIP(hipMalloc(&B->kout, std::max<size_t>(kbytes, 16)));
  FL_HIP(hipMalloc(&B->gout, std::max<size_t>(gbytes, 16)));
  FL_HIP(hipMalloc(&B->state, sizeof(GsState)));
  // no word may carry a tag before a solve writes it: the words start at tag 0, the solves at 1
  FL_HIP(hipMemsetAsync(B->kout, 0, kbytes, B->stream));
  FL_HIP(hipMemsetAsync(B->gout, 0, gbytes, B->stream));
  FL_HIP(hipMalloc(&B->kinit, std::max<size_t>(ibytes, 16)));
  FL_HIP(hipMalloc(&B->d_skews, sizeof(SkewItem) * std::max<size_t>(skews.size(), 1)));
  FL_HIP(hipMemcpy(B->d_skews, skews.data(), sizeof(SkewItem) * skews.size(), hipMemcpyHostToDevice));
  B->nskew = (int)skews.size();
  GsState state{};
  state.solve = 1;
  FL_HIP(hipMemcpy(B->state, &state, sizeof(state), hipMemcpyHostToDevice));
  FL_HIP(hipMemcpy(B->d_tiles, tiles.data(), sizeof(SolveTile) * tiles.size(), hipMemcpyHostToDevice));
  FL_HIP(hipMemcpy(B->d_first, first.data(), sizeof(int) * first.size(), hipMemcpyHostToDevice));
  size_t ko = 0, go = 0, io = 0;
  B->gs_fields.assign(descs.size(), SimDesc{});
  for (size_t e = 0; e < descs.size(); e++) {
    SimDesc& d = B->gs_fields[e];
    d.G = tg[e].G;
    d.KB = tg[e].KB;
    d.rows = tg[e].rows;
    d.kout = B->kout + ko;
    d.gout = B->gout + go;
    d.kinit = B->kinit + io;
    const size_t nt = (size_t)d.G * d.KB;
    ko += 16 * nt * d.rows * LANES;
    go += 16 * (nt + d.G) * d.rows * tk;
    io += (size_t)16 * d.G * (d.rows + 1) * LANES;
  }
  B->tk = tk;
  B->blk = blk;
  B->grid = occupancy_grid<ManySims>(B->dev, tk, blk, std::max(B->ntiles, B->nq * longest));
  return FL_OK;
}
int batch_gs_layout(Batch* B, int N, std::vector<SimDesc>& descs) {
  const int tk = batch_tk(B->prm, descs, N);
  const int blk = pick_blk(B->prm);
  auto fill = [&]() {
    for (size_t e = 0; e < descs.size(); e++) {
      const SimDesc& f = B->gs_fields[e];
      SimDesc& d = descs[e];
      d.G = f.G;
      d.KB = f.KB;
      d.rows = f.rows;
      d.kout = f.kout;
      d.gout = f.gout;
      d.kinit = f.kinit;
    }
  };
  if (B->gs_n == N && B->asked == tk && B->blk == blk && B->gs_fields.size() == descs.size()) {
    fill();
    return FL_OK;
  }
  FL_HIP(hipStreamSynchronize(B->stream));  // earlier solves may still use the old layout
  int rc = FL_OK;
  auto fits = [&](int t) {
    for (const SimDesc& d : descs)
      if (!words_fit(geom(d.g.NX, d.g.NY, N, t, blk), t, blk)) return false;
    return true;
  };
  for (int t = tk; t == tk || (t <= (tk_knob(B->prm) ? 0 : 16) && fits(t)); t *= 2) {  // as in layout()
    batch_free_layout(B);
    if ((rc = batch_plan(B, N, t, blk, descs)) == FL_OK) {
      B->gs_n = N;
      B->asked = tk;
      fill();
      return FL_OK;
    }
  }
  batch_free_layout(B);
  return rc;
}

static int enqueue_batch_solve(Batch* B, int N, int rPin, int rPout, float turb) {
  ManySims m{B->d_sims, B->d_cells, B->d_rings};
  const int E = (int)B->members.size();
  // per-sweep maxima and re-run requests of all members are contiguous
  const GsPrep P{prep_groups(B->nring_items), B->nring_items, rPout, B->maxdiv_pool, 2 * B->nmax * E, B->ctrl_pool, E};
  hipLaunchKernelGGL(k_gs_skew<ManySims>, dim3(P.groups + B->nskew), dim3(SKEW_WAVES * LANES), 0, B->stream, m,
                     B->d_skews, &B->state->solve, B->tk, rPin, P);
  FL_HIP(hipGetLastError());
  GsRun R{};
  R.tiles = B->d_tiles;
  R.first = B->d_first;
  R.nq = B->nq;
  R.mode = B->gs_far ? MODE_FAR : 0;
  R.K = N;
  R.solve = &B->state->solve;
  R.omega = B->d_omega;
  R.damping = B->prm.pressure_damping;
  // every member's cp is density h / dt with the batch's density, h and dt
  const bool full = !regular(B->prm, B->descs.empty() ? 0.0f : B->descs[0].cp);
  const int runs = B->prm.early_exit ? 2 : 1;  // no early exit: nothing to decide or re-run
  for (int which = 0; which < runs; which++) {
    R.which = which;
    R.count = &B->state->run[which];
    R.rerun = which ? &B->state->rerun : nullptr;
    int rc = launch_gs(B->tk, B->blk, B->grid, B->stream, m, R, full);
    if (rc) return rc;
    if (which == 0 && runs > 1) {
      // one wave per member, four per workgroup
      hipLaunchKernelGGL(k_gs_decide, dim3((E + 3) / 4), dim3(4 * LANES), 0, B->stream, m, E, N,
                         &B->state->rerun);
      FL_HIP(hipGetLastError());
    }
  }
  hipLaunchKernelGGL(k_gs_unskew<ManySims>, dim3(B->nskew), dim3(SKEW_WAVES * LANES), 0, B->stream, m, B->d_skews, B->state, N,
                     B->tk, tile_sweeps(B->tk), rPout, false, turb);
  FL_HIP(hipGetLastError());
  return FL_OK;
}
int batch_gs_solve(Batch* B, int N, int rPin, int rPout, float turb) {
  const int rc = enqueue_batch_solve(B, N, rPin, rPout, turb);
  if (rc) B->gs_n = -1;
  return rc;
}

}  // namespace fl

// For the tests, and in no header: puts a solve into states that a program reaches by chance or after
// hours. far: the launches of 16-sweep tiles take MODE_FAR, as if an XCD had not started; number (if
// positive): the number of the next solve (the tags repeat after 32768), of an existing layout.
using namespace fl;
static int set_solve_number(hipStream_t stream, GsState* state, int number) {
  if (number <= 0) return FL_OK;
  if (!state) {
    set_error("no solve has run");
    return FL_ERR_INVALID_ARG;
  }
  FL_HIP(hipStreamSynchronize(stream));
  FL_HIP(hipMemcpy(&state->solve, &number, sizeof(number), hipMemcpyHostToDevice));
  return FL_OK;
}
extern "C" int fl_test_solve(fl_ctx* ctx, int far, int number) {
  Ctx* c = reinterpret_cast<Ctx*>(ctx);
  if (!c) return FL_ERR_INVALID_ARG;
  c->gs_far = far != 0;
  return set_solve_number(c->stream, c->gs.d_state, number);
}
extern "C" int fl_test_batch_solve(fl_batch* b, int far, int number) {
  Batch* B = reinterpret_cast<Batch*>(b);
  if (!B) return FL_ERR_INVALID_ARG;
  B->gs_far = far != 0;
  B->graph_gen++;
  return set_solve_number(B->stream, B->state, number);
}
