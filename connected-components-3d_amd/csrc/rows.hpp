// Row kernel: local labelling of multilabel, binary and continuous volumes on
// link bit masks, one 16-voxel row segment per lane.
//
// Replaces the first raster pass of the reference for these paths
// (cc3d/cc3d.hpp:344-1076, cc3d/cc3d_binary.hpp:31-761,
// cc3d/cc3d_continuous.hpp:90-296).  The tile is 64 x 8 x 8 voxels, 64 rows
// of 64; a 256-thread workgroup gives every lane one row and every wave one
// 16-voxel segment of all rows.  A lane reads its own row and the four
// backward rows its connectivity reaches (B: y-1; C, D, E: z-1 at y, y-1,
// y+1) from the tile staged in LDS and holds, per relation p -> q, one bit
// for each voxel of the segment:
//
//   F            foreground
//   a            linked to the voxel before it in the row
//   b0 bm bp     linked to (x, y-1, z), (x-1, y-1, z), (x+1, y-1, z); the
//   c* d* e*     same for the rows C, D, E
//
// multilabel: a bit is one compare and one add-with-carry (push_*), which
// shifts the condition into the mask: 2 VALU operations per voxel and
// relation.  binary: the segments are staged as foreground bits and every
// relation is a shift and an AND.
//
// A link is dropped when another one covers it: p's link to q is implied by
// a linked backward neighbour r of p that is taken before q in the order a,
// c0, b0, bm, bp, cm, cp, e0, d0, em, ep, dm, dp, is adjacent to q and is
// linked to q (equal values are, so adjacency is enough for multilabel and
// binary; continuous links need the bit of the pair r - q, which is another
// bit of the same masks).  The pair r - q belongs to a voxel before p, so by
// induction over (voxel, order) every dropped link follows from kept ones,
// whatever tiles its voxels lie in.  At a tile's first column the link a
// crosses into the next tile: there it comes last in the order and covers
// nothing.  On the 512^3 uint32 Voronoi workload at 26-connectivity this
// leaves 0.10 unions and 0.017 cross-tile requests per voxel.
//
// Union-find nodes are the tile's voxels (LDS position row * 68 + x, raster
// order, so every tree is rooted at its member with the smallest key); a
// voxel points at its run's first voxel in the segment, and the first voxel of a
// segment that continues a run at the voxel before it, from the start.  Kept
// links go to a per-wave queue and are made 64 at a time, one per lane: links
// inside the tile as LDS unions, links out of it as cross-tile requests
// (voxel position | relation << 12) for the global kernels.  Outputs (GP, TR,
// J8/J16, REQ/TQ, tcnt) are those of the voxel kernel in local.hpp except
// for the request format; J is row-major: entry x + 2^jl * (y + 8 * z).
//
// What bounds it: VALU issue, 1,430 to 1,500 instructions per 1,024-voxel wave and
// 75 to 85 % of the issue slots for voxels of up to 4 bytes (grey levels 1,975 and
// 94 %), of which about a third form the masks and a sixth make the unions; LDS is
// busy 40 to 50 % of the time (8-byte voxels, whose masks are formed by halves:
// VALU 62 %, LDS 59 %). Against the kernels it replaced,
// per launch: 512^3 uint32 Voronoi 26 988 -> 390 us, uint64 at 6 1,646 -> 466,
// float32 grey levels 3,068 -> 440, p = 0.3 mask 26 1,057 -> 357, 16384^2 p =
// 0.5 mask 8 1,571 -> 809. That is 64 rows of 64 because a wave then reads
// whole 256-byte rows, the x border (the only one that costs a segment its
// left link) is 1 voxel in 64, and a lane's 16 voxels make masks of one half
// word, two to a register.
#pragma once

#include "common.hpp"
#include "local.hpp"  // LocalParams

namespace cc3d_amd {

// Tile geometry of the row kernels: 64 rows of 64 voxels, 8 x 8 of them for
// volumes (GeoR) and 64 x 1 for single planes (GeoP); GeoRN and GeoPN are the
// same tiles with shorter J rows, for narrow volumes (row_pitch).  Box rows (by, bz): by =
// y + 1, bz = z + 1 (0 in a plane), one halo row or plane on each side that
// backward neighbours reach.
template <int TY_, int TZ_, bool NARROW_ = false>
struct RowGeo {
  static constexpr bool NARROW = NARROW_;
  static constexpr int TX = 64, TY = TY_, TZ = TZ_;
  static constexpr bool IS3D = TZ > 1;
  static constexpr int NT = 256;
  static constexpr int TV = TX * TY * TZ;
  static constexpr int BY = IS3D ? TY + 2 : TY + 1, BZ = IS3D ? TZ + 1 : 1;
  static constexpr int NROWS = BY * BZ;
  static_assert(TY * TZ == 64, "one row per lane of a wave");
  // J: 2^jl entries a row
  __device__ static inline int jlog(int jl) { return NARROW ? jl : 6; }
  __device__ static inline int jidx(int lx, int ly, int lz, int jl) { return lx + ((ly + TY * lz) << jlog(jl)); }
};
using GeoR = RowGeo<8, 8>;
using GeoP = RowGeo<64, 1>;
using GeoRN = RowGeo<8, 8, true>;
using GeoPN = RowGeo<64, 1, true>;
template <class G>
constexpr bool is_row_geo = std::is_same<G, GeoR>::value || std::is_same<G, GeoP>::value ||
                            std::is_same<G, GeoRN>::value || std::is_same<G, GeoPN>::value;

// Relations in covering order; index 12 is a.  Offsets as (d + 1) in 2-bit
// fields per axis.
enum : int { R_C0, R_B0, R_BM, R_BP, R_CM, R_CP, R_E0, R_D0, R_EM, R_EP, R_DM, R_DP, R_A, R_N };
__host__ __device__ constexpr Off rel_off(int r) {
  switch (r) {
    case R_C0: return {0, 0, -1};
    case R_B0: return {0, -1, 0};
    case R_BM: return {-1, -1, 0};
    case R_BP: return {1, -1, 0};
    case R_CM: return {-1, 0, -1};
    case R_CP: return {1, 0, -1};
    case R_E0: return {0, 1, -1};
    case R_D0: return {0, -1, -1};
    case R_EM: return {-1, 1, -1};
    case R_EP: return {1, 1, -1};
    case R_DM: return {-1, -1, -1};
    case R_DP: return {1, -1, -1};
    default: return {-1, 0, 0};
  }
}
__host__ __device__ constexpr uint32_t rel_packed(int axis) {
  uint32_t m = 0;
  for (int r = 0; r < R_N; r++) {
    const Off o = rel_off(r);
    m |= (uint32_t)((axis == 0 ? o.dx : axis == 1 ? o.dy : o.dz) + 1) << (2 * r);
  }
  return m;
}
// Does an offset belong to connectivity nb?  (Also: are two voxels that far
// apart adjacent.)
__host__ __device__ constexpr bool off_in(int dx, int dy, int dz, int nb) {
  const int ax = dx < 0 ? -dx : dx, ay = dy < 0 ? -dy : dy, az = dz < 0 ? -dz : dz;
  const int l1 = ax + ay + az;
  if (ax > 1 || ay > 1 || az > 1) return false;
  if (nb == 8 || nb == 4) return az == 0 && (nb == 8 || l1 <= 1);
  return nb == 26 || (nb == 18 && l1 <= 2) || (nb == 6 && l1 <= 1);
}
__host__ __device__ constexpr bool rel_in(int r, int nb) {
  return off_in(rel_off(r).dx, rel_off(r).dy, rel_off(r).dz, nb);
}
__host__ __device__ constexpr bool rel_adj(int i, int j, int nb) {
  const Off a = rel_off(i), b = rel_off(j);
  return off_in(a.dx - b.dx, a.dy - b.dy, a.dz - b.dz, nb);
}
// Offset of relation r (run time).
__device__ inline void rel_decode(uint32_t r, int& dx, int& dy, int& dz) {
  constexpr uint32_t PX = rel_packed(0), PY = rel_packed(1), PZ = rel_packed(2);
  dx = (int)((PX >> (2 * r)) & 3u) - 1;
  dy = (int)((PY >> (2 * r)) & 3u) - 1;
  dz = (int)((PZ >> (2 * r)) & 3u) - 1;
}

// J entries per row of a tile, as a power of two: 16, 32 or 64 columns.  A
// narrow volume has one tile in x, of whose 64 columns the rest would be scratch
// that nothing uses (at 16 x N x N and 26-connectivity 24 bytes of scratch a
// voxel, 34 for continuous links; voxel tiles of 32 x 8 x 8 take 18).  Kernels of
// their own, because the general address costs the others up to 1.5 % (16384^2
// mask at 8: 801 and 813 us).
__host__ constexpr int row_pitch(int64_t sx) { return sx <= 16 ? 4 : sx <= 32 ? 5 : 6; }

// Whether a tile's requests may be link masks (see there).
__host__ __device__ constexpr bool row_masks(bool cont, int nb) { return cont && (nb == 26 || nb == 18); }

// Bound on the requests of a tile.  Multilabel and binary: the largest number
// of kept relations that leave the tile, over every set of links a voxel can
// have, summed over the tile's voxels (4,036 at 26-connectivity, 2,537 at
// 18, 1,088 at 6).  Narrow tiles have no neighbour in x: what is left is the
// sum over a column of 64 rows (60, 38, 16).  Planes and 6-connected continuous
// volumes: all relations that leave the tile (382 in a plane).  Continuous
// links at 26 and 18 could leave 9,316 and 5,280, but only in a lattice made for
// it (noise at its worst tolerance leaves 2,520): there a tile has 1,024 entries
// per segment, and one that says which segments hold link masks instead (in
// 16 bytes).  Never below the 128 that the union kernels load unasked.
__host__ __device__ constexpr int row_req_cap(bool cont, int nb, int jl) {
  if (row_masks(cont, nb)) return (64 << jl) + 8;
  if (jl < 6) {
    const int n = (nb == 8 || nb == 4 ? 3 : nb == 6 ? 16 : nb == 18 ? 38 : 60) << jl;
    return n < 128 ? 128 : n;
  }
  return nb == 8 || nb == 4 ? 384 : nb == 6 ? 1088 : nb == 18 ? 2540 : 4036;
}

// Staged voxel type: 4 bytes for every type up to 4 bytes.  Multilabel 8-byte
// voxels are staged as 4-byte halves one after the other (their masks are
// ANDed), which keeps 6 workgroups per CU instead of 3; continuous ones whole.
template <class T, int MODE>
struct RowVal {
  using type = uint32_t;
  static constexpr bool SPLIT = sizeof(T) == 8;
};
template <int MODE>
struct RowVal<float, MODE> {
  using type = float;
  static constexpr bool SPLIT = false;
};
template <>
struct RowVal<uint64_t, M_CONT> {
  using type = uint64_t;
  static constexpr bool SPLIT = false;
};
template <>
struct RowVal<double, M_CONT> {
  using type = double;
  static constexpr bool SPLIT = false;
};
// Half H of an 8-byte voxel.  Doubles compare as bits once -0 is 0 and every
// NaN the default one, which links to nothing (NANHI, a high half that only
// NaNs have).
constexpr uint32_t NANHI = 0x7FF80000u;
template <int H>
__device__ inline uint32_t half_of(uint64_t v) {
  return (uint32_t)(v >> (32 * H));
}
template <int H>
__device__ inline uint32_t half_of(double v) {
  const uint64_t b = v == 0.0 ? 0ull : v != v ? (uint64_t)NANHI << 32 : __builtin_bit_cast(uint64_t, v);
  return (uint32_t)(b >> (32 * H));
}

constexpr int RSTR = 68;   // row stride of staged values and nodes: 16-byte accesses of 64 rows spread over all banks
constexpr int PSTR = 704;  // plane stride of staged values: 10 rows, and 24 more so that planes start on the same bank
constexpr uint32_t SLOW = 0x8000u;
constexpr int RQCAP = 1024;  // queued links per wave; one relation of a wave's segments always fits

// LDS index of a tile voxel's node: raster order, or for the binary 2D
// 8-connected numbering the order of the 2x2 block keys (pairs of rows, 4
// nodes a block, 132 a pair).
template <int QK>
__device__ inline uint32_t row_node(uint32_t x, uint32_t row) {
  if (QK == Q_BLOCK8) return 132u * (row >> 1) + 4u * (x >> 1) + 2u * (row & 1u) + (x & 1u);
  return RSTR * row + x;
}
// Node of voxel k of a segment whose first voxel has node n0.
template <int QK>
__device__ inline uint32_t seg_node(uint32_t n0, uint32_t k) {
  return QK == Q_BLOCK8 ? n0 + 4u * (k >> 1) + (k & 1u) : n0 + k;
}

template <class T, int MODE, class G_ = GeoR>
struct RowLds {
  using G = G_;
  using VT = typename RowVal<T, MODE>::type;
  struct Work {
    uint32_t par[64 * RSTR];
    uint16_t queue[4][RQCAP];  // per wave; later, per wave: segment bits [row]
  };
  union alignas(16) {
    // staged box: x = -1 at 3, x = 0..63 at 4..67, x = 64 at 68 (the next row's unused first element)
    VT v[MODE == M_BINARY ? 4 : G::IS3D ? G::BZ * PSTR : G::NROWS * RSTR + 4];
    // staged foreground bits, 16 per half-word: x = -1 in bit 15 of 0, segments in 1..4, x = 64 in bit 0 of 5
    uint16_t fb[G::NROWS][6];
    Work w;
  } u;
  // binary 2D-4: values of the plane's first row that differ from the one
  // before; continuous volumes: bound on the wave's requests (SLOW: more links
  // than its queue holds)
  uint16_t ne0[4];
  uint32_t nreq;
  uint32_t wtot[4], red_epl[4], red_prov[4];
  uint64_t rows[4];
};

// m = 2 m + condition
__device__ inline void push_bit(uint32_t& m, bool c) { m = m + m + (c ? 1u : 0u); }
__device__ inline void push_eq(uint32_t& m, uint32_t a, uint32_t b) {
  asm("v_cmp_eq_u32_e32 vcc, %1, %2\n\tv_addc_co_u32_e32 %0, vcc, %0, %0, vcc" : "+v"(m) : "v"(a), "v"(b) : "vcc");
}
__device__ inline void push_eq(uint32_t& m, float a, float b) {
  asm("v_cmp_eq_f32_e32 vcc, %1, %2\n\tv_addc_co_u32_e32 %0, vcc, %0, %0, vcc" : "+v"(m) : "v"(a), "v"(b) : "vcc");
}
__device__ inline void push_eq(uint32_t& m, uint64_t a, uint64_t b) {
  asm("v_cmp_eq_u64_e32 vcc, %1, %2\n\tv_addc_co_u32_e32 %0, vcc, %0, %0, vcc" : "+v"(m) : "v"(a), "v"(b) : "vcc");
}
__device__ inline void push_eq(uint32_t& m, double a, double b) {
  asm("v_cmp_eq_f64_e32 vcc, %1, %2\n\tv_addc_co_u32_e32 %0, vcc, %0, %0, vcc" : "+v"(m) : "v"(a), "v"(b) : "vcc");
}
__device__ inline void push_fg(uint32_t& m, uint32_t a) {
  asm("v_cmp_ne_u32_e32 vcc, 0, %1\n\tv_addc_co_u32_e32 %0, vcc, %0, %0, vcc" : "+v"(m) : "v"(a) : "vcc");
}
__device__ inline void push_fg(uint32_t& m, float a) {
  asm("v_cmp_neq_f32_e32 vcc, 0, %1\n\tv_addc_co_u32_e32 %0, vcc, %0, %0, vcc" : "+v"(m) : "v"(a) : "vcc");
}
template <class V>
__device__ inline void push_fg(uint32_t& m, V a) {
  push_bit(m, a != V(0));
}

// Continuous link between two staged values (cc3d/cc3d_continuous.hpp:79-88).
// Floating-point background is staged as a NaN, which links to nothing, so
// the link is one subtraction and one compare; integers test both for zero.
template <class V>
__device__ inline void push_link(uint32_t& m, V a, V b, V delta) {
  push_bit(m, a != V(0) && b != V(0) && match<V>(a, b, delta));
}
__device__ inline void push_link(uint32_t& m, float a, float b, float delta) {
  asm("v_cmp_le_f32_e64 vcc, |%1|, %2\n\tv_addc_co_u32_e32 %0, vcc, %0, %0, vcc"
      : "+v"(m) : "v"(a - b), "s"(delta) : "vcc");
}
__device__ inline void push_link(uint32_t& m, double a, double b, double delta) {
  asm("v_cmp_le_f64_e64 vcc, |%1|, %2\n\tv_addc_co_u32_e32 %0, vcc, %0, %0, vcc"
      : "+v"(m) : "v"(a - b), "s"(delta) : "vcc");
}
// Staged form of a value of a continuous volume: background becomes the NaN
// of all ones, every other NaN the default one.
__device__ inline float cont_stage(float v) {
  const uint32_t b = v == 0.0f ? 0xFFFFFFFFu : v != v ? 0x7FC00000u : __builtin_bit_cast(uint32_t, v);
  return __builtin_bit_cast(float, b);
}
__device__ inline double cont_stage(double v) {
  const uint64_t b = v == 0.0 ? ~0ull : v != v ? 0x7FF8000000000000ull : __builtin_bit_cast(uint64_t, v);
  return __builtin_bit_cast(double, b);
}
template <class V>
__device__ inline V cont_stage(V v) {
  return v;
}
__device__ inline bool cont_fg(float v) { return __builtin_bit_cast(uint32_t, v) != 0xFFFFFFFFu; }
__device__ inline bool cont_fg(double v) { return __builtin_bit_cast(uint64_t, v) != ~0ull; }
template <class V>
__device__ inline bool cont_fg(V v) {
  return v != V(0);
}

// Orders the wave's memory accesses before and after (its LDS accesses are
// performed in order, so this is a matter for the compiler only).
__device__ inline void wave_order() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ inline uint64_t wave_ballot(bool p) { return (uint64_t)__ballot(p); }

// Lanes below this one in m.
__device__ inline uint32_t mbcnt64(uint64_t m) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// LDS union-find over 32-bit parents.  A parent is never larger than its
// node, so walks end.  A union climbs on the side of the larger parent and
// lowers that parent to the other side's on the way (an atomic minimum that
// returns what it replaced): either the node was a root and is linked now, or
// the parent it gave up is the next node to join.  A join left undone is
// always some lane's next step, so no link is lost.  Two finds to the roots
// and then the link took 440 us on 512^3 uint32 Voronoi (26) and 1,025 us on
// a 16384^2 mask (8), this 410 and 831 us.
__device__ inline void lstore(uint32_t* p, uint32_t v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ inline uint32_t rfind_ro(const uint32_t* par, uint32_t a) {
  uint32_t p = lload(par + a);
  while (p != a) {
    a = p;
    p = lload(par + a);
  }
  return a;
}
__device__ inline void runion(uint32_t* par, uint32_t a, uint32_t b) {
  while (true) {
    const uint32_t pa = lload(par + a), pb = lload(par + b);
    if (pa == pb) return;
    const uint32_t c = pa > pb ? a : b, lo = pa > pb ? pb : pa;
    const uint32_t old = atomicMin(par + c, lo);
    if (old == c) return;  // c was a root: linked under lo
    a = old;
    b = lo;
  }
}

// N consecutive voxels from p (aligned to a voxel), as the widest loads that
// alignment allows.
template <class T, int N>
__device__ inline void load_run(const T* p, T (&v)[N]) {
  typedef T V4 __attribute__((ext_vector_type(4), aligned(sizeof(T))));
#pragma unroll
  for (int i = 0; i < N; i += 4) {
    const V4 k = *reinterpret_cast<const V4*>(p + i);
#pragma unroll
    for (int j = 0; j < 4; j++) v[i + j] = k[j];
  }
}

// Bit k of the result: byte k of w is not zero, for the 16 bytes of four
// words; t has 0x80 in each such byte and a dot product gathers them.
__device__ inline uint32_t nonzero_bytes(const uint32_t (&w)[4]) {
  uint32_t acc = 0, out[2];
#pragma unroll
  for (int h = 0; h < 2; h++) {
    acc = 0;
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const uint32_t x = w[2 * h + i];
      const uint32_t t = (((x & 0x7F7F7F7Fu) + 0x7F7F7F7Fu) | x) & 0x80808080u;
      acc = __builtin_amdgcn_udot4(t, i ? 0x80402010u : 0x08040201u, acc, false);
    }
    out[h] = acc >> 7;
  }
  return out[0] | (out[1] << 8);
}

template <class T, int MODE, int NB, class G, int QK>
__device__ inline void rows_tile(const LocalParams& p, const T* in, int64_t sx, int64_t sy, int64_t sz, int64_t ntx,
                                 int64_t nty, Div dxy, Div dx, int64_t tile, int64_t slot, uint32_t keybase,
                                 RowLds<T, MODE, G>& L) {
  constexpr bool IS3D = G::IS3D;
  constexpr bool FACE = NB == 6 || NB == 4;  // face links only
  using VT = typename RowVal<T, MODE>::type;
  constexpr bool SPLIT = RowVal<T, MODE>::SPLIT;
  const int t = threadIdx.x, lane = t & 63;
  const int seg = __builtin_amdgcn_readfirstlane(t >> 6);  // one segment per wave
  int64_t tx, ty, tz;
  tile_coords((uint32_t)tile, ntx, nty, dxy, dx, tx, ty, tz);
  const int64_t x0 = tx * G::TX, y0 = ty * G::TY, z0 = tz * G::TZ;
  uint32_t my_epl = 0, my_prov = 0;
  if (t == 0) L.nreq = 0;

  // 2. masks of the wave's segment: bit k is voxel 16 seg + k of row `lane`
  const int ly = lane & (G::TY - 1), lz = lane / G::TY;
  const bool first = seg == 0;  // bit 0 is the tile's first column
  uint32_t F = 0, a = 0;
  uint32_t U[R_N];  // kept links
#pragma unroll
  for (int i = 0; i < R_N; i++) U[i] = 0;
  uint32_t M[R_N];  // all links
#pragma unroll
  for (int i = 0; i < R_N; i++) M[i] = 0;
  uint32_t hD0 = 0;       // 6-connectivity: equal to the voxel of d0 (bm, cm are in M)
  uint32_t left_cov = 0;  // continuous: bit 0, the link a of the tile's first column is covered
  // offsets of the staged rows B, C, D, E from a row
  constexpr int RB = -RSTR, RC = -PSTR, RD = -PSTR - RSTR, RE = -PSTR + RSTR;
  [[maybe_unused]] auto masks = [&](auto half) {
    [[maybe_unused]] constexpr int H = decltype(half)::value;
    const VT* base = static_cast<const VT*>(__builtin_assume_aligned(
      L.u.v + ((ly + 1) * RSTR + (IS3D ? (lz + 1) * PSTR : 0) + 4 + 16 * seg), 16));
    VT cur[16];
#pragma unroll
    for (int k = 0; k < 16; k++) cur[k] = base[k];
    const VT left = base[-1];
    if constexpr (MODE == M_MULTI) {
      // one half of a split voxel: nonzero halves ORed, equal halves ANDed
      auto both = [&](uint32_t& m, uint32_t half_m) { m = H ? (m & half_m) : half_m; };
      uint32_t f = 0, e = 0;
#pragma unroll
      for (int k = 15; k >= 0; k--) {
        push_fg(f, cur[k]);
        push_eq(e, cur[k], k > 0 ? cur[k > 0 ? k - 1 : 0] : left);
      }
      F |= f;
      both(a, e);
      // W0/WM/WP: which of the row's three relations to form
      auto rel = [&](int dr, int i0, int im, int ip, bool W0, bool WM, bool WP) {
        const VT* w = base + dr;
        VT wv[18];  // x = -1 .. 16 of the segment
#pragma unroll
        for (int k = 0; k < 18; k++)
          if ((k > 0 || WM) && (k < 17 || WP)) wv[k] = w[k - 1];
        uint32_t m0 = 0, mm = 0, mp = 0;
#pragma unroll
        for (int k = 15; k >= 0; k--) {
          if (W0) push_eq(m0, cur[k], wv[k + 1]);
          if (WM) push_eq(mm, cur[k], wv[k]);
          if (WP) push_eq(mp, cur[k], wv[k + 2]);
        }
        if (W0) both(M[i0], m0);
        if (WM) both(M[im], mm);
        if (WP) both(M[ip], mp);
      };
      rel(RB, R_B0, R_BM, R_BP, true, true, !FACE);
      if constexpr (IS3D) {
        rel(RC, R_C0, R_CM, R_CP, true, true, !FACE);
        rel(RD, R_D0, R_DM, R_DP, true, NB == 26, NB == 26);
        if constexpr (!FACE) rel(RE, R_E0, R_EM, R_EP, true, NB == 26, NB == 26);
      }
      if (H == 1 || !SPLIT) {
        uint32_t lk = F;
        if constexpr (std::is_same<T, double>::value) {
          uint32_t nan = 0;
#pragma unroll
          for (int k = 15; k >= 0; k--) push_eq(nan, cur[k], NANHI);
          lk &= ~nan;
        }
        a &= lk;
#pragma unroll
        for (int i = 0; i < R_A; i++) M[i] &= lk;
        hD0 = M[R_D0];
        my_epl = (uint32_t)__popc(F & ~a);
      }
    }
    if constexpr (MODE == M_CONT) {
      const VT delta = (VT)from_bits<T>(p.delta_bits);
      uint32_t eq = 0;
#pragma unroll
      for (int k = 15; k >= 0; k--) {
        const VT pv = k > 0 ? cur[k > 0 ? k - 1 : 0] : left;
        push_bit(F, cont_fg(cur[k]));
        push_eq(eq, cur[k], pv);
        push_link(a, cur[k], pv, delta);
      }
      my_epl = (uint32_t)__popc(F & ~eq);
      const uint32_t inner = first ? (a & ~1u) : a;
      // One backward row: its links, and the kept ones.  Masks of 17 bits
      // have the voxel before the segment in bit 0: the link of voxel k - 1
      // to the voxel at x is a pair (a, q), so it covers p - q where p has
      // the link a; xw: links along the row itself, w[k] - w[k + 1].
      uint32_t bd = 0, ce = 0;
      VT prow[16];  // rows B and C at 18-connectivity, for the pairs (b0, d0) and (c0, e0)
      auto rel = [&](int dr, int i0, int im, int ip, bool diag, bool quirk, bool keep, uint32_t* pair,
                     bool left_rule) {
        const VT* w = base + dr;
        VT wv[18];
#pragma unroll
        for (int k = 0; k < 18; k++)
          if (k < 17 || !FACE) wv[k] = w[k - 1];
        uint32_t x0m = 0, xpm = 0, xw = 0, eqm = 0;
#pragma unroll
        for (int k = 15; k >= -1; k--) {
          const VT c = k >= 0 ? cur[k >= 0 ? k : 0] : left;
          push_link(x0m, c, wv[k + 1], delta);
          if (quirk) push_eq(eqm, c, wv[k + 1]);
          if (diag) push_link(xpm, c, wv[k + 2], delta);
          if (k >= 0 && diag) push_link(M[im], c, wv[k], delta);
          if (FACE) {
            if (k >= 0) push_link(xw, wv[k + 1], wv[k], delta);
          } else if (diag) {
            push_link(xw, wv[k + 2], wv[k + 1], delta);
          }
        }
        if (pair) {
#pragma unroll
          for (int k = 15; k >= 0; k--) push_link(*pair, prow[k], wv[k + 1], delta);
        }
        if (keep) {
#pragma unroll
          for (int k = 0; k < 16; k++) prow[k] = wv[k + 1];
        }
        // equal to the voxel below: linked under 26-connectivity whatever delta says
        // (cc3d/cc3d_continuous.hpp:147-150); a background c is masked by F below
        if (quirk) {
          const uint32_t f17 = (F << 1) | (cont_fg(left) ? 1u : 0u);
          x0m |= eqm & f17;
        }
        M[i0] = x0m >> 1;
        const uint32_t s0 = x0m & 0xFFFFu;  // voxel k - 1 to the voxel of im
        if constexpr (FACE) {
          const uint32_t cov = s0 & xw;
          U[i0] = M[i0] & ~(inner & cov);
          left_cov |= M[i0] & cov;
        } else {
          const uint32_t sp = xpm & 0xFFFFu;  // voxel k - 1 to the voxel of i0
          uint32_t cov0 = rel_adj(R_A, i0, NB) ? (inner & sp) : 0u;
          if (pair) cov0 |= M[i0 == R_D0 ? R_B0 : R_C0] & *pair;
          U[i0] = M[i0] & ~cov0;
          if (diag) {
            M[ip] = xpm >> 1;
            U[im] = M[im] & ~(inner & s0) & ~(M[i0] & xw);
            U[ip] = M[ip] & ~(M[i0] & (xw >> 1));
          }
          if (left_rule) left_cov |= M[i0] & sp;
        }
      };
      constexpr bool D = !FACE, D26 = NB == 26, P18 = NB == 18;
      rel(RB, R_B0, R_BM, R_BP, D, false, P18, nullptr, true);
      if constexpr (IS3D && !FACE) rel(RD, R_D0, R_DM, R_DP, D26, false, false, P18 ? &bd : nullptr, false);
      if constexpr (IS3D) rel(RC, R_C0, R_CM, R_CP, D, NB == 26, P18, nullptr, true);
      if constexpr (IS3D && !FACE) rel(RE, R_E0, R_EM, R_EP, D26, false, false, P18 ? &ce : nullptr, false);
    }
  };

  // 1. stage the box: rows r = by + BY * bz.  Row BY - 1 of the last plane is
  //    reached by no voxel.  Voxels outside the volume are background.
  // box position (-1, -1, -1) ((-1, -1) in a plane); dereferenced inside the volume only
  const T* box = in + ((x0 - 1) + sx * ((y0 - 1) + (IS3D ? sy * (z0 - 1) : 0)));
  const int xleft = (int)(sx - x0 < 128 ? sx - x0 : 128);  // voxels of a row from x0 on
  // box rows and planes inside the volume: [ylo, yhi) and [zlo, zhi)
  const int ylo = y0 == 0 ? 1 : 0, yhi = (int)(sy - y0 + 1 < G::BY ? sy - y0 + 1 : G::BY);
  const int zlo = IS3D && z0 == 0 ? 1 : 0, zhi = IS3D && sz - z0 + 1 < G::BZ ? (int)(sz - z0 + 1) : G::BZ;
  auto row_ok = [&](int by, int bz) -> bool { return by >= ylo && by < yhi && bz >= zlo && bz < zhi; };
  const int64_t pitch = sx * sy;
  auto row_ptr = [&](int by, int bz) -> const T* {  // its x0
    return box + (1 + (int64_t)by * sx + (IS3D ? (int64_t)bz * pitch : 0));
  };
  auto row_of = [&](int r, int& by, int& bz) {  // box row r < 128
    bz = IS3D ? (r * 205) >> 11 : 0;  // r / 10
    static_assert(!IS3D || G::BY == 10, "division by 10");
    by = r - bz * G::BY;
  };
  if constexpr (MODE == M_BINARY) {
    // 16 voxels (one segment) per thread and pass
    constexpr int ITEMS = 4 * G::NROWS;
    constexpr int PASSES = (ITEMS + G::NT - 1) / G::NT;
#pragma unroll
    for (int q = 0; q < PASSES; q++) {
      const int i = t + G::NT * q;
      if (i >= ITEMS) break;
      const int r = i >> 2, s = i & 3;
      int by, bz;
      row_of(r, by, bz);
      uint32_t F = 0, NE = 0;  // NE: differs from the voxel before it (tile rows)
      if (row_ok(by, bz) && 16 * s < xleft) {
        const T* e = row_ptr(by, bz) + 16 * s;
        const bool own = by >= 1 && by <= G::TY && (!IS3D || bz >= 1);
        T prev = T(0);
        if (own && x0 + 16 * s > 0) prev = e[-1];
        if (16 * s + 16 <= xleft) {
          T v[16];
          if constexpr (sizeof(T) == 1) {
            typedef uint32_t Words __attribute__((ext_vector_type(4), aligned(1)));
            const Words q4 = *reinterpret_cast<const Words*>(e);
            const uint32_t w[4] = {q4[0], q4[1], q4[2], q4[3]};
            uint32_t d[4];
            F = nonzero_bytes(w);
            d[0] = w[0] ^ ((w[0] << 8) | (uint32_t)(uint8_t)prev);
#pragma unroll
            for (int k = 1; k < 4; k++) d[k] = w[k] ^ __builtin_amdgcn_alignbyte(w[k], w[k - 1], 3);
            NE = nonzero_bytes(d);
          } else {
            load_run<T, 16>(e, v);
#pragma unroll
            for (int k = 15; k >= 0; k--) {
              push_bit(F, v[k] != T(0));
              push_bit(NE, v[k] != (k > 0 ? v[k - 1] : prev));
            }
          }
        } else {
          const int n = (int)(xleft - 16 * s);
          for (int k = 0; k < n; k++) {
            const T c = e[k];
            F |= (uint32_t)(c != T(0)) << k;
            NE |= (uint32_t)(c != prev) << k;
            prev = c;
          }
        }
        if (own) my_epl += (uint32_t)__popc(F & NE);
        if (QK == Q_BIN4 && by == 1) L.ne0[s] = (uint16_t)NE;
      }
      L.u.fb[r][s + 1] = (uint16_t)F;
    }
    if (t < 2 * G::NROWS) {
      const int r = t >> 1, right = t & 1;
      int by, bz;
      row_of(r, by, bz);
      const bool ok = row_ok(by, bz) && (right ? xleft > 64 : x0 > 0);
      const bool f = ok && row_ptr(by, bz)[right ? 64 : -1] != T(0);
      L.u.fb[r][right ? 5 : 0] = (uint16_t)(f ? (right ? 1u : 0x8000u) : 0u);
    }
  } else {
    // 4 voxels per lane and load, 4 rows a wave; all loads first.  The rows of
    // load l = seg + 4 q: in a volume rows 0-3 or 4-7 of plane l / 2 for l <
    // 18, then rows 8 and 9 of planes 2 (l - 18) and the next; in a plane
    // rows 4 l to 4 l + 3.  Bases are wave-uniform, a lane's offset is one of
    // two constants.
    constexpr int PASSES = IS3D ? 6 : (G::NROWS + 15) / 16;
    const int q4 = 4 * (lane & 15), sub = lane >> 4;
    T v[PASSES][4];
    const bool inner = x0 + G::TX <= sx && ylo == 0 && yhi == G::BY && zlo == 0 && zhi == G::BZ;
    auto base_row = [&](int q, int& by, int& bz) -> bool {  // false: the two-plane form
      const int l = seg + 4 * q;
      if (!IS3D) {
        by = 4 * l;
        bz = 0;
        return true;
      }
      if (l < 18) {
        by = (l & 1) * 4;
        bz = l >> 1;
        return true;
      }
      by = 8;
      bz = 2 * (l - 18);
      return false;
    };
    const int64_t offa = (int64_t)sub * sx + q4, offb = (int64_t)(sub & 1) * sx + (int64_t)(sub >> 1) * pitch + q4;
    const int sub_y = sub & 1, sub_z = sub >> 1;
#pragma unroll
    for (int q = 0; q < PASSES; q++) {
      int by, bz;
      const bool quad = base_row(q, by, bz);
#pragma unroll
      for (int k = 0; k < 4; k++) v[q][k] = T(0);
      const T* e = row_ptr(by, bz) + (quad ? offa : offb);
      if (inner && quad && by + 3 < G::BY && bz < G::BZ) {
        load_run<T, 4>(e, v[q]);
      } else if (quad ? row_ok(by + sub, bz) : row_ok(by + sub_y, bz + sub_z)) {
        if (q4 + 4 <= xleft) {
          load_run<T, 4>(e, v[q]);
        } else {
#pragma unroll
          for (int k = 0; k < 4; k++)
            if (q4 + k < xleft) v[q][k] = e[k];
        }
      }
    }
    T hx = T(0);
    const int hr = t >> 1, right = t & 1;
    int hby, hbz;
    row_of(hr, hby, hbz);
    if (t < 2 * G::NROWS && row_ok(hby, hbz) && (right ? xleft > 64 : x0 > 0))
      hx = row_ptr(hby, hbz)[right ? 64 : -1];
    // half: which half of a split voxel
    auto put = [&](auto half) {
      auto staged = [&](T c) -> VT {
        if constexpr (SPLIT) return half_of<decltype(half)::value>(c);
        else if constexpr (MODE == M_CONT) return cont_stage((VT)c);
        else return (VT)c;
      };
#pragma unroll
      for (int q = 0; q < PASSES; q++) {
        int by, bz;
        const bool quad = base_row(q, by, bz);
        const int dy = quad ? sub : sub_y, dz = quad ? 0 : sub_z;
        if (by + dy < G::BY && bz + dz < G::BZ) {
          VT* d = static_cast<VT*>(
            __builtin_assume_aligned(L.u.v + (by * RSTR + bz * PSTR + (dy * RSTR + dz * PSTR + 4 + q4)), 16));
#pragma unroll
          for (int k = 0; k < 4; k++) d[k] = staged(v[q][k]);
        }
      }
      if (t < 2 * G::NROWS) L.u.v[hby * RSTR + hbz * PSTR + (right ? 68 : 3)] = staged(hx);
    };
    put(std::integral_constant<int, 0>());
    __syncthreads();
    masks(std::integral_constant<int, 0>());
    if constexpr (SPLIT) {
      __syncthreads();
      put(std::integral_constant<int, 1>());
      __syncthreads();
      masks(std::integral_constant<int, 1>());
    }
  }
  if constexpr (MODE == M_BINARY) {
    __syncthreads();
    const int r0 = (ly + 1) + (IS3D ? G::BY * (lz + 1) : 0);
    constexpr int B = -1, C = -G::BY, D = -G::BY - 1, E = -G::BY + 1;  // box rows from r0
    auto bits = [&](int r, uint32_t& m0, uint32_t& mm, uint32_t& mp) {
      const uint16_t* b = &L.u.fb[r][seg];
      const uint32_t c = b[1];
      m0 = c;
      mm = ((c << 1) | (uint32_t)(b[0] >> 15)) & 0xFFFFu;
      mp = (c >> 1) | (((uint32_t)b[2] & 1u) << 15);
    };
    uint32_t mm, mp;
    bits(r0, F, mm, mp);
    a = F & mm;
    auto rel = [&](int dr, int i0, int im, int ip) {
      uint32_t m0;
      bits(r0 + dr, m0, mm, mp);
      M[i0] = F & m0;
      M[im] = F & mm;
      M[ip] = F & mp;
    };
    rel(B, R_B0, R_BM, R_BP);
    if constexpr (IS3D) {
      rel(C, R_C0, R_CM, R_CP);
      rel(D, R_D0, R_DM, R_DP);
      if constexpr (!FACE) rel(E, R_E0, R_EM, R_EP);
      hD0 = M[R_D0];
    }
    if constexpr (QK == Q_BIN4) {
      // the first row links on equal values, later rows to the left unless
      // the two pixels above are both set (cc3d/cc3d_binary.hpp:822-935)
      a &= y0 + ly == 0 ? ~(uint32_t)L.ne0[seg] : ~(M[R_B0] & M[R_BM]);
    }
  }
  {
    uint32_t any;
    const uint32_t ain = first ? (a & ~1u) : a;  // links a inside the tile
    if constexpr (MODE != M_CONT) {
      if constexpr (QK == Q_BIN4) {
        any = a | M[R_B0];
        U[R_B0] = M[R_B0];  // the reference's own links, none covered
        U[R_A] = a & ~ain;
      } else if constexpr (FACE) {
        any = a | M[R_B0] | M[R_C0];
        U[R_B0] = M[R_B0] & ~(ain & M[R_BM]);
        U[R_C0] = M[R_C0] & ~(ain & M[R_CM]) & ~(M[R_B0] & hD0);
        U[R_A] = a & ~ain & ~((M[R_B0] & M[R_BM]) | (M[R_C0] & M[R_CM]));
      } else {
        any = a;
        uint32_t cova = 0;
#pragma unroll
        for (int i = 0; i < R_A; i++) {
          if (!rel_in(i, NB)) continue;
          any |= M[i];
          uint32_t cov = rel_adj(R_A, i, NB) ? ain : 0u;
#pragma unroll
          for (int j = 0; j < i; j++)
            if (rel_in(j, NB) && rel_adj(j, i, NB)) cov |= M[j];
          if (rel_adj(R_A, i, NB)) cova |= M[i];
          U[i] = M[i] & ~cov;
        }
        U[R_A] = a & ~ain & ~cova;
      }
    } else {
      any = a;
#pragma unroll
      for (int i = 0; i < R_A; i++)
        if (rel_in(i, NB)) any |= M[i];
      U[R_A] = a & ~ain & ~left_cov;
    }
    if (QK != Q_BLOCK8) my_prov = (uint32_t)__popc(F & ~any);  // block labels are counted separately
  }
  const uint32_t S = F & (first ? ~(a & ~1u) : ~a);  // run starts inside the tile
  const uint64_t fgrows = wave_ballot(F != 0u);
  __syncthreads();  // the staged box is dead: par and the queues take its place

  // 3. parents, and the wave's queue of kept links
  uint32_t* par = L.u.w.par;
  uint16_t* queue = L.u.w.queue[seg];
  {
    const uint32_t n0 = row_node<QK>(16u * (uint32_t)seg, (uint32_t)lane);
    // a segment that continues a run hangs on the voxel before it
    uint32_t v = QK == Q_BLOCK8 ? n0 - 3u : n0 - 1u;
    constexpr int ST = QK == Q_BLOCK8 ? 2 : 4;  // consecutive nodes
#pragma unroll
    for (int k = 0; k < 16; k += ST) {
      uint32_t w[ST];
#pragma unroll
      for (int i = 0; i < ST; i++) {
        if (k + i == 1) v = (S & 1u) ? v : n0;
        v = ((S >> (k + i)) & 1u) ? seg_node<QK>(n0, (uint32_t)(k + i)) : v;
        w[i] = v;
      }
      uint32_t* d = static_cast<uint32_t*>(__builtin_assume_aligned(par + seg_node<QK>(n0, (uint32_t)k), 4 * ST));
#pragma unroll
      for (int i = 0; i < ST; i++) d[i] = w[i];
    }
  }
  constexpr int NWORD = FACE ? 1 : NB == 8 ? 2 : NB == 18 ? 4 : 6;
  const uint32_t pos0 = (uint32_t)(lane * G::TX + 16 * seg);
  uint32_t W[6];  // two relations each: 2 i in the low half, 2 i + 1 in the high half
  uint32_t cnt = U[R_A];
#pragma unroll
  for (int i = 0; i < 6; i++) {
    W[i] = i < NWORD ? (U[2 * i] | (U[2 * i + 1] << 16)) : 0u;
    if (i < NWORD) cnt += (uint32_t)__popc(W[i]);
  }
  // writes this lane's links from slot q on, two words per loop
  auto emit = [&](uint16_t* q, uint32_t ua) {
    if (first && ua) *q++ = (uint16_t)(pos0 | ((uint32_t)R_A << 12));
#pragma unroll
    for (int i = 0; i < NWORD; i += 2) {
      uint32_t m = W[i], m2 = i + 1 < NWORD ? W[i + 1] : 0u;
      uint32_t code = pos0 + ((uint32_t)(2 * i) << 12);
      while (m | m2) {
        if (m == 0) {
          m = m2;
          m2 = 0;
          code += 2u << 12;
        }
        const uint32_t k = (uint32_t)__builtin_ctz(m);
        m &= m - 1u;
        *q++ = (uint16_t)(code + (k & 15u) + ((k >> 4) << 12));
      }
    }
  };
  // the n queued links of the wave, one per lane; those that leave the tile are
  // appended to its list if that is asked for
  uint16_t* REQt = reinterpret_cast<uint16_t*>(p.REQ) + slot * p.reqcap;
  constexpr bool MASKS = row_masks(MODE == M_CONT, NB);
  auto drain = [&](uint32_t n, bool append) {
    for (uint32_t i0 = 0; i0 < n; i0 += 64) {
      const uint32_t i = i0 + (uint32_t)lane;
      bool out = false;
      uint32_t e = 0;
      if (i < n) {
        e = queue[i];
        int dx, dy, dz;
        rel_decode(e >> 12, dx, dy, dz);
        const uint32_t ps = e & 0xFFFu;
        const int x = (int)(ps & 63u) + dx, y = (int)((ps >> 6) & (G::TY - 1)) + dy, z = (int)(ps / (64u * G::TY)) + dz;
        out = x < 0 || x >= G::TX || y < 0 || y >= G::TY || z < 0;
        if (!out)
          runion(par, row_node<QK>(ps & 63u, ps >> 6), row_node<QK>((uint32_t)x, (uint32_t)(y + G::TY * z)));
      }
      const uint64_t m = wave_ballot(out && append);
      if (m) {
        uint32_t b = 0;
        if (lane == 0) b = atomicAdd(&L.nreq, (uint32_t)__builtin_popcountll(m));
        b = (uint32_t)__builtin_amdgcn_readfirstlane((int)b);
        if (out) REQt[b + mbcnt64(m)] = (uint16_t)e;
      }
    }
  };
  const uint32_t incl = wave_incl_add(cnt);
  const uint32_t total = wave_lane63(incl);
  if (total <= RQCAP) emit(queue + (incl - cnt), U[R_A]);
  if constexpr (MASKS) {
    uint32_t bound = total;
    if (total > RQCAP) {  // the links that leave the tile
      bound = U[R_A];
#pragma unroll
      for (int i = 0; i < 2 * NWORD; i++) {
        constexpr uint32_t ALL = 0xFFFFu;
        const Off o = rel_off(i);
        const uint32_t face = (o.dz < 0 && lz == 0) || (o.dy < 0 && ly == 0) || (o.dy > 0 && ly == G::TY - 1) ? ALL : 0u;
        const uint32_t side = (o.dx < 0 && first ? 1u : 0u) | (o.dx > 0 && seg == 3 ? 0x8000u : 0u);
        bound += (uint32_t)__popc((W[i >> 1] >> (16 * (i & 1))) & (face | side));
      }
      bound = SLOW | wave_lane63(wave_incl_add(bound));
    }
    if (lane == 0) L.ne0[seg] = (uint16_t)bound;
  }
  __syncthreads();

  // 4. unions and requests
  // segments whose links are stored as masks: none unless the list may be too short
  auto masked_segments = [&]() -> uint32_t {
    uint32_t sum = 0, m = 0;
#pragma unroll
    for (int w = 0; w < 4; w++) {
      const uint32_t b = L.ne0[w];
      sum += b & (SLOW - 1u);
      m |= b & SLOW ? 1u << w : 0u;
    }
    return sum <= 64u << G::jlog(p.jl) ? 0u : m;
  };
  if (total <= RQCAP) {
    drain(total, true);
  } else {
    // more links than the queue holds: one relation at a time
    uint32_t keep[6];
#pragma unroll
    for (int i = 0; i < 6; i++) keep[i] = W[i];
    const uint32_t masked = MASKS ? masked_segments() : 0u;
    if (MASKS && masked) {
      // link masks: 13 bits per voxel of the segment, relation r in bit r, row by
      // row; the first such segment at the end of the tile's entries, the next
      // before it.  The list needs no more than the other segments' places.
      const uint32_t at = (64u << G::jlog(p.jl)) - 1024u * (uint32_t)__popc(masked & ((2u << seg) - 1u));
      uint16_t* d = REQt + at + 16 * lane;
#pragma unroll 1
      for (int k = 0; k < 16; k++) {
        uint32_t m = ((U[R_A] >> k) & 1u) << R_A;
#pragma unroll
        for (int i = 0; i < NWORD; i++)
          m |= (((keep[i] >> k) & 1u) << (2 * i)) | (((keep[i] >> (16 + k)) & 1u) << (2 * i + 1));
        d[k] = (uint16_t)m;
      }
    }
#pragma unroll 1
    for (int r = 0; r <= 2 * NWORD; r++) {
      uint32_t c = 0;
#pragma unroll
      for (int i = 0; i < 6; i++) {
        W[i] = (r >> 1) == i ? (keep[i] & ((r & 1) ? 0xFFFF0000u : 0xFFFFu)) : 0u;
        c += (uint32_t)__popc(W[i]);
      }
      const uint32_t ua = r == 2 * NWORD ? U[R_A] : 0u;
      c += ua;
      const uint32_t inc = wave_incl_add(c);
      emit(queue + (inc - c), ua);
      wave_order();
      drain(wave_lane63(inc), masked == 0);
      wave_order();
    }
  }
  // the wave's queue is dead: its place takes the segment bits by row
  wave_order();
  uint32_t* segbits = reinterpret_cast<uint32_t*>(queue);
  segbits[lane] = S | (F << 16);
  my_epl = wave_lane63(wave_incl_add(my_epl));
  my_prov = wave_lane63(wave_incl_add(my_prov));
  if (lane == 0) {
    L.red_epl[seg] = my_epl;
    L.red_prov[seg] = my_prov;
    L.rows[seg] = fgrows;
  }
  __syncthreads();

  // 5. roots.  From here thread t has segment t & 3 of row t >> 2, so its
  //    outputs are in raster order over the workgroup.  Heads (run starts and
  //    the first voxel of a segment) take their root as parent; all walks
  //    only read otherwise.
  const int hrow = t >> 2, hseg = t & 3;
  uint32_t* qs = reinterpret_cast<uint32_t*>(L.u.w.queue[hseg]);
  const uint32_t sf = qs[hrow];
  const uint32_t hS = sf & 0xFFFFu, hF = sf >> 16;
  const uint32_t H = hS | (hF & 1u);
  const uint32_t h0 = row_node<QK>(16u * (uint32_t)hseg, (uint32_t)hrow);
  uint32_t rb = 0;  // roots of this segment
  for (uint32_t m = H; m; m &= m - 1u) {
    const uint32_t k = (uint32_t)__builtin_ctz(m), n = seg_node<QK>(h0, k);
    const uint32_t r = rfind_ro(par, n);
    if (r == n) rb |= 1u << k;
    else lstore(par + n, r);
  }
  const uint32_t nr = (uint32_t)__popc(rb);
  const uint32_t rincl = wave_incl_add(nr);
  if (lane == 63) L.wtot[t >> 6] = rincl;
  __syncthreads();
  uint32_t rbase = 0, R = 0;
#pragma unroll
  for (int w = 0; w < 4; w++) {
    if (w < (t >> 6)) rbase += L.wtot[w];
    R += L.wtot[w];
  }
  rbase += rincl - nr;

  // 6. roots take 1 + their rank as parent and go to the global forest.  Keys
  //    in 32-bit arithmetic (below 2^32; intermediate wraps cancel).  A
  //    segment's keys are consecutive, so its root marks are one or two words.
  const uint32_t root0 = tile_root0<G>(sx, sy, sz, tx, ty, tz, keybase);
  const int hx = x0 + 16 * hseg, hy = y0 + (hrow & (G::TY - 1)), hz = z0 + hrow / G::TY;
  const uint32_t key0 =
    QK == Q_BLOCK8 ? 0u : (uint32_t)hx + (uint32_t)sx * ((uint32_t)hy + (uint32_t)sy * (uint32_t)hz) + keybase;
  uint32_t rk = rbase;
  for (uint32_t m = rb; m; m &= m - 1u) {
    const uint32_t k = (uint32_t)__builtin_ctz(m);
    uint32_t key = key0 + k;
    if (QK == Q_BLOCK8) {
      key = gkey<QK>(hx + (int)k, hy, 0, sx, sy, p.osx) + keybase;
      atomicOr(p.bits + (key >> 5), 1u << (key & 31));
    }
    p.GP[root0 + rk] = make_uint2(root0 + rk, key);
    par[seg_node<QK>(h0, k)] = ++rk;
  }
  if (QK != Q_BLOCK8) {
    if ((sx & 15) == 0) {
      // every segment is a half-word of the bitmask that no other tile holds:
      // stored whether or not it has roots, so nothing clears the bitmask
      // before; the volume's last half-word clears the rest of its word
      if (hx < sx && hy < sy && hz < sz) {
        uint16_t* half = reinterpret_cast<uint16_t*>(p.bits) + (key0 >> 4);
        half[0] = (uint16_t)rb;
        if (!((key0 >> 4) & 1u) && hx + 16 == sx && hy + 1 == sy && hz + 1 == sz) half[1] = 0;
      }
    } else if (rb) {
      const uint32_t sh = key0 & 31u, lo = rb << sh, hi = sh > 16u ? rb >> (32u - sh) : 0u;
      if (lo) atomicOr(p.bits + (key0 >> 5), lo);
      if (hi) atomicOr(p.bits + (key0 >> 5) + 1, hi);
    }
  }
  __syncthreads();

  // 7. the other heads take their root's, and the outputs
  for (uint32_t m = H & ~rb; m; m &= m - 1u) {
    const uint32_t n = seg_node<QK>(h0, (uint32_t)__builtin_ctz(m));
    par[n] = par[par[n]];
  }
  {
    uint32_t j = 0, pk[8];
    uint32_t v[16];
    constexpr int ST = QK == Q_BLOCK8 ? 2 : 4;
#pragma unroll
    for (int k = 0; k < 16; k += ST) {
      const uint32_t* q =
        static_cast<const uint32_t*>(__builtin_assume_aligned(par + seg_node<QK>(h0, (uint32_t)k), 4 * ST));
#pragma unroll
      for (int i = 0; i < ST; i++) v[k + i] = q[i];
    }
#pragma unroll
    for (int k = 0; k < 16; k += 4) {
      uint32_t o[4];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        j = ((H >> (k + i)) & 1u) ? v[k + i] : j;
        o[i] = ((hF >> (k + i)) & 1u) ? j : 0u;
      }
      pk[k / 2] = o[0] | (o[1] << 16);
      pk[k / 2 + 1] = o[2] | (o[3] << 16);
    }
    uint4* o8 = reinterpret_cast<uint4*>(p.J8 + slot * (2 * G::TV)) + t;
    uint4* o16 = reinterpret_cast<uint4*>(p.J16 + slot * G::TV) + 2 * t;
    bool stored = true;
    if constexpr (G::NARROW) {
      const uint32_t at = ((uint32_t)hrow << p.jl) + 16u * (uint32_t)hseg;
      o8 = reinterpret_cast<uint4*>(p.J8 + (slot << (7 + p.jl)) + at);
      o16 = reinterpret_cast<uint4*>(p.J16 + (slot << (6 + p.jl)) + at);
      stored = 16 * hseg < 1 << p.jl;  // else columns that the volume does not have
    }
    if (R <= 255) {
      uint32_t b[4];
#pragma unroll
      for (int i = 0; i < 4; i++) b[i] = __builtin_amdgcn_perm(pk[2 * i + 1], pk[2 * i], 0x06040200u);
      if (stored) *o8 = make_uint4(b[0], b[1], b[2], b[3]);
    } else if (stored) {
      o16[0] = make_uint4(pk[0], pk[1], pk[2], pk[3]);
      o16[1] = make_uint4(pk[4], pk[5], pk[6], pk[7]);
    }
  }
  if (t == 0) {
    uint32_t e = 0, pv = 0;
    uint64_t rows = 0;
    for (int w = 0; w < 4; w++) {
      e += L.red_epl[w];
      pv += L.red_prov[w];
      rows |= L.rows[w];
    }
    long long f = 0x7FFFFFFFFFFFFFFFll, l = -1;
    if (rows) {
      const int fl = __builtin_ctzll(rows), ll = 63 - __builtin_clzll(rows);
      f = (y0 + fl % G::TY) + sy * (z0 + fl / G::TY);
      l = (y0 + ll % G::TY) + sy * (z0 + ll / G::TY);
    }
    p.TR[slot] = R;
    p.TQ[slot] = L.nreq;
    if constexpr (MODE == M_CONT && IS3D) {
      // 6-connected volumes of a batch with others say it too
      const int n = 64 << G::jlog(p.jl);
      if (MASKS || p.reqcap > n) REQt[n] = (uint16_t)(MASKS ? masked_segments() : 0u);
    }
    TileCnt c;
    c.epl = e;
    c.prov = pv;
    c.first_row = f;
    c.last_row = l;
    p.tcnt[slot] = c;
  }
}

// Does one label gather much of a volume?  64 voxels at uneven distances, each
// compared with six others: 192 pairs, of which a label that holds the share s
// of the volume makes 192 s^2 equal (mask at p = 0.2: 8, 0.3: 17), the labels
// of a segmentation none.  By one wave of the launch's first workgroup, which
// runs beside thousands of others.
constexpr int EQUAL_PAIRS = 5;
template <class T>
__device__ inline void label_spread(const T* in, uint64_t n, uint32_t* spread) {
  const uint32_t lane = threadIdx.x & 63;
  const uint64_t step = n >> 6;  // at least one voxel a tile
  const T v = in[lane * step + (((uint64_t)(lane * 0x9E3779B1u) * step) >> 32)];
  uint64_t bits = 0;
  __builtin_memcpy(&bits, &v, sizeof(T));
  int twice = 0;  // every pair is seen from both ends
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const uint64_t w = __shfl_xor((unsigned long long)bits, o);
    twice += __builtin_popcountll(wave_ballot(v != T(0) && w == bits));
  }
  if (lane == 0) *spread = twice < 2 * EQUAL_PAIRS ? 1u : 0u;
}

// Waves per SIMD the row kernel is compiled for: what the LDS of one tile
// admits (6 workgroups of 4 waves per CU; 3 for continuous 8-byte voxels),
// less one for 8-byte voxels staged by halves, which hold a tile's share in
// registers meanwhile.
template <class T, int MODE>
__host__ __device__ constexpr int rows_waves() {
  return sizeof(T) < 8 || MODE == M_BINARY ? 6 : MODE == M_CONT ? 3 : 5;
}

template <class T, int MODE, int NB, class G>
__global__ __launch_bounds__(G::NT, (rows_waves<T, MODE>())) void k_rows_local(LocalParams p) {
  __shared__ RowLds<T, MODE, G> L;
  const int64_t tile = xcd_tile(blockIdx.x, p.ntiles);
  rows_tile<T, MODE, NB, G, Q_NONE>(p, static_cast<const T*>(p.in), p.sx, p.sy, p.sz, p.ntx, p.nty, p.dxy, p.dx, tile,
                                    tile, 0u, L);
  if (MODE == M_MULTI && blockIdx.x == 0 && threadIdx.x < 64 && p.spread)
    label_spread(static_cast<const T*>(p.in), (uint64_t)(p.sx * p.sy * p.sz), p.spread);
}

// Single planes of at least 64 rows.
template <class T, int MODE, int NB, int QK, class G>
__global__ __launch_bounds__(G::NT, (rows_waves<T, MODE>())) void k_rows_plane(LocalParams p) {
  __shared__ RowLds<T, MODE, G> L;
  const int64_t tile = xcd_tile(blockIdx.x, p.ntiles);
  rows_tile<T, MODE, NB, G, QK>(p, static_cast<const T*>(p.in), p.sx, p.sy, 1, p.ntx, p.nty, p.dxy, p.dx, tile, tile,
                                0u, L);
  if (MODE == M_MULTI && blockIdx.x == 0 && threadIdx.x < 64 && p.spread)
    label_spread(static_cast<const T*>(p.in), (uint64_t)(p.sx * p.sy), p.spread);
}

// Batch: tiles [gtile0, gtile0 + gtiles) of volumes of connectivity NB; each
// workgroup reads its volume's table entry.
template <class T, int MODE, int NB, class G>
__global__ __launch_bounds__(G::NT, (rows_waves<T, MODE>())) void k_rows_local_batch(LocalParams p,
                                                                                    const BatchVol* vols,
                                                                                    const uint32_t* vix,
                                                                                    int64_t gtile0, int64_t gtiles) {
  __shared__ RowLds<T, MODE, G> L;
  const int64_t slot = gtile0 + xcd_tile(blockIdx.x, gtiles);
  const BatchVol& v = vols[vix[slot]];
  rows_tile<T, MODE, NB, G, Q_NONE>(p, static_cast<const T*>(v.in), v.sx, v.sy, v.sz, v.ntx, v.nty, v.dxy, v.dx,
                                    slot - v.tile0, slot, v.key0, L);
}

hipError_t launch_rows_multi(int dt, int nb, const LocalParams& p, hipStream_t s);
hipError_t launch_rows_binary(int dt, int nb, const LocalParams& p, hipStream_t s);
// Planes on the row tiles: every mode and numbering but continuous 2D-8
// (Q_CONT8), whose links depend on the plane's extremes.
hipError_t launch_rows_plane_multi(int dt, int nb, int qk, const LocalParams& p, hipStream_t s);
hipError_t launch_rows_plane_binary(int dt, int nb, int qk, const LocalParams& p, hipStream_t s);
hipError_t launch_rows_plane_cont(int dt, int nb, int qk, const LocalParams& p, hipStream_t s);
hipError_t launch_rows_cont(int dt, int nb, const LocalParams& p, hipStream_t s);
hipError_t launch_rows_batch_cont(int dt, int nb, const LocalParams& p, const BatchVol* vols, const uint32_t* vix,
                                  int64_t gtile0, int64_t gtiles, hipStream_t s);
hipError_t launch_rows_batch_multi(int dt, int nb, const LocalParams& p, const BatchVol* vols, const uint32_t* vix,
                                   int64_t gtile0, int64_t gtiles, hipStream_t s);
hipError_t launch_rows_batch_binary(int dt, int nb, const LocalParams& p, const BatchVol* vols, const uint32_t* vix,
                                    int64_t gtile0, int64_t gtiles, hipStream_t s);

template <int MODE>
hipError_t launch_rows_mode(int dt, int nb, const LocalParams& p, hipStream_t s) {
  const dim3 grid((unsigned)p.ntiles), block(GeoR::NT);
#define CC3D_R(T, NB)                                                                            \
  if (p.jl < 6) hipLaunchKernelGGL((k_rows_local<T, MODE, NB, GeoRN>), grid, block, 0, s, p);    \
  else hipLaunchKernelGGL((k_rows_local<T, MODE, NB, GeoR>), grid, block, 0, s, p)
#define CC3D_RNB(T)                       \
  switch (nb) {                           \
    case 26: CC3D_R(T, 26); break;        \
    case 18: CC3D_R(T, 18); break;        \
    case 6: CC3D_R(T, 6); break;          \
    default: return hipErrorInvalidValue; \
  }
  switch (dt) {
    case DT_U8: CC3D_RNB(uint8_t); break;
    case DT_U16: CC3D_RNB(uint16_t); break;
    case DT_U32: CC3D_RNB(uint32_t); break;
    case DT_U64: CC3D_RNB(uint64_t); break;
    case DT_F32: CC3D_RNB(float); break;
    case DT_F64: CC3D_RNB(double); break;
    default: return hipErrorInvalidValue;
  }
#undef CC3D_RNB
#undef CC3D_R
  return hipGetLastError();
}

template <int MODE>
hipError_t launch_rows_plane_mode(int dt, int nb, int qk, const LocalParams& p, hipStream_t s) {
  const dim3 grid((unsigned)p.ntiles), block(GeoP::NT);
#define CC3D_R(T, NB, QK)                                                                        \
  if (p.jl < 6) hipLaunchKernelGGL((k_rows_plane<T, MODE, NB, QK, GeoPN>), grid, block, 0, s, p); \
  else hipLaunchKernelGGL((k_rows_plane<T, MODE, NB, QK, GeoP>), grid, block, 0, s, p)
#define CC3D_RNB(T)                                                                            \
  if (nb == 8 && qk == Q_BLOCK8 && MODE == M_BINARY) {                                         \
    CC3D_R(T, 8, (MODE == M_BINARY ? Q_BLOCK8 : Q_NONE));                                      \
  } else if (nb == 4 && qk == Q_BIN4 && MODE == M_BINARY) {                                    \
    CC3D_R(T, 4, (MODE == M_BINARY ? Q_BIN4 : Q_NONE));                                        \
  } else if (nb == 8 && qk == Q_NONE) {                                                        \
    CC3D_R(T, 8, Q_NONE);                                                                      \
  } else if (nb == 4 && qk == Q_NONE) {                                                        \
    CC3D_R(T, 4, Q_NONE);                                                                      \
  } else {                                                                                     \
    return hipErrorInvalidValue;                                                               \
  }
  switch (dt) {
    case DT_U8: CC3D_RNB(uint8_t); break;
    case DT_U16: CC3D_RNB(uint16_t); break;
    case DT_U32: CC3D_RNB(uint32_t); break;
    case DT_U64: CC3D_RNB(uint64_t); break;
    case DT_F32: CC3D_RNB(float); break;
    case DT_F64: CC3D_RNB(double); break;
    default: return hipErrorInvalidValue;
  }
#undef CC3D_RNB
#undef CC3D_R
  return hipGetLastError();
}

template <int MODE>
hipError_t launch_rows_batch_mode(int dt, int nb, const LocalParams& p, const BatchVol* vols, const uint32_t* vix,
                                  int64_t gtile0, int64_t gtiles, hipStream_t s) {
  const dim3 grid((unsigned)gtiles), block(GeoR::NT);
#define CC3D_R(T, NB)                                                                                              \
  if (p.jl < 6)                                                                                                    \
    hipLaunchKernelGGL((k_rows_local_batch<T, MODE, NB, GeoRN>), grid, block, 0, s, p, vols, vix, gtile0, gtiles); \
  else hipLaunchKernelGGL((k_rows_local_batch<T, MODE, NB, GeoR>), grid, block, 0, s, p, vols, vix, gtile0, gtiles)
#define CC3D_RNB(T)                       \
  switch (nb) {                           \
    case 26: CC3D_R(T, 26); break;        \
    case 18: CC3D_R(T, 18); break;        \
    case 6: CC3D_R(T, 6); break;          \
    default: return hipErrorInvalidValue; \
  }
  switch (dt) {
    case DT_U8: CC3D_RNB(uint8_t); break;
    case DT_U16: CC3D_RNB(uint16_t); break;
    case DT_U32: CC3D_RNB(uint32_t); break;
    case DT_U64: CC3D_RNB(uint64_t); break;
    case DT_F32: CC3D_RNB(float); break;
    case DT_F64: CC3D_RNB(double); break;
    default: return hipErrorInvalidValue;
  }
#undef CC3D_RNB
#undef CC3D_R
  return hipGetLastError();
}

}  // namespace cc3d_amd
