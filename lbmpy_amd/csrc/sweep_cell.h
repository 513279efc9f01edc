// Per-cell pieces of the stream-collide sweep shared by every kernel that updates cells: the
// single-domain sweeps (sweep.hip) and the batched ensemble sweep (batch.hip).  Both call
// collide_cell / sweep_cell, so a cell updated in a batch runs exactly the instructions of the
// same cell updated on its own.
#pragma once
#include <type_traits>

#include "lbm_common.h"
#include "collide_moment.h"
#include "collide_cumulant.h"
#include "collide_central.h"

namespace lbm355 {

template <class S, int FAM, class TC>
struct Collider;

template <class S, class TC>
struct Collider<S, LBM355_FAMILY_MOMENT, TC> {
  static constexpr bool deviation_form = false;
  template <bool NEQ>
  static __device__ __forceinline__ void run(TC (&f)[S::Q], const SweepArgs<TC>& a, int64_t o, TC& rho, TC (&u)[3],
                                             CellExtras<TC>&) {
    collide_moment<S, TC>(f, a, o, rho, u);
  }
};

// kernel-variant family code of the cumulant sweep with the learned closure (internal, not in the ABI)
constexpr int FAMILY_CUMULANT_LEARNED = 0x102;

template <class TC>
struct Collider<D3Q27, FAMILY_CUMULANT_LEARNED, TC> {
  static constexpr bool deviation_form = true;
  template <bool NEQ>
  static __device__ __forceinline__ void run(TC (&f)[27], const SweepArgs<TC>& a, int64_t, TC& rho, TC (&u)[3],
                                             CellExtras<TC>& ex) {
    collide_cumulant_d3q27<TC, true, false, NEQ>(f, a, rho, u, ex);
  }
};

// the learned-closure sweep when every cumulant of order >= 3 relaxes with rate 1
constexpr int FAMILY_CUMULANT_LEARNED_EQ3 = 0x106;

template <class TC>
struct Collider<D3Q27, FAMILY_CUMULANT_LEARNED_EQ3, TC> {
  static constexpr bool deviation_form = true;
  template <bool NEQ>
  static __device__ __forceinline__ void run(TC (&f)[27], const SweepArgs<TC>& a, int64_t, TC& rho, TC (&u)[3],
                                             CellExtras<TC>& ex) {
    collide_cumulant_d3q27<TC, true, false, NEQ, false, true>(f, a, rho, u, ex);
  }
};

// kernel-variant family code of the cumulant sweep with the Galilean / fourth-order corrections (internal)
constexpr int FAMILY_CUMULANT_CORRECTED = 0x103;

template <class TC>
struct Collider<D3Q27, FAMILY_CUMULANT_CORRECTED, TC> {
  static constexpr bool deviation_form = true;
  template <bool NEQ>
  static __device__ __forceinline__ void run(TC (&f)[27], const SweepArgs<TC>& a, int64_t, TC& rho, TC (&u)[3],
                                             CellExtras<TC>& ex) {
    collide_cumulant_d3q27<TC, false, true, NEQ>(f, a, rho, u, ex);
  }
};

// kernel-variant family code of the cumulant sweep for cumulant sets other than the default polynomial one
constexpr int FAMILY_CUMULANT_GENERAL = 0x104;

template <class TC>
struct Collider<D3Q27, FAMILY_CUMULANT_GENERAL, TC> {
  static constexpr bool deviation_form = true;
  template <bool NEQ>
  static __device__ __forceinline__ void run(TC (&f)[27], const SweepArgs<TC>& a, int64_t, TC& rho, TC (&u)[3],
                                             CellExtras<TC>& ex) {
    collide_cumulant_d3q27<TC, false, false, NEQ, true>(f, a, rho, u, ex);
  }
};

// kernel-variant family code of the cumulant sweep when every cumulant of order >= 3 relaxes with rate 1
constexpr int FAMILY_CUMULANT_EQ3 = 0x105;

template <class TC>
struct Collider<D3Q27, FAMILY_CUMULANT_EQ3, TC> {
  static constexpr bool deviation_form = true;
  template <bool NEQ>
  static __device__ __forceinline__ void run(TC (&f)[27], const SweepArgs<TC>& a, int64_t, TC& rho, TC (&u)[3],
                                             CellExtras<TC>& ex) {
    collide_cumulant_d3q27<TC, false, false, NEQ, false, true>(f, a, rho, u, ex);
  }
};

template <class TC>
struct Collider<D3Q27, LBM355_FAMILY_CUMULANT, TC> {
  static constexpr bool deviation_form = true;
  template <bool NEQ>
  static __device__ __forceinline__ void run(TC (&f)[27], const SweepArgs<TC>& a, int64_t, TC& rho, TC (&u)[3],
                                             CellExtras<TC>& ex) {
    collide_cumulant_d3q27<TC, false, false, NEQ>(f, a, rho, u, ex);
  }
};

// number of directions with a non-zero x component (those are shifted through LDS)
template <class S>
__host__ __device__ constexpr int n_xshift() {
  int n = 0;
  for (int i = 0; i < S::Q; ++i) n += S::c[i][0] != 0;
  return n;
}

// Non-temporal accesses for aligned, streamed-once data (each PDF is read and written exactly
// once per sweep); misaligned accesses (x +- 1, or all of them, see AccessMode) keep the default policy so that
// the partially used cache lines are served from cache to the neighbouring wavefront.
template <class TS, class TC>
__device__ __forceinline__ TC load_nt(const TS* p) {
  return (TC)__builtin_nontemporal_load(p);
}
template <class TS, class TC>
__device__ __forceinline__ void store_nt(TS* p, TC v) {
  __builtin_nontemporal_store((TS)v, p);
}

// ROWLDS: the block spans one whole row and x is periodic (blockDim.x == nx).  The +-1
// x-shifts of pull / AA-odd streaming are then done in LDS, so every global load and store
// is an aligned, contiguous, non-temporal 64-lane access:
//   read : tile[j][x] = row(y - c_y, z - c_z)[x];  f_i(x) = tile[j][(x - c_x) mod nx]
//   write: tile[j][x] = f_i(x);  row(y + c_y, z + c_z)[x] = tile[j][(x - c_x) mod nx]
template <class S, class TC>
struct Collider<S, LBM355_FAMILY_CENTRAL, TC> {
  static constexpr bool deviation_form = true;
  template <bool NEQ>
  static __device__ __forceinline__ void run(TC (&f)[S::Q], const SweepArgs<TC>& a, int64_t, TC& rho, TC (&u)[3],
                                             CellExtras<TC>&) {
    collide_central<S, TC>(f, a, rho, u);
  }
};

// 32-bit integer hash (xorshift-multiply): mixes a cell index with a launch seed
__device__ __forceinline__ uint32_t mix32(uint32_t v) {
  v ^= v >> 16;
  v *= 0x7FEB352Du;
  v ^= v >> 15;
  v *= 0x846CA68Bu;
  v ^= v >> 16;
  return v;
}

// Stochastic rounding of a cell's populations to FP16 values (kept in TC, so that the store's conversion is
// exact): each value goes to one of its two neighbouring FP16 numbers with probability proportional to its
// closeness, gfx950's v_cvt_sr_f16_f32, which compares the high bits of its random operand with the dropped
// mantissa bits (measured: a value 1/8, 2/8, ... 7/8 of an FP16 ulp above an FP16 number rounds up with those
// frequencies when bits 19..31 of the operand are uniform, and never when only bits 0..12 vary).  The operand of
// direction i is the low 24 bits of the cell's hash times an odd 24-bit constant of i (one full-rate v_mul_u32_u24),
// whose high bits are well mixed.
template <class S, class TC>
__device__ __forceinline__ void round_stochastic_f16(TC (&f)[S::Q], uint32_t seed, int x, int y, int z, int nx,
                                                     int ny) {
  typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
  const uint32_t cell = (uint32_t)x + (uint32_t)nx * ((uint32_t)y + (uint32_t)ny * (uint32_t)z);
  const uint32_t h = mix32(cell * 0x9E3779B9u + seed);
#pragma unroll
  for (int i = 0; i < S::Q; ++i) {
    const uint32_t k = (0x5BD1E9u + 0x3C6EF2u * (uint32_t)i) & 0xFFFFFFu;   // odd (bit 0 of both terms: 1, 0)
    const uint32_t r = __umul24(h, k);
    const half2_t zero = {0, 0};
    const half2_t v = __builtin_amdgcn_cvt_sr_f16_f32(zero, (float)f[i], r, false);
    f[i] = (TC)(float)v[0];
  }
}

// Collision of one cell's populations plus the optional per-cell outputs (density, velocity, the Smagorinsky
// rate and eddy viscosity).  Shared by every sweep kernel (single domain, row-LDS and batched), so all of them
// run the same arithmetic.  TS is the storage type: FP16 storage may round stochastically.
template <class S, int FAM, class TC, class TS = TC>
__device__ __forceinline__ void collide_cell(TC (&f)[S::Q], const SweepArgs<TC>& a, int x, int y, int z) {
  constexpr int Q = S::Q, D = S::D;
  const bool absolute = !(a.flags & LBM355_FLAG_ZERO_CENTERED);
  if (Collider<S, FAM, TC>::deviation_form && absolute) {
#pragma unroll
    for (int i = 0; i < Q; ++i) f[i] -= TC(weight<S>(i));
  }
  // offset of the cell in the optional per-cell fields
  const int64_t o = (int64_t)(x + a.g) + (int64_t)(y + a.g) * a.osy + (D == 3 ? (int64_t)(z + a.g) * a.osz : 0);
  TC rho, u[3];
  CellExtras<TC> ex = {a.omega_shear, TC(0)};
  // the cumulant collision transforms f - f_eq for FP32 storage with FP32 arithmetic (collide_cumulant.h)
  constexpr bool NEQ = std::is_same<TC, float>::value && std::is_same<TS, float>::value;
  Collider<S, FAM, TC>::template run<NEQ>(f, a, o, rho, u, ex);
  if (Collider<S, FAM, TC>::deviation_form && absolute) {
#pragma unroll
    for (int i = 0; i < Q; ++i) f[i] += TC(weight<S>(i));
  }
  if (a.rho_out) a.rho_out[o] = rho;
  if (a.u_out) {
#pragma unroll
    for (int d = 0; d < D; ++d) a.u_out[o + d * a.osc] = u[d];
  }
  if (a.omega_out) a.omega_out[o] = ex.omega_sgs;
  if (a.nut_out) a.nut_out[o] = a.nut_scale * ex.omega_sgs * ex.pi;
  if constexpr (std::is_same<TS, _Float16>::value) {
    if (a.flags & LBM355_FLAG_STOCHASTIC_ROUNDING) round_stochastic_f16<S, TC>(f, a.seed, x, y, z, a.nx, a.ny);
  }
}

// Loads and stores of element `off` (0 <= off < 2^31) of a population plane.  With 2-byte storage the byte offset
// fits in 32 bits (a plane holds < 2^31 elements): the accesses take the plane's base from scalar registers and one
// 32-bit vector offset for every plane.  They are global accesses: the base in a buffer descriptor has to lie on a
// dword, which every other plane of an odd number of elements does not, and near walls, where the lanes of a wavefront
// differ in plane, each descriptor takes a pass of its own (D3Q27 cumulant 250x200x180 AA: 173 us with descriptors,
// 170 without).  Wider storage uses ordinary pointers.  NT: non-temporal.
template <class TS>
__device__ __forceinline__ TS* plane_at(TS* plane, int off) {
  using Byte = std::conditional_t<std::is_const<TS>::value, const char, char>;
  if constexpr (sizeof(TS) == 2) return reinterpret_cast<TS*>(reinterpret_cast<Byte*>(plane) + (uint32_t)off * 2u);
  return plane + off;
}

template <class TS, class TC, bool NT>
__device__ __forceinline__ TC plane_load(const TS* plane, int off) {
  const TS* p = plane_at(plane, off);
  return NT ? load_nt<TS, TC>(p) : load_as<TS, TC>(p);
}
template <class TS, class TC, bool NT>
__device__ __forceinline__ void plane_store(TS* plane, int off, TC value) {
  TS* p = plane_at(plane, off);
  if (NT)
    store_nt<TS, TC>(p, value);
  else
    store_as<TS, TC>(p, value);
}

// One cell of the sweep with direct (non-LDS) addressing: load with streaming, collide, store.
// With WALLS, only cells next to a NoSlip face take the bounce-back addressing; the test is per cell and
// the wall-free addressing is the same code as without WALLS, so interior cells pay nothing for walls.
// NT: the accesses at the cell itself start on cache lines and are non-temporal.
template <class S, int FAM, int PAT, bool WALLS, bool NT, class TS, class TC>
__device__ __forceinline__ void sweep_cell(const SweepArgs<TC>& a, int x, int y, int z) {
  constexpr int Q = S::Q, D = S::D;
  const AxisNb ax = axis_neighbours(x, a.nx, a.g, a.face[0]);
  const AxisNb ay = axis_neighbours(y, a.ny, a.g, a.face[1]);
  AxisNb az = {0, 0, false, false};
  if (D == 3) az = axis_neighbours(z, a.nz, a.g, a.face[2]);
  // in-plane element offsets of the 3 x positions, 3 rows and 3 planes around the cell
  const int sy = (int)a.sy, sz = (int)a.sz;
  int X[3] = {ax.lo, x + a.g, ax.hi};
  int Y[3] = {ay.lo * sy, (y + a.g) * sy, ay.hi * sy};
  int Z[3] = {D == 3 ? az.lo * sz : 0, D == 3 ? (z + a.g) * sz : 0, D == 3 ? az.hi * sz : 0};
  const int center = X[1] + Y[1] + Z[1];
  const TS* __restrict__ src = reinterpret_cast<const TS*>(a.src);
  TS* __restrict__ dst = reinterpret_cast<TS*>(a.dst);
  const int64_t sq = a.sq;
  const bool near_wall =
      WALLS && (ax.wall_lo || ax.wall_hi || ay.wall_lo || ay.wall_hi || az.wall_lo || az.wall_hi);

  TC f[Q];
  if constexpr (table_pattern(PAT)) {
    // Eso patterns and push: every access from the pattern's table (periodic wrap or ghost layer in X/Y/Z).
    // In place, a cell reads exactly the locations it writes, so one thread per cell needs no synchronisation.
    // With NT, accesses without an x offset are row-aligned and non-temporal.
    constexpr AccessTable<S, PAT> acc{};
#pragma unroll
    for (int i = 0; i < Q; ++i) {
      const Access& t = acc.a[i];
      const TS* p = src + t.rslot * sq + X[1 + t.r[0]] + Y[1 + t.r[1]] + Z[1 + t.r[2]];
      f[i] = NT && t.r[0] == 0 ? load_nt<TS, TC>(p) : load_as<TS, TC>(p);
    }
    collide_cell<S, FAM, TC, TS>(f, a, x, y, z);
#pragma unroll
    for (int i = 0; i < Q; ++i) {
      const Access& t = acc.a[i];
      TS* p = dst + t.wslot * sq + X[1 + t.w[0]] + Y[1 + t.w[1]] + Z[1 + t.w[2]];
      if (NT && t.w[0] == 0)
        store_nt<TS, TC>(p, f[i]);
      else
        store_as<TS, TC>(p, f[i]);
    }
    return;
  }
  // pull reads src[i] at x - c_i; AA odd reads slot inv(i) there.  At a wall the
  // bounce-back value sits in the cell itself: pull slot inv(i), AA odd slot i.
  auto load = [&](auto walls) {
    constexpr bool W = decltype(walls)::value;
#pragma unroll
    for (int i = 0; i < Q; ++i) {
      const int cx = S::c[i][0], cy = S::c[i][1], cz = S::c[i][2];
      const int ii = S::inv[i];
      const int plane = (PAT == LBM355_PULL) ? i : ii;
      const int wplane = (PAT == LBM355_PULL) ? ii : i;
      bool wall = false;
      if (W)
        wall = (cx == 1 && ax.wall_lo) || (cx == -1 && ax.wall_hi) || (cy == 1 && ay.wall_lo) ||
               (cy == -1 && ay.wall_hi) || (cz == 1 && az.wall_lo) || (cz == -1 && az.wall_hi);
      f[i] = wall ? plane_load<TS, TC, false>(src + wplane * sq, center)
                  : plane_load<TS, TC, false>(src + plane * sq, X[1 - cx] + Y[1 - cy] + Z[1 - cz]);
    }
  };
  // AA odd writes f_i to x + c_i slot i; at a wall it is bounced into the cell's slot inv(i)
  auto store = [&](auto walls) {
    constexpr bool W = decltype(walls)::value;
#pragma unroll
    for (int i = 0; i < Q; ++i) {
      const int cx = S::c[i][0], cy = S::c[i][1], cz = S::c[i][2];
      const int ii = S::inv[i];
      bool wall = false;
      if (W)
        wall = (cx == -1 && ax.wall_lo) || (cx == 1 && ax.wall_hi) || (cy == -1 && ay.wall_lo) ||
               (cy == 1 && ay.wall_hi) || (cz == -1 && az.wall_lo) || (cz == 1 && az.wall_hi);
      if (wall)
        plane_store<TS, TC, false>(dst + ii * sq, center, f[i]);
      else
        plane_store<TS, TC, false>(dst + i * sq, X[1 + cx] + Y[1 + cy] + Z[1 + cz], f[i]);
    }
  };

  if (PAT == LBM355_AA_EVEN) {
#pragma unroll
    for (int i = 0; i < Q; ++i) f[i] = plane_load<TS, TC, NT>(src + i * sq, center);
  } else if (near_wall) {
    load(std::true_type{});
  } else {
    load(std::false_type{});
  }

  collide_cell<S, FAM, TC, TS>(f, a, x, y, z);

  // The stores' offsets are worked out again: kept from the loads they take up to 48 registers over the collision, and
  // with them one to three wavefronts per SIMD (D3Q19 FP32 106 -> 78 registers, D3Q27 cumulant FP16 120 -> 72; AA odd
  // D3Q19 TRT FP32 96^3 with walls 32 -> 27 us, FP16 256^3 248 -> 223).
  if constexpr (PAT == LBM355_AA_ODD) {
#pragma unroll
    for (int k = 0; k < 3; ++k) asm("" : "+v"(X[k]), "+v"(Y[k]), "+v"(Z[k]));
  }
  if (PAT == LBM355_PULL) {
#pragma unroll
    for (int i = 0; i < Q; ++i) plane_store<TS, TC, NT>(dst + i * sq, center, f[i]);
  } else if (PAT == LBM355_AA_EVEN) {
#pragma unroll
    for (int i = 0; i < Q; ++i) plane_store<TS, TC, NT>(dst + S::inv[i] * sq, center, f[i]);
  } else if (near_wall) {
    store(std::true_type{});
  } else {
    store(std::false_type{});
  }
}

// How a sweep launch covers the cells and reaches memory:
// ACCESS_ROWS    one block per whole periodic row, x-shifts through LDS, non-temporal accesses (the row kernels);
// ACCESS_WAVES   one thread per cell, rows of whole wavefronts, accesses at the cell itself non-temporal;
// ACCESS_LINES   the same with rows of any length, consecutive in memory;
// ACCESS_CACHED  one thread per cell, regular accesses, one run of blocks per XCD;
// ACCESS_SHARED  the same kernel with short runs, which every other sweep goes backwards.
enum AccessMode {
  ACCESS_ROWS = LBM355_ACCESS_ROWS, ACCESS_WAVES = LBM355_ACCESS_WAVES, ACCESS_LINES = LBM355_ACCESS_LINES,
  ACCESS_CACHED = LBM355_ACCESS_CACHED, ACCESS_SHARED = LBM355_ACCESS_SHARED
};

// The cell of this thread, or false beyond the last cell.  Threads number the cells consecutively over rows and
// planes, so that wavefronts are full whatever nx is; with ACCESS_WAVES, blocks take up to 256 cells of one row, and y
// and z stay in scalar registers (256^3 FP32 AA even: 593 us, 616 us with numbered cells; FP16 storage 315 and 329).
// The block size is an argument: blockDim.x is a load of its own, waited for before the first address.  (The streamed
// rows keep it: 256^3 AA is 0.4% slower without that wait.)
template <int MODE, class TC>
__device__ __forceinline__ bool thread_cell(const SweepArgs<TC>& a, int& x, int& y, int& z) {
  if constexpr (MODE == ACCESS_WAVES) {
    x = blockIdx.x * blockDim.x + threadIdx.x;
    y = blockIdx.y;
    z = blockIdx.z;
    return x < a.nx;
  }
  const uint32_t t = a.order.number(blockIdx.x) * a.block + threadIdx.x;
  const uint32_t r = a.row.quotient(t), p = a.plane.quotient(r);
  x = (int)(t - r * a.row.d);
  y = (int)(r - p * a.plane.d);
  z = (int)p;
  return t < a.row.d * a.plane.d * (uint32_t)a.nz;
}

// Whether every wavefront's accesses at its own cells start on a 128-byte line, so that no two wavefronts share one:
// the cells are consecutive in memory (no ghost layers, no padding), or rows are whole wavefronts on lines of their own.
inline bool starts_lines(const lbm355_sweep_desc* d, const void* src, const void* dst) {
  const int64_t es = d->store_dtype == LBM355_F64 ? 8 : (d->store_dtype == LBM355_F32 ? 4 : 2);
  const bool flat = d->stencil == LBM355_D2Q9;
  const int64_t first = d->ghost_layers * (1 + d->stride_y + (flat ? 0 : d->stride_z)) * es;
  auto line = [](int64_t bytes) { return bytes % 128 == 0; };
  if (!line((int64_t)(uintptr_t)src + first) || !line((int64_t)(uintptr_t)dst + first) || !line(d->stride_q * es))
    return false;
  if (d->ghost_layers == 0 && d->stride_y == d->nx && (flat || d->stride_z == (int64_t)d->nx * d->ny)) return true;
  return d->nx % 64 == 0 && line(d->stride_y * es) && (flat || line(d->stride_z * es));
}

// Launch shape of a sweep, by what the populations' bytes (both arrays of a two-array pattern) fit into and how they lie.
// Times on MI355X, us per launch before (row-mapped blocks, non-temporal accesses wherever x is unshifted) and now,
// D3Q27 cumulant FP32 AA unless noted, every step on the same array:
// - What fits the Infinity Cache (fits_cache) is found there by the next step, if it was written with regular stores:
//   64^3 13.1 -> 10.0, 128^3 81.8 -> 56.7, 128^3 with ghost layers 145 -> 61, EsoTwist 100x90x80 28.2 -> 23.5, D3Q19 TRT
//   pull 96x96x80 (112 MB) 24.1 -> 21.5.  One run of blocks per XCD keeps a cell's neighbours in its L2 as well: D3Q19 SRT
//   FP64 64x32x32 9.8 -> 6.4.  (The row kernel with regular accesses gave 61.2 at 128^3.)
// - Above that, lines that start with a wavefront are best streamed past the caches, as they come: 256^3 593 (685 with
//   regular accesses, 640 with runs of 16 blocks per XCD), FP16 250x200x180 252 -> 170.
// - Otherwise two wavefronts share most lines, and non-temporal accesses move those twice; regular ones, with
//   neighbouring blocks on one XCD, do not: 256^3 with ghost layers 947 -> 709 (809 without the runs), 251x255x253
//   793 -> 684, FP64 131x117x101 143 -> 117.  Every other sweep backwards takes them to 646 and 102 (meets_cached).
// Full wavefronts whatever nx is matter most for short rows: D3Q19 TRT 35x148x256 84 -> 28.
constexpr uint32_t SHARED_LINES_CHUNK = 16;
constexpr int64_t SMALL_CELLS = 1 << 18;   // below: blocks of one wavefront, to spread over the 256 CUs

// Whether the populations' bytes fit the 256 MiB Infinity Cache to a gain.  In place in FP32 or FP64 they may fill it:
// at 128^3 (216 MiB) regular accesses win also for a program that takes three such arrays in turn (82 -> 71 us, one
// array 57; learned closure 120 -> 90, three in turn 108 -> 101).  Two arrays and FP16 storage lose more to such turns
// than they gain alone (pull D3Q19 128x128x80, 199 MB: 39.3 -> 33.8 us for one pair of arrays, three in turn 38.3 -> 40.9;
// FP16 192x128x128, 162 MiB: 54.7 -> 49.5, 63.5): they may fill half of it, where they do not.
inline int64_t population_bytes(const lbm355_sweep_desc* d, bool in_place) {
  const int64_t es = d->store_dtype == LBM355_F64 ? 8 : (d->store_dtype == LBM355_F32 ? 4 : 2);
  const int q = d->stencil == LBM355_D2Q9 ? 9 : (d->stencil == LBM355_D3Q19 ? 19 : 27);
  return (in_place ? 1 : 2) * q * es * d->nx * d->ny * d->nz;
}
constexpr int64_t HALF_CACHE_BYTES = int64_t(128) << 20;
inline bool fits_cache(int64_t bytes, int store, bool in_place) {
  return bytes <= (!in_place || store == LBM355_F16 ? HALF_CACHE_BYTES : 2 * HALF_CACHE_BYTES);
}

// Larger populations still meet a part of themselves in the cache, what the sweep before reached last, if every other
// sweep goes backwards: the even one of an in-place pattern; of two arrays, the one from the lower address.  us per
// launch forwards and so, one array (three in turn, two sweeps on each): D3Q27 cumulant AA FP64 131x117x101 117 (127)
// and 102 (111), FP32 181x175x153 222 (223) and 177 (202), 251x255x253 687 (688) and 646 (666), D3Q19 TRT AA 192x180x144
// with ghost layers and walls 152 (155) and 121 (135), pull 192x160x144 with ghost layers, 672 MB, 165 (164) and 150
// (159).  Two arrays of 1.8 GB lose 1%.
inline bool backwards_sweep(int pattern, const void* src, const void* dst) {
  switch (pattern) {
    case LBM355_AA_EVEN: case LBM355_ESOTWIST_EVEN: case LBM355_ESOPULL_EVEN: case LBM355_ESOPUSH_EVEN: return true;
  }
  return src != dst && (uintptr_t)src < (uintptr_t)dst;
}
inline bool meets_cached(int64_t bytes, bool in_place) { return in_place || bytes <= 8 * HALF_CACHE_BYTES; }
inline bool has_walls(const lbm355_sweep_desc* d) {
  for (int a = 0; a < (d->stencil == LBM355_D2Q9 ? 2 : 3); ++a)
    if (d->face[a] == LBM355_FACE_NOSLIP) return true;
  return false;
}
// Whether that is worth regular accesses where the lines would allow non-temporal ones: D3Q27 cumulant AA FP32 160^3,
// 442 MB, 151 (151) streamed and 132 (151) so, 192^3, 764 MB, 276 (276) and 248 (266), but 224^3, 1.2 GB, 438 (437) and
// 433 (444); FP64 128^3 161 (162) and 136 (158); EsoTwist FP32 192x128x128 127 (125) and 108 (114).  With walls arrays in
// turn lose (D3Q19 TRT 200x200x160 156 (156) and 152 (165)), FP16 too (200^3 146 (145) and 134 (153)), and two arrays
// gain nothing (D3Q19 TRT pull 160^3 119 (119) and 117 (118)).  Fewer populations gain less at the upper end: D3Q19 TRT AA
// 192x192x208, 583 MB, 210 (210) and 189 (202), 256x192x192, 717 MB, 242 (241) and 238 (248), and D2Q9 AA, up to 576 MiB,
// FP32 3520^2, 446 MB, 143 (143) and 135 (145), but 4096^2, 604 MB, 193 (194) and 196 (215), FP64 3072^2, 679 MB, 221 (221)
// and 220 (235).
inline bool cached_anyway(const lbm355_sweep_desc* d, int64_t bytes, bool in_place) {
  const bool flat_aa = d->stencil == LBM355_D2Q9 && !table_pattern(d->pattern);
  return in_place && !has_walls(d) && d->store_dtype != LBM355_F16 &&
         (flat_aa ? 2 * bytes < 9 * HALF_CACHE_BYTES : bytes <= 6 * HALF_CACHE_BYTES);
}

// The streamed modes that a sweep has a kernel for.
struct StreamedModes {
  bool rows, waves, lines;
};

inline bool admits(const StreamedModes& m, int access) {
  switch (access) {
    case ACCESS_ROWS: return m.rows;
    case ACCESS_WAVES: return m.waves;
    case ACCESS_LINES: return m.lines;
    case ACCESS_CACHED: case ACCESS_SHARED: return true;
  }
  return false;
}

inline AccessMode choose_access(const lbm355_sweep_desc* d, const void* src, const void* dst, const StreamedModes& m) {
  const bool in_place = src == dst;
  const int64_t bytes = population_bytes(d, in_place);
  if (fits_cache(bytes, d->store_dtype, in_place)) return ACCESS_CACHED;
  if (!cached_anyway(d, bytes, in_place) && starts_lines(d, src, dst)) {
    if (m.rows) return ACCESS_ROWS;
    if (m.waves) return ACCESS_WAVES;
    if (m.lines) return ACCESS_LINES;
  }
  return ACCESS_SHARED;
}

struct SweepLaunch {
  AccessMode mode;
  dim3 grid, block;
  XcdOrder order;
  bool half_cache;   // the populations take at most HALF_CACHE_BYTES
};

inline SweepLaunch sweep_launch(const lbm355_sweep_desc* d, const void* src, const void* dst, AccessMode access) {
  const bool in_place = src == dst;
  const int64_t bytes = population_bytes(d, in_place);
  const bool half = bytes <= HALF_CACHE_BYTES;
  if (access == ACCESS_ROWS) return {access, dim3(1, d->ny, d->nz), dim3(d->nx), XcdOrder::of(1, 1), half};
  if (access == ACCESS_WAVES) {
    const unsigned bx = d->nx < 256 ? d->nx : 256;
    return {access, dim3((d->nx + bx - 1) / bx, d->ny, d->nz), dim3(bx), XcdOrder::of(1, 1), half};
  }
  const int64_t cells = (int64_t)d->nx * d->ny * d->nz;
  const unsigned bx = cells < SMALL_CELLS ? 64 : 256;
  const unsigned blocks = (unsigned)((cells + bx - 1) / bx);
  const unsigned chunk = access == ACCESS_LINES ? 1 : access == ACCESS_CACHED ? blocks / 8 : SHARED_LINES_CHUNK;
  const bool backwards = access == ACCESS_SHARED && meets_cached(bytes, in_place) && backwards_sweep(d->pattern, src, dst);
  return {access, dim3(blocks), dim3(bx), XcdOrder::of(blocks, chunk, backwards), half};
}

// Kernel arguments from a public descriptor (include/lbm355.h).
template <class TC>
inline SweepArgs<TC> make_args(const lbm355_sweep_desc* d, const void* src, void* dst, void* rho, void* u) {
  SweepArgs<TC> a;
  a.src = src;
  a.dst = dst;
  a.rho_out = (TC*)rho;
  a.u_out = (TC*)u;
  a.tab = (const TC*)d->tables;
  a.nx = d->nx;
  a.ny = d->ny;
  a.nz = d->nz;
  a.g = d->ghost_layers;
  a.sy = d->stride_y;
  a.sz = d->stride_z;
  a.sq = d->stride_q;
  a.osy = d->out_stride_y;
  a.osz = d->out_stride_z;
  a.osc = d->out_stride_c;
  for (int i = 0; i < 3; ++i) {
    a.face[i] = d->face[i];
    a.force[i] = (TC)d->force[i];
  }
  a.flags = d->flags;
  a.nactive = d->n_active;
  a.smag_cs2x18 = (TC)(18.0 * d->smagorinsky_constant * d->smagorinsky_constant);
  a.omega_shear = (TC)d->omega_shear;
  a.closure = d->closure;
  a.omega_out = (TC*)d->omega_out;
  a.nut_out = (TC*)d->eddy_viscosity_out;
  a.rho_in = (const TC*)d->density_in;
  a.u_in = (const TC*)d->velocity_in;
  a.nut_scale = (TC)(1.5 * d->smagorinsky_constant * d->smagorinsky_constant);
  a.seed = d->rounding_seed;
  a.row = CellDivider::of((uint32_t)d->nx);
  a.plane = CellDivider::of((uint32_t)d->ny);
  a.order = XcdOrder::of(1, 1);
  a.block = 0;
  return a;
}

}  // namespace lbm355

// checks a sweep descriptor (sizes, strides, dtypes, table pointer); defined in sweep.hip
int lbm355_validate_desc(const lbm355_sweep_desc* d);

// sweeps of the Eso patterns and push (sweep_eso.hip); the descriptor has been validated
int lbm355_launch_sweep_eso(const lbm355_sweep_desc* d, const void* src, void* dst, void* rho, void* u,
                            const lbm355::SweepLaunch& l, size_t row_lds, hipStream_t s);
// whether they have a row kernel for this domain, and the LDS bytes of a row
bool lbm355_eso_row_lds(const lbm355_sweep_desc* d, size_t* lds_bytes);
