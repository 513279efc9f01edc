// The pull / AA sweep kernel template and its per-(pattern, storage) pickers, shared by the translation
// units that instantiate it (sweep_<family>_<compute type>.hip, one per collision family and compute type, so
// that the library builds in parallel).  The C ABI and the launch code are in sweep.hip.
#pragma once
#include <type_traits>

#include "sweep_cell.h"

namespace lbm355 {

template <class S, int FAM, int PAT, bool WALLS, int MODE, class TS, class TC>
__global__ void __launch_bounds__(MODE == ACCESS_ROWS ? 512 : 256) sweep_kernel(SweepArgs<TC> a) {
  if constexpr (MODE != ACCESS_ROWS) {
    int x, y, z;
    if (!thread_cell<MODE>(a, x, y, z)) return;
    sweep_cell<S, FAM, PAT, WALLS, MODE != ACCESS_CACHED, TS, TC>(a, x, y, z);
  } else {
    const int x = blockIdx.x * blockDim.x + threadIdx.x;
    // The block spans one whole periodic row (blockDim.x == nx).  The +-1 x-shifts of pull / AA-odd
    // streaming go through LDS, so every global access is an aligned, contiguous, non-temporal one.
    constexpr int Q = S::Q, D = S::D;
    const int y = blockIdx.y;
    const int z = blockIdx.z;
    const AxisNb ax = axis_neighbours(x, a.nx, a.g, a.face[0]);
    const AxisNb ay = axis_neighbours(y, a.ny, a.g, a.face[1]);
    AxisNb az = {0, 0, false, false};
    if (D == 3) az = axis_neighbours(z, a.nz, a.g, a.face[2]);
    const int sy = (int)a.sy, sz = (int)a.sz;
    const int X1 = x + a.g;
    const int Y[3] = {ay.lo * sy, (y + a.g) * sy, ay.hi * sy};
    const int Z[3] = {D == 3 ? az.lo * sz : 0, D == 3 ? (z + a.g) * sz : 0, D == 3 ? az.hi * sz : 0};
    const int center = X1 + Y[1] + Z[1];
    // LDS row positions of x - 1 and x + 1 (periodic)
    const int XL[3] = {ax.lo - a.g, x, ax.hi - a.g};
    const TS* __restrict__ src = reinterpret_cast<const TS*>(a.src);
    TS* __restrict__ dst = reinterpret_cast<TS*>(a.dst);
    const int64_t sq = a.sq;
    extern __shared__ unsigned char lds_raw[];
    TS* tile = reinterpret_cast<TS*>(lds_raw);
    const int nx = a.nx;

    // walls are only in y / z here (x is periodic), so whether a block's row touches one is uniform
    const bool row_walls = WALLS && (ay.wall_lo || ay.wall_hi || az.wall_lo || az.wall_hi);

    TC f[Q];
    auto load = [&](auto walls) {
      constexpr bool W = decltype(walls)::value;
      int j = 0;
#pragma unroll
      for (int i = 0; i < Q; ++i) {
        const int cx = S::c[i][0], cy = S::c[i][1], cz = S::c[i][2];
        const int ii = S::inv[i];
        const int plane = (PAT == LBM355_PULL) ? i : ii;
        const int wplane = (PAT == LBM355_PULL) ? ii : i;
        bool wall = false;
        if (W)
          wall = (cy == 1 && ay.wall_lo) || (cy == -1 && ay.wall_hi) || (cz == 1 && az.wall_lo) ||
                 (cz == -1 && az.wall_hi);
        if (cx != 0) {
          if (wall)
            f[i] = load_nt<TS, TC>(src + wplane * sq + center);
          else
            tile[j * nx + x] = __builtin_nontemporal_load(src + plane * sq + X1 + Y[1 - cy] + Z[1 - cz]);
          ++j;
        } else {
          const TS* p = wall ? (src + wplane * sq + center) : (src + plane * sq + X1 + Y[1 - cy] + Z[1 - cz]);
          f[i] = load_nt<TS, TC>(p);
        }
      }
      __syncthreads();
      j = 0;
#pragma unroll
      for (int i = 0; i < Q; ++i) {
        const int cx = S::c[i][0], cy = S::c[i][1], cz = S::c[i][2];
        if (cx == 0) continue;
        bool wall = false;
        if (W)
          wall = (cy == 1 && ay.wall_lo) || (cy == -1 && ay.wall_hi) || (cz == 1 && az.wall_lo) ||
                 (cz == -1 && az.wall_hi);
        if (!wall) f[i] = (TC)tile[j * nx + XL[1 - cx]];
        ++j;
      }
      __syncthreads();
    };
    // AA odd writes f_i to x + c_i slot i; at a wall it is bounced into the cell's slot inv(i)
    auto store = [&](auto walls) {
      constexpr bool W = decltype(walls)::value;
      int j = 0;
#pragma unroll
      for (int i = 0; i < Q; ++i) {
        const int cx = S::c[i][0], cy = S::c[i][1], cz = S::c[i][2];
        const int ii = S::inv[i];
        bool wall = false;
        if (W)
          wall = (cy == -1 && ay.wall_lo) || (cy == 1 && ay.wall_hi) || (cz == -1 && az.wall_lo) ||
                 (cz == 1 && az.wall_hi);
        if (cx != 0) {
          if (wall)
            store_as<TS, TC>(dst + ii * sq + center, f[i]);
          else
            tile[j * nx + x] = (TS)f[i];
          ++j;
        } else {
          TS* p = wall ? (dst + ii * sq + center) : (dst + i * sq + X1 + Y[1 + cy] + Z[1 + cz]);
          store_nt<TS, TC>(p, f[i]);
        }
      }
      __syncthreads();
      j = 0;
#pragma unroll
      for (int i = 0; i < Q; ++i) {
        const int cx = S::c[i][0], cy = S::c[i][1], cz = S::c[i][2];
        if (cx == 0) continue;
        bool wall = false;
        if (W)
          wall = (cy == -1 && ay.wall_lo) || (cy == 1 && ay.wall_hi) || (cz == -1 && az.wall_lo) ||
                 (cz == 1 && az.wall_hi);
        if (!wall) __builtin_nontemporal_store(tile[j * nx + XL[1 - cx]], dst + i * sq + X1 + Y[1 + cy] + Z[1 + cz]);
        ++j;
      }
    };

    if (row_walls) {
      load(std::true_type{});
    } else {
      load(std::false_type{});
    }

    collide_cell<S, FAM, TC, TS>(f, a, x, y, z);

    if (PAT == LBM355_PULL) {
#pragma unroll
      for (int i = 0; i < Q; ++i) store_nt<TS, TC>(dst + i * sq + center, f[i]);
    } else if (row_walls) {
      store(std::true_type{});
    } else {
      store(std::false_type{});
    }
  }
}

// Whether AA odd has a kernel of ACCESS_WAVES, without walls (streamed_modes in sweep.hip).
constexpr bool odd_waves_kernel(int family, int store) {
  return store == LBM355_F16 && (family == LBM355_FAMILY_MOMENT || family == LBM355_FAMILY_CENTRAL);
}

// AA even has no x-shifts (no row kernel); AA odd reaches no population but the centre's at the cell itself, so its
// per-cell kernel is the ACCESS_CACHED one, but for odd_waves_kernel's.
template <class S, int FAM, bool WALLS, class TS, class TC>
void* pick_walls(int pat, int mode) {
#define LBM_K(P, M) (void*)sweep_kernel<S, FAM, P, WALLS, M, TS, TC>
  if (pat == LBM355_PULL) {
    if (mode == ACCESS_ROWS) return LBM_K(LBM355_PULL, ACCESS_ROWS);
    if (mode == ACCESS_WAVES) return LBM_K(LBM355_PULL, ACCESS_WAVES);
    return mode == ACCESS_LINES ? LBM_K(LBM355_PULL, ACCESS_LINES) : LBM_K(LBM355_PULL, ACCESS_CACHED);
  }
  if constexpr (!WALLS && odd_waves_kernel(FAM, sizeof(TS) == 2 ? LBM355_F16 : LBM355_F32))
    if (pat == LBM355_AA_ODD && mode == ACCESS_WAVES) return LBM_K(LBM355_AA_ODD, ACCESS_WAVES);
  if (pat == LBM355_AA_ODD) return mode == ACCESS_ROWS ? LBM_K(LBM355_AA_ODD, ACCESS_ROWS) : LBM_K(LBM355_AA_ODD, ACCESS_CACHED);
  return nullptr;
#undef LBM_K
}

template <class S, int FAM, class TS, class TC>
void* pick_pattern(int pat, bool walls, int mode) {
#define LBM_K(M) (void*)sweep_kernel<S, FAM, LBM355_AA_EVEN, false, M, TS, TC>
  if (pat == LBM355_AA_EVEN)
    return mode == ACCESS_WAVES ? LBM_K(ACCESS_WAVES) : mode == ACCESS_LINES ? LBM_K(ACCESS_LINES) : LBM_K(ACCESS_CACHED);
#undef LBM_K
  return walls ? pick_walls<S, FAM, true, TS, TC>(pat, mode) : pick_walls<S, FAM, false, TS, TC>(pat, mode);
}

template <class S, int FAM, class TC>
void* pick_store(int store, int pat, bool walls, int mode) {
  if (store == LBM355_F64) return pick_pattern<S, FAM, double, TC>(pat, walls, mode);
  if (store == LBM355_F32) return pick_pattern<S, FAM, float, TC>(pat, walls, mode);
  if constexpr (sizeof(TC) == 4) {
    if (store == LBM355_F16) return pick_pattern<S, FAM, _Float16, TC>(pat, walls, mode);
  }
  return nullptr;
}

// Kernel pickers of each (family, compute type), one per translation unit; NULL when there is no kernel.
#define LBM355_PICKER(NAME) void* NAME(int stencil, int store, int pat, bool walls, int mode)
LBM355_PICKER(pick_sweep_moment_f64);
LBM355_PICKER(pick_sweep_moment_f32);
LBM355_PICKER(pick_sweep_central_f64);
LBM355_PICKER(pick_sweep_central_f32);
LBM355_PICKER(pick_sweep_cumulant_f64);
LBM355_PICKER(pick_sweep_cumulant_f32);
LBM355_PICKER(pick_sweep_cumulant_corrected_f64);
LBM355_PICKER(pick_sweep_cumulant_corrected_f32);
LBM355_PICKER(pick_sweep_cumulant_general_f64);
LBM355_PICKER(pick_sweep_cumulant_general_f32);
LBM355_PICKER(pick_sweep_cumulant_eq3_f64);
LBM355_PICKER(pick_sweep_cumulant_eq3_f32);
LBM355_PICKER(pick_sweep_cumulant_learned_f32);
LBM355_PICKER(pick_sweep_cumulant_learned_eq3_f32);

}  // namespace lbm355
