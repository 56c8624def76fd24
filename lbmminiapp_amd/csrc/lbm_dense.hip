// lbm_dense.hip -- host side of the structured-grid engine: handle, link-mask
// builder, state initialisation and readout, moments, FP64 mass reduction,
// and the time loop (the replacement of PropagationAA::run / PropagationAB::run,
// src/propagation/PropagationAA.cpp:126-215, src/propagation/PropagationAB.cpp:155-219).
//
// State conventions (pre-collision populations f_s(x) at time t):
//   AA, t even      f_s(x) in slot opp(s) at x (src/propagation/PropagationAA.cpp:111)
//   AA, t odd       f_s(x) in slot s at x - c_s, or slot opp(s) at x when x - c_s is
//                   solid (src/propagation/PropagationAA.cpp:243-257)
//   AB push         f_s(x) in slot s at x of the current array
//   AB pull         the current array holds post-collision values; f_s(x) is gathered
//                   like the AA odd case (src/kernels/KernelAB_SOA_Pull.cpp:139-140)
//   through walls   AB pull with f_s(x) in slot s at x - c_s also where x - c_s is solid
//                   or outside (wrapped)
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <utility>
#include <vector>

#include "lbm_dense_internal.hpp"

namespace lbm {

enum CanonMode { C_LOCAL = 0, C_OPP = 1, C_GATHER = 2, C_WALL = 3 };

// storage cell of cell = (x, y, z): on interleaved rows element x of the row
// sits at position ir_pos(x)
__device__ __forceinline__ int64_t store_cell(const DenseArgs& a, int64_t cell, int x) {
  return a.xk ? cell - x + ir_pos(x, a.xk, a.xlg) : cell;
}

// storage index of f_s(x) for a given state convention
template <int Q, int LAYOUT>
__device__ __forceinline__ int64_t canon_index(int mode, int s, int64_t cell, int x, uint32_t lk,
                                               const Offsets& off, const DenseArgs& a) {
  const int64_t n = a.ncell;
  const int o = Lattice<Q>::opp(s);
  if (mode == C_LOCAL) return slot<Q, LAYOUT>(n, s, store_cell(a, cell, x));
  if (mode == C_OPP || (mode == C_GATHER && ((lk >> o) & 1u)))
    return slot<Q, LAYOUT>(n, o, store_cell(a, cell, x));
  const int cx = Lattice<Q>::c(s, 0);
  return slot<Q, LAYOUT>(
      n, s,
      store_cell(a, cell + off.at(-cx, -Lattice<Q>::c(s, 1), -Lattice<Q>::c(s, 2)),
                 wrap1(x - cx, a.nx)));
}

__device__ __forceinline__ bool cell_coords(const DenseArgs& a, int& x, int& y, int& z,
                                            int64_t& cell) {
  x = blockIdx.x * blockDim.x + threadIdx.x;
  y = blockIdx.y;
  z = blockIdx.z;
  if (x >= a.nx) return false;
  cell = x + (int64_t)a.nx * (y + (int64_t)a.ny * z);
  return true;
}

// ---------------------------------------------------------------- link mask
template <int Q>
__global__ void __launch_bounds__(256)
    k_build_links(const uint8_t* __restrict__ solid, uint32_t* __restrict__ links, int nx, int ny,
                  int nz, int px, int py, int pz, int xk) {
  const int x = blockIdx.x * blockDim.x + threadIdx.x;
  const int y = blockIdx.y, z = blockIdx.z;
  if (x >= nx) return;
  const int64_t cell = x + (int64_t)nx * (y + (int64_t)ny * z);
  // bit s: x + c_s is solid or outside; solid cells carry the same bits (they
  // place the zeros of the whole-line stores) plus SOLID_BIT
  uint32_t m = solid[cell] ? SOLID_BIT : 0u;
  for (int s = 0; s < Q; s++) {
    int p[3] = {x + Lattice<Q>::c(s, 0), y + Lattice<Q>::c(s, 1), z + Lattice<Q>::c(s, 2)};
    const int dims[3] = {nx, ny, nz};
    const int per[3] = {px, py, pz};
    bool wall = false;
    for (int k = 0; k < 3; k++) {
      if (p[k] < 0 || p[k] >= dims[k]) {
        if (!per[k]) wall = true;
        else p[k] = p[k] < 0 ? p[k] + dims[k] : p[k] - dims[k];
      }
    }
    if (!wall) wall = solid[p[0] + (int64_t)nx * (p[1] + (int64_t)ny * p[2])] != 0;
    if (wall) m |= 1u << s;
  }
  // stored like the populations: at the cell's position on interleaved rows
  links[xk ? cell - x + ir_pos(x, xk) : cell] = m;
}

// ---------------------------------------------------------------- state in / out
// Sign of the pressure-drop jump between the stored value at canon_index and
// the canonical f_s(x): non-zero only where a gathering convention reads
// across the periodic x boundary (canonical = stored + sign * w_s * djump).
template <int Q>
__device__ __forceinline__ int canon_jump_sign(int mode, int s, int x, uint32_t lk, int nx) {
  if (mode < C_GATHER || ((lk >> Lattice<Q>::opp(s)) & 1u)) return 0;
  return gather_crossing(Lattice<Q>::c(s, 0), x, nx);
}

// f_s(x) -> storage, for every fluid cell; src is canonical [Q][ncell] (device).
template <int Q, int STORE, int LAYOUT>
__global__ void __launch_bounds__(256)
    k_set_canonical(const double* __restrict__ src, void* fv, DenseArgs a, int mode) {
  auto* f = static_cast<typename Storage<STORE>::T*>(fv);
  int x, y, z;
  int64_t cell;
  if (!cell_coords(a, x, y, z, cell)) return;
  const uint32_t lk = a.links ? a.links[store_cell(a, cell, x)] : 0u;
  if (lk & SOLID_BIT) return;
  const Offsets off(x, y, z, a.nx, a.ny, a.nz);
  for (int s = 0; s < Q; s++) {
    double v = with_jump<Q>(src[a.ncell * s + cell], -canon_jump_sign<Q>(mode, s, x, lk, a.nx), s,
                            a.djump);
    if constexpr (STORE != LBM_STORE_F64) v -= Lattice<Q>::w(s);
    st<STORE>(f, canon_index<Q, LAYOUT>(mode, s, cell, x, lk, off, a),
              (typename Storage<STORE>::C)v, a.scale);
  }
}

template <int STORE>
__device__ __forceinline__ double to_f(typename Storage<STORE>::C v, double w) {
  if constexpr (STORE == LBM_STORE_F64) return v;
  else return w + (double)v;
}

template <int Q, int STORE, int LAYOUT>
__global__ void __launch_bounds__(256)
    k_get_canonical(const void* fv, double* __restrict__ dst, DenseArgs a, int mode) {
  const auto* f = static_cast<const typename Storage<STORE>::T*>(fv);
  int x, y, z;
  int64_t cell;
  if (!cell_coords(a, x, y, z, cell)) return;
  const uint32_t lk = a.links ? a.links[store_cell(a, cell, x)] : 0u;
  const Offsets off(x, y, z, a.nx, a.ny, a.nz);
  for (int s = 0; s < Q; s++) {
    double v = 0.0;
    if (!(lk & SOLID_BIT))
      v = with_jump<Q>(
          to_f<STORE>(ld<STORE>(f, canon_index<Q, LAYOUT>(mode, s, cell, x, lk, off, a),
                                a.inv_scale),
                      Lattice<Q>::w(s)),
          canon_jump_sign<Q>(mode, s, x, lk, a.nx), s, a.djump);
    dst[a.ncell * s + cell] = v;
  }
}

// rho, u = m / rho of the pre-collision state (reference readout: no F/2 shift,
// src/propagation/PropagationAA.cpp:260-327).
template <int Q, int STORE, int LAYOUT>
__global__ void __launch_bounds__(256)
    k_moments(const void* fv, double* __restrict__ rho_out, double* __restrict__ u_out,
              DenseArgs a, int mode) {
  const auto* f = static_cast<const typename Storage<STORE>::T*>(fv);
  int x, y, z;
  int64_t cell;
  if (!cell_coords(a, x, y, z, cell)) return;
  const uint32_t lk = a.links ? a.links[store_cell(a, cell, x)] : 0u;
  double rho = 0.0, m0 = 0.0, m1 = 0.0, m2 = 0.0;
  if (!(lk & SOLID_BIT)) {
    const Offsets off(x, y, z, a.nx, a.ny, a.nz);
    for (int s = 0; s < Q; s++) {
      const double v = with_jump<Q>(
          to_f<STORE>(ld<STORE>(f, canon_index<Q, LAYOUT>(mode, s, cell, x, lk, off, a),
                                a.inv_scale),
                      Lattice<Q>::w(s)),
          canon_jump_sign<Q>(mode, s, x, lk, a.nx), s, a.djump);
      rho += v;
      m0 += v * Lattice<Q>::c(s, 0);
      m1 += v * Lattice<Q>::c(s, 1);
      m2 += v * Lattice<Q>::c(s, 2);
    }
    const double inv = 1.0 / rho;
    m0 *= inv;
    m1 *= inv;
    m2 *= inv;
  }
  rho_out[cell] = rho;
  u_out[3 * cell + 0] = m0;
  u_out[3 * cell + 1] = m1;
  u_out[3 * cell + 2] = m2;
}

// ---------------------------------------------------------------- initial states
__device__ __forceinline__ uint64_t splitmix64(uint64_t z) {
  z += 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

__device__ __forceinline__ double uniform01(uint64_t seed, uint64_t counter) {
  const uint64_t key = seed * 0x9E3779B97F4A7C15ull + counter;
  return (double)(splitmix64(key) >> 11) * (1.0 / 9007199254740992.0);
}

// src_kind 0: rest; 1: rho/u device arrays; 2: Taylor-Green vortex + seeded noise.
template <int Q, int STORE, int LAYOUT>
__global__ void __launch_bounds__(256)
    k_init(void* fv, DenseArgs a, int mode, int src_kind,
           const double* __restrict__ rho_in, const double* __restrict__ u_in, double u0,
           double noise, uint64_t seed) {
  auto* f = static_cast<typename Storage<STORE>::T*>(fv);
  int x, y, z;
  int64_t cell;
  if (!cell_coords(a, x, y, z, cell)) return;
  const uint32_t lk = a.links ? a.links[store_cell(a, cell, x)] : 0u;
  if (lk & SOLID_BIT) return;
  double rho = 1.0, u[3] = {0.0, 0.0, 0.0};
  if (src_kind == 1) {
    if (rho_in) rho = rho_in[cell];
    for (int k = 0; k < 3; k++) u[k] = u_in[3 * cell + k];
  } else if (src_kind == 2) {
    const double kx = 2.0 * M_PI / a.nx, ky = 2.0 * M_PI / a.ny, kz = 2.0 * M_PI / a.nz;
    u[0] = u0 * sin(kx * x) * cos(ky * y) * cos(kz * z);
    u[1] = -u0 * cos(kx * x) * sin(ky * y) * cos(kz * z);
    if (noise != 0.0)
      for (int k = 0; k < 3; k++)
        u[k] += noise * (2.0 * uniform01(seed, 3ull * (uint64_t)cell + k) - 1.0);
  }
  const Offsets off(x, y, z, a.nx, a.ny, a.nz);
  // f^eq with the collision's association (src/kernels/KernelAA_SOA_Base.cpp:227-238, F = 0)
  const double vdotv = 3.0 * (u[0] * u[0] + u[1] * u[1] + u[2] * u[2]);
  for (int s = 0; s < Q; s++) {
    const double c0 = Lattice<Q>::c(s, 0), c1 = Lattice<Q>::c(s, 1), c2 = Lattice<Q>::c(s, 2);
    const double cdotv = 3.0 * (c0 * u[0] + c1 * u[1] + c2 * u[2]);
    const double w = Lattice<Q>::w(s);
    double feq = w * rho * (1.0 + cdotv + 0.5 * cdotv * cdotv - 0.5 * vdotv);
    if constexpr (STORE != LBM_STORE_F64) feq = w * ((rho - 1.0) + rho * (cdotv + 0.5 * cdotv * cdotv - 0.5 * vdotv));
    feq = with_jump<Q>(feq, -canon_jump_sign<Q>(mode, s, x, lk, a.nx), s, a.djump);
    st<STORE>(f, canon_index<Q, LAYOUT>(mode, s, cell, x, lk, off, a),
              (typename Storage<STORE>::C)feq, a.scale);
  }
}

// The state of every fluid cell from one gathering convention and row order into
// another, in another array; values as they are stored.  Bound by the accesses of the
// side whose rows are permuted (512^3, plain or split to interleaved rows: FP64 10.2
// ms, FP32 6.6, FP16 5.8).
template <int Q, int STORE>
__global__ void __launch_bounds__(256)
    k_convert(const void* __restrict__ src, DenseArgs sa, int smode, void* __restrict__ dst,
              DenseArgs da, int dmode) {
  using T = typename Storage<STORE>::T;
  int x, y, z;
  int64_t cell;
  if (!cell_coords(sa, x, y, z, cell)) return;
  const uint32_t lk = sa.links ? sa.links[cell] : 0u;  // (masked boxes: plain rows)
  if (lk & SOLID_BIT) return;
  const Offsets off(x, y, z, sa.nx, sa.ny, sa.nz);
  // positions of x - 1, x and x + 1 in the rows of both sides
  int from[3], to[3];
  for (int i = 0; i < 3; i++) {
    const int xx = wrap1(x + i - 1, sa.nx);
    from[i] = sa.xk ? ir_pos(xx, sa.xk, sa.xlg) : xx;
    to[i] = da.xk ? ir_pos(xx, da.xk, da.xlg) : xx;
  }
  const int64_t n = sa.ncell, row = cell - x;
#pragma unroll
  for (int s = 0; s < Q; s++) {
    const int o = Lattice<Q>::opp(s), cx = Lattice<Q>::c(s, 0);
    const int64_t there = slot<Q, LBM_LAYOUT_SOA>(
        n, s, row + off.oy[1 - Lattice<Q>::c(s, 1)] + off.oz[1 - Lattice<Q>::c(s, 2)]);
    const int64_t back = slot<Q, LBM_LAYOUT_SOA>(n, o, row);
    const bool blocked = (lk >> o) & 1u;
    const int64_t i = blocked && smode == C_GATHER ? back + from[1] : there + from[1 - cx];
    const int64_t j = blocked && dmode == C_GATHER ? back + to[1] : there + to[1 - cx];
    static_cast<T*>(dst)[j] = static_cast<const T*>(src)[i];
  }
}

// ---------------------------------------------------------------- mass
// Sum over every fluid cell of its Q stored values (any state convention but
// through walls is a permutation of the canonical populations over the fluid
// slots; there the values are gathered).
template <int Q, int STORE, int LAYOUT>
__global__ void __launch_bounds__(256)
    k_mass_partial(const void* fv, DenseArgs a, int mode, double* partial) {
  const auto* f = static_cast<const typename Storage<STORE>::T*>(fv);
  __shared__ double red[256];
  double acc = 0.0;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t cell = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; cell < a.ncell;
       cell += stride) {
    if (a.links && (a.links[cell] & SOLID_BIT)) continue;
    if (mode == C_WALL) {
      const int64_t row = cell / a.nx;
      const int x = (int)(cell - row * a.nx), y = (int)(row % a.ny), z = (int)(row / a.ny);
      const Offsets off(x, y, z, a.nx, a.ny, a.nz);
      for (int s = 0; s < Q; s++)
        acc += to_f<STORE>(ld<STORE>(f, canon_index<Q, LAYOUT>(mode, s, cell, x, 0u, off, a), a.inv_scale),
                           Lattice<Q>::w(s));
      continue;
    }
    for (int s = 0; s < Q; s++)
      acc += to_f<STORE>(ld<STORE>(f, slot<Q, LAYOUT>(a.ncell, s, cell), a.inv_scale),
                         Lattice<Q>::w(s));
  }
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

__global__ void __launch_bounds__(256) k_sum_partials(const double* partial, int n, double* out) {
  __shared__ double red[256];
  double acc = 0.0;
  for (int i = threadIdx.x; i < n; i += blockDim.x) acc += partial[i];
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) *out = red[0];
}

// ---------------------------------------------------------------- dispatch helpers
template <template <int, int, int> class K, typename... A>
void launch_util(int q, int storage, int layout, dim3 g, dim3 b, hipStream_t st, A... args) {
#define LBM_UTIL_CASE(QQ, SS, LL) \
  if (q == QQ && storage == SS && layout == LL) return K<QQ, SS, LL>::launch(g, b, st, args...);
#define LBM_UTIL_Q(QQ)                                      \
  LBM_UTIL_CASE(QQ, LBM_STORE_F64, LBM_LAYOUT_SOA)          \
  LBM_UTIL_CASE(QQ, LBM_STORE_F32S, LBM_LAYOUT_SOA)         \
  LBM_UTIL_CASE(QQ, LBM_STORE_F16S, LBM_LAYOUT_SOA)         \
  LBM_UTIL_CASE(QQ, LBM_STORE_F64, LBM_LAYOUT_AOS)          \
  LBM_UTIL_CASE(QQ, LBM_STORE_F32S, LBM_LAYOUT_AOS)         \
  LBM_UTIL_CASE(QQ, LBM_STORE_F16S, LBM_LAYOUT_AOS)
  LBM_UTIL_Q(19)
  LBM_UTIL_Q(27)
#undef LBM_UTIL_Q
#undef LBM_UTIL_CASE
}

#define LBM_UTIL_KERNEL(name)                                                             \
  template <int Q, int S, int L>                                                          \
  struct name##_u {                                                                       \
    template <typename... A>                                                              \
    static void launch(dim3 g, dim3 b, hipStream_t st, A... a) {                          \
      hipLaunchKernelGGL((name<Q, S, L>), g, b, 0, st, a...);                             \
    }                                                                                     \
  };
LBM_UTIL_KERNEL(k_set_canonical)
LBM_UTIL_KERNEL(k_get_canonical)
LBM_UTIL_KERNEL(k_moments)
LBM_UTIL_KERNEL(k_init)
LBM_UTIL_KERNEL(k_mass_partial)
#undef LBM_UTIL_KERNEL
template <int Q, int S, int L>
struct k_convert_u {  // SOA boxes only: the ones that have two-step launches
  template <typename... A>
  static void launch(dim3 g, dim3 b, hipStream_t st, A... a) {
    if constexpr (L == LBM_LAYOUT_SOA) hipLaunchKernelGGL((k_convert<Q, S>), g, b, 0, st, a...);
  }
};

}  // namespace lbm

using namespace lbm;


namespace lbm {

// Utility kernels: 256-wide x segments.
dim3 block_for(int nx) {
  int bx = nx >= 256 ? 256 : ((nx + 63) / 64) * 64;
  return dim3(bx);
}

dim3 grid_for(const lbm_dense* h) {
  const dim3 b = block_for(h->nx);
  return dim3((h->nx + b.x - 1) / b.x, h->ny, h->nz);
}

// Default block width of the unstaged time-step kernels: a whole x-row per
// workgroup when it fits (kDenseMaxBlock), else 256-wide segments.  FP32
// deviation storage measured faster with 256-wide segments when they tile the
// row exactly (D3Q19 AA at nx = 512: 35.6k vs 31.8k MLUPS); otherwise whole
// rows (porous push at nx = 384: 2.50 vs 2.95 ms per step).
int default_step_bx(int nx, int storage) {
  if (nx <= kDenseMaxBlock && !(storage == LBM_STORE_F32S && nx % 256 == 0))
    return ((nx + 63) / 64) * 64;
  return 256;
}

// Dynamic LDS that leaves room for at most k workgroups per CU (160 KiB LDS).
size_t lds_for_blocks_per_cu(int k) {
  return k > 0 ? (size_t)(160 * 1024 / k) & ~(size_t)1023 : (size_t)0;
}

// Launch shapes, fixed at create.  The SOA AA even step reads and writes only
// row-aligned slots, so it needs no whole rows; it measured fastest with
// small workgroups at low occupancy, like the 19-stream in-place copy pattern,
// whose DRAM efficiency drops as more streams are open per CU.  512^3 even
// step, best of a sweep over widths 64-512 and 0-8 workgroups per CU:
//   D3Q19 FP64   128 wide, <= 3 per CU: 7.09-7.12 ms per step, even and odd
//                averaged over 100-step runs alternating with <= 4 per CU
//                (7.16-7.20), <= 5 (7.15-7.20) and <= 2 (7.09-7.13); single
//                even steps 6.91 ms (512-wide rows: 7.86 ms)
//   D3Q19 FP32   256 wide, <= 4 per CU: 3.39 ms (256 wide, no cap: 3.47 ms)
//   D3Q19 FP16   512 wide, <= 4 per CU: 1.74 ms per step, even and odd
//                averaged over 100-step runs with the interleaved-row odd
//                step (256 wide, no cap: 1.76-1.78; 128 wide: 1.84-1.85)
//   D3Q27 FP64   128 wide, <= 2 per CU: 9.75-9.83 ms alternating with 256 wide,
//                <= 2 per CU (10.30-10.33; step pairs 10.67-10.94 vs 10.86-11.28
//                ms per step); 512-wide rows: 10.83 ms
//   D3Q27 FP32   256 wide, no cap: 4.92-4.95 ms per step, even and odd
//                averaged over 100-step runs on plain rows, alternating with
//                128 wide, no cap (5.01-5.07; in single launches right after
//                initialisation 128 wide had ranked first, 4.69 vs 4.86 ms)
//   D3Q27 FP16   512 wide, <= 4 per CU: 2.49-2.50 ms per step, even and odd
//                averaged over 100-step runs with the interleaved-row odd
//                step (128 wide, <= 8 per CU: 2.61-2.67; 256 / 4: 2.53)
// The first handle of a process measured faster than later ones, so shape
// comparisons alternate the candidates, none of them first.
// Environment overrides (tuning): LBM_DENSE_BLOCK_X and LBM_DENSE_BLOCKS_PER_CU
// for the unstaged kernels (the latter also for the staged ones),
// LBM_DENSE_EVEN_BLOCK_X and LBM_DENSE_EVEN_BLOCKS_PER_CU for the even step.
void set_launch_shapes(lbm_dense* h) {
  auto env_int = [](const char* name, int dflt) {
    const char* e = std::getenv(name);
    return e ? std::atoi(e) : dflt;
  };
  auto clamp_bx = [](int bx) { return bx < 64 ? 64 : (bx > kDenseMaxBlock ? kDenseMaxBlock : bx); };
  h->step_bx = clamp_bx(env_int("LBM_DENSE_BLOCK_X", default_step_bx(h->nx, h->storage)));
  h->step_lds = lds_for_blocks_per_cu(env_int("LBM_DENSE_BLOCKS_PER_CU", 0));
  int even_bx = h->step_bx, even_k = 0, odd_ir_bx = h->step_bx, odd_ir_k = 0;
  if (h->layout == LBM_LAYOUT_SOA) {
    static const int shape[2][3][2] = {
        // {width, workgroups per CU} for F64, F32S, F16S
        {{128, 3}, {256, 4}, {512, 4}},  // D3Q19
        {{128, 2}, {256, 0}, {512, 4}},  // D3Q27
    };
    const int* sh = shape[h->q == 19 ? 0 : 1][h->storage];
    even_bx = sh[0];
    even_k = sh[1];
    // The AA odd step on interleaved rows makes only whole aligned block
    // accesses, like the even step.  512^3, best of widths 64-512 and 0-8
    // workgroups per CU; ms per step over 100-step runs, interleaved / plain
    // rows (the plain-row odd step staged, segmented or unstaged as set
    // below):
    //   D3Q19 FP64   64 wide, <= 4 per CU: 7.11-7.14 / 7.20-7.24
    //   D3Q19 FP32  256 wide, <= 4 per CU: 3.42-3.44 / 3.41-3.44
    //   D3Q19 FP16  512 wide, no cap:      1.77-1.78 / 1.89-1.90
    //   D3Q27 FP64  128 wide, <= 4 per CU: 10.62-10.77 / 10.75-10.96
    //   D3Q27 FP16  512 wide, no cap:      2.68-2.69 / 2.87-2.89
    // D3Q27 FP32 ran slower on interleaved rows (5.16-5.18 / 4.96-5.02) and
    // keeps plain rows (dense_create).
    static const int odd_shape[2][3][2] = {
        {{64, 4}, {256, 4}, {512, 0}},   // D3Q19
        {{128, 4}, {128, 4}, {512, 0}},  // D3Q27
    };
    const int* so = odd_shape[h->q == 19 ? 0 : 1][h->storage];
    odd_ir_bx = so[0];
    odd_ir_k = so[1];
  }
  // Non-temporal streaming pays when the populations exceed the 256 MiB
  // memory-side cache; a grid that fits there runs cached (LBM_DENSE_NT=0|1
  // overrides).
  {
    const size_t pop_bytes =
        (h->pattern == LBM_PATTERN_AB ? 2 : 1) * (size_t)h->ncell * h->q * h->esize;
    h->nt = env_int("LBM_DENSE_NT", pop_bytes > ((size_t)256 << 20) ? 1 : 0) != 0;
  }
  int dev = 0, lds = 0;
  if (hipGetDevice(&dev) == hipSuccess &&
      hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) == hipSuccess &&
      lds > 0)
    h->lds_max = (size_t)lds;
  h->even_bx = clamp_bx(env_int("LBM_DENSE_EVEN_BLOCK_X", even_bx));
  h->even_lds = lds_for_blocks_per_cu(env_int("LBM_DENSE_EVEN_BLOCKS_PER_CU", even_k));
  // LBM_DENSE_ODD_IR_BLOCK_X, LBM_DENSE_ODD_IR_BLOCKS_PER_CU: tuning
  h->odd_ir_bx = clamp_bx(env_int("LBM_DENSE_ODD_IR_BLOCK_X", odd_ir_bx));
  h->odd_ir_lds = lds_for_blocks_per_cu(env_int("LBM_DENSE_ODD_IR_BLOCKS_PER_CU", odd_ir_k));
  // Segmented odd step (k_dense_seg_odd): unmasked periodic SOA boxes whose
  // rows split into segments of a multiple of 64 cells.  512^3 D3Q19 odd step,
  // ms (whole-row staged / best segmented shape): FP32 deviations 3.55 / 3.34
  // (256 wide, <= 4 per CU), so FP32 rows of 512 or more take it; FP64 7.46 /
  // 7.86 and FP16 1.99 (unstaged) / 2.74 stay as they are.  LBM_DENSE_ODD_SEG
  // = width (0 off) and LBM_DENSE_ODD_SEG_BLOCKS_PER_CU override (tuning).  The
  // mask is known only later in create, so dense_create clears it for masked
  // grids.
  {
    const bool dflt = h->storage == LBM_STORE_F32S && h->q == 19 && h->nx >= 512 &&
                      h->nx % 256 == 0;
    const int w = env_int("LBM_DENSE_ODD_SEG", dflt ? 256 : 0);
    const bool ok = h->layout == LBM_LAYOUT_SOA && h->pattern == LBM_PATTERN_AA && w >= 64 &&
                    w <= 256 && w % 64 == 0 && h->nx % w == 0;
    h->odd_seg_w = ok ? w : 0;
    h->odd_seg_lds = lds_for_blocks_per_cu(env_int("LBM_DENSE_ODD_SEG_BLOCKS_PER_CU", dflt ? 4 : 0));
  }
}

// state convention of the current array
int canon_mode(const lbm_dense* h) {
  if (h->pattern == LBM_PATTERN_AA) return h->opp ? C_OPP : C_GATHER;
  return h->walls ? C_WALL : (h->pull ? C_GATHER : C_LOCAL);
}

// kernels with the Guo forcing terms: a nonzero force, or the policy set at create
bool use_force_terms(const lbm_dense* h) {
  return h->force_terms || h->args.F0 != 0.0 || h->args.F1 != 0.0 || h->args.F2 != 0.0;
}

DenseLaunchFn pick_step(const lbm_dense* h, int kind) {
  const bool mask = h->links != nullptr;
  const bool force = use_force_terms(h);
  return h->q == 19 ? pick_dense19(h->storage, h->layout, kind, mask, force, h->nt)
                    : pick_dense27(h->storage, h->layout, kind, mask, force, h->nt);
}

// The LDS-staged kernels cover SOA grids whose rows fit one workgroup (nx a
// multiple of 64, nx <= kDenseMaxBlock): every kind on fully periodic boxes,
// and the pull gather also with solid cells and walls.  By default (staged
// mode 1, set at create from LBM_DENSE_STAGED) they run where they measured
// faster: 512^3 steps, staged vs unstaged handles alternating in one process,
// ms per step (unmasked periodic boxes):
//               AA (odd staged)     AB push            AB pull
//   D3Q19 FP64  staged (7.68/8.47)  8.46 / 8.93        8.10 / 7.83 unstaged
//   D3Q19 FP32  staged (3.64/3.79)  4.23 / 4.94        3.86 / 3.56 unstaged
//   D3Q19 FP16  1.94 / 1.91 unst.   1.86 / 2.05        1.90 / 2.05
//   D3Q27 FP64  10.65 / 11.35       11.65 / 12.69      11.71 / 10.77 unstaged
//   D3Q27 FP32  4.64 / 4.90         5.96 / 6.45        5.75 / 5.29 unstaged
//   D3Q27 FP16  unstaged (kernel alone 3.08 / 2.90)  push 2.81 / 3.27  pull unstaged (3.12 / 3.02)
// Masked gathers run unstaged (35% solid porous pull at 384^3: 20.4k vs 18.7k
// MLUPS staged; a 5% solid channel: equal).  Mode 0 never stages, mode 2
// stages every case covered (tuning and cross-checks).
DenseLaunchFn pick_staged(const lbm_dense* h, int kind) {
  const int mode = h->staged_mode;
  const bool mask = h->links != nullptr;
  if (mode == 0 || h->layout != LBM_LAYOUT_SOA || h->nx % 64 != 0 || h->nx > kDenseMaxBlock ||
      h->xk)
    return nullptr;
  if (mode < 2) {
    const bool f16 = h->storage == LBM_STORE_F16S;
    const bool staged = kind == K_AB_PUSH || (kind == K_AA_ODD && !f16) ||
                        (kind == K_AB_PULL && f16 && h->q == 19);
    if (mask || !staged) return nullptr;
  }
  const bool force = use_force_terms(h);
  return h->q == 19 ? pick_staged19(h->storage, kind, force, h->nx, mask, h->lds_max, h->nt)
                    : pick_staged27(h->storage, kind, force, h->nx, mask, h->lds_max, h->nt);
}

lbm_status launch_kind(lbm_dense* h, int kind, void* f0, void* f1, int z0, int nzl) {
  if (nzl < 0) {
    z0 = 0;
    nzl = h->nz;
  }
  DenseArgs a = h->args;
  a.z0 = z0;
  if (kind == K_AA_ODD && h->xk && !h->links) {
    DenseLaunchFn fn = pick_step(h, K_AA_ODD_IR);
    LBM_REQUIRE(fn, LBM_ERR_UNSUPPORTED, "no interleaved-row odd kernel for this configuration");
    const dim3 b(h->odd_ir_bx);
    fn(dim3((h->nx + b.x - 1) / b.x, h->ny, nzl), b, h->stream, f0, f1, a, h->odd_ir_lds);
    LBM_LAUNCH_CHECK();
    return LBM_OK;
  }
  if (kind == K_AA_ODD && h->odd_seg_w > 0) {
    const int w = h->odd_seg_w;
    const bool force = use_force_terms(h);
    DenseLaunchFn fn = h->q == 19 ? pick_seg_odd19(h->storage, force, h->nt)
                                  : pick_seg_odd27(h->storage, force, h->nt);
    LBM_REQUIRE(fn, LBM_ERR_UNSUPPORTED, "no segmented odd kernel for this configuration");
    fn(dim3((unsigned)((h->nx / w) * h->ny * nzl)), dim3(w), h->stream, f0, f1, a, h->odd_seg_lds);
    LBM_LAUNCH_CHECK();
    return LBM_OK;
  }
  if (DenseLaunchFn st = pick_staged(h, kind)) {
    st(dim3(1, h->ny, nzl), dim3(h->nx), h->stream, f0, f1, a, h->step_lds);
  } else {
    DenseLaunchFn fn = pick_step(h, kind);
    LBM_REQUIRE(fn, LBM_ERR_UNSUPPORTED, "no kernel for this configuration");
    const bool even = kind == K_AA_EVEN;
    const dim3 b(even ? h->even_bx : h->step_bx);
    const dim3 g((h->nx + b.x - 1) / b.x, h->ny, nzl);
    fn(g, b, h->stream, f0, f1, a, even ? h->even_lds : h->step_lds);
  }
  LBM_LAUNCH_CHECK();
  return LBM_OK;
}

// One AA step pair (even, then odd) as z-slabs of P planes, so that the odd
// step of a slab runs right after the even steps it reads, while their planes
// are still in the memory-side cache.  The odd step at z reads and writes
// slots of planes z - 1 .. z + 1, all of which the even step must have
// updated first (and no odd step may precede the even step of a plane it
// writes).  Order with S slabs: even(S-1), even(0), then for k = 0 .. S-2
// even(k+1), odd(k), then odd(S-1).  Every node still gets one even and one
// odd update with the same arithmetic, so the result equals the whole-box
// launches bit for bit.
lbm_status enqueue_aa_pair_by_slabs(lbm_dense* h) {
  const int P = h->slab_planes, S = (h->nz + P - 1) / P;
  void* f = h->f[h->cur];
  auto run = [&](int kind, int k) {
    const int z0 = k * P;
    return launch_kind(h, kind, f, f, z0, std::min(P, h->nz - z0));
  };
  if (lbm_status st = run(K_AA_EVEN, S - 1)) return st;
  if (S > 1)
    if (lbm_status st = run(K_AA_EVEN, 0)) return st;
  for (int k = 0; k + 1 < S; k++) {
    if (k + 1 < S - 1)
      if (lbm_status st = run(K_AA_EVEN, k + 1)) return st;
    if (lbm_status st = run(K_AA_ODD, k)) return st;
  }
  return run(K_AA_ODD, S - 1);
}

// Whether a caller records the handle's stream into a graph of its own.
bool caller_captures(const lbm_dense* h) {
  hipStreamCaptureStatus s = hipStreamCaptureStatusNone;
  if (h->own_capture) return false;
  if (hipStreamIsCapturing(h->stream, &s) != hipSuccess) (void)hipGetLastError();
  return s == hipStreamCaptureStatusActive;
}

// The other way of storing the state and stepping, without moving the state.
void swap_modes(lbm_dense* h) {
  std::swap(static_cast<StepMode&>(*h), h->other);
  h->in_pairs = !h->in_pairs;
  h->args.xk = h->xk;
  h->args.xlg = h->xlg;
  h->ones = h->several = 0;
}

// ... with the state, which is in a gathering convention, into the other array.
lbm_status convert_mode(lbm_dense* h) {
  const DenseArgs from = h->args;
  const int mode = canon_mode(h);
  swap_modes(h);
  h->opp = false;
  launch_util<k_convert_u>(h->q, h->storage, h->layout, grid_for(h), block_for(h->nx), h->stream,
                           (const void*)h->f[h->cur], from, mode, h->f[1 - h->cur], h->args,
                           canon_mode(h));
  LBM_LAUNCH_CHECK();
  h->cur = 1 - h->cur;
  return LBM_OK;
}

// One step of the present mode.
lbm_status enqueue_step(lbm_dense* h) {
  lbm_status st;
  if (h->pattern == LBM_PATTERN_AA) {
    st = launch_kind(h, h->opp ? K_AA_EVEN : K_AA_ODD, h->f[h->cur], h->f[h->cur]);
    h->opp = !h->opp;
  } else {
    const int pull = h->xk && h->xlg == 1 ? K_AB_PULL_SPLIT : K_AB_PULL;
    st = launch_kind(h, h->walls ? K_AB_WALL : (h->pull ? pull : K_AB_PUSH), h->f[h->cur],
                     h->f[1 - h->cur]);
    h->cur = 1 - h->cur;
  }
  h->t++;
  return st;
}

// The mode for a call of `nsteps` steps; takes the first of them where the state has
// to leave the AA even convention (whose stored values include the pressure jump)
// before it can go into pairs.  A change of mode costs one and a half (FP64) to three
// (FP16) steps, so a handle changes when the calls of a kind repeat: to pairs for 8
// steps asked for in calls of two and more, back at the third call of one step in a row.
lbm_status choose_mode(lbm_dense* h, int nsteps, int* taken) {
  h->ones = nsteps == 1 ? h->ones + 1 : 0;
  h->several = nsteps == 1 ? 0 : std::min(h->several + nsteps, 8);
  if (h->in_pairs) return h->alone_ok && h->ones >= 3 ? convert_mode(h) : LBM_OK;
  if (h->alone_ok && h->several < 8) return LBM_OK;
  if (h->pattern == LBM_PATTERN_AA && h->opp) {
    if (lbm_status st = enqueue_step(h)) return st;
    *taken = 1;
  }
  return convert_mode(h);
}

lbm_status enqueue_steps(lbm_dense* h, int nsteps) {
  int i = 0;
  if (h->pair.launch && nsteps > 0) {
    // A caller's graph keeps the arrays and the mode it was captured with.  For a
    // replay to find the state there, an even run has to end in the array it starts
    // in, as with one step per launch: the captured run, and every run of the handle
    // from then on.
    if (caller_captures(h)) h->caller_graphs = true;
    if (!h->caller_graphs && !h->own_capture)
      if (lbm_status st = choose_mode(h, nsteps, &i)) return st;
  }
  if (h->in_pairs) {
    int pairs = (nsteps - i) / 2;
    if (pairs % 2 && h->caller_graphs) pairs--;
    for (; pairs > 0; pairs--, i += 2) {
      h->pair.launch(h->stream, h->f[h->cur], h->f[1 - h->cur], h->args, h->pair_args);
      LBM_LAUNCH_CHECK();
      h->cur = 1 - h->cur;
      h->t += 2;
    }
  }
  for (; i < nsteps; i++) {
    lbm_status st;
    if (h->pattern == LBM_PATTERN_AA && h->slab_planes > 0 && h->opp && i + 1 < nsteps) {
      st = enqueue_aa_pair_by_slabs(h);
      if (st != LBM_OK) return st;
      h->t += 2;
      i++;
      continue;
    }
    if ((st = enqueue_step(h)) != LBM_OK) return st;
  }
  return LBM_OK;
}

void free_all(lbm_dense* h) {
  if (!h) return;
  for (int i = 0; i < 2; i++)
    if (h->f[i]) (void)hipFree(h->f[i]);
  if (h->links) (void)hipFree(h->links);
  if (h->omega_field) (void)hipFree(h->omega_field);
  if (h->gamma_field) (void)hipFree(h->gamma_field);
  if (h->partial) (void)hipFree(h->partial);
  free_stage(h->stage);
  if (h->e0) (void)hipEventDestroy(h->e0);
  if (h->e1) (void)hipEventDestroy(h->e1);
  if (h->own_stream) (void)hipStreamDestroy(h->own_stream);
  delete h;
}

lbm_status dmalloc(lbm_dense* h, void** p, size_t bytes, const char* what) {
  hipError_t e = hipMalloc(p, bytes);
  if (e != hipSuccess) {
    *p = nullptr;
    set_error("lbm_dense_create: hipMalloc of %zu bytes for %s failed: %s", bytes, what,
              hipGetErrorString(e));
    return LBM_ERR_OOM;
  }
  h->device_bytes += bytes;
  return LBM_OK;
}

// Step 0 again, in the array that an even step from here would be in: a caller's
// graphs rely on it (enqueue_steps).  Without pairs of steps that is array 0.
// AA and push boxes with a pressure drop start in the mode without pairs: a
// gathering convention would subtract the jump that its next step adds again, and
// so round the state.
void restart(lbm_dense* h) {
  if (!h->pair.launch) {
    h->cur = 0;
    h->opp = true;
  } else {
    if (h->starts_alone && h->in_pairs && !h->caller_graphs) swap_modes(h);
    if (h->pattern == LBM_PATTERN_AB) h->cur ^= (int)(h->t & 1);
    else h->opp = h->caller_graphs ? h->opp != (bool)(h->t & 1) : true;
  }
  h->t = 0;
}

lbm_status init_from(lbm_dense* h, int src_kind, const double* rho_d, const double* u_d,
                     double u0, double noise, uint64_t seed) {
  restart(h);
  const int mode = canon_mode(h);
  launch_util<k_init_u>(h->q, h->storage, h->layout, grid_for(h), block_for(h->nx), h->stream,
                        h->f[h->cur], h->args, mode, src_kind, rho_d, u_d, u0, noise, seed);
  LBM_LAUNCH_CHECK();
  return LBM_OK;
}

// Number of planes per chunk of the two-step kernel: the launch takes as many
// rounds as the resident workgroups need for all work items, and a round as long
// as a chunk's planes and its two halo planes (and about half a plane to start).
// With this rule a 256^3 D3Q19 FP64 box runs 256-plane chunks, 493 us per step
// (64 planes: 545); 100^3 runs 12-plane chunks, 39.8 us (64 planes: 152).
PairArgs plan_pair(const PairKernel& k, int nx, int ny, int nz, int slots) {
  PairArgs p{};
  p.ntx = (nx / k.v + k.w - 1) / k.w;
  p.nty = (ny + k.ty - 1) / k.ty;
  double best = 0.0;
  for (int lz = 1; lz <= nz; lz++) {
    const int64_t items = (int64_t)p.ntx * p.nty * ((nz + lz - 1) / lz);
    const double cost = (double)((items + slots - 1) / slots) * (lz + 2.5);
    if (lz == 1 || cost < best) {
      best = cost;
      p.lz = lz;
    }
  }
  p.nch = (nz + p.lz - 1) / p.lz;
  p.per_xcd = (int)(((int64_t)p.ntx * p.nty * p.nch + 7) / 8);
  return p;
}

// Whether pairs of steps fill their tiles: rows of a tile past the box idle, and a
// chunk collides two planes more than it finishes.  Measured (us per step, single /
// pairs, 20 steps a call, boxes of 20,000 to 17M cells):
//   FP64   ny = 2 111 / 118 (1024 x 2 x 1024), 3 167 / 132; nz = 1 214 / 234 (2048^2),
//          2 17.4 / 19.2 (384^2), 3 650 / 548 (2048^2); D3Q27 ny = 2 as 3, nz = 3 938 /
//          966, 4 on 3000 x 10 12.0 / 13.4, 6 122 / 97 (512^2), ny = 5 in tiles of 4 1,590
//          / 1,670 (2048 x 5 x 2048), 6 471 / 372
//   FP32   ny = 3 72.7 / 69.6 and D3Q27 113 / 119, 4 107 / 93 and 153 / 130; 9 rows in
//          tiles of 8 54.4 / 59.2 and 75 / 91, 11 294 / 231 and 442 / 376; nz = 3 71.8 /
//          75.0 (1024^2), 4 107 / 90
//   FP16   gains little, so it needs nearly full tiles: 100^3 25.6 / 22.0, 96 x 100 x 90
//          20.9 / 19.3; 17 rows 262 / 284 (1024 x 17 x 1024), 25 rows 342 / 358, 128 x
//          128 x 16 8.7 / 10.0, 320 x 100 x 90 (lanes) 41.1 / 46.5; small boxes 48^3
//          8.8 / 9.0, 64^3 10.2 / 9.2; AB 64^3 7.5 / 9.3, 128^3 27.4 / 27.6, 256 x 200 x
//          128 93.3 / 79.2
// Small boxes of a few planes are launch-bound and gain (256^2 x 1 FP64 8.5 / 5.2), but the
// smallest ones wait for the march along z (64 x 64 x 12 FP32 4.4 / 4.7, 79 x 14 x 47 pull
// FP64 with a force 8.2 / 9.6, 28^3 5.9 / 5.5).
//   masked AA, push: 128^2 x 24 FP64 22.6 / 20.1 and 21.4 / 20.1, x 12 12.8 / 12.6 and
//          12.1 / 12.6, 100^2 x 20 14.0 / 14.4 and 12.4 / 14.4; large ones 512^2 x 8
//          122 / 106, 6 72 / 81 (AA); the pull's single step is faster while both arrays
//          fit the memory-side cache: 64^3 FP64 13.6 / 14.6, 80^3 25.9 / 28.0, 100^3
//          69.1 / 57.5, D3Q27 FP32 channel 41.9 / 45.4, 128^3 87.8 / 69.9
bool tiles_full(const lbm_dense* h, bool need_links) {
  const int ty = h->q == 27 && h->storage == LBM_STORE_F64 ? 4 : 8;
  const double rows = (double)h->ny / ((h->ny + ty - 1) / ty * ty);
  const bool ab = h->pattern == LBM_PATTERN_AB;
  const bool past_cache = 2 * (size_t)h->ncell * h->q * h->esize > ((size_t)256 << 20);
  if (h->storage == LBM_STORE_F16S) {
    auto fill = [](int n, int w) { return (double)n / ((n + w - 1) / w * w); };
    const int nc = h->nx / 2;
    return (ab ? past_cache : h->ncell >= 250000) && rows * h->nz / (h->nz + 2.0) >= 0.9 &&
           fill(nc, nc <= 32 ? 32 : 64) >= 0.85 * fill(h->nx, 64);
  }
  const bool f64 = h->storage == LBM_STORE_F64;
  if (need_links)
    return h->nz >= (h->ncell >= (1 << 21) ? 8 : 24) && (!h->pull || past_cache);
  if (h->ncell < 60000 && (rows < 0.9 || h->nz < 16)) return false;
  if (h->ny < (f64 ? 3 : 4) || (h->ny > ty && rows < (f64 && h->q == 19 ? 0.0 : 0.65)))
    return false;
  if (h->ncell <= (1 << 17) && rows >= 0.9) return true;
  return h->nz >= (!f64 ? 4 : (h->q == 19 ? 3 : 6));
}

// Two steps per launch (lbm_dense_pair.hpp) on SOA boxes in FP64, FP32 and (even
// unmasked rows) FP16 deviations, without per-cell fields, and with a pressure drop only where there
// is a mask.  Default from 20,000 cells on; below, the march along z is a longer chain than two
// launches (us per step, one step / two steps per launch, D3Q19 FP64: 16^3 3.9 /
// 4.6, 128 x 16 x 8 3.8 / 5.4, 24^3 5.0 / 4.8, 28^3 6.3 / 5.0, 12 x 12 x 200
// 11.6 / 7.2), where they fill their tiles (tiles_full).  LBM_DENSE_PAIR=0|1 overrides;
// a variable that tunes the one-step kernels asks for them.  Sets h->pair,
// h->pair_args and the two-step mode, and the cache policy: stores stream past the caches when both
// arrays exceed 320 MiB (100^3 FP64, 290 MiB: 44.0 us cached / 44.7 streaming;
// 112^3, 408 MiB: 54.4 / 52.9; 120^3 FP32, 250 MiB: 34.4 / 39.8).
// Masked boxes gain about 1.2x, so they take pairs only where the tiles waste
// less than 15% of that against the one-step kernels: tile rows past the box,
// lanes past the end of narrow rows, and rows that are solid all along, which
// the one-step kernels skip (`live`: the share of rows that are not).  The
// reference's pipe, 20% of such rows, loses: simulationSize 2 12.5 / 14.4 us per
// step, 4 59.5 / 74.7.  An AA box whose array fits the memory-side cache where
// two do not keeps its one array (100^3 porous D3Q19 FP64 52.8 / 55.8).
void choose_pair(lbm_dense* h, const lbm_dense_config* cfg, bool need_links, double live,
                 StepMode* mode) {
  const char* e = std::getenv("LBM_DENSE_PAIR");
  bool on = h->ncell >= 20000;
  for (const char* v : {"LBM_DENSE_IROWS", "LBM_DENSE_ODD_SEG", "LBM_DENSE_ODD_SEG_BLOCKS_PER_CU",
                        "LBM_DENSE_SLAB_PLANES", "LBM_DENSE_STAGED", "LBM_DENSE_FORCE_TERMS",
                        "LBM_DENSE_PUSH_GATHER", "LBM_DENSE_FILL_SOLID", "LBM_DENSE_BLOCK_X",
                        "LBM_DENSE_BLOCKS_PER_CU", "LBM_DENSE_EVEN_BLOCK_X",
                        "LBM_DENSE_EVEN_BLOCKS_PER_CU", "LBM_DENSE_ODD_IR_BLOCK_X",
                        "LBM_DENSE_ODD_IR_BLOCKS_PER_CU"})
    on = on && !std::getenv(v);
  on = on && tiles_full(h, need_links);
  if (e) on = e[0] != '0';
  const size_t plane_bytes = (size_t)h->nx * h->ny * h->esize;
  if (!on || h->layout != LBM_LAYOUT_SOA || cfg->tau || cfg->gamma ||
      (!need_links && cfg->density_jump_x != 0.0) || plane_bytes >= UINT32_MAX)
    return;
  const bool force = cfg->force[0] != 0.0 || cfg->force[1] != 0.0 || cfg->force[2] != 0.0;
  bool nt = h->nt;
  if (!std::getenv("LBM_DENSE_NT"))
    nt = 2 * (size_t)h->ncell * h->q * h->esize > ((size_t)320 << 20);
  const auto pick = h->q == 19 ? (need_links ? pick_pair19_mask : pick_pair19)
                               : (need_links ? pick_pair27_mask : pick_pair27);
  auto slots = [](const PairKernel& k) {
    int dev = 0, cus = 0, per_cu = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k.fn, k.threads, k.lds) != hipSuccess)
      return 0;
    return cus * per_cu;
  };
  // cells per lane (split rows) and tile width, see lbm_dense_pair.hpp
  auto lanes = [](int columns, int w) { return (columns + w - 1) / w * w; };
  int v = 1;
  if (h->storage == LBM_STORE_F16S) {
    // No kernel with one cell per lane, and none for masks.  It works on scaled values:
    // the scale has to be a power of two.
    v = 2;
    int exponent = 0;
    const double scale = cfg->f16_scale > 0.0 ? cfg->f16_scale : 4096.0;
    if (std::frexp(scale, &exponent) != 0.5 || std::abs(exponent) > 32) return;
    if (h->nx % 2 || need_links) return;
  } else if (h->storage == LBM_STORE_F32S && h->q == 19 && !need_links && h->nx % 2 == 0 &&
             h->ncell >= ((int64_t)1 << 22) && 2 * lanes(h->nx / 2, 64) <= lanes(h->nx, 64)) {
    v = 2;
  }
  if (const char* s = std::getenv("LBM_DENSE_PAIR_CELLS"))  // tuning: 1 or 2 where there is a choice
    if (h->storage == LBM_STORE_F32S && h->q == 19 && !need_links && h->nx % 2 == 0)
      v = std::atoi(s) == 2 ? 2 : 1;
  const int nc = h->nx / v;
  const bool narrow = nc <= 32 || (h->q == 19 && h->storage == LBM_STORE_F64 && !need_links &&
                                   lanes(nc, 32) < 0.9 * lanes(nc, 64));
  // Small tiles where single planes of the large ones do not fill the GPU (32^3
  // D3Q19 FP64: 5.2 us per step against 6.7; 48^3, where they do: 9.6 / 8.7).
  for (const bool small : {false, true}) {
    const PairKernel k = pick(h->storage, force, nt, narrow, small, v);
    const int s = k.launch ? slots(k) : 0;
    if (s <= 0) return;
    const PairArgs p = plan_pair(k, h->nx, h->ny, h->nz, s);
    if ((int64_t)p.ntx * p.nty * p.nch >= ((int64_t)1 << 28)) return;
    if (need_links && !e) {
      const size_t cache = (size_t)256 << 20, one = (size_t)h->ncell * h->q * h->esize;
      const double rows = (double)h->ny / (p.nty * k.ty),
                   lanes = (double)((h->nx + 63) / 64 * 64) / (p.ntx * k.w);
      if (live * rows * lanes < 0.85) return;
      if (h->pattern == LBM_PATTERN_AA && one <= cache && 2 * one > cache) return;
    }
    h->pair = k;
    h->pair_args = p;
    mode->pattern = LBM_PATTERN_AB;
    mode->pull = 1;
    mode->walls = need_links;
    mode->nt = h->nt;
    mode->xk = v > 1 ? h->nx / v : 0;
    mode->xlg = v > 1 ? 1 : 6;
    if ((int64_t)p.ntx * p.nty * h->nz > s) return;
  }
}

lbm_status dense_create(const lbm_dense_config* cfg, lbm_dense** out, bool push_by_gather,
                        bool irows_ok, bool pair_ok) {
  LBM_REQUIRE(cfg && out, LBM_ERR_ARG, "lbm_dense_create: null pointer");
  *out = nullptr;
  LBM_REQUIRE(cfg->nx > 0 && cfg->ny > 0 && cfg->nz > 0, LBM_ERR_ARG,
              "lbm_dense_create: dimensions must be positive (got %d x %d x %d)", cfg->nx,
              cfg->ny, cfg->nz);
  LBM_REQUIRE(cfg->ny <= 65535 && cfg->nz <= 65535, LBM_ERR_ARG,
              "lbm_dense_create: ny and nz must be <= 65535");
  LBM_REQUIRE(cfg->q == 19 || cfg->q == 27, LBM_ERR_ARG, "lbm_dense_create: q must be 19 or 27");
  LBM_REQUIRE(cfg->pattern == LBM_PATTERN_AA || cfg->pattern == LBM_PATTERN_AB, LBM_ERR_ARG,
              "lbm_dense_create: bad pattern %d", cfg->pattern);
  LBM_REQUIRE(cfg->layout == LBM_LAYOUT_SOA || cfg->layout == LBM_LAYOUT_AOS, LBM_ERR_ARG,
              "lbm_dense_create: bad layout %d", cfg->layout);
  LBM_REQUIRE(cfg->storage == LBM_STORE_F64 || cfg->storage == LBM_STORE_F32S ||
                  cfg->storage == LBM_STORE_F16S,
              LBM_ERR_ARG, "lbm_dense_create: storage must be F64, F32S or F16S");
  LBM_REQUIRE(std::isfinite(cfg->omega) && cfg->omega > 0.0 && cfg->omega < 2.0, LBM_ERR_ARG,
              "lbm_dense_create: omega must be in (0, 2)");
  LBM_REQUIRE(std::isfinite(cfg->density_jump_x) && (cfg->density_jump_x == 0.0 || cfg->periodic[0]),
              LBM_ERR_ARG, "lbm_dense_create: density_jump_x needs a finite value and periodic x");
  lbm_dense* h = new lbm_dense;
  h->nx = cfg->nx;
  h->ny = cfg->ny;
  h->nz = cfg->nz;
  h->q = cfg->q;
  h->pattern = cfg->pattern;
  h->pull = cfg->pattern == LBM_PATTERN_AB ? (cfg->pull ? 1 : 0) : 0;
  h->layout = cfg->layout;
  h->storage = cfg->storage;
  for (int k = 0; k < 3; k++) h->periodic[k] = cfg->periodic[k] ? 1 : 0;
  if (const char* e = std::getenv("LBM_DENSE_STAGED")) h->staged_mode = std::atoi(e);
  if (const char* e = std::getenv("LBM_DENSE_SLAB_PLANES")) h->slab_planes = std::max(0, std::atoi(e));
  h->ncell = (int64_t)cfg->nx * cfg->ny * cfg->nz;
  h->esize = cfg->storage == LBM_STORE_F64 ? 8 : (cfg->storage == LBM_STORE_F32S ? 4 : 2);
  set_launch_shapes(h);  // after ncell and esize: the cache policy depends on the footprint
  // fluid count (host mask)
  h->nfluid = h->ncell;
  double live = 1.0;  // share of x-rows with fluid cells
  if (cfg->solid) {
    int64_t ns = 0, dead = 0;
    for (int64_t c = 0; c < h->ncell; c += h->nx) {
      int64_t n = 0;
      for (int x = 0; x < h->nx; x++) n += cfg->solid[c + x] != 0;
      ns += n;
      dead += n == h->nx;
    }
    h->nfluid = h->ncell - ns;
    live = 1.0 - (double)dead / ((double)h->ny * h->nz);
  }
  const bool need_links =
      cfg->solid != nullptr || !h->periodic[0] || !h->periodic[1] || !h->periodic[2];
  if (need_links) h->odd_seg_w = 0;  // the segmented odd step covers unmasked periodic boxes
  // Two steps per launch work out of place, in the AB pull convention.  For an AA
  // box they take a second population array, so only while both fit easily: a
  // quarter of the GPU's memory, and half of what is free (512^3 D3Q19 FP64:
  // 41 of 288 GB), and a readback of the state, which takes q doubles per cell,
  // beside them.  Larger boxes, and a GPU that is nearly full, step in place.
  StepMode paired;
  if (pair_ok) choose_pair(h, cfg, need_links, live, &paired);
  const size_t one_array = (size_t)h->ncell * h->q * h->esize;
  const bool aa_as_pairs = h->pair.launch && h->pattern == LBM_PATTERN_AA;
  if (aa_as_pairs) {
    size_t room = 0, total = 0;
    if (hipMemGetInfo(&room, &total) != hipSuccess || 2 * one_array > total / 4 ||
        2 * one_array > room / 2 ||
        2 * one_array + sizeof(double) * (size_t)h->ncell * h->q > room)
      h->pair = {};
  }
  // Interleaved rows (lbm_dense_kernels.hpp) for AA on unmasked periodic SOA
  // boxes whose rows are whole 64-element blocks: the odd step then makes only
  // whole aligned block accesses, like the even step.  Per-cell fields are
  // stored in the same order.  Default for grids that stream from HBM (h->nt),
  // except D3Q27 FP32 deviations, where plain rows measured faster
  // (set_launch_shapes).  Grids that fit the memory-side cache gained nothing
  // (D3Q19 100-400-step runs, MLUPS interleaved / plain rows: 64^3 FP64 18.7k
  // uncapped, 16.6k with the streaming shape / 19.1-19.5k; 128^3 FP16 65.8-67.3k
  // / 66.4-67.8k), while streaming ones did (256^3 FP16 73.0k / 68.0-68.6k;
  // 256^3 FP64 18.7k / 18.5k).  LBM_DENSE_IROWS=0|1 overrides (A/B timing).
  {
    const char* e = std::getenv("LBM_DENSE_IROWS");
    const bool dflt = h->pattern == LBM_PATTERN_AA && !need_links && h->nt &&
                      !(h->q == 27 && h->storage == LBM_STORE_F32S);
    const bool on = e ? e[0] != '0' : dflt;
    // (a mask is stored once, and the two-step kernels address plain rows)
    if (on && irows_ok && !(h->pair.launch && need_links) && h->layout == LBM_LAYOUT_SOA && h->nx % 64 == 0) {
      h->xk = h->nx / 64;
      h->xlg = 6;
      h->odd_seg_w = 0;
    }
  }
  // a per-cell field in the storage order of the populations
  auto store_order = [h](std::vector<double>& v) {
    if (!h->xk) return;
    std::vector<double> t(v.size());
    for (int64_t row = 0; row < h->ncell; row += h->nx)
      for (int x = 0; x < h->nx; x++) t[row + ir_pos(x, h->xk)] = v[row + x];
    v.swap(t);
  };
  // AB push on a masked SOA grid runs the pull (gather) kernel one streaming
  // step out of phase: with P_0 = S^-1 f_0, (C S)^T P_0 = S^-1 (S C)^T f_0, so
  // the push state f_T is the gather of the pull storage, which is how every
  // readout of a pull handle reads it.  Same per-node arithmetic, bit-identical
  // states.  The gather measured faster when the two arrays stream from HBM
  // (384^3 porous, 8.6 GB: 20.4k vs 14.7k MLUPS; reference cylinder at
  // simulationSize 8, 3.5 GB: 18.1k vs 14.9k) and slower when they nearly fit
  // the 256 MiB memory-side cache (simulationSize 4, 460 MB: 14.6k vs 17.9k),
  // so it applies above 1 GiB of populations.  LBM_DENSE_PUSH_GATHER=0|1
  // overrides (A/B timing).
  if (push_by_gather && h->pattern == LBM_PATTERN_AB && !h->pull && need_links &&
      h->layout == LBM_LAYOUT_SOA) {
    const size_t pop_bytes = 2 * (size_t)h->ncell * h->q * h->esize;
    const char* e = std::getenv("LBM_DENSE_PUSH_GATHER");
    const bool gather = e ? e[0] != '0' : pop_bytes > ((size_t)1 << 30);
    if (gather) h->pull = 1;
  }
  lbm_status st = LBM_OK;
  auto fail = [&](lbm_status s) {
    free_all(h);
    return s;
  };
  if (hipStreamCreateWithFlags(&h->own_stream, hipStreamNonBlocking) != hipSuccess ||
      hipEventCreate(&h->e0) != hipSuccess || hipEventCreate(&h->e1) != hipSuccess) {
    set_error("lbm_dense_create: stream/event creation failed");
    return fail(LBM_ERR_HIP);
  }
  h->stream = h->own_stream;
  const size_t fbytes = (size_t)h->ncell * h->q * h->esize;
  const int narrays = h->pattern == LBM_PATTERN_AA && !h->pair.launch ? 1 : 2;
  for (int i = 0; i < narrays; i++)
    if ((st = dmalloc(h, &h->f[i], fbytes, "populations"))) {
      (void)fail(st);
      return aa_as_pairs && narrays == 2
                 ? dense_create(cfg, out, push_by_gather, irows_ok, false)  // in place after all
                 : st;
    }
  if ((st = dmalloc(h, (void**)&h->partial, sizeof(double) * (h->npartial + 1), "reduction")))
    return fail(st);
  if (need_links) {
    if ((st = dmalloc(h, (void**)&h->links, sizeof(uint32_t) * h->ncell, "link mask")))
      return fail(st);
    uint8_t* solid_d = nullptr;
    if (hipMalloc(&solid_d, h->ncell) != hipSuccess) {
      set_error("lbm_dense_create: hipMalloc of the solid mask failed");
      return fail(LBM_ERR_OOM);
    }
    hipError_t e = cfg->solid
                       ? hipMemcpyAsync(solid_d, cfg->solid, h->ncell, hipMemcpyHostToDevice,
                                        h->stream)
                       : hipMemsetAsync(solid_d, 0, h->ncell, h->stream);
    if (e == hipSuccess) {
      const dim3 g = grid_for(h), b = block_for(h->nx);
      if (h->q == 19)
        hipLaunchKernelGGL(k_build_links<19>, g, b, 0, h->stream, solid_d, h->links, h->nx,
                           h->ny, h->nz, h->periodic[0], h->periodic[1], h->periodic[2], h->xk);
      else
        hipLaunchKernelGGL(k_build_links<27>, g, b, 0, h->stream, solid_d, h->links, h->nx,
                           h->ny, h->nz, h->periodic[0], h->periodic[1], h->periodic[2], h->xk);
      e = hipGetLastError();
      if (e == hipSuccess) e = hipStreamSynchronize(h->stream);
    }
    (void)hipFree(solid_d);
    if (e != hipSuccess) {
      set_error("lbm_dense_create: link mask build failed: %s", hipGetErrorString(e));
      return fail(LBM_ERR_HIP);
    }
  }
  if (cfg->tau) {
    std::vector<double> om(h->ncell);
    for (int64_t c = 0; c < h->ncell; c++) {
      const double tau = cfg->tau[c];
      const bool is_solid = cfg->solid && cfg->solid[c];
      if (!is_solid && !(std::isfinite(tau) && tau > 0.5)) {
        set_error("lbm_dense_create: tau[%lld] = %g must be > 0.5", (long long)c, tau);
        return fail(LBM_ERR_ARG);
      }
      om[c] = is_solid ? 1.0 : 1.0 / tau;
    }
    store_order(om);
    if ((st = dmalloc(h, (void**)&h->omega_field, sizeof(double) * h->ncell, "omega field")))
      return fail(st);
    if (hipMemcpy(h->omega_field, om.data(), sizeof(double) * h->ncell, hipMemcpyHostToDevice) !=
        hipSuccess) {
      set_error("lbm_dense_create: omega field copy failed");
      return fail(LBM_ERR_HIP);
    }
  }
  if (cfg->gamma) {
    if ((st = dmalloc(h, (void**)&h->gamma_field, sizeof(double) * h->ncell, "gamma field")))
      return fail(st);
    std::vector<double> gm(cfg->gamma, cfg->gamma + h->ncell);
    store_order(gm);
    if (hipMemcpy(h->gamma_field, gm.data(), sizeof(double) * h->ncell, hipMemcpyHostToDevice) !=
        hipSuccess) {
      set_error("lbm_dense_create: gamma field copy failed");
      return fail(LBM_ERR_HIP);
    }
  }
  const double scale = cfg->f16_scale > 0.0 ? cfg->f16_scale : 4096.0;
  DenseArgs& a = h->args;
  a.nx = h->nx;
  a.ny = h->ny;
  a.nz = h->nz;
  a.ncell = h->ncell;
  a.periodic_bits = (h->periodic[0] ? 1u : 0u) | (h->periodic[1] ? 2u : 0u) |
                    (h->periodic[2] ? 4u : 0u);
  // Zeros into solid cells' slots complete the SOA row segments (+12% on a 35%
  // solid D3Q19 push step); in AOS the extra scattered stores cost more than
  // they save (-33%).  LBM_DENSE_FILL_SOLID=0 turns it off (A/B timing).
  {
    const char* e = std::getenv("LBM_DENSE_FILL_SOLID");
    a.fill_solid = h->layout == LBM_LAYOUT_SOA && !(e && e[0] == '0');
  }
  a.links = h->links;
  a.omega_field = h->omega_field;
  a.gamma_field = h->gamma_field;
  a.omega = cfg->omega;
  a.F0 = cfg->force[0];
  a.F1 = cfg->force[1];
  a.F2 = cfg->force[2];
  a.scale = (float)scale;
  a.inv_scale = (float)(1.0 / scale);
  a.djump = cfg->density_jump_x;
  // With F = 0 the Guo terms are exact zeros, so the kernels that evaluate
  // them give the same bits as the specialised ones.  For D3Q19 FP64 AA on
  // SOA boxes without solids and with plain rows of more than 256 cells
  // (whole-row staged workgroups of more than 4 wavefronts) they also
  // measured faster: two handles alternating in one process, MLUPS without /
  // with the terms, 512^3: 17,436 / 18,304; 256^3: 18,437 / 18,414; 128^3:
  // 19,083 / 18,965; 64^3: 18,373 / 16,990.  In every other case measured
  // (FP32/FP16 deviations, D3Q27, AB, the interleaved-row odd step: 7.33 /
  // 7.37 ms at 512^3) they were equal or slower.  LBM_DENSE_FORCE_TERMS=0|1
  // overrides.
  {
    const bool dflt = h->q == 19 && h->storage == LBM_STORE_F64 && h->pattern == LBM_PATTERN_AA &&
                      h->layout == LBM_LAYOUT_SOA && h->links == nullptr && h->nx > 256 && !h->xk;
    const char* e = std::getenv("LBM_DENSE_FORCE_TERMS");
    h->force_terms = e ? e[0] == '1' : dflt;
  }
  // What has been set up so far is the mode without pairs.  Single steps go back to
  // it where it is faster than out of place (us per step, in place / out of place,
  // D3Q19): AA boxes whose two arrays exceed the memory-side cache (FP64 100^3 52.5 /
  // 60.7, 512^3 7,090 / 7,880; FP32 128^3 46.9 / 59.5; below, FP64 64^3 15.8 / 13.4,
  // FP32 100^3 31.5 / 29.3) or, masked, very small ones (32^3 FP32 5.8 / 6.4, 64^3
  // 12.8 / 12.0); gathers through walls (pull / through walls: 64^3 channel FP32 8.8 /
  // 12.0, porous 384 x 250 x 260 FP32 768 / 1,011) and split rows (pull, 64^3 FP16 7.9
  // / 8.4), where it is the pull.
  if (h->pair.launch) {
    const bool aa = h->pattern == LBM_PATTERN_AA;
    h->alone_ok = aa ? 2 * one_array > ((size_t)256 << 20) || (need_links && h->ncell < 40000)
                     : (paired.walls && h->pull) || paired.xk;
    h->starts_alone = a.djump != 0.0 && !(h->pattern == LBM_PATTERN_AB && h->pull);
    if (!aa) {
      // push: the state of the mode without pairs is one that pairs can take
      if (h->starts_alone) h->pattern = LBM_PATTERN_AA;
      h->pull = h->pattern == LBM_PATTERN_AB;
    }
    h->other = paired;
    swap_modes(h);
  }
  a.xk = h->xk;
  a.xlg = h->xlg;
  // rest state, as PropagationAA/AB::initialize (src/propagation/PropagationAA.cpp:60-123)
  if ((st = init_from(h, 0, nullptr, nullptr, 0.0, 0.0, 0))) return fail(st);
  // (the two-step kernels store every cell of the second array before it is read)
  if (narrays == 2 && !h->pair.launch &&
      hipMemcpyAsync(h->f[1], h->f[0], fbytes, hipMemcpyDeviceToDevice, h->stream) != hipSuccess) {
    set_error("lbm_dense_create: initial copy failed");
    return fail(LBM_ERR_HIP);
  }
  if (hipStreamSynchronize(h->stream) != hipSuccess) {
    set_error("lbm_dense_create: initialisation failed");
    return fail(LBM_ERR_HIP);
  }
  *out = h;
  return LBM_OK;
}

}  // namespace lbm

extern "C" {

lbm_status lbm_dense_create(const lbm_dense_config* cfg, lbm_dense** out) {
  return dense_create(cfg, out, true, true, true);
}

lbm_status lbm_dense_destroy(lbm_dense* h) {
  if (!h) return LBM_OK;
  LBM_REQUIRE(h->live_graphs == 0, LBM_ERR_STATE,
              "lbm_dense_destroy: %d graph(s) of this handle are still alive; destroy them first",
              h->live_graphs);
  (void)hipStreamSynchronize(h->stream);
  free_all(h);
  return LBM_OK;
}

lbm_status lbm_dense_get_info(lbm_dense* h, lbm_dense_info* info) {
  LBM_REQUIRE(h && info, LBM_ERR_ARG, "lbm_dense_get_info: null pointer");
  info->ncell = h->ncell;
  info->n_fluid = h->nfluid;
  info->time_step = h->t;
  info->bytes_per_lup = 2.0 * h->q * (double)h->esize;
  info->device_bytes = h->device_bytes;
  return LBM_OK;
}

lbm_status lbm_dense_set_state(lbm_dense* h, const double* f) {
  LBM_REQUIRE(h && f, LBM_ERR_ARG, "lbm_dense_set_state: null pointer");
  const size_t bytes = sizeof(double) * h->q * h->ncell;
  double* stage = nullptr;
  LBM_HIP_CHECK(hipMalloc(&stage, bytes));
  hipError_t e = hipMemcpyAsync(stage, f, bytes, hipMemcpyHostToDevice, h->stream);
  if (e == hipSuccess) {
    restart(h);
    launch_util<k_set_canonical_u>(h->q, h->storage, h->layout, grid_for(h), block_for(h->nx),
                                   h->stream, (const double*)stage, h->f[h->cur], h->args,
                                   canon_mode(h));
    e = hipGetLastError();
    if (e == hipSuccess) e = hipStreamSynchronize(h->stream);
  }
  (void)hipFree(stage);
  if (e != hipSuccess) {
    set_error("lbm_dense_set_state: %s", hipGetErrorString(e));
    return LBM_ERR_HIP;
  }
  return LBM_OK;
}

lbm_status lbm_dense_get_state(lbm_dense* h, double* f) {
  LBM_REQUIRE(h && f, LBM_ERR_ARG, "lbm_dense_get_state: null pointer");
  const size_t bytes = sizeof(double) * h->q * h->ncell;
  double* stage = nullptr;
  LBM_HIP_CHECK(hipMalloc(&stage, bytes));
  launch_util<k_get_canonical_u>(h->q, h->storage, h->layout, grid_for(h), block_for(h->nx),
                                 h->stream, (const void*)h->f[h->cur], stage, h->args,
                                 canon_mode(h));
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = copy_to_host(h->stage, h->stream, f, stage, bytes);
  (void)hipFree(stage);
  if (e != hipSuccess) {
    set_error("lbm_dense_get_state: %s", hipGetErrorString(e));
    return LBM_ERR_HIP;
  }
  return LBM_OK;
}

lbm_status lbm_dense_init_equilibrium(lbm_dense* h, const double* rho, const double* u) {
  LBM_REQUIRE(h && u, LBM_ERR_ARG, "lbm_dense_init_equilibrium: null pointer");
  double *rho_d = nullptr, *u_d = nullptr;
  LBM_HIP_CHECK(hipMalloc(&u_d, sizeof(double) * 3 * h->ncell));
  hipError_t e = hipMemcpyAsync(u_d, u, sizeof(double) * 3 * h->ncell, hipMemcpyHostToDevice,
                                h->stream);
  if (e == hipSuccess && rho) {
    e = hipMalloc(&rho_d, sizeof(double) * h->ncell);
    if (e == hipSuccess)
      e = hipMemcpyAsync(rho_d, rho, sizeof(double) * h->ncell, hipMemcpyHostToDevice,
                         h->stream);
  }
  lbm_status st = LBM_OK;
  if (e == hipSuccess) st = init_from(h, 1, rho_d, u_d, 0.0, 0.0, 0);
  if (e == hipSuccess && st == LBM_OK) e = hipStreamSynchronize(h->stream);
  (void)hipFree(u_d);
  if (rho_d) (void)hipFree(rho_d);
  if (st != LBM_OK) return st;
  if (e != hipSuccess) {
    set_error("lbm_dense_init_equilibrium: %s", hipGetErrorString(e));
    return LBM_ERR_HIP;
  }
  return LBM_OK;
}

lbm_status lbm_dense_init_tgv(lbm_dense* h, double u0, double noise, uint64_t seed) {
  LBM_REQUIRE(h, LBM_ERR_ARG, "lbm_dense_init_tgv: null handle");
  if (lbm_status st = init_from(h, 2, nullptr, nullptr, u0, noise, seed)) return st;
  LBM_HIP_CHECK(hipStreamSynchronize(h->stream));
  return LBM_OK;
}

lbm_status lbm_dense_step(lbm_dense* h, int32_t nsteps) {
  LBM_REQUIRE(h && nsteps >= 0, LBM_ERR_ARG, "lbm_dense_step: bad arguments");
  return enqueue_steps(h, nsteps);
}

lbm_status lbm_dense_run_timed(lbm_dense* h, int32_t nsteps, double* elapsed_ms) {
  LBM_REQUIRE(h && elapsed_ms && nsteps >= 0, LBM_ERR_ARG, "lbm_dense_run_timed: bad arguments");
  LBM_HIP_CHECK(hipEventRecord(h->e0, h->stream));
  if (lbm_status st = enqueue_steps(h, nsteps)) return st;
  LBM_HIP_CHECK(hipEventRecord(h->e1, h->stream));
  LBM_HIP_CHECK(hipEventSynchronize(h->e1));
  float ms = 0.f;
  LBM_HIP_CHECK(hipEventElapsedTime(&ms, h->e0, h->e1));
  *elapsed_ms = ms;
  return LBM_OK;
}

// Every call on the handle enqueues on h->stream.  Switching waits for the
// work already on the old stream, so the order of calls is kept.
lbm_status lbm_dense_set_stream(lbm_dense* h, void* stream) {
  LBM_REQUIRE(h, LBM_ERR_ARG, "lbm_dense_set_stream: null handle");
  LBM_HIP_CHECK(hipStreamSynchronize(h->stream));
  h->stream = stream ? (hipStream_t)stream : h->own_stream;
  return LBM_OK;
}

// A captured run of an even number of steps.  After an even number of steps
// every convention holds its states as it did before, so a replay continues the
// run from any state an even number of steps from the one at capture.  The
// out-of-place kernels read one array and write the other: one step per launch
// brings an even run back to the array it started in, but two steps per launch
// may not, and the handle may have changed arrays since the capture, so a
// handle with two-step launches captures the run once from each array and
// replays the one that starts in the current array; while it is in its mode
// without pairs, a launch runs the steps as lbm_dense_step does.  The kernels take
// the handle's device pointers, which stay fixed for the handle's lifetime;
// capture records kernel launches only.
struct lbm_dense_graph {
  lbm_dense* h = nullptr;
  int32_t nsteps = 0;
  int phase = 0;                             // parity of the step at capture
  hipGraph_t graph[2] = {nullptr, nullptr};  // by the array the run starts in
  hipGraphExec_t exec[2] = {nullptr, nullptr};
  int end[2] = {0, 0};                       // the array it ends in
  bool pairs = false;                        // captured in the two-step mode
  bool counted = false;                      // included in h->live_graphs
};

lbm_status lbm_dense_graph_destroy(lbm_dense_graph* g) {
  if (!g) return LBM_OK;
  for (int c = 0; c < 2; c++) {
    if (g->exec[c]) (void)hipGraphExecDestroy(g->exec[c]);
    if (g->graph[c]) (void)hipGraphDestroy(g->graph[c]);
  }
  if (g->counted) g->h->live_graphs--;
  delete g;
  return LBM_OK;
}

lbm_status lbm_dense_graph_create(lbm_dense* h, int32_t nsteps, lbm_dense_graph** out) {
  LBM_REQUIRE(h && out, LBM_ERR_ARG, "lbm_dense_graph_create: null pointer");
  LBM_REQUIRE(nsteps > 0 && nsteps % 2 == 0, LBM_ERR_ARG,
              "lbm_dense_graph_create: nsteps must be even and positive (got %d)", nsteps);
  *out = nullptr;
  auto* g = new lbm_dense_graph;
  g->h = h;
  g->nsteps = nsteps;
  g->phase = (int)(h->t % 2);
  // capture on a stream of its own: the caller's stream may be the null
  // stream, which cannot be captured, and nothing captured runs now
  hipStream_t cap = nullptr;
  hipError_t e = hipStreamCreateWithFlags(&cap, hipStreamNonBlocking);
  if (e != hipSuccess) {
    delete g;
    set_error("lbm_dense_graph_create: %s", hipGetErrorString(e));
    return LBM_ERR_HIP;
  }
  const hipStream_t user = h->stream;
  const int64_t t0 = h->t;
  const int cur0 = h->cur;
  const bool opp0 = h->opp, in_pairs0 = h->in_pairs;
  const int ones0 = h->ones, several0 = h->several;
  h->stream = cap;
  h->own_capture = true;
  // (a handle whose mode a caller's graph holds on to is captured in that mode)
  g->pairs = h->pair.launch && (h->in_pairs || !h->caller_graphs);
  if (g->pairs != h->in_pairs) swap_modes(h);
  lbm_status st = LBM_OK;
  for (int c = 0; c < 2 && st == LBM_OK && e == hipSuccess; c++) {
    if (!g->pairs && c != cur0) continue;
    h->t = t0;
    h->cur = c;
    e = hipStreamBeginCapture(cap, hipStreamCaptureModeThreadLocal);
    if (e != hipSuccess) break;
    st = enqueue_steps(h, nsteps);
    const hipError_t e2 = hipStreamEndCapture(cap, &g->graph[c]);
    if (st == LBM_OK && e2 != hipSuccess) e = e2;
    if (st == LBM_OK && e == hipSuccess)
      e = hipGraphInstantiate(&g->exec[c], g->graph[c], nullptr, nullptr, 0);
    g->end[c] = h->cur;
  }
  h->stream = user;
  h->own_capture = false;
  if (in_pairs0 != h->in_pairs) swap_modes(h);
  h->t = t0;
  h->cur = cur0;
  h->opp = opp0;
  h->ones = ones0;
  h->several = several0;
  (void)hipStreamDestroy(cap);
  if (st != LBM_OK || e != hipSuccess) {
    if (st == LBM_OK) set_error("lbm_dense_graph_create: %s", hipGetErrorString(e));
    lbm_dense_graph_destroy(g);
    return st != LBM_OK ? st : LBM_ERR_HIP;
  }
  g->counted = true;
  h->live_graphs++;
  *out = g;
  return LBM_OK;
}

lbm_status lbm_dense_graph_launch(lbm_dense_graph* g, int32_t nlaunch) {
  LBM_REQUIRE(g && nlaunch >= 0, LBM_ERR_ARG, "lbm_dense_graph_launch: bad arguments");
  lbm_dense* h = g->h;
  if (h->pair.launch && caller_captures(h)) h->caller_graphs = true;
  LBM_REQUIRE((int)(h->t % 2) == g->phase && (g->pairs || g->exec[h->cur]), LBM_ERR_ARG,
              "lbm_dense_graph_launch: the handle is an odd number of steps away from the "
              "state the graph was captured in");
  for (int32_t i = 0; i < nlaunch; i++) {
    // not the captured mode, or a caller's graph relies on the array (enqueue_steps)
    if (g->pairs != h->in_pairs || (h->caller_graphs && g->end[h->cur] != h->cur)) {
      if (lbm_status st = enqueue_steps(h, g->nsteps)) return st;
      continue;
    }
    h->ones = 0;
    LBM_HIP_CHECK(hipGraphLaunch(g->exec[h->cur], h->stream));
    h->cur = g->end[h->cur];
    h->t += g->nsteps;
  }
  return LBM_OK;
}

lbm_status lbm_dense_moments(lbm_dense* h, double* rho, double* u) {
  LBM_REQUIRE(h && rho && u, LBM_ERR_ARG, "lbm_dense_moments: null pointer");
  double* buf = nullptr;
  LBM_HIP_CHECK(hipMalloc(&buf, sizeof(double) * 4 * h->ncell));
  launch_util<k_moments_u>(h->q, h->storage, h->layout, grid_for(h), block_for(h->nx), h->stream,
                           (const void*)h->f[h->cur], buf, buf + h->ncell, h->args,
                           canon_mode(h));
  hipError_t e = hipGetLastError();
  const size_t nb = sizeof(double) * h->ncell;
  if (worth_staging(h->stage, 3 * nb)) {
    if (e == hipSuccess) e = copy_to_host(h->stage, h->stream, u, buf + h->ncell, 3 * nb);
    if (e == hipSuccess) e = copy_to_host(h->stage, h->stream, rho, buf, nb);
  } else {
    if (e == hipSuccess) e = hipMemcpyAsync(rho, buf, nb, hipMemcpyDeviceToHost, h->stream);
    if (e == hipSuccess)
      e = hipMemcpyAsync(u, buf + h->ncell, 3 * nb, hipMemcpyDeviceToHost, h->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(h->stream);
  }
  (void)hipFree(buf);
  if (e != hipSuccess) {
    set_error("lbm_dense_moments: %s", hipGetErrorString(e));
    return LBM_ERR_HIP;
  }
  return LBM_OK;
}

lbm_status lbm_dense_mass(lbm_dense* h, double* mass) {
  LBM_REQUIRE(h && mass, LBM_ERR_ARG, "lbm_dense_mass: null pointer");
  launch_util<k_mass_partial_u>(h->q, h->storage, h->layout, dim3(h->npartial), dim3(256),
                                h->stream, (const void*)h->f[h->cur], h->args, canon_mode(h), h->partial);
  LBM_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_sum_partials, dim3(1), dim3(256), 0, h->stream, (const double*)h->partial,
                     h->npartial, h->partial + h->npartial);
  LBM_LAUNCH_CHECK();
  LBM_HIP_CHECK(hipMemcpyAsync(mass, h->partial + h->npartial, sizeof(double),
                               hipMemcpyDeviceToHost, h->stream));
  LBM_HIP_CHECK(hipStreamSynchronize(h->stream));
  LBM_REQUIRE(std::isfinite(*mass), LBM_ERR_NUMERIC, "lbm_dense_mass: mass is not finite (%g)",
              *mass);
  return LBM_OK;
}

lbm_status lbm_dense_synchronize(lbm_dense* h) {
  LBM_REQUIRE(h, LBM_ERR_ARG, "lbm_dense_synchronize: null handle");
  LBM_HIP_CHECK(hipStreamSynchronize(h->stream));
  return LBM_OK;
}

}  // extern "C"
