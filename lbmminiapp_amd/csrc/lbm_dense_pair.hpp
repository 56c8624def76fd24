// lbm_dense_pair.hpp -- two time steps in one pass over memory.
//
// A time step reads and writes every population once and does about one
// operation per byte, so on its own it runs at the copy rate of the memory
// (D3Q19 FP64 512^3: 40.8 GB in 7.1 ms, 5.8 TB/s, 0.88 of a copy) and only
// moving less can make it faster.  k_dense_pair advances two steps per read and
// write of the state: the intermediate populations live in registers and LDS.
//
// Storage is the AB pull convention (post-collision values, a step gathers slot
// s at x - c_s), out of place: reads are the x-shifted ones and go through the
// caches, where neighbouring workgroups share them; writes are whole aligned
// row segments.  A handle that the caller created as AA or AB push runs it too
// (dense_create): every convention holds the same states, bit for bit (k_convert
// moves them).
//
// A workgroup owns a tile of W x TY cells in (x, y) and marches along z through
// a chunk of lz planes.  At plane p it
//   1. collides the tile and a ring of one cell around it (first step) from
//      registers loaded one plane ahead, and puts the results that change lane
//      (c_x or c_y != 0) into LDS;
//   2. starts the loads of plane p + 1;
//   3. gathers from LDS what the tile's cells receive from plane p: the c_z < 0
//      part completes plane p - 1, whose second step is collided and stored; the
//      c_z = 0 and c_z > 0 parts wait in registers for planes p and p + 1.
// One plane of the Q - 3 exchanged directions is all the LDS holds, so the tile
// can be large: the ring costs (W + 2)(TY + 2) / (W TY), 1.29 for 64 x 8, in
// the first step's arithmetic; in memory traffic the caches absorb part of it
// (measured, 512^3 D3Q19 FP64: 24 to 26 GB read per launch where the state is 20.4,
// 20.4 written).
//
// Waves: W TY / 64 of tile rows, 2 W / 64 of the rows above and below, one of
// the two columns beside the tile.  Only the tile's waves do the second step.
// The two roles have loops of their own, and a lane without a cell repeats its
// neighbour's: with no branch around loads and stores the compiler can count
// them, and the wait for plane p + 1's loads leaves the stores of plane p - 1 in
// flight (one loop with the second step in a branch: 4.6 ms per step at 512^3
// FP64, where two loops take 4.1).
//
// Work items go to the XCDs in contiguous runs (x fastest, then y, then chunks),
// so that the tiles whose rings overlap share an L2.
//
// Split rows (V = 2): a lane takes the cells x and x + nx / 2, which are stored
// side by side (ir_pos with blocks of two), so that its accesses are vectors of
// two and a shift along x is one column for both; across the end of the row the
// two parts change places.  It halves the instructions per byte: FP16 with one
// cell per lane was no faster in pairs than in single steps (128-byte accesses),
// with two 512^3 D3Q19 takes 1.45 ms per step (single steps 1.73), 128^3 27.5 us
// (32.9).  FP32 D3Q19 gains from 4M cells on (512^3 2.57 -> 2.05 ms, 200 x 180 x
// 220 0.209 -> 0.187; 160^3 79.0 -> 97.5 us); D3Q27 FP32 spills, and four cells per
// lane were slower in FP16 (2% at 512^3, 5% at 256^3).
//
// Masked boxes (MASK) hold their state through walls (K_AB_WALL): the gather
// needs no links, so loads stay whole rows, and the stores put what a blocked
// link sends back where the next gather looks for it.  Between the two steps a
// blocked link takes the cell's own result instead of the neighbour's, from its
// own LDS position or register.  Per-lane addresses chosen by link in the gather
// made the pairs slower than single steps (384 x 250 x 260 porous, D3Q19 FP32:
// 968 us per step; now 628, single steps 763).
//
// Measured, ms per step, one-step kernels -> pairs (tile as choose_pair takes it):
//   D3Q19 FP64 512^3 7.08 -> 4.00 to 4.23   256^3 0.970 -> 0.493   128^3 0.110 -> 0.069
//   D3Q19 FP32 512^3 3.39 -> 2.05   256^3 0.424 -> 0.268
//   D3Q19 FP16 512^3 1.74 -> 1.45   256^3 0.219 -> 0.186   D3Q27 FP16 256^3 0.325 -> 0.263
//   D3Q27 FP64 384^3 4.44 -> 3.09   FP32 256^3 0.635 -> 0.414
//   channel with 5% spheres 256^3 D3Q19 FP64 0.930 -> 0.778   FP32 0.456 -> 0.350
//   porous 384 x 250 x 260, 35% solid, D3Q19 FP64 1.37 -> 1.14   FP32 0.763 -> 0.628
#pragma once
#include "lbm_dense_kernels.hpp"

#define LBM_INLINE __attribute__((always_inline))

namespace lbm {

// Launch geometry of k_dense_pair.
struct PairArgs {
  int ntx, nty, nch;  // tiles along x and y, chunks along z
  int lz;             // planes per chunk
  int per_xcd;        // work items per XCD (the grid is 8 times as large)
};

// LDS slot of direction s, or -1 where the receiving cell is in the same lane.
template <int Q>
__host__ __device__ constexpr int pair_slot(int s) {
  if (Lattice<Q>::c(s, 0) == 0 && Lattice<Q>::c(s, 1) == 0) return -1;
  int k = 0;
  for (int r = 0; r < s; r++) k += Lattice<Q>::c(r, 0) != 0 || Lattice<Q>::c(r, 1) != 0;
  return k;
}

template <int W, int TY>
constexpr int pair_threads() {
  return W * TY + 2 * W + 64;
}

template <int Q, int STORE, int W, int TY, int V>
constexpr size_t pair_lds_bytes() {
  return (size_t)(Q - 3) * (W + 2) * (TY + 2) * V * sizeof(typename Storage<STORE>::T);
}

// V values of a lane: a vector, or for V = 1 the value itself.
template <typename T, int V>
struct Lanes {
  typedef T type __attribute__((ext_vector_type(V)));
  static __device__ __forceinline__ T get(type v, int i) { return v[i]; }
  static __device__ __forceinline__ void set(type& v, int i, T x) { v[i] = x; }
  // element i from i + d (mod V)
  static __device__ __forceinline__ type turn(type v, int d) {
    static_assert(V == 2, "two cells: either way is a swap");
    return __builtin_shufflevector(v, v, 1, 0);
  }
};
template <typename T>
struct Lanes<T, 1> {
  using type = T;
  static __device__ __forceinline__ T get(T v, int) { return v; }
  static __device__ __forceinline__ void set(T& v, int, T x) { v = x; }
  static __device__ __forceinline__ T turn(T v, int) { return v; }
};

// A wave-uniform address kept in scalar registers, so that an access is one
// instruction with a scalar base and the lane's 32-bit byte offset.
__device__ __forceinline__ global_ptr<char> scalar_base(const void* p) {
  const uint64_t v = (uint64_t)p;
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return (global_ptr<char>)(((uint64_t)hi << 32) | lo);
}
// The lane's offset, opaque next to its use: extended to 64 bits outside the
// loop it would make every access a 64-bit sum per lane.
__device__ __forceinline__ uint32_t lane_offset(uint32_t v) {
  asm("" : "+v"(v));
  return v;
}

// Directions with a component of the given sign along axis d, as link bits.
template <int Q>
__host__ __device__ constexpr uint32_t dirs_along(int d, int sign) {
  uint32_t m = 0;
  for (int s = 0; s < Q; s++) m |= (uint32_t)(Lattice<Q>::c(s, d) == sign) << s;
  return m;
}

// Store of one element at a lane's byte offset from a uniform base, dropped by
// the buffer's range check where `keep` is false: no branch around the store.
template <bool NT, typename T>
__device__ __forceinline__ void buffer_put(void* base, uint32_t bytes, uint32_t off, bool keep, T v) {
  const auto r = __builtin_amdgcn_make_buffer_rsrc((void*)scalar_base(base), 0, bytes, 0x00020000);
  const uint32_t o = keep ? off : 0xffffffffu;
  constexpr int aux = NT ? 2 : 0;  // nt
  if constexpr (sizeof(T) == 8) {
    typedef unsigned int v2u __attribute__((ext_vector_type(2)));
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(v2u, v), r, o, 0, aux);
  } else {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned int, v), r, o, 0, aux);
  }
}

template <int Q, int STORE, bool MASK, bool FORCE, bool NT, int W, int TY, int V>
__global__ void __launch_bounds__((pair_threads<W, TY>()))
    k_dense_pair(const typename Storage<STORE>::T* __restrict__ f0,
                 typename Storage<STORE>::T* __restrict__ f1, DenseArgs a, PairArgs pa) {
  using T = typename Storage<STORE>::T;
  using C = typename Storage<STORE>::C;
  using L = Lanes<T, V>;
  using VT = typename L::type;  // a lane's V cells: x, x + nc, x + 2 nc ... (split rows)
  static_assert(V == 1 || !MASK, "masked boxes: plain rows");
  constexpr int EX = W + 2, EY = TY + 2, PL = EX * EY;
  extern __shared__ unsigned char lbm_smem[];
  VT* lds = reinterpret_cast<VT*>(lbm_smem);  // [Q - 3][EY][EX]
  const int nc = a.nx / V;                    // columns of V cells

  int t = (blockIdx.x & 7) * pa.per_xcd + (blockIdx.x >> 3);
  if (t >= pa.ntx * pa.nty * pa.nch) return;
  const int x0 = t % pa.ntx * W;
  t /= pa.ntx;
  const int y0 = t % pa.nty * TY;
  const int zc = t / pa.nty * pa.lz, ze = zc + pa.lz < a.nz ? zc + pa.lz : a.nz;
  const int xe = x0 + W < nc ? x0 + W : nc, ye = y0 + TY < a.ny ? y0 + TY : a.ny;

  // The lane's cell (X, Y), which may lie one outside the box (the wrapped
  // neighbour); lanes past the end of the tile or of their role repeat a cell.
  constexpr int RW = 64 / W;   // rows per wave
  constexpr int NI = TY / RW;  // waves of tile rows
  static_assert(W <= 64 && 64 % W == 0 && TY % RW == 0 && 2 * EY <= 64, "tile shape");
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  int X = x0 + lane % W < xe ? x0 + lane % W : xe - 1, Y;
  bool inner = false;  // the wave does the second step
  if (w < NI) {
    inner = y0 + w * RW < ye;
    Y = y0 + w * RW + lane / W;
    Y = inner ? (Y < ye ? Y : ye - 1) : ye;
  } else if (w < NI + 2 * W / 64) {
    Y = (w - NI) * RW + lane / W == 0 ? y0 - 1 : ye;
  } else {
    const int i = lane < 2 * EY ? lane : 2 * EY - 1;
    X = i < EY ? x0 - 1 : xe;
    Y = y0 - 1 + i % EY;
    Y = Y < ye ? Y : ye;
  }
  const int lo = (Y - y0 + 1) * EX + X - x0 + 1;  // the cell's position in an LDS slot
  const int x = wrap1(X, nc), y = wrap1(Y, a.ny);
  // byte offsets, within a plane, of the cells at (x - cx, y - cy)
  uint32_t off[3][3];
#pragma unroll
  for (int i = 0; i < 3; i++)
#pragma unroll
    for (int j = 0; j < 3; j++)
      off[i][j] = ((uint32_t)wrap1(y - (j - 1), a.ny) * (uint32_t)nc +
                   (uint32_t)wrap1(x - (i - 1), nc)) * (uint32_t)sizeof(VT);
  const int64_t n = a.ncell, plane = (int64_t)a.nx * a.ny;
  const double F[3] = {a.F0, a.F1, a.F2};

  uint32_t lk = 0, lk_next = 0, lk_prev = 0;  // links of planes p, p + 1, p - 1
  auto load_links = [&](int p) -> uint32_t {
    if constexpr (MASK) {
      const auto base = scalar_base(a.links + plane * wrap1(p < ze ? p : ze, a.nz));
      return *(global_ptr<const uint32_t>)(base + lane_offset(off[1][1] / (uint32_t)sizeof(T) * 4u));
    }
    return 0u;
  };
  // a population that crossed the periodic x boundary along an open link
  auto jump = [&](VT(&d)[Q], uint32_t k) LBM_INLINE {
    if constexpr (MASK) {
      if (a.djump != 0.0) {
#pragma unroll
        for (int s = 0; s < Q; s++) {
          const int cx = Lattice<Q>::c(s, 0);
          const bool wall = (k >> Lattice<Q>::opp(s)) & 1u;
          if (cx != 0) d[s] = with_jump<Q>(d[s], wall ? 0 : gather_crossing(cx, x, a.nx), s, a.djump);
        }
      }
    }
  };
  // To the storage type.  FP16: the FP32 result is rounded first, as in the
  // one-step kernels (one instruction for the last FMA and the conversion would
  // round once).
  auto pack = [&](C v) LBM_INLINE -> T {
    if constexpr (STORE == LBM_STORE_F16S) asm("" : "+v"(v));
    return (T)v;
  };
  // the lane's cells, one after the other; FP16 deviations stay scaled
  auto collide = [&](VT(&f)[Q]) LBM_INLINE {
    double G[3] = {F[0], F[1], F[2]};
    // masked FP64 keeps no products with the force in registers across the loop
    if constexpr (MASK && FORCE && STORE == LBM_STORE_F64)
      asm volatile("" : "+v"(G[0]), "+v"(G[1]), "+v"(G[2]));
    auto cell = [&](auto part) LBM_INLINE {
      constexpr int i = decltype(part)::value;
      C d[Q];
#pragma unroll
      for (int s = 0; s < Q; s++) d[s] = (C)L::get(f[s], i);
      if constexpr (STORE == LBM_STORE_F64) collide_ref<Q, double, false, FORCE>(d, d, a.omega, G, 0.0);
      else collide_shifted<Q, false, FORCE, STORE == LBM_STORE_F16S>(
          d, a.omega, G, 0.0, STORE == LBM_STORE_F16S, a.scale, a.inv_scale);
#pragma unroll
      for (int s = 0; s < Q; s++) L::set(f[s], i, pack(d[s]));
      if constexpr (V > 1) {
        // packed again before the next part (the compiler would unpack all parts at once)
        if constexpr (sizeof(VT) == 8) {
#pragma unroll
          for (int s = 0; s < Q; s++) {
            uint64_t u = __builtin_bit_cast(uint64_t, f[s]);
            asm volatile("" : "+v"(u));
            f[s] = __builtin_bit_cast(VT, u);
          }
        } else if constexpr (sizeof(VT) == 4) {
#pragma unroll
          for (int s = 0; s < Q; s++) {
            uint32_t u = __builtin_bit_cast(uint32_t, f[s]);
            asm volatile("" : "+v"(u));
            f[s] = __builtin_bit_cast(VT, u);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    cell(std::integral_constant<int, 0>{});
    if constexpr (V > 1) cell(std::integral_constant<int, 1>{});
  };
  // ncell, opaque: the Q slot offsets are summed up again at each use rather than
  // kept in (and spilled from) scalar registers
  auto slot_stride = [&]() -> int64_t {
    return (int64_t)(((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)((uint64_t)n >> 32)) << 32) |
                     (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)n));
  };
  // gathers the populations of plane p (past the chunk: of its last halo plane again)
  auto load_plane = [&](int p, VT(&f)[Q]) LBM_INLINE {
    const int z = wrap1(p < ze ? p : ze, a.nz);
    const T* src[3] = {f0 + plane * wrap1(z + 1, a.nz), f0 + plane * z,
                       f0 + plane * wrap1(z - 1, a.nz)};  // plane of cz = -1, 0, 1
    const int64_t step = slot_stride();
    int64_t at = 0;
#pragma unroll
    for (int s = 0; s < Q; s++) {
      const auto base = scalar_base(src[Lattice<Q>::c(s, 2) + 1] + at);
      at += step;
      f[s] = *(global_ptr<const VT>)(
          base + lane_offset(off[Lattice<Q>::c(s, 0) + 1][Lattice<Q>::c(s, 1) + 1]));
    }
  };
  VT own[3];  // the first step's results that stay in the lane, by cz + 1
  auto first_step = [&](VT(&f)[Q], auto beside) LBM_INLINE {
    if constexpr (V > 1) {
      // across the end of the row, the neighbour of part i is in part i -+ 1
#pragma unroll
      for (int s = 0; s < Q; s++) {
        const int cx = Lattice<Q>::c(s, 0);
        if (cx > 0) f[s] = x == 0 ? L::turn(f[s], -1) : f[s];
        if (cx < 0) f[s] = x == nc - 1 ? L::turn(f[s], 1) : f[s];
      }
    }
    jump(f, lk);
    collide(f);
    if constexpr (V > 1 && decltype(beside)::value) {
      // a wrapped column as the tile's end column sees it
#pragma unroll
      for (int s = 0; s < Q; s++)
        if (pair_slot<Q>(s) >= 0)
          f[s] = X < 0 ? L::turn(f[s], -1) : (X >= nc ? L::turn(f[s], 1) : f[s]);
    }
#pragma unroll
    for (int s = 0; s < Q; s++) {
      const int k = pair_slot<Q>(s);
      if (k < 0) own[Lattice<Q>::c(s, 2) + 1] = f[s];
      else lds[k * PL + lo] = f[s];
    }
    __builtin_amdgcn_sched_barrier(0);
  };

  VT f[Q];
  lk = load_links(zc - 1);
  lk_next = load_links(zc);
  load_plane(zc - 1, f);
  if (!inner) {
    for (int p = zc - 1; p <= ze; p++) {
      first_step(f, std::true_type{});
      const uint32_t lk_after = load_links(p + 2);
      load_plane(p + 1, f);
      __builtin_amdgcn_sched_barrier(0);
      __syncthreads();  // LDS holds plane p
      __syncthreads();  // LDS has been read
      lk = lk_next;
      lk_next = lk_after;
    }
    return;
  }

  // Populations of the second step: h of cz = 0 and cz = 1 for plane p - 1, and
  // of cz = 1 for plane p (next), by direction.  Masked, h of cz = -1 is what a
  // blocked link sends back: the cell's own result in the opposite direction.
  VT h[Q] = {}, next[Q] = {};
  auto blocked = [&](uint32_t k, int s) { return MASK && ((k >> Lattice<Q>::opp(s)) & 1u); };
  // what the cell receives in direction s from the plane in LDS
  auto receive = [&](int s, bool wall) LBM_INLINE -> VT {
    const int k = pair_slot<Q>(s);
    if (k < 0) return own[(wall ? -1 : 1) * Lattice<Q>::c(s, 2) + 1];
    int pos = k * PL + lo - Lattice<Q>::c(s, 1) * EX - Lattice<Q>::c(s, 0);
    if (wall) pos = pair_slot<Q>(Lattice<Q>::opp(s)) * PL + lo;
    return lds[pos];
  };
  auto second_step = [&](int z) LBM_INLINE {
    VT d[Q];
#pragma unroll
    for (int s = 0; s < Q; s++) {
      d[s] = h[s];
      if (Lattice<Q>::c(s, 2) < 0) {
        const VT v = receive(s, false);
        d[s] = blocked(lk_prev, s) ? h[s] : v;
      }
    }
    jump(d, lk_prev);
    collide(d);
    const uint32_t here = off[1][1];
    if constexpr (!MASK) {
      T* dst = f1 + plane * z;
      const int64_t step = slot_stride();
#pragma unroll
      for (int s = 0; s < Q; s++) {
        const auto q = (global_ptr<VT>)(scalar_base(dst) + lane_offset(here));
        dst += step;
        if constexpr (NT) __builtin_nontemporal_store(d[s], q);
        else *q = d[s];
      }
    } else {
      // Links that leave the box through a non-periodic face: there the slot
      // belongs to the cell at the other end.
      const uint32_t open = a.periodic_bits;
      uint32_t out = 0;
      if (!(open & 1u)) out |= (x == 0 ? dirs_along<Q>(0, -1) : 0u) | (x == a.nx - 1 ? dirs_along<Q>(0, 1) : 0u);
      if (!(open & 2u)) out |= (y == 0 ? dirs_along<Q>(1, -1) : 0u) | (y == a.ny - 1 ? dirs_along<Q>(1, 1) : 0u);
      if (!(open & 4u)) out |= (z == 0 ? dirs_along<Q>(2, -1) : 0u) | (z == a.nz - 1 ? dirs_along<Q>(2, 1) : 0u);
      const bool solid = (lk_prev & SOLID_BIT) != 0;
      const uint32_t wall = solid ? 0u : lk_prev;
      const uint32_t keep = solid ? (__all(solid) ? 0u : lk_prev & ~out) : ~(lk_prev & out);
      const uint32_t bytes = (uint32_t)(plane * sizeof(T));
      // What blocked links send back, then the whole rows: the branches of the
      // first leave a known number of stores after them.  (The barriers keep the
      // lane offsets of all 37 stores from being live at once.)
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int s = 0; s < Q; s++) {
        const int cx = Lattice<Q>::c(s, 0), cy = Lattice<Q>::c(s, 1), cz = Lattice<Q>::c(s, 2);
        if ((cx != 0 || cy != 0 || cz != 0) && ((wall >> s) & 1u)) {
          const auto base = scalar_base(f1 + (n * Lattice<Q>::opp(s) + plane * wrap1(z + cz, a.nz)));
          *(global_ptr<T>)(base + lane_offset(off[1 - cx][1 - cy])) = L::get(d[s], 0);
        }
      }
      T* dst = f1 + plane * z;
      const int64_t step = slot_stride();
#pragma unroll
      for (int s = 0; s < Q; s++) {
        buffer_put<NT>(dst + step * s, bytes, here, (keep >> s) & 1u, solid ? T(0) : L::get(d[s], 0));
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  auto plane_step = [&](int p, auto second) LBM_INLINE {
    first_step(f, std::false_type{});
    if constexpr (MASK) {  // c_z > 0 of plane p: what its blocked links send back
#pragma unroll
      for (int s = 0; s < Q; s++)
        if (Lattice<Q>::c(s, 2) > 0 && blocked(lk, s)) next[s] = f[Lattice<Q>::opp(s)];
    }
    const uint32_t lk_after = load_links(p + 2);
    load_plane(p + 1, f);
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();  // LDS holds plane p
    if constexpr (decltype(second)::value) second_step(p - 1);
#pragma unroll
    for (int s = 0; s < Q; s++) {
      const int cz = Lattice<Q>::c(s, 2);
      if (cz == 0) {
        h[s] = receive(s, blocked(lk, s));
      } else if (cz > 0) {
        h[s] = next[s];
        next[s] = receive(s, false);
      } else if (MASK) {
        h[s] = receive(s, true);
      }
      // In registers before the barrier that lets the LDS be overwritten: the
      // compiler has moved such a read, used only later, below the barrier.
      if (cz == 0 || (MASK && cz < 0)) asm volatile("" : "+v"(h[s]));
      if (cz > 0) asm volatile("" : "+v"(h[s]), "+v"(next[s]));
    }
    __syncthreads();  // LDS has been read
    lk_prev = lk;
    lk = lk_next;
    lk_next = lk_after;
  };
  plane_step(zc - 1, std::false_type{});
  plane_step(zc, std::false_type{});
  for (int p = zc + 1; p <= ze; p++) plane_step(p, std::true_type{});
}

// A compiled tile shape: its launch, and what a launch plan needs to know of it.
struct PairKernel {
  void (*launch)(hipStream_t stream, const void* f0, void* f1, const DenseArgs& a,
                 const PairArgs& pa);
  const void* fn;
  int w, ty, v, threads;
  size_t lds;
};

template <int Q, int STORE, bool MASK, bool FORCE, bool NT, int W, int TY, int V>
void launch_pair(hipStream_t stream, const void* f0, void* f1, const DenseArgs& a,
                 const PairArgs& pa) {
  using T = typename Storage<STORE>::T;
  hipLaunchKernelGGL((k_dense_pair<Q, STORE, MASK, FORCE, NT, W, TY, V>), dim3(8 * pa.per_xcd),
                     dim3(pair_threads<W, TY>()), (pair_lds_bytes<Q, STORE, W, TY, V>()), stream,
                     (const T*)f0, (T*)f1, a, pa);
}

template <int Q, int STORE, bool MASK, bool FORCE, bool NT, int W, int TY, int V>
PairKernel pair_kernel() {
  return {launch_pair<Q, STORE, MASK, FORCE, NT, W, TY, V>,
          (const void*)k_dense_pair<Q, STORE, MASK, FORCE, NT, W, TY, V>, W, TY, V,
          pair_threads<W, TY>(), pair_lds_bytes<Q, STORE, W, TY, V>()};
}

template <int Q, int STORE, bool MASK, int W, int TY, int V>
PairKernel pick_pair_flags(bool force, bool nt) {
  if (nt) return force ? pair_kernel<Q, STORE, MASK, true, true, W, TY, V>()
                       : pair_kernel<Q, STORE, MASK, false, true, W, TY, V>();
  return force ? pair_kernel<Q, STORE, MASK, true, false, W, TY, V>()
               : pair_kernel<Q, STORE, MASK, false, false, W, TY, V>();
}

// Tile shapes: W = 64 columns of a row, or 32 for rows of up to 32 (a 24 x 200 x
// 100 box, D3Q19 FP64: 18.4 us per step with 32 x 16 tiles, 24.1 with 64 x 8) and,
// D3Q19 FP64, where they leave a tenth fewer lanes empty (200 x 180 x 220: 269 us
// against 287).
// Large tiles have the smaller ring (512^3 D3Q19 FP64, 64 x 8: 4.10 ms per step,
// 64 x 4: 5.03); the smaller ones give small boxes twice the workgroups.  Waves
// bound the registers: 11 of them (64 x 8) leave 168 per lane, which D3Q27 FP64
// and masked D3Q19 FP64 exceed, and spills cost more than a larger ring (D3Q27
// FP64 384^3: 64 x 4 3.09 ms, 64 x 8 3.60; masked channel with a force, 256^3
// D3Q19 FP64: 64 x 5 778 us, 64 x 8 1,130).  Masked D3Q27 FP64 spills in every
// tile and has no two-step kernel.
template <int Q, int STORE, bool MASK, int V>
PairKernel pick_pair_tile(bool force, bool nt, bool narrow, bool small) {
  if constexpr (MASK && !masked_pairs<Q, STORE>()) {
    return {};
  } else if constexpr (MASK && STORE == LBM_STORE_F64) {
    return narrow ? pick_pair_flags<Q, STORE, MASK, 32, 10, V>(force, nt)
                       : pick_pair_flags<Q, STORE, MASK, 64, 5, V>(force, nt);
  } else {
    if constexpr (!(Q == 27 && STORE == LBM_STORE_F64)) {
      if (!small) return narrow ? pick_pair_flags<Q, STORE, MASK, 32, 16, V>(force, nt)
                                : pick_pair_flags<Q, STORE, MASK, 64, 8, V>(force, nt);
    }
    return narrow ? pick_pair_flags<Q, STORE, MASK, 32, 8, V>(force, nt)
                  : pick_pair_flags<Q, STORE, MASK, 64, 4, V>(force, nt);
  }
}

template <int Q, bool MASK>
PairKernel pick_pair_q(int storage, bool force, bool nt, bool narrow, bool small, int v) {
  if (storage == LBM_STORE_F64 && v == 1)
    return pick_pair_tile<Q, LBM_STORE_F64, MASK, 1>(force, nt, narrow, small);
  if (storage == LBM_STORE_F32S && v == 1)
    return pick_pair_tile<Q, LBM_STORE_F32S, MASK, 1>(force, nt, narrow, small);
  if constexpr (!MASK) {
    if constexpr (Q == 19)
      if (storage == LBM_STORE_F32S && v == 2)
        return pick_pair_tile<Q, LBM_STORE_F32S, MASK, 2>(force, nt, narrow, small);
    if (storage == LBM_STORE_F16S && v == 2)
      return pick_pair_tile<Q, LBM_STORE_F16S, MASK, 2>(force, nt, narrow, small);
  }
  return {};
}

// Defined in lbm_dense_pair{19,27}.hip and, masked, lbm_dense_pair{19,27}_mask.hip;
// launch is nullptr where there is no two-step kernel.  narrow: W = 32; small:
// half the rows; v: cells per lane.
PairKernel pick_pair19(int storage, bool force, bool nt, bool narrow, bool small, int v);
PairKernel pick_pair27(int storage, bool force, bool nt, bool narrow, bool small, int v);
PairKernel pick_pair19_mask(int storage, bool force, bool nt, bool narrow, bool small, int v);
PairKernel pick_pair27_mask(int storage, bool force, bool nt, bool narrow, bool small, int v);

}  // namespace lbm
