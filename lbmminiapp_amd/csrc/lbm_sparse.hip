// lbm_sparse.hip -- drop-in GPU replacement of the reference's kernel classes on
// its fluid-only, indirectly addressed node list.
//
// One work-item per fluid node, exactly the reference's parallel_for shape
// (src/kernels/KernelAA_SOA_Base.cpp:180, :263; KernelAB_SOA_Base.cpp:116;
// KernelAB_SOA_Pull.cpp:118), with the node's Q populations held in registers
// and the collision fully unrolled at compile time.  The arithmetic is
// collide_ref (the Base kernels' association and order, no FMA contraction),
// so FP64 results and -D_PRECISION_SINGLE_ FP32 results equal the reference's
// bit for bit.
//
// Launches go to the null stream by default, so that they are ordered with the
// caller's blocking hipMemcpy traffic, as the reference's kernel calls are
// ordered with its host code; lbm_sparse_set_stream moves them to a caller's
// stream (which can then be captured into a HIP graph: the step calls only
// launch kernels).
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <mutex>

#include "lbm_collide.hpp"
#include "lbm_internal.hpp"

namespace lbm {

template <int Q, int LAYOUT>
__device__ __forceinline__ int64_t pidx(int64_t n, int s, int64_t i) {
  return LAYOUT == LBM_LAYOUT_SOA ? n * s + i : (int64_t)Q * i + s;
}

// Node-aligned accesses (a work-item's own slots and adjacency entries) are
// touched once per step.  With NT they stream past the caches, which pays when
// the arrays exceed the memory-side cache; arrays that fit in it are faster
// cached (the reference's simulationSize 4 deck, 175 MB: 15.2k vs 13.6k MLUPS
// AA; simulationSize 8, 1.35 GB: 13.7k vs 14.8k).  Accesses through the
// adjacency stay cacheable, since neighbouring work-items share their lines.
template <bool NT, typename T>
__device__ __forceinline__ T ldn(const T* p) {
  if constexpr (NT) return __builtin_nontemporal_load(p);
  else return *p;
}
template <bool NT, typename T>
__device__ __forceinline__ void stn(T* p, T v) {
  if constexpr (NT) __builtin_nontemporal_store(v, p);
  else *p = v;
}

// Node block of this workgroup.  Workgroups are dispatched to the 8 XCDs in
// turn (block b to XCD b mod 8), each with its own L2.  group > 0 (the launch
// then has a multiple of 8 * group blocks) gives each XCD runs of `group`
// consecutive node blocks, so that cache lines shared by neighbouring blocks
// (accesses through the adjacency) mostly meet in one L2: physical block p,
// round r = p / 8, XCD k = p mod 8, takes node block
// (r / group) 8 group + k group + r mod group, a bijection; blocks past the
// range exit through the count check.
__device__ __forceinline__ int64_t node_block(uint32_t group) {
  if (!group) return blockIdx.x;
  const uint32_t r = blockIdx.x / 8u, k = blockIdx.x % 8u;
  return (int64_t)(r / group) * 8 * group + (int64_t)k * group + r % group;
}

// Node of this work-item.  Node blocks start at multiples of 64, wherever the
// range starts, so that a wavefront covers one group of kGroup nodes of the
// compressed adjacency; work-items before the range and past its end idle.
__device__ __forceinline__ int64_t node_of(int64_t start, uint32_t group) {
  return (start & ~(int64_t)63) + node_block(group) * blockDim.x + threadIdx.x;
}

// ---------------------------------------------------------------- adjacency
// The caller's adjacency costs 4 Q bytes per node and step, 76 of 380 in D3Q19
// FP64.  In the fluid order of a real geometry the 64 nodes of a group reach
// their neighbours at a few distances only: within a row of the list the
// distance adj - own slot is the same, and every bounce-back has one.  So each
// group holds a table of up to kDeltas distances per direction, and each node a
// 3-bit code per direction (10 codes a word): 8 + 9.5 bytes per node for D3Q19,
// built at create on the GPU (k_sparse_compress).  A group with more distances in
// some direction (about 1 in 1000 at the reference's simulationSize 2, most at
// 0.5, whose rows are 10 nodes) keeps reading the caller's table.
// simulationSize 8, D3Q19, us per step, caller's table -> compressed: FP64 AA 573
// -> 521, push 771 -> 569, pull 653 -> 559; FP32 322 -> 282, 504 -> 336, 387 -> 305.
// (The push loads its populations before it decodes: 658 us the other way round.)
constexpr int kGroup = 64;
constexpr int kDeltas = 8;
template <int Q>
__host__ __device__ constexpr int code_words() {
  return (Q + 9) / 10;
}

struct AdjTables {
  const int32_t* adj;    // the caller's adjacency
  const uint32_t* code;  // [code_words][groups * kGroup]
  const int32_t* table;  // [groups][Q][kDeltas]
  const uint32_t* raw;   // [groups]: nonzero where the group is not compressed
  int64_t groups;
};

// One wavefront per group.
template <int Q, int LAYOUT>
__global__ void __launch_bounds__(kGroup)
    k_sparse_compress(const int32_t* __restrict__ adj, uint32_t* __restrict__ code,
                      int32_t* __restrict__ table, uint32_t* __restrict__ raw, int64_t n) {
  const int64_t g = blockIdx.x;
  const int lane = threadIdx.x;
  const int64_t i = g * kGroup + lane;
  uint32_t words[code_words<Q>()] = {};
  bool fits = true;
#pragma unroll
  for (int s = 0; s < Q; s++) {
    const int64_t own = pidx<Q, LAYOUT>(n, s, i);
    const int32_t delta = i < n ? (int32_t)(adj[own] - own) : 0;
    uint64_t left = __ballot(i < n);
    uint32_t mine = 0;
    int32_t entry = 0;
    for (int k = 0; k < kDeltas && left; k++) {
      const int32_t d = __builtin_amdgcn_readlane(delta, __builtin_ctzll(left));
      const uint64_t same = __ballot(delta == d) & left;
      if ((same >> lane) & 1u) mine = k;
      if (lane == k) entry = d;
      left &= ~same;
    }
    fits = fits && !left;
    words[s / 10] |= mine << (3 * (s % 10));
    if (lane < kDeltas) table[(g * Q + s) * kDeltas + lane] = entry;
  }
  for (int w = 0; w < code_words<Q>(); w++) code[(int64_t)w * gridDim.x * kGroup + i] = words[w];
  if (lane == 0) raw[g] = !fits;
}

// The adjacency of this work-item's node.  load() and index() take the whole
// wavefront (a node past the range holds its group's codes too); only index()
// of a node that exists means something.
template <int Q, int LAYOUT, bool NT>
struct AdjReader {
  static constexpr int kRegs = (Q * kDeltas + 63) / 64;
  bool raw;
  uint32_t code[code_words<Q>()];
  int32_t table[kRegs];  // lane l, register r: entry 64 r + l of the group's table

  __device__ __forceinline__ void load(const AdjTables& t, int64_t i) {
    const int64_t g = __builtin_amdgcn_readfirstlane((uint32_t)(i / kGroup));
    raw = t.raw[g] != 0;
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int w = 0; w < code_words<Q>(); w++) code[w] = ldn<NT>(t.code + (w * t.groups * kGroup + i));
#pragma unroll
    for (int r = 0; r < kRegs; r++) {
      const int e = 64 * r + lane;
      table[r] = ldn<NT>(t.table + (g * Q * kDeltas + (e < Q * kDeltas ? e : Q * kDeltas - 1)));
    }
  }
  __device__ __forceinline__ int32_t index(int s, int64_t n, int64_t i) const {
    const int c = (code[s / 10] >> (3 * (s % 10))) & (kDeltas - 1);
    const int d = __builtin_amdgcn_ds_bpermute(4 * ((s * kDeltas) % 64 + c), table[s * kDeltas / 64]);
    return (int32_t)(pidx<Q, LAYOUT>(n, s, i)) + d;
  }
};

// All Q neighbour slots of a node, compressed (COMP; the whole wavefront takes
// part) or from the caller's table.
template <int Q, int LAYOUT, bool NT, bool COMP>
__device__ __forceinline__ void neighbour_slots(const AdjTables& t, int64_t n, int64_t i, bool active,
                                                int32_t* loc) {
  if constexpr (COMP) {
    AdjReader<Q, LAYOUT, NT> r;
    r.load(t, i);
    if (!r.raw) {
#pragma unroll
      for (int s = 0; s < Q; s++) loc[s] = r.index(s, n, i);
      return;
    }
  }
#pragma unroll
  for (int s = 0; s < Q; s++)
    loc[s] = COMP && !active ? 0 : ldn<NT>(t.adj + pidx<Q, LAYOUT>(n, s, i));
}

// AA even: src/kernels/KernelAA_SOA_Base.cpp:173-254 (AOS: KernelAA_AOS_Base.cpp:174-254)
template <int Q, typename T, int LAYOUT, bool NT>
__global__ void __launch_bounds__(256)
    k_sparse_aa_even(T* __restrict__ f, int64_t n, int64_t start, int64_t count, double omega,
                     T F0, T F1, T F2, uint32_t group) {
  const int64_t i = node_of(start, group);
  if (i < start || i >= start + count) return;
  T d[Q];
#pragma unroll
  for (int s = 0; s < Q; s++) d[s] = ldn<NT>(f + pidx<Q, LAYOUT>(n, Lattice<Q>::opp(s), i));
  const T F[3] = {F0, F1, F2};
  collide_ref<Q, T, false>(d, d, omega, F, 0.0);
#pragma unroll
  for (int s = 0; s < Q; s++) stn<NT>(f + pidx<Q, LAYOUT>(n, s, i), d[s]);
}

// AA odd: src/kernels/KernelAA_SOA_Base.cpp:257-342 (AOS: KernelAA_AOS_Base.cpp:258-342)
template <int Q, typename T, int LAYOUT, bool NT, bool COMP>
__global__ void __launch_bounds__(256)
    k_sparse_aa_odd(T* __restrict__ f, AdjTables adj, int64_t n, int64_t start, int64_t count,
                    double omega, T F0, T F1, T F2, uint32_t group) {
  const int64_t i = node_of(start, group);
  const bool active = i >= start && i < start + count;
  if (COMP ? i / kGroup >= adj.groups : !active) return;
  int32_t loc[Q];
  neighbour_slots<Q, LAYOUT, NT, COMP>(adj, n, i, active, loc);
  if (!active) return;
  T d[Q];
#pragma unroll
  for (int s = 0; s < Q; s++) d[s] = f[loc[s]];
  const T F[3] = {F0, F1, F2};
  collide_ref<Q, T, false>(d, d, omega, F, 0.0);
#pragma unroll
  for (int s = 0; s < Q; s++) f[loc[Lattice<Q>::opp(s)]] = d[s];
}

// AB push: src/kernels/KernelAB_SOA_Base.cpp:111-186 (AOS: KernelAB_AOS_Base.cpp:108-182)
template <int Q, typename T, int LAYOUT, bool NT, bool COMP>
__global__ void __launch_bounds__(256)
    k_sparse_ab_push(const T* __restrict__ src, T* __restrict__ tgt, AdjTables adj, int64_t n,
                     int64_t start, int64_t count, double omega, T F0, T F1, T F2, uint32_t group) {
  const int64_t i = node_of(start, group);
  const bool active = i >= start && i < start + count;
  if (COMP ? i / kGroup >= adj.groups : !active) return;
  T d[Q];
  const T F[3] = {F0, F1, F2};
  if constexpr (COMP) {
    if (active) {
#pragma unroll
      for (int s = 0; s < Q; s++) d[s] = ldn<NT>(src + pidx<Q, LAYOUT>(n, s, i));
    }
    int32_t loc[Q];
    neighbour_slots<Q, LAYOUT, NT, true>(adj, n, i, active, loc);
    if (!active) return;
    collide_ref<Q, T, false>(d, d, omega, F, 0.0);
#pragma unroll
    for (int s = 0; s < Q; s++) tgt[loc[s]] = d[s];
  } else {
#pragma unroll
    for (int s = 0; s < Q; s++) d[s] = ldn<NT>(src + pidx<Q, LAYOUT>(n, s, i));
    collide_ref<Q, T, false>(d, d, omega, F, 0.0);
#pragma unroll
    for (int s = 0; s < Q; s++) tgt[ldn<NT>(adj.adj + pidx<Q, LAYOUT>(n, s, i))] = d[s];
  }
}

// AB pull: src/kernels/KernelAB_SOA_Pull.cpp:113-194
template <int Q, typename T, int LAYOUT, bool NT, bool COMP>
__global__ void __launch_bounds__(256)
    k_sparse_ab_pull(const T* __restrict__ src, T* __restrict__ tgt, AdjTables adj, int64_t n,
                     int64_t start, int64_t count, double omega, T F0, T F1, T F2, uint32_t group) {
  const int64_t i = node_of(start, group);
  const bool active = i >= start && i < start + count;
  if (COMP ? i / kGroup >= adj.groups : !active) return;
  T d[Q];
  if constexpr (COMP) {
    int32_t loc[Q];
    neighbour_slots<Q, LAYOUT, NT, true>(adj, n, i, active, loc);
    if (!active) return;
#pragma unroll
    for (int s = 0; s < Q; s++) d[s] = src[loc[s]];
  } else {
#pragma unroll
    for (int s = 0; s < Q; s++) d[s] = src[ldn<NT>(adj.adj + pidx<Q, LAYOUT>(n, s, i))];
  }
  const T F[3] = {F0, F1, F2};
  collide_ref<Q, T, false>(d, d, omega, F, 0.0);
#pragma unroll
  for (int s = 0; s < Q; s++) stn<NT>(tgt + pidx<Q, LAYOUT>(n, s, i), d[s]);
}

// PropagationAA::initialize (slot opp(s) := w_s) and PropagationAB::initialize (slot s := w_s).
template <int Q, typename T, int LAYOUT, bool NT>
__global__ void __launch_bounds__(256) k_sparse_init_rest(T* __restrict__ f, int64_t n, int aa) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
#pragma unroll
  for (int s = 0; s < Q; s++) {
    const int slot = aa ? Lattice<Q>::opp(s) : s;
    f[pidx<Q, LAYOUT>(n, slot, i)] = T(Lattice<Q>::w(s));
  }
}

// FP64 mass of a fluid-index range: the sum of the Q stored values of every
// node in [start, start + count) (over the whole range this is the total mass
// in any slot convention, which only permutes the populations over the
// slots).  Deterministic two-pass reduction with a fixed shape: workgroup b of
// 256 lanes sums the kMassChunk nodes start + b kMassChunk + ... (lane t takes
// nodes t, t + 256, ... of the chunk, each node's values in s order, in FP64)
// into partial[b]; one workgroup then sums the partials in a fixed order.
constexpr int kMassBlock = 256;
constexpr int64_t kMassChunk = 16 * kMassBlock;

__device__ __forceinline__ double mass_block_sum(double v) {
  __shared__ double red[kMassBlock];
  red[threadIdx.x] = v;
  __syncthreads();
  for (int w = kMassBlock / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  return red[0];
}

// (NT is unused: the launcher instantiates every kernel for both cache policies.)
template <int Q, typename T, int LAYOUT, bool NT>
__global__ void __launch_bounds__(kMassBlock)
    k_sparse_mass_partial(const T* __restrict__ f, int64_t n, int64_t start, int64_t count,
                          double* __restrict__ partial) {
  const int64_t c0 = (int64_t)blockIdx.x * kMassChunk;
  double acc = 0.0;
  for (int64_t k = threadIdx.x; k < kMassChunk; k += kMassBlock) {
    if (c0 + k >= count) break;
    const int64_t i = start + c0 + k;
#pragma unroll
    for (int s = 0; s < Q; s++) acc += (double)f[pidx<Q, LAYOUT>(n, s, i)];
  }
  const double tot = mass_block_sum(acc);
  if (threadIdx.x == 0) partial[blockIdx.x] = tot;
}

__global__ void __launch_bounds__(kMassBlock)
    k_sparse_mass_final(const double* __restrict__ partial, int64_t nb, double* __restrict__ out) {
  double acc = 0.0;
  for (int64_t b = threadIdx.x; b < nb; b += kMassBlock) acc += partial[b];
  const double tot = mass_block_sum(acc);
  if (threadIdx.x == 0) *out = tot;
}

// Partial sums of lbm_sparse_mass_noalloc: a fixed device array instead of an
// allocation, kMassScratchPartials doubles (32 KiB) on every GPU the library
// runs on, held until the process ends.  It bounds that entry point's range to
// kMassScratchPartials * kMassChunk = 16,777,216 nodes.  In host code `scratch`
// only names the array; its device address comes from hipGetSymbolAddress
// (scratch_on_current_device), once per device.  The two-pass reduction
// writes every partial it reads, so nothing needs clearing between calls;
// calls that overlap on one GPU share the array and race.
constexpr int64_t kMassScratchPartials = 4096;
static __device__ __align__(256) double scratch[kMassScratchPartials];

}  // namespace lbm

struct lbm_sparse {
  int64_t n = 0;
  int q = 19;
  int layout = LBM_LAYOUT_SOA;
  int storage = LBM_STORE_F64;
  int adjacency_mode = 1;
  double omega = 1.0;
  double force[3] = {1e-6, 0.0, 0.0};
  int32_t* adj = nullptr;  // device copy of the adjacency
  uint32_t* code = nullptr;  // the adjacency compressed (AdjTables), in adj's allocation
  int32_t* table = nullptr;
  uint32_t* raw = nullptr;
  int64_t groups = 0;
  lbm::AdjTables tables() const { return {adj, code, table, raw, groups}; }
  // launch shapes: the AA even step (all node-aligned) and the other steps
  unsigned even_bx = 256, step_bx = 256, push_bx = 256;
  size_t even_lds = 0, step_lds = 0, push_lds = 0;
  bool nt = true;  // non-temporal node-aligned accesses (arrays beyond the memory-side cache)
  hipStream_t stream = nullptr;  // null stream unless the caller set one
  int xcd_env = -1;              // LBM_SPARSE_XCD: node blocks per XCD run (-1: by footprint)
};

namespace {

using namespace lbm;

inline unsigned grid_for(int64_t count, unsigned bx = 256) {
  return (unsigned)((count + bx - 1) / bx);
}

struct Shape {
  unsigned grid, block;
  size_t lds;
  uint32_t group;  // node_block: 0, or node blocks per XCD run (grid a multiple of 8 group)
};

#define LBM_SPARSE_KERNEL_FN(fn, name, ...)                                                \
  template <int Q, typename T, int L>                                                      \
  struct fn {                                                                              \
    template <typename... A>                                                               \
    static void launch(Shape sh, bool nt, hipStream_t st, A... a) {                        \
      if (nt)                                                                              \
        hipLaunchKernelGGL((lbm::name<Q, T, L, true __VA_ARGS__>), dim3(sh.grid),          \
                           dim3(sh.block), sh.lds, st, a...);                              \
      else                                                                                 \
        hipLaunchKernelGGL((lbm::name<Q, T, L, false __VA_ARGS__>), dim3(sh.grid),         \
                           dim3(sh.block), sh.lds, st, a...);                              \
    }                                                                                      \
  };
#define LBM_COMMA ,
LBM_SPARSE_KERNEL_FN(k_sparse_aa_even_fn, k_sparse_aa_even)
LBM_SPARSE_KERNEL_FN(k_sparse_aa_odd_fn, k_sparse_aa_odd, LBM_COMMA true)
LBM_SPARSE_KERNEL_FN(k_sparse_aa_odd_raw_fn, k_sparse_aa_odd, LBM_COMMA false)
LBM_SPARSE_KERNEL_FN(k_sparse_ab_push_fn, k_sparse_ab_push, LBM_COMMA true)
LBM_SPARSE_KERNEL_FN(k_sparse_ab_push_raw_fn, k_sparse_ab_push, LBM_COMMA false)
LBM_SPARSE_KERNEL_FN(k_sparse_ab_pull_fn, k_sparse_ab_pull, LBM_COMMA true)
LBM_SPARSE_KERNEL_FN(k_sparse_ab_pull_raw_fn, k_sparse_ab_pull, LBM_COMMA false)
LBM_SPARSE_KERNEL_FN(k_sparse_init_rest_fn, k_sparse_init_rest)
LBM_SPARSE_KERNEL_FN(k_sparse_mass_partial_fn, k_sparse_mass_partial)
#undef LBM_COMMA
#undef LBM_SPARSE_KERNEL_FN

template <template <int, typename, int> class K, typename T, typename... A>
void launch_qt(const lbm_sparse* h, Shape sh, A... a) {
  if (h->q == 19) {
    if (h->layout == LBM_LAYOUT_SOA) K<19, T, LBM_LAYOUT_SOA>::launch(sh, h->nt, h->stream, a...);
    else K<19, T, LBM_LAYOUT_AOS>::launch(sh, h->nt, h->stream, a...);
  } else {
    if (h->layout == LBM_LAYOUT_SOA) K<27, T, LBM_LAYOUT_SOA>::launch(sh, h->nt, h->stream, a...);
    else K<27, T, LBM_LAYOUT_AOS>::launch(sh, h->nt, h->stream, a...);
  }
}

// A kernel that reads the adjacency: COMP where it is compressed, RAW otherwise.
template <template <int, typename, int> class COMP, template <int, typename, int> class RAW,
          typename T, typename... A>
void launch_adj(const lbm_sparse* h, Shape sh, A... a) {
  if (h->code) launch_qt<COMP, T>(h, sh, a...);
  else launch_qt<RAW, T>(h, sh, a...);
}

// Node blocks per XCD run (node_block).  Measured on the reference's decks
// (drop-in driver, MLUPS, none -> chosen):
//   arrays in the memory-side cache (simulationSize 4, 175 MB): one run per
//   XCD, AA 15.2k -> 16.2k, AB 12.8k -> 14.0k, pull 11.6k -> 11.9k;
//   streaming (simulationSize 8, 1.35 GB): runs of 8-32 blocks raise AB push
//   10.6k -> 11.2k, while AA and pull lost with long runs (14.7k -> 13.3k,
//   13.4k -> 11.4k with one run per XCD) and gained nothing with short ones.
//   With the push's 128-wide capped blocks (set_shapes), runs of 64-128
//   blocks measured best: 11.46-11.47k (16: 11.16-11.20k; 256: 11.34k).
// LBM_SPARSE_XCD (read at create) overrides: 0 off, g > 0 runs of g blocks.
uint32_t xcd_group(const lbm_sparse* h, bool push, unsigned nb) {
  if (h->xcd_env >= 0) return (uint32_t)h->xcd_env;
  if (!h->nt) return (nb + 7) / 8;
  if (!push) return 0u;
  return h->push_bx == 128 ? 64u : 16u;
}

Shape make_shape(const lbm_sparse* h, int64_t count, unsigned bx, size_t lds, bool push) {
  const unsigned nb = grid_for(count, bx);
  const uint32_t g = xcd_group(h, push, nb);
  if (!g || nb < 16) return {nb, bx, lds, 0};
  const unsigned span = 8 * g;
  return {(nb + span - 1) / span * span, bx, lds, g};
}
// (node blocks start at the multiple of 64 at or before `start`, node_of)
Shape even_shape(const lbm_sparse* h, int64_t start, int64_t count) {
  return make_shape(h, count + (start & 63), h->even_bx, h->even_lds, false);
}
Shape step_shape(const lbm_sparse* h, int64_t start, int64_t count, bool push = false) {
  count += start & 63;
  return push ? make_shape(h, count, h->push_bx, h->push_lds, true)
              : make_shape(h, count, h->step_bx, h->step_lds, false);
}

// Launch shapes, fixed at create.  The AA even step is all node-aligned, like
// the dense engine's even step, which measured fastest with small workgroups
// at capped occupancy.  So did the AB push on streaming FP64 arrays
// (simulationSize-8 deck, MLUPS: 128 wide, <= 4 per CU with XCD runs of 64,
// 11.46k; 256 wide, no cap, runs of 16: 11.18-11.21k; 64 wide, <= 8 per CU:
// 10.9-11.3k).  The other steps keep 256-wide workgroups.  Environment
// overrides (tuning): LBM_SPARSE_EVEN_BLOCK_X, LBM_SPARSE_EVEN_BLOCKS_PER_CU,
// LBM_SPARSE_BLOCK_X, LBM_SPARSE_BLOCKS_PER_CU (all other steps, the push
// included).
void set_shapes(lbm_sparse* h) {
  auto env_int = [](const char* name, int dflt) {
    const char* e = std::getenv(name);
    return e ? std::atoi(e) : dflt;
  };
  auto clamp_bx = [](int bx) { return (unsigned)(bx < 64 ? 64 : (bx > 256 ? 256 : bx / 64 * 64)); };
  auto lds_for = [](int k) { return k > 0 ? (size_t)(160 * 1024 / k) & ~(size_t)1023 : (size_t)0; };
  // footprint of one step: populations (two arrays for AB) and adjacency,
  // against the 256 MiB memory-side cache of the MI355X (LBM_SPARSE_NT=0|1
  // overrides)
  const size_t esize = h->storage == LBM_STORE_F64 ? 8 : 4;
  const size_t nq = (size_t)h->n * h->q;
  const size_t bytes = nq * (esize * (h->adjacency_mode == 1 ? 1 : 2) + 4);
  h->nt = env_int("LBM_SPARSE_NT", bytes > ((size_t)256 << 20) ? 1 : 0) != 0;
  // the small capped even shape is for grids that stream from HBM; cached
  // grids are small enough that the cap leaves the GPU partly idle
  const bool big = h->nt && h->storage == LBM_STORE_F64;
  h->even_bx = clamp_bx(env_int("LBM_SPARSE_EVEN_BLOCK_X", big ? 128 : 256));
  h->even_lds = lds_for(env_int("LBM_SPARSE_EVEN_BLOCKS_PER_CU", big ? 4 : 0));
  h->step_bx = clamp_bx(env_int("LBM_SPARSE_BLOCK_X", 256));
  h->step_lds = lds_for(env_int("LBM_SPARSE_BLOCKS_PER_CU", 0));
  h->push_bx = clamp_bx(env_int("LBM_SPARSE_BLOCK_X", big ? 128 : 256));
  h->push_lds = lds_for(env_int("LBM_SPARSE_BLOCKS_PER_CU", big ? 4 : 0));
}

template <int Q>
void launch_compress(const lbm_sparse* h) {
  const dim3 g((unsigned)h->groups), b(kGroup);
  if (h->layout == LBM_LAYOUT_SOA)
    hipLaunchKernelGGL((k_sparse_compress<Q, LBM_LAYOUT_SOA>), g, b, 0, h->stream, h->adj, h->code,
                       h->table, h->raw, h->n);
  else
    hipLaunchKernelGGL((k_sparse_compress<Q, LBM_LAYOUT_AOS>), g, b, 0, h->stream, h->adj, h->code,
                       h->table, h->raw, h->n);
}

// Device copy of the adjacency and its compressed form.  Waits for both: later
// steps may run on another stream.
lbm_status upload_adjacency(lbm_sparse* h, const int32_t* adjacency) {
  const size_t nq = (size_t)h->n * h->q;
  h->groups = (h->n + kGroup - 1) / kGroup;
  // Short lists are bound by latency and one more dependent load costs more than
  // the traffic it saves.  Reference pipes, D3Q19, caller's table / compressed,
  // us per step: FP64 103k nodes (simulationSize 1.75) push 8.0 / 7.9, pull 8.2 /
  // 8.0, 153k (2) AA 9.6 / 9.2, push 10.5 / 10.4, pull 11.4 / 10.7, 1.15M (4) 66.6
  // / 54.3, 74.6 / 64.9, 87.2 / 76.6; FP32 153k push 7.2 / 7.5, 296k (2.5) push
  // 12.6 / 11.4, pull 12.6 / 11.5.  LBM_SPARSE_COMPRESS=0|1 overrides.
  const char* env = std::getenv("LBM_SPARSE_COMPRESS");
  const size_t esize = h->storage == LBM_STORE_F64 ? 8 : 4;
  bool compress = env ? env[0] != '0' : h->n * esize >= 1100000;
  // one allocation: the caller's table, codes, tables of distances, raw flags
  const size_t words = h->q == 19 ? code_words<19>() : code_words<27>();
  auto pad = [](size_t b) { return (b + 255) / 256 * 256; };
  const size_t adj_b = pad(sizeof(int32_t) * nq),
               code_b = pad(sizeof(uint32_t) * words * h->groups * kGroup),
               table_b = pad(sizeof(int32_t) * h->groups * h->q * kDeltas),
               raw_b = pad(sizeof(uint32_t) * h->groups);
  // no room for the compressed form: the caller's table alone serves
  if (compress && hipMalloc(&h->adj, adj_b + code_b + table_b + raw_b) != hipSuccess) {
    (void)hipGetLastError();
    h->adj = nullptr;
    compress = false;
  }
  if (!compress && hipMalloc(&h->adj, adj_b) != hipSuccess) {
    h->adj = nullptr;
    set_error("lbm_sparse_create: hipMalloc of the adjacency failed");
    return LBM_ERR_OOM;
  }
  if (compress) {
    char* p = (char*)h->adj + adj_b;
    h->code = (uint32_t*)p;
    h->table = (int32_t*)(p + code_b);
    h->raw = (uint32_t*)(p + code_b + table_b);
  }
  hipError_t e = hipMemcpy(h->adj, adjacency, sizeof(int32_t) * nq, hipMemcpyHostToDevice);
  if (e == hipSuccess && compress) {
    if (h->q == 19) launch_compress<19>(h);
    else launch_compress<27>(h);
    e = hipGetLastError();
    if (e == hipSuccess) e = hipStreamSynchronize(h->stream);
  }
  if (e != hipSuccess) {
    set_error("lbm_sparse_create: adjacency copy failed: %s", hipGetErrorString(e));
    return LBM_ERR_HIP;
  }
  return LBM_OK;
}

lbm_status check_range(const lbm_sparse* h, int64_t start, int64_t count) {
  LBM_REQUIRE(start >= 0 && count >= 0 && start + count <= h->n, LBM_ERR_ARG,
              "fluid range [%lld, %lld) outside [0, %lld)", (long long)start,
              (long long)(start + count), (long long)h->n);
  return LBM_OK;
}

// The two mass-reduction launches of a range into `partial` (nb entries) and
// `out`, on the handle's stream.  Shared by the allocating and the
// allocation-free entry points, so both give the same bits.
lbm_status launch_mass(const lbm_sparse* h, const void* dstrb, int64_t start, int64_t count,
                       double* partial, int64_t nb, double* out) {
  if (nb > 0) {
    const Shape g{(unsigned)nb, (unsigned)kMassBlock, 0, 0};
    if (h->storage == LBM_STORE_F64)
      launch_qt<k_sparse_mass_partial_fn, double>(h, g, (const double*)dstrb, h->n, start, count,
                                                  partial);
    else
      launch_qt<k_sparse_mass_partial_fn, float>(h, g, (const float*)dstrb, h->n, start, count,
                                                 partial);
    LBM_LAUNCH_CHECK();
  }
  hipLaunchKernelGGL(k_sparse_mass_final, dim3(1), dim3(kMassBlock), 0, h->stream,
                     (const double*)partial, nb, out);
  LBM_LAUNCH_CHECK();
  return LBM_OK;
}

int64_t mass_blocks(int64_t count) { return (count + kMassChunk - 1) / kMassChunk; }

// Device address of `scratch` on the current device, looked up once per device
// (at lbm_sparse_create, or at the first allocation-free call on a device).
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
double* g_scratch_ptr[kMaxDevices] = {};

lbm_status scratch_on_current_device(double** out) {
  int dev = 0;
  LBM_HIP_CHECK(hipGetDevice(&dev));
  LBM_REQUIRE(dev >= 0 && dev < kMaxDevices, LBM_ERR_UNSUPPORTED, "device %d beyond %d", dev,
              kMaxDevices);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    LBM_HIP_CHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    LBM_REQUIRE(p, LBM_ERR_HIP, "no device address for the mass scratch on device %d", dev);
    g_scratch_ptr[dev] = static_cast<double*>(p);
  }
  *out = g_scratch_ptr[dev];
  return LBM_OK;
}

// true when the device can read and write *p: device, managed or pinned host memory
bool device_accessible(const void* p) {
  hipPointerAttribute_t attr{};
  if (hipPointerGetAttributes(&attr, p) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return attr.type == hipMemoryTypeDevice || attr.type == hipMemoryTypeManaged ||
         attr.type == hipMemoryTypeHost || attr.type == hipMemoryTypeUnified;
}

}  // namespace

extern "C" {

lbm_status lbm_sparse_create(const lbm_sparse_config* cfg, lbm_sparse** out) {
  LBM_REQUIRE(cfg && out, LBM_ERR_ARG, "lbm_sparse_create: null pointer");
  *out = nullptr;
  LBM_REQUIRE(cfg->q == 19 || cfg->q == 27, LBM_ERR_ARG, "lbm_sparse_create: q must be 19 or 27");
  LBM_REQUIRE(cfg->layout == LBM_LAYOUT_SOA || cfg->layout == LBM_LAYOUT_AOS, LBM_ERR_ARG,
              "lbm_sparse_create: bad layout %d", cfg->layout);
  LBM_REQUIRE(cfg->storage == LBM_STORE_F64 || cfg->storage == LBM_STORE_F32, LBM_ERR_ARG,
              "lbm_sparse_create: storage must be LBM_STORE_F64 or LBM_STORE_F32");
  LBM_REQUIRE(cfg->n_fluid > 0 && cfg->adjacency, LBM_ERR_ARG,
              "lbm_sparse_create: need n_fluid > 0 and an adjacency");
  LBM_REQUIRE(cfg->n_fluid * cfg->q < ((int64_t)1 << 31), LBM_ERR_ARG,
              "lbm_sparse_create: n_fluid * q must fit the int32 adjacency");
  const int64_t nq = cfg->n_fluid * cfg->q;
  // every entry in [0, nq): first without a branch (negative ones wrap to large
  // ones), then, if one is not, which
  uint32_t bad = 0;
  for (int64_t k = 0; k < nq; k++) bad |= (uint32_t)cfg->adjacency[k] >= (uint32_t)nq;
  for (int64_t k = 0; bad && k < nq; k++)
    LBM_REQUIRE(cfg->adjacency[k] >= 0 && cfg->adjacency[k] < nq, LBM_ERR_ARG,
                "lbm_sparse_create: adjacency[%lld] = %d outside [0, %lld)", (long long)k,
                cfg->adjacency[k], (long long)nq);
  lbm_sparse* h = new lbm_sparse;
  h->n = cfg->n_fluid;
  h->q = cfg->q;
  h->layout = cfg->layout;
  h->storage = cfg->storage;
  h->adjacency_mode = cfg->adjacency_mode;
  h->omega = cfg->omega;
  for (int d = 0; d < 3; d++) h->force[d] = cfg->force[d];
  set_shapes(h);
  {
    const char* e = std::getenv("LBM_SPARSE_XCD");
    h->xcd_env = e ? std::max(0, std::min(4096, std::atoi(e))) : -1;
  }
  if (lbm_status st = upload_adjacency(h, cfg->adjacency)) {
    if (h->adj) (void)hipFree(h->adj);
    delete h;
    return st;
  }
  double* scr = nullptr;  // set-up of lbm_sparse_mass_noalloc's scratch on this device
  if (lbm_status st = scratch_on_current_device(&scr)) {
    if (h->adj) (void)hipFree(h->adj);
    delete h;
    return st;
  }
  *out = h;
  return LBM_OK;
}

lbm_status lbm_sparse_destroy(lbm_sparse* h) {
  if (!h) return LBM_OK;
  // kernels still queued on the handle's stream read the adjacency
  (void)hipStreamSynchronize(h->stream);
  if (h->adj) LBM_HIP_CHECK(hipFree(h->adj));
  delete h;
  return LBM_OK;
}

lbm_status lbm_sparse_aa_even(lbm_sparse* h, void* dstrb, int64_t start, int64_t count) {
  LBM_REQUIRE(h && dstrb, LBM_ERR_ARG, "lbm_sparse_aa_even: null pointer");
  if (lbm_status st = check_range(h, start, count)) return st;
  if (count == 0) return LBM_OK;
  const Shape g = even_shape(h, start, count);
  if (h->storage == LBM_STORE_F64)
    launch_qt<k_sparse_aa_even_fn, double>(h, g, (double*)dstrb, h->n, start, count, h->omega,
                                          h->force[0], h->force[1], h->force[2], g.group);
  else
    launch_qt<k_sparse_aa_even_fn, float>(h, g, (float*)dstrb, h->n, start, count, h->omega,
                                         (float)h->force[0], (float)h->force[1],
                                         (float)h->force[2], g.group);
  LBM_LAUNCH_CHECK();
  return LBM_OK;
}

lbm_status lbm_sparse_aa_odd(lbm_sparse* h, void* dstrb, int64_t start, int64_t count) {
  LBM_REQUIRE(h && dstrb, LBM_ERR_ARG, "lbm_sparse_aa_odd: null pointer");
  LBM_REQUIRE(h->adjacency_mode == 1, LBM_ERR_STATE,
              "lbm_sparse_aa_odd: AA needs the x - c_s adjacency (adjacency_mode 1)");
  if (lbm_status st = check_range(h, start, count)) return st;
  if (count == 0) return LBM_OK;
  const Shape g = step_shape(h, start, count);
  if (h->storage == LBM_STORE_F64)
    launch_adj<k_sparse_aa_odd_fn, k_sparse_aa_odd_raw_fn, double>(h, g, (double*)dstrb, h->tables(), h->n,
                                         start, count, h->omega, h->force[0], h->force[1],
                                         h->force[2], g.group);
  else
    launch_adj<k_sparse_aa_odd_fn, k_sparse_aa_odd_raw_fn, float>(h, g, (float*)dstrb, h->tables(), h->n, start,
                                        count, h->omega, (float)h->force[0], (float)h->force[1],
                                        (float)h->force[2], g.group);
  LBM_LAUNCH_CHECK();
  return LBM_OK;
}

lbm_status lbm_sparse_ab(lbm_sparse* h, const void* src, void* tgt, int64_t start, int64_t count,
                         int32_t pull) {
  LBM_REQUIRE(h && src && tgt, LBM_ERR_ARG, "lbm_sparse_ab: null pointer");
  LBM_REQUIRE(src != tgt, LBM_ERR_ARG, "lbm_sparse_ab: source and target must differ");
  LBM_REQUIRE(h->adjacency_mode == (pull ? 1 : 0), LBM_ERR_STATE,
              "lbm_sparse_ab: %s needs adjacency_mode %d", pull ? "pull" : "push", pull ? 1 : 0);
  LBM_REQUIRE(!pull || h->layout == LBM_LAYOUT_SOA, LBM_ERR_UNSUPPORTED,
              "lbm_sparse_ab: the reference has no AOS pull kernel");
  if (lbm_status st = check_range(h, start, count)) return st;
  if (count == 0) return LBM_OK;
  const Shape g = step_shape(h, start, count, !pull);
  const AdjTables adj = h->tables();
  if (h->storage == LBM_STORE_F64) {
    if (pull)
      launch_adj<k_sparse_ab_pull_fn, k_sparse_ab_pull_raw_fn, double>(h, g, (const double*)src, (double*)tgt, adj, h->n,
                                            start, count, h->omega, h->force[0], h->force[1],
                                            h->force[2], g.group);
    else
      launch_adj<k_sparse_ab_push_fn, k_sparse_ab_push_raw_fn, double>(h, g, (const double*)src, (double*)tgt, adj, h->n,
                                            start, count, h->omega, h->force[0], h->force[1],
                                            h->force[2], g.group);
  } else {
    const float F0 = (float)h->force[0], F1 = (float)h->force[1], F2 = (float)h->force[2];
    if (pull)
      launch_adj<k_sparse_ab_pull_fn, k_sparse_ab_pull_raw_fn, float>(h, g, (const float*)src, (float*)tgt, adj, h->n,
                                           start, count, h->omega, F0, F1, F2, g.group);
    else
      launch_adj<k_sparse_ab_push_fn, k_sparse_ab_push_raw_fn, float>(h, g, (const float*)src, (float*)tgt, adj, h->n,
                                           start, count, h->omega, F0, F1, F2, g.group);
  }
  LBM_LAUNCH_CHECK();
  return LBM_OK;
}

lbm_status lbm_sparse_init_rest(lbm_sparse* h, void* dstrb, int32_t aa) {
  LBM_REQUIRE(h && dstrb, LBM_ERR_ARG, "lbm_sparse_init_rest: null pointer");
  const Shape g{grid_for(h->n), 256, 0};
  if (h->storage == LBM_STORE_F64)
    launch_qt<k_sparse_init_rest_fn, double>(h, g, (double*)dstrb, h->n, (int)aa);
  else
    launch_qt<k_sparse_init_rest_fn, float>(h, g, (float*)dstrb, h->n, (int)aa);
  LBM_LAUNCH_CHECK();
  return LBM_OK;
}

lbm_status lbm_sparse_mass(lbm_sparse* h, const void* dstrb, int64_t start, int64_t count,
                           double* mass) {
  LBM_REQUIRE(h && dstrb && mass, LBM_ERR_ARG, "lbm_sparse_mass: null pointer");
  if (lbm_status st = check_range(h, start, count)) return st;
  const int64_t nb = mass_blocks(count);
  double* partial = nullptr;
  LBM_HIP_CHECK(hipMalloc(&partial, sizeof(double) * (nb + 1)));
  lbm_status st = launch_mass(h, dstrb, start, count, partial, nb, partial + nb);
  hipError_t e = hipSuccess;
  if (st == LBM_OK) e = hipMemcpyAsync(mass, partial + nb, sizeof(double), hipMemcpyDeviceToHost,
                                       h->stream);
  if (st == LBM_OK && e == hipSuccess) e = hipStreamSynchronize(h->stream);
  (void)hipFree(partial);
  if (st != LBM_OK) return st;
  if (e != hipSuccess) {
    set_error("lbm_sparse_mass: %s", hipGetErrorString(e));
    return LBM_ERR_HIP;
  }
  LBM_REQUIRE(std::isfinite(*mass), LBM_ERR_NUMERIC, "lbm_sparse_mass: mass is not finite (%g)",
              *mass);
  return LBM_OK;
}

lbm_status lbm_sparse_mass_noalloc(lbm_sparse* h, const void* dstrb, int64_t start,
                                   int64_t count, double* mass_device) {
  LBM_REQUIRE(h && dstrb && mass_device, LBM_ERR_ARG, "lbm_sparse_mass_noalloc: null pointer");
  if (lbm_status st = check_range(h, start, count)) return st;
  const int64_t nb = mass_blocks(count);
  LBM_REQUIRE(nb <= kMassScratchPartials, LBM_ERR_ARG,
              "lbm_sparse_mass_noalloc: %lld nodes exceed the fixed scratch (at most %lld nodes "
              "per call); use lbm_sparse_mass or split the range",
              (long long)count, (long long)(kMassScratchPartials * kMassChunk));
  LBM_REQUIRE(device_accessible(dstrb) && device_accessible(mass_device), LBM_ERR_ARG,
              "lbm_sparse_mass_noalloc: the populations and the result must be device-accessible "
              "memory (device, managed or pinned host)");
  double* scr = nullptr;
  if (lbm_status st = scratch_on_current_device(&scr)) return st;
  return launch_mass(h, dstrb, start, count, scr, nb, mass_device);
}

lbm_status lbm_sparse_synchronize(lbm_sparse* h) {
  LBM_REQUIRE(h, LBM_ERR_ARG, "lbm_sparse_synchronize: null handle");
  LBM_HIP_CHECK(hipStreamSynchronize(h->stream));
  return LBM_OK;
}

// Later launches go to `stream` (NULL: the null stream).  Waits for the work
// already enqueued on the previous stream, so the order of calls is kept.
lbm_status lbm_sparse_set_stream(lbm_sparse* h, void* stream) {
  LBM_REQUIRE(h, LBM_ERR_ARG, "lbm_sparse_set_stream: null handle");
  LBM_HIP_CHECK(hipStreamSynchronize(h->stream));
  h->stream = (hipStream_t)stream;
  return LBM_OK;
}

}  // extern "C"
