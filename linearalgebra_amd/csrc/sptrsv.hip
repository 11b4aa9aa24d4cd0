// Sparse triangular solves on gfx950 and the ILU(k)/IC(k) apply.
//
// Analysis (host): level sets by TopologicalSort2
// (sparse_mat_op/matrix_utils.hpp:637-675); the triangle is stored with its
// rows in level order (the reference's permuteRow in
// OptimizedTriangularSolve::analysis, triangle_solve.tpp:87-91) so each
// level is a contiguous, coalesced stream; columns keep original ids.
//
// Solve, two modes:
//  * LEVEL: one launch per level (the Barrier mode, triangle_solve.tpp:
//    127-155), captured once into a HIP graph and replayed.
//  * SYNCFREE: one launch; workgroups claim chunks of rows in level order
//    from an atomic ticket (the NoBarrier mode, triangle_solve.tpp:157-187).
//    x is pre-filled with a sentinel; a row waits until each x_j it reads is
//    no longer the sentinel (value and readiness in one word) and publishes
//    its own x_i the same way. Chunks never span levels, so rows inside one
//    workgroup never wait on each other, and every wait is on an earlier
//    ticket, which a running workgroup already holds: the solve always
//    drains. Waits are bounded; a timeout sets an error flag instead of
//    hanging.
//  * JACOBI (no counterpart in the reference): k Jacobi sweeps on the
//    triangle, y_0 = D^-1 b, y_{s+1} = D^-1 (b - N y_s), each sweep an
//    SpMV with the column-scaled strict triangle N D^-1. D^-1 N is nilpotent (its
//    index is the number of levels), so k >= levels - 1 sweeps give the
//    exact solution; fewer give the truncated Neumann series, an
//    approximate solve whose cost is k bandwidth-bound passes instead of a
//    chain of level-to-level dependencies (Anzt, Chow, Dongarra, "Iterative
//    sparse triangular solves for preconditioning", Euro-Par 2015). For an
//    IC factor both triangles use the same k, so the applied operator
//    P_k^T P_k stays symmetric positive definite and PCG stays valid.
// Row formula (triangle_solve.hpp:32-71): x_i = (b_i - sum_j T_ij x_j) / d_i,
// computed as a product with 1/d_i stored in the plan (within an ulp of the
// quotient; keeps a divide off the sync-free dependency chain).
#include <algorithm>
#include <climits>
#include <cstdlib>
#include <type_traits>

#include "dev_util.hpp"
#include "device.hpp"
#include "host_algos.hpp"

namespace laamd {
using namespace dev;

namespace {
constexpr int kB = 256;

template <typename T>
__device__ __forceinline__ auto ldt(const T *p, int64_t i) {
  return ldm(p, i);
}

template <int G, typename T, typename V, typename A, bool DIAG>
__global__ __launch_bounds__(kB) void k_trsv_level(int k0, int k1, const int *__restrict__ rowptr,
                                                   const int *__restrict__ col,
                                                   const T *__restrict__ val,
                                                   const T *__restrict__ diag,
                                                   const int *__restrict__ perm,
                                                   const V *__restrict__ b, V *x) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * kB + threadIdx.x;
  const int64_t k = k0 + t / G;
  const int sub = threadIdx.x & (G - 1);
  if (k >= k1) return;
  const int rs = rowptr[k], re = rowptr[k + 1];
  A acc = 0;
  for (int q = rs + sub; q < re; q += G) acc += A(ldt(val, q)) * A(x[ldi(col, q)]);
  acc = group_sum<G>(acc);
  if (sub == 0) {
    const int r = perm[k];
    A v = A(b[r]) - acc;
    if constexpr (DIAG) v = v * A(ldt(diag, k));
    x[r] = V(v);
  }
}

// x <- sentinel everywhere; the control words ctl[0..15] (ctl[0]: ticket,
// ctl[1]: owning XCD + 1) reset for the next sync-free solve.
template <typename V>
__global__ void k_fill_sentinel(int64_t n, V *x, unsigned *ctl) {
  using U = typename Sentinel<V>::U;
  U *xb = reinterpret_cast<U *>(x);
  for (int64_t t = static_cast<int64_t>(blockIdx.x) * kB + threadIdx.x; t < n;
       t += static_cast<int64_t>(gridDim.x) * kB)
    xb[t] = Sentinel<V>::bits;
  if (blockIdx.x == 0 && threadIdx.x < 16) ctl[threadIdx.x] = 0;
}

// Sync-free solve. Readiness is polled with agent-scope relaxed loads (they
// bypass the CU's L1).
//  XLOCAL = true: confined to one XCD. The first workgroup to start claims
//    its XCD (device-coherent CAS on ctl[1]); workgroups that land on another
//    XCD leave at once. Results are published with plain stores into that
//    XCD's L2, where the agent-scope polls of the same XCD see them: about
//    0.3 us from store to poll on MI355X, against 0.55 us when producer and
//    consumer sit on different XCDs.
//  XLOCAL = false: every XCD takes part; results are published with
//    agent-scope stores so polls from any XCD see them.
// A workgroup claims one chunk ticket from ctl[0] at a time (one device
// atomic per NT/G rows; the tickets of one counter are handed out about
// 12 ns apart, so a per-wavefront ticket would bound wide levels). Chunks
// are in level order. A wait longer than kWaitTicks of the 100 MHz
// real-time clock sets *err and gives up; every other waiter checks *err
// every 256 polls and gives up too, so the kernel always drains quickly.
constexpr uint64_t kWaitTicks = 20000000;  // 0.2 s

// a wait ran out of time: *err for the polling wavefronts, and the host's copy
// (its address sits behind the flag), which trsv_check_timeout reads
__device__ __forceinline__ void flag_late(int *err) {
  __hip_atomic_fetch_or(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  int *const host = *reinterpret_cast<int *const *>(err + 2);
  __hip_atomic_store(host, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// One row of a sync-free solve, G lanes: wait for each x_j, accumulate,
// publish x_r. `sub` is the lane's index inside its group.
template <int G, typename T, typename V, typename A, bool DIAG, bool XLOCAL>
__device__ __forceinline__ void sf_row(int k, int sub, const int *__restrict__ rowptr,
                                       const int *__restrict__ col, const T *__restrict__ val,
                                       const T *__restrict__ diag, const int *__restrict__ perm,
                                       const V *__restrict__ b, V *x, int *err) {
  using U = typename Sentinel<V>::U;
  // everything that does not depend on x first
  const int rs = rowptr[k], re = rowptr[k + 1];
  const int r = perm[k];
  const A bb = A(b[r]);
  A dd = A(1);
  if constexpr (DIAG) dd = A(ldt(diag, k));
  A acc = 0;
  bool gave_up = false;
  // one entry per lane at a time: a lane that loads only entries of its own
  // row issues no extra request (the polls below go to the memory side, and
  // their count is what the solve pays for)
  for (int q = rs + sub; q < re; q += G) {
    const int j = ldi(col, q);
    const A a = A(ldt(val, q));
    V xv = load_ready(x + j);
    if (is_sentinel(xv) && !gave_up) {
      const uint64_t t0 = __builtin_amdgcn_s_memrealtime();
      unsigned polls = 0;
      while (is_sentinel(xv)) {
        __builtin_amdgcn_s_sleep(1);
        xv = load_ready(x + j);
        if ((++polls & 255u) == 0) {
          if (__hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0 ||
              __builtin_amdgcn_s_memrealtime() - t0 > kWaitTicks) {
            gave_up = true;
            break;
          }
        }
      }
    }
    acc += a * A(is_sentinel(xv) ? V(0) : xv);
  }
  if (gave_up) flag_late(err);
  acc = group_sum<G>(acc);
  if (sub == 0) {
    A v = bb - acc;
    if constexpr (DIAG) v = v * dd;
    U o = to_bits<V>(V(v));
    if (o == Sentinel<V>::bits) o = Sentinel<V>::qnan;
    if constexpr (XLOCAL)
      __hip_atomic_store(reinterpret_cast<U *>(x + r), o, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_WORKGROUP);
    else
      __hip_atomic_store(reinterpret_cast<U *>(x + r), o, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
  }
}

template <int G, int NT, typename T, typename V, typename A, bool DIAG, bool XLOCAL>
__global__ __launch_bounds__(NT) void k_trsv_syncfree(
    int nchunks, const int *__restrict__ chunk_start, const int *__restrict__ rowptr,
    const int *__restrict__ col, const T *__restrict__ val, const T *__restrict__ diag,
    const int *__restrict__ perm, const V *__restrict__ b, V *x, unsigned *ctl, int *err) {
  if constexpr (XLOCAL) {
    __shared__ int s_go;
    if (threadIdx.x == 0) {
      const unsigned me = xcc_id() + 1;
      const unsigned prev = atomicCAS(&ctl[1], 0u, me);
      s_go = (prev == 0u || prev == me) ? 1 : 0;
    }
    __syncthreads();
    if (!s_go) return;
  }
  // row of this lane group inside a chunk of NT/G rows
  const int gi = static_cast<int>(threadIdx.x) / G, sub = threadIdx.x & (G - 1);
  // two ticket slots: while a chunk is solved, thread 0 already claims the
  // next ticket into the other slot, so the claim's round trip overlaps the
  // work; one barrier per chunk. Holding one ticket ahead keeps the drain
  // argument: the lowest unfinished chunk is either some workgroup's
  // current chunk or the next one of a workgroup whose current chunk is
  // finished.
  __shared__ int s_c[2];
  if (threadIdx.x == 0) s_c[0] = static_cast<int>(atomicAdd(&ctl[0], 1u));
  __syncthreads();
  for (int it = 0;; ++it) {
    const int c = s_c[it & 1];
    if (c >= nchunks) break;
    if (threadIdx.x == 0) s_c[(it + 1) & 1] = static_cast<int>(atomicAdd(&ctl[0], 1u));
    const int k = chunk_start[c] + gi;
    if (k < chunk_start[c + 1])
      sf_row<G, T, V, A, DIAG, XLOCAL>(k, sub, rowptr, col, val, diag, perm, b, x, err);
    __syncthreads();
  }
}

// ------------------------------------------------------- tiled schedule
// One workgroup per tile (see tiling.cpp). Wavefront 0, the solver, takes
// the tile's groups (at most 64 rows of one level each) in level order, one
// lane per row (or RL lanes), reading every x_j from LDS: its own results,
// kept in a ring of `ring` groups, or the values of other tiles (the halo).
// What bounds it is the number of instructions it issues per group: it is
// alone on its dependency chain, one wavefront issues at most about one
// instruction per 4-5 cycles, and a scattered access costs it about 64
// cycles of address processing. So everything but the chain is done by the
// other wavefronts:
//  * wavefronts 1..H, the fetchers: poll the values of other tiles that each
//    group reads first (agent-scope loads) into the halo. Blocks of NB
//    consecutive groups go round the fetchers; a fetcher polls a block's
//    values together, one lane per value, and counts the groups whose values
//    have all arrived in s_prog. Halo slots are never reused within a tile,
//    so the fetchers run ahead freely.
//  * the last kTileIo wavefronts: gather b (by row id) into a ring in LDS
//    ahead of the solver, store its results to x (by row id) behind it, and
//    touch the cache lines of the row data it will load next, so that those
//    loads find them in the L2. A block of kTileDepth groups at a time.
// The solver loads its row data (values, LDS addresses, 1/d: one packed
// record per group, every load contiguous over the lanes) into registers
// kTileDepth groups ahead, and hands the rows that other tiles read over in
// `mail`: mstride slots per group, the group's shared rows first, so one
// group's hand-over is one short contiguous store and its readers poll one
// or two lines instead of a line per row. x itself is not polled by anyone.
// A wavefront's LDS accesses are carried out in the order it issues them, so
// the solver needs no wait after its own writes (a compiler-only fence keeps
// the order in the code); the others wait for their LDS writes before they
// report. Every wait on another tile is bounded like the level-chunk
// kernel's; a timeout sets *err.
// Measured per apply of both triangles, this form against one whose solver
// issued every access but the polls, and whose tiles polled x: 128^3 7-point
// IC(0) FP64 425 -> 290 us, FP32 in natural order 631 -> 253 us; 100x96x90
// FP64 494 -> 200 us; 512^2 FP64 569 -> 372 us; 128^2 225 -> 171 us; 27-point
// ILU(1) 56^3 FP32 740 -> 447 us, 90^3 FP64 1470 -> 929 us (with larger tiles,
// smaller records and one synchronisation per apply now 259, 225, 172, 303, 85,
// 407 and 736 us in this order, repeated on the same vectors; with others on
// each pass 271 us for the first and 426 us for the sixth). A group takes the
// solver 0.12 us (0.245 us before), and a hand-over about 1 us at the
// median; the chain of hand-overs between tiles and of groups inside them is
// what bounds the solve now. (With the hand-over slots alone the 3-D solves
// gained 20-40%, but 512^2 lost 8%: one more store per group on the solver.)
constexpr int kTileLanes = 64;
constexpr int kTileIo = 2;     // I/O wavefronts
// bytes of LDS control words, ahead of the slots (where b is staged no more
// than they need: the halo is wide)
constexpr int tile_ctl(bool staged) { return staged ? 40 : 64; }
// Groups of padding the packed rows end with (the solver runs up to
// kTileDepth - 1 groups past a tile's last one and loads kTileDepth ahead),
// and mail slots' spare groups per tile for the same reason.
constexpr int kTilePad = 2 * kTileDepth;
constexpr int kTileNever = INT_MAX / 2;  // "all groups ready"

__device__ __forceinline__ void lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup", "local");
}
__device__ __forceinline__ void code_order() { __atomic_signal_fence(__ATOMIC_SEQ_CST); }
__device__ __forceinline__ int lds_load(const int *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void lds_store(int *p, int v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// A group's packed record: E values, E LDS addresses and 1/d per lane. Values
// and addresses are cut into pieces of at most 16 bytes per lane, piece by
// piece for all 64 lanes, so that every load covers one contiguous run. Issuing
// the loads is a quarter of the solving wavefront's time (128^2, FP64: 273
// cycles a group, 200-210 without them; the LDS write, read and four
// multiply-adds take the rest), so with two FP64 values per lane 1/d sits in the
// addresses' piece: two loads a group instead of four (5-point IC(0) per
// apply, FP64: 128^2 94.4 -> 84.8 us, 512^2 338 -> 303 us). An
// address is a byte address in 32 bits, ready to use; with eight values per
// lane it is a slot number in 16 bits, which takes half the registers (eight
// FP64 values at kTileDepth groups spilled otherwise: 256 are all a wavefront
// of these workgroups gets) and one load less (27-point ILU(1) per apply: 90^3
// FP64 921 -> 762 us, 56^3 FP32 451 -> 438 us).
template <int E, typename T>
struct TileRec {
  static constexpr bool kWide = E < 8;
  using Code = std::conditional_t<kWide, uint32_t, uint16_t>;
  // from an LDS byte address
  static __host__ __device__ Code code(int a) { return static_cast<Code>(kWide ? a : a / 8); }
  static __device__ uint32_t address(Code c) { return kWide ? c : static_cast<uint32_t>(c) * 8u; }
  static constexpr int kVal = E * static_cast<int>(sizeof(T));
  static constexpr int kValPiece = kVal < 16 ? kVal : 16;
  static constexpr int kCode = E * static_cast<int>(sizeof(Code));
  static constexpr bool kJoined = E == 2 && sizeof(T) == 8;  // 1/d behind the addresses
  static constexpr int kCodePiece = kJoined || kCode > 16 ? 16 : kCode;
  static constexpr int kCodeAt = kTileLanes * kVal;
  static constexpr int kDinvAt = kCodeAt + (kJoined ? kCode : kTileLanes * kCode);
  static constexpr int kDinvStep = kJoined ? kCodePiece : static_cast<int>(sizeof(T));
  static constexpr int kBytes =
      kCodeAt + kTileLanes * (kJoined ? kCodePiece : kCode + static_cast<int>(sizeof(T)));
  static_assert(kBytes % 128 == 0, "whole cache lines");
};

typedef unsigned int tile_u2 __attribute__((ext_vector_type(2)));
typedef unsigned int tile_u4 __attribute__((ext_vector_type(4)));
// `total` bytes per lane in pieces of `piece` bytes; base is the same for
// every lane
template <int total, int piece>
__device__ __forceinline__ void ld_pieces(const char *base, unsigned lane, void *out) {
  static_assert(piece == 4 || piece == 8 || piece == 16, "piece size");
#pragma unroll
  for (int q = 0; q < total / piece; ++q) {
    if constexpr (piece == 4)
      reinterpret_cast<unsigned *>(out)[q] = __builtin_nontemporal_load(
          reinterpret_cast<const unsigned *>(base + q * piece * kTileLanes + lane * 4u));
    else if constexpr (piece == 16)
      reinterpret_cast<tile_u4 *>(out)[q] = __builtin_nontemporal_load(
          reinterpret_cast<const tile_u4 *>(base + q * piece * kTileLanes + lane * 16u));
    else
      reinterpret_cast<tile_u2 *>(out)[q] = __builtin_nontemporal_load(
          reinterpret_cast<const tile_u2 *>(base + q * piece * kTileLanes + lane * 8u));
  }
}

template <typename T> struct TileDt;
template <> struct TileDt<double> { static constexpr la_dtype v = LA_F64; };
template <> struct TileDt<float> { static constexpr la_dtype v = LA_F32; };
template <> struct TileDt<bf16> { static constexpr la_dtype v = LA_BF16; };

template <typename T> __device__ __forceinline__ float tile_val(T v) { return float(v); }
template <> __device__ __forceinline__ float tile_val<bf16>(bf16 v) {
  return __uint_as_float(static_cast<uint32_t>(v.bits) << 16);
}
__device__ __forceinline__ double tile_val(double v) { return v; }

// one pipeline stage: a group's record for this lane
template <int E, typename T, typename V>
struct TileStage {
  alignas(16) T val[E];
  struct alignas(16) Tail {
    typename TileRec<E, T>::Code code[E];
    T dinv;
  } tail;
  V b;  // (only where b is staged)
};

// the LDS word at a byte address (as kept in the packed records)
template <typename V>
__device__ __forceinline__ const __attribute__((address_space(3))) V *lds_at(uint32_t a) {
  return (const __attribute__((address_space(3))) V *)a;
}

// waits until *p exceeds `have`; false after kTilePolls polls, which take at
// least kWaitTicks. No global access on this path: the solver's loads in
// flight are counted in issue order, and a global access here would make the
// compiler wait for all of them; nor a clock, whose read the LDS polls would
// wait for.
constexpr int kTilePolls = 1 << 23;  // at least 60 cycles each
__device__ __forceinline__ bool tile_wait(const int *p, int have) {
  for (int polls = 0; lds_load(p) <= have; ++polls) {
    if (polls == kTilePolls) return false;
    __builtin_amdgcn_s_sleep(0);
  }
  return true;
}

// STAGED: the halo (18424 to 19450 values) leaves no room for a ring of b. b
// then holds the right-hand side in the order of the records (64 slots per
// group, k_tile_stage), which the solver loads along with them: a launch and a
// pass over b more, but the tiles stay. 27-point ILU(1) on 2304 x 6 x 6, lower
// triangle, FP64 / FP32: 464 / 360 us, level chunks 1096 / 977 us (2302 x 6 x 6
// with the ring 452 / 373 us); 7-point on 8 x 8 x 4700 715 / 538 us, level
// chunks 1707 / 1625 us.
template <int E, int RL, int NB, int H, typename T, typename V, typename A, bool DIAG,
          bool STAGED>
__global__ __launch_bounds__(kTileLanes * (1 + H + kTileIo)) void k_trsv_tiled(
    int nparts, const int *__restrict__ gptr, const int2 *__restrict__ rows,
    const char *__restrict__ pack, const int2 *__restrict__ reads, int rstride,
    const V *__restrict__ b, V *__restrict__ x, V *mail, int mstride, int ring, int hmax,
    int touch, unsigned *ctl, int *err) {
  constexpr int D = kTileDepth, kCtl = tile_ctl(STAGED);
  static_assert(D % (NB * H) == 0, "a group's fetcher is fixed by its place in the loop");
  static_assert(kTileIo <= kTileWindow / D, "a block's rows are listed before its results go out");
  using R = TileRec<E, T>;
  // LDS, all of it dynamic so that it starts at address 0 (a record's
  // addresses are then used as they are): control words, then 8-byte slots:
  // results of `ring` groups, the zero slot, the halo, b of `ring` groups
  // (not if staged)
  extern __shared__ __align__(16) unsigned char smem[];
  int *const s_prog = reinterpret_cast<int *>(smem), *const s_b = s_prog + H;
  int &s_part = s_b[kTileIo], &s_late = s_b[kTileIo + 1], &s_done = s_b[kTileIo + 2];
  static_assert((H + kTileIo + 3) * 4 <= kCtl, "control words");
  const int wave = static_cast<int>(threadIdx.x) / kTileLanes;
  const int lane = static_cast<int>(threadIdx.x) % kTileLanes;
  unsigned char *const bring = smem + kCtl + 8 * (ring * kTileLanes + 1 + hmax);
  auto slot = [&](int q) -> V & { return *reinterpret_cast<V *>(smem + kCtl + 8 * q); };
  auto bslot = [&](int q) -> V & { return *reinterpret_cast<V *>(bring + 8 * q); };
  // The next tile's ticket and cleared control words, between two barriers.
  // The loop below must stay one loop of whole wavefronts: thread 0's work on
  // both sides of the back edge with no barrier between would let the
  // compiler send the other threads ahead to the next tile without it.
  auto next_tile = [&] {
    if (threadIdx.x == 0) {
      s_part = static_cast<int>(atomicAdd(&ctl[0], 1u));
      s_late = 0;
      s_done = 0;
    }
    if (threadIdx.x < H) s_prog[threadIdx.x] = 0;
    if (threadIdx.x < kTileIo) s_b[threadIdx.x] = 0;
    __syncthreads();
    return __builtin_amdgcn_readfirstlane(s_part);
  };
  if (threadIdx.x == 0) slot(ring * kTileLanes) = V(0);
  for (int p = next_tile(); p < nparts; p = next_tile()) {
    const int g0 = gptr[p], ng = gptr[p + 1] - g0;
    const int nblk = (ng + D - 1) / D;
    if (wave == 0) {
      __builtin_amdgcn_s_setprio(3);  // issue priority over the other wavefronts
      TileStage<E, T, V> st[D];
      int64_t at = static_cast<int64_t>(g0) * R::kBytes;
      const V *bat = b + static_cast<int64_t>(g0) * kTileLanes;
      auto load_rows = [&](int k) {  // the next group's record
        // (the offset is kept in scalar registers: scalar additions instead
        // of 64-bit vector address arithmetic per load)
        asm volatile("" : "+s"(at));
        const char *rec = pack + at;
        ld_pieces<R::kVal, R::kValPiece>(rec, lane, st[k].val);
        // (a load's registers must all be used: the compiler puts other values
        // into those that are not, and then waits for the load at once)
        if constexpr (R::kJoined && DIAG) {
          static_assert(sizeof(st[k].tail) == R::kCodePiece, "addresses and 1/d in one load");
          ld_pieces<R::kCodePiece, R::kCodePiece>(rec + R::kCodeAt, lane, &st[k].tail);
        } else if constexpr (R::kJoined) {
          *reinterpret_cast<tile_u2 *>(st[k].tail.code) = __builtin_nontemporal_load(
              reinterpret_cast<const tile_u2 *>(rec + R::kCodeAt + lane * 16u));
        } else {
          ld_pieces<R::kCode, R::kCodePiece>(rec + R::kCodeAt, lane, st[k].tail.code);
          if constexpr (DIAG)
            st[k].tail.dinv = *reinterpret_cast<const T *>(
                rec + R::kDinvAt + static_cast<unsigned>(lane) * sizeof(T));
        }
        at += R::kBytes;
        if constexpr (STAGED) {
          st[k].b = __builtin_nontemporal_load(bat + lane);
          bat += kTileLanes;
        }
      };
      // sched_barrier keeps the scheduler from reordering the groups' loads,
      // so that the loads in flight when the loop starts are as old as in
      // any later pass (the compiler's count of loads allowed in flight then
      // stays high)
#pragma unroll
      for (int k = 0; k < D; ++k) {
        load_rows(k);
        __builtin_amdgcn_sched_barrier(0);
      }
      // the group's hand-over slots (each tile has kTileDepth groups of spare
      // ones, so groups past the last one need no test)
      V *mg = mail + (static_cast<int64_t>(g0) + static_cast<int64_t>(p) * D) * mstride;
      const bool shared = lane % RL == 0 && lane / RL < mstride;
      // A group's LDS reads are issued right behind the previous group's
      // write, the fetcher's count first: reads are carried out in order, so
      // values read after a sufficient count are good, and are read again
      // in the rare other case. Hand-over and loads are issued while those
      // reads are on their way.
      V bv, xv[E];
      auto read_row = [&](const TileStage<E, T, V> &g, int bpos) {
        if constexpr (STAGED) bv = g.b;
        else bv = bslot(bpos);
#pragma unroll
        for (int e = 0; e < E; ++e) xv[e] = *lds_at<V>(R::address(g.tail.code[e]));
      };
      if (nblk > 0 && !tile_wait(&s_b[0], 0)) s_late = 1;
      lds_fence();
      int rdy = lds_load(&s_prog[0]), rdb = 0;
      code_order();
      read_row(st[0], lane);
      // groups past the last one (at most D - 1) repeat whatever follows in
      // the arrays; nothing reads their results. A loop without early exits
      // keeps the compiler's count of loads in flight across iterations.
      for (int blk = 0; blk < nblk; ++blk) {
        lds_store(&s_done, blk * D);
        const int base = (blk * D & (ring - 1)) * kTileLanes + lane;
#pragma unroll
        for (int k = 0; k < D; ++k) {
          // the halo values of the group are in LDS once its fetcher has
          // counted it
          constexpr int per = D / (NB * H);  // blocks of a fetcher per pass
          const int f = (k / NB) % H, need = (blk * per + k / (NB * H)) * NB + k % NB;
          if (rdy <= need) {
            if (!tile_wait(&s_prog[f], need)) s_late = 1;
            lds_fence();
            read_row(st[k], base + k * kTileLanes);
          }
          A acc = A(tile_val(st[k].val[0])) * A(xv[0]);
#pragma unroll
          for (int e = 1; e < E; ++e) acc += A(tile_val(st[k].val[e])) * A(xv[e]);
          // a row on RL lanes: every lane gets the same sum (the first
          // lane's result is the one read and published)
          acc = group_sum<RL>(acc);
          A v = A(bv) - acc;
          if constexpr (DIAG) v = v * A(tile_val(st[k].tail.dinv));
          const V out = V(v);
          slot(base + k * kTileLanes) = out;
          code_order();
          if (k == D - 2) rdb = lds_load(&s_b[(blk + 1) % kTileIo]);
          if (k == D - 1 && blk + 1 < nblk && rdb <= (blk + 1) / kTileIo) {
            if (!tile_wait(&s_b[(blk + 1) % kTileIo], (blk + 1) / kTileIo)) s_late = 1;
            lds_fence();
          }
          rdy = lds_load(&s_prog[((k + 1) / NB) % H]);
          code_order();
          read_row(st[(k + 1) % D], k + 1 < D ? base + (k + 1) * kTileLanes
                                              : ((blk + 1) * D & (ring - 1)) * kTileLanes + lane);
          code_order();
          // an arithmetic result is never the sentinel: it is a signalling
          // NaN, and arithmetic returns quiet ones (IEEE mode, the default
          // of every kernel)
          if (shared) store_ready(mg + lane / RL, out);
          mg += mstride;
          load_rows(k);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      lds_store(&s_done, kTileNever);
    } else if (wave <= H) {
      // blocks hw, hw + H, ... of NB groups. A group's list has rstride places
      // (x: its hand-over slot, -1 past the list; y: its halo slot), so a
      // block's places are one run whose address needs no look-up; the lists
      // of the next two blocks are on their way while one is polled
      const int hw = wave - 1, nfb = (ng + NB - 1) / NB, places = NB * rstride;
      const int lane_grp = lane / rstride;
      auto list = [&](int jb, int q) {
        int2 e = make_int2(-1, 0);
        if (jb < nfb && q < places)
          e = reads[(static_cast<int64_t>(g0) + jb * NB) * rstride + q];
        return e;
      };
      int2 next = list(hw, lane), next2 = list(hw + H, lane);
      for (int jb = hw; jb < nfb; jb += H) {
        int2 e = next;
        next = next2;
        next2 = list(jb + 2 * H, lane);
        const int done0 = jb / H * NB;
        int grp = lane_grp, told = 0;  // the place's group; groups reported
        for (int q = lane;; q += kTileLanes) {
          bool pending = e.x >= 0 && jb * NB + grp < ng;
          V xv = V(0);
          if (pending) xv = load_ready(mail + e.x);
          const uint64_t w0 = __builtin_amdgcn_s_memrealtime();
          for (unsigned polls = 1;; ++polls) {
            if (pending && !is_sentinel(xv)) {
              slot(e.y) = xv;
              pending = false;
            }
            const uint64_t left = __ballot(pending);
            if (!left) break;
            if constexpr (NB > 1) {
              const int ready = __builtin_amdgcn_readlane(grp, __builtin_ctzll(left));
              if (ready > told) {
                told = ready;
                lds_fence();
                if (lane == 0) lds_store(&s_prog[hw], done0 + told);
              }
            }
            __builtin_amdgcn_s_sleep(1);
            if ((polls & 255u) == 0 &&
                (__hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0 ||
                 __builtin_amdgcn_s_memrealtime() - w0 > kWaitTicks)) {
              flag_late(err);
              if (pending) slot(e.y) = V(0);
              break;
            }
            if (pending) xv = load_ready(mail + e.x);
          }
          if (q - lane + kTileLanes >= places) break;
          // (rare: more places than lanes)
          e = list(jb, q + kTileLanes);
          grp = (q + kTileLanes) / rstride;
        }
        lds_fence();
        __builtin_amdgcn_wave_barrier();
        if (lane == 0) lds_store(&s_prog[hw], done0 + NB);
      }
      lds_fence();
      if (lane == 0) lds_store(&s_prog[hw], kTileNever);
    } else {
      // blocks io, io + kTileIo, ... of D groups. b of a block goes into the
      // ring once the results of the block that held its place `ring` groups
      // earlier are in x; the gather of the next block of this wavefront is
      // issued before that wait. The solver's progress ends every wait here.
      // A block's rows are listed by row id (x: the row, -1 past the last; y:
      // its place in the block), so that neighbouring rows of b and x, which
      // sit in different groups of the block, are accessed together: in a
      // natural-order grid 8 runs of 8 rows per access instead of 64 single
      // rows. Every line of such an access costs the CU's address unit a
      // cycle or more that the polls and the solver's loads wait for.
      const int io = wave - 1 - H, back = ring / D;
      constexpr int NI = D / RL;  // accesses per block
      constexpr int kTouch = (D * R::kBytes / 128 + kTileLanes - 1) / kTileLanes;
      const int2 *const rp = rows + (static_cast<int64_t>(g0 / D) + p) * (NI * kTileLanes) + lane;
      int2 rid[NI], rx[NI], rb[NI];
      int tv[kTouch] = {}, tl = 0;
      V bn[NI];
      auto list = [&](int2(&to)[NI], int m) {
#pragma unroll
        for (int u = 0; u < NI; ++u) to[u] = rp[(m * NI + u) * kTileLanes];
      };
      auto gather = [&] {
        if constexpr (STAGED) return;
#pragma unroll
        for (int u = 0; u < NI; ++u) {
          rb[u] = rid[u];
          bn[u] = b[max(rid[u].x, 0)];
        }
      };
#pragma unroll
      for (int u = 0; u < NI; ++u) {
        rid[u] = rx[u] = rb[u] = make_int2(-1, 0);
        bn[u] = V(0);
      }
      if (io < nblk) {
        list(rid, io);
        gather();
      }
      if (io + kTileIo < nblk) list(rid, io + kTileIo);
      for (int m = io; m < nblk + back; m += kTileIo) {
        const int mx = m - back;  // the block whose results go out
        if (mx >= 0) {
          while (lds_load(&s_done) < mx * D + D) __builtin_amdgcn_s_sleep(1);
          lds_fence();
          const int xb = (mx * D & (ring - 1)) * kTileLanes;
#pragma unroll
          for (int u = 0; u < NI; ++u)
            if (rx[u].x >= 0) x[rx[u].x] = slot(xb + rx[u].y);
        }
        if (m < nblk) {
          const int bb = (m * D & (ring - 1)) * kTileLanes;
#pragma unroll
          for (int u = 0; u < NI; ++u)
            if (rb[u].x >= 0) bslot(bb + rb[u].y) = bn[u];
          lds_fence();
          __builtin_amdgcn_wave_barrier();
          if (lane == 0) lds_store(&s_b[io], m / kTileIo + 1);
        }
        const int mt = m - back + 1 + kTileAhead;  // the block touched
        if (touch && mt >= 0 && mt < nblk) {
          // one lane per 128-byte line of the block's records and lists
          const char *rec = pack + (static_cast<int64_t>(g0) + mt * D) * R::kBytes;
#pragma unroll
          for (int l = 0; l < kTouch; ++l) {
            asm volatile("" ::"v"(tv[l]));
            const int line = l * kTileLanes + lane;
            if (line < D * R::kBytes / 128) tv[l] = *reinterpret_cast<const int *>(rec + line * 128);
          }
          asm volatile("" ::"v"(tl));
          if (lane * 16 < D * rstride)
            tl = reads[(static_cast<int64_t>(g0) + mt * D) * rstride + lane * 16].x;
        }
        if (m + kTileIo < nblk) gather();
        if (m + 2 * kTileIo < nblk) list(rid, m + 2 * kTileIo);
        const int nx = m + kTileIo - back;
        if (nx >= 0 && nx < nblk) list(rx, nx);
      }
    }
    // a wait of the solver that ran out of time
    if (wave == 0 && s_late && lane == 0) flag_late(err);
    __syncthreads();
  }
}

inline int pick_G(double avg) {
  int G = 1;
  while (G < 64 && G < avg) G <<= 1;
  return G;
}

template <typename T, typename V, typename A, bool DIAG>
void launch_level_range(const TrsvPlan &P, int l0, int l1, const T *val, const T *diag,
                        const V *b, V *x, hipStream_t s) {
  for (int l = l0; l < l1; ++l) {
    const int k0 = P.level_ptr[l], k1 = P.level_ptr[l + 1];
    if (k1 <= k0) continue;
    const int64_t threads = static_cast<int64_t>(k1 - k0) * P.G;
    const unsigned grid = static_cast<unsigned>((threads + kB - 1) / kB);
#define LA_LVL(GG)                                                                           \
  hipLaunchKernelGGL((k_trsv_level<GG, T, V, A, DIAG>), dim3(grid), dim3(kB), 0, s, k0, k1, \
                     P.rowptr.as<int>(), P.col.as<int>(), val, diag, P.perm.as<int>(), b, x)
    switch (P.G) {
      case 1: LA_LVL(1); break;
      case 2: LA_LVL(2); break;
      case 4: LA_LVL(4); break;
      case 8: LA_LVL(8); break;
      case 16: LA_LVL(16); break;
      case 32: LA_LVL(32); break;
      default: LA_LVL(64); break;
    }
#undef LA_LVL
  }
  LA_HIP(hipGetLastError());
}

template <int G, int NT, bool XL, typename T, typename V, typename A, bool DIAG>
void sf_launch(TrsvPlan &P, const T *val, const T *diag, const V *b, V *x, hipStream_t s) {
  int *rp = P.rowptr.as<int>(), *cl = P.col.as<int>(), *pm = P.perm.as<int>();
  unsigned *ctl = P.counter.as<unsigned>();
  int *err = P.err_flag.as<int>();
  // XLOCAL launches 8x the workgroups it needs (the others exit at once);
  // otherwise the whole chip, `sf_wgs` workgroups in total
  const unsigned need = std::max(1u, static_cast<unsigned>(P.nchunks));
  const unsigned grid = XL ? 8u * std::min(need, P.sf_wgs) : std::min(need, P.sf_wgs);
  hipLaunchKernelGGL((k_trsv_syncfree<G, NT, T, V, A, DIAG, XL>), dim3(grid), dim3(NT), 0, s,
                     P.nchunks, P.chunk_start.as<int>(), rp, cl, val, diag, pm, b, x, ctl, err);
}

// the hand-over slots <- sentinel, control words reset
template <typename V>
__global__ void k_tile_prep(int64_t n, V *mail, unsigned *ctl) {
  using U = typename Sentinel<V>::U;
  U *m = reinterpret_cast<U *>(mail);
  for (int64_t t = static_cast<int64_t>(blockIdx.x) * kB + threadIdx.x; t < n;
       t += static_cast<int64_t>(gridDim.x) * kB)
    m[t] = Sentinel<V>::bits;
  if (blockIdx.x == 0 && threadIdx.x < 16) ctl[threadIdx.x] = 0;
}

// b in the order of the records: slot t's row (dpos: its level position, -1:
// padding; perm: that position's row)
template <typename V>
__global__ void k_tile_stage(int64_t slots, const int *__restrict__ dpos,
                             const int *__restrict__ perm, const V *__restrict__ b, V *out) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * kB + threadIdx.x;
  if (t < slots) out[t] = dpos[t] >= 0 ? b[perm[dpos[t]]] : V(0);
}

// 8-byte LDS slots: results and, unless staged, b of `ring` groups, the zero
// slot, the halo
inline size_t tile_lds_bytes(int ring, int h_max, bool staged) {
  const size_t rings = (staged ? 1 : 2) * static_cast<size_t>(ring) * kTileLanes;
  return tile_ctl(staged) + 8 * (rings + 1 + h_max);
}

// The packed records: slot t's entries from the level-ordered values
// (src, -1: padding), LDS addresses and reciprocal diagonal (dpos).
template <int E, typename T>
__global__ void k_tile_pack(int64_t slots, const int *__restrict__ src,
                            const int *__restrict__ code, const int *__restrict__ dpos,
                            const T *__restrict__ val, const T *__restrict__ dinv, char *out) {
  using R = TileRec<E, T>;
  const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= slots) return;
  const int lane = static_cast<int>(t % kTileLanes);
  char *rec = out + t / kTileLanes * R::kBytes;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int q = src[t * E + e];
    constexpr int sT = static_cast<int>(sizeof(T));
    const int vb = e * sT, cb = e * static_cast<int>(sizeof(typename R::Code));
    *reinterpret_cast<T *>(rec + vb / R::kValPiece * R::kValPiece * kTileLanes +
                           lane * R::kValPiece + vb % R::kValPiece) = q >= 0 ? val[q] : T();
    *reinterpret_cast<typename R::Code *>(
        rec + R::kCodeAt + cb / R::kCodePiece * R::kCodePiece * kTileLanes +
        lane * R::kCodePiece + cb % R::kCodePiece) = R::code(code[t * E + e]);
  }
  T d = T();
  if (dinv && dpos[t] >= 0) d = dinv[dpos[t]];
  *reinterpret_cast<T *>(rec + R::kDinvAt + lane * R::kDinvStep) = d;
}

template <int E, typename T>
void tile_pack(TrsvPlan &P, hipStream_t s) {
  constexpr la_dtype dt = TileDt<T>::v;
  const int64_t groups = P.t_ngroups + kTilePad, slots = groups * kTileLanes;
  if (!P.t_pack[dt].p)
    P.t_pack[dt].alloc(static_cast<size_t>(groups) * TileRec<E, T>::kBytes);
  hipLaunchKernelGGL((k_tile_pack<E, T>), dim3(static_cast<unsigned>((slots + kB - 1) / kB)),
                     dim3(kB), 0, s, slots, P.t_lsrc.as<int>(), P.t_pcode.as<int>(),
                     P.t_dpos.as<int>(), P.val.v[dt].as<T>(),
                     P.unit ? nullptr : P.diag.v[dt].as<T>(), P.t_pack[dt].as<char>());
  LA_HIP(hipGetLastError());
}

// the packed records of one precision follow the level-ordered values
void tile_pack(TrsvPlan &P, la_dtype dt, hipStream_t s) {
  auto pack = [&](auto v) {
    using T = decltype(v);
    if (P.t_maxe == 2) tile_pack<2, T>(P, s);
    else if (P.t_maxe == 4) tile_pack<4, T>(P, s);
    else tile_pack<kTileMaxEntries, T>(P, s);
  };
  if (dt == LA_F64) pack(double());
  else if (dt == LA_F32) pack(float());
  else pack(bf16());
}

template <int E, int RL, int NB, int H, typename T, typename V, typename A, bool DIAG,
          bool STAGED = false>
void tiled_launch(TrsvPlan &P, const V *b, V *x, hipStream_t s) {
  if constexpr (!STAGED) {
    if (P.t_stage.p) {
      const int64_t slots = (static_cast<int64_t>(P.t_ngroups) + kTilePad) * kTileLanes;
      hipLaunchKernelGGL(k_tile_stage<V>, dim3(static_cast<unsigned>((slots + kB - 1) / kB)),
                         dim3(kB), 0, s, slots, P.t_dpos.as<int>(), P.perm.as<int>(), b,
                         P.t_stage.as<V>());
      LA_HIP(hipGetLastError());
      tiled_launch<E, RL, NB, H, T, V, A, DIAG, true>(P, P.t_stage.as<V>(), x, s);
      return;
    }
  }
  auto kern = k_trsv_tiled<E, RL, NB, H, T, V, A, DIAG, STAGED>;
  const size_t lds = tile_lds_bytes(P.t_ring, P.t_hmax, STAGED);
  static size_t lds_set = 0;  // per instantiation: the largest size allowed so far
  if (lds > lds_set) {
    LA_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                               hipFuncAttributeMaxDynamicSharedMemorySize,
                               static_cast<int>(lds)));
    lds_set = lds;
  }
  const int touch = tile_touch(P.t_ngroups, std::max(P.nlevels, 1), TileRec<E, T>::kBytes);
  const unsigned fg = static_cast<unsigned>(std::min<int64_t>(1024, (P.t_nmail + kB - 1) / kB));
  hipLaunchKernelGGL(k_tile_prep<V>, dim3(std::max(fg, 1u)), dim3(kB), 0, s, P.t_nmail,
                     P.t_mail.as<V>(), P.counter.as<unsigned>());
  hipLaunchKernelGGL(kern, dim3(P.t_wgs), dim3(kTileLanes * (1 + H + kTileIo)), lds, s,
                     P.t_nparts, P.t_gptr.as<int>(), P.t_rows.as<int2>(),
                     P.t_pack[TileDt<T>::v].template as<const char>(), P.t_reads.as<int2>(),
                     P.t_rstride, b, x, P.t_mail.as<V>(), P.t_mstride, P.t_ring, P.t_hmax, touch,
                     P.counter.as<unsigned>(), P.err_flag.as<int>());
}

template <typename T, typename V, typename A, bool DIAG>
void launch_syncfree(TrsvPlan &P, const T *val, const T *diag, const V *b, V *x, hipStream_t s) {
  const int64_t n = P.n;
  if (P.tiled) {
    constexpr int E8 = kTileMaxEntries, RW = kTileRowLanes;
    // fetchers: two with blocks of four groups, or four with blocks of two
    // where a group takes longer (up to 18 values each). Measured per apply,
    // 4 x 1 / 4 x 2 / 2 x 4 (fetchers x groups): 512^2 428 / 400 / 393 us,
    // 56^3 27-point FP32 525 / 472 / 582 us
    if (P.t_maxe == 2) tiled_launch<2, 1, 4, 2, T, V, A, DIAG>(P, b, x, s);
    else if (P.t_maxe == 4) tiled_launch<4, 1, 4, 2, T, V, A, DIAG>(P, b, x, s);
    else if (P.t_rlanes == 1) tiled_launch<E8, 1, 4, 2, T, V, A, DIAG>(P, b, x, s);
    else tiled_launch<E8, RW, 2, 4, T, V, A, DIAG>(P, b, x, s);
    LA_HIP(hipGetLastError());
    return;
  }
  unsigned fg = static_cast<unsigned>(std::min<int64_t>(4096, (n + kB - 1) / kB));
  if (fg == 0) fg = 1;
  hipLaunchKernelGGL(k_fill_sentinel<V>, dim3(fg), dim3(kB), 0, s, n, x, P.counter.as<unsigned>());
  LA_HIP(hipGetLastError());
#define LA_SF2(GG, NT)                                      \
  if (P.sf_xlocal) {                                        \
    sf_launch<GG, NT, true, T, V, A, DIAG>(P, val, diag, b, x, s);  \
  } else {                                                  \
    sf_launch<GG, NT, false, T, V, A, DIAG>(P, val, diag, b, x, s); \
  }
#define LA_SF(GG)              \
  if (P.sf_nt == 1024) {       \
    LA_SF2(GG, 1024);          \
  } else if (P.sf_nt == 512) { \
    LA_SF2(GG, 512);           \
  } else {                     \
    LA_SF2(GG, 256);           \
  }
  switch (P.G) {
    case 1: LA_SF(1); break;
    case 2: LA_SF(2); break;
    case 4: LA_SF(4); break;
    case 8: LA_SF(8); break;
    case 16: LA_SF(16); break;
    case 32: LA_SF(32); break;
    default: LA_SF(64); break;
  }
#undef LA_SF2
#undef LA_SF
  LA_HIP(hipGetLastError());
}

template <typename T, typename V, typename A>
void solve_typed(TrsvPlan &P, la_trsv_mode mode, const void *valp, const void *diagp,
                 const void *b, void *x, hipStream_t s) {
  const T *val = static_cast<const T *>(valp);
  const T *diag = static_cast<const T *>(diagp);
  const V *bb = static_cast<const V *>(b);
  V *xx = static_cast<V *>(x);
  if (mode == LA_TRSV_SYNCFREE) {
    if (P.unit) launch_syncfree<T, V, A, false>(P, val, diag, bb, xx, s);
    else launch_syncfree<T, V, A, true>(P, val, diag, bb, xx, s);
  } else {
    if (P.unit) launch_level_range<T, V, A, false>(P, 0, P.nlevels, val, diag, bb, xx, s);
    else launch_level_range<T, V, A, true>(P, 0, P.nlevels, val, diag, bb, xx, s);
  }
}

void solve_dispatch(TrsvPlan &P, la_trsv_mode mode, la_dtype val, la_dtype vec, const void *b,
                    void *x, hipStream_t s) {
  const void *v = P.nnz ? P.val.get(val) : nullptr;
  const void *d = P.unit ? nullptr : P.diag.get(val);
  if (val == LA_F64 && vec == LA_F64) return solve_typed<double, double, double>(P, mode, v, d, b, x, s);
  if (vec == LA_F64) {
    if (val == LA_F64) return solve_typed<double, double, float>(P, mode, v, d, b, x, s);
    if (val == LA_F32) return solve_typed<float, double, float>(P, mode, v, d, b, x, s);
    return solve_typed<bf16, double, float>(P, mode, v, d, b, x, s);
  }
  if (val == LA_F64) return solve_typed<double, float, float>(P, mode, v, d, b, x, s);
  if (val == LA_F32) return solve_typed<float, float, float>(P, mode, v, d, b, x, s);
  return solve_typed<bf16, float, float>(P, mode, v, d, b, x, s);
}

// ------------------------------------------------------------ JACOBI mode
// Sweeps in the column-scaled form: with w = D y, y_{s+1} = D^-1 (b - N y_s)
// becomes w_{s+1} = b - (N D^-1) w_s from w_0 = b, and x = D^-1 w_k; the
// last sweep applies D^-1 in its epilogue, so a solve is k launches (no
// separate scaling pass).

// out_i = dinv_i * b_i (k = 0, or the last sweep without a sliced-ELL form)
template <typename T, typename V, typename A>
__global__ void k_jac_scale(int n, const T *__restrict__ dinv, const V *__restrict__ b, V *out) {
  const int i = static_cast<int>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) out[i] = static_cast<V>(static_cast<A>(ldt(dinv, i)) * static_cast<A>(b[i]));
}

// D^-1 from a device factor array f
__global__ void k_jac_dinv(int n, const int64_t *__restrict__ dsrc, const double *__restrict__ f,
                           double *dinv) {
  const int i = static_cast<int>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) dinv[i] = 1.0 / f[dsrc[i]];
}

// N D^-1 from f, row by row (dinv null: unit diagonal)
__global__ void k_jac_vals(int n, const int *__restrict__ ai, const int *__restrict__ aj,
                           const int64_t *__restrict__ src, const double *__restrict__ f,
                           const double *__restrict__ dinv, double *nv) {
  const int i = static_cast<int>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  for (int q = ai[i]; q < ai[i + 1]; ++q) nv[q] = dinv ? f[src[q]] * dinv[aj[q]] : f[src[q]];
}

void jacobi_refresh(TrsvPlan &T, const double *f, hipStream_t s) {
  Mat &J = *T.jac;
  if (T.h_src.empty() || T.n == 0) return;
  const unsigned grid = static_cast<unsigned>((T.n + 255) / 256);
  double *dv = T.unit ? nullptr : T.jdinv.v[LA_F64].as<double>();
  if (!T.unit && !T.h_dsrc.empty()) {
    hipLaunchKernelGGL(k_jac_dinv, dim3(grid), dim3(256), 0, s, T.n, T.jdsrc.as<int64_t>(), f,
                       dv);
    LA_HIP(hipGetLastError());
    T.jdinv.set_from_device_f64(dv, T.n, s);
  }
  if (J.nnz) {
    double *nv = J.vals.v[LA_F64].as<double>();
    hipLaunchKernelGGL(k_jac_vals, dim3(grid), dim3(256), 0, s, T.n, J.ai.as<int>(),
                       J.aj.as<int>(), T.jsrc.as<int64_t>(), f, dv, nv);
    LA_HIP(hipGetLastError());
    J.vals.set_from_device_f64(nv, J.nnz, s);
  }
}

void build_jacobi(TrsvPlan &T, hipStream_t s) {
  const int n = T.n;
  std::vector<double> sv(static_cast<size_t>(T.nnz)), dv(T.unit ? 0 : n);
  for (int i = 0; i < n && !T.unit; ++i) dv[i] = 1.0 / T.h_diag[i];
  for (int i = 0; i < n; ++i)
    for (int q = T.h_ai[i]; q < T.h_ai[i + 1]; ++q)
      sv[q] = T.unit ? T.h_av[q] : T.h_av[q] * dv[T.h_aj[q]];
  T.jac = make_mat(n, n, 0, T.h_ai.data(), T.h_aj.data(), sv.data(), s);
  if (!T.unit) T.jdinv.set_from_host(dv.data(), n, s);
  T.jtmp[0].alloc(sizeof(double) * static_cast<size_t>(n));
  T.jtmp[1].alloc(sizeof(double) * static_cast<size_t>(n));
  if (!T.h_src.empty()) {
    T.jsrc.alloc(sizeof(int64_t) * std::max<size_t>(T.h_src.size(), 1));
    T.jsrc.upload(T.h_src.data(), sizeof(int64_t) * T.h_src.size(), s);
    if (!T.h_dsrc.empty()) {
      T.jdsrc.alloc(sizeof(int64_t) * T.h_dsrc.size());
      T.jdsrc.upload(T.h_dsrc.data(), sizeof(int64_t) * T.h_dsrc.size(), s);
    }
  }
  if (T.fsrc) jacobi_refresh(T, T.fsrc, s);
  LA_HIP(hipStreamSynchronize(s));
}

void jac_scale(int n, la_dtype val, la_dtype vec, const void *d, const void *b, void *o,
               hipStream_t s) {
  const dim3 grid(static_cast<unsigned>((n + 255) / 256)), blk(256);
#define LA_JS(T, V, A)                                                                          \
  hipLaunchKernelGGL((k_jac_scale<T, V, A>), grid, blk, 0, s, n, static_cast<const T *>(d),     \
                     static_cast<const V *>(b), static_cast<V *>(o))
  if (vec == LA_F64) {
    if (val == LA_F64) LA_JS(double, double, double);
    else if (val == LA_F32) LA_JS(float, double, float);
    else LA_JS(bf16, double, float);
  } else {
    if (val == LA_F64) LA_JS(double, float, float);
    else if (val == LA_F32) LA_JS(float, float, float);
    else LA_JS(bf16, float, float);
  }
#undef LA_JS
  LA_HIP(hipGetLastError());
}

void jacobi_solve(TrsvPlan &T, la_dtype val, la_dtype vec, const void *b, void *x,
                  hipStream_t s) {
  if (!T.jac) build_jacobi(T, s);
  Mat &J = *T.jac;
  const int n = T.n;
  const size_t esz = vec == LA_F64 ? 8 : 4;
  const la_dtype acc = val == LA_F64 && vec == LA_F64 ? LA_F64 : LA_F32;
  const int k = T.sweeps;
  const void *d = nullptr;
  if (!T.unit) {
    if (!T.jdinv.has[val]) T.jdinv.add(val, s);
    d = T.jdinv.get(val);
  }
  if (k == 0) {
    if (d) jac_scale(n, val, vec, d, b, x, s);
    else LA_HIP(hipMemcpyAsync(x, b, esz * n, hipMemcpyDeviceToDevice, s));
    return;
  }
  void *t0 = T.jtmp[0].p, *t1 = T.jtmp[1].p;
  // sweeps 1 .. k-1 alternate between the two spare vectors (a unit
  // triangle's sweep q writes x when k - q is even instead)
  const void *prev = b;
  for (int q = 1; q < k; ++q) {
    void *dst = d ? (q % 2 ? t0 : t1) : ((k - q) % 2 == 0 ? x : (prev == t0 ? t1 : t0));
    spmv(J, LA_SPMV_AUTO, val, vec, acc, -1.0, prev, 1.0, b, dst, s);
    prev = dst;
  }
  if (!d) {
    spmv(J, LA_SPMV_AUTO, val, vec, acc, -1.0, prev, 1.0, b, x, s);
    return;
  }
  // last sweep: x = D^-1 (b - (N D^-1) w_{k-1})
  if (spmv_sell_rowscaled(J, val, vec, d, prev, b, x, s)) return;
  void *tmp = prev == t0 ? t1 : t0;
  spmv(J, LA_SPMV_AUTO, val, vec, acc, -1.0, prev, 1.0, b, tmp, s);
  jac_scale(n, val, vec, d, tmp, x, s);
}

void tiled_refresh(TrsvPlan &T, hipStream_t s) {
  if (!T.tiled) return;
  for (int dt = 0; dt < 3; ++dt)
    if (T.t_pack[dt].p) tile_pack(T, static_cast<la_dtype>(dt), s);
}

// The tiled schedule when the triangle's pattern is recognised as a grid
// and a tile's window and halo fit one workgroup's LDS; one workgroup per
// tile, at most one per CU, so every tile is resident.
void build_tiled(TrsvPlan &P, const std::vector<int> &iperm, const std::vector<int> &lrp,
                 hipStream_t s) {
  const int n = P.n;
  if (P.nnz == 0) {
    P.t_why = "no entries";
    return;
  }
  std::vector<int> level(static_cast<size_t>(n)), lpos(static_cast<size_t>(n));
  for (int l = 0; l < P.nlevels; ++l)
    for (int k = P.level_ptr[l]; k < P.level_ptr[l + 1]; ++k) {
      level[iperm[k]] = l;
      lpos[iperm[k]] = k;
    }
  int dev = 0, ncu = 0, budget = 0;
  LA_HIP(hipGetDevice(&dev));
  LA_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
  LA_HIP(hipDeviceGetAttribute(&budget, hipDeviceAttributeMaxSharedMemoryPerBlock, dev));
  // halo slots: what LDS holds beyond the results of kTileWindow groups (and a
  // ring of b as long, and both twice as long, where the halo leaves room: the
  // I/O wavefronts then run further ahead)
  const int64_t avail =
      static_cast<int64_t>(budget) - static_cast<int64_t>(tile_lds_bytes(kTileWindow, 0, true));
  const int max_halo = static_cast<int>(avail / 8);
  if (max_halo < 128 || ncu < 1) {
    P.t_why = "LDS too small for the tiled schedule";
    return;
  }
  TileLayout L;
  if (!build_tile_layout(n, P.h_ai.data(), P.h_aj.data(), level.data(), kTileLanes, ncu, n,
                         max_halo, L, P.t_why))
    return;
  const int E = L.maxe, RL = L.rlanes;
  const int G = L.ngroups;
  // (the solve loads groups past a tile's last one)
  const int64_t slots = static_cast<int64_t>(G + kTilePad) * kTileLanes, m = slots * E;
  std::vector<int> dpos(static_cast<size_t>(slots), -1);
  std::vector<int> lsrc(static_cast<size_t>(m), -1);
  P.t_ring = tile_lds_bytes(2 * kTileWindow, L.h_max, false) <= static_cast<size_t>(budget)
                 ? 2 * kTileWindow : kTileWindow;
  const bool staged = tile_lds_bytes(P.t_ring, L.h_max, false) > static_cast<size_t>(budget);
  // byte addresses into LDS: the results of group i sit in place i % t_ring
  const int zero = P.t_ring * kTileLanes, ctl = tile_ctl(staged);
  std::vector<int> pcode(static_cast<size_t>(m), ctl + 8 * zero), gtile(static_cast<size_t>(G));
  for (int p = 0; p < L.nparts; ++p)
    for (int g = L.part_gptr[p]; g < L.part_gptr[p + 1]; ++g) gtile[g] = p;
  // a row of RL lanes: its first lane carries the row id, 1/d and the
  // level position; the others only entries (no id: they publish nothing)
  for (int g = 0; g < G; ++g)
    for (int kk = L.grp_row[g]; kk < L.grp_row[g + 1]; ++kk)
      for (int w = 0; w < RL; ++w) {
        const int64_t sl = static_cast<int64_t>(g) * kTileLanes + RL * (kk - L.grp_row[g]) + w;
        const int r = L.tperm[kk];
        if (w == 0) {
          dpos[sl] = lpos[r];
        }
        for (int e = 0; e < E; ++e) {
          const size_t te = (static_cast<size_t>(kk) * RL + w) * E + e;
          const size_t pe = static_cast<size_t>(sl) * E + e;
          const int c = L.tcode[te], q = L.tsrc[te];
          if (c < 0) {
            pcode[pe] = ctl + 8 * (zero + 1 + (-c - 1));
          } else if (q >= 0) {
            // the layout counts places modulo kTileWindow: the group is the
            // last one before this one at that place
            const int gi = g - L.part_gptr[gtile[g]];
            const int gd = gi - 1 - (gi - 1 - c / kTileLanes) % kTileWindow;
            pcode[pe] = ctl + 8 * (gd % P.t_ring * kTileLanes + c % kTileLanes);
          }
          lsrc[pe] = q >= 0 ? lrp[lpos[r]] + (q - P.h_ai[r]) : -1;
        }
      }
  // shared rows: a fixed run of hand-over slots per group, and kTileDepth
  // groups of spare ones per tile
  P.t_mstride = std::max(4, (L.shared_max + 3) / 4 * 4);
  P.t_nmail = (static_cast<int64_t>(G) + static_cast<int64_t>(L.nparts) * kTileDepth) * P.t_mstride;
  if (P.t_nmail > INT32_MAX) {
    P.t_why = "too many hand-over slots";
    return;
  }
  // per block of kTileDepth groups its rows by row id: (row, place in the
  // block); block m of tile p is number first group / kTileDepth + p + m
  const int per = kTileDepth * kTileLanes / RL;
  std::vector<int2> rows(static_cast<size_t>(G / kTileDepth + L.nparts + 1) * per,
                         make_int2(-1, 0));
#pragma omp parallel for schedule(dynamic, 4)
  for (int p = 0; p < L.nparts; ++p) {
    const int ga = L.part_gptr[p], gb = L.part_gptr[p + 1];
    for (int g = ga; g < gb; g += kTileDepth) {
      int2 *out = &rows[static_cast<size_t>(ga / kTileDepth + p + (g - ga) / kTileDepth) * per];
      int2 *end = out;
      for (int h = g; h < std::min(gb, g + kTileDepth); ++h)
        for (int kk = L.grp_row[h]; kk < L.grp_row[h + 1]; ++kk)
          *end++ = make_int2(L.tperm[kk], (h - g) * kTileLanes + RL * (kk - L.grp_row[h]));
      std::sort(out, end, [](const int2 &a, const int2 &b) { return a.x < b.x; });
    }
  }
  // what each group reads from other tiles: (hand-over slot, halo slot), as
  // many places per group as the longest list has
  int longest = 1;
  for (int g = 0; g < G; ++g) longest = std::max(longest, L.rf_ptr[g + 1] - L.rf_ptr[g]);
  P.t_rstride = longest;
  std::vector<int2> reads(static_cast<size_t>(G + kTilePad) * longest, make_int2(-1, 0));
  for (int g = 0; g < G; ++g)
    for (int t = L.rf_ptr[g]; t < L.rf_ptr[g + 1]; ++t) {
      const int from = L.rf_grp[t];
      reads[static_cast<size_t>(g) * longest + t - L.rf_ptr[g]] =
          make_int2((from + gtile[from] * kTileDepth) * P.t_mstride + L.rf_pos[t],
                    zero + 1 + L.rf_slot[t]);
    }
  P.t_mail.alloc(sizeof(double) * static_cast<size_t>(P.t_nmail));
  if (staged) P.t_stage.alloc(sizeof(double) * static_cast<size_t>(slots));
  auto up = [&](DevBuf &d, const void *h, size_t bytes) {
    d.alloc(std::max<size_t>(bytes, 4));
    d.upload(h, bytes, s);
  };
  up(P.t_gptr, L.part_gptr.data(), sizeof(int) * L.part_gptr.size());
  up(P.t_rows, rows.data(), sizeof(int2) * rows.size());
  up(P.t_pcode, pcode.data(), sizeof(int) * pcode.size());
  up(P.t_reads, reads.data(), sizeof(int2) * reads.size());
  up(P.t_lsrc, lsrc.data(), sizeof(int) * lsrc.size());
  up(P.t_dpos, dpos.data(), sizeof(int) * dpos.size());
  P.t_nparts = L.nparts;
  P.t_ngroups = G;
  P.t_mmax = L.m_max;
  P.t_hmax = L.h_max;
  P.t_maxe = E;
  P.t_rlanes = RL;
  P.t_tau = L.tau;
  P.t_remote = L.remote_frac;
  P.t_wgs = static_cast<unsigned>(std::min(L.nparts, ncu));
  P.tiled = true;
  tile_pack(P, LA_F64, s);
}

// LEVEL mode records at most this many levels in a graph. One of 131072 levels
// ended in a segmentation fault of the host process (65536 ran), so longer
// chains are launched level by level.
constexpr int kGraphLevels = 65536;

hipStream_t capture_stream() {
  static thread_local hipStream_t cs = nullptr;
  if (!cs) LA_HIP(hipStreamCreateWithFlags(&cs, hipStreamNonBlocking));
  return cs;
}
}  // namespace

TrsvPlan::~TrsvPlan() {
  if (err_host) (void)hipHostFree(err_host);
  for (auto &kv : graphs) (void)hipGraphExecDestroy(kv.second);
}

std::unique_ptr<TrsvPlan> make_trsv(int n, int base, const int *ai, const int *aj,
                                    const double *av, const double *diag, bool upper,
                                    hipStream_t s) {
  LA_CHECK_ARG(n >= 0 && ai, "bad triangle");
  auto P = std::make_unique<TrsvPlan>();
  P->n = n;
  P->upper = upper;
  P->unit = diag == nullptr;
  P->stream = s;
  const int64_t nnz = static_cast<int64_t>(ai[n]) - ai[0];
  LA_CHECK_ARG(ai[0] == base, "ai[0] must equal base");
  LA_CHECK_ARG(nnz == 0 || (aj && av), "aj/av null");
  P->nnz = nnz;
  P->h_ai.resize(static_cast<size_t>(n) + 1);
  P->h_aj.resize(static_cast<size_t>(nnz));
  P->h_av.assign(av, av + nnz);
  for (int i = 0; i <= n; ++i) P->h_ai[i] = ai[i] - base;
  for (int i = 0; i < n; ++i)
    for (int q = P->h_ai[i]; q < P->h_ai[i + 1]; ++q) {
      const int c = aj[q] - base;
      LA_CHECK_ARG(c >= 0 && c < n, "column out of range");
      LA_CHECK_ARG(upper ? c > i : c < i,
                   "triangular solve needs a strictly triangular matrix (diagonal apart)");
      P->h_aj[q] = c;
    }
  if (diag) P->h_diag.assign(diag, diag + n);
  // level sets
  std::vector<int> iperm(std::max(n, 1)), prefix(static_cast<size_t>(n) + 2);
  const int L = topo_sort2(n, 0, P->h_ai.data(), P->h_aj.data(), upper, iperm.data(), prefix.data());
  P->nlevels = L;
  P->level_ptr.assign(prefix.begin(), prefix.begin() + L + 1);
  P->h_perm.assign(iperm.begin(), iperm.begin() + n);
  // level-ordered copy
  std::vector<int> rp(static_cast<size_t>(n) + 1), cl(static_cast<size_t>(nnz));
  std::vector<double> vl(static_cast<size_t>(nnz)), dg(diag ? n : 0);
  rp[0] = 0;
  for (int k = 0; k < n; ++k) {
    const int r = iperm[k];
    const int len = P->h_ai[r + 1] - P->h_ai[r];
    std::copy(P->h_aj.begin() + P->h_ai[r], P->h_aj.begin() + P->h_ai[r + 1], cl.begin() + rp[k]);
    std::copy(P->h_av.begin() + P->h_ai[r], P->h_av.begin() + P->h_ai[r + 1], vl.begin() + rp[k]);
    rp[k + 1] = rp[k] + len;
    if (diag) dg[k] = 1.0 / diag[r];  // kernels multiply: no divide on the chain
  }
  P->G = pick_G(n ? static_cast<double>(nnz) / n : 1.0);

  // sync-free launch shape. Narrow levels (few rows per level): the solve is
  // a chain of dependency hops, so keep it on one XCD, where a hop costs
  // ~0.3 us instead of ~0.55 us, with 32 workgroups of 256. Wide levels:
  // the whole chip, 256 workgroups of 512 (fewer tickets per level). The
  // 1024 rows/level switch point sits between the 512^2 5-point grid (256
  // rows/level, 6x faster on one XCD than level launches) and the RCM 128^3
  // 7-point grid (5490 rows/level, 3.3x faster over all XCDs).
  const double rows_per_level = L > 0 ? static_cast<double>(n) / L : 0.0;
  if (rows_per_level < 1024.0) {
    P->sf_xlocal = true;
    P->sf_wgs = 32;
    P->sf_nt = 256;
  } else {
    // wide levels: the whole chip, 256 workgroups; rows of 16+ lanes get
    // 1024-thread workgroups, so a level costs half the tickets (27-point
    // ILU(1) at 160^3: 5.4 ms per apply against 6.9 ms with 512)
    P->sf_xlocal = false;
    P->sf_wgs = 256;
    P->sf_nt = P->G >= 16 ? 1024 : 512;
  }
  // chunks: one workgroup's worth of rows (sf_nt/G), never spanning a level
  if (const char *e = std::getenv("LAAMD_SF_NT")) {
    const int v = std::atoi(e);
    P->sf_nt = v >= 1024 ? 1024 : v >= 512 ? 512 : 256;
  }
  const int R = P->sf_nt / P->G;
  std::vector<int> chunks;
  for (int l = 0; l < L; ++l)
    for (int k = P->level_ptr[l]; k < P->level_ptr[l + 1]; k += R) chunks.push_back(k);
  chunks.push_back(n);
  P->nchunks = static_cast<int>(chunks.size()) - 1;
  // launch-shape overrides for tuning: LAAMD_SF_XLOCAL=0|1, LAAMD_SF_WGS=1..4096
  if (const char *e = std::getenv("LAAMD_SF_XLOCAL")) P->sf_xlocal = std::atoi(e) != 0;
  if (const char *e = std::getenv("LAAMD_SF_WGS"))
    P->sf_wgs = static_cast<unsigned>(std::clamp(std::atoi(e), 1, 4096));
  P->rowptr.alloc(sizeof(int) * (static_cast<size_t>(n) + 1));
  P->col.alloc(sizeof(int) * static_cast<size_t>(nnz));
  P->perm.alloc(sizeof(int) * static_cast<size_t>(std::max(n, 1)));
  P->chunk_start.alloc(sizeof(int) * chunks.size());
  P->counter.alloc(sizeof(unsigned) * 16);
  P->err_flag.alloc(sizeof(int) * 4);
  P->rowptr.upload(rp.data(), sizeof(int) * (n + 1), s);
  P->col.upload(cl.data(), sizeof(int) * nnz, s);
  P->perm.upload(iperm.data(), sizeof(int) * n, s);
  P->chunk_start.upload(chunks.data(), sizeof(int) * chunks.size(), s);
  LA_HIP(hipHostMalloc(reinterpret_cast<void **>(&P->err_host), sizeof(int) * 4,
                       hipHostMallocMapped | hipHostMallocCoherent));
  *P->err_host = 0;
  struct {
    int flag[2];
    int *host;
  } flag = {{0, 0}, nullptr};
  static_assert(sizeof(flag) == sizeof(int) * 4, "the host copy's address behind the flag");
  LA_HIP(hipHostGetDevicePointer(reinterpret_cast<void **>(&flag.host), P->err_host, 0));
  P->err_flag.upload(&flag, sizeof(flag), s);
  LA_HIP(hipMemsetAsync(P->counter.p, 0, sizeof(unsigned) * 16, s));
  P->val.set_from_host(vl.data(), nnz, s);
  if (diag) P->diag.set_from_host(dg.data(), n, s);
  const char *te = std::getenv("LAAMD_SF_TILED");
  if (!(te && te[0] == '0') && n > 0) build_tiled(*P, iperm, rp, s);
  LA_HIP(hipStreamSynchronize(s));
  return P;
}

void trsv_add_dtype(TrsvPlan &T, la_dtype dt) {
  if (T.nnz) T.val.add(dt, T.stream);
  else if (!T.val.has[LA_F64]) { /* empty triangle: nothing stored */ }
  if (!T.unit) T.diag.add(dt, T.stream);
  if (T.tiled && !T.t_pack[dt].p) tile_pack(T, dt, T.stream);
  if (T.transposed) trsv_add_dtype(*T.transposed, dt);
  LA_HIP(hipStreamSynchronize(T.stream));
}

void trsv_solve(TrsvPlan &T, la_trsv_mode mode, la_dtype val, la_dtype vec, const void *b,
                void *x, hipStream_t s) {
  LA_CHECK_ARG(mode == LA_TRSV_LEVEL || mode == LA_TRSV_SYNCFREE || mode == LA_TRSV_JACOBI,
               "bad trsv mode");
  LA_CHECK_ARG(val >= LA_F64 && val <= LA_BF16, "bad value dtype");
  LA_CHECK_ARG(vec == LA_F64 || vec == LA_F32, "vectors must be FP64 or FP32");
  LA_CHECK_ARG(T.n == 0 || (b && x), "null vector");
  LA_CHECK_ARG(b != x || T.n == 0, "b and x must be distinct");
  if (T.n == 0) return;
  if (mode == LA_TRSV_JACOBI) {
    jacobi_solve(T, val, vec, b, x, s);
    return;
  }
  if ((T.nnz && !T.val.has[val]) || (!T.unit && !T.diag.has[val])) trsv_add_dtype(T, val);
  if (mode == LA_TRSV_SYNCFREE || T.nlevels <= 2 || T.nlevels > kGraphLevels) {
    solve_dispatch(T, mode, val, vec, b, x, s);
    return;
  }
  // LEVEL: replay a captured graph of the per-level launches
  auto key = std::make_tuple(static_cast<int>(val), static_cast<int>(vec), b, x);
  auto it = T.graphs.find(key);
  if (it == T.graphs.end()) {
    if (T.graphs.size() >= 16) {
      for (auto &kv : T.graphs) (void)hipGraphExecDestroy(kv.second);
      T.graphs.clear();
    }
    hipStream_t cs = capture_stream();
    hipGraph_t g = nullptr;
    LA_HIP(hipStreamBeginCapture(cs, hipStreamCaptureModeThreadLocal));
    try {
      solve_dispatch(T, mode, val, vec, b, x, cs);
    } catch (...) {
      (void)hipStreamEndCapture(cs, &g);
      if (g) (void)hipGraphDestroy(g);
      throw;
    }
    LA_HIP(hipStreamEndCapture(cs, &g));
    hipGraphExec_t ge = nullptr;
    LA_HIP(hipGraphInstantiate(&ge, g, nullptr, nullptr, 0));
    (void)hipGraphDestroy(g);
    it = T.graphs.emplace(key, ge).first;
  }
  LA_HIP(hipGraphLaunch(it->second, s));
}

TrsvPlan &trsv_transposed(TrsvPlan &T) {
  if (!T.transposed) {
    std::vector<int> ti(static_cast<size_t>(T.n) + 1), tj(static_cast<size_t>(T.nnz));
    std::vector<double> tv(static_cast<size_t>(T.nnz));
    transpose(T.n, T.n, 0, T.h_ai.data(), T.h_aj.data(), T.h_av.data(), ti.data(), tj.data(),
              tv.data());
    T.transposed = make_trsv(T.n, 0, ti.data(), tj.data(), tv.data(),
                             T.unit ? nullptr : T.h_diag.data(), !T.upper, T.stream);
    T.transposed->sweeps = T.sweeps;
    if (!T.h_src.empty() || !T.h_dsrc.empty()) {
      // the same transpose carries the source positions (exact as doubles)
      std::vector<double> sv(T.h_src.begin(), T.h_src.end()), st(static_cast<size_t>(T.nnz));
      std::vector<int> ti2(static_cast<size_t>(T.n) + 1), tj2(static_cast<size_t>(T.nnz));
      transpose(T.n, T.n, 0, T.h_ai.data(), T.h_aj.data(), sv.data(), ti2.data(), tj2.data(),
                st.data());
      std::vector<int64_t> tsrc(st.begin(), st.end());
      trsv_set_sources(*T.transposed, tsrc.data(), T.h_dsrc.empty() ? nullptr : T.h_dsrc.data(),
                       T.stream);
      if (T.fsrc) trsv_refresh(*T.transposed, T.fsrc, T.stream);
    }
    for (int dt = 1; dt < 3; ++dt)
      if (T.val.has[dt] || T.diag.has[dt]) trsv_add_dtype(*T.transposed, static_cast<la_dtype>(dt));
  }
  return *T.transposed;
}

namespace {
__global__ void k_gather(int64_t m, const int64_t *__restrict__ src, const double *__restrict__ f,
                         double *out) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t < m) out[t] = f[src[t]];
}
__global__ void k_gather_recip(int64_t m, const int64_t *__restrict__ src,
                               const double *__restrict__ f, double *out) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t < m) out[t] = 1.0 / f[src[t]];
}
}  // namespace

void trsv_set_sources(TrsvPlan &T, const int64_t *src, const int64_t *dsrc, hipStream_t s) {
  const int n = T.n;
  T.jac.reset();  // the JACOBI copy is rebuilt with the new sources
  T.h_src.assign(src, src + T.nnz);
  if (dsrc) T.h_dsrc.assign(dsrc, dsrc + n);
  else T.h_dsrc.clear();
  // level order: entries of row perm[k] in their stored order
  std::vector<int64_t> ls(static_cast<size_t>(std::max<int64_t>(T.nnz, 1))),
      ld(static_cast<size_t>(std::max(n, 1)));
  int64_t p = 0;
  for (int k = 0; k < n; ++k) {
    const int r = T.h_perm[k];
    for (int q = T.h_ai[r]; q < T.h_ai[r + 1]; ++q) ls[p++] = src[q];
    if (dsrc) ld[k] = dsrc[r];
  }
  T.val_src.alloc(sizeof(int64_t) * ls.size());
  T.val_src.upload(ls.data(), sizeof(int64_t) * ls.size(), s);
  if (dsrc) {
    T.diag_src.alloc(sizeof(int64_t) * ld.size());
    T.diag_src.upload(ld.data(), sizeof(int64_t) * ld.size(), s);
  }
  LA_HIP(hipStreamSynchronize(s));
}

void trsv_refresh(TrsvPlan &T, const double *f, hipStream_t s) {
  T.fsrc = f;
  if (T.nnz) {
    double *v = T.val.v[LA_F64].as<double>();
    hipLaunchKernelGGL(k_gather, dim3(static_cast<unsigned>((T.nnz + 255) / 256)), dim3(256), 0,
                       s, T.nnz, T.val_src.as<int64_t>(), f, v);
    LA_HIP(hipGetLastError());
    T.val.set_from_device_f64(v, T.nnz, s);
  }
  if (!T.unit && !T.h_dsrc.empty() && T.n) {
    double *d = T.diag.v[LA_F64].as<double>();
    hipLaunchKernelGGL(k_gather_recip, dim3(static_cast<unsigned>((T.n + 255) / 256)), dim3(256),
                       0, s, static_cast<int64_t>(T.n), T.diag_src.as<int64_t>(), f, d);
    LA_HIP(hipGetLastError());
    T.diag.set_from_device_f64(d, T.n, s);
  }
  tiled_refresh(T, s);
  if (T.jac) jacobi_refresh(T, f, s);
  if (T.transposed) trsv_refresh(*T.transposed, f, s);
}

void trsv_set_sweeps(TrsvPlan &T, int sweeps) {
  LA_CHECK_ARG(sweeps >= 0 && sweeps <= 1000000, "sweeps out of range");
  T.sweeps = sweeps;
  if (T.transposed) trsv_set_sweeps(*T.transposed, sweeps);
}

// The flag reaches the host as a store of the kernel that set it, so one
// synchronisation is all a check costs (a copy of the flag and another
// synchronisation per triangle took 35 us more per apply).
bool trsv_check_timeout(std::initializer_list<TrsvPlan *> plans, hipStream_t s) {
  LA_HIP(hipStreamSynchronize(s));
  bool bad = false;
  for (TrsvPlan *T : plans)
    for (; T; T = T->transposed.get())
      if (__atomic_load_n(T->err_host, __ATOMIC_ACQUIRE) != 0) {
        bad = true;
        LA_HIP(hipMemsetAsync(T->err_flag.p, 0, sizeof(int), s));
        LA_HIP(hipStreamSynchronize(s));
        __atomic_store_n(T->err_host, 0, __ATOMIC_RELEASE);
      }
  return bad;
}

// ------------------------------------------------------------------ ILU / IC
std::unique_ptr<Prec> make_prec_ilu(int n, int base, const int *fai, const int *faj,
                                    const double *fav, hipStream_t s) {
  auto P = std::make_unique<Prec>();
  P->n = n;
  P->stream = s;
  std::vector<int> Lai(static_cast<size_t>(n) + 1), Uai(static_cast<size_t>(n) + 1);
  int64_t ln = 0, un = 0;
  split_ldu(n, base, fai, faj, fav, Lai.data(), nullptr, nullptr, nullptr, Uai.data(), nullptr,
            nullptr, &ln, &un);
  std::vector<int> Laj(ln), Uaj(un);
  std::vector<double> Lav(ln), Uav(un), D(n);
  split_ldu(n, base, fai, faj, fav, Lai.data(), Laj.data(), Lav.data(), D.data(), Uai.data(),
            Uaj.data(), Uav.data(), &ln, &un);
  for (int i = 0; i < n; ++i)
    if (D[i] == 0.0) throw la_error(LA_ERR_NUMERIC, "ILU factor has a zero or missing diagonal");
  P->lower = make_trsv(n, base, Lai.data(), Laj.data(), Lav.data(), nullptr, false, s);
  P->upper = make_trsv(n, base, Uai.data(), Uaj.data(), Uav.data(), D.data(), true, s);
  P->tmp[0].alloc(sizeof(double) * std::max(n, 1));
  P->tmp[1].alloc(sizeof(float) * std::max(n, 1));
  return P;
}

std::unique_ptr<Prec> make_prec_ic(int n, int base, const int *rai, const int *raj,
                                   const double *rav, hipStream_t s) {
  auto P = std::make_unique<Prec>();
  P->ic = true;
  P->n = n;
  P->stream = s;
  std::vector<int> Lai(static_cast<size_t>(n) + 1), Uai(static_cast<size_t>(n) + 1);
  int64_t ln = 0, un = 0;
  split_ldu(n, base, rai, raj, rav, Lai.data(), nullptr, nullptr, nullptr, Uai.data(), nullptr,
            nullptr, &ln, &un);
  LA_CHECK_ARG(ln == 0, "IC factor must be upper triangular");
  std::vector<int> Uaj(un);
  std::vector<double> Uav(un), D(n);
  split_ldu(n, base, rai, raj, rav, Lai.data(), nullptr, nullptr, D.data(), Uai.data(),
            Uaj.data(), Uav.data(), &ln, &un);
  for (int i = 0; i < n; ++i)
    if (!(D[i] > 0.0)) throw la_error(LA_ERR_NUMERIC, "IC factor has a non-positive diagonal");
  std::vector<int> ti(static_cast<size_t>(n) + 1), tj(un);
  std::vector<double> tv(un);
  transpose(n, n, base, Uai.data(), Uaj.data(), Uav.data(), ti.data(), tj.data(), tv.data());
  P->lower = make_trsv(n, base, ti.data(), tj.data(), tv.data(), D.data(), false, s);
  P->upper = make_trsv(n, base, Uai.data(), Uaj.data(), Uav.data(), D.data(), true, s);
  P->tmp[0].alloc(sizeof(double) * std::max(n, 1));
  P->tmp[1].alloc(sizeof(float) * std::max(n, 1));
  return P;
}

void prec_add_dtype(Prec &P, la_dtype dt) {
  trsv_add_dtype(*P.lower, dt);
  trsv_add_dtype(*P.upper, dt);
}

void prec_apply(Prec &P, la_trsv_mode mode, la_dtype val, la_dtype vec, const void *r, void *z,
                hipStream_t s) {
  void *t = P.tmp[vec == LA_F64 ? 0 : 1].p;
  trsv_solve(*P.lower, mode, val, vec, r, t, s);
  trsv_solve(*P.upper, mode, val, vec, t, z, s);
}

void prec_apply_transpose(Prec &P, la_trsv_mode mode, la_dtype val, la_dtype vec,
                          const void *r, void *z, hipStream_t s) {
  if (P.ic) return prec_apply(P, mode, val, vec, r, z, s);  // M = R^T R is symmetric
  void *t = P.tmp[vec == LA_F64 ? 0 : 1].p;
  // (LU)^-T = L^-T U^-T: solve U^T first (a lower solve), then L^T
  trsv_solve(trsv_transposed(*P.upper), mode, val, vec, r, t, s);
  trsv_solve(trsv_transposed(*P.lower), mode, val, vec, t, z, s);
}

}  // namespace laamd
