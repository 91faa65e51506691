// Pieces shared by the interpreted pass kernels (sv_passes.hip) and the lifted ones (sv_lift.hip): dispatch of
// run-time bits to compile-time op templates, tile movement between HBM and LDS, ragged records, and the
// argument checks and launch shape of a pass.
#pragma once

#include "sv_ops.h"

namespace tedq {

// Dispatch a runtime (target bit, control mask) to Op<R, B, CM> when the mask
// has at most one bit; returns false otherwise.
template <int R, template <int, int, int> class Op, int B, typename... A>
__device__ __forceinline__ bool by_ctrl(int cmask, A&... a) {
  switch (cmask) {
    case 0: Op<R, B, 0>::run(a...); return true;
    case 1: if constexpr (B != 0 && R > 1) { Op<R, B, 1>::run(a...); return true; } break;
    case 2: if constexpr (B != 1 && R > 2) { Op<R, B, 2>::run(a...); return true; } break;
    case 4: if constexpr (B != 2 && R > 4) { Op<R, B, 4>::run(a...); return true; } break;
    case 8: if constexpr (B != 3 && R > 8) { Op<R, B, 8>::run(a...); return true; } break;
    case 16: if constexpr (B != 4 && R > 16) { Op<R, B, 16>::run(a...); return true; } break;
    default: break;
  }
  return false;
}

template <int R, template <int, int, int> class Op, typename... A>
__device__ __forceinline__ bool by_bit(int b, int cmask, A&... a) {
  switch (b) {
    case 0: if constexpr (R > 1) return by_ctrl<R, Op, 0>(cmask, a...); break;
    case 1: if constexpr (R > 2) return by_ctrl<R, Op, 1>(cmask, a...); break;
    case 2: if constexpr (R > 4) return by_ctrl<R, Op, 2>(cmask, a...); break;
    case 3: if constexpr (R > 8) return by_ctrl<R, Op, 3>(cmask, a...); break;
    case 4: if constexpr (R > 16) return by_ctrl<R, Op, 4>(cmask, a...); break;
    default: break;
  }
  return false;
}

#define TEDQ_BIT_SWITCH(b, CALL)                        \
  switch (b) {                                          \
    case 0: if constexpr (R > 1) { CALL(0); } break;    \
    case 1: if constexpr (R > 2) { CALL(1); } break;    \
    case 2: if constexpr (R > 4) { CALL(2); } break;    \
    case 3: if constexpr (R > 8) { CALL(3); } break;    \
    case 4: if constexpr (R > 16) { CALL(4); } break;   \
    default: break;                                     \
  }

// ---------------------------------------------------------------------------
// tile addressing
// ---------------------------------------------------------------------------
struct TileCtx {
  int64_t circuit;     // circuit index of this thread's tile
  int64_t gbase;       // global element offset of local index 0 (G == 1 layout)
  uint64_t lo;         // physical offset contributed by the thread-id bits
  bool valid;
};

// Tiles are moved with buffer instructions: the resource (tile base, uniform
// per workgroup) lives in SGPRs, each lane adds a 32-bit offset and each
// register row a scalar offset, so no 64-bit address is held per element.
// Out-of-range buffer loads return 0 and stores are dropped, which covers the
// partial last workgroup of whole-circuit tiles.  States with more than 2^28
// amplitudes per circuit use plain global addressing.
//
// The swizzle is XOR-linear and a thread's LDS index is (thread part) |
// (register part) with disjoint bits, so swz(base | off) = swz(base) ^
// swz(off): register offsets in the stage header are stored pre-swizzled and
// each element costs one XOR.
template <int R, bool MULTI>
__device__ __forceinline__ void load_tiles(const float2* __restrict__ src, float2* lds, const int* __restrict__ prog,
                                           const PassArgs& a, int tid, int T, const TileCtx& c, int64_t blk) {
  const int sw = swz(tid);
  if (MULTI) {
    const int64_t wg_base = blk * T * R;
    const int64_t left = (a.batch << a.n) - wg_base;
    const int64_t cnt = left < (int64_t)T * R ? left : (int64_t)T * R;
    const __amdgpu_buffer_rsrc_t r = make_rsrc(src + wg_base, (uint32_t)(cnt * 8));
#pragma unroll
    for (int m = 0; m < R; ++m) lds[sw ^ swz(m * T)] = bload(r, (uint32_t)tid * 8u, (uint32_t)(m * T) * 8u);
  } else if (a.n <= 28) {
    const __amdgpu_buffer_rsrc_t r = make_rsrc(src + c.gbase, (uint32_t)(8u << a.n));
    const int64_t* hi = reinterpret_cast<const int64_t*>(prog + kHdrHiOff);
    const uint32_t vo = (uint32_t)c.lo * 8u;
#pragma unroll
    for (int m = 0; m < R; ++m) lds[sw ^ swz(m * T)] = bload(r, vo, (uint32_t)hi[m] * 8u);
  } else {
    const int64_t* hi = reinterpret_cast<const int64_t*>(prog + kHdrHiOff);
    const float2* p = src + c.gbase + c.lo;
#pragma unroll
    for (int m = 0; m < R; ++m) lds[sw ^ swz(m * T)] = p[hi[m]];
  }
}

template <int R, bool MULTI>
__device__ __forceinline__ void store_tiles(float2* __restrict__ dst, const float2* lds, const int* __restrict__ prog,
                                            const PassArgs& a, int tid, int T, const TileCtx& c, int64_t blk) {
  const int sw = swz(tid);
  if (MULTI) {
    const int64_t wg_base = blk * T * R;
    const int64_t left = (a.batch << a.n) - wg_base;
    const int64_t cnt = left < (int64_t)T * R ? left : (int64_t)T * R;
    const __amdgpu_buffer_rsrc_t r = make_rsrc(dst + wg_base, (uint32_t)(cnt * 8));
#pragma unroll
    for (int m = 0; m < R; ++m) bstore(lds[sw ^ swz(m * T)], r, (uint32_t)tid * 8u, (uint32_t)(m * T) * 8u);
  } else if (a.n <= 28) {
    const __amdgpu_buffer_rsrc_t r = make_rsrc(dst + c.gbase, (uint32_t)(8u << a.n));
    const int64_t* hi = reinterpret_cast<const int64_t*>(prog + kHdrHiOff);
    const uint32_t vo = (uint32_t)c.lo * 8u;
#pragma unroll
    for (int m = 0; m < R; ++m) bstore(lds[sw ^ swz(m * T)], r, vo, (uint32_t)hi[m] * 8u);
  } else {
    const int64_t* hi = reinterpret_cast<const int64_t*>(prog + kHdrHiOff);
    float2* p = dst + c.gbase + c.lo;
#pragma unroll
    for (int m = 0; m < R; ++m) p[hi[m]] = lds[sw ^ swz(m * T)];
  }
}

__device__ __forceinline__ TileCtx make_ctx(const PassArgs& a, const int* __restrict__ prog, int tid, bool multi,
                                            int64_t blk) {
  TileCtx c;
  if (multi) {
    const int64_t tile = (blk << a.gT) + (tid >> a.tT);
    c.circuit = tile;  // whole-circuit tiles
    c.valid = tile < a.batch;
    c.gbase = 0;
    c.lo = 0;
  } else {
    c.valid = true;
    tile_origin(a, blk, &c.circuit, &c.gbase);
    uint64_t lo = 0;
    for (int i = 0; i < a.tT; ++i)
      if ((tid >> i) & 1) lo |= 1ull << prog[kHdrTileBits + i];
    c.lo = lo;
  }
  return c;
}

// ---------------------------------------------------------------------------
// ragged passes: circuits of different structures and sizes in one launch
// (a serving batch).  Every circuit has its own state, program, matrices and
// partial rows; all share the tile bits k and register bits r, so one grid of
// 2^(k-r)-thread workgroups covers the tiles of all of them.  Workgroup b
// belongs to the first record whose tile_end exceeds b.
// ---------------------------------------------------------------------------
struct RaggedRec {
  float2* psi;           // the circuit's state [2^n]
  float2* lam;           // adjoint: its lambda [2^n]
  const int* prog;       // its program for this pass (forward or adjoint)
  const float2* mats;    // its slot matrices (one table row)
  float* partials;       // adjoint: its partial rows [n_gslots][2^(n-k) * W][8]
  uint64_t rest_mask;    // physical bits of the circuit that are not tile bits of this pass
  int64_t tile_end;      // tiles of this and all earlier records
  int n;
  int n_gslots;
};
static_assert(sizeof(RaggedRec) == 64, "ragged record layout is part of the C ABI");

__device__ __forceinline__ int ragged_record(const RaggedRec* __restrict__ recs, int nrec, int64_t blk) {
  int lo = 0, hi = nrec - 1;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (recs[mid].tile_end > blk) hi = mid;
    else lo = mid + 1;
  }
  return __builtin_amdgcn_readfirstlane(lo);
}

// The record is the same for the whole workgroup: read every word through readfirstlane so that the
// compiler keeps pointers, masks and sizes in scalar registers (as kernel arguments are).
__device__ __forceinline__ uint64_t uniform64(uint64_t v) {
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return ((uint64_t)hi << 32) | lo;
}

// A pointer read from memory is generic (flat); taking it through the global address space lets the
// compiler issue global (and, for uniform read-only words such as the program, scalar) loads, as it does
// for pointer kernel arguments.
template <class T>
__device__ __forceinline__ T* global_ptr(const void* p) {
  return (T*)(__attribute__((address_space(1))) T*)uniform64(reinterpret_cast<uint64_t>(p));
}

__device__ __forceinline__ RaggedRec load_record(const RaggedRec* __restrict__ recs, int c) {
  RaggedRec r;
  const RaggedRec& g = recs[c];
  r.psi = global_ptr<float2>(g.psi);
  r.lam = global_ptr<float2>(g.lam);
  r.prog = global_ptr<const int>(g.prog);
  r.mats = global_ptr<const float2>(g.mats);
  r.partials = global_ptr<float>(g.partials);
  r.rest_mask = uniform64(g.rest_mask);
  r.tile_end = (int64_t)uniform64((uint64_t)g.tile_end);
  r.n = __builtin_amdgcn_readfirstlane(g.n);
  r.n_gslots = __builtin_amdgcn_readfirstlane(g.n_gslots);
  return r;
}

__device__ __forceinline__ PassArgs ragged_args(const RaggedRec& rc, int k, int tT) {
  PassArgs a;
  a.mat_stride = 0;
  a.batch = 1;
  a.total_tiles = 1ll << (rc.n - k);
  a.rest_mask = rc.rest_mask;
  a.n = rc.n;
  a.k = k;
  a.tT = tT;
  a.gT = 0;
  const int W = tT > 6 ? 1 << (tT - 6) : 1;
  a.np = (1ll << (rc.n - k)) * W;
  a.n_gslots = rc.n_gslots;
  a.flags = 0;
  return a;
}

// gfx950 provides 160 KiB of LDS per workgroup; above 64 KiB the kernel must opt in once.
constexpr size_t kMaxLds = 160 * 1024;

template <typename K>
static bool allow_lds(K kernel, size_t lds) {
  if (lds <= 65536) return true;
  return hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                             (int)lds) == hipSuccess;
}

// Arguments of a pass over [batch][2^n] states, checked, and its launch shape.  Returns kOk or an error (set).
struct PassLaunch {
  PassArgs a;
  unsigned blocks, threads;
  size_t lds;
  bool multi;
};

static inline int plan_pass(bool adjoint, const void* psi, const void* lam, int64_t batch, int n, int k, int r,
                            int threads_log2, const int* dev_prog, uint64_t tile_mask, uint64_t zero_mask,
                            int64_t mat_stride, const float* partials, int64_t np, int n_gslots, PassLaunch* L) {
  if (psi == nullptr || (adjoint && (lam == nullptr || (n_gslots > 0 && partials == nullptr))) ||
      dev_prog == nullptr || batch <= 0 || n < 1 || n > 40 || k < 1 || k > n || r < 1 || r > 5 || r > k) {
    set_error("sv pass: bad arguments (batch=%lld n=%d k=%d r=%d)", (long long)batch, n, k, r);
    return kBadArgument;
  }
  const int tT = k - r;
  if (threads_log2 < tT || threads_log2 > 9 || (threads_log2 > tT && k != n)) {
    set_error("sv pass: threads_log2=%d incompatible with k=%d r=%d n=%d", threads_log2, k, r, n);
    return kBadArgument;
  }
  // whole circuits, several to a workgroup; a circuit that fills its workgroup is an ordinary tile, whose
  // matrix row is then uniform
  const bool multi = L->multi = threads_log2 > tT;
  const uint64_t full = (n >= 64) ? ~0ull : ((1ull << n) - 1);
  if (__builtin_popcountll(tile_mask & full) != k || (tile_mask & ~full) != 0) {
    set_error("sv pass: tile mask does not have k=%d bits below n=%d", k, n);
    return kBadArgument;
  }
  if ((zero_mask & (tile_mask | ~full)) != 0) {
    set_error("sv pass: zero mask 0x%llx holds tile bits or bits above n", (unsigned long long)zero_mask);
    return kBadArgument;
  }
  PassArgs& a = L->a;
  a.mat_stride = mat_stride;
  a.batch = batch;
  a.rest_mask = full & ~tile_mask & ~zero_mask;
  a.total_tiles = batch << __builtin_popcountll(a.rest_mask);
  a.n = n;
  a.k = k;
  a.tT = tT;
  a.gT = threads_log2 - tT;
  a.np = np;
  a.n_gslots = n_gslots;
  a.flags = 0;
  const int T = 1 << threads_log2;
  const int R = 1 << r;
  int64_t blocks;
  if (multi) {
    const int64_t tiles_per_wg = 1ll << a.gT;
    blocks = (batch + tiles_per_wg - 1) / tiles_per_wg;
  } else {
    blocks = a.total_tiles;
  }
  if (blocks > 0x7fffffffll) {
    set_error("sv pass: grid too large (%lld blocks)", (long long)blocks);
    return kBadArgument;
  }
  L->blocks = (unsigned)blocks;
  L->threads = (unsigned)T;
  L->lds = (size_t)T * R * sizeof(float2) * (adjoint ? 2 : 1);
  if (L->lds > kMaxLds) {
    set_error("sv pass: LDS request %zu bytes exceeds %zu", L->lds, kMaxLds);
    return kBadArgument;
  }
  return kOk;
}

}  // namespace tedq
