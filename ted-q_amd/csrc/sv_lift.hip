// Lifted state-vector passes: the interpreted pass kernels of plans whose stages are rounds of in-place
// register ops (tedq_amd/engine/lift.py).
//
// What bounds an interpreted pass is VALU issue: in sv_passes.hip every arm of the op dispatch leaves its
// results in registers of its own, the join after it copies them back, and only about 40% of the VALU
// instructions do arithmetic.  A round has no dispatch: under wave-uniform branches, in a fixed order, it
// multiplies by a diagonal, rotates the register bits that have a gate (one multiply-add per output, the
// common factor left to the second diagonal), multiplies by a diagonal that holds every phase and factor, and
// permutes by the order in which it writes its amplitudes to LDS.  Trained rotations stay unfused, so a
// gradient is one number per parameter instead of a fused gate's 8 bilinears, and the diagonal gates of a
// round share the products of their gradients (Im conj(lambda) psi per amplitude).
//
// Tiles, LDS layout and partial rows are those of sv_passes.hip; stage words (lift.py) hold, per round:
// [0] flags (1: amplitudes still in registers, 2: leave them there, 4: barrier, 8: D0, 16: D1, 32: D1 is the
// rotations' factor alone)
// [1] register mask [2] RX bits | RY bits << 8 [3] table offset (complex64) of D1, rotations, forms, D0 [4] sign per amplitude [5] general ops [6] their word offset [7] gradient bits of
// rotations | D1 << 8 | D0 << 16 [8] PhaseShift bits of D1 | D0 << 8 [9] gradient slot of rotations and D1
// [10] of D0 [12..44) LDS offsets read from [44..76) written to.
// Replaces the reference loop tedq/backends/pytorch_backend.py:358-380 and torch autograd through it.
#include "sv_tiles.h"

namespace tedq {

constexpr int kLiftWords = 80;
enum LiftWord : int { kLwFlags, kLwRegmask, kLwRot, kLwCoef, kLwSign, kLwNGen, kLwGen, kLwGrads, kLwKindP, kLwGroup,
                      kLwGroupPre, kLwIn = 12, kLwOut = 44 };
constexpr int kLiftSkipRead = 1, kLiftSkipWrite = 2, kLiftBarrier = 4, kLiftD0 = 8, kLiftD1 = 16, kLiftScale = 32;

// ---------------------------------------------------------------------------
// general ops (dense 4x4, controlled rotations, user matrices): dispatched, as in sv_passes.hip
// ---------------------------------------------------------------------------
// x = t with the output tied to x's own register, so that every arm leaves its results where they were:
// without it the compiler gives arms result registers of their own and copies all amplitudes at every join
struct InPlace {
  __device__ __forceinline__ void operator()(float& x, float t) const {
    asm("v_mov_b32 %0, %1" : "+v"(x) : "v"(t));
  }
};
__device__ __forceinline__ void set_in_place(float2& x, float2 t) {
  InPlace()(x.x, t.x);
  InPlace()(x.y, t.y);
}

template <int R, int B, int CM>
struct LiftU1 {
  static __device__ __forceinline__ void run(float2 (&v)[R], float2 m0, float2 m1, float2 m2, float2 m3) {
#pragma unroll
    for (int i = 0; i < R; ++i) {
      if ((i & (1 << B)) || (i & CM) != CM) continue;
      const int j = i | (1 << B);
      const float2 x = cmul2(m0, v[i], m1, v[j]), y = cmul2(m2, v[i], m3, v[j]);
      set_in_place(v[i], x);
      set_in_place(v[j], y);
    }
  }
};
template <int R, int B, int CM>
struct LiftPhase {
  static __device__ __forceinline__ void run(float2 (&v)[R], float2 p) {
#pragma unroll
    for (int i = 0; i < R; ++i)
      if ((i & (CM | (1 << B))) == (CM | (1 << B))) set_in_place(v[i], cmul(p, v[i]));
  }
};
template <int R, int B, int CM> struct GradXOp : PauliGradOp<R, B, CM, kGradX, false> {};
template <int R, int B, int CM> struct GradYOp : PauliGradOp<R, B, CM, kGradY, false> {};
template <int R, int B, int CM> struct GradZOp : PauliGradOp<R, B, CM, kGradZ, false> {};
template <int R, int B, int CM> struct GradPOp : PauliGradOp<R, B, CM, kGradP, false> {};

template <int R, int B1, int B0>
__device__ __forceinline__ void lift_u2_pair(float2 (&v)[R], const float2 (&m)[16]) {
#pragma unroll
  for (int i = 0; i < R; ++i) {
    if (i & ((1 << B1) | (1 << B0))) continue;
    const int j[4] = {i, i | (1 << B0), i | (1 << B1), i | (1 << B0) | (1 << B1)};
    float2 o[4];
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      o[a] = make_float2(0.f, 0.f);
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        const float2 u = m[a * 4 + b], x = v[j[b]];
        o[a].x = fmaf(u.x, x.x, fmaf(-u.y, x.y, o[a].x));
        o[a].y = fmaf(u.x, x.y, fmaf(u.y, x.x, o[a].y));
      }
    }
#pragma unroll
    for (int a = 0; a < 4; ++a) set_in_place(v[j[a]], o[a]);
  }
}
template <int R>
__device__ __forceinline__ void lift_u2(float2 (&v)[R], int b1, int b0, const float2 (&m)[16]) {
  switch (b1 * (b1 - 1) / 2 + b0) {   // pairs b1 > b0: (1,0) (2,0) (2,1) (3,0) ...
    case 0: if constexpr (R > 2) lift_u2_pair<R, 1, 0>(v, m); break;
    case 1: if constexpr (R > 4) lift_u2_pair<R, 2, 0>(v, m); break;
    case 2: if constexpr (R > 4) lift_u2_pair<R, 2, 1>(v, m); break;
    case 3: if constexpr (R > 8) lift_u2_pair<R, 3, 0>(v, m); break;
    case 4: if constexpr (R > 8) lift_u2_pair<R, 3, 1>(v, m); break;
    case 5: if constexpr (R > 8) lift_u2_pair<R, 3, 2>(v, m); break;
    case 6: if constexpr (R > 16) lift_u2_pair<R, 4, 0>(v, m); break;
    case 7: if constexpr (R > 16) lift_u2_pair<R, 4, 1>(v, m); break;
    case 8: if constexpr (R > 16) lift_u2_pair<R, 4, 2>(v, m); break;
    case 9: if constexpr (R > 16) lift_u2_pair<R, 4, 3>(v, m); break;
    default: break;
  }
}

template <int R, bool TWO>
__device__ __forceinline__ void general_op(float2 (&v)[R], float2 (&w)[R], const int* __restrict__ op,
                                           const float2* __restrict__ mb) {
  const int type = op[0] & 0xff;
  const bool dag = (op[0] >> 8) & 1;
  if (type == kOpU2) {
    float2 m[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) m[i] = mb[op[4] + i];
    lift_u2<R>(v, op[1], op[2], m);
    if (TWO) lift_u2<R>(w, op[1], op[2], m);
  } else if (type == kOpPhaseLift) {
    float2 p = dag ? cconj(mb[op[4]]) : mb[op[4]];
    by_bit<R, LiftPhase>(op[1], op[3], v, p);
    if (TWO) by_bit<R, LiftPhase>(op[1], op[3], w, p);
  } else {
    float2 m[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) m[i] = mb[op[4] + i];
    if (type == kOpD1 || type == kOpCD1) m[1] = m[2] = make_float2(0.f, 0.f);
    if (dag) {
      const float2 t = m[1];
      m[0] = cconj(m[0]);
      m[1] = cconj(m[2]);
      m[2] = cconj(t);
      m[3] = cconj(m[3]);
    }
    by_bit<R, LiftU1>(op[1], op[3], v, m[0], m[1], m[2], m[3]);
    if (TWO) by_bit<R, LiftU1>(op[1], op[3], w, m[0], m[1], m[2], m[3]);
  }
}

template <int R>
__device__ __forceinline__ float general_grad(const float2 (&p)[R], const float2 (&l)[R], const int* __restrict__ op) {
  float v = 0.f;
  switch (op[6] & 15) {
    case kGradX: by_bit<R, GradXOp>(op[1], op[3], p, l, v); break;
    case kGradY: by_bit<R, GradYOp>(op[1], op[3], p, l, v); break;
    case kGradZ: by_bit<R, GradZOp>(op[1], op[3], p, l, v); break;
    default: by_bit<R, GradPOp>(op[1], op[3], p, l, v); break;
  }
  return (op[6] >> 4) ? -v : v;
}

// ---------------------------------------------------------------------------
// a round's fixed part; masks and coefficients are uniform, R = 2^r with r <= 5 register bits
// ---------------------------------------------------------------------------
#define TEDQ_EACH_BIT(CALL)       \
  do {                            \
    if constexpr (R > 1) CALL(0)  \
    if constexpr (R > 2) CALL(1)  \
    if constexpr (R > 4) CALL(2)  \
    if constexpr (R > 8) CALL(3)  \
    if constexpr (R > 16) CALL(4) \
  } while (0)

// rotations on the bits of `mask` by the q at rt[bit].x, in the second form on the bits of `cots`; DAG: the
// transposed.  The two forms are two branches without an else, kept apart by an empty asm: where two arms meet,
// the compiler gives their results new registers and copies all amplitudes at the join (64 copies per 64
// multiply-adds in the adjoint, read off the generated code); behind a branch without an else they stay.
template <int R, bool TWO, bool DAG, int KIND>
__device__ __forceinline__ void round_rotations(float2 (&v)[R], float2 (&w)[R], int mask, int cots,
                                                const float (&qs)[5]) {
#define CALL(B)                                             \
  if ((mask >> B) & 1) {                                    \
    const float q = qs[B];                                  \
    if ((cots >> B) & 1) {                                  \
      rotate_unscaled<R, B, KIND, true, DAG>(v, q);         \
      if (TWO) rotate_unscaled<R, B, KIND, true, DAG>(w, q);  \
    }                                                       \
    asm volatile("");                                       \
    if (!((cots >> B) & 1)) {                               \
      rotate_unscaled<R, B, KIND, false, DAG>(v, q);        \
      if (TWO) rotate_unscaled<R, B, KIND, false, DAG>(w, q); \
    }                                                       \
  }
  TEDQ_EACH_BIT(CALL);
#undef CALL
}

template <int R, int KIND>
__device__ __forceinline__ void rotation_grads(const float2 (&p)[R], const float2 (&l)[R], int bits, float (&acc)[8]) {
#define CALL(B) \
  if constexpr (B < 4) { if ((bits >> B) & 1) PauliGradOp<R, B, 0, KIND, false>::run(p, l, acc[B]); }
  TEDQ_EACH_BIT(CALL);
#undef CALL
}

// swizzled LDS index of this thread's register 0 in a stage: the tile's thread bits with a zero inserted at
// every register bit (regmask, ascending)
__device__ __forceinline__ int lift_stage_base(int tid, int tT, int k, int regmask) {
  int x = tid & ((1 << tT) - 1);
  for (int mask = regmask; mask; mask &= mask - 1) {
    const int low = x & ((mask & -mask) - 1);
    x = ((x - low) << 1) | low;
  }
  return swz(((tid >> tT) << k) + x);
}

// partial row of a gradient group: acc summed over the tile's lanes, and cleared
__device__ __forceinline__ void flush_group(float (&acc)[8], float* dst, int seg, int lane, bool writer) {
  if (seg == 64) {
    const float tot = reduce8_wave(acc, lane);
    if ((lane & 7) == 0) dst[(lane >> 3) & 7] = tot;
  } else {
#pragma unroll
    for (int q = 0; q < 8; ++q)
      for (int off = 1; off < seg; off <<= 1) acc[q] += __shfl_xor(acc[q], off, 64);
    if (writer) {
      float4* d4 = reinterpret_cast<float4*>(dst);
      d4[0] = make_float4(acc[0], acc[1], acc[2], acc[3]);
      d4[1] = make_float4(acc[4], acc[5], acc[6], acc[7]);
    }
  }
#pragma unroll
  for (int q = 0; q < 8; ++q) acc[q] = 0.f;
}

// A uniform value made to arrive in a scalar register at this point.
__device__ __forceinline__ void pin(int& x) {
  x = __builtin_amdgcn_readfirstlane(x);
  asm volatile("" : "+s"(x));
}
__device__ __forceinline__ void pin(float& x) {
  int i = __builtin_bit_cast(int, x);
  pin(i);
  x = __builtin_bit_cast(float, i);
}

// What a round's control flow needs, held in scalar registers and read one round ahead: its first words, then
// its table row's ratios and forms (and a touch of the row's other lines).  Read where it is used, each is a
// scalar load that the wave waits for alone, about ten in turn per round.
template <int R>
struct RoundHead {
  int flags, regmask, rot, coef, sign, grads, kindp, group, group_pre, cots;
  float q[5], line0, line1;
  __device__ __forceinline__ void words(const int* __restrict__ st) {
    flags = st[kLwFlags];
    regmask = st[kLwRegmask];
    rot = st[kLwRot];
    coef = st[kLwCoef];
    sign = st[kLwSign];
    grads = st[kLwGrads];
    kindp = st[kLwKindP];
    group = st[kLwGroup];
    group_pre = st[kLwGroupPre];
  }
  template <bool MULTI>
  __device__ __forceinline__ void row(const float2* __restrict__ mb) {
    const float2* d1 = mb + coef;
#pragma unroll
    for (int i = 0; i < 5; ++i) q[i] = i < log2c(R) ? d1[R + i].x : 0.f;
    cots = __builtin_bit_cast(int, d1[R + log2c(R)].x);
    if (!MULTI) {
      line0 = d1[0].x;
      line1 = d1[R / 2].x;
    }
  }
  // the loads are issued before here and waited for here (the row of whole-circuit tiles is the lane's own)
  template <bool MULTI>
  __device__ __forceinline__ void arrive() {
    pin(flags), pin(regmask), pin(rot), pin(coef), pin(sign), pin(grads), pin(kindp), pin(group), pin(group_pre);
    if (!MULTI) {
      pin(cots), pin(line0), pin(line1);
#pragma unroll
      for (int i = 0; i < log2c(R); ++i) pin(q[i]);
    }
  }
};

// Touch the lines of the pass's program and of the circuit's table rows while the tile loads are in flight.
// Both were written by another kernel, so the first scalar load of each line misses this XCD's L2 and every
// round waits for two or three of them in turn; with one tile per circuit there is no other workgroup to hide
// it behind.  With the reads ahead of RoundHead: first pass of 32 17-qubit circuits 60 -> 45 us forward and
// 88 -> 71 us adjoint; 48 20-qubit forwards, 12288 tiles a pass, 3.74 -> 3.46 ms.
__device__ __forceinline__ void warm_lines(const int* __restrict__ prog, const float2* __restrict__ mb, int nst, int row) {
  const int t = threadIdx.x, T = blockDim.x;
  const int words = kHdrStages + kLiftWords * nst;
  const int c0 = prog[kHdrStages + kLwCoef], c1 = prog[kHdrStages + kLiftWords * (nst - 1) + kLwCoef];
  const int lo = c0 < c1 ? c0 : c1, hi = (c0 < c1 ? c1 : c0) + row;
  int w = 0;
  float c = 0.f;
  for (int i = 32 * t; i < words; i += 32 * T) w ^= prog[i];
  for (int i = lo + 16 * t; i < hi; i += 16 * T) c += mb[i].x;
  asm volatile("" ::"v"(w), "v"(c));
}

// Workgroup `blk` of a lifted pass (a tile, or G whole circuits when MULTI), forward or adjoint.  GEN: the pass
// has general ops (without them the kernel needs a third fewer registers and no copies around their dispatch).
template <int R, bool ADJ, bool MULTI, bool GEN>
__device__ __forceinline__ void lift_body(float2* __restrict__ psi, float2* __restrict__ lam,
                                          const int* __restrict__ prog, const float2* __restrict__ mats,
                                          float* __restrict__ partials, const PassArgs& a, int64_t blk) {
  extern __shared__ float2 lds[];
  const int T = blockDim.x;
  float2* ldp = lds;
  float2* ldl = ADJ ? lds + T * R : lds;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const TileCtx c = make_ctx(a, prog, tid, MULTI, blk);
  const float2* mb = mats + (c.valid ? c.circuit : 0) * a.mat_stride;
  const int nst = prog[2];
  if (!MULTI) warm_lines(prog, mb, nst, R + log2c(R) + 1);
  load_tiles<R, MULTI>(psi, ldp, prog, a, tid, T, c, blk);
  if (ADJ) load_tiles<R, MULTI>(lam, ldl, prog, a, tid, T, c, blk);
  __syncthreads();

  // partial rows: W waves per tile when a tile spans several waves
  const int tpt = 1 << a.tT;                 // threads per tile
  const int seg = tpt < 64 ? tpt : 64;       // lanes reduced together
  const int W = tpt >> 6 > 0 ? tpt >> 6 : 1; // partial rows per tile
  const int tl = tid & (tpt - 1);
  const int64_t tile_in_circuit = MULTI ? 0 : (blk & ((1ll << tiles_log2(a)) - 1));
  const int64_t prow = tile_in_circuit * W + (tl >> 6);
  const bool writer = c.valid && (tid & (seg - 1)) == 0;
  float* const pbase = partials + (c.circuit * a.n_gslots * a.np + prow) * 8;
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  float2 vp[R], vl[R];
#pragma unroll
  for (int m = 0; m < R; ++m) vp[m] = vl[m] = make_float2(0.f, 0.f);
  RoundHead<R> h;
  h.words(prog + kHdrStages);
  h.template row<MULTI>(mb);
  for (int s = 0; s < nst; ++s) {
    const int* st = prog + kHdrStages + kLiftWords * s;
    const int flags = h.flags, rx = h.rot & 31, ry = (h.rot >> 8) & 31;
    const int sb = lift_stage_base(tid, a.tT, a.k, h.regmask);
    const float2* d1 = mb + h.coef;
    const float2* d0 = d1 + R + log2c(R) + 1;
    const int cots = (rx | ry) ? h.cots : 0;
    RoundHead<R> nx;
    const int* next = s + 1 < nst ? st + kLiftWords : st;
    if (!GEN) nx.words(next);  // (the general ops' words and matrices need the scalar registers)
    if (!(flags & kLiftSkipRead)) {
#pragma unroll
      for (int m = 0; m < R; ++m) {
        vp[m] = ldp[sb ^ st[kLwIn + m]];
        if (ADJ) vl[m] = ldl[sb ^ st[kLwIn + m]];
      }
    }
    const uint32_t sign = (uint32_t)h.sign;
    const int ngen = GEN ? st[kLwNGen] : 0;
    if (!ADJ) {
      if (flags & kLiftD0) scale_diagonal<R, false>(vp, d0, InPlace());
      if (rx) round_rotations<R, false, false, 0>(vp, vl, rx, cots, h.q);
      if (ry) round_rotations<R, false, false, 1>(vp, vl, ry, cots, h.q);
      if (flags & kLiftD1) scale_diagonal<R, false>(vp, d1, InPlace());
      if (flags & kLiftScale) scale_all<R>(vp, d1->x);
      for (int o = 0; o < ngen; ++o) general_op<R, false>(vp, vl, prog + st[kLwGen] + 8 * o, mb);
      if (sign) round_signs<R>(vp, sign);
    } else {
      const int gr = h.grads, kindp = h.kindp;
      if (sign) {
        round_signs<R>(vp, sign);
        round_signs<R>(vl, sign);
      }
      for (int o = 0; o < ngen; ++o) {
        const int* op = prog + st[kLwGen] + 8 * o;
        if ((op[0] & 0xff) == kOpPauliGrad) {
          float g[8] = {general_grad<R>(vp, vl, op), 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
          flush_group(g, pbase + (int64_t)op[5] * a.np * 8, seg, lane, writer);
        } else {
          general_op<R, true>(vp, vl, op, mb);
        }
      }
      if ((gr >> 8) & 31) phase_grads<R>(vp, vl, (gr >> 8) & 31, kindp & 31, acc);
      if (flags & kLiftD1) {
        scale_diagonal<R, true>(vp, d1, InPlace());
        scale_diagonal<R, true>(vl, d1, InPlace());
      }
      if (flags & kLiftScale) {
        const float f = d1->x;
        scale_all<R>(vp, f);
        scale_all<R>(vl, f);
      }
      if (rx) round_rotations<R, true, true, 0>(vp, vl, rx, cots, h.q);
      if (ry) round_rotations<R, true, true, 1>(vp, vl, ry, cots, h.q);
      // (a rotation commutes with its generator: its gradient may be taken before it, where no factor is pending)
      if (gr & rx) rotation_grads<R, kGradX>(vp, vl, gr & rx, acc);
      if (gr & ry) rotation_grads<R, kGradY>(vp, vl, gr & ry, acc);
      if (h.group >= 0) flush_group(acc, pbase + (int64_t)h.group * a.np * 8, seg, lane, writer);
      if (h.group_pre >= 0) {
        phase_grads<R>(vp, vl, (gr >> 16) & 31, (kindp >> 8) & 31, acc);
        flush_group(acc, pbase + (int64_t)h.group_pre * a.np * 8, seg, lane, writer);
      }
      if (flags & kLiftD0) {
        scale_diagonal<R, true>(vp, d0, InPlace());
        scale_diagonal<R, true>(vl, d0, InPlace());
      }
    }
    if (GEN) nx.words(next);
    nx.template row<MULTI>(mb);
    if (!(flags & kLiftSkipWrite)) {
#pragma unroll
      for (int m = 0; m < R; ++m) {
        ldp[sb ^ st[kLwOut + m]] = vp[m];
        if (ADJ) ldl[sb ^ st[kLwOut + m]] = vl[m];
      }
    }
    nx.template arrive<MULTI>();
    h = nx;
    if (flags & kLiftBarrier) __syncthreads();
  }
  store_tiles<R, MULTI>(psi, ldp, prog, a, tid, T, c, blk);
  if (ADJ) store_tiles<R, MULTI>(lam, ldl, prog, a, tid, T, c, blk);
}

template <int R, bool ADJ, bool MULTI, bool GEN>
__global__ void __launch_bounds__(512) k_lift(float2* __restrict__ psi, float2* __restrict__ lam,
                                              const int* __restrict__ prog, const float2* __restrict__ mats,
                                              float* __restrict__ partials, PassArgs a) {
  lift_body<R, ADJ, MULTI, GEN>(psi, lam, prog, mats, partials, a, blockIdx.x);
}

template <int R, bool ADJ, bool GEN>
__global__ void __launch_bounds__(512) k_lift_ragged(const RaggedRec* __restrict__ recs, int nrec, int k, int tT) {
  const int c = ragged_record(recs, nrec, blockIdx.x);
  const RaggedRec rc = load_record(recs, c);
  const int64_t first = c ? (int64_t)uniform64((uint64_t)recs[c - 1].tile_end) : 0;
  lift_body<R, ADJ, false, GEN>(rc.psi, rc.lam, rc.prog, rc.mats, rc.partials, ragged_args(rc, k, tT),
                                (int64_t)blockIdx.x - first);
}

template <int R, bool ADJ, bool GEN>
static int launch_lift(const PassLaunch& L, hipStream_t st, float2* psi, float2* lam, const int* prog,
                       const float2* mats, float* partials) {
  bool ok;
  if (L.multi) {
    ok = allow_lds(k_lift<R, ADJ, true, GEN>, L.lds);
    if (ok)
      hipLaunchKernelGGL((k_lift<R, ADJ, true, GEN>), dim3(L.blocks), dim3(L.threads), L.lds, st, psi, lam, prog, mats,
                         partials, L.a);
  } else {
    ok = allow_lds(k_lift<R, ADJ, false, GEN>, L.lds);
    if (ok)
      hipLaunchKernelGGL((k_lift<R, ADJ, false, GEN>), dim3(L.blocks), dim3(L.threads), L.lds, st, psi, lam, prog, mats,
                         partials, L.a);
  }
  if (!ok) {
    set_error("lifted pass: could not enable %zu bytes of LDS", L.lds);
    return kLaunchFailed;
  }
  return check_launch("tedq_sv_lift_pass");
}

template <int R, bool ADJ, bool GEN>
static int launch_lift_ragged(const RaggedRec* recs, int nrec, int64_t tiles, int k, int r, hipStream_t st) {
  const size_t lds = ((size_t)8 << k) * (ADJ ? 2 : 1);
  if (!allow_lds(k_lift_ragged<R, ADJ, GEN>, lds)) {
    set_error("lifted ragged pass: could not enable %zu bytes of LDS", lds);
    return kLaunchFailed;
  }
  hipLaunchKernelGGL((k_lift_ragged<R, ADJ, GEN>), dim3((unsigned)tiles), dim3(1u << (k - r)), lds, st, recs, nrec, k,
                     k - r);
  return check_launch("tedq_sv_lift_pass_ragged");
}

}  // namespace tedq

using namespace tedq;

// flags: 1 adjoint, 2 the pass has general ops.  r registers per thread: 1..5 forward, 1..4 adjoint (psi and
// lambda of 32 amplitudes would spill, and a gradient group has four bits' values)
#define TEDQ_LIFT_R(RUN, ADJ, GEN, FIVE)       \
  switch (r) {                                 \
    case 1: return RUN(2, ADJ, GEN);           \
    case 2: return RUN(4, ADJ, GEN);           \
    case 3: return RUN(8, ADJ, GEN);           \
    case 4: return RUN(16, ADJ, GEN);          \
    FIVE                                       \
    default: break;                            \
  }
#define TEDQ_LIFT_CASES(RUN)                                                    \
  switch (flags) {                                                              \
    case 0: TEDQ_LIFT_R(RUN, false, false, case 5: return RUN(32, false, false);) break;  \
    case 2: TEDQ_LIFT_R(RUN, false, true, case 5: return RUN(32, false, true);) break;    \
    case 1: TEDQ_LIFT_R(RUN, true, false, ) break;                              \
    case 3: TEDQ_LIFT_R(RUN, true, true, ) break;                               \
    default: break;                                                             \
  }

extern "C" int tedq_sv_lift_pass(int flags, void* psi, void* lam, int64_t batch, int n_qubits, int tile_bits,
                                 int reg_bits, int threads_log2, const int* dev_prog, uint64_t tile_mask,
                                 uint64_t zero_mask, const void* mats, int64_t mat_stride, float* partials,
                                 int64_t partial_rows, int n_gslots, void* stream) {
  PassLaunch L;
  const int r = reg_bits;
  const int rc = plan_pass(flags & 1, psi, lam, batch, n_qubits, tile_bits, r, threads_log2, dev_prog, tile_mask,
                           zero_mask, mat_stride, partials, partial_rows, n_gslots, &L);
  if (rc != kOk) return rc;
  float2* p = static_cast<float2*>(psi);
  float2* l = static_cast<float2*>(lam);
  const float2* mt = static_cast<const float2*>(mats);
  hipStream_t st = static_cast<hipStream_t>(stream);
#define RUN(R, ADJ, GEN) launch_lift<R, ADJ, GEN>(L, st, p, l, dev_prog, mt, partials)
  TEDQ_LIFT_CASES(RUN)
#undef RUN
  set_error("tedq_sv_lift_pass: flags %d or register bits %d out of range", flags, r);
  return kBadArgument;
}

extern "C" int tedq_sv_lift_pass_ragged(int flags, const void* dev_recs, int n_recs, int64_t total_tiles, int k,
                                        int r, void* stream) {
  const int adjoint = flags & 1;
  if (dev_recs == nullptr || n_recs < 1 || total_tiles < n_recs || total_tiles > 0x7fffffffll || k < 1 || k > 20 ||
      flags < 0 || flags > 3 || r < 1 || r > (adjoint ? 4 : 5) || r > k || k - r > 9 ||
      ((size_t)8 << k) * (adjoint ? 2 : 1) > kMaxLds) {
    set_error("tedq_sv_lift_pass_ragged: bad arguments (records=%d tiles=%lld k=%d r=%d flags=%d)", n_recs,
              (long long)total_tiles, k, r, flags);
    return kBadArgument;
  }
  const RaggedRec* recs = static_cast<const RaggedRec*>(dev_recs);
  hipStream_t st = static_cast<hipStream_t>(stream);
#define RUN(R, ADJ, GEN) launch_lift_ragged<R, ADJ, GEN>(recs, n_recs, total_tiles, k, r, st)
  TEDQ_LIFT_CASES(RUN)
#undef RUN
  return kBadArgument;
}
