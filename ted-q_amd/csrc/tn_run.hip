// Runs of gates on one large tensor, a tile of address bits at a time.
//
// A contraction path applies gate-sized tensors one after another to the same
// state-like intermediate.  k_tn_gate does one of them per launch and is
// bound by HBM: 2^25 elements are read and written in 92 us (5.8 TB/s) for 16
// multiply-adds per element.  Here the host groups such steps into square
// matrices on two or three address bits and the matrices into passes; a pass
// loads a tile of up to 2^12 elements into LDS, applies all its matrices in
// place and stores it, so the tensor crosses HBM once per pass.
//
// Matrices are applied on the FP32 matrix cores: v_mfma_f32_4x4x1 (16 blocks)
// takes one column per lane and gives back the four results in the same lane,
// so a lane reads the 4 (8) elements of a row of the tile, issues 16 (64)
// MFMAs and writes them back; the multiply-adds are the same fused ones as on
// the vector units at twice their rate (packed FP32 is not used).
//
//   * k_tn_run_coefs: the matrices, as products of the ops' factors;
//   * k_tn_run_pass: one forward pass;
//   * k_tn_run_bwd: one backward pass: from the pass's result C and its
//     environment E it undoes the ops (their matrices are unitary), leaving
//     the environment of the pass's input and, per op, the environment of its
//     matrix;
//   * k_tn_run_env: adds those over workgroups into the gates' tensors.
#include "tedq_common.h"

namespace tedq {

namespace {

constexpr int kTileMax = 12, kTileMin = 9, kOuterMax = 20;
constexpr int kRunOps = 32, kRunCoef = 512;
constexpr int kOpWords = 52, kPassWords = 128, kFactors = 4;
constexpr int kBwdLog = 9, kBwdThreads = 1 << kBwdLog;

typedef float f32x4 __attribute__((ext_vector_type(4)));

// op words (host: tn/runs.py encode_op)
enum { W_ARITY = 0, W_SLOT = 1, W_DELTA = 4, W_INTERNAL = 5, W_FACTORS = 6, W_COEF = 7, W_EBASE = 8, W_EOFF = 9, W_F = 12 };

struct TNRunPlan {
  int n_local, n_outer, n_ops, coef;
  unsigned char in_bit[kTileMax];    // address bit of slot i in the input
  unsigned char out_slot[kTileMax];  // slot of the i-th lowest of the tile's result bits
  unsigned char out_bit[kTileMax];   // its address bit
  unsigned char outer_in[kOuterMax], outer_out[kOuterMax];
};

struct TNRunBases {
  const float2* p[3];
  int64_t stride[3];
};

// LDS word of tile element a.  Rows of an op on low slots step over two or
// three address bits; folding bits 5..9 onto 0..4 keeps 32 adjacent rows on
// different banks for every choice of slots.  Linear in the bits of a, so
// offsets combine by XOR.
__device__ __forceinline__ uint32_t sw(uint32_t a) { return a ^ ((a >> 5) & 31u); }

__device__ __forceinline__ uint32_t insert0(uint32_t r, int p) {
  return ((r >> p) << (p + 1)) | (r & ((1u << p) - 1u));
}

// LDS byte of row r of an op of arity A: the tile element with the op's slots
// clear.  Linear (XOR) in the bits of r: the part of a thread's own bits is
// formed once per op, the rest is uniform and left to the scalar unit.
template <int A>
__device__ __forceinline__ uint32_t row_byte(uint32_t r, const int* s) {
  uint32_t a = insert0(insert0(r, s[0]), s[1]);
  if (A == 3) a = insert0(a, s[2]);
  return sw(a) << 3;
}

// LDS byte offset of element k of a row
template <int A>
__device__ __forceinline__ uint32_t slot_byte(uint32_t k, const int* s) {
  uint32_t a = 0;
#pragma unroll
  for (int j = 0; j < A; ++j) a |= ((k >> j) & 1u) << s[j];
  return sw(a) << 3;
}

__device__ __forceinline__ float2& at(float2* base, uint32_t byte) {
  return *reinterpret_cast<float2*>(reinterpret_cast<char*>(base) + byte);
}

__device__ __forceinline__ f32x4 mm(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_4x4x1f32(a, b, c, 0, 0, 0);
}

// y = M x over the rows of the tile; m: 2^A x 2^A, [out][in]
template <int A>
__device__ __forceinline__ void apply_op(float2* tile, const float2* m, const int* s, int n_local, int threads) {
  constexpr int D = 1 << A, Q = D / 4;
  const int t = threadIdx.x, rows = 1 << (n_local - A);
  if (t >= rows) return;  // whole waves
  float ar[Q][D], ai[Q][D], an[Q][D];
#pragma unroll
  for (int q = 0; q < Q; ++q)
#pragma unroll
    for (int k = 0; k < D; ++k) {
      const float2 v = m[(4 * q + (t & 3)) * D + k];
      ar[q][k] = v.x;
      ai[q][k] = v.y;
      an[q][k] = -v.y;
    }
  const uint32_t w0 = row_byte<A>(t, s);
#pragma unroll 2
  for (int r = 0; r < rows; r += threads) {
    const uint32_t w = w0 ^ row_byte<A>(r, s);
    float2 x[D];
#pragma unroll
    for (int k = 0; k < D; ++k) x[k] = at(tile, w ^ slot_byte<A>(k, s));
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      f32x4 re = {0.f, 0.f, 0.f, 0.f}, im = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < D; ++k) {
        re = mm(an[q][k], x[k].y, re);
        im = mm(ai[q][k], x[k].x, im);
        re = mm(ar[q][k], x[k].x, re);
        im = mm(ar[q][k], x[k].y, im);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) at(tile, w ^ slot_byte<A>(4 * q + i, s)) = make_float2(re[i], im[i]);
    }
  }
}

__device__ __forceinline__ uint32_t outer_offset(uint32_t g, int n, const unsigned char* bit) {
  uint32_t o = 0;
  for (int i = 0; i < n; ++i) o |= ((g >> i) & 1u) << bit[i];
  return o;
}

// Matrix entry e = out << arity | in of op w: the product of the factors'
// entries summed over the internal indices, zero where an index that goes
// straight through differs between out and in.
__device__ __forceinline__ double2 op_entry(const TNRunBases& bases, const int32_t* __restrict__ w, int64_t b, int e) {
  const int a = w[W_ARITY];
  const uint32_t in = e & ((1 << a) - 1), out = e >> a;
  double2 sum = make_double2(0.0, 0.0);
  if (((in ^ out) & (uint32_t)w[W_DELTA]) == 0) {
    for (uint32_t z = 0; z < (1u << w[W_INTERNAL]); ++z) {
      const uint32_t vars = in | (out << 3) | (z << 6);
      double2 p = make_double2(1.0, 0.0);
      for (int f = 0; f < w[W_FACTORS]; ++f) {
        const int32_t* v = w + W_F + 10 * f;
        uint32_t off = 0;
        for (int i = 0; i < v[2]; ++i) off |= ((vars >> v[3 + i]) & 1u) << i;
        const float2 g = bases.p[v[0]][b * bases.stride[v[0]] + v[1] + off];
        p = make_double2(p.x * g.x - p.y * g.y, p.x * g.y + p.y * g.x);
      }
      sum.x += p.x;
      sum.y += p.y;
    }
  }
  return sum;
}

__device__ __forceinline__ double wave_total(double v) {
#pragma unroll
  for (int h = 32; h > 0; h >>= 1) v += __shfl_xor(v, h, 64);
  return v;
}

}  // namespace

// The matrices of the ops.  A product of several factors is rounded to fp32
// once more than its factors applied one after another would be, and the part
// of that rounding that scales the whole matrix is the same for every row: over
// hundreds of ops it adds up in the result.  Where dev is given, dev[op] holds it
// (|M|, relative to the unrounded product), for k_tn_run_balance.
__global__ void __launch_bounds__(64) k_tn_run_coefs(TNRunBases bases, const int32_t* __restrict__ ops,
                                                     float2* __restrict__ coef, int64_t coef_bs,
                                                     float2* __restrict__ dev) {
  const int32_t* w = ops + (int64_t)blockIdx.x * kOpWords;
  const int e = threadIdx.x, size = 1 << (2 * w[W_ARITY]);
  const int64_t b = blockIdx.y;
  double exact = 0.0, stored = 0.0;
  if (e < size) {
    const double2 p = op_entry(bases, w, b, e);
    const float2 m = make_float2((float)p.x, (float)p.y);
    coef[b * coef_bs + w[W_COEF] + e] = m;
    exact = p.x * p.x + p.y * p.y;
    stored = (double)m.x * m.x + (double)m.y * m.y;
  }
  if (dev == nullptr) return;
  exact = wave_total(exact);
  stored = wave_total(stored);
  const double d = 0.5 * (stored / exact - 1.0);
  // (no finite product has more than its rounding: a zero or an overflowed one is left out)
  if (e == 0) dev[b * coef_bs + blockIdx.x] = make_float2(fabs(d) < 1e-6 ? (float)d : 0.f, 0.f);
}

// Divides the scale of all the roundings out of one op's matrix (a scale
// commutes with everything, so it does not matter which), whose own rounding
// is what remains.  Values of 20-qubit lattices with 280 ops: 1.10 times the
// error of the steps without it, 1.02 with it (960 rows).
__global__ void __launch_bounds__(256) k_tn_run_balance(TNRunBases bases, const int32_t* __restrict__ ops, int n_ops,
                                                        int op, float2* __restrict__ coef, int64_t coef_bs,
                                                        const float2* __restrict__ dev) {
  __shared__ double part[4];
  const int32_t* w = ops + (int64_t)op * kOpWords;
  const int t = threadIdx.x;
  const int64_t b = blockIdx.x;
  double d = 0.0;
  for (int o = t; o < n_ops; o += 256)
    if (o != op) d += dev[b * coef_bs + o].x;
  d = wave_total(d);
  if ((t & 63) == 0) part[t >> 6] = d;
  __syncthreads();
  if (t >= (1 << (2 * w[W_ARITY]))) return;
  const double f = 1.0 - (part[0] + part[1] + part[2] + part[3]);
  const double2 p = op_entry(bases, w, b, t);
  coef[b * coef_bs + w[W_COEF] + t] = make_float2((float)(f * p.x), (float)(f * p.y));
}

// One forward pass: workgroup (g, b) owns tile g of batch element b.
// 256 threads, 32 KB of LDS at 2^12 elements and 8 B per matrix entry: four
// workgroups per CU, whose loads, matrices and stores overlap.  Measured on
// 2^25 elements: 128 us a pass with one matrix (a copy takes 102), 188 with 8,
// 304 with 16, 534 with 32, against 92 us per matrix step by step.
template <bool A3>
__global__ void __launch_bounds__(256) k_tn_run_pass(const float2* __restrict__ X, int64_t x_bs,
                                                     float2* __restrict__ C, int64_t c_bs,
                                                     const float2* __restrict__ coef, int64_t coef_bs,
                                                     const int32_t* __restrict__ ops, TNRunPlan P) {
  extern __shared__ float2 lds[];
  const int t = threadIdx.x, N = 1 << P.n_local;
  float2* tile = lds;
  float2* m = lds + N;
  const int64_t b = blockIdx.y;
  const int coef0 = ops[W_COEF];
  {
    uint32_t lo = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) lo |= ((t >> i) & 1u) << P.in_bit[i];
    const float2* x = X + b * x_bs + (lo | outer_offset(blockIdx.x, P.n_outer, P.outer_in));
    float2 v[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      uint32_t hi = 0;
#pragma unroll
      for (int i = 0; i < 4; ++i) hi |= ((j >> i) & 1u) << P.in_bit[8 + i];
      if (j * 256 < N) v[j] = x[hi];
    }
    for (int e = t; e < P.coef; e += 256) m[e] = coef[b * coef_bs + coef0 + e];
#pragma unroll
    for (int j = 0; j < 16; ++j)
      if (j * 256 < N) tile[sw(j * 256 + t)] = v[j];
  }
  __syncthreads();
  for (int o = 0; o < P.n_ops; ++o) {
    const int32_t* w = ops + o * kOpWords;
    const int s[3] = {w[W_SLOT], w[W_SLOT + 1], w[W_SLOT + 2]};
    const float2* mo = m + (w[W_COEF] - coef0);
    if (A3 && w[W_ARITY] == 3)
      apply_op<3>(tile, mo, s, P.n_local, 256);
    else
      apply_op<2>(tile, mo, s, P.n_local, 256);
    __syncthreads();
  }
  uint32_t lo = 0, ls = 0;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    lo |= ((t >> i) & 1u) << P.out_bit[i];
    ls |= ((t >> i) & 1u) << P.out_slot[i];
  }
  float2* c = C + b * c_bs + (lo | outer_offset(blockIdx.x, P.n_outer, P.outer_out));
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    uint32_t hi = 0, hs = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      hi |= ((j >> i) & 1u) << P.out_bit[8 + i];
      hs |= ((j >> i) & 1u) << P.out_slot[8 + i];
    }
    if (j * 256 < N) c[hi] = tile[sw(hs | ls)];
  }
}

namespace {

// Sum of v over the 16 blocks of a 4x4x1 result (lanes with equal lane & 3),
// scattered: lane holds component lane >> 5 (re, im) of row (lane >> 3) & 3,
// column lane & 3.
__device__ __forceinline__ float block_sum(const f32x4& re, const f32x4& im, int lane) {
  const bool h5 = lane & 32, h4 = lane & 16, h3 = lane & 8;
  float k[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float send = h5 ? re[i] : im[i];
    k[i] = (h5 ? im[i] : re[i]) + __shfl_xor(send, 32, 64);
  }
  float l[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const float send = h4 ? k[i] : k[i + 2];
    l[i] = (h4 ? k[i + 2] : k[i]) + __shfl_xor(send, 16, 64);
  }
  const float send = h3 ? l[0] : l[1];
  float s = (h3 ? l[1] : l[0]) + __shfl_xor(send, 8, 64);
  s += __shfl_xor(s, 4, 64);
  return s;
}

// Backward of one op on the tile: x <- M^H x (the op's input, M unitary),
// red <- sum over rows of E[out] x[in] (per wave), E <- M^T E.
// The rows of a wave are its own until the next barrier, so the second,
// transposed read (lane 4 b + i: element i of row b, as the matrix cores take
// an outer product) needs no barrier: LDS serves one wave in order.
template <int A>
__device__ __forceinline__ void undo_op(float2* xt, float2* et, const float2* m, const int* s, int n_local, float* red) {
  constexpr int D = 1 << A, Q = D / 4;
  const int t = threadIdx.x, lane = t & 63, i4 = lane & 3;
  const int rows = 1 << (n_local - A);
  if (t >= rows) return;  // whole waves
  const uint32_t w0 = row_byte<A>(t, s);
  const uint32_t wt0 = row_byte<A>((t & ~63) | (lane >> 2), s) ^ slot_byte<A>(i4, s);
  f32x4 gr[Q][Q], gn[Q][Q], gi[Q][Q];
#pragma unroll
  for (int q = 0; q < Q; ++q)
#pragma unroll
    for (int k = 0; k < Q; ++k) gr[q][k] = gn[q][k] = gi[q][k] = f32x4{0.f, 0.f, 0.f, 0.f};
  // arity 2 keeps its column of the matrix in registers, arity 3 reads it again
  float mr[A == 2 ? D : 1], mi[A == 2 ? D : 1], mn[A == 2 ? D : 1];
  if (A == 2)
#pragma unroll
    for (int k = 0; k < D; ++k) {
      const float2 v = m[k * D + i4];
      mr[A == 2 ? k : 0] = v.x;
      mi[A == 2 ? k : 0] = v.y;
      mn[A == 2 ? k : 0] = -v.y;
    }
  for (int r = 0; r < rows; r += kBwdThreads) {
    const uint32_t wr = row_byte<A>(r, s), w = w0 ^ wr;
    float2 x[D], e[D];
#pragma unroll
    for (int k = 0; k < D; ++k) {
      x[k] = at(xt, w ^ slot_byte<A>(k, s));
      e[k] = at(et, w ^ slot_byte<A>(k, s));
    }
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      f32x4 re = {0.f, 0.f, 0.f, 0.f}, im = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < D; ++k) {
        const float2 v = A == 2 ? make_float2(mr[A == 2 ? k : 0], mi[A == 2 ? k : 0]) : m[k * D + 4 * q + i4];
        const float vn = A == 2 ? mn[A == 2 ? k : 0] : -v.y;
        re = mm(v.y, x[k].y, re);
        im = mm(vn, x[k].x, im);
        re = mm(v.x, x[k].x, re);
        im = mm(v.x, x[k].y, im);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) at(xt, w ^ slot_byte<A>(4 * q + i, s)) = make_float2(re[i], im[i]);
    }
    __builtin_amdgcn_wave_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const uint32_t wt = wt0 ^ (wr ^ row_byte<A>(16 * u, s));
      float2 xv[Q], ev[Q];
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        xv[q] = at(xt, wt ^ slot_byte<A>(4 * q, s));
        ev[q] = at(et, wt ^ slot_byte<A>(4 * q, s));
      }
#pragma unroll
      for (int q = 0; q < Q; ++q)
#pragma unroll
        for (int k = 0; k < Q; ++k) {
          gr[q][k] = mm(ev[q].x, xv[k].x, gr[q][k]);
          gi[q][k] = mm(ev[q].x, xv[k].y, gi[q][k]);
          gn[q][k] = mm(ev[q].y, xv[k].y, gn[q][k]);
          gi[q][k] = mm(ev[q].y, xv[k].x, gi[q][k]);
        }
    }
    __builtin_amdgcn_wave_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      f32x4 re = {0.f, 0.f, 0.f, 0.f}, im = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < D; ++k) {
        const float2 v = A == 2 ? make_float2(mr[A == 2 ? k : 0], mi[A == 2 ? k : 0]) : m[k * D + 4 * q + i4];
        const float vn = A == 2 ? mn[A == 2 ? k : 0] : -v.y;
        re = mm(vn, e[k].y, re);
        im = mm(v.y, e[k].x, im);
        re = mm(v.x, e[k].x, re);
        im = mm(v.x, e[k].y, im);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) at(et, w ^ slot_byte<A>(4 * q + i, s)) = make_float2(re[i], im[i]);
    }
  }
  float* rw = red + (t >> 6) * (2 * D * D);
#pragma unroll
  for (int q = 0; q < Q; ++q)
#pragma unroll
    for (int k = 0; k < Q; ++k) {
      const float v = block_sum(gr[q][k] - gn[q][k], gi[q][k], lane);
      const int row = 4 * q + ((lane >> 3) & 3), col = 4 * k + i4;
      if ((lane & 4) == 0) rw[2 * (row * D + col) + (lane >> 5)] = v;
    }
}

}  // namespace

// One backward pass.  Workgroups walk over the tiles (grid.x of them per
// batch element) and keep the matrices' environments in LDS, so that the
// partial sums written are per workgroup, not per tile.  EX may be EC when the
// pass keeps the layout: a tile is read whole before it is written.
// 512 threads, two tiles of 32 KB: two workgroups, 16 waves per CU.  Measured
// on 2^25 elements, with k_tn_run_env: 212 us a pass with one matrix, 572 with
// 8, 1019 with 16, 1888 with 32, against 152 us per matrix step by step.
template <bool A3>
__global__ void __launch_bounds__(kBwdThreads) k_tn_run_bwd(const float2* __restrict__ C, int64_t c_bs,
                                                            const float2* EC, int64_t ec_bs, float2* EX,
                                                            int64_t ex_bs, const float2* __restrict__ coef,
                                                            int64_t coef_bs, const int32_t* __restrict__ ops,
                                                            float* __restrict__ part, TNRunPlan P) {
  extern __shared__ float2 lds[];
  constexpr int kPer = 1 << (kTileMax - kBwdLog);
  constexpr int kRed = (kBwdThreads / 64) * (A3 ? 128 : 32);
  const int t = threadIdx.x, N = 1 << P.n_local;
  float2* xt = lds;
  float2* et = lds + (1 << kTileMax);  // a constant distance: one address serves both
  float2* m = lds + (2 << kTileMax);
  float* acc = reinterpret_cast<float*>(m + P.coef);
  float* red = acc + 2 * P.coef;
  const int64_t b = blockIdx.y;
  const int coef0 = ops[W_COEF];
  for (int e = t; e < P.coef; e += kBwdThreads) m[e] = coef[b * coef_bs + coef0 + e];
  for (int e = t; e < 2 * P.coef; e += kBwdThreads) acc[e] = 0.f;
  uint32_t lo_in = 0, lo_out = 0, ls = 0;
#pragma unroll
  for (int i = 0; i < kBwdLog; ++i) {
    lo_in |= ((t >> i) & 1u) << P.in_bit[i];
    lo_out |= ((t >> i) & 1u) << P.out_bit[i];
    ls |= ((t >> i) & 1u) << P.out_slot[i];
  }
  const uint32_t tiles = 1u << P.n_outer;
  for (uint32_t g = blockIdx.x; g < tiles; g += gridDim.x) {
    const uint32_t oo = lo_out | outer_offset(g, P.n_outer, P.outer_out);
    const float2* c = C + b * c_bs + oo;
    const float2* ec = EC + b * ec_bs + oo;
    float2 vx[kPer], ve[kPer];
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      uint32_t hi = 0;
#pragma unroll
      for (int i = 0; i < kTileMax - kBwdLog; ++i) hi |= ((j >> i) & 1u) << P.out_bit[kBwdLog + i];
      if (j * kBwdThreads < N) {
        vx[j] = c[hi];
        ve[j] = ec[hi];
      }
    }
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      uint32_t hs = 0;
#pragma unroll
      for (int i = 0; i < kTileMax - kBwdLog; ++i) hs |= ((j >> i) & 1u) << P.out_slot[kBwdLog + i];
      if (j * kBwdThreads < N) {
        xt[sw(hs | ls)] = vx[j];
        et[sw(hs | ls)] = ve[j];
      }
    }
    __syncthreads();
    for (int o = P.n_ops - 1; o >= 0; --o) {
      const int32_t* w = ops + o * kOpWords;
      const int s[3] = {w[W_SLOT], w[W_SLOT + 1], w[W_SLOT + 2]};
      const int off = w[W_COEF] - coef0, a = w[W_ARITY];
      // two buffers: the sums below read this op's while the next op fills the other
      float* rd = red + (o & 1) * kRed;
      if (A3 && a == 3)
        undo_op<3>(xt, et, m + off, s, P.n_local, rd);
      else
        undo_op<2>(xt, et, m + off, s, P.n_local, rd);
      __syncthreads();
      const int size = 2 << (2 * a);
      if (t < size) {
        const int waves = min(kBwdThreads / 64, (1 << (P.n_local - a)) / 64);
        float v = 0.f;
        for (int q = 0; q < waves; ++q) v += rd[q * size + t];
        acc[2 * off + t] += v;
      }
    }
    float2* ex = EX + b * ex_bs + (lo_in | outer_offset(g, P.n_outer, P.outer_in));
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      uint32_t hi = 0;
#pragma unroll
      for (int i = 0; i < kTileMax - kBwdLog; ++i) hi |= ((j >> i) & 1u) << P.in_bit[kBwdLog + i];
      if (j * kBwdThreads < N) ex[hi] = et[sw(j * kBwdThreads + t)];
    }
    __syncthreads();
  }
  float* p = part + (b * gridDim.x + blockIdx.x) * (int64_t)(2 * P.coef);
  for (int e = t; e < 2 * P.coef; e += kBwdThreads) p[e] = acc[e];
}

// Environment of an op's gate: the workgroups' sums of its matrix entries,
// written to the gate tensor's own address order (an op on one address bit
// carries a spectator bit, which is summed here).
// 1024 threads: the workgroups' rows are 128 B apart reads of one matrix, a
// chain of loads per thread (39 us per pass with 256 threads and no unrolling).
// A rotation rounded to fp32 is a unitary matrix times 1 + O(1e-7): M^H M = s,
// the same for every row, so undoing the ops o, o + 1, ... of the pass left
// their inputs scaled by the product of their s, which no sum averages out.  It
// is divided out here in fp64 (16 qubits, 6 layers of a lattice: 1.11 times the
// error of stored inputs without it).
__global__ void __launch_bounds__(1024) k_tn_run_env(const float* __restrict__ part, int n_wg, int coef,
                                                     const int32_t* __restrict__ ops, int n_ops,
                                                     const float2* __restrict__ m, int64_t m_bs, float2* env0,
                                                     int64_t bs0, float2* env1, int64_t bs1) {
  __shared__ double sum[1024], scale[16];
  __shared__ float2 val[64];
  const int32_t* w = ops + (int64_t)blockIdx.x * kOpWords;
  if (w[W_EBASE] < 0) return;
  const int64_t b = blockIdx.y;
  const int t = threadIdx.x, a = w[W_ARITY], size = 2 << (2 * a), off = 2 * (w[W_COEF] - ops[W_COEF]);
  // sum of s - 1 = tr(M^H M) / D - 1 over the ops, a wave per op (first order: the squares are below 1e-11)
  double dev = 0.0;
  for (int o = blockIdx.x + (t >> 6); o < n_ops; o += 16) {
    const int32_t* wo = ops + o * kOpWords;
    const int ao = wo[W_ARITY], e = t & 63;
    if (e < (1 << (2 * ao))) {
      const float2 v = m[b * m_bs + wo[W_COEF] + e];
      dev += ((double)v.x * v.x + (double)v.y * v.y) / (1 << ao);
    }
    if (e == 0) dev -= 1.0;
  }
  dev = wave_total(dev);
  if ((t & 63) == 0) scale[t >> 6] = dev;
  const int step = 1024 / size;
  const float* p = part + b * n_wg * (int64_t)(2 * coef) + off + (t & (size - 1));
  double s = 0.0;
#pragma unroll 8
  for (int g = t / size; g < n_wg; g += step) s += p[g * (int64_t)(2 * coef)];
  sum[t] = s;
  __syncthreads();
  if (t < size) {
    for (int q = 1; q < step; ++q) s += sum[q * size + t];
    double d = 0.0;
    for (int q = 0; q < 16; ++q) d += scale[q];
    reinterpret_cast<float*>(val)[t] = (float)(s - d * s);
  }
  __syncthreads();
  const int32_t* f = w + W_F;
  const int nb = f[2];
  if (t >= (1 << nb)) return;
  uint32_t vars = 0;
  for (int i = 0; i < nb; ++i) vars |= ((t >> i) & 1u) << f[3 + i];
  const uint32_t spect = (uint32_t)w[W_DELTA];
  float2 r = make_float2(0.f, 0.f);
  for (uint32_t z = 0; z < (1u << a); ++z) {
    if (z & ~spect) continue;
    const uint32_t in = (vars & 7u) | z, out = ((vars >> 3) & 7u) | z;
    r.x += val[(out << a) | in].x;
    r.y += val[(out << a) | in].y;
  }
  float2* e = w[W_EBASE] == 0 ? env0 + b * bs0 : env1 + b * bs1;
  e[w[W_EOFF] + t] = r;
}

namespace {

bool parse_run_plan(const int32_t* words, TNRunPlan* P) {
  P->n_local = words[0];
  P->n_outer = words[1];
  P->n_ops = words[2];
  P->coef = words[3];
  if (P->n_local < kTileMin || P->n_local > kTileMax || P->n_outer < 0 || P->n_outer > kOuterMax || P->n_ops < 1 ||
      P->n_ops > kRunOps || P->coef < 16 || P->coef > kRunCoef)
    return false;
  const int n = P->n_local + P->n_outer;
  if (n > 30) return false;
  uint32_t in = 0, out = 0, slots = 0;
  auto take = [n](int32_t bit, int lim, uint32_t* seen) {
    if (bit < 0 || bit >= lim || (*seen >> bit) & 1u) return false;
    *seen |= 1u << bit;
    return true;
  };
  for (int i = 0; i < kTileMax; ++i) {
    P->in_bit[i] = P->out_slot[i] = P->out_bit[i] = 0;
    if (i >= P->n_local) continue;
    if (!take(words[4 + i], n, &in) || !take(words[16 + i], P->n_local, &slots) || !take(words[28 + i], n, &out))
      return false;
    P->in_bit[i] = (unsigned char)words[4 + i];
    P->out_slot[i] = (unsigned char)words[16 + i];
    P->out_bit[i] = (unsigned char)words[28 + i];
  }
  for (int i = 0; i < P->n_outer; ++i) {
    if (!take(words[40 + i], n, &in) || !take(words[72 + i], n, &out)) return false;
    P->outer_in[i] = (unsigned char)words[40 + i];
    P->outer_out[i] = (unsigned char)words[72 + i];
  }
  return true;
}

// ops of a pass: slots inside the tile, coefficients packed in order
bool check_pass_ops(const int32_t* ops, const TNRunPlan& P, bool* a3) {
  *a3 = false;
  int64_t at = ops[W_COEF];
  if (at < 0) return false;
  for (int o = 0; o < P.n_ops; ++o) {
    const int32_t* w = ops + (int64_t)o * kOpWords;
    const int a = w[W_ARITY];
    if ((a != 2 && a != 3) || w[W_COEF] != at) return false;
    at += 1 << (2 * a);
    for (int j = 0; j < a; ++j)
      if (w[W_SLOT + j] < 0 || w[W_SLOT + j] >= P.n_local || (j > 0 && w[W_SLOT + j] <= w[W_SLOT + j - 1])) return false;
    *a3 = *a3 || a == 3;
  }
  return at - ops[W_COEF] == P.coef;
}

int run_groups(const TNRunPlan& P, int64_t batch) {
  const int64_t tiles = 1ll << P.n_outer;
  // about two rounds of the resident workgroups (two per CU)
  const int64_t want = (1024 + batch - 1) / batch;
  return (int)(tiles < want ? tiles : want);
}

}  // namespace

}  // namespace tedq

using namespace tedq;

// The matrices of n_ops ops for every batch element: coef [batch][coef_bs].
// bases / strides / lens: the three arenas the factors are read from (gate
// leaves, constants, small results); ops / ops_dev: 52 int32 words per op,
// host and device copies.  All offsets are checked on the host.  Where a row of
// coef has room for n_ops more entries after the matrices, the scale of the
// roundings of several factors' products is balanced (k_tn_run_balance).
extern "C" int tedq_tn_run_coefs(const void* const* bases, const int64_t* strides, const int64_t* lens,
                                 const int32_t* ops, const int32_t* ops_dev, int n_ops, void* coef, int64_t coef_bs,
                                 int64_t batch, void* stream) {
  if (bases == nullptr || strides == nullptr || lens == nullptr || ops == nullptr || ops_dev == nullptr ||
      coef == nullptr || n_ops <= 0 || batch <= 0 || batch > 65535) {
    set_error("tedq_tn_run_coefs: bad arguments");
    return kBadArgument;
  }
  TNRunBases tb;
  for (int i = 0; i < 3; ++i) {
    if (bases[i] == nullptr || strides[i] < 0 || lens[i] < 0) {
      set_error("tedq_tn_run_coefs: bad arena %d", i);
      return kBadArgument;
    }
    tb.p[i] = static_cast<const float2*>(bases[i]);
    tb.stride[i] = strides[i];
  }
  int product = -1;
  int64_t entries = 0;
  for (int o = 0; o < n_ops; ++o) {
    const int32_t* w = ops + (int64_t)o * kOpWords;
    const int a = w[W_ARITY];
    bool ok = (a == 2 || a == 3) && w[W_DELTA] >= 0 && w[W_DELTA] < (1 << a) && w[W_INTERNAL] >= 0 &&
              w[W_INTERNAL] <= 3 && w[W_FACTORS] >= 1 && w[W_FACTORS] <= kFactors && w[W_COEF] >= 0 &&
              w[W_COEF] + (1ll << (2 * a)) <= coef_bs;
    for (int f = 0; ok && f < w[W_FACTORS]; ++f) {
      const int32_t* v = w + W_F + 10 * f;
      ok = v[0] >= 0 && v[0] < 3 && v[1] >= 0 && v[2] >= 0 && v[2] <= 6 && v[1] + (1ll << v[2]) <= lens[v[0]];
      for (int i = 0; ok && i < v[2]; ++i) ok = v[3 + i] >= 0 && v[3 + i] < 9;
    }
    if (!ok) {
      set_error("tedq_tn_run_coefs: op %d does not fit (shape or arena bounds)", o);
      return kBadArgument;
    }
    if (w[W_FACTORS] > 1) product = o;
    const int64_t end = w[W_COEF] + (1ll << (2 * a));
    if (end > entries) entries = end;
  }
  float2* c = static_cast<float2*>(coef);
  const bool balance = product >= 0 && coef_bs - entries >= n_ops;
  float2* dev = balance ? c + entries : nullptr;
  hipStream_t st = static_cast<hipStream_t>(stream);
  hipLaunchKernelGGL(k_tn_run_coefs, dim3((unsigned)n_ops, (unsigned)batch), dim3(64), 0, st, tb, ops_dev, c, coef_bs,
                     dev);
  const int rc = check_launch("tedq_tn_run_coefs");
  if (rc != kOk || !balance) return rc;
  hipLaunchKernelGGL(k_tn_run_balance, dim3((unsigned)batch), dim3(256), 0, st, tb, ops_dev, n_ops, product, c, coef_bs,
                     dev);
  return check_launch("tedq_tn_run_coefs(balance)");
}

// One forward pass: plan = 128 int32 words (tile, slots and address bits),
// ops / ops_dev = the pass's ops.  x and c hold 2^(n_local + n_outer) elements
// per batch element and must not overlap.
extern "C" int tedq_tn_run_pass(const void* x, int64_t x_bs, void* c, int64_t c_bs, int64_t batch,
                                const int32_t* plan, const int32_t* ops, const int32_t* ops_dev, const void* coef,
                                int64_t coef_bs, void* stream) {
  TNRunPlan P;
  bool a3;
  if (x == nullptr || c == nullptr || x == c || plan == nullptr || ops == nullptr || ops_dev == nullptr ||
      coef == nullptr || batch <= 0 || batch > 65535 || !parse_run_plan(plan, &P) || !check_pass_ops(ops, P, &a3) ||
      ops[W_COEF] + (int64_t)P.coef > coef_bs) {
    set_error("tedq_tn_run_pass: bad arguments or plan");
    return kBadArgument;
  }
  const dim3 grid(1u << P.n_outer, (unsigned)batch);
  const size_t lds = sizeof(float2) * ((size_t)(1 << P.n_local) + P.coef);
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (a3)
    hipLaunchKernelGGL(k_tn_run_pass<true>, grid, dim3(256), lds, st, static_cast<const float2*>(x), x_bs,
                       static_cast<float2*>(c), c_bs, static_cast<const float2*>(coef), coef_bs, ops_dev, P);
  else
    hipLaunchKernelGGL(k_tn_run_pass<false>, grid, dim3(256), lds, st, static_cast<const float2*>(x), x_bs,
                       static_cast<float2*>(c), c_bs, static_cast<const float2*>(coef), coef_bs, ops_dev, P);
  return check_launch("tedq_tn_run_pass");
}

// Workspace bytes of tedq_tn_run_backward, or -1 for an invalid plan.
extern "C" int64_t tedq_tn_run_backward_workspace(const int32_t* plan, int64_t batch) {
  TNRunPlan P;
  if (plan == nullptr || batch <= 0 || !parse_run_plan(plan, &P)) return -1;
  return batch * run_groups(P, batch) * 2 * (int64_t)P.coef * (int64_t)sizeof(float);
}

// One backward pass: c = the pass's result, ec = its environment; ex receives
// the environment of the pass's input (it may be ec when the pass keeps the
// layout).  Gate environments go to env0 / env1 (batch strides, elements valid
// per batch row) at the ops' words 8 and 9 (base, offset; base -1: none).
extern "C" int tedq_tn_run_backward(const void* c, int64_t c_bs, const void* ec, int64_t ec_bs, void* ex,
                                    int64_t ex_bs, int64_t batch, const int32_t* plan, const int32_t* ops,
                                    const int32_t* ops_dev, const void* coef, int64_t coef_bs, void* env0,
                                    int64_t bs0, int64_t len0, void* env1, int64_t bs1, int64_t len1,
                                    void* workspace, int64_t workspace_bytes, void* stream) {
  TNRunPlan P;
  bool a3;
  if (c == nullptr || ec == nullptr || ex == nullptr || c == ex || plan == nullptr || ops == nullptr ||
      ops_dev == nullptr || coef == nullptr || env0 == nullptr || env1 == nullptr || batch <= 0 || batch > 65535 ||
      !parse_run_plan(plan, &P) || !check_pass_ops(ops, P, &a3) || ops[W_COEF] + (int64_t)P.coef > coef_bs) {
    set_error("tedq_tn_run_backward: bad arguments or plan");
    return kBadArgument;
  }
  bool same = true;
  for (int i = 0; i < P.n_local; ++i) same = same && P.out_slot[i] == i && P.out_bit[i] == P.in_bit[i];
  for (int i = 0; i < P.n_outer; ++i) same = same && P.outer_in[i] == P.outer_out[i];
  if (ec == ex && !same) {
    set_error("tedq_tn_run_backward: a pass that changes the layout cannot run in place");
    return kBadArgument;
  }
  for (int o = 0; o < P.n_ops; ++o) {
    const int32_t* w = ops + (int64_t)o * kOpWords;
    if (w[W_EBASE] < 0) continue;
    const int32_t* f = w + W_F;
    bool ok = w[W_EBASE] <= 1 && w[W_FACTORS] == 1 && w[W_INTERNAL] == 0 && f[2] >= 0 && f[2] <= 6 && w[W_EOFF] >= 0 &&
              w[W_EOFF] + (1ll << f[2]) <= (w[W_EBASE] == 0 ? len0 : len1);
    for (int i = 0; ok && i < f[2]; ++i) ok = f[3 + i] >= 0 && f[3 + i] < 6 && f[3 + i] % 3 < w[W_ARITY];
    if (!ok) {
      set_error("tedq_tn_run_backward: op %d has no single-gate environment in bounds", o);
      return kBadArgument;
    }
  }
  const int groups = run_groups(P, batch);
  const int64_t need = batch * groups * 2 * (int64_t)P.coef * (int64_t)sizeof(float);
  if (workspace == nullptr || workspace_bytes < need) {
    set_error("tedq_tn_run_backward: workspace of %lld bytes required, %lld given", (long long)need,
              (long long)workspace_bytes);
    return kBadArgument;
  }
  const size_t lds = sizeof(float2) * ((size_t)(2 << kTileMax) + P.coef) + sizeof(float) * 2 * P.coef +
                     sizeof(float) * 2 * (kBwdThreads / 64) * (a3 ? 128 : 32);
  hipStream_t st = static_cast<hipStream_t>(stream);
  const dim3 grid((unsigned)groups, (unsigned)batch);
  const void* fn = a3 ? reinterpret_cast<const void*>(k_tn_run_bwd<true>) : reinterpret_cast<const void*>(k_tn_run_bwd<false>);
  const hipError_t he = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (he != hipSuccess) {
    set_error("tedq_tn_run_backward: %zu bytes of LDS: %s", lds, hipGetErrorString(he));
    return kBadArgument;
  }
  if (a3)
    hipLaunchKernelGGL(k_tn_run_bwd<true>, grid, dim3(kBwdThreads), lds, st, static_cast<const float2*>(c), c_bs,
                       static_cast<const float2*>(ec), ec_bs, static_cast<float2*>(ex), ex_bs,
                       static_cast<const float2*>(coef), coef_bs, ops_dev, static_cast<float*>(workspace), P);
  else
    hipLaunchKernelGGL(k_tn_run_bwd<false>, grid, dim3(kBwdThreads), lds, st, static_cast<const float2*>(c), c_bs,
                       static_cast<const float2*>(ec), ec_bs, static_cast<float2*>(ex), ex_bs,
                       static_cast<const float2*>(coef), coef_bs, ops_dev, static_cast<float*>(workspace), P);
  const int rc = check_launch("tedq_tn_run_backward");
  if (rc != kOk) return rc;
  hipLaunchKernelGGL(k_tn_run_env, dim3((unsigned)P.n_ops, (unsigned)batch), dim3(1024), 0, st,
                     static_cast<const float*>(workspace), groups, P.coef, ops_dev, P.n_ops,
                     static_cast<const float2*>(coef), coef_bs, static_cast<float2*>(env0), bs0,
                     static_cast<float2*>(env1), bs1);
  return check_launch("tedq_tn_run_backward(env)");
}
