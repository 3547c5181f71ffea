// Backward of the packed chunk attention on the matrix cores (training: the
// gradient of one streaming block, litgpt/log_kv_cache.py:6867-7098, whose
// per-block autograd.grad this replaces; slot attention's gradient,
// litgpt/log_kv_cache.py:6501-6630).
//
// Forward: o_i = sum_j p_ij v_j, p_ij = softmax_j(scale * [q_i, 1/scale] . [k_j, bias_j])
// over the packed rows, the last causal_tail rows causal. With D_i = dO_i . o_i
// (= sum_j p_ij dO_i . v_j, formed in float32 here: the rounded forward output would lose the
// bits that cancel in dS) and dS_ij = p_ij (dO_i . v_j - D_i):
//   dq_i = scale * sum_j dS_ij k_j      (key features only; the bias coordinate has no gradient)
//   dk_j = scale * sum_i dS_ij q_i,  dv_j = sum_i p_ij dO_i
// for the last `grad_rows` packed rows (the in-flight chunk; every row for slot attention).
//
// All products are v_mfma_f32_32x32x16_bf16 with the forward's fragment layout. A wave's own
// 32 rows (queries for dq, keys for dk / dv) are the B operand and stay in registers for the
// whole walk; the other side streams through double-buffered LDS tiles of 64 rows, loaded into
// registers one tile ahead, one barrier per tile. Both operands of a streamed tile come from
// one row-major copy: as rows by 16-byte reads (S and dP), transposed by ds_read_b64_tr_b16
// (dQ^T += K^T dS^T, dK^T += Q^T dS, dV^T += dO^T P).
//  * stats_kernel: the online maximum, sum and sum of p dP of each query over one part of
//    its key range;
//  * dq_kernel: the parts combined to the log-sum-exp and D (also stored for dkv_kernel), then
//    S^T = K Q^T, dP^T = V dO^T, dS^T and dQ^T += K^T dS^T over one part of the key range;
//  * dkv_kernel: 128 gradient rows per block over one part of the query rows;
//  * sum_dq_kernel / sum_dkv_kernel: the parts' float32 partials added in part order.
// The ranges are split so that the launches fill the 256 CUs (bwd_splits). P and dS are the
// lanes' own accumulator registers (the k-index permutation of the forward's P^T operand), each
// as a high and a low bf16 part; accumulation is float32.
//
// Measured at 2 x 1024 query rows, 16 heads of 128 on 8 groups, 9.3K packed rows and a 1024-row
// chunk: dq 264 us and statistics 185 us (one 128-row block of four waves, tiles staged by element
// and re-read from LDS as both operands: 1880 us together), dk / dv 99 us with its rows loaded as
// 16-byte units (1224 us by element); dq and statistics bound by the matrix products and the
// exponentials, which the two waves of a SIMD run in step and so one after the other; dk / dv, one
// wave per SIMD, by the latency of that same chain (matrix cores 22% busy).
#include <algorithm>

#include "route.hpp"

namespace logkv {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef short s16x4 __attribute__((ext_vector_type(4)));

constexpr int kQWaves = 8;                // waves per query block (two per SIMD), 32 queries each
constexpr int kQRows = 32 * kQWaves;
constexpr int kKWaves = 4;                // waves per gradient-row block: dk and dv accumulators take one wave per SIMD
constexpr int kKRows = 32 * kKWaves;
constexpr int kTile = 64;                 // streamed rows per tile
constexpr int kLdK = 152;                 // row stride of packed-key / query tiles (bf16; 16-byte reads of 8 rows: 8 bank groups)
constexpr int kLdD = 136;                 // row stride of value / dO tiles (dv <= 128)
constexpr int kMaxSplits = 16;
constexpr float kLog2e = 1.44269504088896341f;

__device__ __forceinline__ bf16x8 load8(const uint16_t* p) { return *reinterpret_cast<const bf16x8*>(p); }

// Transposed A operand of a row-major tile: for feature f0 + lane % 32, rows 16 st + 8 (j / 4) +
// 4 (lane / 32) + j % 4 (the order of the accumulator registers' elements). ds_read_b64_tr_b16
// turns a 16-lane group's 4 rows x 16 features (lane i reads row i / 4, features 4 (i % 4) .. + 4)
// into 4 rows of feature i per lane.
template <int LD>
__device__ __forceinline__ bf16x8 load_tr(const uint16_t* tile, int f0, int st) {
  typedef __attribute__((address_space(3))) s16x4* lds4;
  const int l = lane_id(), i = l & 15, h = l >> 5;
  const uint16_t* p = tile + (16 * st + 4 * h + (i >> 2)) * LD + f0 + (l & 16) + 4 * (i & 3);
  const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)(p));
  const s16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)(p + 8 * LD));
  const uint2 x = __builtin_bit_cast(uint2, a), y = __builtin_bit_cast(uint2, b);
  return __builtin_bit_cast(bf16x8, make_uint4(x.x, x.y, y.x, y.y));
}

// B operand of step st from accumulator blocks acc[2] (elements 8 (st % 2) .. + 8 of block
// st / 2) as two bf16 parts: the truncated high half and the rounded remainder, so the two
// products keep about 16 significant bits (the softmax backward sums dS terms that cancel).
__device__ __forceinline__ void regs_b(const f32x16 (&acc)[2], int st, bf16x8& hi, bf16x8& lo) {
  uint32_t hw[4], lw[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float x0 = acc[st / 2][8 * (st % 2) + 2 * j], x1 = acc[st / 2][8 * (st % 2) + 2 * j + 1];
    const uint32_t u0 = __float_as_uint(x0), u1 = __float_as_uint(x1);
    hw[j] = __builtin_amdgcn_perm(u1, u0, 0x07060302u);
    const float r0 = x0 - __uint_as_float(u0 & 0xffff0000u), r1 = x1 - __uint_as_float(u1 & 0xffff0000u);
    lw[j] = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{r0, r1}, bf16x2));
  }
  hi = __builtin_bit_cast(bf16x8, make_uint4(hw[0], hw[1], hw[2], hw[3]));
  lo = __builtin_bit_cast(bf16x8, make_uint4(lw[0], lw[1], lw[2], lw[3]));
}

__device__ __forceinline__ int packed_total(const logkv_attention_args& a, const int32_t* width_ptr) {
  return min(*width_ptr + a.tail + (a.alpha_count_dev ? *a.alpha_count_dev : 0), a.cap);
}

// Features d .. d + 7 of a strided bf16 row (those past n zero): one 16-byte load where the rows
// are 16-byte aligned (`vec`; n is a multiple of 8), else by element.
__device__ __forceinline__ uint4 row_unit(const LOGKV_G uint16_t* row, int d, int n, bool vec) {
  if (d >= n) return make_uint4(0, 0, 0, 0);
  if (vec) return *(const LOGKV_G uint4*)(row + d);
  uint32_t x[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) x[j] = row[d + 2 * j] | (static_cast<uint32_t>(row[d + 2 * j + 1]) << 16);
  return make_uint4(x[0], x[1], x[2], x[3]);
}

// The query row [q, 1/scale, 0...], features d .. d + 7 (dk is a multiple of 8).
__device__ __forceinline__ uint4 query_unit(const logkv_attention_args& a, const LOGKV_G uint16_t* row, int d, bool vec) {
  if (d == a.dk) return make_uint4(f32_to_bf16(a.inv_scale_bf16), 0, 0, 0);
  return row_unit(row, d, a.dk, vec);
}

// Workgroups go to the 8 XCDs round robin: dispatched block n takes logical block (n % 8) (N / 8)
// + n / 8 (N a multiple of 8), so the blocks of a lane, which stream the same rows, share one L2.
struct BwdBlock {
  int x, split, lane;
};
__device__ __forceinline__ BwdBlock bwd_block() {
  const int nx = static_cast<int>(gridDim.x), ny = static_cast<int>(gridDim.y);
  const int n = nx * ny * static_cast<int>(gridDim.z);
  int lin = static_cast<int>(blockIdx.x) + nx * (static_cast<int>(blockIdx.y) + ny * static_cast<int>(blockIdx.z));
  if (n % 8 == 0) lin = (lin % 8) * (n / 8) + lin / 8;
  return BwdBlock{lin % nx, (lin / nx) % ny, lin / (nx * ny)};
}

struct BwdLayout {
  int q_splits;    // parts of the key range (stats_kernel, dq_kernel)
  int k_splits;    // parts of the query rows (dkv_kernel)
  int vec_q, vec_do, vec_dq;   // rows of q / dO 16-byte aligned, of dq 8-byte aligned
  float* stats;    // [lanes, nq, 2]: log-sum-exp, D
  float* part;     // [lanes, q_splits, nq, 4]: maximum, sum, sum of p dP
  float* grad;     // partials of dq [lanes, q_splits, nq, dk], then of dk / dv [lanes, k_splits, grad_rows, dk + dv]
};

// A block's streamed K / V tiles: rows t0 .. of the lane's packed rows, those past `stop` zero.
template <int NKS, int NDV, int THREADS>
struct KvTiles {
  static constexpr int kUnitsK = 2 * NKS, kUnitsV = 4 * NDV;
  static constexpr int kTasksK = (kTile * kUnitsK + THREADS - 1) / THREADS, kTasksV = (kTile * kUnitsV + THREADS - 1) / THREADS;
  uint4 kx[kTasksK], vx[kTasksV];
  __device__ __forceinline__ void load(const logkv_attention_args& a, const LOGKV_G uint16_t* kbase,
                                       const LOGKV_G uint16_t* vbase, int t0, int stop) {
#pragma unroll
    for (int q = 0; q < kTasksK; ++q) {
      const int i = threadIdx.x + THREADS * q, r = i / kUnitsK, u = i % kUnitsK;
      const bool on = r < kTile && t0 + r < stop && 8 * u < a.dim;
      kx[q] = *(const LOGKV_G uint4*)(kbase + static_cast<int64_t>(on ? t0 + r : t0) * a.dim + (on ? 8 * u : 0));
      if (!on) kx[q] = make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (int q = 0; q < kTasksV; ++q) {
      const int i = threadIdx.x + THREADS * q, r = i / kUnitsV, u = i % kUnitsV;
      const bool on = r < kTile && t0 + r < stop && 8 * u < a.dv;
      vx[q] = *(const LOGKV_G uint4*)(vbase + static_cast<int64_t>(on ? t0 + r : t0) * a.dim + (on ? 8 * u : 0));
      if (!on) vx[q] = make_uint4(0, 0, 0, 0);
    }
  }
  __device__ __forceinline__ void store(uint16_t* k_s, uint16_t* v_s) const {
#pragma unroll
    for (int q = 0; q < kTasksK; ++q) {
      const int i = threadIdx.x + THREADS * q, r = i / kUnitsK, u = i % kUnitsK;
      if (r < kTile) *reinterpret_cast<uint4*>(k_s + r * kLdK + 8 * u) = kx[q];
    }
#pragma unroll
    for (int q = 0; q < kTasksV; ++q) {
      const int i = threadIdx.x + THREADS * q, r = i / kUnitsV, u = i % kUnitsV;
      if (r < kTile) *reinterpret_cast<uint4*>(v_s + r * kLdD + 8 * u) = vx[q];
    }
  }
};

// One query block over one part of its key range: the own query and dO fragments, and a walk of
// the key tiles that hands f(s, dp, t0, k tile) the tile's masked scores S^T and dP^T.
template <int NKS, int NDV>
struct QueryWalk {
  int lane_ix, b, qi, head, t, total, tail0, k_begin, k_stop;
  bool q_ok;
  bf16x8 qf[NKS], df[2 * NDV];

  __device__ __forceinline__ QueryWalk(const logkv_attention_args& a, const int32_t* width_ptr,
                                       const logkv_attention_grad_args& gr, const BwdLayout& lay, const BwdBlock& id) {
    const int G = a.n_groups, rep = a.n_heads / G, nq = rep * a.tq;
    lane_ix = id.lane;
    b = lane_ix / G;
    const int w = wave_id(), l = lane_id(), h = l >> 5, col = l & 31;
    qi = id.x * kQRows + w * 32 + col;
    q_ok = qi < nq;
    const int qc = q_ok ? qi : nq - 1;
    head = (lane_ix % G) * rep + qc / a.tq;
    t = qc % a.tq;
    total = packed_total(a, width_ptr);
    tail0 = total - a.causal_tail;
    // Last key row any query of the block can see, and this block's part of the range in whole tiles.
    const int q_first = id.x * kQRows, q_last = min(q_first + kQRows, nq) - 1;
    const int t_max = q_first / a.tq == q_last / a.tq ? q_last % a.tq : a.tq - 1;
    const int key_end = a.causal_tail ? min(total, tail0 + t_max + 1) : total;
    const int tiles = (key_end + kTile - 1) / kTile, per = (tiles + lay.q_splits - 1) / lay.q_splits;
    k_begin = min(id.split * per, tiles) * kTile;
    k_stop = min(min((id.split + 1) * per, tiles) * kTile, key_end);
    const LOGKV_G uint16_t* qrow = gp(a.q) + b * a.q_sb + head * a.q_sh + t * a.q_st;
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks)
      qf[ks] = __builtin_bit_cast(bf16x8, query_unit(a, qrow, 16 * ks + 8 * h, lay.vec_q));
    const LOGKV_G uint16_t* drow = gp(gr.dout) + b * gr.do_sb + head * gr.do_sh + t * gr.do_st;
#pragma unroll
    for (int st = 0; st < 2 * NDV; ++st)
      df[st] = __builtin_bit_cast(bf16x8, row_unit(drow, 16 * st + 8 * h, a.dv, lay.vec_do));
  }

  template <class F>
  __device__ __forceinline__ void walk(const logkv_attention_args& a, uint16_t (*k_s)[kTile * kLdK],
                                       uint16_t (*v_s)[kTile * kLdD], F&& f) const {
    const LOGKV_G uint16_t* kbase = gp(a.k) + static_cast<int64_t>(lane_ix) * a.cap * a.dim;
    const LOGKV_G uint16_t* vbase = gp(a.v) + static_cast<int64_t>(lane_ix) * a.cap * a.dim;
    const int l = lane_id(), h = l >> 5, col = l & 31;
    const int n = k_begin < k_stop ? (k_stop - k_begin + kTile - 1) / kTile : 0;
    KvTiles<NKS, NDV, 64 * kQWaves> tiles;
    if (n > 0) {
      tiles.load(a, kbase, vbase, k_begin, k_stop);
      tiles.store(k_s[0], v_s[0]);
      if (n > 1) tiles.load(a, kbase, vbase, k_begin + kTile, k_stop);
    }
    __syncthreads();
    for (int it = 0; it < n; ++it) {
      const int t0 = k_begin + it * kTile, bf = it & 1;
      const uint16_t* kt = k_s[bf];
      const uint16_t* vt = v_s[bf];
      f32x16 s[2], dp[2];
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          s[kb][i] = 0.f;
          dp[kb][i] = 0.f;
        }
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks)
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
          s[kb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(load8(kt + (32 * kb + col) * kLdK + 16 * ks + 8 * h), qf[ks],
                                                          s[kb], 0, 0, 0);
#pragma unroll
      for (int st = 0; st < 2 * NDV; ++st)
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
          dp[kb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(load8(vt + (32 * kb + col) * kLdD + 16 * st + 8 * h), df[st],
                                                           dp[kb], 0, 0, 0);
      // Tiles with rows past the end or past some query's causal limit (uniform over the block).
      if (t0 + kTile > k_stop || (a.causal_tail && t0 + kTile > tail0)) {
        const int lim = (a.causal_tail ? min(k_stop, tail0 + t + 1) : k_stop) - t0 - 4 * h;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
          for (int i = 0; i < 16; ++i)
            s[kb][i] = 32 * kb + 8 * (i / 4) + (i % 4) < lim ? s[kb][i] : -__builtin_inff();
      }
      f(s, dp, kt);
      if (it + 1 < n) {
        tiles.store(k_s[bf ^ 1], v_s[bf ^ 1]);
        if (it + 2 < n) tiles.load(a, kbase, vbase, t0 + 2 * kTile, k_stop);
      }
      __syncthreads();
    }
  }
};

}  // namespace

template <int NKS, int NDV>
__global__ __launch_bounds__(64 * kQWaves, 2) void stats_kernel(logkv_attention_args a, const int32_t* __restrict__ width_ptr,
                                                       logkv_attention_grad_args gr, BwdLayout lay) {
  __shared__ __align__(16) uint16_t k_s[2][kTile * kLdK];
  __shared__ __align__(16) uint16_t v_s[2][kTile * kLdD];
  const BwdBlock id = bwd_block();
  const QueryWalk<NKS, NDV> me(a, width_ptr, gr, lay, id);
  const float c2 = a.scale * kLog2e;
  float m = -__builtin_inff(), lsum = 0.f, dacc = 0.f;
  me.walk(a, k_s, v_s, [&](f32x16 (&s)[2], f32x16 (&dp)[2], const uint16_t*) {
    float mx = -__builtin_inff();
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[kb][i]);
    mx = fmaxf(mx, __shfl_xor(mx, 32, kWave));
    const float m_new = fmaxf(m, mx * c2);
    const float mb = m_new == -__builtin_inff() ? 0.f : m_new;
    float sum = 0.f, dsum = 0.f;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[kb][i], c2, -mb));
        sum += p;
        dsum = __builtin_fmaf(p, dp[kb][i], dsum);
      }
    const float corr = __builtin_amdgcn_exp2f(m - mb);
    lsum = lsum * corr + sum;     // this lane's half of the keys; the halves are added below
    dacc = dacc * corr + dsum;
    m = m_new;
  });
  lsum += __shfl_xor(lsum, 32, kWave);
  dacc += __shfl_xor(dacc, 32, kWave);
  if (me.q_ok && lane_id() < 32) {
    const int nq = a.n_heads / a.n_groups * a.tq;
    *reinterpret_cast<float4*>(lay.part + ((static_cast<int64_t>(id.lane) * lay.q_splits + id.split) * nq + me.qi) * 4) =
        make_float4(m, lsum, dacc, 0.f);
  }
}

template <int NKS, int NDV>
__global__ __launch_bounds__(64 * kQWaves, 2) void dq_kernel(logkv_attention_args a, const int32_t* __restrict__ width_ptr,
                                                    logkv_attention_grad_args gr, BwdLayout lay) {
  __shared__ __align__(16) uint16_t k_s[2][kTile * kLdK];
  __shared__ __align__(16) uint16_t v_s[2][kTile * kLdD];
  const BwdBlock id = bwd_block();
  const QueryWalk<NKS, NDV> me(a, width_ptr, gr, lay, id);
  const int nq = a.n_heads / a.n_groups * a.tq, h = lane_id() >> 5;
  const float c2 = a.scale * kLog2e;
  // The parts of this lane's query, combined in part order.
  const float4* pp = reinterpret_cast<const float4*>(lay.part) +
                     static_cast<int64_t>(id.lane) * lay.q_splits * nq + (me.q_ok ? me.qi : nq - 1);
  float m = -__builtin_inff(), lsum = 0.f, dacc = 0.f;
  for (int sp = 0; sp < lay.q_splits; ++sp) m = fmaxf(m, pp[static_cast<int64_t>(sp) * nq].x);
  for (int sp = 0; sp < lay.q_splits; ++sp) {
    const float4 x = pp[static_cast<int64_t>(sp) * nq];
    const float f = x.x == -__builtin_inff() ? 0.f : __builtin_amdgcn_exp2f(x.x - m);
    lsum += x.y * f;
    dacc += x.z * f;
  }
  const float lse = lsum > 0.f ? m + __log2f(lsum) : 0.f;
  const float dsum = lsum > 0.f ? dacc / lsum : 0.f;
  if (id.split == 0 && me.q_ok && h == 0)
    *reinterpret_cast<float2*>(lay.stats + (static_cast<int64_t>(id.lane) * nq + me.qi) * 2) = make_float2(lse, dsum);
  f32x16 dq[NDV];
#pragma unroll
  for (int blk = 0; blk < NDV; ++blk)
#pragma unroll
    for (int i = 0; i < 16; ++i) dq[blk][i] = 0.f;
  me.walk(a, k_s, v_s, [&](f32x16 (&s)[2], f32x16 (&dp)[2], const uint16_t* kt) {
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[kb][i], c2, -lse));
        dp[kb][i] = p * (dp[kb][i] - dsum);
      }
#pragma unroll
    for (int st = 0; st < 4; ++st) {
      bf16x8 dh, dl;
      regs_b(dp, st, dh, dl);
      bf16x8 kf[NDV];
#pragma unroll
      for (int blk = 0; blk < NDV; ++blk) kf[blk] = load_tr<kLdK>(kt, 32 * blk, st);
#pragma unroll
      for (int blk = 0; blk < NDV; ++blk) dq[blk] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[blk], dh, dq[blk], 0, 0, 0);
#pragma unroll
      for (int blk = 0; blk < NDV; ++blk) dq[blk] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[blk], dl, dq[blk], 0, 0, 0);
    }
  });
  if (!me.q_ok) return;
  if (lay.q_splits > 1) {
    float* out = lay.grad + ((static_cast<int64_t>(id.lane) * lay.q_splits + id.split) * nq + me.qi) * a.dk;
#pragma unroll
    for (int blk = 0; blk < NDV; ++blk)
#pragma unroll
      for (int i4 = 0; i4 < 4; ++i4) {
        const int d = 32 * blk + 8 * i4 + 4 * h;
        if (d < a.dk)
          *reinterpret_cast<float4*>(out + d) =
              make_float4(dq[blk][4 * i4], dq[blk][4 * i4 + 1], dq[blk][4 * i4 + 2], dq[blk][4 * i4 + 3]);
      }
    return;
  }
  LOGKV_G uint16_t* drow = gp(gr.dq) + me.b * gr.dq_sb + me.head * gr.dq_sh + me.t * gr.dq_st;
#pragma unroll
  for (int blk = 0; blk < NDV; ++blk)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int d = 32 * blk + 8 * (i / 4) + 4 * h + (i % 4);
      if (d < a.dk) drow[d] = f32_to_bf16(dq[blk][i] * a.scale);
    }
}

// dq = scale * (the parts' partials in part order): one thread per query and four features.
__global__ __launch_bounds__(256) void sum_dq_kernel(logkv_attention_args a, logkv_attention_grad_args gr, BwdLayout lay) {
  const int nq = a.n_heads / a.n_groups * a.tq, units = a.dk / 4;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nq * units) return;
  const int qi = i / units, d = 4 * (i % units), lane_ix = blockIdx.y;
  const float* part = lay.grad + (static_cast<int64_t>(lane_ix) * lay.q_splits * nq + qi) * a.dk + d;
  float x[4] = {0.f, 0.f, 0.f, 0.f};
  for (int sp = 0; sp < lay.q_splits; ++sp) {
    const float4 p = *reinterpret_cast<const float4*>(part + static_cast<int64_t>(sp) * nq * a.dk);
    x[0] += p.x;
    x[1] += p.y;
    x[2] += p.z;
    x[3] += p.w;
  }
  uint32_t o[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) o[j] = f32_to_bf16(x[j] * a.scale);
  const int b = lane_ix / a.n_groups, head = (lane_ix % a.n_groups) * (a.n_heads / a.n_groups) + qi / a.tq, t = qi % a.tq;
  LOGKV_G uint16_t* row = gp(gr.dq) + b * gr.dq_sb + head * gr.dq_sh + t * gr.dq_st + d;
  if (lay.vec_dq) {
    *(LOGKV_G uint2*)(row) = make_uint2(o[0] | (o[1] << 16), o[2] | (o[3] << 16));
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j) row[j] = static_cast<uint16_t>(o[j]);
  }
}

template <int NKS, int NDV>
__global__ __launch_bounds__(64 * kKWaves, 1) void dkv_kernel(logkv_attention_args a, const int32_t* __restrict__ width_ptr,
                                                     logkv_attention_grad_args gr, BwdLayout lay) {
  constexpr int kThreads = 64 * kKWaves, kUnitsQ = 2 * NKS, kUnitsD = 4 * NDV;
  constexpr int kTasksQ = (kTile * kUnitsQ + kThreads - 1) / kThreads, kTasksD = (kTile * kUnitsD + kThreads - 1) / kThreads;
  __shared__ __align__(16) uint16_t q_s[2][kTile * kLdK];
  __shared__ __align__(16) uint16_t d_s[2][kTile * kLdD];
  __shared__ __align__(16) float lse_s[2][kTile];
  __shared__ __align__(16) float dsum_s[2][kTile];
  __shared__ __align__(16) int t_s[2][kTile];
  const BwdBlock id = bwd_block();
  const int lane_ix = id.lane, G = a.n_groups, b = lane_ix / G, g = lane_ix % G;
  const int rep = a.n_heads / G, nq = rep * a.tq;
  const int w = wave_id(), l = lane_id(), h = l >> 5, col = l & 31, tid = static_cast<int>(threadIdx.x);
  const int total = packed_total(a, width_ptr);
  const int tail0 = total - a.causal_tail;
  const int first = total - gr.grad_rows;                // first gradient row
  const int r_first = first + id.x * kKRows;
  const int key = r_first + w * 32 + col;                  // this lane's key row
  const bool key_ok = key < total && key >= 0 && key >= first;
  const float c2 = a.scale * kLog2e;
  // The lane's own key and value as B fragments (columns past the packed width / dv zero).
  bf16x8 kf[NKS], vf[2 * NDV];
  {
    const int64_t row = (static_cast<int64_t>(lane_ix) * a.cap + (key_ok ? key : 0)) * a.dim;
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks)
      kf[ks] = __builtin_bit_cast(bf16x8, row_unit(gp(a.k) + row, 16 * ks + 8 * h, a.dim, true));
#pragma unroll
    for (int st = 0; st < 2 * NDV; ++st)
      vf[st] = __builtin_bit_cast(bf16x8, row_unit(gp(a.v) + row, 16 * st + 8 * h, a.dv, true));
  }
  // Query tiles of this part whose last causal index reaches the block's first row: a tile
  // all of whose queries come before every row of the block has no visible pair.
  const int tiles = (nq + kTile - 1) / kTile, per = (tiles + lay.k_splits - 1) / lay.k_splits;
  const int tile_end = min((id.split + 1) * per, tiles);
  const int min_t = a.causal_tail ? r_first - tail0 : 0;
  auto next_tile = [&](int tile) {
    for (; tile < tile_end; ++tile) {
      const int q0 = tile * kTile, qe = min(q0 + kTile, nq) - 1;
      if (!a.causal_tail || (q0 / a.tq == qe / a.tq ? qe % a.tq : a.tq - 1) >= min_t) break;
    }
    return tile;
  };
  uint4 qx[kTasksQ], dx[kTasksD];
  float lse_x = 0.f, dsum_x = 0.f;
  int t_x = 0;
  auto load = [&](int tile) {
    const int q0 = tile * kTile;
    auto row_of = [&](int r, int64_t sb, int64_t sh, int64_t st) {
      const int qr = min(q0 + r, nq - 1);
      return b * sb + (g * rep + qr / a.tq) * sh + (qr % a.tq) * st;
    };
#pragma unroll
    for (int q = 0; q < kTasksQ; ++q) {
      const int i = tid + kThreads * q, r = min(i / kUnitsQ, kTile - 1), u = i % kUnitsQ;
      qx[q] = query_unit(a, gp(a.q) + row_of(r, a.q_sb, a.q_sh, a.q_st), 8 * u, lay.vec_q);
      if (q0 + r >= nq) qx[q] = make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (int q = 0; q < kTasksD; ++q) {
      const int i = tid + kThreads * q, r = min(i / kUnitsD, kTile - 1), u = i % kUnitsD;
      dx[q] = row_unit(gp(gr.dout) + row_of(r, gr.do_sb, gr.do_sh, gr.do_st), 8 * u, a.dv, lay.vec_do);
      if (q0 + r >= nq) dx[q] = make_uint4(0, 0, 0, 0);
    }
    if (tid < kTile) {
      const int qr = min(q0 + tid, nq - 1);
      const float2 x = *reinterpret_cast<const float2*>(lay.stats + (static_cast<int64_t>(lane_ix) * nq + qr) * 2);
      lse_x = x.x;
      dsum_x = x.y;
      t_x = q0 + tid < nq ? qr % a.tq : INT32_MIN;   // rows past the queries see no key: p = 0
    }
  };
  auto store = [&](int bf) {
#pragma unroll
    for (int q = 0; q < kTasksQ; ++q) {
      const int i = tid + kThreads * q, r = i / kUnitsQ, u = i % kUnitsQ;
      if (r < kTile) *reinterpret_cast<uint4*>(&q_s[bf][r * kLdK + 8 * u]) = qx[q];
    }
#pragma unroll
    for (int q = 0; q < kTasksD; ++q) {
      const int i = tid + kThreads * q, r = i / kUnitsD, u = i % kUnitsD;
      if (r < kTile) *reinterpret_cast<uint4*>(&d_s[bf][r * kLdD + 8 * u]) = dx[q];
    }
    if (tid < kTile) {
      lse_s[bf][tid] = lse_x;
      dsum_s[bf][tid] = dsum_x;
      t_s[bf][tid] = t_x;
    }
  };
  f32x16 dk[NDV], dv[NDV];
#pragma unroll
  for (int blk = 0; blk < NDV; ++blk)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      dk[blk][i] = 0.f;
      dv[blk][i] = 0.f;
    }
  // A query sees this lane's key where its causal index reaches kq.
  const int kq = a.causal_tail ? key - tail0 : -1;
  int tile = next_tile(id.split * per), ahead = tile;
  if (tile < tile_end) {
    load(tile);
    store(0);
    ahead = next_tile(tile + 1);
    if (ahead < tile_end) load(ahead);
  }
  __syncthreads();
  for (int bf = 0; tile < tile_end; bf ^= 1) {
    const uint16_t* qt = q_s[bf];
    const uint16_t* dt = d_s[bf];
    f32x16 s[2], dp[2];
#pragma unroll
    for (int qb = 0; qb < 2; ++qb)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        s[qb][i] = 0.f;
        dp[qb][i] = 0.f;
      }
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks)
#pragma unroll
      for (int qb = 0; qb < 2; ++qb)
        s[qb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(load8(qt + (32 * qb + col) * kLdK + 16 * ks + 8 * h), kf[ks], s[qb], 0, 0, 0);
#pragma unroll
    for (int st = 0; st < 2 * NDV; ++st)
#pragma unroll
      for (int qb = 0; qb < 2; ++qb)
        dp[qb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(load8(dt + (32 * qb + col) * kLdD + 16 * st + 8 * h), vf[st], dp[qb], 0, 0, 0);
    // P and dS of this lane's key against the tile's queries (element i of block qb is query
    // 32 qb + 8 (i / 4) + 4 h + i % 4).
#pragma unroll
    for (int qb = 0; qb < 2; ++qb)
#pragma unroll
      for (int i4 = 0; i4 < 4; ++i4) {
        const int r = 32 * qb + 8 * i4 + 4 * h;
        const float4 lse = *reinterpret_cast<const float4*>(&lse_s[bf][r]), ds = *reinterpret_cast<const float4*>(&dsum_s[bf][r]);
        const int4 tt = *reinterpret_cast<const int4*>(&t_s[bf][r]);
        const float lse4[4] = {lse.x, lse.y, lse.z, lse.w}, ds4[4] = {ds.x, ds.y, ds.z, ds.w};
        const int t4[4] = {tt.x, tt.y, tt.z, tt.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int i = 4 * i4 + j;
          const float p = kq <= t4[j] ? __builtin_amdgcn_exp2f(__builtin_fmaf(s[qb][i], c2, -lse4[j])) : 0.f;
          s[qb][i] = p;
          dp[qb][i] = p * (dp[qb][i] - ds4[j]);
        }
      }
#pragma unroll
    for (int st = 0; st < 4; ++st) {
      bf16x8 ph, pl, dh, dl;
      regs_b(s, st, ph, pl);
      regs_b(dp, st, dh, dl);
#pragma unroll
      for (int blk = 0; blk < NDV; ++blk) {
        const bf16x8 of = load_tr<kLdD>(dt, 32 * blk, st), qf = load_tr<kLdK>(qt, 32 * blk, st);
        dv[blk] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(of, ph, dv[blk], 0, 0, 0);
        dk[blk] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(qf, dh, dk[blk], 0, 0, 0);
        dv[blk] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(of, pl, dv[blk], 0, 0, 0);
        dk[blk] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(qf, dl, dk[blk], 0, 0, 0);
      }
    }
    tile = ahead;
    if (tile < tile_end) {
      store(bf ^ 1);
      ahead = next_tile(tile + 1);
      if (ahead < tile_end) load(ahead);
    }
    __syncthreads();
  }
  if (!key_ok) return;
  if (lay.k_splits > 1) {
    float* out = lay.grad + ((static_cast<int64_t>(lane_ix) * lay.k_splits + id.split) * gr.grad_rows + (key - first)) * (a.dk + a.dv);
#pragma unroll
    for (int blk = 0; blk < NDV; ++blk)
#pragma unroll
      for (int i4 = 0; i4 < 4; ++i4) {
        const int d = 32 * blk + 8 * i4 + 4 * h, i = 4 * i4;
        if (d < a.dk) *reinterpret_cast<float4*>(out + d) = make_float4(dk[blk][i], dk[blk][i + 1], dk[blk][i + 2], dk[blk][i + 3]);
        if (d < a.dv) *reinterpret_cast<float4*>(out + a.dk + d) = make_float4(dv[blk][i], dv[blk][i + 1], dv[blk][i + 2], dv[blk][i + 3]);
      }
    return;
  }
  const int64_t row = static_cast<int64_t>(lane_ix) * gr.grad_rows + (key - first);
#pragma unroll
  for (int blk = 0; blk < NDV; ++blk)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int d = 32 * blk + 8 * (i / 4) + 4 * h + (i % 4);
      if (d < a.dk) gp(gr.dk)[row * a.dk + d] = f32_to_bf16(dk[blk][i] * a.scale);
      if (d < a.dv) gp(gr.dv)[row * a.dv + d] = f32_to_bf16(dv[blk][i]);
    }
}

// dk = scale * and dv = the parts' partials in part order: one thread per row and four features.
__global__ __launch_bounds__(256) void sum_dkv_kernel(logkv_attention_args a, logkv_attention_grad_args gr, BwdLayout lay) {
  const int wid = a.dk + a.dv, units = wid / 4;
  const int i = blockIdx.x * blockDim.x + threadIdx.x, lane_ix = blockIdx.y;
  if (i >= gr.grad_rows * units) return;
  const int r = i / units, d = 4 * (i % units);
  const int64_t step = static_cast<int64_t>(gr.grad_rows) * wid;
  const float* part = lay.grad + static_cast<int64_t>(lane_ix) * lay.k_splits * step + static_cast<int64_t>(r) * wid + d;
  float x[4] = {0.f, 0.f, 0.f, 0.f};
  for (int sp = 0; sp < lay.k_splits; ++sp) {
    const float4 p = *reinterpret_cast<const float4*>(part + sp * step);
    x[0] += p.x;
    x[1] += p.y;
    x[2] += p.z;
    x[3] += p.w;
  }
  const int64_t row = static_cast<int64_t>(lane_ix) * gr.grad_rows + r;
  const bool key = d < a.dk;
  LOGKV_G uint16_t* out = key ? gp(gr.dk) + row * a.dk + d : gp(gr.dv) + row * a.dv + (d - a.dk);
#pragma unroll
  for (int j = 0; j < 4; ++j) out[j] = f32_to_bf16(key ? x[j] * a.scale : x[j]);
}

namespace {

// Parts of a walk of `tiles` tiles for `blocks` blocks at one block per CU: the count that costs
// least in tiles (dq and statistics together 6.4 us, dk / dv 5.3 us at 128 features): rounds over
// the 256 CUs, each of a part's tiles and one more for its start, and with more than one part a tile
// for the summing launch and 1/128 tile for every block's float32 partials, written and read back
// (0.13 MB at 128 features; at 1/64 a 512-row chunk of 8 lanes lost parts that pay, 99 -> 104 us).
// Without that charge 480 query blocks over 12K rows took 9 parts and 570 MB of partials to save
// three tiles: 3111 us, with one part 2908 us (288 over 5K: 8 parts 982, 5 parts 866 us).
int bwd_splits(int64_t blocks, int tiles) {
  int best = 1;
  int64_t best_cost = INT64_MAX;   // in 1/128 tiles
  for (int s = 1; s <= std::min(kMaxSplits, std::max(1, tiles / 2)); ++s) {
    const int64_t rounds = (blocks * s + 255) / 256;
    const int64_t cost = 128 * rounds * ((tiles + s - 1) / s + 1) + (s > 1 ? 128 + blocks * s : 0);
    if (cost < best_cost) {
      best_cost = cost;
      best = s;
    }
  }
  return best;
}

int dq_splits(const logkv_attention_args& a) {
  const int nq = a.n_heads / a.n_groups * a.tq;
  return bwd_splits(static_cast<int64_t>((nq + kQRows - 1) / kQRows) * a.n_batch * a.n_groups, (a.cap + kTile - 1) / kTile);
}

int dkv_splits(const logkv_attention_args& a, int grad_rows) {
  const int nq = a.n_heads / a.n_groups * a.tq;
  return bwd_splits(static_cast<int64_t>((grad_rows + kKRows - 1) / kKRows) * a.n_batch * a.n_groups, (nq + kTile - 1) / kTile);
}

// Workspace floats: [stats][parts][gradient partials], the last for dq and for the dk / dv of a
// chunk (grad_rows = tq); more gradient rows take as many parts as fit it.
struct BwdSizes {
  int64_t stats, part, grad;
};
BwdSizes bwd_sizes(const logkv_attention_args& a) {
  const int nq = a.n_heads / a.n_groups * a.tq, qs = dq_splits(a), ks = dkv_splits(a, a.tq);
  const int64_t lanes = static_cast<int64_t>(a.n_batch) * a.n_groups;
  const int64_t dq = qs > 1 ? lanes * qs * nq * a.dk : 0, dkv = ks > 1 ? lanes * ks * a.tq * (a.dk + a.dv) : 0;
  return {(lanes * nq * 2 + 3) / 4 * 4, lanes * qs * nq * 4, std::max(dq, dkv)};
}

bool aligned(const void* p, int64_t sb, int64_t sh, int64_t st, int bytes) {
  const int64_t n = bytes / 2;
  return reinterpret_cast<uintptr_t>(p) % bytes == 0 && sb % n == 0 && sh % n == 0 && st % n == 0;
}

}  // namespace

int64_t chunk_backward_workspace_floats(const logkv_attention_args& a) {
  const BwdSizes z = bwd_sizes(a);
  return z.stats + z.part + z.grad + 3;   // the regions start at the workspace's first 16-byte boundary
}

int launch_chunk_backward(const logkv_attention_args& a, const int32_t* width, const logkv_attention_grad_args& g,
                          float* ws, hipStream_t stream) {
  const int nq = (a.n_heads / a.n_groups) * a.tq;
  const int lanes = a.n_batch * a.n_groups;
  const BwdSizes z = bwd_sizes(a);
  BwdLayout lay{};
  lay.q_splits = dq_splits(a);
  lay.k_splits = 1;
  if (g.grad_rows > 0) {
    const int64_t fit = z.grad / (static_cast<int64_t>(lanes) * g.grad_rows * (a.dk + a.dv));
    lay.k_splits = static_cast<int>(std::max<int64_t>(1, std::min<int64_t>(dkv_splits(a, g.grad_rows), fit)));
  }
  lay.vec_q = aligned(a.q, a.q_sb, a.q_sh, a.q_st, 16);
  lay.vec_do = aligned(g.dout, g.do_sb, g.do_sh, g.do_st, 16);
  lay.vec_dq = aligned(g.dq, g.dq_sb, g.dq_sh, g.dq_st, 8);
  lay.stats = reinterpret_cast<float*>((reinterpret_cast<uintptr_t>(ws) + 15) / 16 * 16);
  lay.part = lay.stats + z.stats;
  lay.grad = lay.part + z.part;
  const dim3 qgrid((nq + kQRows - 1) / kQRows, lay.q_splits, lanes);
  const dim3 kgrid((g.grad_rows + kKRows - 1) / kKRows, lay.k_splits, lanes);
  auto run = [&](auto stats, auto dq, auto dkv) {
    hipLaunchKernelGGL(stats, qgrid, dim3(64 * kQWaves), 0, stream, a, width, g, lay);
    hipLaunchKernelGGL(dq, qgrid, dim3(64 * kQWaves), 0, stream, a, width, g, lay);
    if (lay.q_splits > 1)
      hipLaunchKernelGGL(sum_dq_kernel, dim3((nq * (a.dk / 4) + 255) / 256, lanes), dim3(256), 0, stream, a, g, lay);
    if (g.grad_rows > 0) {
      hipLaunchKernelGGL(dkv, kgrid, dim3(64 * kKWaves), 0, stream, a, width, g, lay);
      if (lay.k_splits > 1)
        hipLaunchKernelGGL(sum_dkv_kernel, dim3((static_cast<unsigned>(g.grad_rows) * ((a.dk + a.dv) / 4) + 255) / 256, lanes),
                           dim3(256), 0, stream, a, g, lay);
    }
  };
  // Head dim 64 (5 steps of the packed width, 2 blocks of dk and dv) has its own kernels; every
  // other shape runs the full ones on zero padding.
  if (a.dim <= 80 && a.dk <= 64 && a.dv <= 64) run(stats_kernel<5, 2>, dq_kernel<5, 2>, dkv_kernel<5, 2>);
  else run(stats_kernel<9, 4>, dq_kernel<9, 4>, dkv_kernel<9, 4>);
  return hipGetLastError() == hipSuccess ? LOGKV_OK : LOGKV_ERUNTIME;
}

}  // namespace logkv
