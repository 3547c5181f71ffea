// Decode attention on the matrix cores: at most 16 query rows per KV group (heads per group x
// query rows of a decode step) over the packed rows [pooled | exact | recent | current].
//
// Decode attention (litgpt/log_kv_cache.py:6428-6464, :6751-6758):
// softmax(scale * [q, 1/scale] . [k, bias]) v, the last causal_tail rows causal. A block of four
// waves takes one share of a lane's rows; its waves walk alternate 32-row tiles on their own,
// with no block barrier until their results are combined:
//   S^T = K Q^T by v_mfma_f32_16x16x32_bf16 (keys x queries: a lane holds 8 keys of its query
//   l % 16), K fragments loaded from global memory in operand layout;
//   online softmax per lane (the other 24 keys of the tile in the lanes of the same l % 16);
//   O^T += V^T P^T, V staged row-major in the wave's own LDS and read transposed
//   (ds_read_b64_tr_b16), P as three bf16 parts (8 + 8 + 8 bits: the float32 value).
// The next tile's K and V are in registers, or on their way there, while a tile is computed: the
// kernel is bound by HBM, the products cost 34 of the 16-cycle matrix instructions per 17 KB tile.
// Measured, packed rows of 128 features: 8 x 8 lanes of 8.4K rows, 2 queries each, 51 us (5.7 TB/s;
// a per-row-group form with vector dot products and no LDS 58 us); 4 x 8 lanes of 6K rows, 8
// queries, 27 us (staged tiles with scalar products 136 us); 8 lanes of 3K rows, 9.6 us (16.2 us).
#include <algorithm>

#include "route.hpp"

namespace logkv {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

constexpr int kWaves = 4;
constexpr int kRows = 32;          // packed rows per wave tile
constexpr int kQ = 16;             // query columns

// LDS row stride of a V tile (bf16): 8 dwords modulo 32, so the four rows of a transposed read
// fall into distinct banks.
constexpr int v_stride(int blocks) { return 16 * blocks + 16; }

}  // namespace

// NS 32-wide steps of the packed width, NB 16-wide blocks of dv.
template <int NS, int NB>
__global__ __launch_bounds__(64 * kWaves, NB <= 8 ? 2 : 1) void decode_mfma_kernel(logkv_attention_args a,
                                                                     const int32_t* __restrict__ width_ptr,
                                                                     float* __restrict__ part) {
  typedef __attribute__((address_space(3))) s16x4* lds4;
  constexpr int kLd = v_stride(NB), kVLoads = kRows * 2 * NB / 64;
  constexpr int kTileBytes = kRows * kLd * 2, kOutBytes = kQ * 16 * NB * 4;
  __shared__ __align__(16) uint8_t buf[kWaves][kTileBytes > kOutBytes ? kTileBytes : kOutBytes];
  __shared__ float m_s[kWaves][kQ], l_s[kWaves][kQ];
  const int lane = blockIdx.y, G = a.n_groups, b = lane / G, g = lane % G;
  const int rep = a.n_heads / G, nq = rep * a.tq, dim = a.dim, units = dim / 8, vunits = (a.dv + 7) / 8;
  const int w = wave_id(), l = lane_id(), col = l & 15, hq = l >> 4;
  const int total = min(*width_ptr + a.tail + (a.alpha_count_dev ? *a.alpha_count_dev : 0), a.cap);
  const int tail0 = total - a.causal_tail;
  // The lane's rows in gridDim.x equal shares, multiples of a pass of the block's waves; shares
  // past the rows write empty partials.
  constexpr int kPass = kWaves * kRows;
  const int splits = static_cast<int>(gridDim.x);
  const int share = max(kPass, (total + kPass * splits - 1) / (kPass * splits) * kPass);
  const int r_begin = min(static_cast<int>(blockIdx.x) * share, total), r_end = min(r_begin + share, total);
  float* out = part + (static_cast<int64_t>(lane) * splits + blockIdx.x) * nq * (a.dv + 2);

  // Query col as B fragments of [q, 1/scale, 0...]; columns past nq are zero.
  const int t = col % a.tq;
  bf16x8 qf[NS];
  {
    const int qc = col < nq ? col : nq - 1;
    const LOGKV_G uint16_t* qrow = gp(a.q) + b * a.q_sb + (g * rep + qc / a.tq) * a.q_sh + (qc % a.tq) * a.q_st;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      uint32_t e[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int d = 32 * s + 8 * hq + j;
        e[j] = d < a.dk ? qrow[d] : (d == a.dk ? f32_to_bf16(a.inv_scale_bf16) : 0u);
        if (col >= nq) e[j] = 0u;
      }
      qf[s] = __builtin_bit_cast(bf16x8, make_uint4(e[0] | (e[1] << 16), e[2] | (e[3] << 16), e[4] | (e[5] << 16),
                                                    e[6] | (e[7] << 16)));
    }
  }
  const LOGKV_G uint16_t* kbase = gp(a.k) + static_cast<int64_t>(lane) * a.cap * dim;
  const LOGKV_G uint16_t* vbase = gp(a.v) + static_cast<int64_t>(lane) * a.cap * dim;
  uint16_t* v_s = reinterpret_cast<uint16_t*>(buf[w]);

  uint4 kx[2][NS], vx[kVLoads];
  // Rows past the share: K repeats its last row (masked in the scores), V is zero.
  auto load = [&](int t0) {
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      const LOGKV_G uint16_t* row = kbase + static_cast<int64_t>(min(t0 + 16 * kb + col, r_end - 1)) * dim;
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        kx[kb][s] = make_uint4(0, 0, 0, 0);
        if (4 * s + hq < units) kx[kb][s] = *(const LOGKV_G uint4*)(row + 32 * s + 8 * hq);
      }
    }
#pragma unroll
    for (int i = 0; i < kVLoads; ++i) {
      const int e = l + 64 * i, r = e / (2 * NB), u = e % (2 * NB);
      vx[i] = make_uint4(0, 0, 0, 0);
      if (u < vunits && t0 + r < r_end) vx[i] = *(const LOGKV_G uint4*)(vbase + static_cast<int64_t>(t0 + r) * dim + 8 * u);
    }
  };
  f32x4 o[NB];
#pragma unroll
  for (int n = 0; n < NB; ++n) o[n] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -__builtin_inff(), lsum = 0.f;
  const int first = r_begin + w * kRows;
  if (first < r_end) load(first);
  for (int t0 = first; t0 < r_end; t0 += kPass) {
    f32x4 s[2];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) s[kb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int st = 0; st < NS; ++st)
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
        s[kb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, kx[kb][st]), qf[st], s[kb], 0, 0, 0);
    // An infinity or NaN in V takes P's high part only: the lower parts, which can be zero where P
    // is not, meet it as zero.
    u16x2 top = {0, 0};
#pragma unroll
    for (int i = 0; i < kVLoads; ++i) {
      const uint32_t x4[4] = {vx[i].x, vx[i].y, vx[i].z, vx[i].w};
#pragma unroll
      for (int j = 0; j < 4; ++j) top = __builtin_elementwise_max(top, __builtin_bit_cast(u16x2, x4[j] & 0x7fff7fffu));
    }
    const bool finite = __ballot(top[0] >= 0x7f80 || top[1] >= 0x7f80) == 0;
    // The wave's own V tile: written and read by this wave only (LDS accesses of a wave complete
    // in order; the fences keep the compiler's order).
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int i = 0; i < kVLoads; ++i) {
      const int e = l + 64 * i, r = e / (2 * NB), u = e % (2 * NB);
      *reinterpret_cast<uint4*>(v_s + r * kLd + 8 * u) = vx[i];
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (t0 + kPass < r_end) load(t0 + kPass);
    // Scores in base 2: rows past the share and past the causal limit are masked (element i of
    // block kb is row t0 + 16 kb + 4 hq + i).
    const int lim = (a.causal_tail ? min(r_end, tail0 + t + 1) : r_end) - t0 - 4 * hq;
    float mx = -__builtin_inff();
    const float c2 = a.scale * 1.44269504088896341f;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        s[kb][i] = 16 * kb + i < lim ? s[kb][i] * c2 : -__builtin_inff();
        mx = fmaxf(mx, s[kb][i]);
      }
    mx = fmaxf(mx, __shfl_xor(mx, 16, kWave));
    mx = fmaxf(mx, __shfl_xor(mx, 32, kWave));
    const float m_new = fmaxf(m, mx);
    const float mb = m_new == -__builtin_inff() ? 0.f : m_new;
    if (__ballot(m_new != m)) {
      const float corr = __builtin_amdgcn_exp2f(m - mb);
      lsum *= corr;
#pragma unroll
      for (int n = 0; n < NB; ++n) o[n] *= corr;
    }
    m = m_new;
    // P = hi + mid + lo, each the truncated top 8 significant bits of what is left.
    uint32_t part_w[3][4];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        float x0 = __builtin_amdgcn_exp2f(s[kb][2 * j] - mb), x1 = __builtin_amdgcn_exp2f(s[kb][2 * j + 1] - mb);
        lsum += x0 + x1;
#pragma unroll
        for (int q = 0; q < 3; ++q) {
          const uint32_t u0 = __float_as_uint(x0), u1 = __float_as_uint(x1);
          part_w[q][2 * kb + j] = __builtin_amdgcn_perm(u1, u0, 0x07060302u);
          x0 -= __uint_as_float(u0 & 0xffff0000u);
          x1 -= __uint_as_float(u1 & 0xffff0000u);
        }
      }
    bf16x8 pf[3];
#pragma unroll
    for (int q = 0; q < 3; ++q)
      pf[q] = __builtin_bit_cast(bf16x8, make_uint4(part_w[q][0], part_w[q][1], part_w[q][2], part_w[q][3]));
    // V^T fragments: features 16 n + col, rows 4 hq .. + 3 and 16 + 4 hq .. + 3 (P's own order).
#pragma unroll
    for (int n = 0; n < NB; ++n) {
      const uint16_t* p = v_s + (4 * hq + (col >> 2)) * kLd + 16 * n + 4 * (col & 3);
      const uint2 x = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)(p)));
      const uint2 y = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)(p + 16 * kLd)));
      uint32_t vw[4] = {x.x, x.y, y.x, y.y};
      o[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, make_uint4(vw[0], vw[1], vw[2], vw[3])),
                                                     pf[0], o[n], 0, 0, 0);
      if (!finite) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if ((vw[j] & 0x7f80u) == 0x7f80u) vw[j] &= 0xffff0000u;
          if ((vw[j] & 0x7f800000u) == 0x7f800000u) vw[j] &= 0xffffu;
        }
      }
#pragma unroll
      for (int q = 1; q < 3; ++q)
        o[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, make_uint4(vw[0], vw[1], vw[2], vw[3])),
                                                       pf[q], o[n], 0, 0, 0);
    }
  }
  // Waves combined in wave order: [m, l, acc[dv]] per query of this share (base-e maximum).
  lsum += __shfl_xor(lsum, 16, kWave);
  lsum += __shfl_xor(lsum, 32, kWave);
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  float* acc_w = reinterpret_cast<float*>(buf[w]);
#pragma unroll
  for (int n = 0; n < NB; ++n)
    *reinterpret_cast<f32x4*>(acc_w + col * (16 * NB) + 16 * n + 4 * hq) = o[n];
  if (hq == 0) {
    m_s[w][col] = m;
    l_s[w][col] = lsum;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < nq * (a.dv + 2); e += blockDim.x) {
    const int q = e / (a.dv + 2), c = e % (a.dv + 2);
    float mx = -__builtin_inff();
#pragma unroll
    for (int i = 0; i < kWaves; ++i) mx = fmaxf(mx, m_s[i][q]);
    float val = 0.f;
#pragma unroll
    for (int i = 0; i < kWaves; ++i) {
      const float x = c < 2 ? l_s[i][q] : reinterpret_cast<const float*>(buf[i])[q * (16 * NB) + c - 2];
      if (m_s[i][q] != -__builtin_inff()) val += x * __builtin_amdgcn_exp2f(m_s[i][q] - mx);
    }
    out[e] = c == 0 ? mx * 0.693147180559945309f : val;
  }
}

int launch_decode_mfma(const logkv_attention_args& a, const int32_t* width, float* part, int n_split, hipStream_t stream) {
  const dim3 grid(n_split, a.n_batch * a.n_groups);
  // By packed width and value width: head dims up to 64 and up to 128, wider keys with values up to
  // 128 (all at two waves per SIMD), and the rest up to the packed limit of 264 and dv of 256 (one).
  // Units a shape does not have are zero and not read. Keys of 192 with values of 128, 64 lanes of 4K
  // rows, 2 queries: 40 us (47 us in the widest kernel, which also read the values' padding).
  if (a.dim <= 96 && a.dv <= 64)
    hipLaunchKernelGGL((decode_mfma_kernel<3, 4>), grid, dim3(64 * kWaves), 0, stream, a, width, part);
  else if (a.dim <= 160 && a.dv <= 128)
    hipLaunchKernelGGL((decode_mfma_kernel<5, 8>), grid, dim3(64 * kWaves), 0, stream, a, width, part);
  else if (a.dv <= 128)
    hipLaunchKernelGGL((decode_mfma_kernel<9, 8>), grid, dim3(64 * kWaves), 0, stream, a, width, part);
  else
    hipLaunchKernelGGL((decode_mfma_kernel<9, 16>), grid, dim3(64 * kWaves), 0, stream, a, width, part);
  return hipGetLastError() == hipSuccess ? LOGKV_OK : LOGKV_ERUNTIME;
}

}  // namespace logkv
