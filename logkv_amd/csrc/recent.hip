// The recent window's row moves on the device: one launch appends a block of
// rows to every recent buffer, one launch moves the rows left after a flush to
// the front and clears the vacated rows (litgpt/log_kv_cache.py:5668-5718,
// :5640-5659, there as separate tensor copies and fills per buffer).
//
// Bf16 rows move in 16-byte units of eight features (8-byte ones where a width
// or a source row does not allow it), one per thread, a block per 256 units of
// one lane's buffer, so that a block's source and destination are uniform;
// positions and span flags one entry per thread. A launch holds at most 2^31
// threads; longer moves are several launches. Bound by HBM: 224 lanes x 2048
// rows of 3 x 128 features are appended in 159 us (4.4 TB/s; 8-byte units in a
// grid-stride loop over all buffers 191 us; two units per thread 164 us, and
// 18 us instead of 7 us at 8 lanes) and moved and cleared in 183 us (239 us).
#include <algorithm>

#include "route.hpp"

namespace logkv {

namespace {

constexpr int kThreads = 256;
constexpr int64_t kLaunchThreads = int64_t(1) << 31;   // threads of one launch

template <int F>
struct UnitOf;
template <>
struct UnitOf<4> {
  using type = uint2;
  static __device__ __forceinline__ uint2 zero() { return make_uint2(0u, 0u); }
};
template <>
struct UnitOf<8> {
  using type = uint4;
  static __device__ __forceinline__ uint4 zero() { return make_uint4(0u, 0u, 0u, 0u); }
};

// The block's lane, buffer (0 keys, 1 raw keys, 2 values) and first unit of that buffer's rows.
struct RowBlock {
  int lane, buf, first;
};
__device__ __forceinline__ RowBlock row_block(int chunks, int lane0) {
  const int i = static_cast<int>(blockIdx.x) / chunks;
  return RowBlock{lane0 + i / 3, i % 3, (static_cast<int>(blockIdx.x) - i * chunks) * kThreads};
}

}  // namespace

// Rows [0, n) of each source into recent rows [at, at + n); `chunks` blocks to a lane's buffer.
template <int F>
__global__ __launch_bounds__(kThreads) void recent_append_kernel(logkv_recent_args a, int at, int n, int chunks,
                                                                    int lane0) {
  using Unit = typename UnitOf<F>::type;
  const RowBlock blk = row_block(chunks, lane0);
  const int b = blk.lane / a.n_groups, g = blk.lane % a.n_groups, tid = static_cast<int>(threadIdx.x);
  const int d = blk.buf == 0 ? a.dk : (blk.buf == 1 ? a.dkr : a.dv), units = d / F, total = n * units;
  const LOGKV_G uint16_t* src = blk.buf == 0 ? gp(a.k) + b * a.k_sb + g * a.k_sg
                              : blk.buf == 1 ? gp(a.k_raw) + b * a.kr_sb + g * a.kr_sg
                                             : gp(a.v) + b * a.v_sb + g * a.v_sg;
  const int64_t st = blk.buf == 0 ? a.k_st : (blk.buf == 1 ? a.kr_st : a.v_st);
  LOGKV_G uint16_t* dst = (blk.buf == 0 ? gp(a.recent_k) : (blk.buf == 1 ? gp(a.recent_k_raw) : gp(a.recent_v))) +
                          (static_cast<int64_t>(blk.lane) * a.cap + at) * d;
  const int i = blk.first + tid;
  if (i < total) {
    const int t = i / units;
    const Unit x = *reinterpret_cast<const LOGKV_G Unit*>(src + t * st + F * (i - t * units));
    *reinterpret_cast<LOGKV_G Unit*>(dst + static_cast<int64_t>(F) * i) = x;
  }
  if (g != 0 || blk.buf != 0) return;
  for (int t = blk.first + tid; t < n; t += chunks * kThreads) {
    a.recent_pos[static_cast<int64_t>(b) * a.cap + at + t] = a.pos[b * a.pos_sb + t * a.pos_st];
    if (a.recent_ends) a.recent_ends[static_cast<int64_t>(b) * a.cap + at + t] = a.ends[b * a.ends_sb + t];
  }
}

// Rows [0, n): the first `remaining` receive the rows `take` further on, which become zero, and the
// others become zero. Of a window of `count` rows that loses `take` all rows [0, take) are given,
// with count - take of them receiving: count - take <= take, so every source row lies in the
// cleared range past them, and the thread that reads it clears it.
template <int F>
__global__ __launch_bounds__(kThreads) void recent_shift_kernel(logkv_recent_args a, int take, int n, int remaining,
                                                                   int chunks, int lane0) {
  using Unit = typename UnitOf<F>::type;
  const RowBlock blk = row_block(chunks, lane0);
  const int b = blk.lane / a.n_groups, g = blk.lane % a.n_groups, tid = static_cast<int>(threadIdx.x);
  const int d = blk.buf == 0 ? a.dk : (blk.buf == 1 ? a.dkr : a.dv), units = d / F, total = n * units;
  LOGKV_G uint16_t* dst = (blk.buf == 0 ? gp(a.recent_k) : (blk.buf == 1 ? gp(a.recent_k_raw) : gp(a.recent_v))) +
                          static_cast<int64_t>(blk.lane) * a.cap * d;
  LOGKV_G uint16_t* src = dst + static_cast<int64_t>(take) * d;
  const int moved = remaining * units;
  const int i = blk.first + tid;
  if (i < moved) {
    const Unit x = *reinterpret_cast<const LOGKV_G Unit*>(src + static_cast<int64_t>(F) * i);
    *reinterpret_cast<LOGKV_G Unit*>(dst + static_cast<int64_t>(F) * i) = x;
    *reinterpret_cast<LOGKV_G Unit*>(src + static_cast<int64_t>(F) * i) = UnitOf<F>::zero();
  } else if (i < total) {
    *reinterpret_cast<LOGKV_G Unit*>(dst + static_cast<int64_t>(F) * i) = UnitOf<F>::zero();
  }
  if (g != 0 || blk.buf != 0) return;
  const int64_t pos0 = static_cast<int64_t>(b) * a.cap;
  for (int r = blk.first + tid; r < n; r += chunks * kThreads) {
    if (r < remaining) {
      a.recent_pos[pos0 + r] = a.recent_pos[pos0 + take + r];
      a.recent_pos[pos0 + take + r] = 0;
      if (a.recent_ends) {
        a.recent_ends[pos0 + r] = a.recent_ends[pos0 + take + r];
        a.recent_ends[pos0 + take + r] = 0;
      }
    } else {
      a.recent_pos[pos0 + r] = 0;
      if (a.recent_ends) a.recent_ends[pos0 + r] = 0;
    }
  }
}

namespace {

bool rows16(const void* p, int64_t sb, int64_t sg, int64_t st) {
  return reinterpret_cast<uintptr_t>(p) % 16 == 0 && sb % 8 == 0 && sg % 8 == 0 && st % 8 == 0;
}

bool wide_window(const logkv_recent_args& a) {
  return a.dk % 8 == 0 && a.dkr % 8 == 0 && a.dv % 8 == 0 && rows16(a.recent_k, 0, 0, 0) &&
         rows16(a.recent_k_raw, 0, 0, 0) && rows16(a.recent_v, 0, 0, 0);
}

// Calls launch(first row, rows, first lane, grid, chunks) for rows [0, rows) and every lane, in as many
// parts as kLaunchThreads asks for (one, short of tens of GB).
template <class Launch>
void by_parts(const logkv_recent_args& a, int f, int rows, Launch launch) {
  const int units = std::max(a.dk, std::max(a.dkr, a.dv)) / f;   // of a row's widest buffer
  const int lanes = a.n_batch * a.n_groups;
  const int max_rows = static_cast<int>((kLaunchThreads / 3 - kThreads) / units);
  for (int row0 = 0; row0 < rows; row0 += std::min(max_rows, rows - row0)) {
    const int n = std::min(max_rows, rows - row0), total = n * units;
    const int chunks = (total + kThreads - 1) / kThreads;
    const int max_lanes = static_cast<int>(std::min<int64_t>(lanes, kLaunchThreads / (int64_t(3) * chunks * kThreads)));
    for (int lane0 = 0; lane0 < lanes; lane0 += std::min(max_lanes, lanes - lane0))
      launch(row0, n, lane0, dim3(static_cast<unsigned>(chunks) * 3 * std::min(max_lanes, lanes - lane0)), chunks);
  }
}

}  // namespace

int launch_recent_append(const logkv_recent_args& a, int at, int n, hipStream_t stream) {
  const bool wide = wide_window(a) && rows16(a.k, a.k_sb, a.k_sg, a.k_st) && rows16(a.k_raw, a.kr_sb, a.kr_sg, a.kr_st) &&
                    rows16(a.v, a.v_sb, a.v_sg, a.v_st);
  by_parts(a, wide ? 8 : 4, n, [&](int row0, int rows, int lane0, dim3 grid, int chunks) {
    logkv_recent_args p = a;
    p.k += row0 * a.k_st;
    p.k_raw += row0 * a.kr_st;
    p.v += row0 * a.v_st;
    p.pos += row0 * a.pos_st;
    if (p.ends) p.ends += row0;
    hipLaunchKernelGGL(wide ? recent_append_kernel<8> : recent_append_kernel<4>, grid, dim3(kThreads), 0, stream, p,
                       at + row0, rows, chunks, lane0);
  });
  return hipGetLastError() == hipSuccess ? LOGKV_OK : LOGKV_ERUNTIME;
}

int launch_recent_shift(const logkv_recent_args& a, int take, int count, hipStream_t stream) {
  const bool wide = wide_window(a);
  by_parts(a, wide ? 8 : 4, take, [&](int row0, int rows, int lane0, dim3 grid, int chunks) {
    logkv_recent_args p = a;
    p.recent_k += static_cast<int64_t>(row0) * a.dk;
    p.recent_k_raw += static_cast<int64_t>(row0) * a.dkr;
    p.recent_v += static_cast<int64_t>(row0) * a.dv;
    p.recent_pos += row0;
    if (p.recent_ends) p.recent_ends += row0;
    const int remaining = std::max(0, std::min(count - take - row0, rows));
    hipLaunchKernelGGL(wide ? recent_shift_kernel<8> : recent_shift_kernel<4>, grid, dim3(kThreads), 0, stream, p, take,
                       rows, remaining, chunks, lane0);
  });
  return hipGetLastError() == hipSuccess ? LOGKV_OK : LOGKV_ERUNTIME;
}

}  // namespace logkv
