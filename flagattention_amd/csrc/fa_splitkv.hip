// Split-KV forward (flash decoding) and the merge of its partial results.
//
// Replaces `_fwd_split_kv_kernel` (src/flag_attn/split_kv.py:14-160) and `_fwd_combine_kv_splits`
// (split_kv.py:162-227).  The split kernel is the decode core of decode.hpp over a dense K/V
// stream: a workgroup takes one (batch, kv head, split) and up to 16 of the G * M query rows that
// share that kv head, so the keys and values of a split are read once for the whole GQA group.
// Partial outputs are fp16 whatever the input dtype, as in the reference (flash.py:96); a split
// that holds no visible key for a row stores 0 and a log-normalizer of -inf, and the merge weights
// by select so that such splits drop out instead of producing NaN.  A NaN in a split's row sum goes to both and
// through the merge into the result.
#include "decode.hpp"
#include "params.hpp"

namespace fa {

// UNIFORM: rows less than 64 MiB apart, so that the rows of a load instruction are 32-bit offsets from one address.
template <class T, int D, bool UNIFORM>
struct DenseSrc {
  static constexpr bool kUniform = UNIFORM;
  const T* kb;
  const T* vb;
  int64_t k_st, v_st;
  struct Ids {};
  FA_DEVICE void lookup(Ids&, int, int, int) const {}
  static constexpr int RPI = DecCfg<T, D>::RPI;
  FA_DEVICE void resolve(Ids&, int, int) const {}
  FA_DEVICE const T* k_base(const Ids&, int i, int n0) const { return kb + (int64_t)n0 * k_st + i * (RPI * k_st); }
  FA_DEVICE const T* v_base(const Ids&, int i, int n0) const { return vb + (int64_t)n0 * v_st + i * (RPI * v_st); }
  FA_DEVICE const T* k_row(const Ids&, int, int n) const { return kb + (int64_t)n * k_st; }
  FA_DEVICE const T* v_row(const Ids&, int, int n) const { return vb + (int64_t)n * v_st; }
  FA_DEVICE uint32_t k_stride() const { return (uint32_t)k_st * (uint32_t)sizeof(T); }
  FA_DEVICE uint32_t v_stride() const { return (uint32_t)v_st * (uint32_t)sizeof(T); }
};

template <class T, int D, bool UNIFORM>
FA_KERNEL void FA_LAUNCH_BOUNDS2(kThreads, 2) fa_splitkv_kernel(SplitParams p) {
  using C = DecCfg<T, D>;
  FA_LDS_DECL(smem);
  const int tid = hw::thread_id(), lane = tid & 63, li = lane & 15;
  const int rb = hw::block_x(), split = hw::block_y();
  const int batch = hw::block_z() / (p.H / p.group), hk = hw::block_z() % (p.H / p.group);
  const int M = p.M, N = p.N, pseq = N - M;
  const int rows = p.group * M;

  DenseSrc<T, D, UNIFORM> src;
  src.kb = (const T*)p.k.ptr + batch * p.k.sb + hk * p.k.sh;
  src.vb = (const T*)p.v.ptr + batch * p.v.sb + hk * p.v.sh;
  src.k_st = p.k.st;
  src.v_st = p.v.st;

  // this lane's query row: rho = g * M + m
  const int rho = rb * 16 + li;
  const T* q_row = nullptr;
  int lane_limit = 0;
  if (rho < rows) {
    const int g = rho / M, m = rho % M;
    q_row = (const T*)p.q.ptr + batch * p.q.sb + (hk * p.group + g) * p.q.sh + (int64_t)m * p.q.st;
    lane_limit = p.causal ? imin(N, m + pseq + 1) : N;
  }
  const int n_begin = split * p.split_size;
  const int n_end = imin(N, n_begin + p.split_size);

  DecodeOut<D> res;
  decode_block<T, D>(src, q_row, imin(16, rows - rb * 16), n_begin, n_end, lane_limit, p.sm_scale * kLog2e, smem, res);

  const int out_tid = thread_for_output();
#pragma unroll
  for (int e = 0; e < DecodeOut<D>::kPerThread; ++e) {
    const int idx = out_tid + e * kThreads;
    const int row = idx / D, d = idx % D;
    const int r = rb * 16 + row;
    if (r < rows) {
      const int g = r / M, m = r % M;
      const int64_t slot = (((int64_t)batch * p.H + hk * p.group + g) * p.num_splits + split) * M + m;
      const bool empty = res.row_sum[e] == 0.f;
      ((hw::half_t*)p.part_o)[slot * D + d] = (hw::half_t)(empty ? 0.f : res.o[e] / res.row_sum[e]);
      if (d == 0)
        p.part_lse[slot] = empty ? neg_inf() : res.row_max[e] * p.sm_scale + hw::log_nat(res.row_sum[e]);
    }
  }
}

// Merge of the pieces of one row: 8 output elements per thread.  The kernel is a chain of memory latencies, so its
// loads are issued at once: the log-normalizer and output of BATCH pieces together, and with GROUPS > 1 the pieces are
// dealt to as many groups of lanes, which merge through lane exchanges (a group is a row's D / 8 lanes, a wavefront
// holds one row).  One row of 32 pieces took 6.1 us as a serial loop over batches of four and takes 3.0.  Up to 8 pieces
// a thread takes them all (2.3 us), and a wavefront holds 64 / (D / 8) rows, which is what the many rows of a prefill
// chunk want.
template <class T, int D, int BATCH, bool SPREAD>
struct CombineCfg {
  static constexpr int LANES = D / 8;
  static constexpr int GROUPS = SPREAD ? 64 / LANES : 1;
  static constexpr int ROWS = kThreads / (LANES * GROUPS);
};
template <class T, int D, int BATCH, bool SPREAD, class P>   // P: type of the partial outputs, fp16 or float
FA_KERNEL void FA_LAUNCH_BOUNDS(kThreads) fa_combine_kernel(CombineParams p) {
  constexpr int WORDS = (int)sizeof(P) / 2;                  // 16-byte loads for the 8 elements
  using C = CombineCfg<T, D, BATCH, SPREAD>;
  const int tid = hw::thread_id(), group = tid / C::LANES % C::GROUPS;
  const int64_t total_rows = (int64_t)p.B * p.H * p.M;
  const int64_t my_row = (int64_t)hw::block_x() * C::ROWS + tid / (C::LANES * C::GROUPS);  // over B * H * M
  const int64_t row = my_row < total_rows ? my_row : total_rows - 1;
  const int col = (tid % C::LANES) * 8;
  const int m = (int)(row % p.M);
  const int64_t bh = row / p.M;
  const int S = p.num_splits;
  const float* ls = p.part_lse + bh * S * p.M + m;  // stride M between splits
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  float z = 0.f, top = neg_inf();
  auto raise = [&](float t) {   // to the reference maximum t >= top
    const float old = top > neg_inf() ? hw::exp2_fast((top - t) * kLog2e) : 0.f;
    z *= old;
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] *= old;
    top = t;
  };
  for (int s0 = group * BATCH; s0 < S; s0 += C::GROUPS * BATCH) {
    float l[BATCH];
    u32x4 raw[BATCH][WORDS];
#pragma unroll
    for (int u = 0; u < BATCH; ++u) {
      const int s = imin(s0 + u, S - 1);
      l[u] = ls[(int64_t)s * p.M];
      const u32x4* part = (const u32x4*)((const P*)p.part_o + ((bh * S + s) * p.M + m) * D + col);
#pragma unroll
      for (int w = 0; w < WORDS; ++w) raw[u][w] = part[w];
    }
    float t = top;
#pragma unroll
    for (int u = 0; u < BATCH; ++u) t = fmaxf(t, l[u]);
    raise(t);
#pragma unroll
    for (int u = 0; u < BATCH; ++u) {
      if (s0 + u >= S || l[u] == neg_inf()) continue;  // past the end, or a split without a visible key
      const float wgt = hw::exp2_fast((l[u] - top) * kLog2e);
      z += wgt;
      if constexpr (WORDS == 2) {
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] += wgt * __builtin_bit_cast(float, (uint32_t)raw[u][e / 4][e % 4]);
      } else {
        auto v = hw::as_v8<hw::half_t>(raw[u][0]);
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] += wgt * (float)v[e];
      }
    }
  }
  if constexpr (C::GROUPS > 1) {
    float t = top;
#pragma unroll
    for (int x = C::LANES; x < 64; x <<= 1) t = fmaxf(t, hw::shfl_xor(t, x));
    raise(t);
#pragma unroll
    for (int x = C::LANES; x < 64; x <<= 1) {
      z += hw::shfl_xor(z, x);
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] += hw::shfl_xor(acc[e], x);
    }
    if (group > 0) return;
  }
  if (my_row >= total_rows) return;
  const float inv = z == 0.f ? 0.f : 1.f / z;   // z is NaN where a piece's log-normalizer is
  const int b = (int)(bh / p.H), h = (int)(bh % p.H);
  T* o = (T*)p.o.ptr + b * p.o.sb + h * p.o.sh + (int64_t)m * p.o.st + col;
  u32x4 w;
#pragma unroll
  for (int e = 0; e < 4; ++e)
    w[e] = (uint32_t)hw::bits16<T>(acc[2 * e] * inv) | ((uint32_t)hw::bits16<T>(acc[2 * e + 1] * inv) << 16);
  *(u32x4*)o = w;
  if (col == 0) p.lse[row] = z == 0.f ? neg_inf() : top + hw::log_nat(z);
}

template <class T, bool UNIFORM>
static int launch_split(const SplitParams& p, hipStream_t stream) {
  const int rows = p.group * p.M;
  dim3 grid((rows + 15) / 16, p.num_splits, p.B * (p.H / p.group));
  switch (p.D) {
    case 16: return launch(fa_splitkv_kernel<T, 16, UNIFORM>, grid, DecCfg<T, 16>::LDS_BYTES, stream, p);
    case 32: return launch(fa_splitkv_kernel<T, 32, UNIFORM>, grid, DecCfg<T, 32>::LDS_BYTES, stream, p);
    case 64: return launch(fa_splitkv_kernel<T, 64, UNIFORM>, grid, DecCfg<T, 64>::LDS_BYTES, stream, p);
    case 128: return launch(fa_splitkv_kernel<T, 128, UNIFORM>, grid, DecCfg<T, 128>::LDS_BYTES, stream, p);
  }
  return kUnsupported;
}

int run_splitkv(const SplitParams& p, hipStream_t stream) {
  if (p.B <= 0 || p.H <= 0 || p.M <= 0 || p.N <= 0 || p.group <= 0 || p.num_splits <= 0 || p.split_size <= 0)
    return kBadArgument;
  if ((int64_t)p.num_splits * p.split_size < p.N) return kBadArgument;
  if (splitkv_wide_applies(p)) return run_splitkv_wide(p, stream);   // many query rows: 256-row tiles
  const bool uniform = p.k.st < (1 << 25) && p.v.st < (1 << 25);
  if (p.dtype == kDtypeF16) return uniform ? launch_split<hw::half_t, true>(p, stream) : launch_split<hw::half_t, false>(p, stream);
  if (p.dtype == kDtypeBF16) return uniform ? launch_split<hw::bf16_t, true>(p, stream) : launch_split<hw::bf16_t, false>(p, stream);
  return kUnsupported;
}

template <class T, int D, class P>
static int launch_combine_as(const CombineParams& p, hipStream_t stream) {
  const int64_t total = (int64_t)p.B * p.H * p.M;
  auto go = [&](auto kern, auto cfg) {
    using C = decltype(cfg);
    return launch(kern, dim3((unsigned)((total + C::ROWS - 1) / C::ROWS)), 0, stream, p);
  };
  if (p.num_splits <= 4) return go(fa_combine_kernel<T, D, 4, false, P>, CombineCfg<T, D, 4, false>{});
  if (p.num_splits <= 8) return go(fa_combine_kernel<T, D, 8, false, P>, CombineCfg<T, D, 8, false>{});
  return go(fa_combine_kernel<T, D, 8, true, P>, CombineCfg<T, D, 8, true>{});
}
template <class T, int D>
static int launch_combine_d(const CombineParams& p, hipStream_t stream) {
  return p.f32 ? launch_combine_as<T, D, float>(p, stream) : launch_combine_as<T, D, hw::half_t>(p, stream);
}

template <class T>
static int launch_combine(const CombineParams& p, hipStream_t stream) {
  switch (p.D) {
    case 16: return launch_combine_d<T, 16>(p, stream);
    case 32: return launch_combine_d<T, 32>(p, stream);
    case 64: return launch_combine_d<T, 64>(p, stream);
    case 128: return launch_combine_d<T, 128>(p, stream);
  }
  return kUnsupported;
}

int run_combine(const CombineParams& p, hipStream_t stream) {
  if (p.B <= 0 || p.H <= 0 || p.M <= 0 || p.num_splits <= 0) return kBadArgument;
  if (p.dtype == kDtypeF16) return launch_combine<hw::half_t>(p, stream);
  if (p.dtype == kDtypeBF16) return launch_combine<hw::bf16_t>(p, stream);
  return kUnsupported;
}

}  // namespace fa
