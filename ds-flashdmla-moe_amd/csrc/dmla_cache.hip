// The two ends of paged split-KV decoding that are not attention:
//   * the paged latent-cache append (the producer of the [num_pages, 64, 576] pages that
//     dmla_decode_paged reads through the block table);
//   * the split-KV log-sum-exp combine, also usable on its own (e.g. to merge partials that
//     several devices computed over disjoint page ranges of one context).
// Neither has a reference counterpart: the reference has no paged decode (benchmark config 3).
#include <type_traits>

#include "dmla_common.h"
#include "dmla_host.h"

namespace dmla {

// ---- split-KV combine --------------------------------------------------------------------
//   o = sum_s w_s o_s / sum_s w_s, w_s = exp(lse_s - max_s lse_s), lse = max + log(sum w)
// over the first n splits of a (sequence, head) pair; no finite lse leaves o = 0 and lse = -inf
// (max of the inputs); a NaN lse makes o and lse NaN.  A split with lse = -inf is skipped whatever
// its o slot holds.  kW waves share a pair: wave w adds the splits w, w + kW, .. in that order and
// the kW sums meet in LDS, added in wave order, so the result does not depend on timing.
// Bound: HBM latency.  A lane holds 16 bytes of a partial row, so one load instruction takes 1 KB
// (a whole bf16 row), and kBatch rows are in flight per wave; the first batch goes out before the
// lse values have arrived.  One wave per pair adding 79 splits one load at a time took 72 us at one
// sequence of 5000 tokens and 128 heads (11.6 MB of partials); four waves and batches of 8 took
// the decode call there from 93.4 to 28.1 us, and from 52.4 to 36.4 us at 16 sequences x 16 heads
// (~17 splits each); at 64 sequences x 128 heads (3 splits) 115.4 -> 113.4 us.
constexpr int kCombineFew = 4;     // splits of the usual large batch: one batch of 4 rows covers them
constexpr int kCombineBatch = 8;   // rows in flight per wave otherwise

template <typename T>
struct PartVec {
  static constexpr int kN = 16 / (int)sizeof(T);   // elements of one 16-byte load
  T v[kN];
};
template <typename T>
__device__ __forceinline__ PartVec<T> load_part(const T* p) {
  return __builtin_bit_cast(PartVec<T>, *reinterpret_cast<const f32x4*>(p));
}

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  return v;
}
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) v += __shfl_xor(v, o, 64);
  return v;
}

template <typename T, int kW, int kBatch>
__device__ __forceinline__ void combine_pair(const CombineArgs& a, const T* part, int b, int h, int n, int64_t s0,
                                             int lane, int w, DMLA_LDS float* xch) {
  constexpr int kN = PartVec<T>::kN;
  constexpr int kCols = 64 * kN;   // columns of one pass
  const int64_t lbase = (a.split_base != nullptr ? s0 * a.lse_ss : (int64_t)b * a.lse_sb) + (int64_t)h * a.lse_sh;
  const T* rows = part + (a.split_base != nullptr ? s0 * a.po_ss : (int64_t)b * a.po_sb) + (int64_t)h * a.po_sh;
  bf16* orow = a.o + (int64_t)b * a.o_sb + (int64_t)h * a.o_sh;
  auto lse_chunk = [&](int c) { return c + lane < n ? a.part_lse[lbase + (int64_t)(c + lane) * a.lse_ss] : kNegInf; };
  PartVec<T> x[kBatch];
  // Rows w + kW u of the batch at s (wave-uniform); rows past n and columns past d read row 0 or
  // column 0 instead and are not used.
  auto load_batch = [&](int s, int cc) {
#pragma unroll
    for (int u = 0; u < kBatch; ++u) x[u] = load_part(rows + (int64_t)(s + kW * u < n ? s + kW * u : 0) * a.po_ss + cc);
  };
  const float lv0 = lse_chunk(0);
  if (n > 0) load_batch(w, kN * lane < a.d ? kN * lane : 0);
  float mx = lv0;
  bool nan_in = lv0 != lv0;   // a NaN lse (e.g. a split that met an invalid page) poisons the pair
  for (int c = 64; c < n; c += 64) {
    const float lv = lse_chunk(c);
    nan_in = nan_in || lv != lv;
    mx = fmaxf(mx, lv);
  }
  if (__any(nan_in)) {
    const bf16 nb = (bf16)__builtin_nanf("");
    for (int col = 4 * (lane + 64 * w); col < a.d; col += 256 * kW)
      *reinterpret_cast<bf16x4*>(orow + col) = bf16x4{nb, nb, nb, nb};
    if (lane == 0 && w == 0 && a.lse != nullptr) a.lse[(int64_t)b * a.H + h] = __builtin_nanf("");
    return;
  }
  mx = wave_max(mx);
  const float mref = mx == kNegInf ? 0.f : mx;
  float wsum = __expf(lv0 - mref);
  for (int c = 64; c < n; c += 64) wsum += __expf(lse_chunk(c) - mref);
  wsum = wave_sum(wsum);
  const float inv = wsum > 0.f ? 1.f / wsum : 0.f;
  for (int col0 = 0; col0 < a.d; col0 += kCols) {
    const int col = col0 + kN * lane, cc = col < a.d ? col : 0;
    if (col0 > 0 && n > 0) load_batch(w, cc);
    float acc[kN];
#pragma unroll
    for (int e = 0; e < kN; ++e) acc[e] = 0.f;
    for (int c = 0; c < n; c += 64) {
      const float lv = c == 0 ? lv0 : lse_chunk(c);
      const float wl = __expf(lv - mref) * inv;
      const uint64_t live = __ballot(lv != kNegInf);
      for (int s = c + w; s < min(n, c + 64); s += kW * kBatch) {
        if (s != w) load_batch(s, cc);
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
          const int i = s - c + kW * u;
          if (i >= 64 || !((live >> i) & 1)) continue;   // live holds no bit past n
          const float ws = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, wl), i));
#pragma unroll
          for (int e = 0; e < kN; ++e) acc[e] += ws * (float)x[u].v[e];
        }
      }
    }
    if constexpr (kW == 1) {
      if (col < a.d) {
#pragma unroll
        for (int q = 0; q < kN / 4; ++q) {
          bf16x4 v;
          v[0] = (bf16)acc[4 * q]; v[1] = (bf16)acc[4 * q + 1]; v[2] = (bf16)acc[4 * q + 2]; v[3] = (bf16)acc[4 * q + 3];
          *reinterpret_cast<bf16x4*>(orow + col + 4 * q) = v;
        }
      }
    } else {
#pragma unroll
      for (int q = 0; q < kN / 4; ++q)
        *reinterpret_cast<DMLA_LDS f32x4*>(xch + w * kCols + kN * lane + 4 * q) =
            f32x4{acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
      __syncthreads();
      const int t = 64 * w + lane;
      if (4 * t < kCols && col0 + 4 * t < a.d) {
        f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < kW; ++j) v += *reinterpret_cast<const DMLA_LDS f32x4*>(xch + j * kCols + 4 * t);
        bf16x4 r;
        r[0] = (bf16)v[0]; r[1] = (bf16)v[1]; r[2] = (bf16)v[2]; r[3] = (bf16)v[3];
        *reinterpret_cast<bf16x4*>(orow + col0 + 4 * t) = r;
      }
      __syncthreads();   // the sums are read out before the next pass writes its own
    }
  }
  if (lane == 0 && w == 0 && a.lse != nullptr) a.lse[(int64_t)b * a.H + h] = wsum > 0.f ? mref + __logf(wsum) : mx;
}

// kPlan: the decode case, split_base and num_splits both given, so that both loads go out
// together (one round trip before the partials' loads, not one per null check).  kW: waves per
// pair, 1 (four pairs per 256-thread block) or 4.
template <bool kPlan, int kW>
__global__ void __launch_bounds__(256) lse_combine_kernel(CombineArgs a) {
  __shared__ f32x4 xch[kW == 1 ? 1 : kW * 64 * 2];   // kW rows of up to 512 sums, as 16-byte pieces
  const int lane = threadIdx.x & 63;
  const int wave = uniform(threadIdx.x >> 6);
  // 32-bit index math: the launcher checks B * H < 2^31
  const unsigned pair = kW == 1 ? blockIdx.x * 4u + (unsigned)wave : blockIdx.x;
  if (pair >= (unsigned)(a.B * a.H)) return;
  const int b = (int)(pair / (unsigned)a.H), h = (int)(pair - (unsigned)b * (unsigned)a.H);
  int n = a.max_splits;
  int64_t s0 = 0;
  if constexpr (kPlan) {
    int sb = a.split_base[b], ns = a.num_splits[b];
    asm volatile("" : "+s"(sb), "+s"(ns));   // both loads issued before anything waits on either
    s0 = sb;
    n = min(max(ns, 0), a.max_splits);
  } else {
    if (a.split_base != nullptr) s0 = a.split_base[b];
    if (a.num_splits != nullptr) n = min(max(a.num_splits[b], 0), a.max_splits);
  }
  if (a.skip_single && n == 1) return;   // the decode kernel already wrote such rows itself
  DMLA_LDS float* x = (DMLA_LDS float*)xch;
  const int w = kW == 1 ? 0 : wave;
  auto run = [&](const auto* part) {
    using T = std::remove_const_t<std::remove_pointer_t<decltype(part)>>;
    if (kW == 1 && n <= kCombineFew) combine_pair<T, kW, kCombineFew>(a, part, b, h, n, s0, lane, w, x);
    else combine_pair<T, kW, kCombineBatch>(a, part, b, h, n, s0, lane, w, x);
  };
  if (a.part_o16 != nullptr) run(a.part_o16);
  else run(a.part_o);
}

int launch_lse_combine(const CombineArgs& a, hipStream_t stream, const char* what) {
  if (a.B == 0 || a.H == 0) return DMLA_OK;
  const int64_t pairs = (int64_t)a.B * a.H;
  if (pairs >= ((int64_t)1 << 31)) return fail(DMLA_ERR_UNSUPPORTED, "%s: B * H must be below 2^31", what);
  // Four waves per pair where the pairs alone leave most of the chip's 8192 wave slots empty and a
  // pair has more than a handful of splits.
  const bool wide = pairs <= 2048 && a.mean_splits > kCombineFew;
  const bool plan = a.split_base != nullptr && a.num_splits != nullptr;
  const dim3 grid((unsigned)(wide ? pairs : (pairs + 3) / 4));
  const auto kernel = wide ? (plan ? lse_combine_kernel<true, 4> : lse_combine_kernel<false, 4>)
                           : (plan ? lse_combine_kernel<true, 1> : lse_combine_kernel<false, 1>);
  hipLaunchKernelGGL(kernel, grid, dim3(256), 0, stream, a);
  return check_launch(what);
}

namespace {

// ---- paged append ------------------------------------------------------------------------
struct AppendArgs {
  bf16* pool;
  const int32_t* block_table;
  const int32_t* seqlens;
  const int32_t* new_lens;   // nullable: every sequence appends n_new rows
  const bf16* new_kv;
  int32_t* bad;              // nullable: set to 1 when a row's page slot or index is out of range
  int64_t pool_sp, pool_ss, bt_sb, nk_sb, nk_ss;
  int B, n_new, chunks;      // chunks = d / 8 (16-byte pieces per row)
  int page_size, num_pages, max_pages;
};

// One 16-byte piece per thread and step, consecutive threads on consecutive pieces of a row.
__global__ void __launch_bounds__(256) kv_append_kernel(AppendArgs a) {
  const int64_t total = (int64_t)a.B * a.n_new * a.chunks;
  for (int64_t u = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; u < total; u += (int64_t)gridDim.x * blockDim.x) {
    const int c = (int)(u % a.chunks);
    const int64_t bt = u / a.chunks;
    const int t = (int)(bt % a.n_new);
    const int b = (int)(bt / a.n_new);
    const int n = a.new_lens ? min(max(a.new_lens[b], 0), a.n_new) : a.n_new;
    if (t >= n) continue;
    const int64_t pos = (int64_t)max(a.seqlens[b], 0) + t;
    const int64_t slot = pos / a.page_size;
    const int page = slot < a.max_pages ? a.block_table[b * a.bt_sb + slot] : -1;
    if (page < 0 || page >= a.num_pages) {
      if (a.bad != nullptr) a.bad[0] = 1;
      continue;
    }
    const bf16x8 v = *reinterpret_cast<const bf16x8*>(a.new_kv + b * a.nk_sb + t * a.nk_ss + 8 * c);
    *reinterpret_cast<bf16x8*>(a.pool + page * a.pool_sp + (pos % a.page_size) * a.pool_ss + 8 * c) = v;
  }
}

}  // namespace
}  // namespace dmla

using namespace dmla;

extern "C" int dmla_kv_append(void* kv_pool, const int32_t* block_table, const int32_t* cache_seqlens,
                              const int32_t* new_lens, const void* new_kv, int32_t* bad_index_flag, int64_t B,
                              int64_t n_new, int64_t d, int64_t page_size, int64_t num_pages,
                              int64_t max_pages_per_seq, int64_t kv_sp, int64_t kv_ss, int64_t bt_sb,
                              int64_t nk_sb, int64_t nk_ss, dmla_stream_t stream) {
  clear_error();
  if (!kv_pool || !block_table || !cache_seqlens || !new_kv)
    return fail(DMLA_ERR_INVALID_ARG, "dmla_kv_append: null pointer argument");
  if (B < 0 || n_new < 0 || d <= 0 || page_size <= 0 || num_pages < 0 || max_pages_per_seq < 0)
    return fail(DMLA_ERR_INVALID_ARG, "dmla_kv_append: negative or zero size");
  if (d % 8 != 0) return fail(DMLA_ERR_UNSUPPORTED, "dmla_kv_append: d must be a multiple of 8 (got %lld)", (long long)d);
  if (!aligned16(kv_pool) || !aligned16(new_kv))
    return fail(DMLA_ERR_INVALID_ARG, "dmla_kv_append: kv_pool and new_kv must be 16-byte aligned");
  if (!mult8(kv_sp) || !mult8(kv_ss) || !mult8(nk_sb) || !mult8(nk_ss) || kv_ss < d || kv_sp < page_size * kv_ss)
    return fail(DMLA_ERR_INVALID_ARG, "dmla_kv_append: strides must be multiples of 8 and cover a row / page");
  if (bt_sb < max_pages_per_seq)
    return fail(DMLA_ERR_INVALID_ARG, "dmla_kv_append: block_table row stride < max_pages_per_seq");
  if (B > ((int64_t)1 << 24) || n_new > ((int64_t)1 << 24) || num_pages > 0x7fffffff ||
      max_pages_per_seq > ((int64_t)1 << 24) || d / 8 > 0x7fffffff)
    return fail(DMLA_ERR_UNSUPPORTED, "dmla_kv_append: size too large");
  if (B == 0 || n_new == 0) return DMLA_OK;
  AppendArgs a = {};
  a.pool = static_cast<bf16*>(kv_pool);
  a.block_table = block_table;
  a.seqlens = cache_seqlens;
  a.new_lens = new_lens;
  a.new_kv = static_cast<const bf16*>(new_kv);
  a.bad = bad_index_flag;
  a.pool_sp = kv_sp; a.pool_ss = kv_ss; a.bt_sb = bt_sb; a.nk_sb = nk_sb; a.nk_ss = nk_ss;
  a.B = (int)B; a.n_new = (int)n_new; a.chunks = (int)(d / 8);
  a.page_size = (int)page_size; a.num_pages = (int)num_pages; a.max_pages = (int)max_pages_per_seq;
  const int64_t total = B * n_new * (d / 8);
  const int64_t blocks = std::min<int64_t>((total + 255) / 256, (int64_t)device_cu_count() * 16);
  hipLaunchKernelGGL(kv_append_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, a);
  return check_launch("dmla_kv_append");
}

extern "C" int dmla_lse_combine(const float* part_o, const float* part_lse, const int32_t* num_splits, void* o,
                                float* lse, int64_t B, int64_t H, int64_t max_splits, int64_t d, int64_t po_sb,
                                int64_t po_ss, int64_t po_sh, int64_t lse_sb, int64_t lse_ss, int64_t lse_sh,
                                int64_t o_sb, int64_t o_sh, dmla_stream_t stream) {
  clear_error();
  if (!part_o || !part_lse || !o) return fail(DMLA_ERR_INVALID_ARG, "dmla_lse_combine: null pointer argument");
  if (B < 0 || H < 0 || max_splits <= 0 || d <= 0)
    return fail(DMLA_ERR_INVALID_ARG, "dmla_lse_combine: bad size");
  if (d % 4 != 0) return fail(DMLA_ERR_UNSUPPORTED, "dmla_lse_combine: d must be a multiple of 4");
  if (!aligned16(part_o) || (reinterpret_cast<uintptr_t>(o) & 7u) != 0)
    return fail(DMLA_ERR_INVALID_ARG, "dmla_lse_combine: part_o must be 16-byte and o 8-byte aligned");
  if (po_sb % 4 || po_ss % 4 || po_sh % 4 || o_sb % 4 || o_sh % 4)
    return fail(DMLA_ERR_INVALID_ARG, "dmla_lse_combine: part_o / o strides must be multiples of 4 elements");
  if (B * H > 0x7fffffff || max_splits > 0x7fffffff || d > 0x7fffffff)
    return fail(DMLA_ERR_UNSUPPORTED, "dmla_lse_combine: size too large");
  CombineArgs a = {};
  a.part_o = part_o;
  a.part_lse = part_lse;
  a.num_splits = num_splits;
  a.o = static_cast<bf16*>(o);
  a.lse = lse;
  a.B = (int)B; a.H = (int)H; a.max_splits = (int)max_splits; a.d = (int)d;
  a.mean_splits = (int)max_splits;
  a.po_sb = po_sb; a.po_ss = po_ss; a.po_sh = po_sh;
  a.lse_sb = lse_sb; a.lse_ss = lse_ss; a.lse_sh = lse_sh;
  a.o_sb = o_sb; a.o_sh = o_sh;
  return launch_lse_combine(a, (hipStream_t)stream, "dmla_lse_combine");
}
