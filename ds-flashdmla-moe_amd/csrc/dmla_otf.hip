// On-the-fly DMLA forward for gfx950: the per-head latent projections K_lat = K WK and
// V_lat = V WV are computed inside the attention kernel (README.md:14, the on-the-fly mode of
// the absent csrc/attention/fa2_dmla_fwd.cu, README.md:45), then
//     O[b,h] = softmax(scale * Q[b,h] K_lat[b,h]^T (+ causal mask)) V_lat[b,h].
// Shapes: Q [B,H,Sq,64], K and V [B,Sk,H,128], WK and WV [H,128,64], O [B,H,Sq,64].
//
// Workgroup = 8 waves on 512 query rows of one (batch, head); wave w owns rows 64w .. +63
// (otf_fwd_short_kernel: fewer rows per workgroup, for short sequences).
// Key tiles of 64 keys flow through a one-barrier-per-tile pipeline:
//   * the raw K / V rows of tile t+2 are copied global -> LDS (direct copies, two stages);
//   * tile t+1 is projected on MFMA: waves 0-3 compute K_lat^T (16 latent dims each, WK^T in
//     registers), waves 4-7 compute V_lat (WV^T in registers), both written to LDS as fp16 --
//     once per key tile for all 512 rows, so the projection adds 1/4 to the attention MFMAs
//     (a 128-row tile would double them);
//   * tile t is attended: S^T = K_lat Q^T (Q in registers), P in the exp2 domain, O += P V_lat.
// Scores: Q stays in bf16 (exact) and K_lat, multiplied by scale log2(e), is stored as a bf16
// pair hi + lo (hi = bf16(c), lo = bf16(c - hi)), two bf16 MFMAs per k-step: the scores carry
// ~2^-17 relative error, where one fp16 rounding of K_lat (2^-12) moved the row statistics
// m, l by ~1.7e-3 at the benchmark's config 4.  (An fp16 pair does not work: most residuals
// are fp16 subnormals, which the fp16 MFMA loses.)  V_lat and P enter the PV product as fp16,
// rounded from fp32: 3 more significand bits than bf16, which keeps their rounding well inside
// the output tolerance even for rows that see only a few keys.  The score accumulators start
// at -m_ref, so the MFMA hands the softmax its exp2 arguments directly.
// Every MFMA operand read from LDS is a conflict-free 16-byte read: K_lat rows for S^T and a
// V_lat^T tile whose key order matches the C layout of S^T (so P needs no transposition).
//
// Softmax: in log2 units against a per-row reference max m_ref that only moves when a tile's
// max exceeds it by more than kSlack (p <= 2^kSlack in between); moving it rescales O and l.  The exact running max is tracked beside it for the m / l outputs, which
// follow the cache-latent forward's convention (natural-log units).
#include <type_traits>

#include "dmla_common.h"
#include "dmla_host.h"
#include "dmla_rules.h"

namespace dmla {
namespace {

constexpr int kDin = 128;          // raw K / V dims per head
constexpr int kDlat = 64;          // latent dims (Q, K_lat, V_lat, O)
constexpr int kOtfWaves = 8;
constexpr int kOtfThreads = 64 * kOtfWaves;
constexpr int kOtfRows = 64 * kOtfWaves;   // 512 query rows per workgroup
constexpr int kOtfKeys = 64;               // keys per tile
constexpr float kSlack = 8.0f;             // log2 slack of the reference max
// LDS: raw K / V stages (2 x 2 x 64 x 128 bf16), latent buffers (2 x [K_lat hi, V_lat^T, K_lat lo] of
// 64 x 64).  WK and WV pass through the latent buffers once, before the first tile.
constexpr int kWBytes = kDlat * kDin * 2;          // 16 KB
constexpr int kRawBytes = kOtfKeys * kDin * 2;     // 16 KB
constexpr int kLatBytes = kOtfKeys * kDlat * 2;    // 8 KB
constexpr int kRawOff = 0;                         // [stage][K, V]
constexpr int kLatOff = 4 * kRawBytes;             // [buffer][K_lat hi, V_lat^T, K_lat lo]
constexpr int kBufBytes = 3 * kLatBytes;
constexpr int kOtfLds = kLatOff + 2 * kBufBytes;   // 112 KB
static_assert(2 * kWBytes <= 2 * kBufBytes, "W fits in the latent buffers");

struct OtfParams {
  const bf16* q;
  const bf16* k;
  const bf16* v;
  const bf16* wk;
  const bf16* wv;
  bf16* o;
  float* m;
  float* l;
  int64_t q_sb, q_sh, q_ss;
  int64_t k_sb, k_ss, k_sh;
  int64_t v_sb, v_ss, v_sh;
  int64_t w_sh, w_si;          // WK / WV: head stride, row (input dim) stride; latent dims contiguous
  int64_t o_sb, o_sh, o_ss;
  int B, H, Sq, Sk, causal;
  float scale_log2;
  int n_qt;                    // row tiles per (batch, head)
  int o_rows16;                // o strides are multiples of 8 elements (16-byte stores)
};

// Raw tile layout: [key (64)][16 chunks of 16 B], physical chunk = c ^ (key & 15): 16 lanes
// reading one chunk of 16 consecutive keys hit 16 different bank groups.
__device__ __forceinline__ int raw_off(int key, int chunk) { return key * 256 + 16 * (chunk ^ (key & 15)); }
// Latent tiles (K_lat [key][64 dims] and V_lat^T [dim][64 key positions]): 128-byte rows,
// chunk c of row r at c ^ swz(r & 15) as in the cache-latent tiles.
__device__ __forceinline__ int lat_off(int row, int chunk) { return row * 128 + 16 * (chunk ^ swz(row & 15)); }

// WK[h] and WV[h] as they lie ([input (128)][64 latent dims], 128-byte rows) into the latent
// buffers, one copy per 8 rows: chunk c of input row i at c ^ (i & 7).
__device__ __forceinline__ void stage_w(const OtfParams& p, int h, unsigned lds_base, int wave, int lane) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int n = wave + 8 * j;
    const int i = 8 * (n & 15) + (lane >> 3);
    const bf16* w = (n < 16 ? p.wk : p.wv) + h * p.w_sh + i * p.w_si;
    dma16_addr(w + 8 * ((lane & 7) ^ (i & 7)), lds_base + kLatOff + n * 1024);
  }
}
// Eight inputs i0 .. i0 + 7 of latent dim d0 + (lane & 15), W^T as an MFMA operand, by two
// transposed reads (i0, d0 per group of 16 lanes).  Written out transposed with 2-byte LDS writes
// instead, W cost each workgroup 1.3 us more before its first tile (1 x 32 heads x 64: 9.6 -> 8.3 us).
__device__ __forceinline__ bf16x8 w_operand(const DMLA_LDS char* w, int i0, int d0, int lane) {
  const int e = (lane & 15) >> 2, q = lane & 3;
  auto at = [&](int i) {
    return reinterpret_cast<const DMLA_LDS bf16x4*>(w + i * 128 + 16 * ((d0 / 8 + (q >> 1)) ^ (i & 7)) + 8 * (q & 1));
  };
  return concat(lds_read_tr16(at(i0 + e)), lds_read_tr16(at(i0 + 4 + e)));
}

__global__ void __launch_bounds__(kOtfThreads, 1) otf_fwd_kernel(OtfParams p) {
  __shared__ __attribute__((aligned(1024))) char smem[kOtfLds];
  DMLA_LDS char* lds = (DMLA_LDS char*)smem;
  const int wave = uniform(threadIdx.x >> 6);
  const int lane = lane_id();
  const int l16 = lane & 15, g = lane >> 4;
  const int bh = (int)blockIdx.x % (p.B * p.H);
  const int qt = p.n_qt - 1 - (int)blockIdx.x / (p.B * p.H);   // heaviest (latest) tiles first
  const int b = bh / p.H, h = bh % p.H;
  const int off = p.Sk - p.Sq;
  const int row0 = qt * kOtfRows + 64 * wave;                  // this wave's first query row
  const int last_row = min(p.Sq, qt * kOtfRows + kOtfRows) - 1;
  const int key_end = p.causal ? min(p.Sk, last_row + off + 1) : p.Sk;
  const int n_t = key_end > 0 ? (key_end + kOtfKeys - 1) / kOtfKeys : 0;
  const unsigned lds_base = lds_addr(lds);

  stage_w(p, h, lds_base, wave, lane);

  // ---- raw K / V tile copies: 16 per tensor (4 keys x 256 B each), 4 per wave ----
  // Wave w copies tensor x = w / 4 (K, then V): copy c covers keys 4n .. 4n+3 with
  // n = 4 (w % 4) + c; lane l -> key 4n + l/16 (= 16 (w % 4) + 4c + g), physical chunk
  // l16 ^ (key % 16) = l16 ^ (4c + g).  The address is a wave-uniform base (the tile's first key
  // plus 4c rows, scalar arithmetic) and a lane offset that does not change from tile to tile
  // (row strides < 2^24 elements keep it below 2^31 bytes).  Computed per copy from 64-bit
  // strides instead, the addresses had cost ~30 quarter-rate integer multiplies per wave and
  // tile.  Only a tile that reaches past Sk takes per-lane addresses, clamped to the last key
  // (those keys are masked).
  const int xw = wave >> 2;
  const bf16* xbase = xw == 0 ? p.k + b * p.k_sb + h * p.k_sh : p.v + b * p.v_sb + h * p.v_sh;
  const int64_t xss = xw == 0 ? p.k_ss : p.v_ss;
  const unsigned raw_lane = (unsigned)((16 * (wave & 3) + g) * xss * 2);
  auto stage_raw = [&](int t, int st) {
    const unsigned ldst = lds_base + kRawOff + (st * 2 + xw) * kRawBytes + (wave & 3) * 4 * 1024;
    if (t * kOtfKeys + kOtfKeys <= p.Sk) {
#pragma unroll
      for (int c = 0; c < 4; ++c)
        dma16(xbase + (int64_t)(t * kOtfKeys + 4 * c) * xss, raw_lane + 16u * (unsigned)(l16 ^ (4 * c + g)),
              ldst + c * 1024);
    } else {
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int key = 16 * (wave & 3) + 4 * c + g;
        const int gk = min(t * kOtfKeys + key, p.Sk - 1);
        dma16_addr(xbase + (int64_t)gk * xss + 8 * (l16 ^ (4 * c + g)), ldst + c * 1024);
      }
    }
  };
  if (n_t > 0) stage_raw(0, 0);
  if (n_t > 1) stage_raw(1, 1);

  // ---- Q rows of this wave as the B operand of S^T: qreg[rb][ks] = Q[row0 + 16 rb + l16][32 ks + 8 g ..]
  bf16x8 qreg[4][2];
#pragma unroll
  for (int rb = 0; rb < 4; ++rb) {
    const int r = min(row0 + 16 * rb + l16, p.Sq - 1);
    const bf16* qrow = p.q + b * p.q_sb + h * p.q_sh + (int64_t)r * p.q_ss + 8 * g;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      qreg[rb][ks] = *reinterpret_cast<const bf16x8*>(qrow + 32 * ks);
    }
  }
  wait_vmem();
  __syncthreads();   // W and raw tile 0 (and 1) landed

  // Projection operand of this wave: waves 0-3 hold WK^T rows 16 w .. +15 (A operand of
  // K_lat^T), waves 4-7 WV^T rows 16 (w-4) .. (B operand of V_lat); 4 k-steps of 32 input dims.
  const int pdb = wave & 3;
  const bool pk = wave < 4;
  bf16x8 wreg[4];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks)
    wreg[ks] = w_operand(lds + kLatOff + (pk ? 0 : kWBytes), 32 * ks + 8 * g, 16 * pdb, lane);
  // Every wave holds its operands before the latent buffers take the first tile (lgkmcnt(0): the
  // reads above are done).
  __builtin_amdgcn_s_waitcnt(0xc07f);
  __syncthreads();

  // Project tile t (raw stage st) into latent buffer lb.  One wave-uniform branch for the
  // whole projection (a select per MFMA compiles to a branch around every MFMA).
  auto project = [&](int st, int lb) {
    auto proj = [&](auto is_k) {
      constexpr bool kK = decltype(is_k)::value;
      const DMLA_LDS char* raw = lds + kRawOff + (st * 2 + (kK ? 0 : 1)) * kRawBytes;
      DMLA_LDS char* lat = lds + kLatOff + lb * kBufBytes + (kK ? 0 : kLatBytes);
      // The four key blocks' accumulations run interleaved (k-step outer), so consecutive MFMAs
      // are independent, and each k-step's raw reads go out one k-step ahead.  (Key block by key
      // block, every MFMA waited for the previous one's result and every read was awaited
      // right before its MFMA.)
      f32x4 cacc[4];
      bf16x8 xr[2][4];
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) {
        cacc[kb] = f32x4{0.f, 0.f, 0.f, 0.f};
        xr[0][kb] = *reinterpret_cast<const DMLA_LDS bf16x8*>(raw + raw_off(16 * kb + l16, g));
      }
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        if (ks + 1 < 4) {
#pragma unroll
          for (int kb = 0; kb < 4; ++kb)
            xr[(ks + 1) & 1][kb] = *reinterpret_cast<const DMLA_LDS bf16x8*>(raw + raw_off(16 * kb + l16, 4 * (ks + 1) + g));
        }
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) {
          if constexpr (kK) cacc[kb] = mfma_bf16(wreg[ks], xr[ks & 1][kb], cacc[kb]);   // K_lat^T[dim 16 pdb + 4g + i][key 16 kb + l16]
          else cacc[kb] = mfma_bf16(xr[ks & 1][kb], wreg[ks], cacc[kb]);                // V_lat[key 16 kb + 4g + i][dim 16 pdb + l16]
        }
      }
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) {
        f32x4 c = cacc[kb];
        if constexpr (kK) {
          // K_lat is stored pre-multiplied by scale log2(e), so that scores come out of the MFMA
          // in log2 units, as hi + lo with hi = bf16(c) and lo = bf16(c - hi):
          // K_lat[key 16 kb + l16][dims 16 pdb + 4g .. +3]
          c *= p.scale_log2;
          bf16x4 hi, lo;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            hi[i] = (bf16)c[i];
            lo[i] = (bf16)(c[i] - (float)hi[i]);
          }
          const int key = 16 * kb + l16;
          const int o = lat_off(key, 2 * pdb + (g >> 1)) + 8 * (g & 1);
          *reinterpret_cast<DMLA_LDS bf16x4*>(lat + o) = hi;
          *reinterpret_cast<DMLA_LDS bf16x4*>(lat + 2 * kLatBytes + o) = lo;
        } else {
          f16x4 v;
          v[0] = (_Float16)c[0]; v[1] = (_Float16)c[1]; v[2] = (_Float16)c[2]; v[3] = (_Float16)c[3];
          // V_lat^T[dim 16 pdb + l16][position]: keys 4g + i of key block kb sit at positions
          // 32 (kb/2) + 8 g + 4 (kb&1) + i, the key order of the P operand (S^T C layout).
          const int dim = 16 * pdb + l16;
          *reinterpret_cast<DMLA_LDS f16x4*>(lat + lat_off(dim, 4 * (kb >> 1) + g) + 8 * (kb & 1)) = v;
        }
      }
    };
    if (pk) proj(std::true_type{});
    else proj(std::false_type{});
  };

  f32x4 oacc[4][4];   // O[row0 + 16 rb + 4 g + i][16 db + l16]
#pragma unroll
  for (int rb = 0; rb < 4; ++rb)
#pragma unroll
    for (int db = 0; db < 4; ++db) oacc[rb][db] = f32x4{0.f, 0.f, 0.f, 0.f};
  float mref[4], mtrue[4], lsum[4];   // per own row 16 rb + l16 (log2 units; lsum lane-partial)
#pragma unroll
  for (int rb = 0; rb < 4; ++rb) {
    mref[rb] = kNegInf;
    mtrue[rb] = kNegInf;
    lsum[rb] = 0.f;
  }
  const int own_pos0 = row0 + l16;   // position of own row 16 rb + l16 is own_pos0 + 16 rb

  if (n_t > 0) project(0, 0);
  for (int t = 0; t < n_t; ++t) {
    wait_vmem();
    __syncthreads();   // latent tile t written, raw tile t+1 landed, raw stage t%2 and latent buffer (t+1)%2 free
    if (t + 1 < n_t) project((t + 1) & 1, (t + 1) & 1);
    // Tile t+2's raw copies go out after the projection: issued straight after the barrier, the
    // 32 KB of copies of all waves queue in the CU's vector-memory path ahead of the work.
    if (t + 2 < n_t) stage_raw(t + 2, t & 1);

    const DMLA_LDS char* klat = lds + kLatOff + (t & 1) * kBufBytes;
    const DMLA_LDS char* vlat = klat + kLatBytes;
    const DMLA_LDS char* klo = klat + 2 * kLatBytes;
    // x[kb][rb] = S^T in log2 units minus the row's reference: keys 16 kb + 4g + i, row 16 rb +
    // l16.  The MFMA accumulators start at -m_ref (0 while a row has no reference), so x is the
    // exp2 argument as it leaves the matrix core.
    float nmr[4];
#pragma unroll
    for (int rb = 0; rb < 4; ++rb) nmr[rb] = mref[rb] == kNegInf ? 0.f : -mref[rb];
    f32x4 s[4][4];
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      const int o0 = lat_off(16 * kb + l16, g), o1 = lat_off(16 * kb + l16, 4 + g);
      const bf16x8 k0 = *reinterpret_cast<const DMLA_LDS bf16x8*>(klat + o0);
      const bf16x8 k1 = *reinterpret_cast<const DMLA_LDS bf16x8*>(klat + o1);
      const bf16x8 k0l = *reinterpret_cast<const DMLA_LDS bf16x8*>(klo + o0);
      const bf16x8 k1l = *reinterpret_cast<const DMLA_LDS bf16x8*>(klo + o1);
#pragma unroll
      for (int rb = 0; rb < 4; ++rb) {
        s[kb][rb] = mfma_bf16(k0l, qreg[rb][0], f32x4{nmr[rb], nmr[rb], nmr[rb], nmr[rb]});
        s[kb][rb] = mfma_bf16(k1l, qreg[rb][1], s[kb][rb]);
        s[kb][rb] = mfma_bf16(k0, qreg[rb][0], s[kb][rb]);
        s[kb][rb] = mfma_bf16(k1, qreg[rb][1], s[kb][rb]);
      }
    }
    // Only tiles that reach past some row's limit or past Sk are masked, in a block of their own.
    const int key0 = t * kOtfKeys;
    if (key0 + kOtfKeys > p.Sk || (p.causal && key0 + kOtfKeys - 1 > row0 + off)) {
#pragma unroll
      for (int rb = 0; rb < 4; ++rb) {
        const int lim = p.causal ? min(own_pos0 + 16 * rb + off, p.Sk - 1) : p.Sk - 1;
#pragma unroll
        for (int kb = 0; kb < 4; ++kb)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (key0 + 16 * kb + 4 * g + i > lim) s[kb][rb][i] = kNegInf;
      }
    }
    // Tile max per own row (lane-partial, log2 units), exact running max, and the slack test.
    bool raise = false;
#pragma unroll
    for (int rb = 0; rb < 4; ++rb) {
      float mx = kNegInf;
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
        mx = fmaxf(mx, fmaxf(fmaxf(s[kb][rb][0], s[kb][rb][1]), fmaxf(s[kb][rb][2], s[kb][rb][3])));
      mx -= nmr[rb];   // the tile's max score in log2 units
      mtrue[rb] = fmaxf(mtrue[rb], mx);
      raise |= mx > mref[rb] + kSlack;
    }
    if (__any(raise)) {
      // Move the reference to the exact row max so far; rescale l and the O rows.
#pragma unroll
      for (int rb = 0; rb < 4; ++rb) {
        const float mrow = group_max(mtrue[rb]);
        const float mnew = fmaxf(mref[rb], mrow);
        const float f = mnew == kNegInf ? 1.f : fast_exp2(mref[rb] - mnew);   // 0 when mref = -inf
        lsum[rb] *= f;
        mref[rb] = mnew;
        // this tile's arguments move to the new reference
        const float dn = (mnew == kNegInf ? 0.f : -mnew) - nmr[rb];
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) s[kb][rb] += dn;
        // O rows 16 rb + 4 g + i are own rows of lanes with l16 = 4 g + i.
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float fi = __shfl(f, 4 * g + i);
#pragma unroll
          for (int db = 0; db < 4; ++db) oacc[rb][db][i] *= fi;
        }
      }
    }
    // P = exp2(s scale - mref) (0 for masked keys and for rows without a finite reference yet).
    // The row sums add the fp16 P that the PV product multiplies, two per v_dot2c_f32_f16 (fp32
    // accumulation): half the instructions of one fp32 add per score.
    f16x8 pa[4][2];   // A operand of O += P V_lat: [rb][ks], keys of k-step ks in V_lat^T order
    const f16x2 ones = {(_Float16)1.f, (_Float16)1.f};
#pragma unroll
    for (int rb = 0; rb < 4; ++rb) {
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float e = fast_exp2(s[kb][rb][i]);
          pa[rb][kb >> 1][4 * (kb & 1) + i] = (_Float16)e;
        }
      }
      float ps = lsum[rb];
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          ps = __builtin_amdgcn_fdot2(f16x2{pa[rb][ks][2 * j], pa[rb][ks][2 * j + 1]}, ones, ps, false);
      lsum[rb] = ps;
    }
#pragma unroll
    for (int db = 0; db < 4; ++db) {
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        const f16x8 vb = *reinterpret_cast<const DMLA_LDS f16x8*>(vlat + lat_off(16 * db + l16, 4 * ks + g));
#pragma unroll
        for (int rb = 0; rb < 4; ++rb) oacc[rb][db] = mfma_f16(pa[rb][ks], vb, oacc[rb][db]);
      }
    }
  }

  // ---- epilogue: row sums, statistics, normalised O ----
#pragma unroll
  for (int rb = 0; rb < 4; ++rb) {
    const float ltot = group_sum(lsum[rb]);
    const float mrow = group_max(mtrue[rb]);
    const float inv = ltot > 0.f ? 1.f / ltot : 0.f;
    const int r = own_pos0 + 16 * rb;
    if (g == 0 && r < p.Sq && p.m) {
      const int64_t idx = ((int64_t)b * p.H + h) * p.Sq + r;
      const bool any = ltot > 0.f;
      p.m[idx] = any ? mrow * kLn2 : kNegInf;
      p.l[idx] = any ? ltot * fast_exp2(mref[rb] - mrow) : 0.f;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float fi = __shfl(inv, 4 * g + i);
      const int ro = row0 + 16 * rb + 4 * g + i;
      if (ro >= p.Sq) continue;
      bf16* orow = p.o + b * p.o_sb + h * p.o_sh + (int64_t)ro * p.o_ss + l16;
#pragma unroll
      for (int db = 0; db < 4; ++db) orow[16 * db] = (bf16)(oacc[rb][db][i] * fi);
    }
  }
}

// ---- short sequences ------------------------------------------------------------------------
// The kernel above needs 512-row tiles to spread the projection over; where these leave most CUs
// without a workgroup (32 heads of 500 rows: 32 workgroups of 8 serial tiles), this one runs 256 or
// 128 rows per workgroup on v_mfma_f32_32x32x16: a wave owns 32 query rows, and with kKS = 2 two
// waves share them, each taking every tile's keys of one half and the pair's results merged at the
// end.  Same tiles, stages, precision and softmax rules as above.  Bound: the latency of a tile's
// chain (projection, scores, softmax, PV).  At 1 x 32 heads x 500 rows the kernel takes
// 16.9 us with 128 rows per workgroup and 20.4 us with 256, against 35.8 us before (512 rows).
//
// LDS rows.  A 32x32 operand read (lane l: row l % 32, chunk 2 ks + l / 32 of 16 bytes) is served 16
// lanes at a time, the lanes with equal bit 5 and equal parity of bits 2-4: 16 rows whose low four
// bits all differ.
//  * Raw K / V tiles: raw_off, chunk c of row r at c ^ (r & 15): the 16 rows of a group take 16
//    different chunks, all 64 banks once.
//  * Latent tiles (K_lat [key][64 dims], V_lat^T [dim][64 key positions]): rows of 8 chunks, two per
//    256-byte bank line, chunk c of row r at c ^ ((r >> 1) & 7): the even (odd) rows of a group
//    differ in bits 1-3.
// The xor'd offsets of k-step ks are those of k-step 0 xor 32 ks.
__device__ __forceinline__ int lat32_off(int row, int chunk) { return row * 128 + 16 * (chunk ^ ((row >> 1) & 7)); }

template <int kKS>
__global__ void __launch_bounds__(kOtfThreads, 1) otf_fwd_short_kernel(OtfParams p) {
  constexpr int kRowWaves = kOtfWaves / kKS;
  constexpr int kRows = 32 * kRowWaves;
  constexpr int kKb = 2 / kKS;     // 32-key blocks of a tile per wave
  __shared__ __attribute__((aligned(1024))) char smem[kOtfLds];
  DMLA_LDS char* lds = (DMLA_LDS char*)smem;
  const int wave = uniform(threadIdx.x >> 6);
  const int lane = lane_id();
  const int l32 = lane & 31, hf = lane >> 5;
  const int l16 = lane & 15, g = lane >> 4;
  const int kh = wave / kRowWaves;       // first key block of this wave (kKS = 2)
  const int bh = (int)blockIdx.x % (p.B * p.H);
  const int qt = p.n_qt - 1 - (int)blockIdx.x / (p.B * p.H);   // heaviest (latest) tiles first
  const int b = bh / p.H, h = bh % p.H;
  const int off = p.Sk - p.Sq;
  const int row0 = qt * kRows + 32 * (wave % kRowWaves);       // this wave's first query row
  const int last_row = min(p.Sq, qt * kRows + kRows) - 1;
  const int key_end = p.causal ? min(p.Sk, last_row + off + 1) : p.Sk;
  const int n_t = key_end > 0 ? (key_end + kOtfKeys - 1) / kOtfKeys : 0;
  const unsigned lds_base = lds_addr(lds);

  stage_w(p, h, lds_base, wave, lane);
  // ---- raw K / V tile copies: as in the kernel above (wave w: tensor w / 4, keys 16 (w % 4) ..) ----
  const int xw = wave >> 2;
  const bf16* xbase = xw == 0 ? p.k + b * p.k_sb + h * p.k_sh : p.v + b * p.v_sb + h * p.v_sh;
  const int64_t xss = xw == 0 ? p.k_ss : p.v_ss;
  const unsigned raw_lane = (unsigned)((16 * (wave & 3) + g) * xss * 2);
  auto stage_raw = [&](int t, int st) {
    const unsigned ldst = lds_base + (st * 2 + xw) * kRawBytes + (wave & 3) * 4 * 1024;
    if (t * kOtfKeys + kOtfKeys <= p.Sk) {
#pragma unroll
      for (int c = 0; c < 4; ++c)
        dma16(xbase + (int64_t)(t * kOtfKeys + 4 * c) * xss, raw_lane + 16u * (unsigned)(l16 ^ (4 * c + g)),
              ldst + c * 1024);
    } else {
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int gk = min(t * kOtfKeys + 16 * (wave & 3) + 4 * c + g, p.Sk - 1);
        dma16_addr(xbase + (int64_t)gk * xss + 8 * (l16 ^ (4 * c + g)), ldst + c * 1024);
      }
    }
  };
  if (n_t > 0) stage_raw(0, 0);
  if (n_t > 1) stage_raw(1, 1);

  // ---- Q rows of this wave as the B operand of S^T: qreg[ks] = Q[row0 + l32][16 ks + 8 hf ..]
  bf16x8 qreg[4];
  {
    const bf16* qrow = p.q + b * p.q_sb + h * p.q_sh + (int64_t)min(row0 + l32, p.Sq - 1) * p.q_ss + 8 * hf;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) qreg[ks] = *reinterpret_cast<const bf16x8*>(qrow + 16 * ks);
  }
  wait_vmem();
  __syncthreads();   // W and raw tiles 0 and 1 landed
  // This wave's W^T operand: wreg[ks] = W^T[32 dbp + l32][16 ks + 8 hf ..].
  const int dbp = (wave >> 1) & 1, kbp = wave & 1;
  bf16x8 wreg[8];
#pragma unroll
  for (int ks = 0; ks < 8; ++ks)
    wreg[ks] = w_operand(lds + kLatOff + (wave < 4 ? 0 : kWBytes), 16 * ks + 8 * hf, 32 * dbp + 16 * (g & 1), lane);
  // Every wave holds its operands before the latent buffers take the first tile (lgkmcnt(0): the
  // reads above are done).
  __builtin_amdgcn_s_waitcnt(0xc07f);
  __syncthreads();

  // One 32 x 32 block of the projection of a tile (raw stage st) into latent buffer lb: dims 32 dbp ..
  // of keys 32 kbp .., K_lat (kK, waves 0-3) or V_lat (waves 4-7).
  auto proj = [&](auto is_k, int st, int lb) {
    constexpr bool kK = decltype(is_k)::value;
    const int raw = (st * 2 + (kK ? 0 : 1)) * kRawBytes + raw_off(32 * kbp + l32, hf);
    DMLA_LDS char* lat = lds + kLatOff + lb * kBufBytes + (kK ? 0 : kLatBytes);
    f32x16 c = {};
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) {
      const bf16x8 xr = *reinterpret_cast<const DMLA_LDS bf16x8*>(lds + (raw ^ (32 * ks)));
      if constexpr (kK) c = mfma32_bf16(wreg[ks], xr, c);   // K_lat^T[dim 32 dbp + 8a + 4 hf + i][key 32 kbp + l32]
      else c = mfma32_bf16(xr, wreg[ks], c);                // V_lat[key 32 kbp + 8a + 4 hf + i][dim 32 dbp + l32]
    }
    __builtin_amdgcn_sched_group_barrier(0x100, 8, 0);   // all reads ahead of the MFMAs
    __builtin_amdgcn_sched_group_barrier(0x008, 8, 0);
    __builtin_amdgcn_sched_barrier(0);
    const int lrow = lat32_off(kK ? 32 * kbp + l32 : 32 * dbp + l32, 0);   // chunk c of the row: xor 16 c
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      if constexpr (kK) {
        // K_lat[key 32 kbp + l32][dims 32 dbp + 8a + 4 hf .. +3] times scale log2(e), as hi + lo
        bf16x4 hi, lo;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float x = c[4 * a + i] * p.scale_log2;
          hi[i] = (bf16)x;
          lo[i] = (bf16)(x - (float)hi[i]);
        }
        const int o = (lrow ^ (64 * dbp + 16 * a)) + 8 * hf;
        *reinterpret_cast<DMLA_LDS bf16x4*>(lat + o) = hi;
        *reinterpret_cast<DMLA_LDS bf16x4*>(lat + 2 * kLatBytes + o) = lo;
      } else {
        f16x4 v;
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = (_Float16)c[4 * a + i];
        // V_lat^T[dim][position]: key 32 kbp + 8a + 4 hf + i sits at position 32 kbp + 16 (a/2) +
        // 8 hf + 4 (a%2) + i, the key order of the P operand (S^T C layout).
        const int o = lrow ^ (64 * kbp + 16 * hf + 32 * (a >> 1));
        *reinterpret_cast<DMLA_LDS f16x4*>(lat + o + 8 * (a & 1)) = v;
      }
    }
  };
  auto project = [&](int st, int lb) {
    if (wave < 4) proj(std::true_type{}, st, lb);
    else proj(std::false_type{}, st, lb);
  };

  f32x16 oacc[2] = {};   // O^T[dim 32 db + 8a + 4 hf + i][row0 + l32], element 4a + i
  // Of the wave's keys, per own row l32: the reference max, the exact running max and the row sum
  // (log2 units; the last two lane-partial).
  float mref = kNegInf, mtrue = kNegInf, lsum = 0.f;
  const int own_lim = p.causal ? min(row0 + l32 + off, p.Sk - 1) : p.Sk - 1;

  if (n_t > 0) project(0, 0);
  for (int t = 0; t < n_t; ++t) {
    wait_vmem();
    __syncthreads();   // latent tile t written, raw tile t+1 landed, raw stage t%2 and latent buffer (t+1)%2 free
    if (t + 1 < n_t) project((t + 1) & 1, (t + 1) & 1);
    if (t + 2 < n_t) stage_raw(t + 2, t & 1);

    // Operand address of k-step ks in the tile's K_lat hi, V_lat^T (+ kLatBytes) and K_lat lo
    // (+ 2 kLatBytes): the same row and chunk of each.
    const int op0 = kLatOff + (t & 1) * kBufBytes + lat32_off(l32, hf);
    const float nmr = mref == kNegInf ? 0.f : -mref;
    f32x16 s[kKb];   // S^T minus the reference: key 32 (kh + kb) + 8a + 4 hf + i, row l32
#pragma unroll
    for (int kb = 0; kb < kKb; ++kb)
#pragma unroll
      for (int i = 0; i < 16; ++i) s[kb][i] = nmr;
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int kb = 0; kb < kKb; ++kb) {
        const DMLA_LDS char* op = lds + (op0 ^ (32 * ks)) + (kh + kb) * 4096;
        const bf16x8 lo = *reinterpret_cast<const DMLA_LDS bf16x8*>(op + 2 * kLatBytes);
        const bf16x8 hi = *reinterpret_cast<const DMLA_LDS bf16x8*>(op);
        s[kb] = mfma32_bf16(lo, qreg[ks], s[kb]);
        s[kb] = mfma32_bf16(hi, qreg[ks], s[kb]);
      }
    // Six operand reads ahead of the MFMAs.
    __builtin_amdgcn_sched_group_barrier(0x100, 6, 0);
#pragma unroll
    for (int i = 0; i < 8 * kKb - 6; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, 6, 0);
    const int key0 = t * kOtfKeys;
    if (key0 + kOtfKeys > p.Sk || (p.causal && key0 + kOtfKeys - 1 > row0 + off)) {
#pragma unroll
      for (int kb = 0; kb < kKb; ++kb) {
        const int lim = own_lim - key0 - 32 * (kh + kb) - 4 * hf;
#pragma unroll
        for (int i = 0; i < 16; ++i)
          if (8 * (i >> 2) + (i & 3) > lim) s[kb][i] = kNegInf;
      }
    }
    float mx = kNegInf;
#pragma unroll
    for (int kb = 0; kb < kKb; ++kb)
#pragma unroll
      for (int i = 0; i < 16; i += 2) mx = fmaxf(mx, fmaxf(s[kb][i], s[kb][i + 1]));
    mx -= nmr;   // the max score in log2 units
    mtrue = fmaxf(mtrue, mx);
    if (__any(mx > mref + kSlack)) {
      // Move the reference to the exact row max so far; rescale l and the O rows.
      const float mnew = fmaxf(mref, half_max(mtrue));
      const float f = mnew == kNegInf ? 1.f : fast_exp2(mref - mnew);   // 0 when mref = -inf
      lsum *= f;
      mref = mnew;
      const float dn = (mnew == kNegInf ? 0.f : -mnew) - nmr;   // this tile's arguments move along
#pragma unroll
      for (int i = 0; i < 16; ++i) {
#pragma unroll
        for (int kb = 0; kb < kKb; ++kb) s[kb][i] += dn;
        oacc[0][i] *= f;
        oacc[1][i] *= f;
      }
    }
    const f16x2 ones = {(_Float16)1.f, (_Float16)1.f};
#pragma unroll
    for (int ks = 0; ks < 2 * kKb; ++ks) {
      f16x8 pa;   // B operand of O^T += V_lat^T P^T: keys of the k-step in V_lat^T order
#pragma unroll
      for (int j = 0; j < 8; ++j) pa[j] = (_Float16)fast_exp2(s[ks >> 1][8 * (ks & 1) + j]);
#pragma unroll
      for (int j = 0; j < 4; ++j) lsum = __builtin_amdgcn_fdot2(f16x2{pa[2 * j], pa[2 * j + 1]}, ones, lsum, false);
      const int vop = (op0 ^ (32 * ks)) ^ (64 * kh);   // kh: 64 bytes (32 positions) along the row
#pragma unroll
      for (int db = 0; db < 2; ++db) {
        const f16x8 vb = *reinterpret_cast<const DMLA_LDS f16x8*>(lds + vop + kLatBytes + db * 4096);
        oacc[db] = mfma32_f16(vb, pa, oacc[db]);
      }
    }
  }

  // ---- merge of the two key halves: waves 4-7 hand theirs over through LDS ----
  if constexpr (kKS == 2) {
    __syncthreads();   // the last tile is read out
    DMLA_LDS f32x4* ox = reinterpret_cast<DMLA_LDS f32x4*>(lds) + (wave % kRowWaves) * 9 * 64 + lane;
    if (kh == 1) {
#pragma unroll
      for (int j = 0; j < 8; ++j)
        ox[64 * j] = f32x4{oacc[j >> 2][4 * (j & 3)], oacc[j >> 2][4 * (j & 3) + 1], oacc[j >> 2][4 * (j & 3) + 2],
                           oacc[j >> 2][4 * (j & 3) + 3]};
      ox[64 * 8] = f32x4{mref, mtrue, lsum, 0.f};
    }
    __syncthreads();
    if (kh == 1) return;
    const f32x4 st = ox[64 * 8];
    const float mnew = fmaxf(mref, st[0]);
    const float f0 = mnew == kNegInf ? 1.f : fast_exp2(mref - mnew), f1 = mnew == kNegInf ? 0.f : fast_exp2(st[0] - mnew);
    mref = mnew;
    mtrue = fmaxf(mtrue, st[1]);
    lsum = lsum * f0 + st[2] * f1;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const f32x4 o1 = ox[64 * j];
#pragma unroll
      for (int i = 0; i < 4; ++i)
        oacc[j >> 2][4 * (j & 3) + i] = oacc[j >> 2][4 * (j & 3) + i] * f0 + o1[i] * f1;
    }
  }

  // ---- epilogue: row sums, statistics, normalised O ----
  const float ltot = half_sum(lsum);
  const float mrow = half_max(mtrue);
  const float inv = ltot > 0.f ? 1.f / ltot : 0.f;
  const int r = row0 + l32;
  if (r >= p.Sq) return;
  if (hf == 0 && p.m) {
    const int64_t idx = ((int64_t)b * p.H + h) * p.Sq + r;
    const bool any = ltot > 0.f;
    p.m[idx] = any ? mrow * kLn2 : kNegInf;
    p.l[idx] = any ? ltot * fast_exp2(mref - mrow) : 0.f;
  }
  bf16* orow = p.o + b * p.o_sb + h * p.o_sh + (int64_t)r * p.o_ss;
#pragma unroll
  for (int db = 0; db < 2; ++db) {
#pragma unroll
    for (int ap = 0; ap < 2; ++ap) {
      typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
      typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
      bf16x4 x, y;   // dims 32 db + 16 ap + 4 hf .. +3 and 8 more
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        x[i] = (bf16)(oacc[db][8 * ap + i] * inv);
        y[i] = (bf16)(oacc[db][8 * ap + 4 + i] * inv);
      }
      if (p.o_rows16) {
        // Swapping the halves' pieces leaves each lane 8 consecutive dims, 32 db + 16 ap + 8 hf ..
        const u32x2 xu = __builtin_bit_cast(u32x2, x), yu = __builtin_bit_cast(u32x2, y);
        u32x4 v;
#pragma unroll
        for (int w = 0; w < 2; ++w) {
          const auto r2 = __builtin_amdgcn_permlane32_swap(xu[w], yu[w], false, false);
          v[w] = r2[0];
          v[2 + w] = r2[1];
        }
        *reinterpret_cast<u32x4*>(orow + 32 * db + 16 * ap + 8 * hf) = v;
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          orow[32 * db + 16 * ap + 4 * hf + i] = x[i];
          orow[32 * db + 16 * ap + 8 + 4 * hf + i] = y[i];
        }
      }
    }
  }
}

}  // namespace
}  // namespace dmla

using namespace dmla;

extern "C" int dmla_fwd_onthefly(const void* q, const void* k, const void* v, const void* wk, const void* wv,
                                 void* o, float* m, float* l, int64_t B, int64_t H, int64_t Sq, int64_t Sk,
                                 int64_t d_in, int64_t d_lat, int64_t q_sb, int64_t q_sh, int64_t q_ss,
                                 int64_t k_sb, int64_t k_ss, int64_t k_sh, int64_t v_sb, int64_t v_ss,
                                 int64_t v_sh, int64_t w_sh, int64_t w_si, int64_t o_sb, int64_t o_sh,
                                 int64_t o_ss, float softmax_scale, int causal, dmla_stream_t stream) {
  clear_error();
  if (!q || !k || !v || !wk || !wv || !o) return fail(DMLA_ERR_INVALID_ARG, "dmla_fwd_onthefly: null pointer argument");
  if ((m == nullptr) != (l == nullptr))
    return fail(DMLA_ERR_INVALID_ARG, "dmla_fwd_onthefly: m and l must both be set or both be NULL");
  if (B < 0 || H < 0 || Sq < 0 || Sk < 0) return fail(DMLA_ERR_INVALID_ARG, "dmla_fwd_onthefly: negative size");
  if (d_in != kDin || d_lat != kDlat)
    return fail(DMLA_ERR_UNSUPPORTED, "dmla_fwd_onthefly: only d_in=128, d_lat=64 is compiled (got %lld, %lld)",
                (long long)d_in, (long long)d_lat);
  if (!(softmax_scale > 0.f) || !__builtin_isfinite(softmax_scale))
    return fail(DMLA_ERR_INVALID_ARG, "dmla_fwd_onthefly: softmax_scale must be finite and > 0");
  if (!aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(wk) || !aligned16(wv) || !aligned16(o))
    return fail(DMLA_ERR_INVALID_ARG, "dmla_fwd_onthefly: tensors must be 16-byte aligned");
  if (!mult8(q_sb) || !mult8(q_sh) || !mult8(q_ss) || !mult8(k_sb) || !mult8(k_ss) || !mult8(k_sh) ||
      !mult8(v_sb) || !mult8(v_ss) || !mult8(v_sh) || !mult8(w_sh) || !mult8(w_si))
    return fail(DMLA_ERR_INVALID_ARG, "dmla_fwd_onthefly: input strides must be multiples of 8 elements");
  if (Sq > ((int64_t)1 << 30) || Sk > ((int64_t)1 << 30))
    return fail(DMLA_ERR_UNSUPPORTED, "dmla_fwd_onthefly: size too large");
  if (k_ss < 0 || v_ss < 0 || k_ss >= ((int64_t)1 << 24) || v_ss >= ((int64_t)1 << 24))
    return fail(DMLA_ERR_UNSUPPORTED, "dmla_fwd_onthefly: row strides of k and v must be in [0, 2^24)");
  if (B == 0 || H == 0 || Sq == 0) return DMLA_OK;
  OtfParams p = {};
  p.q = static_cast<const bf16*>(q);
  p.k = static_cast<const bf16*>(k);
  p.v = static_cast<const bf16*>(v);
  p.wk = static_cast<const bf16*>(wk);
  p.wv = static_cast<const bf16*>(wv);
  p.o = static_cast<bf16*>(o);
  p.m = m;
  p.l = l;
  p.q_sb = q_sb; p.q_sh = q_sh; p.q_ss = q_ss;
  p.k_sb = k_sb; p.k_ss = k_ss; p.k_sh = k_sh;
  p.v_sb = v_sb; p.v_ss = v_ss; p.v_sh = v_sh;
  p.w_sh = w_sh; p.w_si = w_si;
  p.o_sb = o_sb; p.o_sh = o_sh; p.o_ss = o_ss;
  p.B = (int)B; p.H = (int)H; p.Sq = (int)Sq; p.Sk = (int)Sk;
  p.causal = causal ? 1 : 0;
  p.scale_log2 = softmax_scale * kLog2e;
  p.o_rows16 = mult8(o_sb) && mult8(o_sh) && mult8(o_ss);
  const int rows = otf_rows(device_cu_count(), B * H, Sq, Sk, p.causal);
  p.n_qt = (int)((Sq + rows - 1) / rows);
  const int64_t grid = (int64_t)p.n_qt * B * H;
  if (grid > 0x7fffffff) return fail(DMLA_ERR_UNSUPPORTED, "dmla_fwd_onthefly: grid too large");
  const auto kernel = rows == kOtfRows ? otf_fwd_kernel : rows == 256 ? otf_fwd_short_kernel<1> : otf_fwd_short_kernel<2>;
  hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(kOtfThreads), 0, (hipStream_t)stream, p);
  return check_launch("dmla_fwd_onthefly");
}
