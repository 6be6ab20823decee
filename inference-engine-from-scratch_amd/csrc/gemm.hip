// W8A16 projection GEMMs and the bf16 LM-head GEMM for gfx950.
//
// Replaces Int8Linear.forward (ne/models/int8_quantization.py:55-57), which
// materialises bf16(int8 * scale) for the whole weight before F.linear, and the
// tied-embedding LM head (ne/models/qwen3.py:197-203).
//
// Shapes here are short and wide: M = query rows of a verify step (64 x 5 =
// 320), N up to 6144 (151936 for the LM head), K 1024..3072.  Both kernels stage
// X and W tiles in LDS with DMA copies (global_load_lds_dwordx4) so that copies
// stay in flight while the MFMAs (v_mfma_f32_16x16x32_bf16) consume the previous
// stage.  Each MFMA computes D = W . X^T (weight rows x token rows), so a lane ends
// up holding four consecutive output columns of one token row (8-byte stores).
// int8 weights become bf16 in registers after the LDS read (exact); the per-row
// scale is applied to the fp32 sum.
//
// At M = 320 every N-tile re-reads X; the tiles are sized to keep that traffic per CU
// near its minimum for 256 independent tiles, and the LM head keeps all 320 rows
// resident per work-group to read X once per 256 columns.  A projection's time is its
// work-group's chain (first weight fetch from HBM, then per stage a barrier, the copy
// issue, the fragment reads and the MFMAs, then the k-group exchange), not L2 -> CU
// bandwidth (~30 TB/s with enough loads in flight), HBM or the MFMAs.
#include <type_traits>

#include "ne_common.hpp"
#include "qk_rope_kv.hpp"

namespace ne {

namespace {

struct GemmParams {
  const uint16_t* x;
  int64_t ldx;
  const void* w;
  const void* scale;
  int m, n, k;
  int scale_dtype;   // of the projections' row scales
  uint16_t* y;
  int64_t ldy;
  uint64_t* argmax;  // [m][n / BN] packed (ordered value, ~index)
  int tiles_m, tiles_n;
};

__device__ __forceinline__ float sbyte(uint32_t w, int k) { return (float)(int8_t)(w >> (8 * k)); }

__device__ __forceinline__ bf16x8 int8x8_to_bf16x8(uint32_t a, uint32_t b) {
  u32x4 r = {pack_bf16x2(sbyte(a, 0), sbyte(a, 1)), pack_bf16x2(sbyte(a, 2), sbyte(a, 3)),
             pack_bf16x2(sbyte(b, 0), sbyte(b, 1)), pack_bf16x2(sbyte(b, 2), sbyte(b, 3))};
  return __builtin_bit_cast(bf16x8, r);
}

// order-preserving key: larger value wins, then smaller index wins
__device__ __forceinline__ uint64_t argmax_key(float v, uint32_t idx) {
  v = v + 0.0f;  // -0 compares equal to +0 (torch.argmax): give both one key
  uint32_t b = __builtin_bit_cast(uint32_t, v);
  b = (b & 0x80000000u) ? ~b : (b | 0x80000000u);
  return ((uint64_t)b << 32) | (uint64_t)(0xFFFFFFFFu - idx);
}

__device__ __forceinline__ uint64_t max_u64(uint64_t a, uint64_t b) { return a > b ? a : b; }

__device__ __forceinline__ uint64_t shfl_xor_u64(uint64_t v, int o) {
  const uint32_t lo = __shfl_xor((uint32_t)v, o);
  const uint32_t hi = __shfl_xor((uint32_t)(v >> 32), o);
  return ((uint64_t)hi << 32) | lo;
}

template <int SDT>
__device__ __forceinline__ float scale_at(const void* s, int64_t i) {
  if constexpr (SDT < 0) {
    return 1.f;
  } else {
    return load_scale<SDT>(s, i);
  }
}

// bf16(silu(gate)) * up of four paired outputs, each rounded to bf16 first
__device__ __forceinline__ u32x2 swiglu4(const floatx4& gate4, const floatx4& up4, const float (&gs)[4],
                                         const float (&us)[4]) {
  float out[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float gate = bf16_round(gate4[i] * gs[i]);
    const float up = bf16_round(up4[i] * us[i]);
    const float silu = bf16_round(gate / (1.f + __expf(-gate)));
    out[i] = silu * up;
  }
  return u32x2{pack_bf16x2(out[0], out[1]), pack_bf16x2(out[2], out[3])};
}

// ---- shared pieces -------------------------------------------------------------
// Tiles are copied global -> LDS with global_load_lds_dwordx4: every wave-instruction
// copies 1 KiB of whole 128-byte lines (4 rows of 256 B or 8 rows of 128 B), the access
// shape the vector L1 serves at full rate.  Each lane picks its source so that LDS row
// `row` holds 16-byte chunk c at position c ^ (row % chunks-per-row), which makes the
// MFMA fragment reads bank-conflict free.
constexpr int kArgmaxCols = 64;  // columns per LM-head argmax partial
constexpr int kStageK = 128;     // k per stage of the projection kernel
// the projection kernels address X rows with 32-bit byte offsets from a scalar base
constexpr int64_t kMaxXElems = (int64_t(1) << 31) - 256;

__device__ __forceinline__ void lds_dma16(const void* src, void* lds_wave_base) {
  __builtin_amdgcn_global_load_lds(src, (__attribute__((address_space(3))) void*)lds_wave_base, 16,
                                   0, 0);
}

// s_waitcnt vmcnt(n) leaving lgkmcnt/expcnt unconstrained (gfx9 encoding)
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

// ---- W8A16 projections ----------------------------------------------------------
// Work-group tile: PM * 16 token rows (80 for the plain shapes, 48 for split-K) x 16 *
// NSUB weight rows, sized so that the verify-step shapes give about one work-group per
// CU (M = 320: QKV N = 4096 and gate|up N = 6144 give 256 tiles; o / down N = 1024 give
// 7 x 16 tiles of 48 rows, split 2 ways over K).  For o / down, 48-row tiles and two
// splits (224 work-groups) against 80-row tiles and four (256): the split-K sum +
// RMSNorm that follows reads half the fp32 partials; with 28 distinct weights replayed
// back to back the pair takes 9.5 / 10.6 us instead of 10.6 / 11.3 us, inside the
// verify step the GEMMs take the same time and the norm 0.14 us less.  Fewer rows gain
// more: 288 rows (6 x 16 x 2 work-groups instead of 4 x 16 x 4) and 64 rows (2 x 16 x 4
// instead of 1 x 16 x 4).  The MFMA waves form KG k-groups x NSUB / NPW: wave (kg, nw) runs the
// 4 / KG k-steps kg * 4 / KG .. (32 wide each) of every 128-wide stage for all PM token
// subtiles against weight subtiles nw * NPW .. + NPW, so each X fragment read from LDS
// feeds NPW MFMAs and each weight fragment PM.  At the end, wave (kg, nw) finishes the
// token subtiles mi with mi % KG == kg: the other k-groups' partial tiles of those come
// through LDS and are added in k-group order.  Two k-groups halve that exchange (and
// its barrier wait) against four, for twice the X fragment reads in the loop.
//
// Stages are copied by DMA into two LDS rings: X rows (from L2, where every column
// tile re-reads them) run kRX - 1 stages ahead and weight rows (from HBM, the longer
// way) kRW - 1 stages ahead.  A wave copies either X or weight rows, never both, so
// its vmcnt counts one stream and its wait for a stage is exact.  Each wave reads the
// fragments of stage t from LDS before it runs the MFMAs of stage t - 1 (held in
// registers), so the LDS latency hides under the multiplies.
constexpr int kPM = 5;       // token subtiles per work-group (the fused QKV epilogue uses 3)
constexpr int kSplitPM = 3;  // token subtiles per work-group of the split-K product
constexpr int kQkvKRows = 32;  // rows per work-group of the fused QKV kernel's k heads (q / v: 48)

template <int NSUB, int PM, int KG, int NPW>
struct ProjLayout {
  static_assert(KG == 1 || KG == 2 || KG == 4, "k-groups split the 4 k-steps of a stage");
  static_assert(NSUB % NPW == 0, "weight subtiles per wave");
  static constexpr int kKS = 4 / KG;  // k-steps per wave per stage
  static constexpr int kPRows = PM * 16;
  static constexpr int kNW = NSUB / NPW;
  static constexpr int kWaves = KG * kNW;
  static constexpr int kThreads = kWaves * kWave;
  static constexpr int kXI = PM * 4;    // 1 KiB copies per stage: X rows of 256 B ...
  static constexpr int kWI = NSUB * 2;  // ... and weight rows of 128 B
  static constexpr int kXBytes = kXI * 1024;
  static constexpr int kWBytes = kWI * 1024;
  static constexpr int kRX = 3;
  static constexpr int kRW = 6;
  // copies per X-copying / weight-copying wave: the fewest per wave that fit the waves
  static constexpr int split() {
    int best = -1, cost = 1 << 30;
    for (int dx = 1; dx <= kXI; ++dx)
      for (int dw = 1; dw <= kWI; ++dw)
        if (kXI % dx == 0 && kWI % dw == 0 && kXI / dx + kWI / dw <= kWaves && (dx > dw ? dx : dw) < cost) {
          cost = dx > dw ? dx : dw;
          best = dx * 256 + dw;
        }
    return best;
  }
  static constexpr int kDX = split() / 256;
  static constexpr int kDW = split() % 256;
  static constexpr int kNXW = kXI / kDX;  // waves [0, kNXW) copy X
  static constexpr int kNWW = kWI / kDW;  // waves [kNXW, kNXW + kNWW) copy weights
  static constexpr int kRedBytes = KG * kNW * PM * NPW * 1024;
  static constexpr int kRing = kRX * kXBytes + kRW * kWBytes;
  static constexpr int kLds = kRing > kRedBytes ? kRing : kRedBytes;
  static_assert(split() > 0, "copy split");
  static_assert(kDX * (kRX - 2) < 64 && kDW * (kRW - 2) < 64, "vmcnt range");
  static_assert(kLds <= 160 * 1024, "LDS");
};

// a wave-uniform pointer kept in SGPRs, so that a copy's address is a scalar base plus
// a 32-bit lane offset
__device__ __forceinline__ const char* uniform_ptr(const char* ptr) {
  const uint64_t v = (uint64_t)ptr;
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return (const char*)(((uint64_t)hi << 32) | lo);
}

// s_waitcnt vmcnt(D * pend) for a run-time pend in [0, P]
template <int D, int P>
__device__ __forceinline__ void wait_pending(int pend) {
  if constexpr (P <= 0) {
    wait_vmcnt<0>();
  } else {
    if (pend >= P) {
      wait_vmcnt<D * P>();
    } else {
      wait_pending<D, P - 1>(pend);
    }
  }
}

// Two adjacent 16-column subtiles of a 16-row MFMA result, lane (r, g) with columns 4 g ..
// + 4 of each as packed bf16 (a, b): regrouped so that the lane holds 8 consecutive columns
// from column 16 (g % 2) + 8 (g / 2) of the pair, one 16-byte store instead of two of 8.
__device__ __forceinline__ u32x4 pair_columns(const u32x2& a, const u32x2& b) {
  const auto x = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false);
  const auto y = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
  return u32x4{x[0], y[0], x[1], y[1]};
}
__device__ __forceinline__ int pair_column(int g) { return 16 * (g & 1) + 8 * (g >> 1); }

__device__ __forceinline__ void wait_lgkmcnt0() { __builtin_amdgcn_s_waitcnt(15 | (3 << 14) | (7 << 4)); }

// The k loop of a work-group: kt_n stages of 128 from k = kbase (KT > 0: kt_n = KT).  X rows m0.. (rows past
// m re-read row m - 1 and are never stored) and weight rows n0.. are copied with the
// chunk swizzles below; in k-step kk (0..3) of a stage, lane group g = lane / 16
// supplies logical k = 64 (kk / 2) + 16 g + 8 (kk % 2) + e, e < 8: X chunk
// 8 (kk / 2) + 2 g + kk % 2 of its 256-byte row, weight bytes 16 (4 (kk / 2) + g) +
// 8 (kk % 2) of its 128-byte row.  Wave (kg, nw) runs k-steps kk = kg * KS + s.
template <int NSUB, int PM, int KG, int NPW, int KT>
__device__ __forceinline__ void proj_mainloop(const GemmParams& p, char* smem, int m0, int n0, int kbase,
                                              int kt_runtime, int wave, int lane, int kg, int nw,
                                              floatx4 (&acc)[PM][NPW]) {
  using L = ProjLayout<NSUB, PM, KG, NPW>;
  constexpr int KS = L::kKS;
  // a stage count known at compile time turns every wait below into one instruction
  const int kt_n = KT > 0 ? KT : kt_runtime;
  const int r = lane & 15;
  const int g = lane >> 4;
  const bool xwave = wave < L::kNXW;
  const bool wwave = wave >= L::kNXW && wave < L::kNXW + L::kNWW;
  constexpr int D = L::kDX > L::kDW ? L::kDX : L::kDW;
  // copy j of this wave: LDS position c ^ (row % chunks-per-row) for 16-byte chunk c of
  // LDS row `row`, which makes the fragment reads bank-conflict free
  uint32_t off[D];
#pragma unroll
  for (int j = 0; j < D; ++j) {
    if (xwave) {  // 4 X rows x 16 chunks
      const int row = (wave * L::kDX + j) * 4 + (lane >> 4);
      const int chunk = (lane & 15) ^ (row & 15);
      const int grow = min(m0 + row, p.m - 1);
      off[j] = (uint32_t)grow * (uint32_t)(p.ldx * 2) + (uint32_t)chunk * 16u;
    } else {  // 8 weight rows x 8 chunks
      const int row = ((wave - L::kNXW) * L::kDW + j) * 8 + (lane >> 3);
      const int chunk = (lane & 7) ^ (row & 7);
      off[j] = (uint32_t)row * (uint32_t)p.k + (uint32_t)chunk * 16u;
    }
  }
  const char* xbase = (const char*)p.x + (int64_t)kbase * 2;
  const char* wbase = (const char*)p.w + (int64_t)n0 * p.k + kbase;
  char* xring = smem;
  char* wring = smem + L::kRX * L::kXBytes;
  auto issue_x = [&](int s) {
    if (!xwave) return;
    char* slot = xring + (s % L::kRX) * L::kXBytes + wave * L::kDX * 1024;
    const char* src = uniform_ptr(xbase + s * (kStageK * 2));
#pragma unroll
    for (int j = 0; j < L::kDX; ++j) {
      uint32_t o = off[j];
      __asm__("" : "+v"(o));  // keep the lane offset 32-bit: scalar base + offset addressing
      lds_dma16(src + o, slot + j * 1024);
    }
  };
  auto issue_w = [&](int s) {
    if (!wwave) return;
    char* slot = wring + (s % L::kRW) * L::kWBytes + (wave - L::kNXW) * L::kDW * 1024;
    const char* src = uniform_ptr(wbase + s * kStageK);
#pragma unroll
    for (int j = 0; j < L::kDW; ++j) {
      uint32_t o = off[j];
      __asm__("" : "+v"(o));
      lds_dma16(src + o, slot + j * 1024);
    }
  };
  // stage t needs this wave's copies of stage t; those of later stages may still fly
  auto wait_stage = [&](int t) {
    if (xwave) wait_pending<L::kDX, L::kRX - 2>(min(kt_n - t - 1, L::kRX - 2));
    if (wwave) wait_pending<L::kDW, L::kRW - 2>(min(kt_n - t - 1, L::kRW - 2));
  };
  uint32_t xr[KS], wr[KS];
#pragma unroll
  for (int q = 0; q < KS; ++q) {
    const int kk = kg * KS + q;
    const int cx = 8 * (kk >> 1) + 2 * g + (kk & 1);
    xr[q] = (uint32_t)(r * 256 + ((cx ^ r) * 16));
    const int cw = 4 * (kk >> 1) + g;
    wr[q] = (uint32_t)((nw * NPW * 16 + r) * 128 + ((cw ^ (r & 7)) * 16) + (kk & 1) * 8);
  }
  using XFrag = u32x4[KS][PM];
  using WFrag = u32x2[KS][NPW];
  using AFrag = bf16x8[KS][NPW];
  // weight fragments first: their conversion is the first thing waiting on them
  auto read = [&](int s, XFrag& xf, WFrag& wf) {
    const char* xs = xring + (s % L::kRX) * L::kXBytes;
    const char* ws = wring + (s % L::kRW) * L::kWBytes;
#pragma unroll
    for (int q = 0; q < KS; ++q)
#pragma unroll
      for (int ns = 0; ns < NPW; ++ns) wf[q][ns] = *(const u32x2*)(ws + wr[q] + ns * 2048);
#pragma unroll
    for (int q = 0; q < KS; ++q)
#pragma unroll
      for (int mi = 0; mi < PM; ++mi) xf[q][mi] = *(const u32x4*)(xs + xr[q] + mi * 4096);
  };
  auto convert = [&](const WFrag& wf, AFrag& a) {
#pragma unroll
    for (int q = 0; q < KS; ++q)
#pragma unroll
      for (int ns = 0; ns < NPW; ++ns) a[q][ns] = int8x8_to_bf16x8(wf[q][ns][0], wf[q][ns][1]);
  };
  auto mma = [&](const XFrag& xf, const AFrag& a) {
#pragma unroll
    for (int q = 0; q < KS; ++q)
#pragma unroll
      for (int mi = 0; mi < PM; ++mi)
#pragma unroll
        for (int ns = 0; ns < NPW; ++ns)
          acc[mi][ns] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[q][ns], __builtin_bit_cast(bf16x8, xf[q][mi]),
                                                                acc[mi][ns], 0, 0, 0);
  };
  // stage t: its copies are in LDS after the barrier, and every wave has read stage
  // t - 1 into registers before it (lgkmcnt(0)), so the slots of stage t - 1 take the
  // copies of stages t + kRX - 1 and t + kRW - 1.  The MFMAs of stage t - 1 run on
  // weights converted to bf16 from the int8 read in step t - 1; the compiler places that
  // conversion just before those MFMAs (it keeps the int8 form live across the barrier),
  // so a wave converts and then multiplies.
  auto step = [&](int t, XFrag& xr_, WFrag& wr_, AFrag& ar, const XFrag& xm, const AFrag& am) {
    wait_stage(t);
    wait_lgkmcnt0();
    asm volatile("s_barrier" ::: "memory");
    if (t + L::kRX - 1 < kt_n) issue_x(t + L::kRX - 1);
    if (t + L::kRW - 1 < kt_n) issue_w(t + L::kRW - 1);
    read(t, xr_, wr_);
    __builtin_amdgcn_sched_barrier(0);  // the reads go out before the multiplies
    mma(xm, am);
    convert(wr_, ar);
    __builtin_amdgcn_sched_barrier(0);
  };

#pragma unroll
  for (int s = 0; s < L::kRW - 1; ++s)
    if (s < kt_n) issue_w(s);  // the weights first: they have the longer way to come
#pragma unroll
  for (int s = 0; s < L::kRX - 1; ++s)
    if (s < kt_n) issue_x(s);
  XFrag xa, xb;
  WFrag wa, wb;
  AFrag aa, ab;
  wait_stage(0);
  asm volatile("s_barrier" ::: "memory");
  if (L::kRX - 1 < kt_n) issue_x(L::kRX - 1);
  if (L::kRW - 1 < kt_n) issue_w(L::kRW - 1);
  read(0, xa, wa);
  convert(wa, aa);
  int t = 1;
  for (; t + 1 < kt_n; t += 2) {
    step(t, xb, wb, ab, xa, aa);
    step(t + 1, xa, wa, aa, xb, ab);
  }
  if (t < kt_n) {
    step(t, xb, wb, ab, xa, aa);
    wait_lgkmcnt0();
    mma(xb, ab);
  } else {
    wait_lgkmcnt0();
    mma(xa, aa);
  }
}

// EPI 0: y = bf16(acc * scale); 1: SwiGLU of paired gate/up subtiles; 3: fp32 partial
// sums of K split blockIdx.y, scaled, into partial[split][m][n]; 4: the QKV projection
// with one 128-column head per tile (NSUB 8), each head vector of the bf16 result taken
// through QK-norm + RoPE into q_out or quantised into the KV cache (qk_rope_kv.hpp) --
// the bits the GEMM with EPI 0 followed by the row kernel produce, without the qkv round
// trip through memory.  KV (EPI 4): 1 bf16 cache, 2 int8 + bf16 scales, 3 int8 + fp16.
template <int NSUB, int SDT, int EPI, int KV, int PM, int KG, int NPW, int KT>
__global__ __launch_bounds__((ProjLayout<NSUB, PM, KG, NPW>::kThreads)) void proj_kernel(
    GemmParams p, int k_per_split, float* partial, QkvRopeArgs qa) {
  using L = ProjLayout<NSUB, PM, KG, NPW>;
  constexpr int kPRows = L::kPRows;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  // Every kernel argument the work-group uses, requested in one batch: left to itself
  // the compiler loads each next to its first use, and the tile index, the copy
  // addresses and the epilogue then wait on one scalar-cache round trip after another.
  asm volatile("" ::"s"(p.x), "s"(p.ldx), "s"(p.w), "s"(p.scale), "s"(p.m), "s"(p.k), "s"(p.tiles_m),
               "s"(p.tiles_n), "s"(k_per_split));
  if constexpr (EPI == 3) {
    asm volatile("" ::"s"(partial), "s"(p.n));
  } else if constexpr (EPI != 4) {
    asm volatile("" ::"s"(p.y), "s"(p.ldy));
  } else {
    asm volatile("" ::"s"(qa.q_norm_w), "s"(qa.k_norm_w), "s"(qa.positions), "s"(qa.slot_mapping),
                 "s"(qa.rope), "s"(qa.rope_positions), "s"(qa.hq));
  }
  const int bid = blockIdx.x;
  const int xcd = bid % kNumXcd;
  const int jj = bid / kNumXcd;
  int tm = jj % p.tiles_m;
  int tn = (jj / p.tiles_m) * kNumXcd + xcd;  // the M tiles of one weight tile share an XCD
  int tile_rows = kPRows;
  if constexpr (EPI == 4) {
    // heads xcd, xcd + 8, ... on this XCD, each with all its row tiles: kPRows rows for
    // q / v heads, kQkvKRows for k heads (whose epilogue also quantises, so fewer rows
    // per work-group even out the work-groups' end times)
    int j = jj;
    tn = -1;
    for (int h = xcd; h < p.tiles_n; h += kNumXcd) {
      const bool kh = h >= qa.hq && h < qa.hq + qa.hkv;
      const int t = kh ? qa.tiles_k : p.tiles_m;
      if (j < t) {
        tn = h;
        tm = j;
        tile_rows = kh ? kQkvKRows : kPRows;
        break;
      }
      j -= t;
    }
    if (tn < 0) return;
  }
  if (tn >= p.tiles_n) return;
  const int split = blockIdx.y;
  const int m0 = tm * tile_rows;
  const int n0 = tn * NSUB * 16;
  const int kbase = split * k_per_split;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int lane = threadIdx.x % kWave;
  const int kg = wave / L::kNW;
  const int nw = wave % L::kNW;
  const int r = lane & 15;
  const int g = lane >> 4;

  // the epilogue's weight-row scales, fetched now so that their latency hides under
  // the k loop: lane (r, g) stores columns (nw NPW + ns) 16 + 4 g + i
  float sc[NPW][4] = {};
  if constexpr (EPI != 4) {  // EPI 4 scales its rows' columns instead (e_sc)
#pragma unroll
    for (int ns = 0; ns < NPW; ++ns)
#pragma unroll
      for (int i = 0; i < 4; ++i) sc[ns][i] = scale_at<SDT>(p.scale, n0 + (nw * NPW + ns) * 16 + 4 * g + i);
  }

  // EPI 4: wave w finishes rows w, w + kWaves, ... of the tile (head tn).  Their slots
  // and positions (scalar loads) and the head's norm weights are requested now and
  // used only in the epilogue, so no wait for them precedes the k loop; the RoPE
  // values, which need the positions, are requested right after the k loop.
  constexpr int kEpiRows = (kPRows + L::kWaves - 1) / L::kWaves;
  int e_slot[kEpiRows], e_pos[kEpiRows];
  uint16_t e_w[2] = {0, 0};
  float e_sc[2] = {0.f, 0.f};  // weight-row scales of head columns lane and lane + 64
  if constexpr (EPI == 4) {
    const uint16_t* w = (tn < qa.hq) ? qa.q_norm_w : qa.k_norm_w;  // v heads do not use it
    e_w[0] = w[lane];
    e_w[1] = w[lane + 64];
    e_sc[0] = scale_at<SDT>(p.scale, n0 + lane);
    e_sc[1] = scale_at<SDT>(p.scale, n0 + 64 + lane);
#pragma unroll
    for (int i = 0; i < kEpiRows; ++i) {
      const int m = min(m0 + wave + L::kWaves * i, p.m - 1);
      e_slot[i] = ((const ConstI32*)qa.slot_mapping)[m];
      e_pos[i] = ((const ConstI32*)qa.positions)[m];
    }
  }

  floatx4 acc[PM][NPW];
#pragma unroll
  for (int mi = 0; mi < PM; ++mi)
#pragma unroll
    for (int ns = 0; ns < NPW; ++ns) acc[mi][ns] = floatx4{0.f, 0.f, 0.f, 0.f};

  proj_mainloop<NSUB, PM, KG, NPW, KT>(p, smem, m0, n0, kbase, k_per_split / kStageK, wave, lane, kg, nw,
                                       acc);

  // EPI 4: the rows' cos / sin, in flight while the k-groups are summed
  uint16_t e_rc[kEpiRows], e_rs[kEpiRows];
  if constexpr (EPI == 4) {
    // the loads issued before the k loop are long done: take their values now, so that
    // the compiler's wait for them does not land after the loads below
    __asm__ __volatile__("" ::"v"(e_sc[0]), "v"(e_sc[1]), "v"(e_w[0]), "v"(e_w[1]));
#pragma unroll
    for (int i = 0; i < kEpiRows; ++i) {
      const int64_t pos = min(max(e_pos[i], 0), qa.rope_positions - 1);
      e_rc[i] = qa.rope[pos * 128 + lane];
      e_rs[i] = qa.rope[pos * 128 + 64 + lane];
    }
  }

  // ---- sum the k-groups through LDS (the stage ring is free once all waves pass) ----
  lds_barrier();
  if constexpr (EPI == 4) {
    // partials as rows [kg][row][128 + 4 pad] fp32, so that the row pass below reads a
    // row's columns lane and lane + 64 as consecutive words; each row is summed over the
    // k-groups in order and scaled, the bits the GEMM epilogue stores
    static_assert(NSUB == 8, "one head per tile");
    constexpr int kRowF = 132;
    static_assert(KG * kPRows * kRowF * 4 <= L::kLds, "partials fit the stage ring");
    constexpr bool kInt8 = KV >= 2;
    constexpr int kKvSdt = KV == 3 ? NE_DTYPE_FP16 : NE_DTYPE_BF16;
    float* part = (float*)smem;
#pragma unroll
    for (int mi = 0; mi < PM; ++mi)
#pragma unroll
      for (int ns = 0; ns < NPW; ++ns)
        *(floatx4*)(part + (kg * kPRows + mi * 16 + r) * kRowF + (nw * NPW + ns) * 16 + 4 * g) = acc[mi][ns];
    lds_barrier();
    // this wave's rows all at once, so that their reductions overlap
    auto rows_pass = [&](auto n_rows) {
      constexpr int N = decltype(n_rows)::value;
      int rows_e[N];
      bool valid_e[N];
      float a_e[N], b_e[N], c_e[N], s_e[N];
      int64_t slot_e[N];
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const int rr = min(wave + L::kWaves * i, kPRows - 1);
        rows_e[i] = m0 + rr;
        valid_e[i] = wave + L::kWaves * i < tile_rows && m0 + rr < p.m;
        float va = part[rr * kRowF + lane];
        float vb = part[rr * kRowF + 64 + lane];
#pragma unroll
        for (int q = 1; q < KG; ++q) {
          va += part[(q * kPRows + rr) * kRowF + lane];
          vb += part[(q * kPRows + rr) * kRowF + 64 + lane];
        }
        a_e[i] = bf16_round(va * e_sc[0]);
        b_e[i] = bf16_round(vb * e_sc[1]);
        c_e[i] = bf16_to_f32(e_rc[i]);
        s_e[i] = bf16_to_f32(e_rs[i]);
        slot_e[i] = e_slot[i];
      }
      qk_norm_rope_kv_vectors<kInt8, kKvSdt, N>(qa, rows_e, valid_e, tn, lane, a_e, b_e, slot_e,
                                                bf16_to_f32(e_w[0]), bf16_to_f32(e_w[1]), c_e, s_e);
    };
    static_assert(kQkvKRows % L::kWaves == 0 && kQkvKRows / L::kWaves <= kEpiRows, "k-tile rows per wave");
    if (tile_rows == kQkvKRows) {
      rows_pass(std::integral_constant<int, kQkvKRows / L::kWaves>{});
    } else {
      rows_pass(std::integral_constant<int, kEpiRows>{});
    }
    return;
  }
  // Token subtile mi is finished by k-group mi % KG: each wave hands the partial tiles of
  // the other subtiles to their finishing wave through LDS, [kg][nw][mi][ns][lane].
  floatx4* red = (floatx4*)smem;
  auto red_at = [&](int q, int mi, int ns) -> floatx4& {
    return red[(((q * L::kNW + nw) * PM + mi) * NPW + ns) * kWave + lane];
  };
#pragma unroll
  for (int mi = 0; mi < PM; ++mi)
    if (KG > 1 && mi % KG != kg)
#pragma unroll
      for (int ns = 0; ns < NPW; ++ns) red_at(kg, mi, ns) = acc[mi][ns];
  if constexpr (KG > 1) lds_barrier();

#pragma unroll
  for (int mi = 0; mi < PM; ++mi) {
    if (mi % KG != kg) continue;
    floatx4 v[NPW];
#pragma unroll
    for (int ns = 0; ns < NPW; ++ns) {
      // in k-group order, this wave's own partial from its registers
      v[ns] = kg == 0 ? acc[mi][ns] : red_at(0, mi, ns);
#pragma unroll
      for (int q = 1; q < KG; ++q) v[ns] += q == kg ? acc[mi][ns] : red_at(q, mi, ns);
    }
    // lane holds D[n = 4 g + i][m = r] of weight subtiles nw NPW + ns
    const int m = m0 + mi * 16 + r;
    if (m >= p.m) continue;
    if constexpr (EPI == 0) {
#pragma unroll
      for (int ns = 0; ns < NPW; ++ns) {
        const int n = n0 + (nw * NPW + ns) * 16 + 4 * g;
        const u32x2 bits = {pack_bf16x2(v[ns][0] * sc[ns][0], v[ns][1] * sc[ns][1]),
                            pack_bf16x2(v[ns][2] * sc[ns][2], v[ns][3] * sc[ns][3])};
        *(u32x2*)(p.y + (int64_t)m * p.ldy + n) = bits;
      }
    } else if constexpr (EPI == 1) {
      static_assert(NPW == 2, "a wave holds paired gate / up subtiles");
      // gate rows are subtile 2 nw, the paired up rows subtile 2 nw + 1
      const int ncol = (n0 + 2 * nw * 16) / 2 + 4 * g;
      const u32x2 bits = swiglu4(v[0], v[1], sc[0], sc[1]);
      *(u32x2*)(p.y + (int64_t)m * p.ldy + ncol) = bits;
    } else {
#pragma unroll
      for (int ns = 0; ns < NPW; ++ns) {
        const int n = n0 + (nw * NPW + ns) * 16 + 4 * g;
        const floatx4 sv = {v[ns][0] * sc[ns][0], v[ns][1] * sc[ns][1], v[ns][2] * sc[ns][2],
                            v[ns][3] * sc[ns][3]};
        *(floatx4*)(partial + ((int64_t)split * p.m + m) * p.n + n) = sv;
      }
    }
  }
}

template <int NSUB, int SDT, int EPI, int KV, int PM, int KG, int NPW, int KT>
int launch_proj_kt(GemmParams p, int splits, float* partial, hipStream_t stream, const char* name,
                   QkvRopeArgs qa) {
  using L = ProjLayout<NSUB, PM, KG, NPW>;
  p.tiles_m = ceil_div(p.m, L::kPRows);
  p.tiles_n = p.n / (NSUB * 16);
  const int tiles_n_padded = ceil_div(p.tiles_n, kNumXcd) * kNumXcd;
  dim3 grid((unsigned)(p.tiles_m * tiles_n_padded), (unsigned)splits);
  if constexpr (EPI == 4) {
    // per XCD: its heads' row tiles (k heads in tiles of kQkvKRows); the grid covers the
    // XCD with the most
    qa.tiles_k = ceil_div(p.m, kQkvKRows);
    int most = 0;
    for (int x = 0; x < kNumXcd; ++x) {
      int t = 0;
      for (int h = x; h < p.tiles_n; h += kNumXcd) t += (h >= qa.hq && h < qa.hq + qa.hkv) ? qa.tiles_k : p.tiles_m;
      most = t > most ? t : most;
    }
    grid.x = (unsigned)(most * kNumXcd);
  }
  static const hipError_t attr = hipFuncSetAttribute(
      (const void*)proj_kernel<NSUB, SDT, EPI, KV, PM, KG, NPW, KT>, hipFuncAttributeMaxDynamicSharedMemorySize,
      L::kLds);
  if (attr != hipSuccess) {
    set_error("%s: cannot reserve %d bytes of LDS: %s", name, L::kLds, hipGetErrorString(attr));
    return NE_ELAUNCH;
  }
  hipLaunchKernelGGL((proj_kernel<NSUB, SDT, EPI, KV, PM, KG, NPW, KT>), grid, dim3(L::kThreads), L::kLds,
                     stream, p, p.k / splits, partial, qa);
  return check_launch(name);
}

// Stage counts with a kernel of their own: 8 (K = 1024, the QKV and gate|up
// projections of the 0.6B model), and for split-K 8 and 12 (o and down split 2 ways over
// K = 2048 and 3072) and 4 and 6 (the same split 4 ways, for fewer rows); any other
// count runs the loop with a run-time count.
template <int NSUB, int SDT, int EPI, int KV, int PM, int KG, int NPW>
int launch_proj(GemmParams p, int splits, float* partial, hipStream_t stream, const char* name,
                const QkvRopeArgs& qa = QkvRopeArgs{}) {
  const int kt = p.k / splits / kStageK;
  if constexpr (EPI == 3) {
    if (kt == 4) return launch_proj_kt<NSUB, SDT, EPI, KV, PM, KG, NPW, 4>(p, splits, partial, stream, name, qa);
    if (kt == 6) return launch_proj_kt<NSUB, SDT, EPI, KV, PM, KG, NPW, 6>(p, splits, partial, stream, name, qa);
    if (kt == 8) return launch_proj_kt<NSUB, SDT, EPI, KV, PM, KG, NPW, 8>(p, splits, partial, stream, name, qa);
    if (kt == 12) return launch_proj_kt<NSUB, SDT, EPI, KV, PM, KG, NPW, 12>(p, splits, partial, stream, name, qa);
  } else {
    if (kt == 8) return launch_proj_kt<NSUB, SDT, EPI, KV, PM, KG, NPW, 8>(p, splits, partial, stream, name, qa);
  }
  return launch_proj_kt<NSUB, SDT, EPI, KV, PM, KG, NPW, 0>(p, splits, partial, stream, name, qa);
}

// ---- W8A16 projections over many rows (prefill) ---------------------------------------
// The kernel above is built for a verify step: every wave takes all rows of a tile, 80 at
// most.  Over thousands of rows its 80 x 64 tiles read each X row 64 times and each weight
// 52-100 times, and a wave reads 1.2 LDS fragments per MFMA.  Here a work-group of 8 waves
// owns 256 x 256, 128 x 256 or 128 x 128 outputs and a wave 128 x 64 or 64 x 64 of them:
// 0.38 or 0.5 fragments per MFMA.
//   waves = KG k-groups x MW row groups x NW column groups.  The 128 x 128 tile has two
//           k-groups (each takes half of every stage's k, the halves of the sum meet in LDS
//           at the end), the others one.
//   ring  = three stages of KG blocks of 64 k, copied by DMA: X rows of 128 B and int8
//           weight rows of 64 B, chunk-swizzled so that the fragment reads are free of bank
//           conflicts.  Every wave issues the same number of copies per stage, so one vmcnt
//           wait covers the stage.
//   loop  = a wave holds the fragments of the next k-step while the MFMAs of the current
//           one run; the barrier that admits stage t + 1 sits before the last MFMAs of stage
//           t, so its wait and the first reads of t + 1 hide under them.
//   k order: in k-step q of a block, lane group g holds logical k = 16 g + 8 q + e, so one
//           16-byte weight read feeds both k-steps.
// Measured (four weights in turn from a HIP graph; us, before -> here): 8,192 rows QKV
// N = 4,096 154 -> 72, gate|up N = 6,144 183 -> 104 (990 TFLOP/s), o K = 2,048 83 -> 39,
// down K = 3,072 119 -> 54; 4,096 rows 83 -> 39, 102 -> 62, 49 -> 25, 68 -> 34; the QKV
// product with its epilogue, in the layer, 195 -> 100 and 110 -> 56.  16-byte stores (two
// output subtiles regrouped by pair_columns) instead of 8: QKV 72 -> 65 us at 8,192 rows, o
// 25 -> 23 us at 4,096.  A 256 x 256
// tile's 64 k take ~2.3 us for 2,048 cycles of MFMAs per SIMD: the int8 conversions (48 VALU
// per 32 MFMAs, both waves of a SIMD at once) and the LDS (208 KB per block at 128 B per
// clock) share that time with them.
template <int BM_, int BN_, int MW_, int NW_, int KG_>
struct TileLayout {
  static constexpr int BM = BM_, BN = BN_, MW = MW_, NW = NW_, KG = KG_;
  static constexpr int kWaves = 8;
  static_assert(MW * NW * KG == kWaves && (KG == 1 || KG == 2), "waves");
  static constexpr int PM = BM / MW / 16;   // token subtiles per wave
  static constexpr int NPW = BN / NW / 16;  // weight subtiles per wave
  static constexpr int kXBlock = BM * 128, kWBlock = BN * 64;
  static constexpr int kBlock = kXBlock + kWBlock;  // 64 k of X and W
  static constexpr int kStage = KG * kBlock;
  static constexpr int kStageK = 64 * KG;
  static constexpr int kRing = 3;
  static constexpr int kPerBlock = kBlock / 1024 / kWaves;  // copies per wave and block
  static constexpr int kXPerBlock = kXBlock / 1024 / kWaves;
  static constexpr int kCopies = KG * kPerBlock;  // copies per wave and stage
  static constexpr int kRed = KG > 1 ? kWaves * (PM / 2) * NPW * 1024 : 0;
  static constexpr int kRowB = BN * 2 + 16;       // bytes per row of the staged bf16 tile (QKV epilogue)
  static constexpr int kLds = kRing * kStage;
  static_assert(kBlock % (1024 * kWaves) == 0 && kXBlock % (1024 * kWaves) == 0, "copies split evenly over the waves");
  static_assert(kRed <= kLds && BM * kRowB <= kLds && kLds <= 160 * 1024, "LDS");
};

template <typename L>
struct TileWave {
  uint32_t off[L::kCopies];  // lane offsets of this wave's copies
  uint32_t xr, wr;           // fragment read positions within a block (k-step 0, subtile 0)
  int wave, mw, nw, kg;
};

template <typename L>
__device__ __forceinline__ void tile_mainloop(const GemmParams& p, char* smem, int n0, const TileWave<L>& w,
                                              floatx4 (&acc)[L::PM][L::NPW]) {
  constexpr int PM = L::PM, NPW = L::NPW, D = L::kCopies;
  const int n_stages = p.k / L::kStageK;
  const char* xbase = (const char*)p.x;
  const char* wbase = (const char*)p.w + (int64_t)n0 * p.k;
  // copy j of this wave is KiB 8 j + wave of the stage; a block is X rows, then weight rows
  auto issue = [&](int t) {
    char* slot = smem + (t % L::kRing) * L::kStage;
    const char* xs = uniform_ptr(xbase + (int64_t)t * (L::kStageK * 2));
    const char* ws = uniform_ptr(wbase + (int64_t)t * L::kStageK);
#pragma unroll
    for (int j = 0; j < D; ++j) {
      uint32_t o = w.off[j];
      __asm__("" : "+v"(o));  // keep the lane offset 32-bit: scalar base + offset addressing
      lds_dma16((j % L::kPerBlock < L::kXPerBlock ? xs : ws) + o, slot + (j * L::kWaves + w.wave) * 1024);
    }
  };
  using XFrag = u32x4[PM];
  using AFrag = bf16x8[NPW];
  auto block_at = [&](int t) { return smem + (t % L::kRing) * L::kStage + w.kg * L::kBlock; };
  // X chunk 2 g + q of a 128-byte row sits at position chunk ^ (row % 8): k-step q flips bit 4
  auto read_x = [&](int t, int q, XFrag& xf) {
    const char* xs = block_at(t) + (w.xr ^ (uint32_t)(q * 16));
#pragma unroll
    for (int mi = 0; mi < PM; ++mi) xf[mi] = *(const u32x4*)(xs + mi * 16 * 128);
  };
  u32x4 wf[NPW];  // both k-steps of a block
  auto read_w = [&](int t) {
    const char* ws = block_at(t) + w.wr;
#pragma unroll
    for (int ns = 0; ns < NPW; ++ns) wf[ns] = *(const u32x4*)(ws + ns * 16 * 64);
  };
  auto convert = [&](int q, AFrag& a) {
#pragma unroll
    for (int ns = 0; ns < NPW; ++ns) a[ns] = int8x8_to_bf16x8(wf[ns][2 * q], wf[ns][2 * q + 1]);
  };
  auto mma = [&](const XFrag& xf, const AFrag& a) {
#pragma unroll
    for (int mi = 0; mi < PM; ++mi)
#pragma unroll
      for (int ns = 0; ns < NPW; ++ns)
        acc[mi][ns] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[ns], __builtin_bit_cast(bf16x8, xf[mi]), acc[mi][ns],
                                                              0, 0, 0);
  };

#pragma unroll
  for (int s = 0; s < L::kRing; ++s)
    if (s < n_stages) issue(s);
  wait_pending<D, L::kRing - 1>(min(n_stages, L::kRing) - 1);  // stage 0 has landed
  asm volatile("s_barrier" ::: "memory");

  XFrag x0, x1;
  AFrag a0, a1;
  read_w(0);
  read_x(0, 0, x0);
  for (int t = 0; t + 1 < n_stages; ++t) {
    read_x(t, 1, x1);
    __builtin_amdgcn_sched_barrier(0);  // the reads go out before the multiplies
    convert(0, a0);
    mma(x0, a0);
    convert(1, a1);
    __builtin_amdgcn_sched_barrier(0);
    // stage t + 1 has landed and every wave has read stage t: its slot takes stage t + 3
    if (t + 2 < n_stages) {
      wait_vmcnt<D>();
    } else {
      wait_vmcnt<0>();
    }
    wait_lgkmcnt0();
    asm volatile("s_barrier" ::: "memory");
    if (t + L::kRing < n_stages) issue(t + L::kRing);
    read_w(t + 1);
    read_x(t + 1, 0, x0);
    __builtin_amdgcn_sched_barrier(0);
    mma(x1, a1);
    __builtin_amdgcn_sched_barrier(0);
  }
  read_x(n_stages - 1, 1, x1);
  convert(0, a0);
  mma(x0, a0);
  convert(1, a1);
  mma(x1, a1);
}

// the weight rows' scales first + 16 ns + i in the caller's dtype (one uniform branch)
template <int NPW>
__device__ __forceinline__ void tile_scales(const GemmParams& p, int first, float (&sc)[NPW][4]) {
  auto load = [&](auto dtype) {
#pragma unroll
    for (int ns = 0; ns < NPW; ++ns)
#pragma unroll
      for (int i = 0; i < 4; ++i) sc[ns][i] = load_scale<decltype(dtype)::value>(p.scale, first + ns * 16 + i);
  };
  if (p.scale_dtype == NE_DTYPE_BF16) {
    load(std::integral_constant<int, NE_DTYPE_BF16>{});
  } else if (p.scale_dtype == NE_DTYPE_FP16) {
    load(std::integral_constant<int, NE_DTYPE_FP16>{});
  } else {
    load(std::integral_constant<int, NE_DTYPE_FP32>{});
  }
}

// Sum / maximum over the 16 lanes of a DPP row, every lane ending with the result.  With
// a lane holding the sum of four consecutive leaves, the additions pair up exactly as
// wave_reduce_n pairs 64 lanes of one leaf each.
template <bool MAX, int N>
__device__ __forceinline__ void row16_reduce(float (&v)[N]) {
  auto op = [](float a, float b) { return MAX ? fmaxf(a, b) : a + b; };
#pragma unroll
  for (int i = 0; i < N; ++i) v[i] = op(v[i], dpp_f32<0xB1>(v[i]));  // quad_perm [1, 0, 3, 2]
#pragma unroll
  for (int i = 0; i < N; ++i) v[i] = op(v[i], dpp_f32<0x4E>(v[i]));  // quad_perm [2, 3, 0, 1]
#pragma unroll
  for (int i = 0; i < N; ++i) v[i] = op(v[i], dpp_f32<0x141>(v[i]));  // row_half_mirror
#pragma unroll
  for (int i = 0; i < N; ++i) v[i] = op(v[i], dpp_f32<0x140>(v[i]));  // row_mirror
}

__device__ __forceinline__ void unpack4(const u32x2 v, float (&f)[4]) {
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    f[2 * i] = __uint_as_float(v[i] << 16);
    f[2 * i + 1] = __uint_as_float(v[i] & 0xFFFF0000u);
  }
}

// four values rounded to bf16
__device__ __forceinline__ u32x2 pack4(const float (&f)[4]) {
  return u32x2{pack_bf16x2(f[0], f[1]), pack_bf16x2(f[2], f[3])};
}

__device__ __forceinline__ void round4(float (&f)[4]) { unpack4(pack4(f), f); }

// four int8 codes of quotients: rounded to even, clamped to +-127
__device__ __forceinline__ uint32_t codes4(const float (&t)[4]) {
  uint32_t b[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) b[e] = (uint32_t)(int)fminf(fmaxf(rintf(t[e]), -127.f), 127.f);
  const uint32_t lo = __builtin_amdgcn_perm(b[1], b[0], 0x0c0c0400u);
  return __builtin_amdgcn_perm(__builtin_amdgcn_perm(b[3], b[2], 0x0c0c0400u), lo, 0x05040100u);
}

// QK-norm + RoPE + KV write of the tile's head vectors, staged as bf16 in LDS (the bits the
// plain epilogue stores): the arithmetic of qk_norm_rope_kv_vectors on 16 lanes per vector,
// lane c with elements 4 c .. + 4 and 64 + 4 c .. + 4, so that a wave takes four vectors at
// once, RoPE pairs meet in a lane and stores are 4 or 8 bytes wide.
template <typename L, int KV>
__device__ __forceinline__ void tile_qkv_epilogue(const QkvRopeArgs& qa, const char* smem, int m, int m0, int n0,
                                                  int wave, int lane) {
  constexpr bool kInt8 = KV >= 2;
  constexpr int kSdt = KV == 3 ? NE_DTYPE_FP16 : NE_DTYPE_BF16;
  constexpr int kHeads = L::BN / 128;
  constexpr int kHeadWaves = L::kWaves / kHeads;   // waves per head of the tile
  constexpr int kWaveRows = L::BM / kHeadWaves;    // rows per wave
  constexpr int kSteps = kWaveRows / 4;            // four rows at a time
  constexpr int kBatch = 4;                        // steps whose RoPE loads are in flight together
  static_assert(kSteps % kBatch == 0, "whole batches");
  const int hl = wave / kHeadWaves;
  const int h = n0 / 128 + hl;
  const int c = lane & 15;
  const bool is_q = h < qa.hq;
  const bool is_v = h >= qa.hq + qa.hkv;
  const int kh = is_v ? h - qa.hq - qa.hkv : h - qa.hq;
  void* cache = is_v ? qa.v_cache : qa.k_cache;
  const int wrow0 = (wave % kHeadWaves) * kWaveRows + (lane >> 4);
  // slots and positions of all the wave's rows, then the RoPE values one batch ahead
  int slot[kSteps], pos[kSteps];
#pragma unroll
  for (int i = 0; i < kSteps; ++i) {
    const int row = min(m0 + wrow0 + 4 * i, m - 1);
    slot[i] = is_q ? 0 : qa.slot_mapping[row];
    pos[i] = is_v ? 0 : qa.positions[row];
  }
  float wa[4], wb[4];
  {
    const uint16_t* w = is_q ? qa.q_norm_w : qa.k_norm_w;  // v heads do not use it
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      wa[i] = bf16_to_f32(w[4 * c + i]);
      wb[i] = bf16_to_f32(w[64 + 4 * c + i]);
    }
  }
  u32x2 rope[2][kBatch][2];
  auto load_rope = [&](int b, u32x2 (&dst)[kBatch][2]) {
#pragma unroll
    for (int i = 0; i < kBatch; ++i) {
      const int64_t at = min(max(pos[b * kBatch + i], 0), qa.rope_positions - 1);
      dst[i][0] = *(const u32x2*)(qa.rope + at * 128 + 4 * c);
      dst[i][1] = *(const u32x2*)(qa.rope + at * 128 + 64 + 4 * c);
    }
  };
  load_rope(0, rope[0]);
  lds_barrier();  // the staged tile is complete
#pragma unroll
  for (int b = 0; b < kSteps / kBatch; ++b) {
    const int lrow0 = wrow0 + b * 4 * kBatch;
    if (m0 + lrow0 - (lane >> 4) >= m) return;  // wave-uniform: no rows left
    if (b + 1 < kSteps / kBatch) load_rope(b + 1, rope[(b + 1) & 1]);
    // the batch's vectors stage by stage, so that the steps' chains overlap
    float x[kBatch][4], y[kBatch][4];
#pragma unroll
    for (int i = 0; i < kBatch; ++i) {
      const char* src = smem + (lrow0 + 4 * i) * L::kRowB + hl * 256 + 8 * c;
      unpack4(*(const u32x2*)src, x[i]);
      unpack4(*(const u32x2*)(src + 128), y[i]);
    }
    if (!is_v) {
      float ss[kBatch];
#pragma unroll
      for (int i = 0; i < kBatch; ++i) {
        float leaf[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) leaf[e] = x[i][e] * x[i][e] + y[i][e] * y[i][e];
        ss[i] = (leaf[0] + leaf[1]) + (leaf[2] + leaf[3]);
      }
      row16_reduce<false, kBatch>(ss);
#pragma unroll
      for (int i = 0; i < kBatch; ++i) {
        const float inv = rsqrtf(ss[i] / 128.f + qa.eps);
        float cs[4], sn[4], xc[4], xs[4], yc[4], ys[4];
        unpack4(rope[b & 1][i][0], cs);
        unpack4(rope[b & 1][i][1], sn);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          x[i][e] *= inv;
          y[i][e] *= inv;
        }
        round4(x[i]);
        round4(y[i]);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          x[i][e] *= wa[e];
          y[i][e] *= wb[e];
        }
        round4(x[i]);
        round4(y[i]);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          xc[e] = x[i][e] * cs[e];
          xs[e] = x[i][e] * sn[e];
          yc[e] = y[i][e] * cs[e];
          ys[e] = -y[i][e] * sn[e];
        }
        round4(xc);
        round4(xs);
        round4(yc);
        round4(ys);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          x[i][e] = xc[e] + ys[e];
          y[i][e] = yc[e] + xs[e];
        }
      }
    }
    if (is_q || !kInt8) {
#pragma unroll
      for (int i = 0; i < kBatch; ++i) {
        const int row = m0 + lrow0 + 4 * i;
        uint16_t* dst = (is_q ? qa.q_out + ((int64_t)row * qa.hq + h) * 128
                              : (uint16_t*)cache + ((int64_t)slot[b * kBatch + i] * qa.hkv + kh) * 128) + 4 * c;
        if (row < m) {
          *(u32x2*)dst = pack4(x[i]);
          *(u32x2*)(dst + 64) = pack4(y[i]);
        }
      }
    } else {
      // write_vectors' quantisation: the quotient by the reciprocal (within 3e-5 of the exact
      // one), exact divisions where a lane of the batch is near a rounding tie
      float s[kBatch], tx[kBatch][4], ty[kBatch][4];
#pragma unroll
      for (int i = 0; i < kBatch; ++i) {
        round4(x[i]);
        round4(y[i]);
        s[i] = 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) s[i] = fmaxf(s[i], fmaxf(fabsf(x[i][e]), fabsf(y[i][e])));
      }
      row16_reduce<true, kBatch>(s);
      float dist = 0.f;  // the farthest of this lane's quotients from a whole number
#pragma unroll
      for (int i = 0; i < kBatch; ++i) {
        s[i] = fmaxf(s[i], 1e-8f) / 127.f;
        const float rcp = __builtin_amdgcn_rcpf(s[i]);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          tx[i][e] = x[i][e] * rcp;
          ty[i][e] = y[i][e] * rcp;
          dist = fmaxf(dist, fmaxf(fabsf(tx[i][e] - rintf(tx[i][e])), fabsf(ty[i][e] - rintf(ty[i][e]))));
        }
      }
      if (__builtin_amdgcn_ballot_w64(dist > 0.49996f) != 0) {
#pragma unroll
        for (int i = 0; i < kBatch; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            tx[i][e] = x[i][e] / s[i];
            ty[i][e] = y[i][e] / s[i];
          }
      }
#pragma unroll
      for (int i = 0; i < kBatch; ++i) {
        const uint32_t px = codes4(tx[i]), py = codes4(ty[i]);
        const int64_t vec = (int64_t)slot[b * kBatch + i] * qa.hkv + kh;
        if (m0 + lrow0 + 4 * i < m) {
          int8_t* dst = (int8_t*)cache + vec * 128 + 4 * c;
          *(uint32_t*)dst = px;
          *(uint32_t*)(dst + 64) = py;
          if (c == 0) store_scale<kSdt>(is_v ? qa.v_scale : qa.k_scale, vec, s[i]);
        }
      }
    }
  }
}

// EPI and KV as proj_kernel's (0: store, 1: SwiGLU, 4: QK-norm + RoPE + KV write).
template <typename L, int EPI, int KV>
__global__ __launch_bounds__(L::kWaves* kWave) void proj_tile_kernel(GemmParams p, QkvRopeArgs qa) {
  constexpr int PM = L::PM, NPW = L::NPW;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  asm volatile("" ::"s"(p.x), "s"(p.ldx), "s"(p.w), "s"(p.scale), "s"(p.m), "s"(p.k), "s"(p.tiles_m),
               "s"(p.tiles_n), "s"(p.y), "s"(p.ldy));
  // Each XCD takes a contiguous eighth of the tiles, in an order that walks all weight
  // tiles against groups of four row tiles: the group's X rows stay in that XCD's L2.
  const int total = p.tiles_m * p.tiles_n;
  const int per = (total + kNumXcd - 1) / kNumXcd;
  const int idx = (blockIdx.x % kNumXcd) * per + blockIdx.x / kNumXcd;
  if (idx >= total) return;
  constexpr int kGroup = 4;
  const int grp = idx / (kGroup * p.tiles_n);
  const int in_grp = idx - grp * (kGroup * p.tiles_n);
  const int rows_in = min(kGroup, p.tiles_m - grp * kGroup);
  const int tn = in_grp / rows_in;
  const int m0 = (grp * kGroup + in_grp - tn * rows_in) * L::BM;
  const int n0 = tn * L::BN;
  const int lane = threadIdx.x % kWave;
  const int r = lane & 15;
  const int g = lane >> 4;
  TileWave<L> w;
  w.wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  w.kg = w.wave / (L::MW * L::NW);
  w.mw = (w.wave / L::NW) % L::MW;
  w.nw = w.wave % L::NW;
#pragma unroll
  for (int j = 0; j < L::kCopies; ++j) {
    const int block = j / L::kPerBlock;
    const int i = (j % L::kPerBlock) * L::kWaves + w.wave;  // KiB of the block
    if (j % L::kPerBlock < L::kXPerBlock) {                 // 8 X rows x 8 chunks of 16 B
      const int row = i * 8 + (lane >> 3);
      const int chunk = (lane & 7) ^ (row & 7);
      // rows past m re-read row m - 1 and are never stored
      w.off[j] = (uint32_t)min(m0 + row, p.m - 1) * (uint32_t)(p.ldx * 2) + (uint32_t)(block * 128 + chunk * 16);
    } else {  // 16 weight rows x 4 chunks
      const int row = (i - L::kXBlock / 1024) * 16 + (lane >> 2);
      const int chunk = (lane & 3) ^ ((row >> 1) & 3);
      w.off[j] = (uint32_t)row * (uint32_t)p.k + (uint32_t)(block * 64 + chunk * 16);
    }
  }
  w.xr = (uint32_t)((w.mw * PM * 16 + r) * 128 + (((2 * g) ^ (r & 7)) * 16));
  w.wr = (uint32_t)(L::kXBlock + (w.nw * NPW * 16 + r) * 64 + ((g ^ ((r >> 1) & 3)) * 16));

  floatx4 acc[PM][NPW];
#pragma unroll
  for (int mi = 0; mi < PM; ++mi)
#pragma unroll
    for (int ns = 0; ns < NPW; ++ns) acc[mi][ns] = floatx4{0.f, 0.f, 0.f, 0.f};
  tile_mainloop<L>(p, smem, n0, w, acc);

  // the weight rows' scales: lane (r, g) stores columns 16 ns + 4 g + i of its subtiles
  float sc[NPW][4];
  tile_scales<NPW>(p, n0 + w.nw * NPW * 16 + 4 * g, sc);

  // two k-groups: group kg finishes token subtiles [kg PM / 2, + PM / 2), summed kg 0 + kg 1
  constexpr int kMine = L::KG > 1 ? PM / 2 : PM;
  if constexpr (L::KG > 1) {
    floatx4* red = (floatx4*)smem;
    auto at = [&](int from, int mi, int ns) -> floatx4& {
      return red[(((from * L::MW * L::NW + w.wave % (L::MW * L::NW)) * kMine + mi) * NPW + ns) * kWave + lane];
    };
    lds_barrier();  // every wave is past its last fragment read
#pragma unroll
    for (int mi = 0; mi < kMine; ++mi)
#pragma unroll
      for (int ns = 0; ns < NPW; ++ns) at(w.kg, mi, ns) = w.kg == 0 ? acc[kMine + mi][ns] : acc[mi][ns];
    lds_barrier();
#pragma unroll
    for (int mi = 0; mi < kMine; ++mi)
#pragma unroll
      for (int ns = 0; ns < NPW; ++ns) {
        const floatx4 other = at(1 - w.kg, mi, ns);
        acc[mi][ns] = w.kg == 0 ? acc[mi][ns] + other : other + acc[kMine + mi][ns];
      }
  }
  const int lrow0 = (w.mw * PM + (L::KG > 1 ? w.kg * kMine : 0)) * 16 + r;  // first of this lane's tile rows
  if constexpr (EPI == 4) {
    lds_barrier();  // every wave is past its last read of the ring, or of the partial sums
#pragma unroll
    for (int mi = 0; mi < kMine; ++mi)
#pragma unroll
      for (int ns = 0; ns < NPW; ++ns) {
        const floatx4 v = acc[mi][ns];
        *(u32x2*)(smem + (lrow0 + mi * 16) * L::kRowB + ((w.nw * NPW + ns) * 16 + 4 * g) * 2) =
            u32x2{pack_bf16x2(v[0] * sc[ns][0], v[1] * sc[ns][1]), pack_bf16x2(v[2] * sc[ns][2], v[3] * sc[ns][3])};
      }
    tile_qkv_epilogue<L, KV>(qa, smem, p.m, m0, n0, w.wave, lane);
    return;
  }
  const bool wide = ((uintptr_t)p.y % 16) == 0 && p.ldy % 8 == 0;
#pragma unroll
  for (int mi = 0; mi < kMine; ++mi) {
    const int m = m0 + lrow0 + mi * 16;
    // the row's 16-column output subtiles in pairs: with 16-byte aligned rows one store each
    constexpr int kOut = EPI == 1 ? NPW / 2 : NPW;
    static_assert(kOut % 2 == 0, "output subtiles in pairs");
    uint16_t* dst = p.y + (int64_t)m * p.ldy + (EPI == 1 ? n0 / 2 : n0) + w.nw * kOut * 16;
    auto out4 = [&](int o) {
      if constexpr (EPI == 1) return swiglu4(acc[mi][2 * o], acc[mi][2 * o + 1], sc[2 * o], sc[2 * o + 1]);
      const floatx4 v = acc[mi][o];
      return u32x2{pack_bf16x2(v[0] * sc[o][0], v[1] * sc[o][1]), pack_bf16x2(v[2] * sc[o][2], v[3] * sc[o][3])};
    };
#pragma unroll
    for (int o = 0; o < kOut; o += 2) {
      const u32x2 x = out4(o), y = out4(o + 1);
      if (wide) {
        const u32x4 both = pair_columns(x, y);
        if (m < p.m) *(u32x4*)(dst + o * 16 + pair_column(g)) = both;
      } else if (m < p.m) {
        *(u32x2*)(dst + o * 16 + 4 * g) = x;
        *(u32x2*)(dst + (o + 1) * 16 + 4 * g) = y;
      }
    }
  }
}

template <typename L, int EPI, int KV>
int launch_proj_tile_as(GemmParams p, hipStream_t stream, const char* name, const QkvRopeArgs& qa) {
  p.tiles_m = ceil_div(p.m, L::BM);
  p.tiles_n = p.n / L::BN;
  const int per = ceil_div((int64_t)p.tiles_m * p.tiles_n, kNumXcd);
  static const hipError_t attr = hipFuncSetAttribute((const void*)proj_tile_kernel<L, EPI, KV>,
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, L::kLds);
  if (attr != hipSuccess) {
    set_error("%s: cannot reserve %d bytes of LDS: %s", name, L::kLds, hipGetErrorString(attr));
    return NE_ELAUNCH;
  }
  hipLaunchKernelGGL((proj_tile_kernel<L, EPI, KV>), dim3((unsigned)(per * kNumXcd)), dim3(L::kWaves * kWave),
                     L::kLds, stream, p, qa);
  return check_launch(name);
}

using Tile256x256 = TileLayout<256, 256, 2, 4, 1>;
using Tile128x256 = TileLayout<128, 256, 2, 4, 1>;
using Tile128x128 = TileLayout<128, 128, 2, 2, 2>;

enum class ProjTile { kVerify, k128x128, k128x256, k256x256 };

// The kernel of a product without split-K: the least rounds of one tile per CU times what a
// round costs per 64 k.  Costs in us, measured at N = 1,024-6,144, K = 1,024-3,072 and 320-
// 8,192 rows: 2.3 (256 x 256), 1.32 (128 x 256), 0.8 (128 x 128) and, for the verify step's
// kernel, 0.39 (80 x 64) or 0.45 (SwiGLU's 80 x 96) with rounds that overlap.  At 512 rows
// of N = 4,096 that kernel takes 12.6 us and 128 x 128 tiles 14.0, at 1,024 rows 22.9 and
// 15.7; 2,048 rows of o 24.3 and 23.3, 4,096 rows 49 and 25.  From N = 16,384 on the tiles also
// win below 320 rows (K = 1,024: 200 rows of 16,384 18.2 and 14.8, 81 of 32,768 25.2 and 15.9,
// 33 of 65,536 26.4 and 22.8, 17 of 131,072 47.9 and 43.2; 17 of 65,536 over K = 2,048 45.2 and
// 40.8); up to 16 rows the few-rows kernel goes first (16 of 65,536: 18.6, tiles 22.6).  The
// fused QKV product follows the plain product's choice, so that both sum in one order and round
// to the same bits.
ProjTile choose_proj_tile(int m, int n, bool swiglu) {
  const auto rounds = [&](int bm, int bn) {
    return (int64_t)ceil_div((int64_t)ceil_div(m, bm) * (n / bn), kNumCu);
  };
  const int verify_n = swiglu && n % 96 == 0 ? 96 : 64;
  const double verify_tiles = (double)ceil_div(m, kPM * 16) * (n / verify_n) / kNumCu;
  double best = (verify_tiles > 1.0 ? verify_tiles : 1.0) * (verify_n == 96 ? 0.45 : 0.39);
  ProjTile tile = ProjTile::kVerify;
  const auto offer = [&](ProjTile t, int bm, int bn, double cost) {
    if (n % bn != 0 || rounds(bm, bn) * cost >= best) return;
    best = rounds(bm, bn) * cost;
    tile = t;
  };
  offer(ProjTile::k128x128, 128, 128, 0.8);
  offer(ProjTile::k128x256, 128, 256, 1.32);
  offer(ProjTile::k256x256, 256, 256, 2.3);
  return tile;
}

template <int EPI, int KV>
int launch_proj_tile(ProjTile tile, const GemmParams& p, hipStream_t s, const char* name,
                     const QkvRopeArgs& qa = QkvRopeArgs{}) {
  if (tile == ProjTile::k256x256) return launch_proj_tile_as<Tile256x256, EPI, KV>(p, s, name, qa);
  if (tile == ProjTile::k128x256) return launch_proj_tile_as<Tile128x256, EPI, KV>(p, s, name, qa);
  return launch_proj_tile_as<Tile128x128, EPI, KV>(p, s, name, qa);
}

// ---- W8A16 projections of few rows -----------------------------------------------------
// At up to 16 rows a work-group of the kernel above spends its time in a chain of stages
// (copy, barrier, read, convert, multiply, ~0.5 us each) that hold a dozen MFMAs.  Here
// nothing is staged: X (all of K, at most 32 KB) is copied to LDS once, every wave loads all
// of its weight rows' K into registers in one burst, in the MFMA operand order, and then
// multiplies as they arrive.  One barrier, one memory round trip.
//   wave  = NPW weight subtiles of 16 rows x all PM token subtiles x K = 128 KT
//   sums  = KG accumulators per output (k-step kk of a stage goes to accumulator kk KG / 4),
//           added in order: the k-groups of the kernel above, so the results are its bits
// Measured at 5 rows (kernel trace, fastest of 28; us, before -> here): QKV 8.7 -> 7.8,
// gate|up 7.0 -> 6.4, o 4.5 -> 2.9, down 4.6 -> 3.9; four layers from a HIP graph 174-177
// -> 167-171.  What is left is the launch, one round trip to HBM and, for QKV, 128 KB of weights
// into each of 32 CUs.
template <int PM_, int NPW_, int KG_, int WAVES_, int KT_>
struct FewLayout {
  static constexpr int PM = PM_, NPW = NPW_, KG = KG_, WAVES = WAVES_, KT = KT_;
  static constexpr int kRows = PM * 16;
  static constexpr int kStage = kRows * 256;         // X rows of a 128-wide stage
  static constexpr int kX = KT * kStage;
  static constexpr int kCopies = KT * PM * 4;        // 1 KiB copies: 4 rows of 256 B
  static constexpr int kPerWave = (kCopies + WAVES - 1) / WAVES;
  static constexpr int kLoads = NPW * KT * 2;        // 16-byte weight loads per lane
  static constexpr int kRowF = 132;                  // floats per row of the QKV epilogue's fp32 rows
  static constexpr int kLds = kX > kRows * kRowF * 4 ? kX : kRows * kRowF * 4;
  static_assert(kLoads < 64, "vmcnt range");
  static_assert(kLds <= 160 * 1024, "LDS");
};

template <typename L, int EPI, int KV>
__global__ __launch_bounds__(L::WAVES* kWave) void proj_few_rows_kernel(GemmParams p, float* partial, QkvRopeArgs qa) {
  constexpr int PM = L::PM, NPW = L::NPW, KG = L::KG, KT = L::KT;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  asm volatile("" ::"s"(p.x), "s"(p.ldx), "s"(p.w), "s"(p.scale), "s"(p.m), "s"(p.k), "s"(p.n), "s"(p.y), "s"(p.ldy));
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int lane = threadIdx.x % kWave;
  const int r = lane & 15;
  const int g = lane >> 4;
  const int n0 = (blockIdx.x * L::WAVES + wave) * NPW * 16;  // this wave's first weight row
  const int kbase = blockIdx.y * KT * kStageK;

  // ---- X to LDS: stage t, row, 16-byte chunk c at position c ^ (row % 16) ----
  {
    const char* xsrc = uniform_ptr((const char*)p.x + (int64_t)kbase * 2);
#pragma unroll
    for (int j = 0; j < L::kPerWave; ++j) {
      const int i = j * L::WAVES + wave;  // KiB: stage i / (4 PM), rows 4 (i % (4 PM)) .. + 4
      if (L::kCopies % L::WAVES != 0 && i >= L::kCopies) break;  // wave-uniform
      const int t = i / (4 * PM);
      const int row = (i % (4 * PM)) * 4 + (lane >> 4);
      // rows past m re-read row m - 1 and are never stored
      const uint32_t off = (uint32_t)min(row, p.m - 1) * (uint32_t)(p.ldx * 2) +
                           (uint32_t)(t * 256 + (((lane & 15) ^ (row & 15)) * 16));
      lds_dma16(xsrc + off, smem + i * 1024);
    }
  }
  __asm__ __volatile__("" ::: "memory");  // the X copies are older than the weight loads
  // ---- weights: bytes 128 t + 64 h + 16 g of row r of each subtile feed k-steps 2 h, 2 h + 1 ----
  u32x4 wf[KT][2][NPW];
  {
    const char* wsrc = (const char*)p.w + (int64_t)(n0 + r) * p.k + kbase + 16 * g;
#pragma unroll
    for (int t = 0; t < KT; ++t)
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int ns = 0; ns < NPW; ++ns)
          wf[t][h][ns] = *(const u32x4*)(wsrc + (int64_t)ns * 16 * p.k + t * 128 + 64 * h);
  }
  __asm__ __volatile__("" ::: "memory");
  // EPI 4: wave w finishes rows w, w + WAVES, .. of the head; their slots and positions
  // (scalar loads) now, their RoPE values behind the weights
  constexpr int N = EPI == 4 ? L::kRows / L::WAVES : 1;
  const int head = blockIdx.x;
  int64_t slot_e[N];
  int pos_e[N];
  if constexpr (EPI == 4) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int m = min(wave + L::WAVES * i, p.m - 1);
      slot_e[i] = ((const ConstI32*)qa.slot_mapping)[m];
      pos_e[i] = ((const ConstI32*)qa.positions)[m];
    }
  }
  wait_vmcnt<L::kLoads>();  // this wave's X copies have landed
  asm volatile("s_barrier" ::: "memory");
  uint16_t rc_e[N], rs_e[N], nw_e[2] = {0, 0};
  if constexpr (EPI == 4) {
    const uint16_t* w = head < qa.hq ? qa.q_norm_w : qa.k_norm_w;  // v heads do not use it
    nw_e[0] = w[lane];
    nw_e[1] = w[lane + 64];
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int64_t pos = min(max(pos_e[i], 0), qa.rope_positions - 1);
      rc_e[i] = qa.rope[pos * 128 + lane];
      rs_e[i] = qa.rope[pos * 128 + 64 + lane];
    }
  }
  // the weight rows' scales as they are, behind the weights too (converted at the end: a
  // conversion here would wait for every load)
  uint32_t raw_sc[NPW][4];
#pragma unroll
  for (int ns = 0; ns < NPW; ++ns)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int at = n0 + 4 * g + ns * 16 + i;
      raw_sc[ns][i] = p.scale_dtype == NE_DTYPE_FP32 ? ((const uint32_t*)p.scale)[at] : ((const uint16_t*)p.scale)[at];
    }

  floatx4 acc[KG][PM][NPW];
#pragma unroll
  for (int q = 0; q < KG; ++q)
#pragma unroll
    for (int mi = 0; mi < PM; ++mi)
#pragma unroll
      for (int ns = 0; ns < NPW; ++ns) acc[q][mi][ns] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int t = 0; t < KT; ++t)
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      u32x4 xf[PM];
#pragma unroll
      for (int mi = 0; mi < PM; ++mi)
        xf[mi] = *(const u32x4*)(smem + t * L::kStage + (mi * 16 + r) * 256 +
                                 (((8 * (kk >> 1) + 2 * g + (kk & 1)) ^ r) * 16));
#pragma unroll
      for (int ns = 0; ns < NPW; ++ns) {
        const u32x4 w = wf[t][kk >> 1][ns];
        const bf16x8 a = int8x8_to_bf16x8(w[2 * (kk & 1)], w[2 * (kk & 1) + 1]);
#pragma unroll
        for (int mi = 0; mi < PM; ++mi)
          acc[kk * KG / 4][mi][ns] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              a, __builtin_bit_cast(bf16x8, xf[mi]), acc[kk * KG / 4][mi][ns], 0, 0, 0);
      }
    }

  float sc[NPW][4];
#pragma unroll
  for (int ns = 0; ns < NPW; ++ns)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t b = raw_sc[ns][i];
      sc[ns][i] = p.scale_dtype == NE_DTYPE_FP32   ? __uint_as_float(b)
                  : p.scale_dtype == NE_DTYPE_BF16 ? bf16_to_f32((uint16_t)b)
                                                   : f16_to_f32((uint16_t)b);
    }
  floatx4 v[PM][NPW];
#pragma unroll
  for (int mi = 0; mi < PM; ++mi)
#pragma unroll
    for (int ns = 0; ns < NPW; ++ns) {
      v[mi][ns] = acc[0][mi][ns];
#pragma unroll
      for (int q = 1; q < KG; ++q) v[mi][ns] += acc[q][mi][ns];
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if constexpr (EPI != 1) v[mi][ns][i] *= sc[ns][i];
    }

  if constexpr (EPI == 4) {
    // the head's rows through LDS (fp32 [row][128 + 4], over X once every wave has read it),
    // then wave w takes rows w, w + WAVES, .. as the row kernel does
    static_assert(NPW == 1 && L::WAVES == 8, "one head per work-group");
    constexpr int kRowF = L::kRowF;
    float* rows = (float*)smem;
    lds_barrier();
#pragma unroll
    for (int mi = 0; mi < PM; ++mi) *(floatx4*)(rows + (mi * 16 + r) * kRowF + wave * 16 + 4 * g) = v[mi][0];
    lds_barrier();
    int rows_e[N];
    bool valid_e[N];
    float a_e[N], b_e[N], c_e[N], s_e[N];
#pragma unroll
    for (int i = 0; i < N; ++i) {
      rows_e[i] = wave + L::WAVES * i;
      valid_e[i] = rows_e[i] < p.m;
      a_e[i] = bf16_round(rows[rows_e[i] * kRowF + lane]);
      b_e[i] = bf16_round(rows[rows_e[i] * kRowF + 64 + lane]);
      c_e[i] = bf16_to_f32(rc_e[i]);
      s_e[i] = bf16_to_f32(rs_e[i]);
    }
    qk_norm_rope_kv_vectors<(KV >= 2), KV == 3 ? NE_DTYPE_FP16 : NE_DTYPE_BF16, N>(
        qa, rows_e, valid_e, head, lane, a_e, b_e, slot_e, bf16_to_f32(nw_e[0]), bf16_to_f32(nw_e[1]), c_e, s_e);
    return;
  }
#pragma unroll
  for (int mi = 0; mi < PM; ++mi) {
    const int m = mi * 16 + r;
    if (m >= p.m) continue;
    if constexpr (EPI == 0) {
#pragma unroll
      for (int ns = 0; ns < NPW; ++ns)
        *(u32x2*)(p.y + (int64_t)m * p.ldy + n0 + ns * 16 + 4 * g) =
            u32x2{pack_bf16x2(v[mi][ns][0], v[mi][ns][1]), pack_bf16x2(v[mi][ns][2], v[mi][ns][3])};
    } else if constexpr (EPI == 1) {
      static_assert(NPW == 2, "a wave holds paired gate / up subtiles");
      *(u32x2*)(p.y + (int64_t)m * p.ldy + n0 / 2 + 4 * g) = swiglu4(v[mi][0], v[mi][1], sc[0], sc[1]);
    } else {
#pragma unroll
      for (int ns = 0; ns < NPW; ++ns)
        *(floatx4*)(partial + ((int64_t)blockIdx.y * p.m + m) * p.n + n0 + ns * 16 + 4 * g) = v[mi][ns];
    }
  }
}

template <typename L, int EPI, int KV>
int launch_few_as(const GemmParams& p, int splits, float* partial, hipStream_t stream, const char* name,
                  const QkvRopeArgs& qa) {
  static const hipError_t attr = hipFuncSetAttribute((const void*)proj_few_rows_kernel<L, EPI, KV>,
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, L::kLds);
  if (attr != hipSuccess) {
    set_error("%s: cannot reserve %d bytes of LDS: %s", name, L::kLds, hipGetErrorString(attr));
    return NE_ELAUNCH;
  }
  hipLaunchKernelGGL((proj_few_rows_kernel<L, EPI, KV>),
                     dim3((unsigned)(p.n / (L::WAVES * L::NPW * 16)), (unsigned)splits), dim3(L::WAVES * kWave), L::kLds,
                     stream, p, partial, qa);
  return check_launch(name);
}

// Wave layouts (k-groups, weight subtiles per wave).  The plain and split-K products and
// the fused QKV projection share two k-groups, so the fused epilogue sums every output in
// the order the plain GEMM does and both round to the same bits; SwiGLU pairs gate and
// up subtiles in one wave and keeps four k-groups to keep 12 waves.
constexpr int kKgPlain = 2, kNpwPlain = 1;
constexpr int kKgQkv = 2, kNpwQkv = 2;
constexpr int kKgSwiglu = 4, kNpwSwiglu = 2;

// Whether the few-rows kernel serves a product: one token subtile, and a K (per split) of up
// to kFewMaxStages stages, whose weights a wave holds in registers (128 of them for SwiGLU's
// two subtiles).  Per launch at 5 rows, weights in turn from a HIP graph (us, staged -> here):
// N = 4,096 K = 128 3.5 -> 2.6, 384 4.7 -> 3.3, 640 5.7 -> 3.9, 896 6.7 -> 5.0, 1,024 6.2 -> 5.3;
// SwiGLU N = 6,144 4.5 -> 3.3, 5.8 -> 4.3, 7.2 -> 5.7, 8.4 -> 6.9 and 7.6 -> 7.6; four splits of
// them at N = 1,024 3.2 -> 2.7, 4.2 -> 3.3, 5.0 -> 3.9, 5.9 -> 4.9 and 5.2 -> 5.3.  A larger K
// would need a second burst behind the first.  With three subtiles it lost to the staged kernel at 48 rows (QKV 10.4 ->
// 12.2 us, gate|up 8.2 -> 9.4, down 5.6 -> 6.8: every wave then waits for 96 KB of X before its
// first product).
constexpr int kFewMaxStages = 8;
bool few_rows(const GemmParams& p, int splits) { return p.m <= 16 && p.k / splits <= kFewMaxStages * kStageK; }

template <int NPW, int KG, int WAVES, int EPI, int KV, int KT = kFewMaxStages>
int launch_few(const GemmParams& p, int splits, float* partial, hipStream_t s, const char* name,
               const QkvRopeArgs& qa = QkvRopeArgs{}) {
  if constexpr (KT > 1) {
    if (p.k / splits / kStageK < KT)
      return launch_few<NPW, KG, WAVES, EPI, KV, KT - 1>(p, splits, partial, s, name, qa);
  }
  return launch_few_as<FewLayout<1, NPW, KG, WAVES, KT>, EPI, KV>(p, splits, partial, s, name, qa);
}

template <int SDT>
int dispatch_qkv_fused(GemmParams p, const QkvRopeArgs& qa, int kv_mode, hipStream_t s) {
  const char* name = "w8a16_qkv_norm_rope_kv";
  const bool few = few_rows(p, 1);
  // the tiles' epilogue stores 4 or 8 bytes at a time where the row kernel's stores elements
  const bool aligned = (((uintptr_t)qa.q_out | (uintptr_t)qa.rope | (uintptr_t)qa.k_cache | (uintptr_t)qa.v_cache) % 8) == 0;
  const ProjTile tile = !few && aligned ? choose_proj_tile(p.m, p.n, false) : ProjTile::kVerify;
  if (!few && tile == ProjTile::kVerify) {
    switch (kv_mode) {
      // 48-row tiles: 7 x 32 = 224 work-groups for 320 rows, 3 rows per wave in the epilogue
      case 1: return launch_proj<8, SDT, 4, 1, 3, kKgQkv, kNpwQkv>(p, 1, nullptr, s, name, qa);
      case 2: return launch_proj<8, SDT, 4, 2, 3, kKgQkv, kNpwQkv>(p, 1, nullptr, s, name, qa);
      default: return launch_proj<8, SDT, 4, 3, 3, kKgQkv, kNpwQkv>(p, 1, nullptr, s, name, qa);
    }
  }
  if (few) {
    if (kv_mode == 1) return launch_few<1, kKgQkv, 8, 4, 1>(p, 1, nullptr, s, name, qa);
    if (kv_mode == 2) return launch_few<1, kKgQkv, 8, 4, 2>(p, 1, nullptr, s, name, qa);
    return launch_few<1, kKgQkv, 8, 4, 3>(p, 1, nullptr, s, name, qa);
  }
  if (kv_mode == 1) return launch_proj_tile<4, 1>(tile, p, s, name, qa);
  if (kv_mode == 2) return launch_proj_tile<4, 2>(tile, p, s, name, qa);
  return launch_proj_tile<4, 3>(tile, p, s, name, qa);
}

template <int SDT>
int dispatch_w8a16(GemmParams p, int epilogue, int splits, float* partial, hipStream_t s) {
  const bool swiglu = epilogue == NE_EPILOGUE_SWIGLU;
  const bool few = few_rows(p, partial != nullptr ? splits : 1);
  const ProjTile tile = !few && partial == nullptr ? choose_proj_tile(p.m, p.n, swiglu) : ProjTile::kVerify;
  if (!few && tile == ProjTile::kVerify) {
    if (swiglu) {
      if (p.n % 96 == 0)
        return launch_proj<6, SDT, 1, 0, kPM, kKgSwiglu, kNpwSwiglu>(p, 1, nullptr, s, "w8a16_swiglu");
      return launch_proj<4, SDT, 1, 0, kPM, kKgSwiglu, kNpwSwiglu>(p, 1, nullptr, s, "w8a16_swiglu");
    }
    if (partial != nullptr)
      return launch_proj<4, SDT, 3, 0, kSplitPM, kKgPlain, kNpwPlain>(p, splits, partial, s, "w8a16_splitk");
    return launch_proj<4, SDT, 0, 0, kPM, kKgPlain, kNpwPlain>(p, 1, nullptr, s, "w8a16_gemm");
  }
  if (few) {
    if (swiglu) return launch_few<2, kKgSwiglu, 2, 1, 0>(p, 1, nullptr, s, "w8a16_swiglu");
    if (partial != nullptr) return launch_few<1, kKgPlain, 2, 3, 0>(p, splits, partial, s, "w8a16_splitk");
    return launch_few<1, kKgPlain, 2, 0, 0>(p, 1, nullptr, s, "w8a16_gemm");
  }
  return swiglu ? launch_proj_tile<1, 0>(tile, p, s, "w8a16_swiglu") : launch_proj_tile<0, 0>(tile, p, s, "w8a16_gemm");
}

// ---- LM head: persistent work-groups over the vocabulary -------------------------
// logits = X . W^T for X [m, k] bf16 and the tied embedding W [vocab, k] bf16, plus
// argmax partials: per row, one (value, index) key for each half of each work-group's
// column range (the range's 128-column halves of every block, kept as a running
// maximum, so that the acceptance kernel reduces 512 keys per row, not one per 64
// columns).  Inside the kernel a key is 32 bits: a 16-bit order code of the bf16 value
// over 16 bits of column within the range.  The weight (311 MB for 151936 x 1024) is
// read from HBM once; what limits a tiled GEMM at m = 320 is the L2 -> CU traffic
// of X, which every column tile re-reads (about 2.3 GB over 64 x 128 tiles).  So
// one work-group per CU owns a contiguous range of 64-column groups and walks it in
// blocks of 256 columns against all rows at once: 8 waves, wave (mw, nw) holding
// rows 80 mw .. +80 and columns 128 nw .. +128 of the block in 160 accumulators,
// which cuts the X traffic to one read per 256 columns.  K advances in stages of 64
// (X 40 KiB + W 32 KiB) copied by DMA into a two-stage LDS ring: right after the
// barrier that frees a slot, every wave issues 9 copies of the next stage, 5 of X and 4
// of W, then runs its 80 MFMAs on the current one.  Spreading the weight copies (HBM
// misses) over all waves keeps any one wave from queueing behind them; the two waves of
// a SIMD still finish a stage apart, the older one ahead.  Stages run on across
// blocks.  The logits leave in 16-byte stores (two subtiles regrouped by pair_columns), and
// the stage after a full block waits for its copies only, not for those stores: 320 rows'
// logits 127 -> 122.5 us (their argmax partials alone take ~115).  Holding each next k-step's
// fragments in registers through the current one's MFMAs, as the prefill tiles do, was
// slower (151 us): a wave's reads then wait for each other in order.  A range of ~9.3 groups
// ends in a short block of one or two groups: there the waves whose 128 columns are all past
// the end skip their MFMAs and the weight copies of absent rows are not issued (~23 % of the
// MFMAs were on such columns).  Rows beyond m re-read row m - 1 and are never stored; more
// than 320 rows take further passes.
constexpr int kLmMaxGrid = 256;  // persistent work-groups (one per CU)
constexpr int kLmRows = 320;
constexpr int kLmCols = 256;
constexpr int kLmWaves = 8;
constexpr int kLmSK = 64;
constexpr int kLmRing = 2;
constexpr int kLmXBytes = kLmRows * kLmSK * 2;   // 40 KiB
constexpr int kLmWBytes = kLmCols * kLmSK * 2;   // 32 KiB
constexpr int kLmStage = kLmXBytes + kLmWBytes;
constexpr int kLmInstr = kLmStage / 1024 / kLmWaves;  // DMA instructions per wave per stage (9)
static_assert(kLmStage % (1024 * kLmWaves) == 0, "stage split over waves");

struct LmStage {
  int m0, c0, ccols, k0;
};

// This wave's 9 copies of a stage: copy j moves 8 rows of 128 bytes (64 bf16) into LDS
// slot i = 8 j + wave, so copies 0..4 of every wave are X slots (i < 40) and 5..8 weight
// slots; row r keeps its 16-byte chunk c at position c ^ (r & 7).  A copy's source is a
// scalar base for the stage (X: k0; W: the block's first column and k0) plus a 32-bit
// lane offset that depends only on the pass's first row (X) or the block's width (W), so
// a stage's copies need no 64-bit arithmetic.
constexpr int kLmFullStores = 40;  // 16-byte stores per wave of a full block's logits (5 x 8 / 2 subtile pairs)
constexpr int kLmXCopies = kLmXBytes / 1024 / kLmWaves;  // 5
static_assert(kLmXBytes % (1024 * kLmWaves) == 0, "X slots split evenly over the waves");

struct LmCopies {
  uint32_t off[kLmInstr];
};

__device__ __forceinline__ void lm_offsets(const GemmParams& p, const LmStage& st, int wave, int lane,
                                           LmCopies& c) {
#pragma unroll
  for (int j = 0; j < kLmInstr; ++j) {
    const int i = j * kLmWaves + wave;
    if (j < kLmXCopies) {
      const int row = i * 8 + (lane >> 3);
      const int chunk = (lane & 7) ^ (row & 7);
      const int grow = min(st.m0 + row, p.m - 1);
      c.off[j] = (uint32_t)grow * (uint32_t)(p.ldx * 2) + (uint32_t)chunk * 16u;
    } else {
      const int wrow = (i - kLmXBytes / 1024) * 8 + (lane >> 3);
      const int chunk = (lane & 7) ^ (wrow & 7);
      // a short block re-reads its last column
      c.off[j] = (uint32_t)min(wrow, st.ccols - 1) * (uint32_t)(p.k * 2) + (uint32_t)chunk * 16u;
    }
  }
}

__device__ __forceinline__ void lm_issue(const GemmParams& p, char* stage, const LmStage& st, const LmCopies& c,
                                         int wave) {
  const char* xsrc = uniform_ptr((const char*)p.x + st.k0 * 2);
  const char* wsrc = uniform_ptr((const char*)p.w + ((int64_t)st.c0 * p.k + st.k0) * 2);
#pragma unroll
  for (int j = 0; j < kLmInstr; ++j) {
    // weight slot j * 8 + wave - 40 holds rows (slot) 8 .. + 8 of the block: not copied when
    // they are all past a short block's end (those rows' MFMA outputs are never used)
    if (j >= kLmXCopies && (j * kLmWaves + wave - kLmXBytes / 1024) * 8 >= st.ccols) continue;
    uint32_t o = c.off[j];
    __asm__("" : "+v"(o));  // scalar base + 32-bit lane offset addressing
    lds_dma16((j < kLmXCopies ? xsrc : wsrc) + o, stage + (j * kLmWaves + wave) * 1024);
  }
}

__device__ __forceinline__ bf16x8 lm_frag(const char* base, int row, int chunk) {
  return __builtin_bit_cast(bf16x8, *(const u32x4*)(base + row * 128 + ((chunk ^ (row & 7)) * 16)));
}

// A stage's 80 MFMAs: two k-steps of 32 (lane group g holds k = 32 s + 8 g .. +8), the
// X fragment of token subtile mi + 1 read while the MFMAs of subtile mi run.
__device__ __forceinline__ void lm_mma(const char* stage, int mw, int nw, int lane, floatx4 (&acc)[5][8]) {
  const int r = lane & 15;
  const int g = lane >> 4;
  const char* xs = stage;
  const char* ws = stage + kLmXBytes;
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    bf16x8 b[8];
#pragma unroll
    for (int ns = 0; ns < 8; ++ns) b[ns] = lm_frag(ws, nw * 128 + ns * 16 + r, 4 * s + g);
    bf16x8 a = lm_frag(xs, mw * 80 + r, 4 * s + g);
#pragma unroll
    for (int mi = 0; mi < 5; ++mi) {
      bf16x8 an = a;
      if (mi < 4) an = lm_frag(xs, mw * 80 + (mi + 1) * 16 + r, 4 * s + g);
#pragma unroll
      for (int ns = 0; ns < 8; ++ns)
        acc[mi][ns] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[ns], a, acc[mi][ns], 0, 0, 0);
      a = an;
    }
  }
}

// A bf16 pair (lo in bits 0..15) as two unsigned 16-bit codes in value order: positives
// 0x8000 + magnitude, negatives 0x8000 - magnitude, so -0 and +0 share 0x8000 (as
// torch.argmax treats them) and any finite value codes above 0.
__device__ __forceinline__ uint32_t bf16x2_order(uint32_t pair) {
  typedef short s16x2 __attribute__((ext_vector_type(2)));
  typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
  const uint32_t sgn = __builtin_bit_cast(uint32_t, __builtin_bit_cast(s16x2, pair) >> (short)15);
  const uint32_t t = pair ^ ((sgn & 0x7FFF7FFFu) | 0x80008000u);
  return __builtin_bit_cast(uint32_t, __builtin_bit_cast(u16x2, t) - __builtin_bit_cast(u16x2, sgn));
}

// What a block's end writes, each in a kernel without the others' code (a call of one short
// block per work-group feels the instruction fetches): the argmax partials alone, logits in
// 8-byte stores, or logits whose full blocks leave in 16-byte stores.
enum class LmOut { kArgmax, kLogits, kWideLogits };
template <LmOut OUT>
__global__ __launch_bounds__(kLmWaves * kWave) void lm_head_kernel(GemmParams p) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int lane = threadIdx.x % kWave;
  const int mw = wave & 3;
  const int nw = wave >> 2;
  const int r = lane & 15;
  const int g = lane >> 4;
  // this work-group's 64-column groups [grp0, grp1)
  const int groups = p.n / kArgmaxCols;
  const int grp0 = (int)((int64_t)groups * blockIdx.x / gridDim.x);
  const int grp1 = (int)((int64_t)groups * (blockIdx.x + 1) / gridDim.x);
  const int nblk = (grp1 - grp0 + 3) / 4;
  const int kt = p.k / kLmSK;
  const int mpass = (p.m + kLmRows - 1) / kLmRows;
  const int total = mpass * nblk * kt;  // stages, in order pass, block, k
  if (total == 0) return;
  // stages advance by counters (pass, block, k), so no stage needs a division
  auto make = [&](int pass, int bi, int t) {
    LmStage st;
    st.m0 = pass * kLmRows;
    st.c0 = (grp0 + 4 * bi) * kArgmaxCols;
    st.ccols = min(4, grp1 - grp0 - 4 * bi) * kArgmaxCols;
    st.k0 = t * kLmSK;
    return st;
  };
  int pass = 0, bi = 0, t = 0;
  // per token subtile: the best (value, index) key of row 16 mi + r over this wave's
  // columns of the pass so far; written once per pass as partial (row, 2 block + nw)
  // per token subtile: (order code << 16) | (0xFFFF - column within the range) of the best
  // value of row 16 mi + r over this lane's columns of the pass so far (0: none yet)
  uint32_t row_best[5] = {0, 0, 0, 0, 0};
  const int rc0 = grp0 * kArgmaxCols;
  const int tiles = 2 * (int)gridDim.x;

  floatx4 acc[5][8];
#pragma unroll
  for (int mi = 0; mi < 5; ++mi)
#pragma unroll
    for (int ns = 0; ns < 8; ++ns) acc[mi][ns] = floatx4{0.f, 0.f, 0.f, 0.f};

  LmStage cur = make(0, 0, 0);
  LmCopies copies;
  lm_offsets(p, cur, wave, lane, copies);
  int off_m0 = cur.m0, off_cols = cur.ccols;  // what the offsets were built for
  lm_issue(p, smem, cur, copies, wave);
  constexpr bool LOGITS = OUT != LmOut::kArgmax, WIDE = OUT == LmOut::kWideLogits;
  bool stores = false;  // the last block's stores may still be in flight
  for (int u = 0; u < total; ++u) {
    // this wave's copies of stage u (older than the last block's stores, if any)
    if (WIDE && stores) {
      wait_vmcnt<kLmFullStores>();
      stores = false;
    } else {
      wait_vmcnt<0>();
    }
    asm volatile("s_barrier" ::: "memory");           // everyone's; stage u - 1 fully read
    const bool more = u + 1 < total;
    int npass = pass, nbi = bi, nt = t + 1;
    if (nt == kt) {
      nt = 0;
      if (++nbi == nblk) {
        nbi = 0;
        ++npass;
      }
    }
    const LmStage nst = more ? make(npass, nbi, nt) : cur;
    if (more && (nst.m0 != off_m0 || nst.ccols != off_cols)) {
      lm_offsets(p, nst, wave, lane, copies);
      off_m0 = nst.m0;
      off_cols = nst.ccols;
    }
    const int cur_cols = cur.ccols;
    if (more) lm_issue(p, smem + ((u + 1) & 1) * kLmStage, nst, copies, wave);
    if (nw * 128 < cur_cols) lm_mma(smem + (u & 1) * kLmStage, mw, nw, lane, acc);
    const bool block_done = t == kt - 1;
    const bool pass_done = block_done && (!more || npass != pass);
    const LmStage st = cur;
    cur = nst;
    pass = npass;
    bi = nbi;
    t = nt;
    if (!block_done) continue;

    // ---- block done: logits and argmax partials, then clear the accumulators ----
    // a lane's 32 values of a row are ranked by (order code << 16) | (31 - position),
    // position 4 ns + i in column order, then turned into a range column once per row
    const int ngrp = st.ccols / kArgmaxCols;
    const uint32_t col0 = (uint32_t)(st.c0 - rc0 + nw * 128 + 4 * g);
    const bool pairs = WIDE && ngrp == 4;  // a range's short last block keeps 8-byte stores
    if (pairs) {
      // a block whose rows and columns are all there: its 40 stores per wave are known, so
      // the next stage waits for its copies (issued before them) and not for the stores
      stores = st.m0 + kLmRows <= p.m;
      const int row = st.m0 + mw * 80 + r;
      uint16_t* dst = p.y + (int64_t)row * p.ldy + st.c0 + nw * 128 + pair_column(g);
#pragma unroll
      for (int mi = 0; mi < 5; ++mi)
#pragma unroll
        for (int ns = 0; ns < 8; ns += 2) {
          const floatx4 v = acc[mi][ns], w = acc[mi][ns + 1];
          const u32x4 both = pair_columns(u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])},
                                          u32x2{pack_bf16x2(w[0], w[1]), pack_bf16x2(w[2], w[3])});
          if (row + mi * 16 < p.m)
            *(u32x4*)(dst + (int64_t)mi * 16 * p.ldy + ns * 16) = both;
        }
    }
#pragma unroll
    for (int mi = 0; mi < 5; ++mi) {
      const int m = st.m0 + mw * 80 + mi * 16 + r;
      uint32_t best = 0;
#pragma unroll
      for (int q = 0; q < 2; ++q) {  // the wave's two 64-column groups
        const int grp = 2 * nw + q;
#pragma unroll
        for (int nq = 0; nq < 4; ++nq) {
          const int ns = 4 * q + nq;
          const int n = st.c0 + nw * 128 + ns * 16 + 4 * g;
          const floatx4 v = acc[mi][ns];
          const u32x2 bits = {pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
          if (LOGITS && !pairs && m < p.m && grp < ngrp) *(u32x2*)(p.y + (int64_t)m * p.ldy + n) = bits;
          if ((!LOGITS || p.argmax != nullptr) && grp < ngrp) {
            const uint32_t o0 = bf16x2_order(bits[0]);
            const uint32_t o1 = bf16x2_order(bits[1]);
            const uint32_t rank = 31u - 4u * ns;
            best = max(best, (o0 << 16) | rank);
            best = max(best, (o0 & 0xFFFF0000u) | (rank - 1u));
            best = max(best, (o1 << 16) | (rank - 2u));
            best = max(best, (o1 & 0xFFFF0000u) | (rank - 3u));
          }
          acc[mi][ns] = floatx4{0.f, 0.f, 0.f, 0.f};
        }
      }
      const uint32_t pos = 31u - (best & 31u);
      const uint32_t col = col0 + (pos >> 2) * 16u + (pos & 3u);
      if (best != 0) row_best[mi] = max(row_best[mi], (best & 0xFFFF0000u) | (0xFFFFu - col));
      if (pass_done) {
        uint32_t b2 = row_best[mi];
        b2 = max(b2, (uint32_t)__shfl_xor(b2, 16));
        b2 = max(b2, (uint32_t)__shfl_xor(b2, 32));
        if (p.argmax != nullptr && g == 0 && m < p.m) {
          const uint32_t n = (uint32_t)rc0 + 0xFFFFu - (b2 & 0xFFFFu);
          p.argmax[(int64_t)m * tiles + 2 * blockIdx.x + nw] =
              b2 == 0 ? 0 : ((uint64_t)(b2 >> 16) << 32) | (uint64_t)(0xFFFFFFFFu - n);
        }
        row_best[mi] = 0;
      }
    }
  }
}

// ---- LM head for at most 80 rows (a draft model's one-row-per-sequence decode, small
// verify batches) -------------------------------------------------------------------
// The 320-row kernel's time does not shrink with the rows: its eight waves split the
// rows four ways, so at m <= 80 two waves of one SIMD do all the MFMAs while the weights
// stream through the same two-stage ring.  Here wave c of a work-group owns columns
// 32 c .. +32 of each 256-column block against all 80 rows (5 x 2 subtiles), and a stage
// is X 10 KiB + W 32 KiB, so the ring holds three stages and the weight copies of a stage
// go out two stages ahead.  Work-group ranges, blocks, K stages, the chunk swizzle, the
// MFMA operand order and the argmax key are the 320-row kernel's: every logit is the same
// sum in the same order, hence the same bits, and so is every argmax partial.
constexpr int kLsRows = 80;
constexpr int kLsRing = 3;
constexpr int kLsXSlots = kLsRows * kLmSK * 2 / 1024;    // 10 copies of 8 rows
constexpr int kLsWSlots = kLmCols * kLmSK * 2 / 1024;    // 32
constexpr int kLsSlots = kLsXSlots + kLsWSlots;          // 42 per stage
constexpr int kLsStage = kLsSlots * 1024;
constexpr int kLsMaxCopies = (kLsSlots + kLmWaves - 1) / kLmWaves;  // 6 (waves 0, 1), else 5
static_assert(kLsRing * kLsStage <= 160 * 1024, "LDS");

// copy j of wave w fills stage slot s = 8 j + w (slots 0..9: X rows 8 s .., then W rows)
__device__ __forceinline__ int ls_copies(int wave) { return (kLsSlots - wave + kLmWaves - 1) / kLmWaves; }

__global__ __launch_bounds__(kLmWaves * kWave) void lm_head_small_kernel(GemmParams p) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int lane = threadIdx.x % kWave;
  const int r = lane & 15;
  const int g = lane >> 4;
  const int groups = p.n / kArgmaxCols;
  const int grp0 = (int)((int64_t)groups * blockIdx.x / gridDim.x);
  const int grp1 = (int)((int64_t)groups * (blockIdx.x + 1) / gridDim.x);
  const int nblk = (grp1 - grp0 + 3) / 4;
  const int kt = p.k / kLmSK;
  const int total = nblk * kt;  // stages, in order block, k
  if (total == 0) return;
  const int rc0 = grp0 * kArgmaxCols;
  const int tiles = 2 * (int)gridDim.x;
  const int ncp = ls_copies(wave);

  // per copy: the 32-bit lane offset from the stage's scalar base (X: row and chunk; W:
  // column row within the block and chunk, a short block re-reading its last column)
  auto offset = [&](int j, int ccols) -> uint32_t {
    const int s = j * kLmWaves + wave;
    if (s < kLsXSlots) {
      const int row = s * 8 + (lane >> 3);
      const int chunk = (lane & 7) ^ (row & 7);
      return (uint32_t)min(row, p.m - 1) * (uint32_t)(p.ldx * 2) + (uint32_t)chunk * 16u;
    }
    const int wrow = (s - kLsXSlots) * 8 + (lane >> 3);
    const int chunk = (lane & 7) ^ (wrow & 7);
    return (uint32_t)min(wrow, ccols - 1) * (uint32_t)(p.k * 2) + (uint32_t)chunk * 16u;
  };
  auto issue = [&](int u) {
    const int bi = u / kt, t = u % kt;
    const int c0 = (grp0 + 4 * bi) * kArgmaxCols;
    const int ccols = min(4, grp1 - grp0 - 4 * bi) * kArgmaxCols;
    const int k0 = t * kLmSK;
    char* stage = smem + (u % kLsRing) * kLsStage;
    const char* xsrc = uniform_ptr((const char*)p.x + k0 * 2);
    const char* wsrc = uniform_ptr((const char*)p.w + ((int64_t)c0 * p.k + k0) * 2);
#pragma unroll
    for (int j = 0; j < kLsMaxCopies; ++j) {
      if (j >= ncp) break;
      const int s = j * kLmWaves + wave;
      uint32_t o = offset(j, ccols);
      __asm__("" : "+v"(o));  // scalar base + 32-bit lane offset addressing
      lds_dma16((s < kLsXSlots ? xsrc : wsrc) + o, stage + s * 1024);
    }
  };

  floatx4 acc[5][2];
#pragma unroll
  for (int mi = 0; mi < 5; ++mi) acc[mi][0] = acc[mi][1] = floatx4{0.f, 0.f, 0.f, 0.f};
  uint32_t row_best[5] = {0, 0, 0, 0, 0};

  issue(0);
  if (total > 1) issue(1);
  for (int u = 0; u < total; ++u) {
    // this wave's copies of stage u have landed once at most stage u + 1's are in flight
    if (u + 1 < total) {
      wait_pending<1, kLsMaxCopies>(ncp);
    } else {
      wait_vmcnt<0>();
    }
    asm volatile("s_barrier" ::: "memory");  // everyone's stage u; stage u - 1 fully read
    if (u + 2 < total) issue(u + 2);
    const int bi = u / kt, t = u % kt;
    const int c0 = (grp0 + 4 * bi) * kArgmaxCols;
    const int ccols = min(4, grp1 - grp0 - 4 * bi) * kArgmaxCols;
    const bool live = wave * 32 < ccols;  // a short block's waves past its end skip the MFMAs
    if (live) {
      const char* xs = smem + (u % kLsRing) * kLsStage;
      const char* ws = xs + kLsXSlots * 1024;
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        bf16x8 b[2];
#pragma unroll
        for (int ns = 0; ns < 2; ++ns) b[ns] = lm_frag(ws, wave * 32 + ns * 16 + r, 4 * s + g);
#pragma unroll
        for (int mi = 0; mi < 5; ++mi) {
          const bf16x8 a = lm_frag(xs, mi * 16 + r, 4 * s + g);
#pragma unroll
          for (int ns = 0; ns < 2; ++ns)
            acc[mi][ns] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[ns], a, acc[mi][ns], 0, 0, 0);
        }
      }
    }
    if (t != kt - 1) continue;

    // ---- block done: logits, this lane's best of its 8 values per row, clear ----
    const uint32_t col0 = (uint32_t)(c0 - rc0 + wave * 32 + 4 * g);
#pragma unroll
    for (int mi = 0; mi < 5; ++mi) {
      const int m = mi * 16 + r;
      uint32_t best = 0;
#pragma unroll
      for (int ns = 0; ns < 2; ++ns) {
        const floatx4 v = acc[mi][ns];
        const u32x2 bits = {pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
        if (p.y != nullptr && m < p.m && live)
          *(u32x2*)(p.y + (int64_t)m * p.ldy + c0 + wave * 32 + ns * 16 + 4 * g) = bits;
        if (live) {
          const uint32_t o0 = bf16x2_order(bits[0]);
          const uint32_t o1 = bf16x2_order(bits[1]);
          const uint32_t rank = 7u - 4u * ns;
          best = max(best, (o0 << 16) | rank);
          best = max(best, (o0 & 0xFFFF0000u) | (rank - 1u));
          best = max(best, (o1 << 16) | (rank - 2u));
          best = max(best, (o1 & 0xFFFF0000u) | (rank - 3u));
        }
        acc[mi][ns] = floatx4{0.f, 0.f, 0.f, 0.f};
      }
      const uint32_t pos = 7u - (best & 7u);
      const uint32_t col = col0 + (pos >> 2) * 16u + (pos & 3u);
      if (best != 0) row_best[mi] = max(row_best[mi], (best & 0xFFFF0000u) | (0xFFFFu - col));
    }
  }

  // ---- the range's argmax partials: per row, the best of the four waves of each
  // 128-column half (waves 0..3, 4..7), as the 320-row kernel's waves nw = 0, 1 keep them
  uint32_t* s_best = (uint32_t*)smem;  // [wave][80 rows]
  __syncthreads();                     // every wave is past its last stage
#pragma unroll
  for (int mi = 0; mi < 5; ++mi) {
    uint32_t b2 = row_best[mi];
    b2 = max(b2, (uint32_t)__shfl_xor(b2, 16));
    b2 = max(b2, (uint32_t)__shfl_xor(b2, 32));
    if (g == 0) s_best[wave * kLsRows + mi * 16 + r] = b2;
  }
  __syncthreads();
  if (p.argmax != nullptr && (wave & 3) == 0) {
    const int half = wave >> 2;
    for (int m = lane; m < p.m; m += kWave) {
      uint32_t b2 = 0;
#pragma unroll
      for (int w = 0; w < 4; ++w) b2 = max(b2, s_best[(half * 4 + w) * kLsRows + m]);
      const uint32_t n = (uint32_t)rc0 + 0xFFFFu - (b2 & 0xFFFFu);
      p.argmax[(int64_t)m * tiles + 2 * blockIdx.x + half] =
          b2 == 0 ? 0 : ((uint64_t)(b2 >> 16) << 32) | (uint64_t)(0xFFFFFFFFu - n);
    }
  }
}

template <LmOut OUT>
int launch_lm_head_rows(const GemmParams& p, int grid, hipStream_t stream) {
  static const hipError_t attr = hipFuncSetAttribute(
      (const void*)lm_head_kernel<OUT>, hipFuncAttributeMaxDynamicSharedMemorySize, kLmRing * kLmStage);
  if (attr != hipSuccess) {
    set_error("lm_head: cannot reserve %d bytes of LDS: %s", kLmRing * kLmStage, hipGetErrorString(attr));
    return NE_ELAUNCH;
  }
  hipLaunchKernelGGL((lm_head_kernel<OUT>), dim3((unsigned)grid), dim3(kLmWaves * kWave), kLmRing * kLmStage,
                     stream, p);
  return check_launch("lm_head");
}

int launch_lm_head(GemmParams p, hipStream_t stream) {
  const int groups = p.n / kArgmaxCols;
  const int grid = groups < kLmMaxGrid ? groups : kLmMaxGrid;
  if (p.m <= kLsRows) {
    static const hipError_t attr_small = hipFuncSetAttribute(
        (const void*)lm_head_small_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, kLsRing * kLsStage);
    if (attr_small != hipSuccess) {
      set_error("lm_head: cannot reserve %d bytes of LDS: %s", kLsRing * kLsStage, hipGetErrorString(attr_small));
      return NE_ELAUNCH;
    }
    hipLaunchKernelGGL(lm_head_small_kernel, dim3((unsigned)grid), dim3(kLmWaves * kWave), kLsRing * kLsStage,
                       stream, p);
    return check_launch("lm_head");
  }
  if (p.y == nullptr) return launch_lm_head_rows<LmOut::kArgmax>(p, grid, stream);
  // 16-byte stores: rows that start on 16 bytes, and ranges with a full block of 4 groups
  if (((uintptr_t)p.y % 16) == 0 && p.ldy % 8 == 0 && groups >= 4 * grid)
    return launch_lm_head_rows<LmOut::kWideLogits>(p, grid, stream);
  return launch_lm_head_rows<LmOut::kLogits>(p, grid, stream);
}

}  // namespace

}  // namespace ne

using namespace ne;

namespace {

int w8a16_common(const void* x, int64_t ldx, const int8_t* w, const void* scale, int32_t scale_dtype,
                 int32_t m, int32_t n, int32_t k, void* y, int64_t ldy, int32_t epilogue,
                 int32_t splits, float* partial, void* stream) {
  GemmParams p{};
  p.x = (const uint16_t*)x;
  p.ldx = ldx;
  p.w = w;
  p.scale = scale;
  p.scale_dtype = scale_dtype;
  p.m = m;
  p.n = n;
  p.k = k;
  p.y = (uint16_t*)y;
  p.ldy = ldy;
  hipStream_t s = (hipStream_t)stream;
  switch (scale_dtype) {
    case NE_DTYPE_BF16:
      return dispatch_w8a16<NE_DTYPE_BF16>(p, epilogue, splits, partial, s);
    case NE_DTYPE_FP16:
      return dispatch_w8a16<NE_DTYPE_FP16>(p, epilogue, splits, partial, s);
    case NE_DTYPE_FP32:
      return dispatch_w8a16<NE_DTYPE_FP32>(p, epilogue, splits, partial, s);
    default:
      set_error("scale_dtype must be bf16, fp16 or fp32");
      return NE_EINVAL;
  }
}

}  // namespace

extern "C" int32_t ne_w8a16_kernel(int32_t m, int32_t n, int32_t k, int32_t splits, int32_t epilogue) {
  if (m <= 0 || n <= 0 || k <= 0 || splits < 0) return NE_W8A16_STAGED;
  GemmParams p{};
  p.m = m;
  p.n = n;
  p.k = k;
  if (few_rows(p, splits > 0 ? splits : 1)) return NE_W8A16_FEW_ROWS;
  if (splits > 0) return NE_W8A16_STAGED;
  switch (choose_proj_tile(m, n, epilogue == NE_EPILOGUE_SWIGLU)) {
    case ProjTile::k128x128: return NE_W8A16_TILE_128X128;
    case ProjTile::k128x256: return NE_W8A16_TILE_128X256;
    case ProjTile::k256x256: return NE_W8A16_TILE_256X256;
    default: return NE_W8A16_STAGED;
  }
}

extern "C" int ne_w8a16_gemm(const void* x, int64_t ldx, const int8_t* w, const void* scale,
                             int32_t scale_dtype, int32_t m, int32_t n, int32_t k, void* y,
                             int64_t ldy, int32_t epilogue, void* stream) {
  NE_CHECK_ARG(m >= 0 && n > 0 && k > 0, "bad gemm shape m=%d n=%d k=%d", m, n, k);
  if (m == 0) return NE_OK;
  NE_CHECK_ARG(x && w && scale && y, "null pointer argument");
  NE_CHECK_ARG(epilogue == NE_EPILOGUE_STORE || epilogue == NE_EPILOGUE_SWIGLU,
               "unknown epilogue %d", epilogue);
  NE_CHECK_SUPPORTED(k % 128 == 0, "k must be a multiple of 128 (got %d)", k);
  NE_CHECK_SUPPORTED(n % 64 == 0, "n must be a multiple of 64 (got %d)", n);
  NE_CHECK_ARG(ldx >= k && ldx % 8 == 0, "ldx must be >= k and a multiple of 8");
  NE_CHECK_SUPPORTED((int64_t)m * ldx < kMaxXElems, "x spans more than 4 GiB (m=%d, ldx=%lld)", m, (long long)ldx);
  NE_CHECK_ARG(ldy >= (epilogue == NE_EPILOGUE_SWIGLU ? n / 2 : n) && ldy % 4 == 0,
               "ldy too small or not a multiple of 4");
  NE_CHECK_ARG(((uintptr_t)x % 16) == 0 && ((uintptr_t)w % 16) == 0 && ((uintptr_t)y % 8) == 0,
               "x and w must be 16-byte aligned, y 8-byte aligned");
  return w8a16_common(x, ldx, w, scale, scale_dtype, m, n, k, y, ldy, epilogue, 1, nullptr, stream);
}

extern "C" int ne_w8a16_gemm_splitk(const void* x, int64_t ldx, const int8_t* w, const void* scale,
                                    int32_t scale_dtype, int32_t m, int32_t n, int32_t k,
                                    int32_t splits, float* partials, void* stream) {
  NE_CHECK_ARG(m >= 0 && n > 0 && k > 0, "bad gemm shape m=%d n=%d k=%d", m, n, k);
  if (m == 0) return NE_OK;
  NE_CHECK_ARG(x && w && scale && partials, "null pointer argument");
  NE_CHECK_ARG(splits >= 1 && splits <= 64, "splits must be in [1, 64] (got %d)", splits);
  NE_CHECK_SUPPORTED(k % (128 * splits) == 0, "k must be a multiple of 128 * splits (k=%d, splits=%d)",
                     k, splits);
  NE_CHECK_SUPPORTED(n % 64 == 0, "n must be a multiple of 64 (got %d)", n);
  NE_CHECK_ARG(ldx >= k && ldx % 8 == 0, "ldx must be >= k and a multiple of 8");
  NE_CHECK_SUPPORTED((int64_t)m * ldx < kMaxXElems, "x spans more than 4 GiB (m=%d, ldx=%lld)", m, (long long)ldx);
  NE_CHECK_ARG(((uintptr_t)x % 16) == 0 && ((uintptr_t)w % 16) == 0 && ((uintptr_t)partials % 16) == 0,
               "x, w and partials must be 16-byte aligned");
  return w8a16_common(x, ldx, w, scale, scale_dtype, m, n, k, nullptr, 0, NE_EPILOGUE_STORE, splits,
                      partials, stream);
}

extern "C" int ne_w8a16_qkv_norm_rope_kv(
    const void* x, int64_t ldx, const int8_t* w, const void* scale, int32_t scale_dtype, int32_t m,
    int32_t num_q_heads, int32_t num_kv_heads, int32_t k, const void* q_norm_w, const void* k_norm_w,
    float eps, const int32_t* positions, const void* rope, int32_t rope_positions,
    const int32_t* slot_mapping, int32_t kv_dtype, void* k_cache, void* v_cache, void* k_scale,
    void* v_scale, int32_t kv_scale_dtype, void* q_out, void* stream) {
  NE_CHECK_ARG(m >= 0 && num_q_heads > 0 && num_kv_heads > 0 && k > 0, "bad shape");
  if (m == 0) return NE_OK;
  NE_CHECK_ARG(x && w && scale && q_norm_w && k_norm_w && positions && rope && slot_mapping && k_cache &&
                   v_cache && q_out,
               "null pointer argument");
  NE_CHECK_ARG(rope_positions > 0, "rope_positions must be > 0");
  NE_CHECK_SUPPORTED(k % 128 == 0, "k must be a multiple of 128 (got %d)", k);
  NE_CHECK_ARG(ldx >= k && ldx % 8 == 0, "ldx must be >= k and a multiple of 8");
  NE_CHECK_SUPPORTED((int64_t)m * ldx < kMaxXElems, "x spans more than 4 GiB (m=%d, ldx=%lld)", m, (long long)ldx);
  NE_CHECK_ARG(((uintptr_t)x % 16) == 0 && ((uintptr_t)w % 16) == 0, "x and w must be 16-byte aligned");
  int kv_mode = 0;
  if (kv_dtype == NE_DTYPE_BF16) {
    kv_mode = 1;
  } else if (kv_dtype == NE_DTYPE_INT8) {
    NE_CHECK_ARG(k_scale && v_scale, "an int8 cache needs k_scale and v_scale");
    NE_CHECK_SUPPORTED(kv_scale_dtype == NE_DTYPE_BF16 || kv_scale_dtype == NE_DTYPE_FP16,
                       "fused KV write supports bf16 or fp16 scales");
    kv_mode = kv_scale_dtype == NE_DTYPE_BF16 ? 2 : 3;
  } else {
    set_error("kv_dtype must be int8 or bf16");
    return NE_EINVAL;
  }
  GemmParams p{};
  p.x = (const uint16_t*)x;
  p.ldx = ldx;
  p.w = w;
  p.scale = scale;
  p.scale_dtype = scale_dtype;
  p.m = m;
  p.n = (num_q_heads + 2 * num_kv_heads) * 128;
  p.k = k;
  const QkvRopeArgs qa{num_q_heads, num_kv_heads, (const uint16_t*)q_norm_w, (const uint16_t*)k_norm_w,
                       eps, positions, (const uint16_t*)rope, rope_positions, slot_mapping,
                       k_cache, v_cache, k_scale, v_scale, (uint16_t*)q_out};
  hipStream_t s = (hipStream_t)stream;
  switch (scale_dtype) {
    case NE_DTYPE_BF16: return dispatch_qkv_fused<NE_DTYPE_BF16>(p, qa, kv_mode, s);
    case NE_DTYPE_FP16: return dispatch_qkv_fused<NE_DTYPE_FP16>(p, qa, kv_mode, s);
    case NE_DTYPE_FP32: return dispatch_qkv_fused<NE_DTYPE_FP32>(p, qa, kv_mode, s);
    default:
      set_error("scale_dtype must be bf16, fp16 or fp32");
      return NE_EINVAL;
  }
}

extern "C" int32_t ne_lm_head_num_tiles(int32_t n) {
  return n > 0 ? 2 * min(n / kArgmaxCols, kLmMaxGrid) : 0;  // two waves' halves per work-group
}

extern "C" int ne_lm_head(const void* x, int64_t ldx, const void* w, int32_t m, int32_t n,
                          int32_t k, void* logits, int64_t ld_logits, uint64_t* argmax_partials,
                          void* stream) {
  NE_CHECK_ARG(m >= 0 && n > 0 && k > 0, "bad lm head shape m=%d n=%d k=%d", m, n, k);
  if (m == 0) return NE_OK;
  NE_CHECK_ARG(x && w, "null pointer argument");
  NE_CHECK_ARG(logits || argmax_partials, "lm head needs logits and/or argmax_partials");
  NE_CHECK_SUPPORTED(k % 128 == 0, "k must be a multiple of 128 (got %d)", k);
  NE_CHECK_SUPPORTED(n % 128 == 0, "vocab must be a multiple of 128 (got %d)", n);
  // argmax keys hold a column within a work-group's range in 16 bits
  NE_CHECK_SUPPORTED(n <= (1 << 24), "vocab above 2^24 (got %d)", n);
  NE_CHECK_ARG(ldx >= k && ldx % 8 == 0, "ldx must be >= k and a multiple of 8");
  NE_CHECK_ARG(!logits || (ld_logits >= n && ld_logits % 4 == 0), "bad ld_logits");
  NE_CHECK_ARG(((uintptr_t)x % 16) == 0 && ((uintptr_t)w % 16) == 0 &&
                   ((uintptr_t)logits % 8) == 0,
               "x and w must be 16-byte aligned, logits 8-byte aligned");
  // X copies address rows with 32-bit byte offsets, weight rows of a block likewise
  NE_CHECK_SUPPORTED((int64_t)m * ldx < kMaxXElems, "x spans more than 4 GiB (m=%d, ldx=%lld)", m, (long long)ldx);
  NE_CHECK_SUPPORTED((int64_t)kLmCols * k * 2 < (int64_t(1) << 32), "k too large for the LM head (k=%d)", k);
  GemmParams p{};
  p.x = (const uint16_t*)x;
  p.ldx = ldx;
  p.w = w;
  p.m = m;
  p.n = n;
  p.k = k;
  p.y = (uint16_t*)logits;
  p.ldy = ld_logits;
  p.argmax = argmax_partials;
  hipStream_t s = (hipStream_t)stream;
  return launch_lm_head(p, s);
}
