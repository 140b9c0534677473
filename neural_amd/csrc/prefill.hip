// MXFP4 GEMMs on gfx950 for prompt processing: the reference's mxfp4_gemm / grouped GEMM arithmetic (per 32-element
// group, E2M1 x 2^(s-127) dequantised exactly to bf16, bf16 x bf16 products accumulated in fp32, one bf16 rounding of
// each output; reference neural/q80/mxfp4_kernels.py:87-126, 242-295) and the fused MoE prefill layer (reference
// server.py:1837-1936, _expert_gemms :1977-2040).
//
// The fused layer (k_prefill_gate_up / k_prefill_down) runs on the block-scaled v_mfma_scale_f32_16x16x128_f8f6f4:
// E2M1 codes and E8M0 scales as stored, activations as two E4M3 rows (hi, lo) with one E8M0 scale per 32 elements
// each (x per 32-element block of a row; h per 32 columns of a row, quantised in the gate_up epilogue).  hi w + lo w
// is the reference's bf16 x E2M1 product exactly for every element within 2^13 of its block's largest magnitude m;
// an element further below m is reproduced to within 2^-21 m (the remainder's 4 significant bits on the lo grid),
// so an output deviates from the reference's by at most 2^-21 sum_k |w_k| m_k before its bf16 rounding (t950.h
// states the quantiser).
//
// The plain and grouped GEMM entry points (bf16 activations, no workspace) run the same tiles on bf16 rows and
// v_mfma_f32_16x16x32_bf16, the weights converted to bf16 (exact; gemm8_wide past bf16's range) in registers.  They are HBM-bound where experts have
// few rows: 2,000 Zipf-routed rows over a raw store, gate_up and down (1.7 GB), 1,390 -> 536 us when the scales went
// through LDS instead of scattered byte loads, tiles stopped staging and multiplying their empty 16-row blocks, column
// groups got the XCD order, and the kernels, 400 registers before, came to fit two workgroups per CU; -> 493 us with the
// activation quantiser's one-instruction block maxima; -> 462 us, and one expert's 4,096 rows 320 -> 213 us
// (957 TFLOP/s), when the rows stopped being quantised into hi + lo E4M3 rows by every column group.
//
// Weight layouts (template W): the store's raw and PS4 slots (row r: 1,440 code bytes, then a raw 90-byte or PS4
// 46-byte scale row; lane (q, n) reads the 16 bytes of group 4t + q of row n, already the MFMA's B order) and the t950
// tiles (lane (q, n) reads the 16 bytes at 1024 t + 16 (16 q + n) of the row block: the same operand).
#include "common.h"
#include "t950.h"

#include <hip/hip_ext.h>

namespace na {

enum WLayout : int { kWRaw = 0, kWPs4 = 1, kWT950 = 2 };

constexpr int kPBM = 64;                 // tokens per tile
constexpr int kPKT = 128;                // K elements per k-tile
constexpr int kPTiles = kTTiles;         // 23 k-tiles: 22 full + groups 88, 89

// One matrix (gate_up or down) of one expert, as the kernels address it.
struct WSrc {
  const uint8_t* codes;     // raw/PS4: row 0's code bytes (row pitch 1,440); t950: block 0 of the matrix
  const uint8_t* scales;    // raw/PS4: row 0's scale row (pitch 90 or 46); t950: unused
};

// Two E2M1 codes of byte SEL of `word`, times 2^e of the float `scale` -> packed bf16 pair (low nibble = element 0 in the
// low half): exact for every E8M0 scale byte up to 252 (byte 0, the float 0, is 2^-127), NaN at 255.
template <int SEL>
NA_DEVICE uint32_t fp4x2_scaled(uint32_t word, float scale) {
  return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(word, scale, SEL));
}

// Scale bytes from which a weight can be past bf16's largest value: codes of 4 and 6 at 253, of 2 and above at 254.
constexpr uint32_t kE8m0Wide = 253;

// A quarter of the same two weights from the scale byte: exact for every byte up to 254 (2^-130 .. 1.5 x 2^127), NaN at
// 255.
template <int SEL>
NA_DEVICE uint32_t fp4x2_quarter(uint32_t word, uint32_t byte) {
  const auto v = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(word, 1.0f, SEL);
  const int e = (int)byte - 129;
  return byte == 255 ? 0x7fc07fc0u : pack_bf16x2(__builtin_amdgcn_ldexpf(v[0], e), __builtin_amdgcn_ldexpf(v[1], e));
}

constexpr int kPNB = 3;                  // row blocks per wave in the plain, grouped and down kernels
constexpr int kPRows = 4 * kPNB * 16;    // 192 weight rows per workgroup

template <int W>
NA_DEVICE WSrc w_src(const uint8_t* blocks, long long sb_slot, const uint8_t* scales, long long ss_slot,
                     long long slot) {
  return WSrc{blocks + slot * sb_slot, scales ? scales + slot * ss_slot : nullptr};
}

// ------------------------------------------------------------------------------------ fused MoE prefill layer
// Routing: pairs p = 4 t + k (token t, rank k); valid expert ids in [0, 128).  counts[e], then a stable order of the
// pairs by expert (order[offs[e] + i] = the i-th pair of expert e in increasing p) and a tile table
// tiles[i] = (expert, first sorted position, rows <= 64), ntiles.  Invalid ids are in no expert's list and
// contribute +0 (the combine skips them).
// Quantised row ("q row", kQRow bytes): hi codes [0, 2880), lo codes [2880, 5760), hi scales [5760, 5856) and lo
// scales [5856, 5952), scale bytes 90..95 of each half zero (the last k-tile's groups 90, 91 are padding).
constexpr int kQRow = 2 * kH + 2 * kX8ScPitch;        // 5,952
constexpr int kQLo = kH;
constexpr int kQSh = 2 * kH;
constexpr int kQSl = 2 * kH + kX8ScPitch;

struct PTile {
  int e, p0, cnt, pad;
};

// Expert ids of one round of 8,192 pairs: wave w's 2,048 consecutive ones in 32 coalesced steps of 64, id[j] = that of
// pair p0 + 2048 w + 64 j + lane, -1 past P and for an id outside [0, 128).
constexpr int kRound = 8192;
NA_DEVICE void load_round(const int64_t* __restrict__ ids, int P, int p0, int wave, int lane, int (&id)[32]) {
#pragma unroll
  for (int j = 0; j < 32; ++j) {
    const long long p = (long long)p0 + 2048 * wave + 64 * j + lane;
    const int64_t v = p < P ? ids[p] : -1;
    id[j] = v >= 0 && v < 128 ? (int)v : -1;
  }
}

// Block e of 0..127: the expert's count, tiles and pairs in increasing p.  Every block counts all experts in LDS (one
// histogram per wave), so that the prefix over the experts before e needs no launch of its own; a round's ids stay in
// registers between the counting and the ordering (a layer of up to 2,048 tokens reads them once): one ballot per step
// gives each lane its place among its wave's hits, a 4-entry scan places the waves.  Blocks 128..: x quantised into q
// rows, one 8-element chunk per thread (4 consecutive threads = one 32-element block; 360 chunks per row, so a block
// never straddles rows).  Latency-bound: with the counts (and the quantising) in a launch before the order's, the layer
// took 630 us at 2,048 tokens, 611 so; at 23 tokens 3.5 % more.
__global__ __launch_bounds__(256) void k_prefill_route(const int64_t* __restrict__ ids, int P, int* __restrict__ counts,
                                                       int* __restrict__ order, PTile* __restrict__ tiles,
                                                       int* __restrict__ ntiles, const uint16_t* __restrict__ x, int T,
                                                       uint8_t* __restrict__ xq) {
  if (blockIdx.x >= 128) {
    const long long g = (long long)(blockIdx.x - 128) * 256 + threadIdx.x;
    const bool ok = g < (long long)T * kChunks;
    const long long row = ok ? g / kChunks : 0;
    const int c = ok ? (int)(g - row * kChunks) : 0;
    const uint4 v = ok ? *reinterpret_cast<const uint4*>(x + row * kH + 8 * c) : make_uint4(0, 0, 0, 0);
    uint2 hi, lo;
    uint32_t sh, sl;
    x8_quant_chunk(v, hi, lo, sh, sl);
    if (ok) {
      uint8_t* dst = xq + row * kQRow;
      *reinterpret_cast<uint2*>(dst + 8 * c) = hi;
      *reinterpret_cast<uint2*>(dst + kQLo + 8 * c) = lo;
      if ((c & 3) == 0) {
        dst[kQSh + (c >> 2)] = (uint8_t)sh;
        dst[kQSl + (c >> 2)] = (uint8_t)sl;
      }
      if (c < kX8ScPitch - kGK) {
        dst[kQSh + kGK + c] = 0;
        dst[kQSl + kGK + c] = 0;
      }
    }
    return;
  }
  const int e = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  __shared__ int hist[4][128];
  __shared__ int wcnt[4];
  __shared__ int base_s[3];
  hist[wave][lane] = 0;
  hist[wave][64 + lane] = 0;
  __syncthreads();
  int id[32];
  for (int r = (P - 1) / kRound; r >= 0; --r) {         // the first round last: its ids stay for the ordering
    load_round(ids, P, r * kRound, wave, lane, id);
#pragma unroll
    for (int j = 0; j < 32; ++j)
      if (id[j] >= 0) atomicAdd(&hist[wave][id[j]], 1);
  }
  __syncthreads();
  if (wave == 0) {
    const int c0 = (hist[0][lane] + hist[1][lane]) + (hist[2][lane] + hist[3][lane]);
    const int c1 = (hist[0][64 + lane] + hist[1][64 + lane]) + (hist[2][64 + lane] + hist[3][64 + lane]);
    const int t0 = (c0 + kPBM - 1) / kPBM, t1 = (c1 + kPBM - 1) / kPBM;
    int off = (lane < e ? c0 : 0) + (64 + lane < e ? c1 : 0);
    int tb = (lane < e ? t0 : 0) + (64 + lane < e ? t1 : 0);
    int tt = t0 + t1;
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
      off += __shfl_xor(off, o);
      tb += __shfl_xor(tb, o);
      tt += __shfl_xor(tt, o);
    }
    if (lane == 0) {
      base_s[0] = off;
      base_s[1] = tb;
      if (e == 0) *ntiles = tt;
    }
    if (lane == (e & 63)) {
      base_s[2] = e < 64 ? c0 : c1;
      counts[e] = e < 64 ? c0 : c1;
    }
  }
  __syncthreads();
  const int off = base_s[0], tb = base_s[1], c = base_s[2];
  for (int m = tid; m * kPBM < c; m += 256) tiles[tb + m] = PTile{e, off + m * kPBM, min(kPBM, c - m * kPBM), 0};
  const uint64_t lt = (1ull << lane) - 1;
  int run = 0;                                        // pairs of expert e before this round
  for (int p0 = 0; p0 < P; p0 += kRound) {
    if (p0) load_round(ids, P, p0, wave, lane, id);
    const int wp0 = p0 + 2048 * wave;
    uint64_t bal[32];
    int wn = 0;
#pragma unroll
    for (int j = 0; j < 32; ++j) {
      bal[j] = __ballot(id[j] == e);
      wn += __popcll(bal[j]);
    }
    if (lane == 0) wcnt[wave] = wn;
    __syncthreads();
    int pos = off + run;
    for (int w = 0; w < wave; ++w) pos += wcnt[w];
#pragma unroll
    for (int j = 0; j < 32; ++j) {
      if ((bal[j] >> lane) & 1) order[pos + __popcll(bal[j] & lt)] = wp0 + 64 * j + lane;
      pos += __popcll(bal[j]);
    }
    run += wcnt[0] + wcnt[1] + wcnt[2] + wcnt[3];
    __syncthreads();
  }
}

// ---------------------------------------------------------------- block-scaled products of the fused layer
// The layer's two GEMMs run on v_mfma_scale_f32_16x16x128_f8f6f4 with the E2M1 codes and E8M0 scales as stored (B)
// and the activations as two exact E4M3 rows (A: hi and lo, one E8M0 scale per 32-element block each; the exactness
// argument is the one of x8_quant_chunk in t950.h).  Each k-tile of 128 elements is one MFMA per (16 tokens, 16 weight
// rows) and activation row (hi, lo): the hi + lo products are the reference's bf16 x E2M1 products, accumulated in
// fp32.  Activations are quantised once per row, not per workgroup: x per token by the first launch, h per sorted pair
// by the gate_up epilogue.
//
constexpr int kQPitch = 2 * kPKT + 16;                 // LDS bytes per staged row: hi 128 | lo 128 | pad 16
constexpr int kQStage = kPBM * kQPitch + kPBM * 8;     // one k-tile: 64 rows, then 8 scale bytes per row
constexpr int kGuSlots = 3;                            // gate_up: 23 column groups over 8 XCDs, 3 per XCD
constexpr int kDnSlots = 2;                            // down: 15 column groups, 2 per XCD
constexpr int kYPitch = 2 * kPRows + 16;              // LDS bytes per row of a staged down output tile
constexpr int kOhPitch = 2 * kPKT + 8;                 // LDS bytes per row of gate_up's staged h codes (rows 4 apart
                                                       // start 8 banks apart)

// Staging of one k-tile of the 16 NT q rows that a tile's tokens fill: pieces of 16 B, thread tid owns piece (tid & 15)
// of rows (tid >> 4) + 16 i, i < NT (pieces 0..7 hi, 8..15 lo); threads 0..16 NT - 1 also own the 4 hi and 4 lo scale
// bytes of row tid, stored interleaved (hi g, lo g) per group g of the k-tile.
template <int NT>
struct QStage {
  uint4 v[NT];
  uint2 s;
};

// Activation rows that arrive quantised (q rows): rp[i] = q row of staged row (tid >> 4) + 16 i, srow = q row of
// staged row tid & 63.
struct QRows {
  static constexpr bool kBf16 = false;
  template <int NT>
  using Stage = QStage<NT>;
  const uint8_t* rp[4];
  const uint8_t* srow;

  template <int NT>
  NA_DEVICE void load(int t, int tid, QStage<NT>& a) const {
    const int c16 = tid & 15, e0 = t * kPKT + 16 * (c16 & 7), half = (c16 >> 3) * kQLo;
#pragma unroll
    for (int i = 0; i < NT; ++i)
      a.v[i] = e0 < kH ? *reinterpret_cast<const uint4*>(rp[i] + half + e0) : make_uint4(0, 0, 0, 0);
    if (tid < 16 * NT) {
      a.s.x = *reinterpret_cast<const uint32_t*>(srow + kQSh + 4 * t);
      a.s.y = *reinterpret_cast<const uint32_t*>(srow + kQSl + 4 * t);
    }
  }
  template <int NT>
  NA_DEVICE void store(uint8_t* buf, int tid, const QStage<NT>& a) const {
#pragma unroll
    for (int i = 0; i < NT; ++i)
      *reinterpret_cast<uint4*>(buf + ((tid >> 4) + 16 * i) * kQPitch + 16 * (tid & 15)) = a.v[i];
    if (tid < 16 * NT)                                 // interleaved at the store, so the loads are not waited on early
      *reinterpret_cast<uint2*>(buf + kPBM * kQPitch + 8 * tid) =
          make_uint2(__byte_perm(a.s.x, a.s.y, 0x5140), __byte_perm(a.s.x, a.s.y, 0x7362));
  }
};

// bf16 activation rows staged as they are (the GEMM entry points): thread tid owns the 8-element piece tid & 15 of rows
// (tid >> 4) + 16 i.  rp[i] = bf16 row of staged row (tid >> 4) + 16 i.
template <int NT>
struct BStage {
  uint4 v[NT];
};

struct BRows {
  static constexpr bool kBf16 = true;
  template <int NT>
  using Stage = BStage<NT>;
  const uint16_t* rp[4];
  const uint16_t* x0;                                  // staged row r: row min(r, last) of x0
  int last;

  NA_DEVICE BRows(const uint16_t* x0_, int last_, int tid) : x0(x0_), last(last_) {
#pragma unroll
    for (int i = 0; i < 4; ++i) rp[i] = row((tid >> 4) + 16 * i);
  }
  NA_DEVICE const uint16_t* row(int r) const { return x0 + min(r, last) * kH; }

  template <int NT>
  NA_DEVICE void load(int t, int tid, BStage<NT>& a) const {
    const int e0 = t * kPKT + 8 * (tid & 15);
#pragma unroll
    for (int i = 0; i < NT; ++i)
      a.v[i] = e0 < kH ? *reinterpret_cast<const uint4*>(rp[i] + e0) : make_uint4(0, 0, 0, 0);
  }
  template <int NT>
  NA_DEVICE void store(uint8_t* buf, int tid, const BStage<NT>& a) const {
#pragma unroll
    for (int i = 0; i < NT; ++i)
      *reinterpret_cast<uint4*>(buf + ((tid >> 4) + 16 * i) * kQPitch + 16 * (tid & 15)) = a.v[i];
  }
};

// FP4 B operand of k-tile t in the MFMA order (lane 16 kb + n: the 16 code bytes of group 4t + kb of row n), groups
// beyond K zeroed.  Every layout's load already is in that order.
NA_DEVICE mfma_i32x8_t w_operand8(uint4 c, int t, int lane) {
  if (4 * t + (lane >> 4) >= kGK) c = make_uint4(0, 0, 0, 0);
  return mfma_i32x8_t{(int)c.x, (int)c.y, (int)c.z, (int)c.w, 0, 0, 0, 0};
}

constexpr int kWScBytes = kTRows * kTScalePitch;      // LDS bytes of one row block's staged scale rows (t950: 1,536)

// Store layouts: the scale rows of a row block are contiguous (16 x 90 or 16 x 46 bytes), so they are staged as they
// stand: a k-tile's scale is one LDS byte (PS4: a nibble of one, plus the row's base, which stays in a register).
// Scattered per-k-tile byte loads in their place (one or two per row block, each 16 lines) bound these layouts before.
template <int W>
struct WScales {
  static constexpr int kPitch = W == kWT950 ? kTScalePitch : W == kWRaw ? kGK : kPs4Row;
  static constexpr int kBytes = kTRows * kPitch;       // a multiple of 16 in every layout
  static_assert(kBytes <= kWScBytes && kBytes % 16 == 0, "scale rows of a row block");
};

// One wave's weight stream over its NB row blocks: the code bytes of a k-tile, one 16-byte load per lane and row block
// in the MFMA's operand order (lane (q, n): t950 the 16 bytes at 1024 t + 16 lane of the block, raw / PS4 those of group
// 4t + q of row n; groups 90, 91 re-read group 89 and are zeroed at the use).  The block's own offset is 64-bit and
// wave-uniform (the GEMM entry points take any N: 1.49 M rows of codes pass 2^31 bytes), the lane's within it 32-bit.
// The E8M0 rows of the blocks are staged once in the wave's LDS area wsc (load_scales, store_scales) and read per k-tile
// from there.
template <int W, int NB>
struct WStream {
  WSrc src;
  const int* blk;
  uint8_t* wsc;
  int lane;
  int base[NB];                                        // PS4: base byte of this lane's row, per row block
  uint32_t top;                                        // bf16 rows: this lane's largest scale byte (gemm8_wide)

  NA_DEVICE void load(int t, uint4 (&c)[NB]) const {
    const int g = min(4 * t + (lane >> 4), kGK - 1);
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      if constexpr (W == kWT950)
        c[nb] = load16(src.codes + (long long)blk[nb] * kTBlock + t * 1024 + 16 * lane);
      else
        c[nb] = load16(src.codes + (long long)blk[nb] * (kTRows * kRowBytes) +
                       (uint32_t)((lane & 15) * kRowBytes + 16 * g));
    }
  }
  // The blocks' scale rows through registers to LDS, by 16-byte pieces: the loads are issued before the first k-tiles'
  // and stored behind them, so that their round trip is not a tile's first (a view of byte-aligned scales, which only
  // the GEMM entry points accept, is copied byte by byte at the store).
  static constexpr int kScBytes = WScales<W>::kBytes, kScRounds = (kScBytes / 16 + 63) / 64;
  NA_DEVICE const uint8_t* scale_rows(int nb) const {
    return W == kWT950 ? src.codes + (long long)blk[nb] * kTBlock + kTCodes : src.scales + (long long)blk[nb] * kScBytes;
  }
  NA_DEVICE bool scales_aligned() const {
    return W == kWT950 || (reinterpret_cast<uintptr_t>(src.scales) & 15) == 0;
  }
  NA_DEVICE void load_scales(uint4 (&v)[NB][kScRounds]) {
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      const uint8_t* sp = scale_rows(nb);
#pragma unroll
      for (int r = 0; r < kScRounds; ++r) {
        v[nb][r] = make_uint4(0, 0, 0, 0);
        if (scales_aligned() && 64 * r + lane < kScBytes / 16) v[nb][r] = load16(sp + 16 * (64 * r + lane));
      }
      if constexpr (W == kWPs4) base[nb] = sp[(lane & 15) * kPs4Row];
    }
  }
  NA_DEVICE void store_scales(const uint4 (&v)[NB][kScRounds]) {
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      uint8_t* dst = wsc + nb * kWScBytes;
      if (scales_aligned()) {
#pragma unroll
        for (int r = 0; r < kScRounds; ++r)
          if (64 * r + lane < kScBytes / 16) *reinterpret_cast<uint4*>(dst + 16 * (64 * r + lane)) = v[nb][r];
      } else {
        for (int i = lane; i < kScBytes; i += 64) dst[i] = scale_rows(nb)[i];
      }
    }
  }
  NA_DEVICE int scale(int t, int nb) const {
    const uint8_t* row = wsc + nb * kWScBytes + (lane & 15) * WScales<W>::kPitch;
    const int kb = lane >> 4;
    if constexpr (W == kWT950) {
      return row[4 * t + kb];
    } else if constexpr (W == kWRaw) {
      return row[min(4 * t + kb, kGK - 1)];
    } else {
      return base[nb] + ((row[1 + min(2 * t + (kb >> 1), kGK / 2 - 1)] >> (4 * (kb & 1))) & 15);
    }
  }
};

// The MFMAs of k-tile t on quantised rows staged at cur, weight codes c: block-scaled, hi and lo rows.
template <int W, int NB, int NT>
NA_DEVICE void ktile_x8(int t, const WStream<W, NB>& ws, const uint8_t* cur, const uint4 (&c)[NB], f32x4_t (&acc)[4][NB]) {
  const int lane = threadIdx.x & 63, kb = lane >> 4, m = lane & 15;
  mfma_i32x8_t b[NB];
  int sb[NB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    b[nb] = w_operand8(c[nb], t, lane);
    sb[nb] = ws.scale(t, nb);
  }
  __builtin_amdgcn_s_setprio(1);                     // the MFMA burst issues ahead of the other wave's staging
#pragma unroll
  for (int tt = 0; tt < NT; ++tt) {
    const uint8_t* row = cur + (16 * tt + m) * kQPitch + 16 * kb;
    const uint4 h0 = *reinterpret_cast<const uint4*>(row), h1 = *reinterpret_cast<const uint4*>(row + 64);
    const uint4 l0 = *reinterpret_cast<const uint4*>(row + 128), l1 = *reinterpret_cast<const uint4*>(row + 192);
    const uint32_t s2 = *reinterpret_cast<const uint16_t*>(cur + kPBM * kQPitch + (16 * tt + m) * 8 + 2 * kb);
    const int sh = (int)(s2 & 0xff), sl = (int)(s2 >> 8);
    const mfma_i32x8_t ah = {(int)h0.x, (int)h0.y, (int)h0.z, (int)h0.w, (int)h1.x, (int)h1.y, (int)h1.z, (int)h1.w};
    const mfma_i32x8_t al = {(int)l0.x, (int)l0.y, (int)l0.z, (int)l0.w, (int)l1.x, (int)l1.y, (int)l1.z, (int)l1.w};
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      acc[tt][nb] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(ah, b[nb], acc[tt][nb], 0, 4, 0, sh, 0, sb[nb]);
      acc[tt][nb] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(al, b[nb], acc[tt][nb], 0, 4, 0, sl, 0, sb[nb]);
    }
  }
}

// The MFMAs of k-tile t on bf16 rows: the E2M1 codes x 2^(s - 127) converted to bf16 (exact), 16 conversions per row
// block and k-tile shared by the tile's 16-token blocks.  By itself v_mfma_f32_16x16x32_bf16 is the slower exact route
// (1,546 TFLOP/s when nothing else runs, against 2,391 of the scaled instruction on hi and lo rows); these kernels stay
// below either, and gain from not quantising their rows, which each of the 15 to 30 column groups repeated: about 220
// vector instructions per k-tile of a full tile against the 48 conversions.  MFMA j multiplies elements 8 j .. 8 j + 7
// of each of the k-tile's four 32-element groups (lane 16 kb + m: group kb), on both operands.
template <int W, int NB, int NT>
NA_DEVICE void ktile_bf16(int t, WStream<W, NB>& ws, const uint8_t* cur, const uint4 (&c)[NB],
                          f32x4_t (&acc)[4][NB]) {
  const int lane = threadIdx.x & 63, kb = lane >> 4, m = lane & 15;
  uint4 b[NB][4];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    const bool in = 4 * t + kb < kGK;
    const uint32_t w[4] = {in ? c[nb].x : 0u, in ? c[nb].y : 0u, in ? c[nb].z : 0u, in ? c[nb].w : 0u};
    const uint32_t sb = (uint32_t)ws.scale(t, nb) & 0xff;
    ws.top = max(ws.top, sb);
    const float s = e8m0_f32(sb);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      b[nb][j] = make_uint4(fp4x2_scaled<0>(w[j], s), fp4x2_scaled<1>(w[j], s), fp4x2_scaled<2>(w[j], s),
                            fp4x2_scaled<3>(w[j], s));
  }
  __builtin_amdgcn_s_setprio(1);
#pragma unroll
  for (int tt = 0; tt < NT; ++tt) {
    const uint8_t* row = cur + (16 * tt + m) * kQPitch + 64 * kb;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const bf16x8_t a = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4*>(row + 16 * j));
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
        acc[tt][nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, __builtin_bit_cast(bf16x8_t, b[nb][j]), acc[tt][nb],
                                                              0, 0, 0);
    }
  }
}

// One k-tile of gemm8_tile.  A of k-tile t is staged in LDS at cur and the weights of k-tile t are in c.  It
// issues the loads of A of k-tile t + 2 (into a_in) and of the weights of k-tile t + 2 (into c2), runs the
// MFMAs, stores A of k-tile t + 1 (loaded one step earlier, a_out) at nxt and meets the barrier.
template <int W, int NB, int NT, typename S>
NA_DEVICE void gemm8_step(int t, WStream<W, NB>& ws, bool live, const S& st, const uint8_t* cur, uint8_t* nxt,
                          const typename S::template Stage<NT>& a_out, typename S::template Stage<NT>& a_in,
                          const uint4 (&c)[NB], uint4 (&c2)[NB], f32x4_t (&acc)[4][NB]) {
  const int tid = threadIdx.x;
  if (t + 2 < kPTiles) {
    st.template load<NT>(t + 2, tid, a_in);
    ws.load(t + 2, c2);
  }
  if (live) {
    if constexpr (S::kBf16) ktile_bf16<W, NB, NT>(t, ws, cur, c, acc);
    else ktile_x8<W, NB, NT>(t, ws, cur, c, acc);
  }
  // The MFMAs are issued before the LDS stores, which wait for their k-tile's loads: an empty asm that takes every
  // accumulator (and orders memory) keeps the compiler from sinking the MFMAs below those stores.
#pragma unroll
  for (int tt = 0; tt < NT; ++tt)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) asm volatile("" : "+v"(acc[tt][nb])::"memory");
  __builtin_amdgcn_s_setprio(0);
  if (t + 1 < kPTiles) st.template store<NT>(nxt, tid, a_out);
  __syncthreads();
}

// acc[tt][nb] = D of tokens 16 tt .. 16 tt + 15 x row block blk[nb] (lane (q, n): tokens 16 tt + 4 q + r, row n),
// over the 23 k-tiles for tt < NT (the 16-token blocks that hold rows; the others stay zero); st stages the
// activation rows (QRows or BRows).  Both
// operand streams run two k-tiles ahead of the MFMAs: the activations through three LDS buffers of a k-tile (64 rows'
// 256 code bytes and 8 scale bytes each, loaded into registers two steps before and stored one step before their
// use), each wave's weight codes through three register sets; the k-loop is unrolled by 3 so that every buffer and
// register set is fixed at compile time.  Each wave reads one token tile's hi and lo fragments at a time and feeds
// them to its NB row blocks.  lds: 3 x kQStage bytes; wsc: this wave's LDS area of NB x 1,536 bytes (staged
// scale rows).  A wave without work (live = false) stages and meets every barrier but runs no MFMA.  All 256 threads must
// call it.
template <int W, int NB, int NT, typename S>
NA_DEVICE void gemm8_tile_n(WStream<W, NB>& ws, bool live, const S& st, uint8_t* lds,
                            f32x4_t (&acc)[4][NB]) {
  const int tid = threadIdx.x, lane = tid & 63;
#pragma unroll
  for (int tt = 0; tt < 4; ++tt)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[tt][nb] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  uint4 wsv[NB][WStream<W, NB>::kScRounds];
  ws.load_scales(wsv);
  uint8_t* const b0 = lds;
  uint8_t* const b1 = lds + kQStage;
  uint8_t* const b2 = lds + 2 * kQStage;
  uint4 c0[NB], c1[NB], c2[NB];
  typename S::template Stage<NT> a0, a1, a2;           // a_k: A of the k-tiles = k (mod 3) while in flight
  ws.load(0, c0);
  ws.load(1, c1);
  __builtin_amdgcn_sched_barrier(0);                   // the weights are requested before the row addresses are awaited
  st.template load<NT>(0, tid, a0);
  st.template load<NT>(1, tid, a1);
  __builtin_amdgcn_sched_barrier(0);                   // every load above is issued before the first wait
  ws.store_scales(wsv);
  st.template store<NT>(b0, tid, a0);
  __syncthreads();
  int t = 0;
  for (; t + 3 <= kPTiles; t += 3) {                   // k-tiles 0 .. 20
    gemm8_step<W, NB, NT, S>(t, ws, live, st, b0, b1, a1, a2, c0, c2, acc);
    gemm8_step<W, NB, NT, S>(t + 1, ws, live, st, b1, b2, a2, a0, c1, c0, acc);
    gemm8_step<W, NB, NT, S>(t + 2, ws, live, st, b2, b0, a0, a1, c2, c1, acc);
  }
  gemm8_step<W, NB, NT, S>(t, ws, live, st, b0, b1, a1, a2, c0, c2, acc);       // 21
  gemm8_step<W, NB, NT, S>(t + 1, ws, live, st, b1, b2, a2, a0, c1, c0, acc);   // 22
}

// acc of gemm8_tile again where one of the wave's scale bytes is kE8m0Wide or more: there a weight may be past bf16's
// range though its product with a small x is finite, as the scaled instruction and the GEMV have it.  A quarter of every
// weight is inside the range, and four equal products are added in the place of one.  One wave by itself, without
// barriers: fragments straight from the rows and codes, scales from the wave's LDS area.  Such bytes (weights of 2^126
// and more) occur in no trained model, so this is kept small, not fast; the test for them is one maximum per conversion
// and one branch per tile (a branch per k-tile cost 40 to 90 spilled registers).
template <int W, int NB>
NA_DEVICE void gemm8_wide(const WStream<W, NB>& ws, const BRows& st, int ntt, f32x4_t (&acc)[4][NB]) {
  const int kb = ws.lane >> 4, m = ws.lane & 15;
#pragma unroll
  for (int tt = 0; tt < 4; ++tt)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[tt][nb] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
  for (int t = 0; t < kPTiles; ++t) {
    const bool in = 4 * t + kb < kGK;
    uint4 c[NB];
    ws.load(t, c);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      bf16x8_t a[4];
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) {
        uint4 v = make_uint4(0, 0, 0, 0);
        if (in && tt < ntt) v = *reinterpret_cast<const uint4*>(st.row(16 * tt + m) + t * kPKT + 32 * kb + 8 * j);
        a[tt] = __builtin_bit_cast(bf16x8_t, v);
      }
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        const uint32_t cw[4] = {c[nb].x, c[nb].y, c[nb].z, c[nb].w};
        const uint32_t w = in ? cw[j] : 0u, sb = (uint32_t)ws.scale(t, nb) & 0xff;
        const bf16x8_t b = __builtin_bit_cast(bf16x8_t, make_uint4(fp4x2_quarter<0>(w, sb), fp4x2_quarter<1>(w, sb),
                                                                   fp4x2_quarter<2>(w, sb), fp4x2_quarter<3>(w, sb)));
#pragma unroll 1
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int tt = 0; tt < 4; ++tt)
            acc[tt][nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[tt], b, acc[tt][nb], 0, 0, 0);
      }
    }
  }
}

// gemm8_tile_n for a tile whose rows fill ntt (1..4) 16-token blocks: empty blocks are neither staged nor multiplied.
// ntt is workgroup-uniform.
template <int W, int NB, typename S>
NA_DEVICE void gemm8_tile(const WSrc& src, const int (&blk)[NB], bool live, int ntt, const S& st, uint8_t* lds,
                          uint8_t* wsc, f32x4_t (&acc)[4][NB]) {
  WStream<W, NB> ws{src, blk, wsc, (int)(threadIdx.x & 63), {}, 0};
  if (ntt > 3)
    gemm8_tile_n<W, NB, 4, S>(ws, live, st, lds, acc);
  else if (ntt == 3)
    gemm8_tile_n<W, NB, 3, S>(ws, live, st, lds, acc);
  else if (ntt == 2)
    gemm8_tile_n<W, NB, 2, S>(ws, live, st, lds, acc);
  else
    gemm8_tile_n<W, NB, 1, S>(ws, live, st, lds, acc);
  if constexpr (S::kBf16)
    if (__any(ws.top >= kE8m0Wide)) gemm8_wide<W, NB>(ws, st, ntt, acc);
}

// Workgroup b -> (tile, column group): the dispatcher deals workgroups to the 8 XCDs in turn (XCD b % 8), so XCD x
// is given column groups slots * x .. slots * x + slots - 1 of every tile, tiles in order.  Each XCD's L2 then holds
// the weight rows of its few column groups while the tiles of one expert pass through it, and every weight byte
// crosses from HBM about once.
template <int SLOTS>
NA_DEVICE void xcd_tile(int b, int& tile, int& col) {
  const int s = b >> 3;
  tile = s / SLOTS;
  col = SLOTS * (b & 7) + s % SLOTS;
}

// What bounds it, from stamps of every workgroup (one expert's rows in full tiles, 4 x 1,024 rows, 1,472 workgroups):
// two workgroups on a CU for 81 % of the launch (1.74 on average: six a CU in three rounds, then a part-empty end), each
// 77,300 cycles: 5,800 before its first k-tile, 23 k-tiles of 2,616, of which the two waves of a SIMD fill 2,048 with
// MFMAs, 11,300 of epilogue (32 activations per lane).  The clock is 1.92 GHz under this load (2.2 with one workgroup on
// a third of the CUs, 2.28 by the rate of the bare MFMA loop): matrix cores busy for 0.51 of the cycles, 1,015 TFLOP/s =
// 0.42 of that loop's rate.  Over 128 experts (2,048 Zipf tokens) the clock falls to 1.6 GHz, and a tile of one 16-row
// block takes 55 % of a full one's time for a quarter of its MFMAs.
// The weights, their scales and the row addresses requested side by side, and an epilogue on the hardware exponential,
// block maxima of one instruction per step and shared conversions: 2,048 tokens 665 -> 630 us, 23 tokens 191 -> 182.
//
// gate_up + bias + clamped SwiGLU on the block-scaled MFMA: tile i, column group y (128 intermediate columns).
// Wave w owns intermediate blocks jb, jb + 1 (jb = 8 y + 2 w) and reads their gate rows (blocks jb, jb + 1) and up
// rows (blocks 180 + jb, 181 + jb), so the SwiGLU pairs registers of one lane.  x rows come quantised (xq, one q row
// per token) and are gathered through the pair order; h leaves as q rows in sorted pair order, each 32-column block
// (one wave's columns of one row) with its own E8M0 scales.  Grid: max tiles x 24 (xcd_tile<3>); in column group 22
// waves 2 and 3 have no blocks.
template <int W>
__global__ __launch_bounds__(256, 2) void k_prefill_gate_up(
    const uint8_t* __restrict__ xq, const int* __restrict__ order, const PTile* __restrict__ tiles,
    const int* __restrict__ ntiles, const uint8_t* __restrict__ pool, long long slot_bytes,
    const int64_t* __restrict__ slot_tab, long long expert_base, const uint16_t* __restrict__ bias_gu,
    uint8_t* __restrict__ hq, float alpha, float limit) {
  __shared__ __align__(16) uint8_t lds[3 * kQStage + 4 * 4 * kWScBytes];
  int ti, y;
  xcd_tile<kGuSlots>(blockIdx.x, ti, y);
  const int nt_all = *ntiles;
  const PTile tl = tiles[ti];                          // read beside the count: the table holds max tiles
  if (ti >= nt_all || y >= 23) return;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, q = lane >> 4,
            n = lane & 15;
  const int jb = 8 * y + 2 * wave;
  const bool live = jb < kTUpBlock0;
  const int jl = live ? jb : 0;
  const int blk[4] = {jl, jl + 1, kTUpBlock0 + jl, kTUpBlock0 + jl + 1};
  const long long gid = expert_base + tl.e;
  const long long slot = slot_tab ? slot_tab[gid] : gid;
  const uint8_t* sb = pool + slot * slot_bytes;
  const WSrc src = W == kWT950 ? WSrc{sb, nullptr} : WSrc{sb, sb + kOffGateScales};
  QRows st;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    st.rp[i] = xq + (long long)(order[tl.p0 + min((tid >> 4) + 16 * i, tl.cnt - 1)] >> 2) * kQRow;
  st.srow = xq + (long long)(order[tl.p0 + min(tid & 63, tl.cnt - 1)] >> 2) * kQRow;
  f32x4_t acc[4][4];
  const int ntt = (tl.cnt + 15) >> 4;
  gemm8_tile<W, 4>(src, blk, live, ntt, st, lds, lds + 3 * kQStage + wave * 4 * kWScBytes, acc);
  // h = bf16(SwiGLU(bf16(acc) + bias)) (the reference's bf16 rounding points), quantised per (row, 32-column block)
  // into LDS: oh[row] = hi codes of the workgroup's 128 columns | lo codes, os[row] = 4 hi | 4 lo scale bytes.
  uint8_t* oh = lds;
  uint8_t* os = lds + kPBM * kOhPitch;
  if (live) {
    const uint16_t* bg = bias_gu ? bias_gu + gid * kGU : nullptr;
    float bgv[2], buv[2];
    uint32_t sh_own = 0, sl_own = 0;
#pragma unroll
    for (int hb = 0; hb < 2; ++hb) {
      const int j = 16 * (jl + hb) + n;
      bgv[hb] = bg ? bf16_to_f32(bg[j]) : -0.f;        // x + -0 is x, signed zeros included
      buv[hb] = bg ? bf16_to_f32(bg[kI + j]) : -0.f;
    }
#pragma unroll
    for (int tt = 0; tt < 4; ++tt) {
      if (tt >= ntt) break;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float g[2] = {acc[tt][0][r], acc[tt][1][r]}, u[2] = {acc[tt][2][r], acc[tt][3][r]}, hv[2];
        rb2(g[0], g[1]);
        rb2(u[0], u[1]);
#pragma unroll
        for (int hb = 0; hb < 2; ++hb) {
          g[hb] += bgv[hb];
          u[hb] += buv[hb];
        }
        rb2(g[0], g[1]);
        rb2(u[0], u[1]);
        swiglu_clamp_bf16_2(g, u, alpha, limit, hv);
        const uint32_t mx = max(__float_as_uint(hv[0]) & 0x7fffffffu, __float_as_uint(hv[1]) & 0x7fffffffu);
        const uint32_t sh = x8_scale_byte(__uint_as_float(row16_umax(mx)));
        const float s_hi = e8m0_f32(sh);
        fp8x2_t o2 = {0, 0};
        o2 = __builtin_amdgcn_cvt_scalef32_pk_fp8_f32(o2, hv[0], hv[1], s_hi, false);
        const uint32_t hc = __builtin_bit_cast(uint32_t, o2);
        const auto d = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(hc, s_hi, false);
        const float r0 = hv[0] - d[0], r1 = hv[1] - d[1];
        const uint32_t mr = row16_umax(__float_as_uint(fmaxf(fabsf(r0), fabsf(r1))));
        const uint32_t sl = x8_scale_byte(__uint_as_float(mr));
        fp8x2_t l2 = {0, 0};
        l2 = __builtin_amdgcn_cvt_scalef32_pk_fp8_f32(l2, r0, r1, e8m0_f32(sl), false);
        const uint32_t lc = __builtin_bit_cast(uint32_t, l2);
        const int row = 16 * tt + 4 * q + r, c = 32 * wave + n;
        oh[row * kOhPitch + c] = (uint8_t)hc;
        oh[row * kOhPitch + c + 16] = (uint8_t)(hc >> 8);
        oh[row * kOhPitch + kPKT + c] = (uint8_t)lc;
        oh[row * kOhPitch + kPKT + c + 16] = (uint8_t)(lc >> 8);
        if (n == 4 * tt + r) {                         // a select: lane n keeps the scales of its row, written below
          sh_own = sh;
          sl_own = sl;
        }
      }
    }
    if ((n >> 2) < ntt) {                              // lane (q, n): row 16 (n / 4) + 4 q + n % 4
      const int row = 16 * (n >> 2) + 4 * q + (n & 3);
      os[row * 8 + wave] = (uint8_t)sh_own;
      os[row * 8 + 4 + wave] = (uint8_t)sl_own;
    }
  }
  __syncthreads();
  // q rows out: 16-byte pieces of the valid columns (64 in column group 22), scale bytes 4 y .. 4 y + 3 (group 22:
  // bytes 88, 89 and the zero padding 90..95).
  const int ncol = y == 22 ? 64 : 128;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int pc = tid + 256 * i, row = pc >> 4, c16 = pc & 15, c8 = c16 & 7;
    if (row < tl.cnt && 16 * c8 < ncol) {
      const uint2 a0 = *reinterpret_cast<const uint2*>(oh + row * kOhPitch + 16 * c16);
      const uint2 a1 = *reinterpret_cast<const uint2*>(oh + row * kOhPitch + 16 * c16 + 8);
      *reinterpret_cast<uint4*>(hq + (long long)(tl.p0 + row) * kQRow + (c16 >> 3) * kQLo + kPKT * y + 16 * c8) =
          make_uint4(a0.x, a0.y, a1.x, a1.y);
    }
  }
  if (tid < tl.cnt && tid < kPBM) {
    uint8_t* dst = hq + (long long)(tl.p0 + tid) * kQRow;
    const uint32_t sh4 = *reinterpret_cast<const uint32_t*>(os + tid * 8);
    const uint32_t sl4 = *reinterpret_cast<const uint32_t*>(os + tid * 8 + 4);
    if (y < 22) {
      *reinterpret_cast<uint32_t*>(dst + kQSh + 4 * y) = sh4;
      *reinterpret_cast<uint32_t*>(dst + kQSl + 4 * y) = sl4;
    } else {
      *reinterpret_cast<uint2*>(dst + kQSh + 88) = make_uint2(sh4 & 0xffff, 0);
      *reinterpret_cast<uint2*>(dst + kQSl + 88) = make_uint2(sl4 & 0xffff, 0);
    }
  }
}

// down + bias, x routing weight, scattered back to pair order: ys[p][n] = bf16(bf16(bf16(y) + b) * w[p]) with p the
// pair of sorted position p0 + m.  A = the h q rows of the tile (consecutive sorted positions).  Grid: max tiles x 16
// (xcd_tile<2>); wave w: row blocks 12 y + 3 w + i.
template <int W>
__global__ __launch_bounds__(256, 2) void k_prefill_down(
    const uint8_t* __restrict__ hq, const int* __restrict__ order, const PTile* __restrict__ tiles,
    const int* __restrict__ ntiles, const uint16_t* __restrict__ wts, const uint8_t* __restrict__ pool,
    long long slot_bytes, const int64_t* __restrict__ slot_tab, long long expert_base,
    const uint16_t* __restrict__ bias_dn, uint16_t* __restrict__ ys) {
  __shared__ __align__(16) uint8_t lds[3 * kQStage + 4 * kPNB * kWScBytes];
  int ti, y;
  xcd_tile<kDnSlots>(blockIdx.x, ti, y);
  const int nt_all = *ntiles;
  const PTile tl = tiles[ti];                          // read beside the count: the table holds max tiles
  if (ti >= nt_all || y >= kH / kPRows) return;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, q = lane >> 4,
            n = lane & 15;
  int blk[kPNB];
#pragma unroll
  for (int i = 0; i < kPNB; ++i) blk[i] = y * (4 * kPNB) + kPNB * wave + i;
  const long long gid = expert_base + tl.e;
  const long long slot = slot_tab ? slot_tab[gid] : gid;
  const uint8_t* sb = pool + slot * slot_bytes;
  const WSrc src = W == kWT950 ? WSrc{sb + kTDownOff, nullptr}
                               : WSrc{sb + kOffDownCodes, sb + kOffGateScales + (long long)kGU * (W == kWRaw ? kGK : kPs4Row)};
  QRows st;
#pragma unroll
  for (int i = 0; i < 4; ++i) st.rp[i] = hq + (long long)(tl.p0 + min((tid >> 4) + 16 * i, tl.cnt - 1)) * kQRow;
  st.srow = hq + (long long)(tl.p0 + min(tid & 63, tl.cnt - 1)) * kQRow;
  f32x4_t acc[4][kPNB];
  const int ntt = (tl.cnt + 15) >> 4;
  gemm8_tile<W, kPNB>(src, blk, true, ntt, st, lds, lds + 3 * kQStage + wave * kPNB * kWScBytes, acc);
  // y = bf16(bf16(bf16(acc) + b) * w[p]) per element, staged as the tile's 64 rows x 192 columns in LDS (the A stages
  // are free after the last k-tile's barrier), then written back with 16-byte stores: one 384-byte piece per pair.
  uint8_t* yt = lds;
  float wv[4][4];                                     // routing weight of each of the lane's 16 tokens
#pragma unroll
  for (int tt = 0; tt < 4; ++tt)
#pragma unroll
    for (int r = 0; r < 4; ++r) wv[tt][r] = bf16_to_f32(wts[order[tl.p0 + min(16 * tt + 4 * q + r, tl.cnt - 1)]]);
#pragma unroll
  for (int nb = 0; nb < kPNB; ++nb) {
    const int cl = 16 * (kPNB * wave + nb) + n;        // column within the workgroup's 192
    const float bd = bias_dn ? bf16_to_f32(bias_dn[gid * kH + 16 * blk[nb] + n]) : 0.f;
#pragma unroll
    for (int tt = 0; tt < 4; ++tt) {
      if (tt >= ntt) break;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float yv = rb(acc[tt][nb][r]);
        if (bias_dn) yv = rb(yv + bd);
        const uint32_t v = f32_to_bf16(yv * wv[tt][r]);
        const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xF, 0xF, false) & 0xffff;
        if (!(n & 1))
          *reinterpret_cast<uint32_t*>(yt + (16 * tt + 4 * q + r) * kYPitch + 2 * cl) = v | (hi << 16);
      }
    }
  }
  __syncthreads();
  constexpr int kPieces = kPRows * 2 / 16;            // 24 pieces of 16 bytes per row
#pragma unroll
  for (int i = 0; i < kPBM * kPieces / 256; ++i) {
    const int pc = tid + 256 * i, row = pc / kPieces, piece = pc - row * kPieces;
    if (row < tl.cnt)
      *reinterpret_cast<uint4*>(ys + (long long)order[tl.p0 + row] * kH + kPRows * y + 8 * piece) =
          *reinterpret_cast<const uint4*>(yt + row * kYPitch + 16 * piece);
  }
}

// ------------------------------------------------------------------------------- plain GEMM (mxfp4_gemm)
// out[e][m][n] = bf16(sum_k x[m][k] w_e[n][k]); tiles = E * ceil(M / 64) of 64 rows; column group y, wave w: row
// blocks 12 y + 3 w + i.
// The fused layer's tiles on bf16 rows (ktile_bf16).
NA_DEVICE void store_tile(uint16_t* out_row0, long long pitch, const f32x4_t (&acc)[4][kPNB], const int (&blk)[kPNB],
                          int m_limit) {
  const int lane = threadIdx.x & 63, q = lane >> 4, n = lane & 15;
#pragma unroll
  for (int nb = 0; nb < kPNB; ++nb)
#pragma unroll
    for (int tt = 0; tt < 4; ++tt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = 16 * tt + 4 * q + r;
        const uint32_t v = f32_to_bf16(acc[tt][nb][r]);
        const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xF, 0xF, false) & 0xffff;
        if (m < m_limit && !(n & 1))
          *reinterpret_cast<uint32_t*>(out_row0 + (long long)m * pitch + 16 * blk[nb] + n) = (uint32_t)v | (hi << 16);
      }
}

// Workgroup of the GEMM entry points -> (tile, column group of 192 rows), a linear grid.  slots > 0: xcd_tile's order
// with `slots` column groups per XCD, so that each weight row stays in one XCD's L2 while the tiles of its expert pass;
// slots = 0 (few column groups, which would leave XCDs idle): column groups of a tile in turn.
NA_DEVICE void gemm_tile_col(int b, int slots, int cols, int& tile, int& col) {
  if (slots > 0) {
    const int s = b >> 3;
    tile = s / slots;
    col = slots * (b & 7) + (s - tile * slots);
  } else {
    tile = b / cols;
    col = b - tile * cols;
  }
}

template <int W>
__global__ __launch_bounds__(256, 2) void k_mxfp4_gemm(const uint16_t* __restrict__ x, int M,
                                                       const uint8_t* __restrict__ blocks, long long sb_slot,
                                                       const uint8_t* __restrict__ scales, long long ss_slot,
                                                       const int64_t* __restrict__ slots, uint16_t* __restrict__ out,
                                                       int N, int xcd_slots, int tile0) {
  __shared__ __align__(16) uint8_t lds[3 * kQStage + 4 * kPNB * kWScBytes];
  const int mt = (M + kPBM - 1) / kPBM;
  int i, y;
  gemm_tile_col(blockIdx.x, xcd_slots, N / kPRows, i, y);
  i += tile0;
  if (y >= N / kPRows) return;
  const int e = i / mt, m0 = (i - e * mt) * kPBM;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int blk[kPNB];
#pragma unroll
  for (int i = 0; i < kPNB; ++i) blk[i] = y * (4 * kPNB) + kPNB * wave + i;
  const WSrc src = w_src<W>(blocks, sb_slot, scales, ss_slot, slots[e]);
  const BRows st(x + (long long)m0 * kH, M - 1 - m0, tid);
  f32x4_t acc[4][kPNB];
  const int ntt = (min(M - m0, kPBM) + 15) >> 4;
  gemm8_tile<W, kPNB>(src, blk, true, ntt, st, lds, lds + 3 * kQStage + wave * kPNB * kWScBytes, acc);
  store_tile(out + ((long long)e * M + m0) * N, N, acc, blk, M - m0);
}

// --------------------------------------------------------------- grouped GEMM (GroupedGemmPlan descriptors)
// tiles int64 [ntiles][5] = (x address, out address, slot, pair M, pm); rows [pm * block_m, min(M, pm * block_m +
// block_m)) of the pair, as sub-tiles of 64 rows (block_m <= 64: one).
template <int W>
__global__ __launch_bounds__(256, 2) void k_mxfp4_gemm_grouped(const uint8_t* __restrict__ blocks, long long sb_slot,
                                                               const uint8_t* __restrict__ scales, long long ss_slot,
                                                               const int64_t* __restrict__ tiles, int block_m, int N,
                                                               int xcd_slots) {
  __shared__ __align__(16) uint8_t lds[3 * kQStage + 4 * kPNB * kWScBytes];
  const int sub = max(block_m / kPBM, 1);              // 64-row sub-tiles per tile, one workgroup each
  int i, y;
  gemm_tile_col(blockIdx.x, xcd_slots, N / kPRows, i, y);
  if (y >= N / kPRows) return;
  const int64_t* d = tiles + (long long)(i / sub) * 5;
  const uint16_t* x = reinterpret_cast<const uint16_t*>(d[0]);
  uint16_t* out = reinterpret_cast<uint16_t*>(d[1]);
  const long long slot = d[2];
  const int M = (int)d[3], pm = (int)d[4];
  const long long row0 = (long long)pm * block_m + (i % sub) * kPBM;
  const int r1 = (int)min((long long)M, (pm + 1LL) * block_m);
  if (row0 >= r1) return;
  const int m0 = (int)row0;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int blk[kPNB];
#pragma unroll
  for (int i = 0; i < kPNB; ++i) blk[i] = y * (4 * kPNB) + kPNB * wave + i;
  const WSrc src = w_src<W>(blocks, sb_slot, scales, ss_slot, slot);
  const BRows st(x + (long long)m0 * kH, r1 - 1 - m0, tid);
  f32x4_t acc[4][kPNB];
  const int ntt = (min(r1 - m0, kPBM) + 15) >> 4;
  gemm8_tile<W, kPNB>(src, blk, true, ntt, st, lds, lds + 3 * kQStage + wave * kPNB * kWScBytes, acc);
  store_tile(out + (long long)m0 * N, N, acc, blk, r1 - m0);
}

// out[t][n] = bf16(sum_k ys[4 t + k][n]) over the valid ranks k, fp32 sum in top-k order (server.py:2340-2341).
// One thread per 8 columns of a token: 16-byte loads of the four ranks' rows, one 16-byte store.
__global__ __launch_bounds__(256) void k_prefill_combine(const uint16_t* __restrict__ ys, const int64_t* __restrict__ ids,
                                                         int T, uint16_t* __restrict__ out) {
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i >= (long long)T * (kH / 8)) return;
  const int t = (int)(i / (kH / 8)), c8 = (int)(i - (long long)t * (kH / 8));
  float a[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  uint4 v[4];
  bool ok[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {                       // all four loads in flight before the sums
    const long long e = ids[4 * t + k];
    ok[k] = e >= 0 && e < 128;
    v[k] = ok[k] ? *reinterpret_cast<const uint4*>(ys + (long long)(4 * t + k) * kH + 8 * c8) : make_uint4(0, 0, 0, 0);
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    if (!ok[k]) continue;
    const uint32_t w[4] = {v[k].x, v[k].y, v[k].z, v[k].w};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      a[2 * j] += bf16_to_f32((uint16_t)(w[j] & 0xffff));
      a[2 * j + 1] += bf16_to_f32((uint16_t)(w[j] >> 16));
    }
  }
  uint4 o;
  o.x = (uint32_t)f32_to_bf16(a[0]) | ((uint32_t)f32_to_bf16(a[1]) << 16);
  o.y = (uint32_t)f32_to_bf16(a[2]) | ((uint32_t)f32_to_bf16(a[3]) << 16);
  o.z = (uint32_t)f32_to_bf16(a[4]) | ((uint32_t)f32_to_bf16(a[5]) << 16);
  o.w = (uint32_t)f32_to_bf16(a[6]) | ((uint32_t)f32_to_bf16(a[7]) << 16);
  *reinterpret_cast<uint4*>(out + (long long)t * kH + 8 * c8) = o;
}

// Workspace of the fused prefill layer for T tokens (P = 4 T pairs): byte offsets, 256-aligned.
struct PrefillWs {
  long long counts, ntiles, order, tiles, xq, h, ys, total;
  int max_tiles;
};

static long long align256(long long v) { return (v + 255) & ~255LL; }

static PrefillWs prefill_ws(int T) {
  PrefillWs w;
  const long long P = 4LL * T;
  w.max_tiles = (int)(P / kPBM + 128);
  w.counts = 0;
  w.ntiles = 512;
  w.order = 1024;
  w.tiles = align256(w.order + P * 4);
  w.xq = align256(w.tiles + (long long)w.max_tiles * sizeof(PTile));
  w.h = align256(w.xq + (long long)T * kQRow);
  w.ys = align256(w.h + P * kQRow);
  w.total = align256(w.ys + P * kH * 2);
  return w;
}

// Grid of the GEMM entry points (gemm_tile_col): workgroups per tile of N / 192 column groups, in the XCD order where
// its 8 x slots column groups are at least 7/8 in use (N = 5760: 30 of 32, N = 2880: 15 of 16), else the plain order.
static int gemm_wgs_per_tile(int N, int& xcd_slots) {
  const int cols = N / kPRows, slots = (cols + 7) / 8;
  xcd_slots = 8 * cols >= 7 * 8 * slots ? slots : 0;
  return xcd_slots ? 8 * slots : cols;
}

// Workgroups of 256 threads in one launch: a grid dimension holds fewer than 2^32 threads.  The entry points launch
// more tiles than that in several grids (1,048,576 one-row tiles of 2,880 columns, say).
constexpr long long kMaxWgs = 0xffffffffLL / 256;

template <typename... KArgs, typename... Args>
static void launch_p(void (*kern)(KArgs...), dim3 grid, dim3 block, hipStream_t stream, hipEvent_t e0, hipEvent_t e1,
                     Args... args) {
  if (e0 || e1)
    hipExtLaunchKernelGGL(kern, grid, block, 0, stream, e0, e1, 0, static_cast<KArgs>(args)...);
  else
    hipLaunchKernelGGL(kern, grid, block, 0, stream, static_cast<KArgs>(args)...);
}

}  // namespace na

using namespace na;

extern "C" {

long long na_moe_prefill_workspace_bytes(int T) {
  if (T <= 0 || T > (1 << 20)) return -1;
  return prefill_ws(T).total;
}

int na_moe_prefill_workspace_layout(int T, long long* offsets) {
  if (T <= 0 || T > (1 << 20) || !offsets) return kErrArgs;
  const PrefillWs w = prefill_ws(T);
  const long long v[9] = {w.counts, w.ntiles, w.order, w.tiles, w.xq, w.h, w.ys, w.total, w.max_tiles};
  for (int i = 0; i < 9; ++i) offsets[i] = v[i];
  return kOk;
}

int na_moe_prefill(const void* x, const int64_t* topk_ids, const void* topk_w, int T, const void* pool,
                   long long slot_bytes, int layout, const int64_t* slot_tab, long long expert_base,
                   const void* bias_gu, const void* bias_dn, void* workspace, long long ws_bytes, void* out,
                   float alpha, float limit, void* const* events, hipStream_t stream) {
  if (!x || !topk_ids || !topk_w || !pool || !workspace || !out || T <= 0 || T > (1 << 20)) return kErrArgs;
  if (layout < kWRaw || layout > kWT950) return kErrArgs;
  const long long need = layout == kWT950 ? kTSlot : layout == kWPs4 ? kSlotPs4 : kSlotRaw;
  if (slot_bytes < need || (slot_bytes & 15) || (reinterpret_cast<uintptr_t>(pool) & 15)) return kErrArgs;
  if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(workspace) | reinterpret_cast<uintptr_t>(out)) & 15)
    return kErrArgs;
  const PrefillWs w = prefill_ws(T);
  if (ws_bytes < w.total) return kErrTooLarge;
  uint8_t* ws = (uint8_t*)workspace;
  int* counts = (int*)(ws + w.counts);
  int* ntiles = (int*)(ws + w.ntiles);
  int* order = (int*)(ws + w.order);
  PTile* tiles = (PTile*)(ws + w.tiles);
  uint8_t* xq = ws + w.xq;
  uint8_t* hq = ws + w.h;
  uint16_t* ys = (uint16_t*)(ws + w.ys);
  hipEvent_t ev[10] = {};
  if (events)
    for (int i = 0; i < 10; ++i) ev[i] = (hipEvent_t)events[i];
  const int P = 4 * T;
  const long long qblocks = ((long long)T * kChunks + 255) / 256;
  launch_p(k_prefill_route, dim3((unsigned)(128 + qblocks)), dim3(256), stream, ev[0], ev[1], topk_ids, P, counts, order,
           tiles, ntiles, (const uint16_t*)x, T, xq);
  for (int i = 2; i < 4; ++i)
    if (ev[i] && hipEventRecord(ev[i], stream) != hipSuccess) return kErrLaunch;
  const dim3 gg(w.max_tiles * 8 * kGuSlots), gd(w.max_tiles * 8 * kDnSlots), blk(256);
#define NA_PREFILL_GEMMS(W)                                                                                          \
  launch_p(k_prefill_gate_up<W>, gg, blk, stream, ev[4], ev[5], (const uint8_t*)xq, (const int*)order,                \
           (const PTile*)tiles, (const int*)ntiles, (const uint8_t*)pool, slot_bytes, slot_tab, expert_base,          \
           (const uint16_t*)bias_gu, hq, alpha, limit);                                                                \
  launch_p(k_prefill_down<W>, gd, blk, stream, ev[6], ev[7], (const uint8_t*)hq, (const int*)order,                    \
           (const PTile*)tiles, (const int*)ntiles, (const uint16_t*)topk_w, (const uint8_t*)pool, slot_bytes,        \
           slot_tab, expert_base, (const uint16_t*)bias_dn, ys);
  if (layout == kWT950) {
    NA_PREFILL_GEMMS(kWT950)
  } else if (layout == kWPs4) {
    NA_PREFILL_GEMMS(kWPs4)
  } else {
    NA_PREFILL_GEMMS(kWRaw)
  }
#undef NA_PREFILL_GEMMS
  const long long nc = (long long)T * (kH / 8);
  launch_p(k_prefill_combine, dim3((unsigned)((nc + 255) / 256)), dim3(256), stream, ev[8], ev[9],
           (const uint16_t*)ys, topk_ids, T, (uint16_t*)out);
  return hipGetLastError() == hipSuccess ? kOk : kErrLaunch;
}

int na_mxfp4_gemm(const void* x, int M, int K, const void* blocks, long long sb_slot, const void* scales,
                  long long ss_slot, int layout, const int64_t* slots, int E, void* out, int N, hipStream_t stream) {
  if (!x || !blocks || !slots || !out || M <= 0 || E <= 0 || N <= 0) return kErrArgs;
  if (K != kH || N % kPRows || layout < kWRaw || layout > kWT950 || (layout != kWT950 && !scales)) return kErrArgs;
  if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(out)) & 15) return kErrArgs;
  const long long mt = (M + kPBM - 1) / kPBM;
  if (mt * E > 0x7fffffff) return kErrTooLarge;
  int xcd_slots;
  const int per = gemm_wgs_per_tile(N, xcd_slots);
  const long long all = mt * E, step = kMaxWgs / per;
  if (step == 0) return kErrTooLarge;
  auto kern = layout == kWT950 ? k_mxfp4_gemm<kWT950> : layout == kWPs4 ? k_mxfp4_gemm<kWPs4> : k_mxfp4_gemm<kWRaw>;
  for (long long t0 = 0; t0 < all; t0 += step)
    hipLaunchKernelGGL(kern, dim3((unsigned)(min(step, all - t0) * per)), dim3(256), 0, stream, (const uint16_t*)x, M,
                       (const uint8_t*)blocks, sb_slot, (const uint8_t*)scales, ss_slot, slots, (uint16_t*)out, N,
                       xcd_slots, (int)t0);
  return hipGetLastError() == hipSuccess ? kOk : kErrLaunch;
}

int na_mxfp4_gemm_grouped(const void* blocks, long long sb_slot, const void* scales, long long ss_slot, int layout,
                          const int64_t* tiles, int ntiles, int block_m, int N, int K, hipStream_t stream) {
  if (!blocks || !tiles || ntiles < 0 || N <= 0) return kErrArgs;
  if (K != kH || N % kPRows || layout < kWRaw || layout > kWT950 || (layout != kWT950 && !scales)) return kErrArgs;
  if (block_m < 16 || (block_m & (block_m - 1)) || block_m > 4096) return kErrArgs;
  if (ntiles == 0) return kOk;
  int xcd_slots;
  const long long per = (long long)gemm_wgs_per_tile(N, xcd_slots) * max(block_m / kPBM, 1), step = kMaxWgs / per;
  if (step == 0) return kErrTooLarge;
  auto kern = layout == kWT950 ? k_mxfp4_gemm_grouped<kWT950>
            : layout == kWPs4 ? k_mxfp4_gemm_grouped<kWPs4> : k_mxfp4_gemm_grouped<kWRaw>;
  for (long long t0 = 0; t0 < ntiles; t0 += step)
    hipLaunchKernelGGL(kern, dim3((unsigned)(min(step, ntiles - t0) * per)), dim3(256), 0, stream,
                       (const uint8_t*)blocks, sb_slot, (const uint8_t*)scales, ss_slot, tiles + 5 * t0, block_m, N,
                       xcd_slots);
  return hipGetLastError() == hipSuccess ? kOk : kErrLaunch;
}

}  // extern "C"
