// Block-sparse FlashAttention-2 forward, head dimension 128, launches that fill the GPU.
//
// At D = 128 a wavefront that owns 64 queries would need all 512 registers of its SIMD and be bound by instruction issue.
// Here a row block belongs to a pair of wavefronts, 32 queries each (256 registers: two
// wavefronts per SIMD), which share one K and one V tile buffer: a workgroup is one pair, four
// workgroups fit a compute unit, and the grid has one workgroup per (head, row block) - the
// hardware's dispatcher balances the load - or, where that leaves the GPU idle, several that share a row block's list and
// whose parts a second launch sums (pair_split).  Heads are taken in groups
// of 8, head i of a group on XCD i (place.h), so that the
// row blocks resident on an XCD share one head's K and V in its L2; long row blocks of
// block-causal masks come first.  Two barriers per tile: in front of the one that frees the K buffer both wavefronts wait for their
// halves of V, in front of the one that frees V for those of the next K.  (Four, with waits of their own: 16 heads N = 8192 dense 641 -> 541 us,
// on another card 648 -> 572, keep 0.3 193 -> 187, 28 heads N = 2048 dense 72 -> 70, 16 heads N = 4000 token-causal 125 -> 122; block-causal masks the same.)
//
// Tile arithmetic, softmax and layouts are those of attn_fwd.hip (fa2_custom_mask/fa2_fwd.py:146-196
// of the reference), with a single block of 32 queries per wavefront.
#include "common.h"
#include "fwd_tile.h"
#include "kernel_util.h"

namespace bsattn {

constexpr int PAIR_D = 128;
constexpr int PAIR_COLS_CAP = 1024;                               // column indices of the row block kept in LDS
constexpr int PAIR_LDS_BYTES = 2 * 64 * 2 * PAIR_D + 512 + PAIR_COLS_CAP * 4;     // K tile, V tile, mask words, columns

// TAIL: N is not a multiple of 64 (as in attn_fwd.hip: the copy of the last tile repeats its last key, the scores beyond
// it are -inf, the queries beyond N are not written).
template <int DT, bool EW, bool TAIL>
__global__ __launch_bounds__(128, 2) void fwd_pair_kernel(const FwdParams prm) {
  constexpr int D = PAIR_D, KS = D / 16, DB = D / 32, CPR = D / 8, ROWB = 2 * D, TILE_BYTES = 64 * ROWB;
  constexpr bool BF16 = DT != 0;
  constexpr bool PB = DT == 2;                   // P rounded to bf16, second product in bf16 (V as it is)
  constexpr bool FOLD = !BF16;
  // V read before the softmax (see the loop).  (Elementwise masks too, since a query without mass is looked after by sum_limit and not
  // by every lane in every tile, which spilled V's registers with bf16: 32 heads N = 4000 token window of 1000 92 -> 86 us, token-causal
  // 210 -> 199, 16 heads N = 4000 token-causal 135 -> 125.)
  constexpr int HALF = CPR / 2;                  // copy instructions per wavefront and tile
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ln = lane & 31, g = lane >> 5;
  const int nb = prm.nb, BH = prm.B * prm.H;
  // linear id -> (head, row block): groups of 8 heads, one head per XCD (place.h), long row blocks first
  int chunk;
  const Place p = prm.place.of(blockIdx.x, chunk);
  const int bh = p.head, m = nb - 1 - p.item;
  if (m < 0) return;                             // padding of an incomplete last group
  const int b = (int)prm.per_batch.of((unsigned)bh), h = bh - b * prm.H;
  const int mh = (prm.Bm > 1 ? b : 0) * prm.Hm + (prm.Hm > 1 ? h : 0);
  const cint_ptr_t rp = (cint_ptr_t)(uintptr_t)(prm.row_ptr + (int64_t)mh * nb);
  // Q of this lane's query (second operand of S^T = K Q^T) depends on the block index only: asked for first, it
  // travels while the list is looked up and the first tiles are requested.
  const int64_t qrow = (int64_t)m * 64 + 32 * w + ln;          // this lane's query
  const bool exists = !TAIL || qrow < prm.N;
  const int valid = TAIL ? prm.N - (nb - 1) * 64 : 64, tail_cb = TAIL ? nb - 1 : -1;
  uintx4 qf[1][KS];
  {
    const unsigned short* qp = (const unsigned short*)prm.q + b * prm.qs[0] + h * prm.qs[1] + (exists ? qrow : prm.N - 1) * prm.qs[2];
#pragma unroll
    for (int s = 0; s < KS; ++s) qf[0][s] = *reinterpret_cast<const uintx4*>(qp + 16 * s + 8 * g);
  }
  int* lcols = reinterpret_cast<int*>(lds + 2 * TILE_BYTES + 512);
  const bool listed = EW || prm.mask == nullptr;
  int t0, t1;
  if (listed) { t0 = rp[m]; t1 = rp[m + 1]; }
  else { t0 = 0; t1 = columns_of_row<MASK_MAX_BLOCKS>(prm, b, h, m, lane, lcols, chunk == 0 && w == 0); }
  if (!EW && prm.split > 1) {                    // this workgroup's share of the row block's list (elementwise masks: launches that fill the GPU)
    const int len = t1 - t0;
    if (chunk == 0 && threadIdx.x == 0) prm.part_len[bh * nb + m] = len;
    t1 = t0 + (int)((int64_t)len * (chunk + 1) / prm.split);
    t0 = t0 + (int)((int64_t)len * chunk / prm.split);
    if (t0 == t1) return;                        // (pair_sum_parts_kernel knows which shares are empty)
  }
  void* obase = out_base(prm, b, h);
  if (t0 == t1) {                                // no kept tile: O = 0, lse = -inf
    if (!exists) return;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int i4 = 0; i4 < 4; ++i4)
        store_out4<BF16>(obase, qrow * prm.os[2] + 32 * db + 8 * i4 + 4 * g, prm.out_f32, 0.f, 0.f, 0.f, 0.f);
    if (prm.lse != nullptr && g == 0) prm.lse[(int64_t)bh * prm.N + qrow] = -INFINITY;
    return;
  }

  unsigned char* lds_k = lds;
  unsigned char* lds_v = lds + TILE_BYTES;
  const unsigned long long* lds_bits = reinterpret_cast<const unsigned long long*>(lds + 2 * TILE_BYTES);
  const unsigned lds_k_addr = (unsigned)(uintptr_t)(lds_ptr_t)lds;
  const unsigned lds_v_addr = lds_k_addr + TILE_BYTES;
  const unsigned lds_bits_addr = lds_k_addr + 2 * TILE_BYTES;

  const unsigned short* kg = (const unsigned short*)prm.k + b * prm.ks[0] + h * prm.ks[1];
  const unsigned short* vg = (const unsigned short*)prm.v + b * prm.vs[0] + h * prm.vs[1];
  const float qk_scale = prm.qk_scale;

  // column indices of the row block (EW: "partly set" in bit 30), staged once
  const cint_ptr_t cols = (cint_ptr_t)(uintptr_t)prm.col_idx;
  typedef const unsigned char __attribute__((address_space(4)))* cbyte_ptr_t;
  auto flagged_col = [&](int t) {
    int c = cols[t];
    if constexpr (EW) c |= (int)((cbyte_ptr_t)(uintptr_t)prm.tile_partial)[t] << 30;
    return c;
  };
  constexpr int COL_MASK = 0x3fffffff;
  static_assert(MASK_MAX_BLOCKS <= PAIR_COLS_CAP, "all columns from the mask are in LDS");
  const int first_t = listed ? t0 : 0;           // entry t of the list is lcols[t - first_t] once it is staged
  auto col_of = [&](int t) { return t - first_t < PAIR_COLS_CAP ? lcols[t - first_t] : flagged_col(t); };

  // asynchronous tile copies: copy instruction j covers tile rows [4j, 4j+4); this wavefront issues
  // the instructions [HALF w, HALF (w+1)) of every tile (and 256 of the 512 bytes of mask words)
  // (the swizzles repeat every 16 rows for K and every 4 rows for V: KPER / VPER instructions)
  constexpr int RPI = 64 / CPR, KPER = 16 / RPI, VPER = RPI >= 4 ? 1 : 4 / RPI;
  unsigned koff[KPER], voff[VPER];
  {
    const int row0 = lane / CPR, ch = lane % CPR;
#pragma unroll
    for (int par = 0; par < KPER; ++par)
      koff[par] = 2u * (unsigned)(row0 * (int)prm.ks[2] + ((ch ^ k_swz<D>(par * RPI + row0)) * 8));
#pragma unroll
    for (int par = 0; par < VPER; ++par)
      voff[par] = 2u * (unsigned)(row0 * (int)prm.vs[2] + ((ch ^ v_swz<D>(par * RPI + row0)) * 8));
  }
  const int64_t k_rs = prm.ks[2], v_rs = prm.vs[2];   // row strides
  // (the lane index as a value the compiler cannot trace back, or the offsets are computed before the loop and held)
  auto tail_copy = [&](const unsigned short* tile, int64_t rs, unsigned lds_addr, auto&& swz) {
    int lane_t = lane;
    asm volatile("" : "+v"(lane_t));
#pragma unroll 1
    for (int j = w * HALF; j < (w + 1) * HALF; ++j) {
      const int row = j * RPI + lane_t / CPR, src = row < valid ? row : valid - 1;
      tile_load_async_one(tile, 2u * (unsigned)(src * (int)rs + (((lane_t % CPR) ^ swz(row)) * 8)), lds_addr + j * 1024);
    }
  };
  auto k_copy = [&](int cb, int t) {
    const unsigned short* tile = kg + (int64_t)cb * 64 * k_rs;
    if (TAIL && cb == tail_cb) {
      tail_copy(tile, k_rs, lds_k_addr, [](int row) { return k_swz<D>(row); });
    } else {
#pragma unroll
      for (int jj = 0; jj < HALF; ++jj) {
        const int j = w * HALF + jj;
        tile_load_async_one(tile + (int64_t)j * RPI * k_rs, koff[jj % KPER], lds_k_addr + j * 1024);
      }
    }
    if constexpr (EW) {
      const unsigned long long* src = prm.tile_bits + (int64_t)t * 64;
      words_load_async(src, 4u * (unsigned)lane + 256u * w, lds_bits_addr + w * 256);
    }
  };
  auto v_copy = [&](int cb) {
    const unsigned short* tile = vg + (int64_t)cb * 64 * v_rs;
    if (TAIL && cb == tail_cb) {
      tail_copy(tile, v_rs, lds_v_addr, [](int row) { return v_swz<D>(row); });
    } else {
#pragma unroll
      for (int jj = 0; jj < HALF; ++jj) {
        const int j = w * HALF + jj;
        tile_load_async_one(tile + (int64_t)j * RPI * v_rs, voff[jj % VPER], lds_v_addr + j * 1024);
      }
    }
  };
  static_assert(HALF % KPER == 0 && HALF % VPER == 0, "the swizzle patterns of a wavefront's instructions start at phase 0");

  // fragment addresses (as in attn_fwd.hip)
  int kaddr[2][KS];
#pragma unroll
  for (int kb = 0; kb < 2; ++kb)
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const int row = 32 * kb + ln;
      kaddr[kb][s] = row * ROWB + (((2 * s + g) ^ k_swz<D>(row)) * 16);
    }
  const int vblk = lane >> 4, vs_ = lane & 15;
  const int vkey0 = 4 * (vblk >> 1) + (vs_ >> 2), vcol0 = 16 * (vblk & 1) + 4 * (vs_ & 3);
  const uintx4 ones_frag = {g == 0 ? 0x3c003c00u : 0u, 0u, 0u, 0u};

  // first tile's copies (its column from one scalar load), then the column list into LDS
  int cx = listed ? flagged_col(t0) : __builtin_amdgcn_readfirstlane(lcols[t0]);
  k_copy(cx & COL_MASK, t0);
  v_copy(cx & COL_MASK);
  if (listed) {
    for (int i = threadIdx.x; i < t1 - t0 && i < PAIR_COLS_CAP; i += 128) {
      int c = prm.col_idx[t0 + i];
      if constexpr (EW) c |= (int)prm.tile_partial[t0 + i] << 30;
      lcols[i] = c;
    }
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);               // vmcnt(0), visible to the compiler: Q and the first tiles
  if constexpr (FOLD) {
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const uintx4 raw = qf[0][s];
      const uintx4 scaled = {scale_half2(raw[0], qk_scale), scale_half2(raw[1], qk_scale),
                             scale_half2(raw[2], qk_scale), scale_half2(raw[3], qk_scale)};
      qf[0][s] = scaled;
    }
  }
  floatx16 oacc[DB][2];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int i = 0; i < 16; ++i) { oacc[db][0][i] = 0.f; oacc[db][1][i] = 0.f; }
  // (while a query has no mass every tile is recentred (sum_limit); one that does not exist never would have any)
  float m_i = 0.f, l_i = EW && TAIL && !exists ? 1e-30f : 0.f;
  uintx4 mfrag = {0u, 0u, 0u, 0u};
  bool fresh = true;
  float limit = FOLD ? SUM_LIMIT : 0.f;
  int any_m = 0;     // (wave-uniform) some lane's reference exponent is not zero: the extra contraction slice is needed
  __syncthreads();                                  // both halves of K(t0) and V(t0) and the column list are in LDS

  for (int t = t0; t < t1; ++t) {
    const bool has1 = t + 1 < t1;
    const int cxn = has1 ? __builtin_amdgcn_readfirstlane(col_of(t + 1)) : 0;
    const bool partial = EW ? (cx >> 30) != 0 : TAIL && cx == tail_cb;
    // ---- S^T = K Q^T (- m when FOLD); the K fragments (and the mask word of this lane's query) ----
    floatx16 s0, s1;
#pragma unroll
    for (int i = 0; i < 16; ++i) { s0[i] = 0.f; s1[i] = 0.f; }
    unsigned long long mw = 0ull;
    {
      uintx4 kfr[2][KS];
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int s = 0; s < KS; ++s) kfr[kb][s] = *reinterpret_cast<const uintx4*>(lds_k + kaddr[kb][s]);
      {
        if constexpr (EW) { if (partial) mw = lds_bits[32 * w + ln] >> (4 * g); }
        else if constexpr (TAIL) {
          if (partial) { mw = ((1ull << valid) - 1ull) >> (4 * g); asm volatile("" : "+v"(mw)); }
        }
        wait_vm<0>();                               // this wavefront's half of V(t) has landed
        lds_wait();
        __syncthreads();                            // ... and the other half; both hold their K fragments: the K buffer is free
        if (has1) k_copy(cxn & COL_MASK, t + 1);
      }
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        s0 = mfma_qk<BF16>(kfr[0][s], qf[0][s], s0);
        s1 = mfma_qk<BF16>(kfr[1][s], qf[0][s], s1);
      }
    }
    if constexpr (FOLD) {
      if (any_m) {
        s0 = mfma_qk<BF16>(ones_frag, mfrag, s0);
        s1 = mfma_qk<BF16>(ones_frag, mfrag, s1);
      }
    }
    if constexpr (EW || TAIL) {
      if (partial) {
        const unsigned lo = (unsigned)mw, hi = (unsigned)(mw >> 32);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const unsigned bit = 1u << (8 * (i / 4) + (i % 4));
          s0[i] = (lo & bit) ? s0[i] : -INFINITY;
          s1[i] = (hi & bit) ? s1[i] : -INFINITY;
        }
      }
    }
    uintx4 pf[4][2];
    // ---- V^T fragments ----
    auto read_v = [&](uintx4 (&vfr)[4][DB]) {
#pragma unroll
      for (int ts = 0; ts < 4; ++ts)
#pragma unroll
        for (int db = 0; db < DB; ++db) {
          uintx4 a;
#pragma unroll
          for (int jh = 0; jh < 2; ++jh) {
            const int key = 16 * ts + 8 * jh + vkey0, col = 32 * db + vcol0;
            const int addr = key * ROWB + (((col >> 3) ^ v_swz<D>(key)) * 16) + (col & 7) * 2;
            const short4v rr = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (short4v __attribute__((address_space(3)))*)(lds_v + addr));
            const uintx2 r2 = __builtin_bit_cast(uintx2, rr);
            a[2 * jh] = r2[0]; a[2 * jh + 1] = r2[1];
          }
          if constexpr (BF16 && !PB) a = bf16x8_to_f16x8(a);
          vfr[ts][db] = a;
        }
    };
    auto v_free = [&]() {
      wait_vm<0>();                               // this wavefront's half of K(t+1) has landed
      lds_wait();
      __syncthreads();                            // ... and the other half; both hold their V fragments: the V buffer is free
      if (has1) v_copy(cxn & COL_MASK);
    };
    auto second = [&](uintx4 (&vfr)[4][DB]) {
#pragma unroll
      for (int ts = 0; ts < 4; ++ts)
#pragma unroll
        for (int db = 0; db < DB; ++db)
          oacc[db][0] = mfma_qk<PB>(vfr[ts][db], pf[ts][0], oacc[db][0]);
    };
    auto numerators = [&]() {
      float lnew = softmax_tile<FOLD, PB>(s0, s1, qk_scale, m_i, l_i, pf, 0);
      // (FOLD: the first tile of a row block keeps the reference at 0 when its sums are of moderate size; not with elementwise masks, whose
      // short rows the largest numerators being exact serves most: fp16, 16 heads N = 4000 token-causal 2.54e-4 against 64 bits, so 2.49e-4)
      const bool first = FOLD && fresh && (EW || !(lnew >= 0.25f));
      if (__any(first || !(lnew - l_i < limit))) {
        recentre<DB, FOLD, false>(s0, s1, oacc, 0, qk_scale, m_i, l_i, mfrag, fresh, g);
        any_m = 1;
        lnew = softmax_tile<FOLD, PB>(s0, s1, qk_scale, m_i, l_i, pf, 0);
        limit = sum_limit<false>(lnew);
      }
      l_i = lnew;
      fresh = false;
    };
    {
      // The V fragments are read before the softmax (they take the registers of the K fragments), so
      // that the next V tile is requested that much earlier: its latency was exposed otherwise.
      uintx4 vfr[4][DB];
      read_v(vfr);
      v_free();
      numerators();
      second(vfr);
    }
    cx = cxn;
  }

  // ---- normalise and write ----
  const float lsum = l_i + __shfl_xor(l_i, 32);
  if (!EW && prm.split > 1) {   // unnormalised fp32 part with its reference exponent and row sum
    if (!exists) return;
    float* part = prm.part_o + ((int64_t)chunk * BH + bh) * prm.N * D;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int i4 = 0; i4 < 4; ++i4)
        store_out4<BF16>(part, qrow * D + 32 * db + 8 * i4 + 4 * g, true, oacc[db][0][4 * i4], oacc[db][0][4 * i4 + 1],
                         oacc[db][0][4 * i4 + 2], oacc[db][0][4 * i4 + 3]);
    if (g == 0) {
      float* ml = prm.part_ml + (((int64_t)chunk * BH + bh) * prm.N + qrow) * 2;
      ml[0] = m_i; ml[1] = lsum;
    }
    return;
  }
  const float inv = row_inverse<EW>(lsum);
  // the wavefront's 32 rows of O leave through its half of the (now idle) LDS
  static_assert(2 * rows_out_bytes(D, true) <= PAIR_LDS_BYTES, "room for the result rows of both wavefronts");
  __syncthreads();           // the other wavefront has left its last tile
  rows_out<BF16, D>(lds + w * rows_out_bytes(D, true), obase, ((int64_t)m * 64 + 32 * w) * prm.os[2], prm.os[2], prm.out_f32,
                    lane, TAIL ? prm.N - (m * 64 + 32 * w) : 32, [&](int db, int i) { return oacc[db][0][i] * inv; });
  if (prm.lse != nullptr && g == 0 && exists) prm.lse[(int64_t)bh * prm.N + qrow] = row_lse(m_i, lsum);
}

// split > 1: O = sum_c 2^(m_c - M) O_c / sum_c 2^(m_c - M) l_c over the non-empty shares c of a row block
// (M = max m_c over shares with mass), lse = (M + log2 of the denominator) ln 2.  A share without mass is one whose
// sum is zero: a sum that is not a number (a score that is not finite) goes into the result like any other.  One thread
// per 4 consecutive output values.  Bound by latency: the (m, l) and the values of all S shares are asked for together, an empty share
// (nothing was written) reads the last one's, which is never empty, in its place.  Before, one share's loads
// waited for another's and rows were found by 64-bit divisions: 2 heads of N = 4096, D = 256, 8 shares 21.8 -> 14.9 us (71 MB:
// 4.8 TB/s); 8 heads of N = 4000, D = 128, 2 shares, the whole training step 136.9 -> 132.3.
template <bool BF16, int S>
__global__ __launch_bounds__(256) void pair_sum_parts_kernel(const FwdParams prm, unsigned quads) {
  constexpr int D = PAIR_D, QSHIFT = 5;                      // log2 of the threads per query row
  static_assert(D == 4 << QSHIFT, "four values per thread");
  const unsigned i = blockIdx.x * 256 + threadIdx.x;
  if (i >= quads) return;
  const unsigned rowg = i >> QSHIFT;                         // row over all heads
  const int col = (int)(i & ((1u << QSHIFT) - 1)) * 4;
  const int bh = (int)(rowg / (unsigned)prm.N), row = (int)(rowg - (unsigned)bh * prm.N);
  const int b = bh / prm.H, h = bh % prm.H, BH = prm.B * prm.H;
  const int len = prm.part_len[bh * prm.nb + row / 64];
  floatx4 acc = {0.f, 0.f, 0.f, 0.f};
  float M = -INFINITY, L = 0.f;
  if (len > 0) {
    float m[S], l[S];
    floatx4 part[S];
#pragma unroll
    for (int c = 0; c < S; ++c) {
      const bool on = (int64_t)len * c / S != (int64_t)len * (c + 1) / S;
      const int64_t at = ((int64_t)(on ? c : S - 1) * BH + bh) * prm.N + row;
      m[c] = prm.part_ml[at * 2];
      l[c] = prm.part_ml[at * 2 + 1];
      part[c] = *reinterpret_cast<const floatx4*>(prm.part_o + at * D + col);
      if (!on) l[c] = 0.f;
    }
#pragma unroll
    for (int c = 0; c < S; ++c)
      if (l[c] != 0.f) M = fmaxf(M, m[c]);
#pragma unroll
    for (int c = 0; c < S; ++c) {
      if (l[c] == 0.f) continue;
      const float wgt = __builtin_amdgcn_exp2f(m[c] - M);
      L += wgt * l[c];
      acc += wgt * part[c];
    }
  }
  const float inv = len > 0 && prm.tile_bits == nullptr ? row_inverse<false>(L) : row_inverse<true>(L);
  store_out4<BF16>(out_base(prm, b, h), (int64_t)row * prm.os[2] + col, prm.out_f32, acc[0] * inv, acc[1] * inv, acc[2] * inv,
                   acc[3] * inv);
  if (col == 0 && prm.lse != nullptr) prm.lse[(int64_t)bh * prm.N + row] = row_lse(M, L);
}

// (one thread per 4 results of a launch that shares lists, which has fewer than 2 row blocks per compute unit: 64 D / 4 threads each,
// 2 048 at most, so the values fit 32 bits.)
template <bool BF16, int S = 2>
static void launch_sum_parts_t(const FwdParams& prm, hipStream_t st) {
  if constexpr (S < 4) {
    if (prm.split != S) { launch_sum_parts_t<BF16, S + 1>(prm, st); return; }
  }
  const unsigned quads = (unsigned)((int64_t)prm.B * prm.H * prm.N * PAIR_D / 4);
  hipLaunchKernelGGL((pair_sum_parts_kernel<BF16, S>), dim3((quads + 255) / 256), dim3(256), 0, st, prm, quads);
}

template <int DT, bool EW, bool TAIL>
static void launch_pair_c(const FwdParams& prm, int grid, hipStream_t st) {
  static std::atomic<unsigned long long> configured{0};   // raising the dynamic LDS limit is idempotent
  once_per_device(configured, [] {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&fwd_pair_kernel<DT, EW, TAIL>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, PAIR_LDS_BYTES);
  });
  hipLaunchKernelGGL((fwd_pair_kernel<DT, EW, TAIL>), dim3(grid), dim3(128), PAIR_LDS_BYTES, st, prm);
}

template <int DT, bool EW>
static void launch_pair_t(const FwdParams& prm, hipStream_t st) {
  const int grid = prm.place.per_share * prm.split;
  if (prm.N % 64 != 0) launch_pair_c<DT, EW, true>(prm, grid, st);
  else launch_pair_c<DT, EW, false>(prm, grid, st);
  if (!EW && prm.split > 1) launch_sum_parts_t<DT != 0>(prm, st);
}

template <bool EW>
static void launch_pair_e(const FwdParams& prm, int dt, hipStream_t st) {
  if (dt == 0) launch_pair_t<0, EW>(prm, st);
  else if (dt == 1) launch_pair_t<1, EW>(prm, st);
  else launch_pair_t<2, EW>(prm, st);
}

// dt: 0 fp16, 1 bf16 with P rounded to fp16 (V converted), 2 bf16 with P rounded to bf16.
void launch_fwd_pair(const FwdParams& prm, int dt, bool elementwise, hipStream_t st) {
  if (elementwise) launch_pair_e<true>(prm, dt, st);
  else launch_pair_e<false>(prm, dt, st);
}

}  // namespace bsattn
