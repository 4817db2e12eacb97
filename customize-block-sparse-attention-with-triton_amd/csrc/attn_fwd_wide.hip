// Block-sparse FlashAttention-2 forward, head dimension 256.
//
// A workgroup of four wavefronts has one row block, or a share of its list (quad_shares.h): wavefront (kh, w) takes keys
// 32 kh .. of every tile for queries 32 w .. .  O of 32 queries is 128 registers and Q 64; with the scores of 32 keys in place of
// 64 the rest fits a quarter of a SIMD's registers, so two wavefronts share a SIMD and one's products run beside the other's
// softmax.  A K and a V tile (64 KB) are shared by the four, two workgroups per compute unit; the next K tile is asked for as soon
// as all hold their K fragments, the next V tile as soon as all hold their V fragments.  Two barriers per tile: in front of the one that
// frees the K buffer every wavefront waits for its part of V, in front of the one that frees V for its part of the next K.  (Four, with
// waits of their own: 10 heads N = 4090 keep 0.3 95 -> 92 us, 2 heads N = 20800 dense 978 -> 947, 16 heads N = 8192 keep 0.3 378 -> 369.)  The two
// key halves keep a reference exponent and a sum each and meet in LDS at the end, half of the columns each way.  Shares of a list
// (quad_shares.h) meet in the workspace, in the same launch; the last one in asks for all 16 KB per wavefront of a part at once (four
// round trips per part: 1 head N = 1024 dense 22.0 -> 20.0 us, N = 1536 24.6 -> 23.2).
//
// Before, fwd_pair_kernel: a wavefront with the scores of all 64 keys, up to 512 registers, alone on its SIMD, so that scores, softmax
// and second product came one after the other.  us: 16 heads N = 4096 block-causal keep 0.5 bf16 108 -> 96, results in fp32
// 131 -> 117, dense block-causal fp16 189 -> 168 (831 TFLOP/s); 16 heads N = 8192 keep 0.3 472 -> 409 (806 TFLOP/s).  Ragged: 16 heads
// N = 4000 causal keep 0.5 bf16 168 -> 95 (fwd_pair_kernel spilled), 10 heads N = 4090 keep 0.3 142 -> 93, fp16 N = 4065 dense
// block-causal 214 -> 170.  Elementwise masks: 16 heads N = 4000 token window of 1000 127 -> 81, token-causal 215 -> 143, fp16 N = 4096 101 -> 86
// and 180 -> 156.  Two variants, fp16 elementwise with strided rows, keep 12 bytes per lane in scratch memory.
//
// Tile arithmetic, softmax and layouts are those of attn_fwd.hip (fa2_custom_mask/fa2_fwd.py:146-196 of the reference).
#include "common.h"
#include "fwd_tile.h"
#include "kernel_util.h"

namespace bsattn {

constexpr int WIDE_D = 256, WIDE_COLS_CAP = 1024;                               // column indices of the row block kept in LDS
constexpr int WIDE_TILE_BYTES = 64 * 2 * WIDE_D;
constexpr int WIDE_COLS_OFF = 2 * WIDE_TILE_BYTES;
constexpr int WIDE_BITS_OFF = WIDE_COLS_OFF + WIDE_COLS_CAP * 4;
constexpr int WIDE_LDS_BYTES = WIDE_BITS_OFF + 512;                             // K tile, V tile, columns, mask words
static_assert(MASK_MAX_BLOCKS <= WIDE_COLS_CAP, "all columns from the mask are in LDS");
static_assert(4 * rows_out_bytes(128, true) <= WIDE_LDS_BYTES, "room for the result rows of all wavefronts");

// DT: 0 fp16; 1 bf16 with P rounded to fp16 (V fragments converted); 2 bf16 with P rounded to bf16.
// CONTIG: the rows of K and of V follow each other without gaps (row stride = 256).
// TAIL: N is not a multiple of 64: the copy of the last tile repeats its last key, the scores beyond it are -inf (a half without
// any key leaves the tile out), the queries beyond N are not written.
// PARTS: some first tiles keep their numerators in two parts (attn_fwd_quad.hip).
// EW: elementwise masks (bit 30 of a staged column says "partly set", the tile's 64 row words travel with K).
template <int DT, bool CONTIG, bool TAIL, bool EW, bool PARTS>
__global__ __launch_bounds__(256, 2) void fwd_wide_kernel(const FwdShareParams prm) {
  constexpr int D = WIDE_D, KS = D / 16, DB = D / 32, CPR = D / 8, ROWB = 2 * D, RPI = 64 / CPR;
  constexpr int COPIES = CPR / 4;                // copy instructions per wavefront and tile
  constexpr bool BF16 = DT != 0, PB = DT == 2, FOLD = !BF16;
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), kh = wave >> 1, w = wave & 1;
  const int ln = lane & 31, g = lane >> 5;
  const int nb = prm.nb;
  int chunk;
  const Place p = prm.place.of(blockIdx.x, chunk);
  const int bh = p.head, m = nb - 1 - p.item;
  if (m < 0) return;                             // padding of an incomplete last group
  const int b = (int)prm.per_batch.of((unsigned)bh), h = bh - b * prm.H;
  const int mh = (prm.Bm > 1 ? b : 0) * prm.Hm + (prm.Hm > 1 ? h : 0);
  const cint_ptr_t rp = (cint_ptr_t)(uintptr_t)(prm.row_ptr + (int64_t)mh * nb);
  // Q of this lane's query depends on the block index only: asked for first, it travels while the list is looked up
  const int64_t qrow = (int64_t)m * 64 + 32 * w + ln;
  const int valid = TAIL ? prm.N - (nb - 1) * 64 : 64, tail_cb = TAIL ? nb - 1 : -1;
  uintx4 qf[KS];
  {
    const unsigned short* qp = (const unsigned short*)prm.q + b * prm.qs[0] + h * prm.qs[1] + (!TAIL || qrow < prm.N ? qrow : prm.N - 1) * prm.qs[2];
#pragma unroll
    for (int s = 0; s < KS; ++s) qf[s] = *reinterpret_cast<const uintx4*>(qp + 16 * s + 8 * g);
  }
  int* lcols = reinterpret_cast<int*>(lds + WIDE_COLS_OFF);
  const bool listed = EW || prm.mask == nullptr;
  int t0, t1;
  if (listed) { t0 = rp[m]; t1 = rp[m + 1]; }
  else { t0 = 0; t1 = columns_of_row<MASK_MAX_BLOCKS>(prm, b, h, m, lane, lcols, chunk == 0 && wave == 0); }
  int shares = 1;
  if (prm.split > 1) {                           // this workgroup's share of the row block's list
    const int len = t1 - t0;
    shares = shares_of_list(prm, rp, b, h, len, (int)blockIdx.x - chunk * prm.place.per_share, listed, lane);
    if (chunk >= shares) return;
    t1 = t0 + (int)((int64_t)len * (chunk + 1) / shares);
    t0 = t0 + (int)((int64_t)len * chunk / shares);
  }
  void* obase = out_base(prm, b, h);
  if (t0 == t1) {                                // no kept tile: O = 0, lse = -inf
    if (TAIL && qrow >= prm.N) return;
#pragma unroll
    for (int db = 0; db < DB / 2; ++db)
#pragma unroll
      for (int i4 = 0; i4 < 4; ++i4)
        store_out4<BF16>(obase, qrow * prm.os[2] + 128 * kh + 32 * db + 8 * i4 + 4 * g, prm.out_f32, 0.f, 0.f, 0.f, 0.f);
    if (prm.lse != nullptr && wave == w && g == 0) prm.lse[(int64_t)bh * prm.N + qrow] = -INFINITY;
    return;
  }

  unsigned char* lds_v = lds + WIDE_TILE_BYTES;
  const unsigned lds_k_addr = (unsigned)(uintptr_t)(lds_ptr_t)lds;
  const unsigned lds_v_addr = lds_k_addr + WIDE_TILE_BYTES;
  const unsigned short* kg = (const unsigned short*)prm.k + b * prm.ks[0] + h * prm.ks[1];
  const unsigned short* vg = (const unsigned short*)prm.v + b * prm.vs[0] + h * prm.vs[1];
  const float qk_scale = prm.qk_scale;

  const cint_ptr_t cols = (cint_ptr_t)(uintptr_t)prm.col_idx;
  const int first_t = listed ? t0 : 0;           // entry t of the list is lcols[t - first_t] once it is staged
  typedef const unsigned char __attribute__((address_space(4)))* cbyte_ptr_t;
  constexpr int COL_MASK = 0x3fffffff;
  auto flagged_col = [&](int t) {
    int x = cols[t];
    if constexpr (EW) x |= (int)((cbyte_ptr_t)(uintptr_t)prm.tile_partial)[t] << 30;
    return x;
  };
  auto col_of = [&](int t) { return t - first_t < WIDE_COLS_CAP ? lcols[t - first_t] : flagged_col(t); };

  // asynchronous tile copies: instruction j covers tile rows 2j, 2j + 1; this wavefront issues [8 wave, 8 wave + 8) of a tile.
  // The swizzles repeat every 16 rows for K (8 instructions) and every 4 rows for V (2): instruction j reads chunk
  // (lane % 32) ^ (2 j + row0) % 16 of K's row 2j + row0, ... ^ 4 ((2 j + row0) % 4) of V's.
  constexpr int KPER = 16 / RPI, VPER = 4 / RPI;
  static_assert(COPIES % KPER == 0 && COPIES % VPER == 0, "the swizzle patterns of a wavefront's instructions start at phase 0");
  const int row0 = lane / CPR;
  unsigned kx = 16u * (unsigned)((lane % CPR) ^ row0), vx = 16u * (unsigned)((lane % CPR) ^ (4 * row0));
  const unsigned krow = 2u * (unsigned)(row0 * (int)prm.ks[2]), vrow = 2u * (unsigned)(row0 * (int)prm.vs[2]);
  if constexpr (CONTIG) { kx += row0 * ROWB; vx += row0 * ROWB; }
  auto tile_copy = [&](const unsigned short* tile, int64_t rs, unsigned lds_addr, auto&& off) {
    if constexpr (CONTIG) {            // (instruction j reads at byte 1024 j of the tile and writes at byte 1024 j of the buffer)
#pragma unroll
      for (int jb = 0; jb < COPIES; jb += 4)
        tile_load_async_four(tile + (wave * COPIES + jb) * RPI * D, off(jb), off(jb + 1), off(jb + 2), off(jb + 3),
                             lds_addr + (wave * COPIES + jb) * 1024);
    } else {
#pragma unroll
      for (int jj = 0; jj < COPIES; ++jj) {
        const int j = wave * COPIES + jj;
        tile_load_async_one(tile + (int64_t)j * RPI * rs, off(jj), lds_addr + j * 1024);
      }
    }
  };
  // (the lane index as a value the compiler cannot trace back, or the offsets are computed before the loop and held)
  auto tail_copy = [&](const unsigned short* tile, int64_t rs, unsigned lds_addr, auto&& swz) {
    int lane_t = lane;
    asm volatile("" : "+v"(lane_t));
#pragma unroll 1
    for (int j = wave * COPIES; j < (wave + 1) * COPIES; ++j) {
      const int row = j * RPI + lane_t / CPR, src = row < valid ? row : valid - 1;
      tile_load_async_one(tile, 2u * (unsigned)(src * (int)rs + (((lane_t % CPR) ^ swz(row)) * 8)), lds_addr + j * 1024);
    }
  };
  auto k_copy = [&](int cb, int t) {
    if constexpr (EW) {
      if (wave < 2) words_load_async(prm.tile_bits + (int64_t)t * 64, 4u * (unsigned)lane + 256u * wave, lds_k_addr + WIDE_BITS_OFF + wave * 256);
    }
    if (TAIL && cb == tail_cb) {
      tail_copy(kg + (int64_t)cb * 64 * prm.ks[2], prm.ks[2], lds_k_addr, [](int row) { return k_swz<D>(row); });
      return;
    }
    tile_copy(kg + (int64_t)cb * 64 * (CONTIG ? (int64_t)D : prm.ks[2]), prm.ks[2], lds_k_addr,
              [&](int j) { return (kx ^ (32u * (j % KPER))) + (CONTIG ? 0u : krow); });
  };
  auto v_copy = [&](int cb) {
    if (TAIL && cb == tail_cb) {
      tail_copy(vg + (int64_t)cb * 64 * prm.vs[2], prm.vs[2], lds_v_addr, [](int row) { return v_swz<D>(row); });
      return;
    }
    tile_copy(vg + (int64_t)cb * 64 * (CONTIG ? (int64_t)D : prm.vs[2]), prm.vs[2], lds_v_addr,
              [&](int j) { return (vx ^ (128u * (j % VPER))) + (CONTIG ? 0u : vrow); });
  };

  // Fragment addresses.  K: chunk (2s + g) ^ (row & 15) of row 32 kh + ln, i.e. kbase with bits 5-7 turned by s % 8, and 256 s / 8
  // further on.  V: chunk (4 db + ..) ^ 4 (key & 3), i.e. vbase with bits 6-7 turned by db % 4, and 256 (db / 4) further on.
  int kbase = (32 * kh + ln) * ROWB + ((g ^ k_swz<D>(ln)) * 16);
  int vbase;
  {
    const int blk = lane >> 4, vs = lane & 15, key0 = 4 * (blk >> 1) + (vs >> 2), col0 = 16 * (blk & 1) + 4 * (vs & 3);
    vbase = (32 * kh + key0) * ROWB + (((col0 >> 3) ^ v_swz<D>(key0)) * 16) + (col0 & 7) * 2;
  }
  const uintx4 ones_frag = {g == 0 ? 0x3c003c00u : 0u, 0u, 0u, 0u};

  // first tile's copies (its column from one scalar load), then the column list into LDS
  int cx = listed ? flagged_col(t0) : __builtin_amdgcn_readfirstlane(lcols[t0]);
  k_copy(cx & COL_MASK, t0);
  v_copy(cx & COL_MASK);
  if (listed) {
    for (int i = threadIdx.x; i < t1 - t0 && i < WIDE_COLS_CAP; i += 256) {
      int x = prm.col_idx[t0 + i];
      if constexpr (EW) x |= (int)prm.tile_partial[t0 + i] << 30;
      lcols[i] = x;
    }
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);               // vmcnt(0), visible to the compiler: Q and the first tiles
  if constexpr (FOLD) {
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const uintx4 raw = qf[s];
      const uintx4 scaled = {scale_half2(raw[0], qk_scale), scale_half2(raw[1], qk_scale),
                             scale_half2(raw[2], qk_scale), scale_half2(raw[3], qk_scale)};
      qf[s] = scaled;
    }
  }
  floatx16 oacc[DB][1];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int i = 0; i < 16; ++i) oacc[db][0][i] = 0.f;
  // (while a query has no mass every tile is recentred (sum_limit); one that does not exist never would have any)
  float m_i = 0.f, l_i = EW && TAIL && qrow >= prm.N ? 1e-30f : 0.f;
  uintx4 mfrag = {0u, 0u, 0u, 0u};
  bool fresh = true;
  float limit = FOLD ? SUM_LIMIT : 0.f;
  int any_m = 0;     // (wave-uniform) some lane's reference exponent is not zero: the extra contraction slice is needed
  __syncthreads();                                  // all of K(t0), V(t0) and the column list are in LDS

  const int two_parts_to = t0 + first_tiles<FOLD>(prm.exact, shares);
  for (int t = t0; t < t1; ++t) {
    const bool has1 = t + 1 < t1;
    const int cxn = has1 ? __builtin_amdgcn_readfirstlane(col_of(t + 1)) : 0;
    asm volatile("" : "+v"(kbase), "+v"(vbase), "+v"(kx), "+v"(vx));    // (or the turned addresses are computed before the loop and held)
    // ---- S^T = K Q^T (- m when FOLD), K fragments in portions of four ----
    floatx16 sc;
#pragma unroll
    for (int i = 0; i < 16; ++i) sc[i] = 0.f;
    unsigned mw = 0u;
    uintx4 kfr[2][4];
    auto read_k = [&](int pt) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int s = 4 * pt + i;
        kfr[pt & 1][i] = *reinterpret_cast<const uintx4*>(lds + (kbase ^ (32 * (s & 7))) + 256 * (s >> 3));
      }
    };
    read_k(0);
#pragma unroll
    for (int pt = 0; pt < 4; ++pt) {
      if (pt < 3) read_k(pt + 1);
      if (pt == 3) {
        if constexpr (EW) {
          if ((cx >> 30) != 0) mw = reinterpret_cast<const unsigned*>(lds + WIDE_BITS_OFF)[2 * (32 * w + ln) + kh] >> (4 * g);
        }
        wait_vm<0>();                               // this wavefront's part of V(t) has landed
        lds_wait();
        __syncthreads();                            // ... and the others'; all hold their K fragments: the K buffer is free
        if (has1) k_copy(cxn & COL_MASK, t + 1);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) sc = mfma_qk<BF16>(kfr[pt & 1][i], qf[4 * pt + i], sc);
    }
    if constexpr (FOLD) {
      if (any_m) sc = mfma_qk<BF16>(ones_frag, mfrag, sc);
    }
    uintx4 pf[2];
    const int keys = TAIL && !EW && cx == tail_cb ? valid - 32 * kh : 32;      // of this half
    if constexpr (EW) {
      if ((cx >> 30) != 0) {
#pragma unroll
        for (int i = 0; i < 16; ++i) sc[i] = (mw & (1u << (8 * (i / 4) + (i % 4)))) ? sc[i] : -INFINITY;
      }
    }
    if (TAIL && !EW && keys < 32) {
      int first_key = 4 * g;
      asm volatile("" : "+v"(first_key));
#pragma unroll
      for (int i = 0; i < 16; ++i) sc[i] = 8 * (i / 4) + (i % 4) + first_key < keys ? sc[i] : -INFINITY;
    }
    // V^T fragments, in portions of two column blocks
    uintx4 vfr[2][2][2];
    auto read_v = [&](int pt) {
#pragma unroll
      for (int d = 0; d < 2; ++d)
#pragma unroll
        for (int ts = 0; ts < 2; ++ts) {
          const int db = 2 * pt + d;
          uintx4 a;
#pragma unroll
          for (int jh = 0; jh < 2; ++jh) {
            const short4v rr = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (short4v __attribute__((address_space(3)))*)(lds_v + (vbase ^ (64 * (db & 3))) + 256 * (db >> 2) + (16 * ts + 8 * jh) * ROWB));
            const uintx2 r2 = __builtin_bit_cast(uintx2, rr);
            a[2 * jh] = r2[0]; a[2 * jh + 1] = r2[1];
          }
          vfr[pt & 1][d][ts] = a;
        }
    };
    auto second = [&](int pt, const uintx4 (&p)[2]) {
#pragma unroll
      for (int ts = 0; ts < 2; ++ts)
#pragma unroll
        for (int d = 0; d < 2; ++d) {
          uintx4 a = vfr[pt & 1][d][ts];
          if constexpr (BF16 && !PB) a = bf16x8_to_f16x8(a);
          oacc[2 * pt + d][0] = mfma_qk<PB>(a, p[ts], oacc[2 * pt + d][0]);
        }
    };
    if (TAIL && !EW && keys <= 0) {
      pf[0] = pf[1] = uintx4{0u, 0u, 0u, 0u};
    } else {
      float lnew = 0.f;
      // (which tiles call for a new reference: attn_fwd_quad.hip; elementwise masks take the softmax first, or 8 to 20 bytes more spill in five variants)
      const bool parts = PARTS && t < two_parts_to;
      bool far = PARTS && !FOLD && !EW && fresh;
      if (!far) {
        lnew = softmax_block<FOLD, PB>(sc, qk_scale, m_i, l_i, pf);
        far = __any((FOLD && fresh && !(lnew >= 0.25f)) || !(lnew - l_i < limit));
      }
      if (far || parts) {
        if (far) {
          recentre_block<DB, FOLD>(sc, oacc, qk_scale, m_i, l_i, mfrag, fresh, g);
          any_m = 1;
          if (EW || !parts) lnew = softmax_block<FOLD, PB>(sc, qk_scale, m_i, l_i, pf);
          if (EW) limit = sum_limit<false>(lnew);
        }
        if constexpr (PARTS) {
          if (parts) {
            uintx4 rest[2];
            lnew = softmax_block_parts<FOLD, PB>(sc, qk_scale, m_i, l_i, pf, rest);
#pragma unroll
            for (int pt = 0; pt < 4; ++pt) {
              read_v(pt);
              second(pt, rest);
              __builtin_amdgcn_sched_barrier(0);
            }
          }
        }
        if (!EW && far) limit = sum_limit<false>(lnew);
      }
      l_i = lnew;
      fresh = false;
    }
    // ---- O^T += V^T P^T ----
    read_v(0);
#pragma unroll
    for (int pt = 0; pt < 4; ++pt) {
      if (pt < 3) read_v(pt + 1);
      if (pt == 3) {
        wait_vm<0>();                               // this wavefront's part of K(t+1) has landed
        lds_wait();
        __syncthreads();                            // ... and the others'; all hold their V fragments: the V buffer is free
        if (has1) v_copy(cxn & COL_MASK);
      }
      second(pt, pf);
    }
    if constexpr (TAIL || EW) cx = cxn;
  }

  // ---- the key halves meet: each hands over the columns the other finishes ----
  // (after the last tile's barriers nobody reads a tile or a column any more: all of the LDS is free)
  // (the lane index as a value the compiler cannot trace back: addresses would otherwise be made before the walk and held)
  int lane_e = lane;
  asm volatile("" : "+v"(lane_e));
  const int ln_e = lane_e & 31, g_e = lane_e >> 5;
  const float lsum = l_i + __shfl_xor(l_i, 32);
  const float m_own = lsum != 0.f ? m_i : -INFINITY;       // (a sum that is not a number stays in)
  float* ml = reinterpret_cast<float*>(lds + WIDE_COLS_OFF);    // (m, l) per half and query
  if (g_e == 0) { ml[(64 * kh + 32 * w + ln_e) * 2] = m_own; ml[(64 * kh + 32 * w + ln_e) * 2 + 1] = lsum; }
  floatx4* give = reinterpret_cast<floatx4*>(lds) + (2 * (1 - kh) + w) * (DB / 2) * 4 * 64 + lane_e;
  const floatx4* take = reinterpret_cast<const floatx4*>(lds) + (2 * kh + w) * (DB / 2) * 4 * 64 + lane_e;
  floatx16 res[DB / 2];
#pragma unroll
  for (int db = 0; db < DB / 2; ++db) {
#pragma unroll
    for (int i4 = 0; i4 < 4; ++i4) {
      floatx4 x;
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] = kh == 0 ? oacc[DB / 2 + db][0][4 * i4 + e] : oacc[db][0][4 * i4 + e];
      give[(4 * db + i4) * 64] = x;
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) res[db][i] = kh == 0 ? oacc[db][0][i] : oacc[DB / 2 + db][0][i];
  }
  unsigned long long* arrivals = prm.flags + (int64_t)bh * nb + m;
  unsigned long long seen = 0ull;      // (the read travels beside the merge)
  if (shares > 1 && threadIdx.x == 0) seen = __hip_atomic_load(arrivals, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  const int other = (64 * (1 - kh) + 32 * w + ln_e) * 2;
  const float m_oth = ml[other], l_oth = ml[other + 1];
  float M = fmaxf(m_own, m_oth);
  const float wo = m_own == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_own - M);
  const float wt = m_oth == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_oth - M);
  // (both halves round it the same way: a share's sum is the same whether it comes from the workspace or from registers)
  float L = (kh == 0 ? wo : wt) * (kh == 0 ? lsum : l_oth) + (kh == 0 ? wt : wo) * (kh == 0 ? l_oth : lsum);
#pragma unroll
  for (int db = 0; db < DB / 2; ++db)
#pragma unroll
    for (int i4 = 0; i4 < 4; ++i4) {
      const floatx4 x = take[(4 * db + i4) * 64];
#pragma unroll
      for (int e = 0; e < 4; ++e) res[db][4 * i4 + e] = wo * res[db][4 * i4 + e] + wt * x[e];
    }
  if (shares > 1) {
    // the shares of a list meet in the workspace, as the parts of a row block do in attn_fwd.hip: each is published with device-scope
    // stores and counted in once these are acknowledged, the last one in adds all of them up in their order
    const int64_t first_slot = ((int64_t)bh * nb + m) * prm.split;
    auto slot_of = [&](int p) { return prm.part_o + (first_slot + p) * (64 * D) + wave * (64 * 64) + lane_e * 4; };      // [wavefront][quad][lane][4]
    auto ml_of = [&](int p) { return prm.part_ml + (first_slot + p) * 128 + 2 * (32 * w + ln_e); };
#pragma unroll
    for (int db = 0; db < DB / 2; ++db)
#pragma unroll
      for (int i4 = 0; i4 < 4; ++i4)
        coherent_store4(slot_of(chunk) + (4 * db + i4) * 256, res[db][4 * i4], res[db][4 * i4 + 1], res[db][4 * i4 + 2], res[db][4 * i4 + 3]);
    if (kh == 0 && g_e == 0) { coherent_store(ml_of(chunk), M); coherent_store(ml_of(chunk) + 1, L); }
    wait_vm<0>();
    __syncthreads();
    if (threadIdx.x == 0) lcols[0] = count_in(arrivals, prm.epoch, seen);
    __syncthreads();
    if (__builtin_amdgcn_readfirstlane(*(volatile int*)lcols) != shares) return;
    floatx16 acc[DB / 2];
#pragma unroll
    for (int db = 0; db < DB / 2; ++db)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[db][i] = 0.f;
    float Ms = -INFINITY, Ls = 0.f;
    for (int p = 0; p < shares; ++p) {
      floatx4 x[16];
      static_assert(DB / 2 * 4 == 16, "quads of a part per lane");
      float mp = M, lp = L;
      if (p == chunk) {
#pragma unroll
        for (int db = 0; db < DB / 2; ++db)
#pragma unroll
          for (int i4 = 0; i4 < 4; ++i4) x[4 * db + i4] = {res[db][4 * i4], res[db][4 * i4 + 1], res[db][4 * i4 + 2], res[db][4 * i4 + 3]};
      } else {
        mp = coherent_load(ml_of(p));
        lp = coherent_load(ml_of(p) + 1);
        coherent_load4x16(slot_of(p), x);
      }
      const float mn = fmaxf(Ms, mp);              // a side without mass has maximum -inf and weight 0
      const float ws = Ms == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(Ms - mn), wp = mp == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mp - mn);
      Ls = Ls * ws + lp * wp;
      Ms = mn;
#pragma unroll
      for (int db = 0; db < DB / 2; ++db)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[db][i] = acc[db][i] * ws + wp * x[4 * db + i / 4][i % 4];
    }
    // back to zero, so that a replay of this launch (same mark) starts from a clean counter
    if (threadIdx.x == 0) __hip_atomic_store(arrivals, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    M = Ms; L = Ls;
#pragma unroll
    for (int db = 0; db < DB / 2; ++db) res[db] = acc[db];
  }
  const float inv = row_inverse<EW>(L);
  __syncthreads();           // all have taken what was handed over: the LDS is free for the result rows
  rows_out<BF16, D / 2>(lds + wave * rows_out_bytes(D / 2, true), obase, ((int64_t)m * 64 + 32 * w) * prm.os[2] + 128 * kh, prm.os[2],
                        prm.out_f32, lane_e, TAIL ? prm.N - (m * 64 + 32 * w) : 32, [&](int db, int i) { return res[db][i] * inv; });
  if (prm.lse != nullptr && kh == 0 && g_e == 0 && (!TAIL || qrow < prm.N)) prm.lse[(int64_t)bh * prm.N + qrow] = row_lse(M, L);
}

template <int DT, bool CONTIG, bool TAIL, bool EW, bool PARTS>
static void launch_wide_p(const FwdShareParams& prm, hipStream_t st) {
  static std::atomic<unsigned long long> configured{0};   // raising the dynamic LDS limit is idempotent
  once_per_device(configured, [] {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&fwd_wide_kernel<DT, CONTIG, TAIL, EW, PARTS>), hipFuncAttributeMaxDynamicSharedMemorySize,
                              WIDE_LDS_BYTES);
  });
  const int grid = prm.place.per_share * prm.split;
  hipLaunchKernelGGL((fwd_wide_kernel<DT, CONTIG, TAIL, EW, PARTS>), dim3(grid), dim3(256), WIDE_LDS_BYTES, st, prm);
}

template <int DT, bool CONTIG, bool TAIL, bool EW>
static void launch_wide_c(const FwdShareParams& prm, hipStream_t st) {
  if constexpr (DT == 0) launch_wide_p<DT, CONTIG, TAIL, EW, EW>(prm, st);      // (fp16: as in attn_fwd_quad.hip)
  else if (first_tiles<false>(prm.exact, 1) > 0) launch_wide_p<DT, CONTIG, TAIL, EW, true>(prm, st);
  else launch_wide_p<DT, CONTIG, TAIL, EW, false>(prm, st);
}

template <int DT, bool EW>
static void launch_wide_t(const FwdShareParams& prm, hipStream_t st) {
  const bool contig = prm.ks[2] == WIDE_D && prm.vs[2] == WIDE_D;
  if (prm.N % 64 != 0) { if (contig) launch_wide_c<DT, true, true, EW>(prm, st); else launch_wide_c<DT, false, true, EW>(prm, st); }
  else { if (contig) launch_wide_c<DT, true, false, EW>(prm, st); else launch_wide_c<DT, false, false, EW>(prm, st); }
}

// dt: 0 fp16, 1 bf16 with P rounded to fp16 (V converted), 2 bf16 with P rounded to bf16.
template <bool EW>
static void launch_wide_e(const FwdShareParams& prm, int dt, hipStream_t st) {
  if (dt == 0) launch_wide_t<0, EW>(prm, st);
  else if (dt == 1) launch_wide_t<1, EW>(prm, st);
  else launch_wide_t<2, EW>(prm, st);
}

void launch_fwd_wide(const FwdShareParams& prm, int dt, bool elementwise, hipStream_t st) {
  if (elementwise) launch_wide_e<true>(prm, dt, st);
  else launch_wide_e<false>(prm, dt, st);
}

}  // namespace bsattn
