// Block-sparse FlashAttention-2 forward, head dimension 64, for launches with few row blocks, whose time is the latency of
// a row block's list and not the throughput of the GPU.
//
// A workgroup has one row block (or one of `split` contiguous shares of its list).  It is S pairs of wavefronts; pair c takes
// tiles c, c + S, ... of the list, wavefront w of a pair 32 of the 64 queries, and the pairs' results are merged through
// LDS at the end.  A pair has two stages of a K and a V tile: the next step's tiles are asked for before the current ones
// are worked on, and one barrier per step (of the whole workgroup: all pairs make the same number of steps, a pair that has run
// out of tiles only waits) covers both.  The row block is the workgroup's index: nothing has to be searched or divided
// before the first tile can be asked for.  Latency bound: 1 head N = 1024 keep 0.5 (16 row blocks of 8 tiles) 12.1 -> 8.8 us
// a call (fwd_kernel's ranges before), of which the host is 8.5; 8 heads N = 2048 keep 0.3 15.9 -> 11.2, N = 4096 dense 51.7 ->
// 46.7 (2 pairs); 3 heads N = 2000, token window of 600, 16.7 -> 10.4.  (Single stages and four barriers per tile, as
// in attn_fwd_pair.hip, with as many pairs in workgroups of their own and a launch that sums their parts: 10-11 us at least.)
//
// Tile arithmetic, softmax and layouts are those of attn_fwd.hip (fa2_custom_mask/fa2_fwd.py:146-196 of the reference), with a
// single block of 32 queries per wavefront.
#include "common.h"
#include "fwd_tile.h"
#include "kernel_util.h"

namespace bsattn {

constexpr int SHARING_PAIRS = 4, SHARING_MOST = 4;      // pairs of the workgroups that share lists; shares of a list, at most

// Two quads of each of four parts, 8 KB apart, and the wait for them in one statement (kernel_util.h, coherent_load4x4).
__device__ __forceinline__ void coherent_load_pairs(const float* a, const float* b, const float* c, const float* d, floatx4 (&x)[4][2]) {
  asm volatile("global_load_dwordx4 %0, %8, off sc1\n\tglobal_load_dwordx4 %1, %9, off sc1\n\t"
               "global_load_dwordx4 %2, %10, off sc1\n\tglobal_load_dwordx4 %3, %11, off sc1\n\t"
               "global_load_dwordx4 %4, %12, off sc1\n\tglobal_load_dwordx4 %5, %13, off sc1\n\t"
               "global_load_dwordx4 %6, %14, off sc1\n\tglobal_load_dwordx4 %7, %15, off sc1\n\t"
               "s_waitcnt vmcnt(0)"
               : "=&v"(x[0][0]), "=&v"(x[0][1]), "=&v"(x[1][0]), "=&v"(x[1][1]), "=&v"(x[2][0]), "=&v"(x[2][1]), "=&v"(x[3][0]), "=&v"(x[3][1])
               : "v"(a), "v"(a + 2048), "v"(b), "v"(b + 2048), "v"(c), "v"(c + 2048), "v"(d), "v"(d + 2048) : "memory");
}

// S: pairs of wavefronts per workgroup.  Lists of at most SHORT_MAX_BLOCKS tiles.
template <int S, bool EW> struct ShortCfg {
  static constexpr int TILE_BYTES = 64 * 128;
  static constexpr int STAGE_BYTES = 2 * TILE_BYTES + (EW ? 512 : 0);          // K tile, V tile, mask words
  static constexpr int PAIR_BYTES = 2 * STAGE_BYTES;
  static constexpr int COLS_OFF = S * PAIR_BYTES;
  static constexpr int COLS_CAP = SHORT_MAX_BLOCKS;                             // column indices of the list
  static constexpr int ML_OFF = COLS_OFF + COLS_CAP * 4;                        // (m, l) per pair and query
  static constexpr int LDS_BYTES = ML_OFF + S * 64 * 2 * 4;
  static constexpr int PITCH = 64 + 4;                                          // floats per row of a pair's result in LDS
  static_assert(64 * PITCH * 4 <= PAIR_BYTES, "a pair's result fits its stages");
};

// DT: 0 fp16; 1 bf16 with P rounded to fp16 (V fragments converted); 2 bf16 with P rounded to bf16.
// TAIL: N is not a multiple of 64 (as in attn_fwd.hip: the copy of the last tile repeats its last key, the scores beyond
// it are -inf, the queries beyond N are not written).
// SHARED: lists are shared by workgroups (a variant of its own: the code, even where it is jumped over, costs a launch of one short head 0.3 us).
template <int S, int DT, bool EW, bool TAIL, bool SHARED>
__global__ __launch_bounds__(128 * S, 2) void fwd_short_kernel(const FwdParams prm) {
  using C = ShortCfg<S, EW>;
  constexpr int D = 64, KS = D / 16, DB = D / 32, CPR = D / 8, ROWB = 2 * D, HALF = CPR / 2, RPI = 64 / CPR;
  constexpr bool BF16 = DT != 0, PB = DT == 2, FOLD = !BF16;
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), c = wave >> 1, w = wave & 1;
  const int ln = lane & 31, g = lane >> 5;
  const int nb = prm.nb;
  int chunk;
  const Place p = prm.place.of(blockIdx.x, chunk);
  const int bh = p.head, m = nb - 1 - p.item;
  if (m < 0) return;                              // padding of an incomplete last group
  const int b = (int)prm.per_batch.of((unsigned)bh), h = bh - b * prm.H;
  const int mh = (prm.Bm > 1 ? b : 0) * prm.Hm + (prm.Hm > 1 ? h : 0);
  const cint_ptr_t rp = (cint_ptr_t)(uintptr_t)(prm.row_ptr + (int64_t)mh * nb);
  // Q of this lane's query depends on the block index only: asked for first, it travels while the list is looked up
  const int64_t qrow = (int64_t)m * 64 + 32 * w + ln;
  uintx4 qf[1][KS];
  {
    const unsigned short* qp = (const unsigned short*)prm.q + b * prm.qs[0] + h * prm.qs[1] + (!TAIL || qrow < prm.N ? qrow : prm.N - 1) * prm.qs[2];
#pragma unroll
    for (int s = 0; s < KS; ++s) qf[0][s] = *reinterpret_cast<const uintx4*>(qp + 16 * s + 8 * g);
  }
  int* lcols = reinterpret_cast<int*>(lds + C::COLS_OFF);
  const bool listed = EW || prm.mask == nullptr;
  int t0, t1;
  if (listed) { t0 = rp[m]; t1 = rp[m + 1]; }
  else { t0 = 0; t1 = columns_of_row<SHORT_MAX_BLOCKS>(prm, b, h, m, lane, lcols, chunk == 0 && wave == 0); }
  int shares = 1;
  if constexpr (SHARED) {                         // this workgroup's share of the row block's list
    const int len = t1 - t0;
    shares = short_shares(len, prm.split, prm.share_shift);
    if (chunk >= shares) return;
    t1 = t0 + short_share_begins(len, chunk + 1, shares);
    t0 = t0 + short_share_begins(len, chunk, shares);
  }
  const int valid = TAIL ? prm.N - (nb - 1) * 64 : 64, tail_cb = TAIL ? nb - 1 : -1;
  const unsigned short* kg = (const unsigned short*)prm.k + b * prm.ks[0] + h * prm.ks[1];
  const unsigned short* vg = (const unsigned short*)prm.v + b * prm.vs[0] + h * prm.vs[1];
  const float qk_scale = prm.qk_scale;
  const cint_ptr_t cols = (cint_ptr_t)(uintptr_t)prm.col_idx;
  constexpr int COL_MASK = 0x3fffffff;            // (EW: bit 30 of a staged column says "partly set")
  const int first_t = listed ? t0 : 0;            // entry t of the list is lcols[t - first_t] once it is staged
  unsigned char* mine = lds + c * C::PAIR_BYTES;
  const unsigned mine_addr = (unsigned)(uintptr_t)(lds_ptr_t)lds + c * C::PAIR_BYTES;

  // asynchronous tile copies: instruction j covers tile rows [8j, 8j + 8); this wavefront issues [4w, 4w + 4) of K and of V
  unsigned koff[2], voff;
  {
    const int row0 = lane / CPR, ch = lane % CPR;
#pragma unroll
    for (int par = 0; par < 2; ++par) koff[par] = 2u * (unsigned)(row0 * (int)prm.ks[2] + ((ch ^ k_swz<D>(par * RPI + row0)) * 8));
    voff = 2u * (unsigned)(row0 * (int)prm.vs[2] + ((ch ^ v_swz<D>(row0)) * 8));
  }
  auto tail_copy = [&](const unsigned short* tile, int64_t rs, unsigned lds_addr, auto&& swz) {
    int lane_t = lane;
    asm volatile("" : "+v"(lane_t));
#pragma unroll 1
    for (int j = w * HALF; j < (w + 1) * HALF; ++j) {
      const int row = j * RPI + lane_t / CPR, src = row < valid ? row : valid - 1;
      tile_load_async_one(tile, 2u * (unsigned)(src * (int)rs + (((lane_t % CPR) ^ swz(row)) * 8)), lds_addr + j * 1024);
    }
  };
  auto issue = [&](int cb, int t, int stage) {
    const unsigned short* kt = kg + (int64_t)cb * 64 * prm.ks[2];
    const unsigned short* vt = vg + (int64_t)cb * 64 * prm.vs[2];
    const unsigned ka = mine_addr + stage * C::STAGE_BYTES, va = ka + C::TILE_BYTES;
    if (TAIL && cb == tail_cb) {
      tail_copy(kt, prm.ks[2], ka, [](int row) { return k_swz<D>(row); });
      tail_copy(vt, prm.vs[2], va, [](int row) { return v_swz<D>(row); });
    } else {
#pragma unroll
      for (int jj = 0; jj < HALF; ++jj) tile_load_async_one(kt + (int64_t)(w * HALF + jj) * RPI * prm.ks[2], koff[jj & 1], ka + (w * HALF + jj) * 1024);
#pragma unroll
      for (int jj = 0; jj < HALF; ++jj) tile_load_async_one(vt + (int64_t)(w * HALF + jj) * RPI * prm.vs[2], voff, va + (w * HALF + jj) * 1024);
    }
    if constexpr (EW) {
      const unsigned long long* src = prm.tile_bits + (int64_t)t * 64;
      words_load_async(src, 4u * (unsigned)lane + 256u * w, va + C::TILE_BYTES + w * 256);
    }
  };
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

  // the first step's copies (their column from one scalar load), then the column list into LDS
  int t = t0 + c, cx = 0;
  if (t < t1) {
    cx = listed ? cols[t] : __builtin_amdgcn_readfirstlane(lcols[t]);
    issue(cx, t, 0);
  }
  if (listed) {
    for (int i = threadIdx.x; i < t1 - t0 && i < C::COLS_CAP; i += 128 * S) {
      int x = prm.col_idx[t0 + i];
      if constexpr (EW) x |= (int)prm.tile_partial[t0 + i] << 30;
      lcols[i] = x;
    }
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);             // vmcnt(0), visible to the compiler: Q and the first tiles
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
  // (EW: a query that has no mass yet is recentred in every tile; one that does not exist never will have any)
  float m_i = 0.f, l_i = EW && TAIL && qrow >= prm.N ? 1e-30f : 0.f;
  uintx4 mfrag = {0u, 0u, 0u, 0u};
  bool fresh = true;
  float limit = FOLD || EW ? SUM_LIMIT : 0.f;
  int any_m = 0;     // (wave-uniform) some lane's reference exponent is not zero: the extra contraction slice is needed

  const int steps = (t1 - t0 + S - 1) / S;
  for (int it = 0; it < steps; ++it) {
    wait_vm<0>();
    __syncthreads();                              // the step's tiles are complete; everybody has left the step before
    if constexpr (EW) { if (it == 0 && t < t1) cx = __builtin_amdgcn_readfirstlane(lcols[c]); }     // (with its flag)
    const int tn = t + S;
    int cxn = 0;
    if (tn < t1) {
      cxn = __builtin_amdgcn_readfirstlane(lcols[tn - first_t]);
      issue(cxn & COL_MASK, tn, (it + 1) & 1);
    }
    if (t < t1) {
      const unsigned char* lds_k = mine + (it & 1) * C::STAGE_BYTES;
      const unsigned char* lds_v = lds_k + C::TILE_BYTES;
      const bool partial = EW ? (cx >> 30) != 0 : TAIL && cx == tail_cb;
      // ---- S^T = K Q^T (- m when FOLD) ----
      uintx4 kfr[2][KS];
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int s = 0; s < KS; ++s) kfr[kb][s] = *reinterpret_cast<const uintx4*>(lds_k + kaddr[kb][s]);
      __builtin_amdgcn_sched_barrier(0);
      floatx16 s0, s1;
#pragma unroll
      for (int i = 0; i < 16; ++i) { s0[i] = 0.f; s1[i] = 0.f; }
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        s0 = mfma_qk<BF16>(kfr[0][s], qf[0][s], s0);
        s1 = mfma_qk<BF16>(kfr[1][s], qf[0][s], s1);
      }
      // V^T fragments: on their way while the scores are made
      uintx4 vfr[4][DB];
#pragma unroll
      for (int ts = 0; ts < 4; ++ts)
#pragma unroll
        for (int db = 0; db < DB; ++db) {
          uintx4 a;
#pragma unroll
          for (int jh = 0; jh < 2; ++jh) {
            const int key = 16 * ts + 8 * jh + vkey0, col = 32 * db + vcol0;
            const int addr = key * ROWB + (((col >> 3) ^ v_swz<D>(key)) * 16) + (col & 7) * 2;
            const short4v rr = __builtin_amdgcn_ds_read_tr16_b64_v4i16((short4v __attribute__((address_space(3)))*)(lds_v + addr));
            const uintx2 r2 = __builtin_bit_cast(uintx2, rr);
            a[2 * jh] = r2[0]; a[2 * jh + 1] = r2[1];
          }
          if constexpr (BF16 && !PB) a = bf16x8_to_f16x8(a);
          vfr[ts][db] = a;
        }
      if constexpr (FOLD) {
        if (any_m) {
          s0 = mfma_qk<BF16>(ones_frag, mfrag, s0);
          s1 = mfma_qk<BF16>(ones_frag, mfrag, s1);
        }
      }
      if constexpr (EW || TAIL) {
        if (partial) {
          unsigned long long mw;
          if constexpr (EW) mw = reinterpret_cast<const unsigned long long*>(lds_v + C::TILE_BYTES)[32 * w + ln] >> (4 * g);
          else { mw = ((1ull << valid) - 1ull) >> (4 * g); asm volatile("" : "+v"(mw)); }
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
      float lnew = softmax_tile<FOLD, PB>(s0, s1, qk_scale, m_i, l_i, pf, 0);
      // (FOLD: the first tile keeps the reference at 0 when its sums are of moderate size)
      const bool first = FOLD ? fresh && !(lnew >= 0.25f) : EW && fresh;
      if (__any(first || (EW && l_i == 0.f) || !(lnew - l_i < limit))) {
        recentre<DB, FOLD, EW>(s0, s1, oacc, 0, qk_scale, m_i, l_i, mfrag, fresh, g);
        any_m = 1;
        lnew = softmax_tile<FOLD, PB>(s0, s1, qk_scale, m_i, l_i, pf, 0);
        limit = sum_limit<EW>(lnew);
      }
      l_i = lnew;
      fresh = false;
      // ---- O^T += V^T P^T ----
#pragma unroll
      for (int ts = 0; ts < 4; ++ts)
#pragma unroll
        for (int db = 0; db < DB; ++db) oacc[db][0] = mfma_qk<PB>(vfr[ts][db], pf[ts][0], oacc[db][0]);
    }
    t = tn;
    cx = cxn;
  }

  // ---- merge the pairs: every wavefront's 32 rows into its pair's stages, then 4 consecutive columns of a row per thread ----
  const float lsum = l_i + __shfl_xor(l_i, 32);
  float* ml = reinterpret_cast<float*>(lds + C::ML_OFF);
  unsigned long long* arrivals = prm.flags + (int64_t)bh * nb + m;
  unsigned long long seen = 0ull;      // (the read travels beside the merge)
  if (SHARED && shares > 1 && threadIdx.x == 0) seen = __hip_atomic_load(arrivals, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();           // everybody has left the last step
  {
    float* own = reinterpret_cast<float*>(mine) + (32 * w + ln) * C::PITCH + 4 * g;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int i4 = 0; i4 < 4; ++i4) {
        const floatx4 x = {oacc[db][0][4 * i4], oacc[db][0][4 * i4 + 1], oacc[db][0][4 * i4 + 2], oacc[db][0][4 * i4 + 3]};
        *reinterpret_cast<floatx4*>(own + 32 * db + 8 * i4) = x;
      }
    if (g == 0) {      // (a sum that is not a number stays in)
      ml[(c * 64 + 32 * w + ln) * 2] = lsum != 0.f ? m_i : -INFINITY;
      ml[(c * 64 + 32 * w + ln) * 2 + 1] = lsum;
    }
  }
  __syncthreads();
  void* obase = out_base(prm, b, h);
  auto merge = [&](int i, float& M, float& L) {      // quad i: row i / 16, columns 4 (i % 16) .. + 3
    const int r = i >> 4, col = (i & 15) * 4;
    float mp[S], lp[S];
    floatx4 acc = {0.f, 0.f, 0.f, 0.f}, part[S];
    M = -INFINITY;
    L = 0.f;
#pragma unroll
    for (int cc = 0; cc < S; ++cc) {
      mp[cc] = ml[(cc * 64 + r) * 2];
      lp[cc] = ml[(cc * 64 + r) * 2 + 1];
      part[cc] = *reinterpret_cast<const floatx4*>(reinterpret_cast<const float*>(lds + cc * C::PAIR_BYTES) + r * C::PITCH + col);
    }
#pragma unroll
    for (int cc = 0; cc < S; ++cc) M = fmaxf(M, mp[cc]);
#pragma unroll
    for (int cc = 0; cc < S; ++cc) {
      const float wgt = mp[cc] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mp[cc] - M);
      L += wgt * lp[cc];
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[e] += wgt * part[cc][e];
    }
    return acc;
  };
  auto put = [&](int i, const floatx4& acc, float M, float L) {
    const int col = (i & 15) * 4;
    const int64_t q = (int64_t)m * 64 + (i >> 4);
    if (TAIL && q >= prm.N) return;
    const float inv = EW || steps == 0 ? row_inverse<true>(L) : row_inverse<false>(L);     // (no kept tile or no key: O = 0)
    store_out4<BF16>(obase, q * prm.os[2] + col, prm.out_f32, acc[0] * inv, acc[1] * inv, acc[2] * inv, acc[3] * inv);
    if (col == 0 && prm.lse != nullptr) prm.lse[(int64_t)bh * prm.N + q] = row_lse(M, L);
  };
  if constexpr (SHARED) {
    if (shares > 1) {
      // The shares of a list meet in the workspace, as the parts of a row block do in attn_fwd.hip: each is published with device-scope
      // stores and counted in once these are acknowledged, the last one in asks for all of them at once and adds them up in their order.
      // (A launch that summed the parts took 1 to 2 us more: 1 head N = 6400 keep 0.3 18.6 -> 16.7 us, N = 4096 bf16 keep 0.1 12.7 -> 11.1, dense
      // 17.2 -> 16.4, 2 heads N = 4000 causal keep 0.25 14.0 -> 12.1, N = 8192 token window of 2048 17.3 -> 15.0.)
      constexpr int HALF_QUADS = 64 * 16 / 2;
      static_assert(128 * S == HALF_QUADS && SHARING_MOST == 4, "two quads per thread, four shares at most");
      const int i = threadIdx.x, r = i >> 4;
      const int64_t first = ((int64_t)bh * nb + m) * prm.split;
      auto slot = [&](int p) { return prm.part_o + (first + p) * (64 * D) + 4 * i; };
      auto ml_of = [&](int p) { return prm.part_ml + (first + p) * 128 + 2 * r; };
      float M[2], L[2];
      const floatx4 x0 = merge(i, M[0], L[0]), x1 = merge(i + HALF_QUADS, M[1], L[1]);
      coherent_store4(slot(chunk), x0[0], x0[1], x0[2], x0[3]);
      coherent_store4(slot(chunk) + 4 * HALF_QUADS, x1[0], x1[1], x1[2], x1[3]);
      if ((i & 15) == 0) {
#pragma unroll
        for (int j = 0; j < 2; ++j) { coherent_store(ml_of(chunk) + 64 * j, M[j]); coherent_store(ml_of(chunk) + 64 * j + 1, L[j]); }
      }
      wait_vm<0>();
      __syncthreads();                                   // (and all have read the pairs' results)
      if (threadIdx.x == 0) lcols[0] = count_in(arrivals, prm.epoch, seen);
      __syncthreads();
      if (__builtin_amdgcn_readfirstlane(*(volatile int*)lcols) != shares) return;
      float mp[SHARING_MOST][2], lp[SHARING_MOST][2];
      floatx4 part[SHARING_MOST][2];
#pragma unroll
      for (int p = 0; p < SHARING_MOST; ++p)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const float* at = ml_of(p < shares ? p : 0) + 64 * j;
          mp[p][j] = coherent_load(at);
          lp[p][j] = p < shares ? coherent_load(at + 1) : 0.f;
        }
      coherent_load_pairs(slot(0), slot(1), slot(shares > 2 ? 2 : 0), slot(shares > 3 ? 3 : 0), part);
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        float Ms = -INFINITY, Ls = 0.f;
        floatx4 acc = {0.f, 0.f, 0.f, 0.f};
        // (a share without mass is one whose sum is zero: a sum that is not a number goes into the result like any other)
#pragma unroll
        for (int p = 0; p < SHARING_MOST; ++p) Ms = lp[p][j] != 0.f ? fmaxf(Ms, mp[p][j]) : Ms;
#pragma unroll
        for (int p = 0; p < SHARING_MOST; ++p) {
          if (lp[p][j] == 0.f) continue;
          const float wgt = __builtin_amdgcn_exp2f(mp[p][j] - Ms);
          Ls += wgt * lp[p][j];
          acc += wgt * part[p][j];
        }
        put(i + j * HALF_QUADS, acc, Ms, Ls);
      }
      // back to zero, so that a replay of this launch (same mark) starts from a clean counter
      if (threadIdx.x == 0) __hip_atomic_store(arrivals, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      return;
    }
  }
#pragma unroll
  for (int i = threadIdx.x; i < 64 * 16; i += 128 * S) {
    float M, L;
    const floatx4 acc = merge(i, M, L);
    put(i, acc, M, L);
  }
}

template <int S, int DT, bool EW, bool TAIL, bool SHARED = false>
static void launch_short_t(const FwdParams& prm, hipStream_t st) {
  if constexpr (S == SHARING_PAIRS && !SHARED) {
    if (prm.split > 1) { launch_short_t<S, DT, EW, TAIL, true>(prm, st); return; }
  }
  constexpr int LDS = ShortCfg<S, EW>::LDS_BYTES;
  static std::atomic<unsigned long long> configured{0};   // raising the dynamic LDS limit is idempotent
  once_per_device(configured, [] {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&fwd_short_kernel<S, DT, EW, TAIL, SHARED>), hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
  });
  const int grid = prm.place.per_share * prm.split;
  hipLaunchKernelGGL((fwd_short_kernel<S, DT, EW, TAIL, SHARED>), dim3(grid), dim3(128 * S), LDS, st, prm);
}

template <int S, int DT>
static void launch_short_d(const FwdParams& prm, bool elementwise, hipStream_t st) {
  const bool tail = prm.N % 64 != 0;
  if (!elementwise) { if (tail) launch_short_t<S, DT, false, true>(prm, st); else launch_short_t<S, DT, false, false>(prm, st); }
  else { if (tail) launch_short_t<S, DT, true, true>(prm, st); else launch_short_t<S, DT, true, false>(prm, st); }
}

template <int S>
static void launch_short_s(const FwdParams& prm, int dt, bool elementwise, hipStream_t st) {
  if (dt == 0) launch_short_d<S, 0>(prm, elementwise, st);
  else if (dt == 1) launch_short_d<S, 1>(prm, elementwise, st);
  else launch_short_d<S, 2>(prm, elementwise, st);
}

// pairs: 2 or 4 per workgroup.  dt: 0 fp16, 1 bf16 with P rounded to fp16 (V converted), 2 bf16 with P rounded to bf16.
void launch_fwd_short(const FwdParams& prm, int pairs, int dt, bool elementwise, hipStream_t st) {
  if (pairs == 2) launch_short_s<2>(prm, dt, elementwise, st);
  else launch_short_s<4>(prm, dt, elementwise, st);
}

}  // namespace bsattn
