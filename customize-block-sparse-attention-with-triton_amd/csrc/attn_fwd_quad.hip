// Block-sparse FlashAttention-2 forward, head dimension 128, for launches with few row blocks, whose time is the latency of a row block's
// list and not the throughput of the GPU.
//
// A workgroup has one row block, or a share of its list.  It is S groups of four wavefronts; group c takes tiles c, c + S, ... , and
// wavefront (kh, w) of a group keys 32 kh .. of every tile for queries 32 w .. .  A group has two stages of a K and a V tile: the next
// step's tiles are asked for before the current ones are worked on, and one barrier per step (of the whole workgroup: all groups make the
// same number of steps, a group that has run out of tiles only waits) covers both.  Key halves and groups keep a reference exponent and
// a sum each and are merged through LDS at the end.  The row block is the workgroup's index: nothing has to be searched or divided before
// the first tile can be asked for.
//
// How many shares a list has is decided on the device, by its own length and that of others (quad_shares.h): every workgroup of a row
// block comes to the same number, those beyond it leave at once.  The shares meet in the workspace, in the same launch.
//
// Before, fwd_pair_kernel (a pair of wavefronts per share, single stages and four barriers per tile) and a launch that summed fp32 parts
// of all lists.  us: 11 heads N = 1344 dense 30 -> 20, 4 heads N = 4096 keep 0.1 25 -> 16, dense 55 -> 45, 8 heads N = 3072 block-causal 65 -> 45,
// 8 heads N = 4000 token window of 1000 39 -> 27, 2 heads N = 12032 block-causal 147 -> 108 (there not taken: quad_plan).  A step of a
// lone group takes 0.75 us for 0.22 us of MFMAs: scores, softmax and second product of a wavefront come one after the other.  At D = 64 the same kernel with 1, 2 or 4
// groups was no faster than fwd_short_kernel (8 heads N = 2048 dense 17.3 against 15.9).
//
// Tile arithmetic, softmax and layouts are those of attn_fwd.hip (fa2_custom_mask/fa2_fwd.py:146-196 of the reference), with a
// single block of 32 queries and 32 keys per wavefront and step.
#include "common.h"
#include "fwd_tile.h"
#include "kernel_util.h"

namespace bsattn {

// S: groups of four wavefronts per workgroup.
template <int D, int S, bool EW> struct QuadCfg {
  static constexpr int TILE_BYTES = 64 * 2 * D;
  static constexpr int STAGE_BYTES = 2 * TILE_BYTES + (EW ? 512 : 0);          // K tile, V tile, mask words
  static constexpr int PITCH = D + 4;                                           // floats per row of a key half's result in LDS
  static constexpr int PART_BYTES = 64 * PITCH * 4;
  static constexpr int GROUP_BYTES = 2 * (STAGE_BYTES > PART_BYTES ? STAGE_BYTES : PART_BYTES);     // two stages, then two results
  static constexpr int COLS_OFF = S * GROUP_BYTES;
  static constexpr int COLS_CAP = QUAD_MAX_BLOCKS;                              // column indices of the list kept in LDS
  static constexpr int ML_OFF = COLS_OFF + COLS_CAP * 4;                        // (m, l) per key half, group and query
  static constexpr int LDS_BYTES = ML_OFF + 2 * S * 64 * 2 * 4;
  static_assert(MASK_MAX_BLOCKS <= COLS_CAP, "all columns from the mask are in LDS");
};

// DT: 0 fp16; 1 bf16 with P rounded to fp16 (V fragments converted); 2 bf16 with P rounded to bf16.
// TAIL: N is not a multiple of 64 (as in attn_fwd.hip: the copy of the last tile repeats its last key, the scores beyond
// it are -inf, the queries beyond N are not written; a half without any key leaves the tile out).
// PARTS: some first tiles keep their numerators in two parts (first_tiles; launches that have none run without the code for it: 7 heads
// N = 3000 dense 63 -> 59 us, D = 256 10 heads N = 4090 dense 225 -> 220).
template <int D, int S, int DT, bool EW, bool TAIL, bool PARTS>
__global__ __launch_bounds__(256 * S, 2) void fwd_quad_kernel(const FwdShareParams prm) {
  using C = QuadCfg<D, S, EW>;
  constexpr int KS = D / 16, DB = D / 32, CPR = D / 8, ROWB = 2 * D, RPI = 64 / CPR;
  constexpr int COPIES = CPR / 4;                 // copy instructions per wavefront and tile
  constexpr int KPER = 16 / RPI;                  // the K swizzle repeats every 16 rows, the V swizzle every 4
  static_assert(COPIES % KPER == 0 && RPI >= 4, "the swizzle patterns of a wavefront's instructions start at phase 0");
  constexpr bool BF16 = DT != 0, PB = DT == 2, FOLD = !BF16;
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), c = wave >> 2, quarter = wave & 3, kh = quarter >> 1, w = wave & 1;
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
  uintx4 qf[KS];
  {
    const unsigned short* qp = (const unsigned short*)prm.q + b * prm.qs[0] + h * prm.qs[1] + (!TAIL || qrow < prm.N ? qrow : prm.N - 1) * prm.qs[2];
#pragma unroll
    for (int s = 0; s < KS; ++s) qf[s] = *reinterpret_cast<const uintx4*>(qp + 16 * s + 8 * g);
  }
  int* lcols = reinterpret_cast<int*>(lds + C::COLS_OFF);
  const bool listed = EW || prm.mask == nullptr;
  int t0, t1;
  if (listed) { t0 = rp[m]; t1 = rp[m + 1]; }
  else { t0 = 0; t1 = columns_of_row<MASK_MAX_BLOCKS>(prm, b, h, m, lane, lcols, chunk == 0 && wave == 0); }
  int shares = 1;
  if (prm.split > 1) {                            // this workgroup's share of the row block's list
    const int len = t1 - t0;
    shares = shares_of_list(prm, rp, b, h, len, (int)blockIdx.x - chunk * prm.place.per_share, listed, lane);
    if (chunk >= shares) return;
    t1 = t0 + (int)((int64_t)len * (chunk + 1) / shares);
    t0 = t0 + (int)((int64_t)len * chunk / shares);
  }
  const int valid = TAIL ? prm.N - (nb - 1) * 64 : 64, tail_cb = TAIL ? nb - 1 : -1;
  const unsigned short* kg = (const unsigned short*)prm.k + b * prm.ks[0] + h * prm.ks[1];
  const unsigned short* vg = (const unsigned short*)prm.v + b * prm.vs[0] + h * prm.vs[1];
  const float qk_scale = prm.qk_scale;
  const cint_ptr_t cols = (cint_ptr_t)(uintptr_t)prm.col_idx;
  constexpr int COL_MASK = 0x3fffffff;            // (EW: bit 30 of a staged column says "partly set")
  const int first_t = listed ? t0 : 0;            // entry t of the list is lcols[t - first_t] once it is staged
  unsigned char* mine = lds + c * C::GROUP_BYTES;
  const unsigned mine_addr = (unsigned)(uintptr_t)(lds_ptr_t)lds + c * C::GROUP_BYTES;

  // asynchronous tile copies: instruction j covers tile rows [RPI j, RPI (j + 1)); this wavefront issues COPIES of K and of V
  unsigned koff[KPER], voff;
  {
    const int row0 = lane / CPR, ch = lane % CPR;
#pragma unroll
    for (int par = 0; par < KPER; ++par) koff[par] = 2u * (unsigned)(row0 * (int)prm.ks[2] + ((ch ^ k_swz<D>(par * RPI + row0)) * 8));
    voff = 2u * (unsigned)(row0 * (int)prm.vs[2] + ((ch ^ v_swz<D>(row0)) * 8));
  }
  auto tail_copy = [&](const unsigned short* tile, int64_t rs, unsigned lds_addr, auto&& swz) {
    int lane_t = lane;
    asm volatile("" : "+v"(lane_t));
#pragma unroll 1
    for (int j = quarter * COPIES; j < (quarter + 1) * COPIES; ++j) {
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
      for (int jj = 0; jj < COPIES; ++jj)
        tile_load_async_one(kt + (int64_t)(quarter * COPIES + jj) * RPI * prm.ks[2], koff[jj % KPER], ka + (quarter * COPIES + jj) * 1024);
#pragma unroll
      for (int jj = 0; jj < COPIES; ++jj)
        tile_load_async_one(vt + (int64_t)(quarter * COPIES + jj) * RPI * prm.vs[2], voff, va + (quarter * COPIES + jj) * 1024);
    }
    if constexpr (EW) {
      if (quarter < 2) {
        const unsigned long long* src = prm.tile_bits + (int64_t)t * 64;
        words_load_async(src, 4u * (unsigned)lane + 256u * quarter, va + C::TILE_BYTES + quarter * 256);
      }
    }
  };
  // Fragment addresses.  K: chunk 2s + g, swizzled, of row 32 kh + ln.  V: the transpose reads of keys 32 kh + 16 ts + 8 jh + vkey0.
  int kaddr[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) kaddr[s] = (32 * kh + ln) * ROWB + (((2 * s + g) ^ k_swz<D>(ln)) * 16);
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
    for (int i = threadIdx.x; i < t1 - t0; i += 256 * S) {
      int x = prm.col_idx[t0 + i];
      if constexpr (EW) x |= (int)prm.tile_partial[t0 + i] << 30;
      lcols[i] = x;
    }
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);             // vmcnt(0), visible to the compiler: Q and the first tiles
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

  const int steps = (t1 - t0 + S - 1) / S, two_parts = first_tiles<FOLD>(prm.exact, S * shares);
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
    const int keys = TAIL && !EW && cx == tail_cb ? valid - 32 * kh : 32;      // of this half
    if (t < t1 && (!TAIL || EW || keys > 0)) {
      const unsigned char* lds_k = mine + (it & 1) * C::STAGE_BYTES;
      const unsigned char* lds_v = lds_k + C::TILE_BYTES;
      // ---- S^T = K Q^T (- m when FOLD) ----
      uintx4 kfr[KS];
#pragma unroll
      for (int s = 0; s < KS; ++s) kfr[s] = *reinterpret_cast<const uintx4*>(lds_k + kaddr[s]);
      __builtin_amdgcn_sched_barrier(0);
      floatx16 sc;
#pragma unroll
      for (int i = 0; i < 16; ++i) sc[i] = 0.f;
#pragma unroll
      for (int s = 0; s < KS; ++s) sc = mfma_qk<BF16>(kfr[s], qf[s], sc);
      // V^T fragments: on their way while the scores are made
      uintx4 vfr[2][DB];
#pragma unroll
      for (int ts = 0; ts < 2; ++ts)
#pragma unroll
        for (int db = 0; db < DB; ++db) {
          uintx4 a;
#pragma unroll
          for (int jh = 0; jh < 2; ++jh) {
            const int key = 32 * kh + 16 * ts + 8 * jh + vkey0, col = 32 * db + vcol0;
            const int addr = key * ROWB + (((col >> 3) ^ v_swz<D>(vkey0)) * 16) + (col & 7) * 2;
            const short4v rr = __builtin_amdgcn_ds_read_tr16_b64_v4i16((short4v __attribute__((address_space(3)))*)(lds_v + addr));
            const uintx2 r2 = __builtin_bit_cast(uintx2, rr);
            a[2 * jh] = r2[0]; a[2 * jh + 1] = r2[1];
          }
          if constexpr (BF16 && !PB) a = bf16x8_to_f16x8(a);
          vfr[ts][db] = a;
        }
      if constexpr (FOLD) {
        if (any_m) sc = mfma_qk<BF16>(ones_frag, mfrag, sc);
      }
      if constexpr (EW) {
        if ((cx >> 30) != 0) {
          const unsigned mw = reinterpret_cast<const unsigned*>(lds_v + C::TILE_BYTES)[2 * (32 * w + ln) + kh] >> (4 * g);
#pragma unroll
          for (int i = 0; i < 16; ++i) sc[i] = (mw & (1u << (8 * (i / 4) + (i % 4)))) ? sc[i] : -INFINITY;
        }
      } else if constexpr (TAIL) {
        if (keys < 32) {
          int first_key = 4 * g;
          asm volatile("" : "+v"(first_key));
#pragma unroll
          for (int i = 0; i < 16; ++i) sc[i] = 8 * (i / 4) + (i % 4) + first_key < keys ? sc[i] : -INFINITY;
        }
      }
      uintx4 pf[2];
      float lnew = 0.f;
      // A tile calls for a new reference: the first one (FOLD: it keeps 0 when its sums are of moderate size), and where numerators grow too
      // large.  PARTS: a first one that is known to (all but FOLD) saves a softmax, and another if it is in two parts (us, with them: 1 head N = 1024
      // keep 0.1 11.4, so 11.0; 3 heads N = 3000 keep 0.1 15.5, 14.8; D = 256 1 head N = 1024 keep 0.1 14.5, 13.7; the test for it costs long lists 1 %).
      const bool parts = PARTS && it < two_parts;
      bool far = PARTS && !FOLD && fresh;
      if (!far) {
        lnew = softmax_block<FOLD, PB>(sc, qk_scale, m_i, l_i, pf);
        far = __any((FOLD && fresh && !(lnew >= 0.25f)) || !(lnew - l_i < limit));
      }
      if (far || parts) {
        if (far) {
          recentre_block<DB, FOLD>(sc, oacc, qk_scale, m_i, l_i, mfrag, fresh, g);
          any_m = 1;
          if (!parts) lnew = softmax_block<FOLD, PB>(sc, qk_scale, m_i, l_i, pf);
        }
        if constexpr (PARTS) {
          if (parts) {
            uintx4 rest[2];
            lnew = softmax_block_parts<FOLD, PB>(sc, qk_scale, m_i, l_i, pf, rest);
#pragma unroll
            for (int ts = 0; ts < 2; ++ts)
#pragma unroll
              for (int db = 0; db < DB; ++db) oacc[db][0] = mfma_qk<PB>(vfr[ts][db], rest[ts], oacc[db][0]);
          }
        }
        if (far) limit = sum_limit<false>(lnew);
      }
      l_i = lnew;
      fresh = false;
      // ---- O^T += V^T P^T ----
#pragma unroll
      for (int ts = 0; ts < 2; ++ts)
#pragma unroll
        for (int db = 0; db < DB; ++db) oacc[db][0] = mfma_qk<PB>(vfr[ts][db], pf[ts], oacc[db][0]);
    }
    t = tn;
    cx = cxn;
  }

  // ---- merge: every wavefront's 32 rows into its group's stages, then 4 consecutive columns of a row per thread ----
  const float lsum = l_i + __shfl_xor(l_i, 32);
  float* ml = reinterpret_cast<float*>(lds + C::ML_OFF);
  __syncthreads();           // everybody has left the last step
  {
    float* own = reinterpret_cast<float*>(mine + kh * C::PART_BYTES) + (32 * w + ln) * C::PITCH + 4 * g;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int i4 = 0; i4 < 4; ++i4) {
        const floatx4 x = {oacc[db][0][4 * i4], oacc[db][0][4 * i4 + 1], oacc[db][0][4 * i4 + 2], oacc[db][0][4 * i4 + 3]};
        *reinterpret_cast<floatx4*>(own + 32 * db + 8 * i4) = x;
      }
    if (g == 0) {      // (a sum that is not a number stays in)
      ml[((2 * c + kh) * 64 + 32 * w + ln) * 2] = lsum != 0.f ? m_i : -INFINITY;
      ml[((2 * c + kh) * 64 + 32 * w + ln) * 2 + 1] = lsum;
    }
  }
  unsigned long long* arrivals = prm.flags + (int64_t)bh * nb + m;
  unsigned long long seen = 0ull;      // (a first guess of the compare-and-swap below: the read travels beside the merge)
  if (shares > 1 && threadIdx.x == 0) seen = __hip_atomic_load(arrivals, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  void* obase = out_base(prm, b, h);
  constexpr int QPR = D / 4, QT = 64 * QPR / (256 * S);      // quads per row, per thread
  static_assert(64 * QPR % (256 * S) == 0 && (QT == 4 || QT == 8), "the loads of a part go out together");
  auto put = [&](int r, int col, const floatx4& acc, float M, float L) {
    const int64_t q = (int64_t)m * 64 + r;
    if (TAIL && q >= prm.N) return;
    const float inv = EW || t0 == t1 ? row_inverse<true>(L) : row_inverse<false>(L);     // (no kept tile or no key: O = 0)
    store_out4<BF16>(obase, q * prm.os[2] + col, prm.out_f32, acc[0] * inv, acc[1] * inv, acc[2] * inv, acc[3] * inv);
    if (col == 0 && prm.lse != nullptr) prm.lse[(int64_t)bh * prm.N + q] = row_lse(M, L);
  };
  floatx4 sum[QT];
  float sum_m[QT], sum_l[QT];
#pragma unroll
  for (int it = 0; it < QT; ++it) {
    const int i = threadIdx.x + it * 256 * S, r = i / QPR, col = (i % QPR) * 4;
    float mp[2 * S], lp[2 * S], M = -INFINITY, L = 0.f;
    floatx4 acc = {0.f, 0.f, 0.f, 0.f}, part[2 * S];
#pragma unroll
    for (int cc = 0; cc < 2 * S; ++cc) {
      mp[cc] = ml[(cc * 64 + r) * 2];
      lp[cc] = ml[(cc * 64 + r) * 2 + 1];
      part[cc] = *reinterpret_cast<const floatx4*>(reinterpret_cast<const float*>(lds + (cc >> 1) * C::GROUP_BYTES + (cc & 1) * C::PART_BYTES) + r * C::PITCH + col);
    }
#pragma unroll
    for (int cc = 0; cc < 2 * S; ++cc) M = fmaxf(M, mp[cc]);
#pragma unroll
    for (int cc = 0; cc < 2 * S; ++cc) {
      const float wgt = mp[cc] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mp[cc] - M);
      L += wgt * lp[cc];
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[e] += wgt * part[cc][e];
    }
    if (shares == 1) put(r, col, acc, M, L);
    sum[it] = acc; sum_m[it] = M; sum_l[it] = L;
  }
  if (shares == 1) return;

  // ---- the shares of a list meet in the workspace, as the parts of a row block do in attn_fwd.hip: each is published with
  // device-scope stores and counted in once these are acknowledged, the last one in adds all of them up in their order ----
  const int64_t first_slot = ((int64_t)bh * nb + m) * prm.split;
  {
    float* slot = prm.part_o + (first_slot + chunk) * (64 * D) + wave * (QT * 256) + lane * 4;     // [wavefront][round][lane][4]
    float* slot_ml = prm.part_ml + (first_slot + chunk) * 128;
#pragma unroll
    for (int it = 0; it < QT; ++it) {
      const int i = threadIdx.x + it * 256 * S;
      coherent_store4(slot + it * 256, sum[it][0], sum[it][1], sum[it][2], sum[it][3]);
      if (i % QPR == 0) { coherent_store(slot_ml + 2 * (i / QPR), sum_m[it]); coherent_store(slot_ml + 2 * (i / QPR) + 1, sum_l[it]); }
    }
  }
  wait_vm<0>();
  __syncthreads();
  if (threadIdx.x == 0) lcols[0] = count_in(arrivals, prm.epoch, seen);
  __syncthreads();
  if (__builtin_amdgcn_readfirstlane(*(volatile int*)lcols) != shares) return;
  floatx4 acc[QT];
  float M[QT], L[QT];
#pragma unroll
  for (int it = 0; it < QT; ++it) { acc[it] = {0.f, 0.f, 0.f, 0.f}; M[it] = -INFINITY; L[it] = 0.f; }
  for (int p = 0; p < shares; ++p) {
    floatx4 x[QT];
    float mp[QT], lp[QT];
    if (p == chunk) {
#pragma unroll
      for (int it = 0; it < QT; ++it) { x[it] = sum[it]; mp[it] = sum_m[it]; lp[it] = sum_l[it]; }
    } else {
      const float* slot = prm.part_o + (first_slot + p) * (64 * D) + wave * (QT * 256) + lane * 4;
      const float* slot_ml = prm.part_ml + (first_slot + p) * 128;
#pragma unroll
      for (int it = 0; it < QT; ++it) {
        const int r = (threadIdx.x + it * 256 * S) / QPR;
        mp[it] = coherent_load(slot_ml + 2 * r);
        lp[it] = coherent_load(slot_ml + 2 * r + 1);
      }
      if constexpr (QT == 8) coherent_load4x8(slot, x);
      else coherent_load4x4(slot, x[0], x[1], x[2], x[3]);
    }
#pragma unroll
    for (int it = 0; it < QT; ++it) {
      const float mn = fmaxf(M[it], mp[it]);     // a side without mass has maximum -inf and weight 0
      const float wo = M[it] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(M[it] - mn);
      const float wp = mp[it] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mp[it] - mn);
      L[it] = L[it] * wo + lp[it] * wp;
      M[it] = mn;
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[it][e] = acc[it][e] * wo + wp * x[it][e];
    }
  }
#pragma unroll
  for (int it = 0; it < QT; ++it) {
    const int i = threadIdx.x + it * 256 * S;
    put(i / QPR, (i % QPR) * 4, acc[it], M[it], L[it]);
  }
  // back to zero, so that a replay of this launch (same mark) starts from a clean counter
  if (threadIdx.x == 0) __hip_atomic_store(arrivals, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <int D, int S, int DT, bool EW, bool TAIL, bool PARTS>
static void launch_quad_p(const FwdShareParams& prm, hipStream_t st) {
  constexpr int LDS = QuadCfg<D, S, EW>::LDS_BYTES;
  static std::atomic<unsigned long long> configured{0};   // raising the dynamic LDS limit is idempotent
  once_per_device(configured, [] {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&fwd_quad_kernel<D, S, DT, EW, TAIL, PARTS>), hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
  });
  const int grid = prm.place.per_share * prm.split;
  hipLaunchKernelGGL((fwd_quad_kernel<D, S, DT, EW, TAIL, PARTS>), dim3(grid), dim3(256 * S), LDS, st, prm);
}

template <int D, int S, int DT, bool EW, bool TAIL>
static void launch_quad_t(const FwdShareParams& prm, hipStream_t st) {
  if constexpr (DT == 0) launch_quad_p<D, S, DT, EW, TAIL, EW>(prm, st);       // (fp16: none with block masks, one at least with elementwise ones)
  else if (first_tiles<false>(prm.exact, S) > 0) launch_quad_p<D, S, DT, EW, TAIL, true>(prm, st);
  else launch_quad_p<D, S, DT, EW, TAIL, false>(prm, st);
}

template <int D, int S, int DT>
static void launch_quad_d(const FwdShareParams& prm, bool elementwise, hipStream_t st) {
  const bool tail = prm.N % 64 != 0;
  if (!elementwise) { if (tail) launch_quad_t<D, S, DT, false, true>(prm, st); else launch_quad_t<D, S, DT, false, false>(prm, st); }
  else { if (tail) launch_quad_t<D, S, DT, true, true>(prm, st); else launch_quad_t<D, S, DT, true, false>(prm, st); }
}

template <int D, int S>
static void launch_quad_s(const FwdShareParams& prm, int dt, bool elementwise, hipStream_t st) {
  if (dt == 0) launch_quad_d<D, S, 0>(prm, elementwise, st);
  else if (dt == 1) launch_quad_d<D, S, 1>(prm, elementwise, st);
  else launch_quad_d<D, S, 2>(prm, elementwise, st);
}

// D = 128.  groups: of four wavefronts per workgroup.  dt: 0 fp16, 1 bf16 with P rounded to fp16 (V converted), 2 bf16 with P rounded to bf16.
void launch_fwd_quad(const FwdShareParams& prm, int groups, int dt, bool elementwise, hipStream_t st) {
  if (groups == 1) launch_quad_s<128, 1>(prm, dt, elementwise, st);
  else launch_quad_s<128, 2>(prm, dt, elementwise, st);
}

}  // namespace bsattn
