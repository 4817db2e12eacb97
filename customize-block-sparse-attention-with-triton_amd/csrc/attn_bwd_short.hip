// Block-sparse FlashAttention-2 backward, head dimension 64, for launches with few lists: dK, dV and dQ in one launch.
//
// A workgroup has one column block (dK and dV of its keys) or one row block (dQ of its queries), or one of `split` contiguous
// shares of its list.  It is S pairs of wavefronts; pair c takes tiles c, c + S, ... of the list and the pairs' sums are added
// up in LDS at the end (as fwd_short_kernel does).  The dK/dV workgroups do not wait for delta = rowsum(O dO) of anybody: the
// rows of O travel beside those of Q and dO, and a wavefront has the dO fragments it needs in registers anyway.  So nothing
// orders the two kinds of workgroups, and they fill the GPU together: what a launch of few lists needs.  The products, layouts
// and roundings are those of attn_bwd.hip.
//
// Before, dq_kernel, then dkdv_kernel (which waits for delta), each with up to 8 workgroups per list and fp32 parts of dQ, dK
// and dV that a third launch added up: a third of the time of a short backward was parts and the gaps between launches.
// us, fp16: 8 heads N = 2048 keep 0.3 43 -> 21, block-causal 57 -> 40; 4 heads N = 512 dense 26 -> 13; 12 heads N = 3072 keep 0.3
// 83 -> 57; 4 heads N = 8192 block-causal 237 -> 159.  Bound by the chain of a step (fragments from LDS, products,
// exponentials, products) with two wavefronts per SIMD; the rows of O cost 7 % of a dense launch that has no need to be short.
#include "bwd_tile.h"

namespace bsattn {

// S: pairs of wavefronts per workgroup.  Lists of at most BWD_SHORT_MAX_BLOCKS tiles.
template <int S, bool EW> struct BwdShortCfg {
  static constexpr int D = 64, PITCH = D + 4;                        // PITCH: floats per row of a pair's sums in LDS (add_pairs)
  static constexpr int KV_BYTES = 64 * 2 * D, HALF_BYTES = KV_BYTES / 2, BITS_BYTES = EW ? 512 : 0;
  static constexpr int DQ_STAGE = 2 * KV_BYTES + BITS_BYTES;         // K tile, V tile, mask words
  static constexpr int DKV_STAGE = 3 * HALF_BYTES + 256 + BITS_BYTES;   // 32 rows of Q, dO and O, lse of the 64, mask words
  static constexpr int SUM_BYTES = 64 * PITCH * 4;
  static constexpr int BIGGER = DQ_STAGE > DKV_STAGE ? DQ_STAGE : DKV_STAGE;
  static constexpr int PAIR_BYTES = (2 * BIGGER > 2 * SUM_BYTES ? 2 * BIGGER : 2 * SUM_BYTES) + 255 & ~255;
  static constexpr int COLS_OFF = S * PAIR_BYTES;
  static constexpr int DELTA_OFF = COLS_OFF + BWD_SHORT_MAX_BLOCKS * 4;   // 32 floats per wavefront
  static constexpr int LDS_BYTES = DELTA_OFF + 2 * S * 32 * 4;
  static_assert(LDS_BYTES <= 160 * 1024, "fits a compute unit");
};

// sum of the products of the eight 16-bit elements of a and b: products exact, sums in fp32
template <bool BF16>
__device__ __forceinline__ float dot8_packed(const uintx4& a, const uintx4& b, float acc) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const unsigned au = a[i], bu = b[i];
    if constexpr (BF16) acc = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, au), __builtin_bit_cast(bf16x2, bu), acc, false);
    else acc = __builtin_amdgcn_fdot2(__builtin_bit_cast(half2v, au), __builtin_bit_cast(half2v, bu), acc, false);
  }
  return acc;
}

// The sums over the pairs, four consecutive values of one of the first `rows` rows per thread.  A pair's rows are D + 4 floats apart.
template <int D, int S, typename F>
__device__ __forceinline__ void add_pairs(const unsigned char* lds, int pair_bytes, int rows, F&& put) {
#pragma unroll 4
  for (int i = threadIdx.x; i < 64 * (D / 4); i += 128 * S) {
    const int r = i / (D / 4), col = i % (D / 4) * 4;
    if (r >= rows) break;
    floatx4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < S; ++c) {
      const floatx4 x = *reinterpret_cast<const floatx4*>(reinterpret_cast<const float*>(lds + c * pair_bytes) + r * (D + 4) + col);
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[e] += x[e];
    }
    put(r, col, acc);
  }
}

// dQ of row block m.  D = 64 walks whole tiles, D = 128 halves of 32 keys (attn_bwd.hip's dq_kernel).  C: where what is in LDS.
// delta: where delta of the queries goes for a dK/dV kernel that comes later, or null.
template <int D, int S, typename C, bool BF16, bool EW, bool PB, bool TAIL>
__device__ __forceinline__ void short_dq(const BwdParams& prm, unsigned char* lds, int bh, int b, int h, int mh, int m, int chunk, int split,
                                         float* delta) {
  constexpr int KS = D / 16, DB = D / 32, KB = D == 64 ? 2 : 1, ROWS = 32 * KB, STEPS = 2 / KB;
  constexpr int TILE_BYTES = ROWS * 2 * D, BITS_OFF = 2 * TILE_BYTES;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), c = wave >> 1, w = wave & 1;
  const int ln = lane & 31, g = lane >> 5, nb = prm.nb;
  const cint_ptr_t rp = (cint_ptr_t)(uintptr_t)(prm.row_ptr + (int64_t)mh * nb);
  const cint_ptr_t cols = (cint_ptr_t)(uintptr_t)prm.col_idx;
  const int64_t qrow = (int64_t)m * 64 + 32 * w + ln, qsrc = !TAIL || qrow < prm.N ? qrow : prm.N - 1;
  const int valid = TAIL ? prm.N - (nb - 1) * 64 : 64;
  const unsigned short* qp = (const unsigned short*)prm.q + b * prm.qs[0] + h * prm.qs[1] + qsrc * prm.qs[2];
  const unsigned short* gp = (const unsigned short*)prm.d_o + b * prm.dos[0] + h * prm.dos[1] + qsrc * prm.dos[2];
  const unsigned short* op = (const unsigned short*)prm.o + b * prm.os[0] + h * prm.os[1] + qsrc * prm.os[2];
  uintx4 qfr[KS], dofr[KS], ofr[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    qfr[s] = *reinterpret_cast<const uintx4*>(qp + 16 * s + 8 * g);
    dofr[s] = *reinterpret_cast<const uintx4*>(gp + 16 * s + 8 * g);
  }
#pragma unroll
  for (int s = 0; s < KS; ++s) ofr[s] = *reinterpret_cast<const uintx4*>(op + 16 * s + 8 * g);
  const float lse_q = prm.lse[(int64_t)bh * prm.N + qsrc];
  int t0, t1;
  {
    const int first = rp[m], len = rp[m + 1] - first;
    t0 = first + (int)((int64_t)len * chunk / split);
    t1 = first + (int)((int64_t)len * (chunk + 1) / split);
  }
  int* lcols = reinterpret_cast<int*>(lds + C::COLS_OFF);
  unsigned char* mine = lds + c * C::PAIR_BYTES;
  const unsigned mine_addr = (unsigned)(uintptr_t)(lds_ptr_t)lds + c * C::PAIR_BYTES;
  const unsigned short* kg = (const unsigned short*)prm.k + b * prm.ks[0] + h * prm.ks[1];
  const unsigned short* vg = (const unsigned short*)prm.v + b * prm.vs[0] + h * prm.vs[1];
  auto issue = [&](int cb, int t, int part, int stage) {       // rows ROWS part .. of the tile
    const unsigned sa = mine_addr + stage * C::DQ_STAGE;
    if (TAIL && cb == nb - 1) {
      tail_tile_load_async<2, D, ROWS>(kg + (int64_t)cb * 64 * prm.ks[2], prm.ks[2], part * ROWS, valid, w, lane, sa);
      tail_tile_load_async<2, D, ROWS>(vg + (int64_t)cb * 64 * prm.vs[2], prm.vs[2], part * ROWS, valid, w, lane, sa + TILE_BYTES);
    } else {
      const int64_t key0 = (int64_t)cb * 64 + part * ROWS;
      half_tile_load_async<D, ROWS>(kg + key0 * prm.ks[2], prm.ks[2], w, lane, sa);
      half_tile_load_async<D, ROWS>(vg + key0 * prm.vs[2], prm.vs[2], w, lane, sa + TILE_BYTES);
    }
    if constexpr (EW)   // the tile's 64 mask words, 256 bytes per wavefront
      stat_load_async(reinterpret_cast<const float*>(prm.bits_rows + (int64_t)t * 64) + w * 64, lane, sa + BITS_OFF + w * 256);
  };
  int t = t0 + c, cb = 0;
  if (t < t1) { cb = cols[t]; issue(cb, t, 0, 0); }
  for (int i = threadIdx.x; i < t1 - t0 && i < BWD_SHORT_MAX_BLOCKS; i += 128 * S) lcols[i] = prm.col_idx[t0 + i];
  // a query without any unmasked key has lse = -inf: every P of its row must come out as 0
  float lse2 = EW && lse_q == -INFINITY ? INFINITY : lse_q * kLog2e, dlt;
  {
    float acc = 0.f;
#pragma unroll
    for (int s = 0; s < KS; ++s) acc = dot8<BF16>(ofr[s], dofr[s], acc);
    dlt = acc + __shfl_xor(acc, 32);
    if (delta != nullptr && chunk == 0 && c == 0 && g == 0 && (!TAIL || qrow < prm.N)) delta[(int64_t)bh * prm.N + qrow] = dlt;
  }
#pragma unroll
  for (int s = 0; s < KS; ++s) { settle(qfr[s]); settle(dofr[s]); }
  settle(lse2); settle(dlt);
  const float qk_scale = prm.qk_scale;
  floatx16 dqacc[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) dqacc[db] = zero16();

  const int steps = STEPS * ((t1 - t0 + S - 1) / S);
  for (int it = 0; it < steps; ++it) {
    wait_vm<0>();
    __syncthreads();                              // the step's tiles are complete; everybody has left the step before
    const int part = it % STEPS, tn = part == STEPS - 1 ? t + S : t;
    int cbn = cb;
    if (tn < t1) {
      if (part == STEPS - 1) cbn = __builtin_amdgcn_readfirstlane(lcols[tn - t0]);
      issue(cbn, tn, (it + 1) % STEPS, (it + 1) & 1);
    }
    if (t < t1) {
      const unsigned char* kt = mine + (it & 1) * C::DQ_STAGE;
      const unsigned char* vt = kt + TILE_BYTES;
      floatx16 sacc[KB], dpacc[KB];
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) { sacc[kb] = zero16(); dpacc[kb] = zero16(); }
      {
        uintx4 fk[KB][KS], fv[KB][KS];
#pragma unroll
        for (int s = 0; s < KS; ++s)
#pragma unroll
          for (int kb = 0; kb < KB; ++kb) {
            fk[kb][s] = frag_rows<D>(kt, 32 * kb, s, ln, g);
            fv[kb][s] = frag_rows<D>(vt, 32 * kb, s, ln, g);
          }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < KS; ++s)
#pragma unroll
          for (int kb = 0; kb < KB; ++kb) {
            sacc[kb] = mfma_qk<BF16>(fk[kb][s], qfr[s], sacc[kb]);      // S^T = K Q^T
            dpacc[kb] = mfma_qk<BF16>(fv[kb][s], dofr[s], dpacc[kb]);   // dP^T = V dO^T
          }
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (EW) {
        const unsigned long long mw = *reinterpret_cast<const unsigned long long*>(kt + BITS_OFF + (32 * w + ln) * 8);
        if constexpr (KB == 2) mask_partly(sacc[0], sacc[1], mw >> (4 * g));
        else mask_scores(sacc[0], (unsigned)(mw >> (32 * part + 4 * g)));      // (D = 128: with the test 20 to 52 bytes per lane spilled)
      } else if (TAIL && cb == nb - 1) {
        const unsigned long long mw = tail_word(valid, g);
        if constexpr (KB == 2) mask_scores(sacc[0], sacc[1], mw);
        else mask_scores(sacc[0], (unsigned)(mw >> (32 * part)));
      }
      uintx4 fkt[2 * KB][DB];
#pragma unroll
      for (int ts = 0; ts < 2 * KB; ++ts)
#pragma unroll
        for (int db = 0; db < DB; ++db) fkt[ts][db] = frag_cols<D, BF16 && !PB>(kt, db, ts, lane);
      __builtin_amdgcn_sched_barrier(0);
      uintx4 dsf[2 * KB];       // dS^T = P^T * (dP^T - delta), packed as operand slices of 16 keys
#pragma unroll
      for (int ts = 0; ts < 2 * KB; ++ts)
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
          const int kb = ts >> 1, i = 8 * (ts & 1) + 2 * jj;
          const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(sacc[kb][i], qk_scale, -lse2));
          const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(sacc[kb][i + 1], qk_scale, -lse2));
          dsf[ts][jj] = pack2<PB>(p0 * (dpacc[kb][i] - dlt), p1 * (dpacc[kb][i + 1] - dlt));
        }
#pragma unroll
      for (int ts = 0; ts < 2 * KB; ++ts)
#pragma unroll
        for (int db = 0; db < DB; ++db) dqacc[db] = mfma_qk<PB>(fkt[ts][db], dsf[ts], dqacc[db]);       // dQ^T += K^T dS^T
    }
    t = tn;
    cb = cbn;
  }

  __syncthreads();           // everybody has left the last step
  {
    float* own = reinterpret_cast<float*>(mine) + (32 * w + ln) * (D + 4) + 4 * g;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int i4 = 0; i4 < 4; ++i4) {
        const floatx4 x = {dqacc[db][4 * i4], dqacc[db][4 * i4 + 1], dqacc[db][4 * i4 + 2], dqacc[db][4 * i4 + 3]};
        *reinterpret_cast<floatx4*>(own + 32 * db + 8 * i4) = x;
      }
  }
  __syncthreads();
  const int64_t r0 = (int64_t)m * 64, off = b * prm.dqs[0] + h * prm.dqs[1];
  void* base = prm.out_f32 ? (void*)((float*)prm.dq + off) : (void*)((unsigned short*)prm.dq + off);
  float* part = prm.part_dq + ((int64_t)chunk * prm.B * prm.H + bh) * prm.N * D;
  const float sc = prm.sm_scale;
  add_pairs<D, S>(lds, C::PAIR_BYTES, TAIL && r0 + 64 > prm.N ? prm.N - (int)r0 : 64, [&](int r, int col, const floatx4& x) {
    if (split > 1) *reinterpret_cast<floatx4*>(part + (r0 + r) * D + col) = x;
    else store_out4<BF16>(base, (r0 + r) * prm.dqs[2] + col, prm.out_f32, x[0] * sc, x[1] * sc, x[2] * sc, x[3] * sc);
  });
}

template <int S, bool BF16, bool EW, bool PB, bool TAIL>
__device__ __forceinline__ void short_dkdv(const BwdParams& prm, unsigned char* lds, int bh, int b, int h, int mh, int n, int chunk) {
  using C = BwdShortCfg<S, EW>;
  constexpr int D = 64, KS = D / 16, DB = D / 32, LSE_OFF = 3 * C::HALF_BYTES, BITS_OFF = LSE_OFF + 256;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), c = wave >> 1, w = wave & 1;
  const int ln = lane & 31, g = lane >> 5, nb = prm.nb;
  const cint_ptr_t cp = (cint_ptr_t)(uintptr_t)(prm.col_ptr + (int64_t)mh * nb);
  const cint_ptr_t rows = (cint_ptr_t)(uintptr_t)prm.row_idx;
  const int64_t krow = (int64_t)n * 64 + 32 * w + ln, ksrc = !TAIL || krow < prm.N ? krow : prm.N - 1;
  const int valid = TAIL ? prm.N - (nb - 1) * 64 : 64;
  const unsigned short* kp = (const unsigned short*)prm.k + b * prm.ks[0] + h * prm.ks[1] + ksrc * prm.ks[2];
  const unsigned short* vp = (const unsigned short*)prm.v + b * prm.vs[0] + h * prm.vs[1] + ksrc * prm.vs[2];
  uintx4 kfr[KS], vfr[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    kfr[s] = *reinterpret_cast<const uintx4*>(kp + 16 * s + 8 * g);
    vfr[s] = *reinterpret_cast<const uintx4*>(vp + 16 * s + 8 * g);
  }
  int t0, t1;
  {
    const int first = cp[n], len = cp[n + 1] - first;
    t0 = first + (int)((int64_t)len * chunk / prm.split);
    t1 = first + (int)((int64_t)len * (chunk + 1) / prm.split);
  }
  int* lrows = reinterpret_cast<int*>(lds + C::COLS_OFF);
  float* deltas = reinterpret_cast<float*>(lds + C::DELTA_OFF) + wave * 32;      // of the step's queries, this wavefront's own
  unsigned char* mine = lds + c * C::PAIR_BYTES;
  const unsigned mine_addr = (unsigned)(uintptr_t)(lds_ptr_t)lds + c * C::PAIR_BYTES;
  const unsigned short* qg = (const unsigned short*)prm.q + b * prm.qs[0] + h * prm.qs[1];
  const unsigned short* gg = (const unsigned short*)prm.d_o + b * prm.dos[0] + h * prm.dos[1];
  const unsigned short* og = (const unsigned short*)prm.o + b * prm.os[0] + h * prm.os[1];
  const float* lse_h = prm.lse + (int64_t)bh * prm.N;
  // queries 32 half .. 32 half + 31 of row block rb
  auto issue = [&](int rb, int t, int half, int stage) {
    const unsigned sa = mine_addr + stage * C::DKV_STAGE;
    int stat_lane = lane;
    if (TAIL && rb == nb - 1) {
      const int64_t r0 = (int64_t)rb * 64;
      tail_tile_load_async<2, D, 32>(qg + r0 * prm.qs[2], prm.qs[2], half * 32, valid, w, lane, sa);
      tail_tile_load_async<2, D, 32>(gg + r0 * prm.dos[2], prm.dos[2], half * 32, valid, w, lane, sa + C::HALF_BYTES);
      tail_tile_load_async<2, D, 32>(og + r0 * prm.os[2], prm.os[2], half * 32, valid, w, lane, sa + 2 * C::HALF_BYTES);
      stat_lane = lane < valid ? lane : valid - 1;
    } else {
      const int64_t r0 = (int64_t)rb * 64 + half * 32;
      half_tile_load_async<D, 32>(qg + r0 * prm.qs[2], prm.qs[2], w, lane, sa);
      half_tile_load_async<D, 32>(gg + r0 * prm.dos[2], prm.dos[2], w, lane, sa + C::HALF_BYTES);
      half_tile_load_async<D, 32>(og + r0 * prm.os[2], prm.os[2], w, lane, sa + 2 * C::HALF_BYTES);
    }
    if (w == 0) stat_load_async(lse_h + rb * 64, stat_lane, sa + LSE_OFF);         // of all 64 rows of the tile
    if constexpr (EW)   // the tile's 64 mask words (one per key, bit = query), 256 bytes per wavefront
      stat_load_async(reinterpret_cast<const float*>(prm.bits_cols + (int64_t)t * 64) + w * 64, lane, sa + BITS_OFF + w * 256);
  };
  int t = t0 + c, rb = 0;
  if (t < t1) { rb = rows[t]; issue(rb, t, 0, 0); }
  for (int i = threadIdx.x; i < t1 - t0 && i < BWD_SHORT_MAX_BLOCKS; i += 128 * S) lrows[i] = prm.row_idx[t0 + i];
#pragma unroll
  for (int s = 0; s < KS; ++s) { settle(kfr[s]); settle(vfr[s]); }
  const float qk_scale = prm.qk_scale;
  floatx16 dkacc[DB], dvacc[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) { dkacc[db] = zero16(); dvacc[db] = zero16(); }

  const int steps = 2 * ((t1 - t0 + S - 1) / S);      // a tile is walked in two steps of 32 queries
  for (int it = 0; it < steps; ++it) {
    wait_vm<0>();
    __syncthreads();
    const int half = it & 1, tn = half ? t + S : t;
    int rbn = rb;
    if (tn < t1) {
      if (half) rbn = __builtin_amdgcn_readfirstlane(lrows[tn - t0]);
      issue(rbn, tn, half ^ 1, (it + 1) & 1);
    }
    if (t < t1) {
      const unsigned char* qt = mine + half * C::DKV_STAGE;
      const unsigned char* gt = qt + C::HALF_BYTES;
      const unsigned char* ot = gt + C::HALF_BYTES;
      const float* st_lse = reinterpret_cast<const float*>(qt + LSE_OFF) + 32 * half;
      floatx16 sacc = zero16(), dpacc = zero16();
      {
        uintx4 fq[KS], fg[KS], fo[KS];
#pragma unroll
        for (int s = 0; s < KS; ++s) {
          fq[s] = frag_rows<D>(qt, 0, s, ln, g);
          fg[s] = frag_rows<D>(gt, 0, s, ln, g);
        }
#pragma unroll
        for (int s = 0; s < KS; ++s) fo[s] = frag_rows<D>(ot, 0, s, ln, g);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < KS; ++s) {
          sacc = mfma_qk<BF16>(fq[s], kfr[s], sacc);      // S = Q K^T
          dpacc = mfma_qk<BF16>(fg[s], vfr[s], dpacc);    // dP = dO V^T
        }
        // delta of query ln: this lane holds one half of its rows of dO and O, its neighbour 32 lanes on the other
        float acc = 0.f;
#pragma unroll
        for (int s = 0; s < KS; ++s) acc = dot8_packed<BF16>(fo[s], fg[s], acc);
        acc += __shfl_xor(acc, 32);
        if (g == 0) deltas[ln] = acc;
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (EW) mask_partly(sacc, (unsigned)(*reinterpret_cast<const unsigned long long*>(qt + BITS_OFF + (32 * w + ln) * 8) >> (32 * half + 4 * g)));
      else if (TAIL && rb == nb - 1) mask_scores(sacc, (unsigned)(tail_word(valid, g) >> (32 * half)));
      uintx4 fgt[2][DB], fqt[2][DB];      // dO^T and Q^T fragments of the second products
#pragma unroll
      for (int ts = 0; ts < 2; ++ts)
#pragma unroll
        for (int db = 0; db < DB; ++db) {
          fgt[ts][db] = frag_cols<D, BF16 && !PB>(gt, db, ts, lane);
          fqt[ts][db] = frag_cols<D, BF16 && !PB>(qt, db, ts, lane);
        }
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_sched_barrier(0);
      uintx4 pf[2], dsf[2];               // rows of the results are queries: register i <-> query 8(i/4) + 4g + i%4
#pragma unroll
      for (int ts = 0; ts < 2; ++ts)
#pragma unroll
        for (int jh = 0; jh < 2; ++jh) {
          const int i0 = 8 * ts + 4 * jh, q0 = 8 * (i0 >> 2) + 4 * g;
          const floatx4 l4 = *reinterpret_cast<const floatx4*>(st_lse + q0);
          const floatx4 d4 = *reinterpret_cast<const floatx4*>(deltas + q0);
          float p[4], ds[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            // (a query without any unmasked key has lse = -inf: its P must come out as 0)
            const float nl = EW && l4[e] == -INFINITY ? -INFINITY : -l4[e] * kLog2e;
            p[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(sacc[i0 + e], qk_scale, nl));
            ds[e] = p[e] * (dpacc[i0 + e] - d4[e]);
          }
          pf[ts][2 * jh] = pack2<PB>(p[0], p[1]);   pf[ts][2 * jh + 1] = pack2<PB>(p[2], p[3]);
          dsf[ts][2 * jh] = pack2<PB>(ds[0], ds[1]); dsf[ts][2 * jh + 1] = pack2<PB>(ds[2], ds[3]);
        }
#pragma unroll
      for (int ts = 0; ts < 2; ++ts)
#pragma unroll
        for (int db = 0; db < DB; ++db) {
          dvacc[db] = mfma_qk<PB>(fgt[ts][db], pf[ts], dvacc[db]);    // dV^T += dO^T P
          dkacc[db] = mfma_qk<PB>(fqt[ts][db], dsf[ts], dkacc[db]);   // dK^T += Q^T dS
        }
    }
    t = tn;
    rb = rbn;
  }

  __syncthreads();           // everybody has left the last step
  {
    float* own = reinterpret_cast<float*>(mine) + (32 * w + ln) * C::PITCH + 4 * g;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int i4 = 0; i4 < 4; ++i4) {
        const floatx4 x = {dkacc[db][4 * i4], dkacc[db][4 * i4 + 1], dkacc[db][4 * i4 + 2], dkacc[db][4 * i4 + 3]};
        const floatx4 y = {dvacc[db][4 * i4], dvacc[db][4 * i4 + 1], dvacc[db][4 * i4 + 2], dvacc[db][4 * i4 + 3]};
        *reinterpret_cast<floatx4*>(own + 32 * db + 8 * i4) = x;
        *reinterpret_cast<floatx4*>(own + C::SUM_BYTES / 4 + 32 * db + 8 * i4) = y;
      }
  }
  __syncthreads();
  const int64_t r0 = (int64_t)n * 64, koff = b * prm.dks[0] + h * prm.dks[1], voff = b * prm.dvs[0] + h * prm.dvs[1];
  void* kbase = prm.out_f32 ? (void*)((float*)prm.dk + koff) : (void*)((unsigned short*)prm.dk + koff);
  void* vbase = prm.out_f32 ? (void*)((float*)prm.dv + voff) : (void*)((unsigned short*)prm.dv + voff);
  const int64_t poff = ((int64_t)chunk * prm.B * prm.H + bh) * prm.N * D;
  const int here = TAIL && r0 + 64 > prm.N ? prm.N - (int)r0 : 64;
  const float sc = prm.sm_scale;
  add_pairs<D, S>(lds, C::PAIR_BYTES, here, [&](int r, int col, const floatx4& x) {
    if (prm.split > 1) *reinterpret_cast<floatx4*>(prm.part_dk + poff + (r0 + r) * D + col) = x;
    else store_out4<BF16>(kbase, (r0 + r) * prm.dks[2] + col, prm.out_f32, x[0] * sc, x[1] * sc, x[2] * sc, x[3] * sc);
  });
  add_pairs<D, S>(lds + C::SUM_BYTES, C::PAIR_BYTES, here, [&](int r, int col, const floatx4& x) {
    if (prm.split > 1) *reinterpret_cast<floatx4*>(prm.part_dv + poff + (r0 + r) * D + col) = x;
    else store_out4<BF16>(vbase, (r0 + r) * prm.dvs[2] + col, prm.out_f32, x[0], x[1], x[2], x[3]);
  });
}

// dK and dV, which take longer, in the first `split` shares of the grid, dQ in the others
template <int S, bool BF16, bool EW, bool PB, bool TAIL>
__global__ __launch_bounds__(128 * S, 2) void bwd_short_kernel(const BwdParams prm) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
  int share;
  const Place p = prm.place.of(blockIdx.x, share);
  if (p.item >= prm.nb) return;                   // padding of an incomplete last group
  const int bh = p.head, b = (int)prm.per_batch.of((unsigned)bh), h = bh - b * prm.H;
  const int mh = (prm.Bm > 1 ? b : 0) * prm.Hm + (prm.Hm > 1 ? h : 0);
  if (share < prm.split) short_dkdv<S, BF16, EW, PB, TAIL>(prm, lds, bh, b, h, mh, p.item, share);
  else short_dq<64, S, BwdShortCfg<S, EW>, BF16, EW, PB, TAIL>(prm, lds, bh, b, h, mh, prm.nb - 1 - p.item, share - prm.split, prm.split, nullptr);   // (long rows of causal masks first)
}

// dQ alone at D = 128, for launches with few lists (attn_bwd.hip, bwd_pairs_128): S pairs of wavefronts per row block where dq_kernel
// has one or several workgroups of one.  Bound by the chain of a step, S and dP, exponentials, dQ: at two wavefronts per SIMD one's
// products hide half of the other's chain, and each has 256 registers: ten of the 24 variants keep 12 to 36 bytes per lane in scratch memory
// (most: bf16 with P in fp16, 4 pairs).  One share per list: no parts, no sums.  (D = 256 with two pairs, a lone wavefront per SIMD
// like dq_kernel's, took longer than dq_kernel's shares at every size: 2 heads N = 4096 dense, backward 183 -> 281 us.)
template <int D, int S, bool EW> struct DqPairsCfg {
  static constexpr int DQ_STAGE = 2 * 32 * 2 * D + (EW ? 512 : 0), SUM_BYTES = 64 * (D + 4) * 4;
  static constexpr int PAIR_BYTES = (2 * DQ_STAGE > SUM_BYTES ? 2 * DQ_STAGE : SUM_BYTES) + 255 & ~255;
  static constexpr int COLS_OFF = S * PAIR_BYTES, LDS_BYTES = COLS_OFF + BWD_SHORT_MAX_BLOCKS * 4;
  static_assert(LDS_BYTES <= 160 * 1024, "fits a compute unit");
};

template <int D, int S, bool BF16, bool EW, bool PB, bool TAIL>
__global__ __launch_bounds__(128 * S, 2) void dq_pairs_kernel(const BwdParams prm) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
  int share;
  const Place p = prm.place_dq.of(blockIdx.x, share);
  if (p.item >= prm.nb) return;                   // padding of an incomplete last group
  const int bh = p.head, b = (int)prm.per_batch.of((unsigned)bh), h = bh - b * prm.H;
  const int mh = (prm.Bm > 1 ? b : 0) * prm.Hm + (prm.Hm > 1 ? h : 0);
  short_dq<D, S, DqPairsCfg<D, S, EW>, BF16, EW, PB, TAIL>(prm, lds, bh, b, h, mh, prm.nb - 1 - p.item, 0, 1, prm.delta);
}

template <int D, int S, bool BF16, bool EW, bool PB, bool TAIL>
static void launch_dq_t(const BwdParams& prm, hipStream_t st) {
  constexpr int LDS = DqPairsCfg<D, S, EW>::LDS_BYTES;
  static std::atomic<unsigned long long> configured{0};   // raising the dynamic LDS limit is idempotent
  once_per_device(configured, [] {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&dq_pairs_kernel<D, S, BF16, EW, PB, TAIL>), hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
  });
  hipLaunchKernelGGL((dq_pairs_kernel<D, S, BF16, EW, PB, TAIL>), dim3(prm.place_dq.per_share), dim3(128 * S), LDS, st, prm);
}

// pairs: 2 or 4 per workgroup
void launch_dq_pairs(const BwdParams& prm, int pairs, bool bf16, bool pb, hipStream_t st) {
  const bool ew = prm.bits_rows != nullptr, tail = prm.N % 64 != 0;
  auto pick = [&](auto ss, auto e, auto t) {
    constexpr int SS = decltype(ss)::value;
    constexpr bool E = decltype(e)::value, T = decltype(t)::value;
    if (!bf16) launch_dq_t<128, SS, false, E, false, T>(prm, st);
    else if (pb) launch_dq_t<128, SS, true, E, true, T>(prm, st);
    else launch_dq_t<128, SS, true, E, false, T>(prm, st);
  };
  auto pick_mask = [&](auto ss) {
    if (ew) { if (tail) pick(ss, std::true_type{}, std::true_type{}); else pick(ss, std::true_type{}, std::false_type{}); }
    else { if (tail) pick(ss, std::false_type{}, std::true_type{}); else pick(ss, std::false_type{}, std::false_type{}); }
  };
  if (pairs == 2) pick_mask(std::integral_constant<int, 2>{});
  else pick_mask(std::integral_constant<int, 4>{});
}

template <int S, bool BF16, bool EW, bool PB, bool TAIL>
static void launch_short_t(const BwdParams& prm, hipStream_t st) {
  constexpr int LDS = BwdShortCfg<S, EW>::LDS_BYTES;
  static std::atomic<unsigned long long> configured{0};   // raising the dynamic LDS limit is idempotent
  once_per_device(configured, [] {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&bwd_short_kernel<S, BF16, EW, PB, TAIL>), hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
  });
  hipLaunchKernelGGL((bwd_short_kernel<S, BF16, EW, PB, TAIL>), dim3(prm.place.per_share * 2 * prm.split), dim3(128 * S), LDS, st, prm);
}

template <int S, bool EW, bool TAIL>
static void launch_short_d(const BwdParams& prm, bool bf16, bool pb, hipStream_t st) {
  if (!bf16) launch_short_t<S, false, EW, false, TAIL>(prm, st);
  else if (pb) launch_short_t<S, true, EW, true, TAIL>(prm, st);
  else launch_short_t<S, true, EW, false, TAIL>(prm, st);
}

// pairs: 2 or 4 per workgroup.  prm.place: of 2 split shares.
void launch_bwd_short(const BwdParams& prm, int pairs, bool bf16, bool pb, hipStream_t st) {
  const bool ew = prm.bits_rows != nullptr, tail = prm.N % 64 != 0;
  auto pick = [&](auto s) {
    constexpr int S = decltype(s)::value;
    if (ew) { if (tail) launch_short_d<S, true, true>(prm, bf16, pb, st); else launch_short_d<S, true, false>(prm, bf16, pb, st); }
    else { if (tail) launch_short_d<S, false, true>(prm, bf16, pb, st); else launch_short_d<S, false, false>(prm, bf16, pb, st); }
  };
  if (pairs == 2) pick(std::integral_constant<int, 2>{});
  else pick(std::integral_constant<int, 4>{});
}

}  // namespace bsattn
