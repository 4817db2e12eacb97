// Block-sparse FlashAttention-2 backward for gfx950.
//
// Gradient algebra of the reference (fa2_custom_mask/fa2_bwd.py:17,57-74,117-130,232,284),
// evaluated over exactly the kept tiles:
//   delta = rowsum(O * dO);  P = exp(S*sm_scale - lse);  dV = P^T dO;  dP = dO V^T;
//   dS = P * (dP - delta);   dK = sm_scale * dS^T Q;     dQ = sm_scale * dS K.
// Two kernels, no atomics, results independent of scheduling:
//   dq_kernel     one workgroup (2 wavefronts x 32 queries) per row block, walking the row
//                 lists: per kept tile  S^T = K Q^T,  dP^T = V dO^T,  dQ^T += K^T dS^T;
//                 it also computes delta of its queries on the way in (dO is in its registers
//                 anyway) and leaves it in the workspace for the next kernel;
//   dkdv_kernel   one workgroup (2 wavefronts x 32 keys) per column block, walking the column
//                 lists: per kept tile  S = Q K^T,  dP = dO V^T,  dV^T += dO^T P,  dK^T += Q^T dS.
// Operand roles are chosen so that the fragment a wavefront owns for the whole walk (Q, dO or
// K, V) sits along the lanes: the per-row scalars (lse, delta) are then per-lane values in
// dq_kernel, P and dS leave the first products already in the operand layout of the second
// ones, and the tiles that change per step are staged in LDS by asynchronous copies into a
// double buffer (one barrier per tile).
// (D = 64 with few lists: attn_bwd_short.hip.)
#include <algorithm>
#include "bwd_tile.h"
#include <type_traits>

namespace bsattn {

// Is the list at lp, lp + 1 so short that the first share's workgroup walks all of it?  (The pointer as a value the
// compiler cannot trace back, or it makes these loads, and waits for them, in the workgroups of the first share too.)
__device__ __forceinline__ bool walked_by_first(cint_ptr_t lp, int whole) {
  asm volatile("" : "+s"(lp));
  return lp[1] - lp[0] <= whole;
}

// Entries [u0, u1) of a list [t0, t0 + len) are share `chunk` of it.  Returns the number of its shares (1: chunk is 0).
// BY_LENGTH: short lists may be one workgroup's (only in the kernels that are launched so, bwd_shares: the look at the
// length costs 0.3 us of a launch).
template <bool BY_LENGTH>
__device__ __forceinline__ int share_of_list(const BwdParams& prm, int t0, int len, int chunk, int& u0, int& u1) {
  if constexpr (BY_LENGTH) {
    u0 = t0;
    u1 = t0 + len;
    if (len <= prm.whole || prm.split == 1) return 1;
  }
  u0 = t0 + (int)((int64_t)len * chunk / prm.split);
  u1 = t0 + (int)((int64_t)len * (chunk + 1) / prm.split);
  return prm.split;
}
template <int D, bool EW> constexpr bool by_length = D == 128 && !EW;

// ---------------------------------------------------------------------------------------
// dQ: workgroup = row block m, wavefront wv owns queries 64m + 32wv + ln
// ---------------------------------------------------------------------------------------
// PB (bf16 inputs only): dS is rounded to bf16 and the second product runs in bf16 on the tile as it
// is; otherwise dS is rounded to fp16 and bf16 tiles are converted fragment by fragment.
// KB: 32-key blocks of a tile handled per step.  2: a whole tile per step.  1 (used at D = 128): a
// tile is walked in two steps of 32 keys; the staged halves are 8 KB, four workgroups fit a compute
// unit and the wavefront stays within 256 registers: two wavefronts per SIMD.
// TAIL: N is not a multiple of 64.  The last row block has queries that do not exist (its loads repeat the last query,
// nothing is written for them), the last tile of a list keys that do not exist (the copy repeats the last one, the scores
// are -inf).
template <int D, bool BF16, bool EW, bool PB, int KB, bool TAIL>
__global__ __launch_bounds__(128, D == 256 ? 1 : 2) void dq_kernel(const BwdParams prm) {
  using C = BwdCfg<D, EW, 32 * KB>;
  constexpr int KS = D / 16, DB = D / 32, STEPS = 2 / KB;
  constexpr int PORTIONS = D == 256 ? 2 : 1, KSP = KS / PORTIONS;   // D = 256: the fragments of the first products in two portions
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ln = lane & 31, g = lane >> 5;
  const int nb = prm.nb;
  int chunk;
  const Place p = prm.place.of(blockIdx.x, chunk);   // heads in groups of 8, one per XCD: the tiles its workgroups walk are shared in one L2
  if (p.item >= nb) return;
  const int bh = p.head, m = nb - 1 - p.item;        // long rows of block-causal masks first
  const int b = (int)prm.per_batch.of((unsigned)bh), h = bh - b * prm.H;
  const int mh = (prm.Bm > 1 ? b : 0) * prm.Hm + (prm.Hm > 1 ? h : 0);
  const cint_ptr_t rp = (cint_ptr_t)(uintptr_t)(prm.row_ptr + (int64_t)mh * nb);
  const cint_ptr_t cols = (cint_ptr_t)(uintptr_t)prm.col_idx;
  if (by_length<D, EW> && chunk > 0 && walked_by_first(rp + m, prm.whole)) return;
  // The rows this workgroup owns for its whole walk (Q, dO, O, lse of its queries) depend on the block index only:
  // they are asked for first, and travel while the list is looked up and the first tiles are requested.
  const int64_t qrow = (int64_t)m * 64 + 32 * wv + ln;
  const bool exists = !TAIL || qrow < prm.N;
  const int64_t qsrc = exists ? qrow : prm.N - 1;
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
  int u0, u1, split;                                           // steps: tile u / STEPS, part u % STEPS
  {
    const int t0 = rp[m], len = rp[m + 1] - t0;                // this workgroup's share of the row's list
    split = share_of_list<by_length<D, EW>>(prm, t0, len, chunk, u0, u1);
    u0 *= STEPS;
    u1 *= STEPS;
  }
  const unsigned lds_addr = (unsigned)(uintptr_t)(lds_ptr_t)lds;

  const unsigned short* kg = (const unsigned short*)prm.k + b * prm.ks[0] + h * prm.ks[1];
  const unsigned short* vg = (const unsigned short*)prm.v + b * prm.vs[0] + h * prm.vs[1];
  int blk_issued = 0;        // (TAIL) column block of the step issued last
  auto issue = [&](int u, int stage) {
    const int t = u / STEPS, cb = cols[t];
    const unsigned sa = lds_addr + stage * C::STAGE_BYTES;
    blk_issued = cb;
    if (TAIL && cb == nb - 1) {
      tail_tile_load_async<2, D, 32 * KB>(kg + (int64_t)cb * 64 * prm.ks[2], prm.ks[2], (u % STEPS) * 32 * KB, valid, wv, lane, sa);
      tail_tile_load_async<2, D, 32 * KB>(vg + (int64_t)cb * 64 * prm.vs[2], prm.vs[2], (u % STEPS) * 32 * KB, valid, wv, lane, sa + C::TILE_BYTES);
    } else {
      const int64_t key0 = (int64_t)cb * 64 + (u % STEPS) * 32 * KB;
      half_tile_load_async<D, 32 * KB>(kg + key0 * prm.ks[2], prm.ks[2], wv, lane, sa);
      half_tile_load_async<D, 32 * KB>(vg + key0 * prm.vs[2], prm.vs[2], wv, lane, sa + C::TILE_BYTES);
    }
    if constexpr (EW)   // the tile's 64 mask words, 256 bytes per wavefront
      stat_load_async(reinterpret_cast<const float*>(prm.bits_rows + (int64_t)t * 64) + wv * 64, lane,
                      lds_addr + stage * C::STAGE_BYTES + 2 * C::TILE_BYTES + C::STAT_BYTES + wv * 256);
  };
  if (u0 < u1) issue(u0, 0);

  // a query without any unmasked key has lse = -inf: every P of its row must come out as 0
  float lse2 = EW && lse_q == -INFINITY ? INFINITY : lse_q * kLog2e;
  // delta = rowsum(O * dO) (fa2_bwd.py:17): the lane holds one half of its query's row of dO, its neighbour 32
  // lanes on the other half.  Also kept for the dK/dV kernel, which needs it by key tile.
  float dlt;
  {
    float acc = 0.f;
#pragma unroll
    for (int s = 0; s < KS; ++s) acc = dot8<BF16>(ofr[s], dofr[s], acc);
    dlt = acc + __shfl_xor(acc, 32);
    if (chunk == 0 && g == 0 && exists) prm.delta[(int64_t)bh * prm.N + qrow] = dlt;
  }
#pragma unroll
  for (int s = 0; s < KS; ++s) { settle(qfr[s]); settle(dofr[s]); }
  settle(lse2); settle(dlt);       // everything above has arrived: no vector-memory waits in the loop
  const float qk_scale = prm.qk_scale;

  floatx16 dqacc[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) dqacc[db] = zero16();

  for (int u = u0; u < u1; ++u) {
    const int stage = (u - u0) & 1;
    wait_vm<0>();
    __syncthreads();   // step u complete in `stage`; everyone is done with the other stage
    const bool tail_step = TAIL && !EW && blk_issued == nb - 1;
    if (u + 1 < u1) issue(u + 1, stage ^ 1);
    const unsigned char* kt = lds + stage * C::STAGE_BYTES;
    const unsigned char* vt = kt + C::TILE_BYTES;

    // All operand fragments of a block of MFMAs are read from LDS before the block starts: a read
    // issued next to the MFMA that consumes it costs a full LDS latency per MFMA.
    floatx16 sacc[KB], dpacc[KB];
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) { sacc[kb] = zero16(); dpacc[kb] = zero16(); }
#pragma unroll
    for (int pt = 0; pt < PORTIONS; ++pt) {
      uintx4 fk[KB][KSP], fv[KB][KSP];
#pragma unroll
      for (int s = 0; s < KSP; ++s)
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
          fk[kb][s] = frag_rows<D>(kt, 32 * kb, pt * KSP + s, ln, g);
          fv[kb][s] = frag_rows<D>(vt, 32 * kb, pt * KSP + s, ln, g);
        }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int s = 0; s < KSP; ++s)
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
          sacc[kb] = mfma_qk<BF16>(fk[kb][s], qfr[pt * KSP + s], sacc[kb]);      // S^T = K Q^T
          dpacc[kb] = mfma_qk<BF16>(fv[kb][s], dofr[pt * KSP + s], dpacc[kb]);   // dP^T = V dO^T
        }
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (EW) {
      unsigned long long mw = *reinterpret_cast<const unsigned long long*>(
          vt + C::TILE_BYTES + C::STAT_BYTES + (32 * wv + ln) * 8);
      if constexpr (KB == 1) mw >>= 32 * (u % STEPS);
      mw >>= 4 * g;
      if constexpr (KB == 2) mask_partly(sacc[0], sacc[1], mw);
      else if constexpr (D == 256) mask_scores(sacc[0], (unsigned)mw);
      else mask_partly(sacc[0], (unsigned)mw);
    }
    if (tail_step) {
      const unsigned long long mw = tail_word(valid, g);
      if constexpr (KB == 2) mask_scores(sacc[0], sacc[1], mw);
      else mask_scores(sacc[0], (unsigned)(mw >> (32 * (u % STEPS))));
    }
    // K^T fragments of the second product, read under the exponentials below
    uintx4 fkt[2 * KB][DB];
#pragma unroll
    for (int ts = 0; ts < 2 * KB; ++ts)
#pragma unroll
      for (int db = 0; db < DB; ++db) fkt[ts][db] = frag_cols<D, BF16 && !PB>(kt, db, ts, lane);
    __builtin_amdgcn_sched_barrier(0);
    // dS^T = P^T * (dP^T - delta), this lane's query; packed as operand slices of 16 keys
    uintx4 dsf[2 * KB];
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
      for (int db = 0; db < DB; ++db)
        dqacc[db] = mfma_qk<PB>(fkt[ts][db], dsf[ts], dqacc[db]);       // dQ^T += K^T dS^T
  }

  if (split > 1) {   // unscaled fp32 part; sum_parts_kernel adds the parts up
    if (!exists) return;
    float* part = prm.part_dq + ((int64_t)chunk * prm.B * prm.H + bh) * prm.N * D;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int i4 = 0; i4 < 4; ++i4)
        store_out4<BF16>(part, qrow * D + 32 * db + 8 * i4 + 4 * g, true, dqacc[db][4 * i4], dqacc[db][4 * i4 + 1],
                         dqacc[db][4 * i4 + 2], dqacc[db][4 * i4 + 3]);
    return;
  }
  // dQ rows leave through this wavefront's stage of the (now idle) tile buffers
  static_assert(rows_out_bytes(D, true) <= C::STAGE_BYTES, "a stage holds a wavefront's 32 result rows");
  __syncthreads();           // the other wavefront has left its last step
  const float sc = prm.sm_scale;
  rows_out<BF16, D>(lds + wv * C::STAGE_BYTES, prm.dq, b * prm.dqs[0] + h * prm.dqs[1] + ((int64_t)m * 64 + 32 * wv) * prm.dqs[2],
                    prm.dqs[2], prm.out_f32, lane, TAIL ? prm.N - (m * 64 + 32 * wv) : 32, [&](int db, int i) { return dqacc[db][i] * sc; });
}

// ---------------------------------------------------------------------------------------
// dK, dV: workgroup = column block n, wavefront wv owns keys 64n + 32wv + ln
// ---------------------------------------------------------------------------------------
// A tile is walked in two steps of 32 queries, which halves the fragments in flight.
// (D = 64; larger head dimensions run dkdv4_kernel.)
template <int D, bool BF16, bool EW, bool PB, bool TAIL>
__global__ __launch_bounds__(128, 2) void dkdv_kernel(const BwdParams prm) {
  using C = BwdCfg<D, EW, 32>;
  constexpr int KS = D / 16, STEPS = 2;
  constexpr int DB = D / 32;
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ln = lane & 31, g = lane >> 5;
  const int nb = prm.nb;
  int chunk;
  const Place p = prm.place.of(blockIdx.x, chunk);   // (as in dq_kernel; early columns of block-causal masks are the long ones)
  if (p.item >= nb) return;
  const int bh = p.head, n = p.item;
  const int b = (int)prm.per_batch.of((unsigned)bh), h = bh - b * prm.H;
  const int mh = (prm.Bm > 1 ? b : 0) * prm.Hm + (prm.Hm > 1 ? h : 0);
  const cint_ptr_t cp = (cint_ptr_t)(uintptr_t)(prm.col_ptr + (int64_t)mh * nb);
  const cint_ptr_t rows = (cint_ptr_t)(uintptr_t)prm.row_idx;
  if (by_length<D, EW> && chunk > 0 && walked_by_first(cp + n, prm.whole)) return;
  int u0, u1, split;                                           // steps: tile u / STEPS, part u % STEPS
  {
    const int t0 = cp[n], len = cp[n + 1] - t0;                // this workgroup's share of the column's list
    split = share_of_list<by_length<D, EW>>(prm, t0, len, chunk, u0, u1);
    u0 *= STEPS;
    u1 *= STEPS;
  }
  const unsigned lds_addr = (unsigned)(uintptr_t)(lds_ptr_t)lds;

  const unsigned short* qg = (const unsigned short*)prm.q + b * prm.qs[0] + h * prm.qs[1];
  const unsigned short* gg = (const unsigned short*)prm.d_o + b * prm.dos[0] + h * prm.dos[1];
  const float* lse_h = prm.lse + (int64_t)bh * prm.N;
  const float* dlt_h = prm.delta + (int64_t)bh * prm.N;
  const int valid = TAIL ? prm.N - (nb - 1) * 64 : 64;
  int blk_issued = 0;        // (TAIL) row block of the step issued last
  auto issue = [&](int u, int stage) {
    const int t = u / STEPS;
    const int rb = rows[t];
    const unsigned sa = lds_addr + stage * C::STAGE_BYTES;
    blk_issued = rb;
    int stat_lane = lane;
    if (TAIL && rb == nb - 1) {
      tail_tile_load_async<2, D, 32>(qg + (int64_t)rb * 64 * prm.qs[2], prm.qs[2], (u % STEPS) * 32, valid, wv, lane, sa);
      tail_tile_load_async<2, D, 32>(gg + (int64_t)rb * 64 * prm.dos[2], prm.dos[2], (u % STEPS) * 32, valid, wv, lane, sa + C::TILE_BYTES);
      stat_lane = lane < valid ? lane : valid - 1;
    } else {
      const int64_t row0 = (int64_t)rb * 64 + (u % STEPS) * 32;
      half_tile_load_async<D, 32>(qg + row0 * prm.qs[2], prm.qs[2], wv, lane, sa);
      half_tile_load_async<D, 32>(gg + row0 * prm.dos[2], prm.dos[2], wv, lane, sa + C::TILE_BYTES);
    }
    stat_load_async((wv == 0 ? lse_h : dlt_h) + rb * 64, stat_lane, sa + 2 * C::TILE_BYTES + wv * 256);   // all 64 rows of the tile
    if constexpr (EW)   // the tile's 64 mask words (one per key, bit = query), 256 bytes per wavefront
      stat_load_async(reinterpret_cast<const float*>(prm.bits_cols + (int64_t)t * 64) + wv * 64, lane,
                      sa + 2 * C::TILE_BYTES + C::STAT_BYTES + wv * 256);
  };
  if (u0 < u1) issue(u0, 0);

  const int64_t krow = (int64_t)n * 64 + 32 * wv + ln;
  const bool exists = !TAIL || krow < prm.N;
  const int64_t ksrc = exists ? krow : prm.N - 1;
  const unsigned short* kp = (const unsigned short*)prm.k + b * prm.ks[0] + h * prm.ks[1] + ksrc * prm.ks[2];
  const unsigned short* vp = (const unsigned short*)prm.v + b * prm.vs[0] + h * prm.vs[1] + ksrc * prm.vs[2];
  uintx4 kfr[KS], vfr[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    kfr[s] = *reinterpret_cast<const uintx4*>(kp + 16 * s + 8 * g);
    vfr[s] = *reinterpret_cast<const uintx4*>(vp + 16 * s + 8 * g);
  }
#pragma unroll
  for (int s = 0; s < KS; ++s) { settle(kfr[s]); settle(vfr[s]); }   // no vector-memory waits in the loop, as in dq_kernel
  const float qk_scale = prm.qk_scale;

  floatx16 dkacc[DB], dvacc[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) { dkacc[db] = zero16(); dvacc[db] = zero16(); }

  for (int u = u0; u < u1; ++u) {
    const int stage = (u - u0) & 1;
    wait_vm<0>();
    __syncthreads();
    const bool tail_step = TAIL && !EW && blk_issued == nb - 1;
    if (u + 1 < u1) issue(u + 1, stage ^ 1);
    const unsigned char* qt = lds + stage * C::STAGE_BYTES;
    const unsigned char* gt = qt + C::TILE_BYTES;
    const int qoff = 32 * (u % STEPS);            // first query of this step within the tile
    const float* st_lse = reinterpret_cast<const float*>(gt + C::TILE_BYTES) + qoff;
    const float* st_dlt = st_lse + 64;

    // operand fragments are read from LDS ahead of the block of MFMAs that consumes them
    floatx16 sacc = zero16(), dpacc = zero16();
    {
      uintx4 fq[KS], fg[KS];
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        fq[s] = frag_rows<D>(qt, 0, s, ln, g);
        fg[s] = frag_rows<D>(gt, 0, s, ln, g);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        sacc = mfma_qk<BF16>(fq[s], kfr[s], sacc);      // S = Q K^T
        dpacc = mfma_qk<BF16>(fg[s], vfr[s], dpacc);    // dP = dO V^T
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (EW) {
      unsigned long long mw = *reinterpret_cast<const unsigned long long*>(
          gt + C::TILE_BYTES + C::STAT_BYTES + (32 * wv + ln) * 8);
      mask_partly(sacc, (unsigned)(mw >> (qoff + 4 * g)));
    }
    if (tail_step) mask_scores(sacc, (unsigned)(tail_word(valid, g) >> qoff));
    // dO^T and Q^T fragments of the second products, read under the exponentials below
    uintx4 fgt[2][DB], fqt[2][DB];
#pragma unroll
    for (int ts = 0; ts < 2; ++ts)
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        fgt[ts][db] = frag_cols<D, BF16 && !PB>(gt, db, ts, lane);
        fqt[ts][db] = frag_cols<D, BF16 && !PB>(qt, db, ts, lane);
      }
    __builtin_amdgcn_sched_barrier(0);
    // rows of the results are queries: register i <-> query 8(i/4) + 4g + i%4
    uintx4 pf[2], dsf[2];
#pragma unroll
    for (int ts = 0; ts < 2; ++ts)
#pragma unroll
      for (int jh = 0; jh < 2; ++jh) {
        const int i0 = 8 * ts + 4 * jh, q0 = 8 * (i0 >> 2) + 4 * g;
        const floatx4 l4 = *reinterpret_cast<const floatx4*>(st_lse + q0);
        const floatx4 d4 = *reinterpret_cast<const floatx4*>(st_dlt + q0);
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

  if (!exists) return;
  if (split > 1) {   // unscaled fp32 parts; sum_parts_kernel adds them up
    const int64_t poff = ((int64_t)chunk * prm.B * prm.H + bh) * prm.N * D;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int i4 = 0; i4 < 4; ++i4) {
        const int64_t off = krow * D + 32 * db + 8 * i4 + 4 * g;
        store_out4<BF16>(prm.part_dk + poff, off, true, dkacc[db][4 * i4], dkacc[db][4 * i4 + 1], dkacc[db][4 * i4 + 2],
                         dkacc[db][4 * i4 + 3]);
        store_out4<BF16>(prm.part_dv + poff, off, true, dvacc[db][4 * i4], dvacc[db][4 * i4 + 1], dvacc[db][4 * i4 + 2],
                         dvacc[db][4 * i4 + 3]);
      }
    return;
  }
  const int64_t koffh = b * prm.dks[0] + h * prm.dks[1], voffh = b * prm.dvs[0] + h * prm.dvs[1];
  void* kbase = prm.out_f32 ? (void*)((float*)prm.dk + koffh) : (void*)((unsigned short*)prm.dk + koffh);
  void* vbase = prm.out_f32 ? (void*)((float*)prm.dv + voffh) : (void*)((unsigned short*)prm.dv + voffh);
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int i4 = 0; i4 < 4; ++i4) {
      const int col = 32 * db + 8 * i4 + 4 * g;
      const int64_t off = krow * prm.dks[2] + col;
      store_out4<BF16>(kbase, off, prm.out_f32, dkacc[db][4 * i4] * prm.sm_scale, dkacc[db][4 * i4 + 1] * prm.sm_scale,
                       dkacc[db][4 * i4 + 2] * prm.sm_scale, dkacc[db][4 * i4 + 3] * prm.sm_scale);
      store_out4<BF16>(vbase, krow * prm.dvs[2] + col, prm.out_f32, dvacc[db][4 * i4], dvacc[db][4 * i4 + 1], dvacc[db][4 * i4 + 2],
                       dvacc[db][4 * i4 + 3]);
    }
}

// ---------------------------------------------------------------------------------------
// dK, dV at D = 128 and 256: workgroup = column block n, four wavefronts (one per SIMD).
// Wavefront (kh, dh) owns keys 64n + 32kh + ln and the columns 64dh .. 64dh + 63 of their dK and dV rows: half
// the accumulators of dkdv_kernel's wavefront, which, with K, V, dK and dV of its keys in 192 of 512
// registers, runs alone on its SIMD and leaves the matrix cores idle two thirds of the time.  Here a wavefront
// stays within 256 registers and two workgroups share a compute unit (two wavefronts per SIMD).
// The first products (S, dP) contract over the whole head dimension, so the two wavefronts of a key half share
// them by query block: wavefront dh computes S and dP of queries 32dh .. 32dh + 31, turns them into P and dS,
// and hands both, packed as the operand fragments of the second products, to its partner through LDS (4 KB
// each way, one barrier).  Every wavefront then runs the second products of both query blocks on its columns,
// its own block first, while the partner's P and dS are on their way.
// The per-query terms (- lse in the exponent, - delta beside dP) enter through one extra contraction slice each,
// ones x the term in three 16-bit pieces, as the forward does with its reference exponent: no vector
// instruction per element, and the row statistics need no place in LDS: a lane reads the two values of its
// query from memory a step ahead.  (Two stages of a Q and a dO tile, 64 KB, + 16 KB of exchange are exactly half
// the 160 KB of a compute unit: two workgroups per compute unit, two wavefronts per SIMD.)
// D = 256: the same split with 128 columns, 500 registers and 145 KB of LDS per wavefront and workgroup, one wavefront per
// SIMD; lse and delta are staged in LDS and stay fp32 (the pieces have a limited range).  Before, dkdv_kernel ran twice,
// 128 columns of dK and dV each time: S and dP twice (6 products for 4) and every tile copied twice.  Backward, bf16:
// 12 heads N = 4096 causal 0.5 519 -> 333 us, 16 heads N = 8192 keep 0.3 1780 -> 1540, 2 heads N = 1000 96 -> 61 (two
// shares each).  Bound by its lone wavefront's chain: first products, exponentials, exchange, second products.
// G = 2 (D = 128): two such groups of four wavefronts in a workgroup have half of the column's list each, and their sums are added
// through LDS, dK by the first group and dV by the second.  (The loop is each group's own; the shorter half's group then meets the
// two barriers of the other's last step.  With that case inside the loop the compiler held K and V in scratch.)
// ---------------------------------------------------------------------------------------
template <int NWV, int D, int ROWS>
__device__ __forceinline__ void part_tile_load_async(const unsigned short* tile, int64_t stride, int wv, int lane,
                                                     unsigned lds_addr) {
  constexpr int CPR = D / 8, PER_WAVE = ROWS * CPR / (64 * NWV);
#pragma unroll
  for (int jj = 0; jj < PER_WAVE; ++jj) {
    const int j = wv * PER_WAVE + jj;
    const int c = j * 64 + lane, row = c / CPR, ch = c % CPR;
    const unsigned off = 2u * (unsigned)(row * (int)stride + ((ch ^ u_swz<D>(row)) * 8));
    tile_load_async_one(tile, off, lds_addr + j * 1024);
  }
}

// x as three 16-bit pieces (hi, mid, lo; fp16 or bf16) in the first three contraction slots of an operand slice.
// fp16 pieces hold x / PIECE_GAIN and the other operand of the slice holds PIECE_GAIN instead of ones: lse / sm_scale
// (about the largest raw q k) and delta = rowsum(O dO) (of the order |dO| sqrt(D), large under loss scaling) may lie
// far above fp16's 65504, where the first piece would be infinite and the remainders NaN.  With the gain the
// pieces reach +-4.1e6 (beyond that x is clamped: finite, wrong results instead of NaN) and are exact to
// max(2^-33 |x|, 2e-6).  bf16 pieces have fp32's range and need no gain.
constexpr float PIECE_GAIN = 64.0f;
template <bool BF16>
__device__ __forceinline__ uintx4 three_pieces(float x, bool holder) {
  unsigned short p[3];
  float rest = x;
  if constexpr (!BF16) {
    constexpr float LIM = 65000.0f;
    rest = fminf(fmaxf(x * (1.0f / PIECE_GAIN), -LIM), LIM);
  }
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    if constexpr (BF16) {
      const __bf16 v = (__bf16)rest;
      p[i] = __builtin_bit_cast(unsigned short, v);
      rest -= (float)v;
    } else {
      const _Float16 v = (_Float16)rest;
      p[i] = __builtin_bit_cast(unsigned short, v);
      rest -= (float)v;
    }
  }
  uintx4 r = {0u, 0u, 0u, 0u};
  if (holder) { r[0] = (unsigned)p[0] | ((unsigned)p[1] << 16); r[1] = (unsigned)p[2]; }
  return r;
}

// two stages of a Q and a dO tile, 4 KB of exchange per wavefront, at D = 256 two stages of lse and delta
template <int D> constexpr int dkdv4_lds_bytes() { return 4 * 64 * 2 * D + 4 * 4096 + (D == 256 ? 2 * 512 : 0); }
template <int D, bool BF16, bool PB, bool EW, bool TAIL, int G = 1>
__global__ __launch_bounds__(256 * G, D == 128 ? 2 : 1) void dkdv4_kernel(const BwdParams prm) {
  static_assert(D == 128 || D == 256, "two or four 32-column blocks of dK and dV per wavefront");
  constexpr int KS = D / 16, DBW = D / 64;           // 32-column blocks per wavefront
  constexpr int TILE_BYTES = 64 * 2 * D, STAGE_BYTES = 2 * TILE_BYTES, EXCH_OFF = 2 * STAGE_BYTES, STAT_OFF = EXCH_OFF + 4 * 4096;
  constexpr bool PIECES = D == 128;                  // lse and delta by way of the matrix cores
  constexpr int PORTIONS = KS / 4, KSP = KS / PORTIONS;   // fragments of the first products in portions
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds_all[];
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane((threadIdx.x >> 6) & 3);
  const int grp = G == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
  unsigned char* lds = lds_all + grp * dkdv4_lds_bytes<D>();
  const int kh = wv & 1, dh = wv >> 1;
  const int ln = lane & 31, g = lane >> 5;
  const int nb = prm.nb;
  int chunk;
  const Place p = prm.place.of(blockIdx.x, chunk);   // (as in dq_kernel; early columns of block-causal masks are the long ones)
  if (p.item >= nb) return;
  const int bh = p.head, n = p.item;
  const int b = (int)prm.per_batch.of((unsigned)bh), h = bh - b * prm.H;
  const int mh = (prm.Bm > 1 ? b : 0) * prm.Hm + (prm.Hm > 1 ? h : 0);
  const cint_ptr_t cp = (cint_ptr_t)(uintptr_t)(prm.col_ptr + (int64_t)mh * nb);
  const cint_ptr_t rows = (cint_ptr_t)(uintptr_t)prm.row_idx;
  if (by_length<D, EW> && chunk > 0 && walked_by_first(cp + n, prm.whole)) return;
  // The K and V rows this wavefront owns for the whole walk depend on the block index only: asked for first, they
  // travel while the list is looked up and the first tiles are requested.
  const int64_t krow = (int64_t)n * 64 + 32 * kh + ln;
  const bool exists = !TAIL || krow < prm.N;
  const int64_t ksrc = exists ? krow : prm.N - 1;
  const int valid = TAIL ? prm.N - (nb - 1) * 64 : 64;
  const unsigned short* kp = (const unsigned short*)prm.k + b * prm.ks[0] + h * prm.ks[1] + ksrc * prm.ks[2];
  const unsigned short* vp = (const unsigned short*)prm.v + b * prm.vs[0] + h * prm.vs[1] + ksrc * prm.vs[2];
  uintx4 kfr[KS], vfr[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    kfr[s] = *reinterpret_cast<const uintx4*>(kp + 16 * s + 8 * g);
    vfr[s] = *reinterpret_cast<const uintx4*>(vp + 16 * s + 8 * g);
  }
  int u0, u1, split;
  {
    const int t0 = cp[n], len = cp[n + 1] - t0;                // this workgroup's share of the column's list
    split = share_of_list<by_length<D, EW>>(prm, t0, len, chunk, u0, u1);
  }
  int rounds = 0;            // G = 2: steps of the group with the longer half of the list, one more than the other's at most
  if constexpr (G == 2) {
    const int half = (u1 - u0 + 1) / 2;
    if (grp == 0) u1 = u0 + half;
    else u0 = u0 + half;
    rounds = half;
  }
  const unsigned lds_addr = (unsigned)(uintptr_t)(lds_ptr_t)lds;
  const unsigned short* qg = (const unsigned short*)prm.q + b * prm.qs[0] + h * prm.qs[1];
  const unsigned short* gg = (const unsigned short*)prm.d_o + b * prm.dos[0] + h * prm.dos[1];
  const float* lse_h = prm.lse + (int64_t)bh * prm.N;
  const float* dlt_h = prm.delta + (int64_t)bh * prm.N;
  const float inv_scale = 1.0f / prm.sm_scale;
  int blk_issued = 0;        // (TAIL) row block of the step issued last
  // tile copies of step u into `stage`
  auto issue = [&](int u, int stage) {
    const int rb = rows[u];
    const unsigned sa = lds_addr + stage * STAGE_BYTES;
    blk_issued = rb;
    if constexpr (!PIECES)
      if (wv < 2) stat_load_async((wv == 0 ? lse_h : dlt_h) + (int64_t)rb * 64, TAIL && rb == nb - 1 && lane >= valid ? valid - 1 : lane,
                                  lds_addr + STAT_OFF + stage * 512 + wv * 256);
    if (TAIL && rb == nb - 1) {
      tail_tile_load_async<4, D, 64>(qg + (int64_t)rb * 64 * prm.qs[2], prm.qs[2], 0, valid, wv, lane, sa);
      tail_tile_load_async<4, D, 64>(gg + (int64_t)rb * 64 * prm.dos[2], prm.dos[2], 0, valid, wv, lane, sa + TILE_BYTES);
      return;
    }
    part_tile_load_async<4, D, 64>(qg + (int64_t)rb * 64 * prm.qs[2], prm.qs[2], wv, lane, sa);
    part_tile_load_async<4, D, 64>(gg + (int64_t)rb * 64 * prm.dos[2], prm.dos[2], wv, lane, sa + TILE_BYTES);
  };
  // lse and delta of this lane's query (of the wavefront's query block) in step u.  Ordinary loads, asked for
  // before the step's tile copies and first used after the wait for those copies at the top of the step: the
  // wait the compiler puts in front of that use then finds nothing in flight.
  // Elementwise masks: entry u of the column lists has 64 words, one per key of the tile, bit = query; a lane
  // reads the word of its key the same way.
  float st_lse = 0.f, st_dlt = 0.f;
  unsigned long long st_bits = 0ull;
  auto ask_stats = [&](int u) {
    int q = rows[u] * 64 + 32 * dh + ln;
    if (TAIL && q >= prm.N) q = prm.N - 1;
    if constexpr (PIECES) {
      st_lse = lse_h[q];
      st_dlt = dlt_h[q];
    }
    if constexpr (EW) st_bits = prm.bits_cols[(int64_t)u * 64 + 32 * kh + ln];
  };
  if (u0 < u1) { ask_stats(u0); issue(u0, 0); }

#pragma unroll
  for (int s = 0; s < KS; ++s) { settle(kfr[s]); settle(vfr[s]); }   // K and V are there: no waits for them in the loop
  const float qk_scale = prm.qk_scale;
  // ones in the three slots the pieces occupy (second operand of the extra slices)
  const unsigned one16 = BF16 ? 0x3f80u : 0x5400u;      // 1.0 (bf16) or PIECE_GAIN = 64.0 (fp16), see three_pieces
  static_assert(PIECE_GAIN == 64.0f, "0x5400 is 64.0 in fp16");
  const uintx4 ones_frag = {g == 0 ? (one16 | (one16 << 16)) : 0u, g == 0 ? one16 : 0u, 0u, 0u};

  floatx16 dkacc[DBW], dvacc[DBW];
#pragma unroll
  for (int db = 0; db < DBW; ++db) { dkacc[db] = zero16(); dvacc[db] = zero16(); }
  uintx4* exch_mine = reinterpret_cast<uintx4*>(lds + EXCH_OFF + wv * 4096);
  const uintx4* exch_partner = reinterpret_cast<const uintx4*>(lds + EXCH_OFF + (wv ^ 2) * 4096);
  // one block of second products, the 32 queries of block qb against this wavefront's columns, in two parts: the
  // transposed fragments of dO and Q are read from LDS well ahead of the MFMAs that consume them
  auto read_cols = [&](const unsigned char* qt, const unsigned char* gt, int qb, uintx4 (&fgt)[2][DBW], uintx4 (&fqt)[2][DBW]) {
#pragma unroll
    for (int t2 = 0; t2 < 2; ++t2)
#pragma unroll
      for (int db = 0; db < DBW; ++db) {
        fgt[t2][db] = frag_cols<D, BF16 && !PB>(gt, DBW * dh + db, 2 * qb + t2, lane);
        fqt[t2][db] = frag_cols<D, BF16 && !PB>(qt, DBW * dh + db, 2 * qb + t2, lane);
      }
  };
  auto second = [&](const uintx4 (&fgt)[2][DBW], const uintx4 (&fqt)[2][DBW], const uintx4 (&pf)[2], const uintx4 (&dsf)[2]) {
#pragma unroll
    for (int t2 = 0; t2 < 2; ++t2)
#pragma unroll
      for (int db = 0; db < DBW; ++db) {
        dvacc[db] = mfma_qk<PB>(fgt[t2][db], pf[t2], dvacc[db]);    // dV^T += dO^T P
        dkacc[db] = mfma_qk<PB>(fqt[t2][db], dsf[t2], dkacc[db]);   // dK^T += Q^T dS
      }
  };

  for (int u = u0; u < u1; ++u) {
    const int stage = (u - u0) & 1;
    wait_vm<0>();
    __syncthreads();                 // the step's tiles are complete; everybody has left the previous step
    // the extra slices of this step from the statistics asked for a step ago; then the next step's
    // (a query without any unmasked key has lse = -inf; all its scores are masked below, whatever the slice holds)
    uintx4 lse_slice, dlt_slice;
    if constexpr (PIECES) {
      lse_slice = three_pieces<BF16>(EW && st_lse == -INFINITY ? 0.f : -st_lse * inv_scale, g == 0);
      dlt_slice = three_pieces<BF16>(-st_dlt, g == 0);
    }
    // the mask bits of this lane's key for the queries of this wavefront's block, shifted so that bit
    // 8(i/4) + i%4 belongs to register i
    const unsigned mw = EW ? (unsigned)(st_bits >> (32 * dh)) >> (4 * g) : 0u;
    __builtin_amdgcn_sched_barrier(0);
    const bool tail_step = TAIL && !EW && blk_issued == nb - 1;
    if (u + 1 < u1) { ask_stats(u + 1); issue(u + 1, stage ^ 1); }
    const unsigned char* qt = lds + stage * STAGE_BYTES;
    const unsigned char* gt = qt + TILE_BYTES;

    // ---- first products of this wavefront's query block: S' = Q K^T - lse / sm_scale, dP' = dO V^T - delta ----
    floatx16 sacc = zero16(), dpacc = zero16();
    {
      // (the fragments in portions of four slices: all at once they do not fit beside K, V and the accumulators)
#pragma unroll
      for (int pt = 0; pt < PORTIONS; ++pt) {
        uintx4 fq[KSP], fg[KSP];
#pragma unroll
        for (int s = 0; s < KSP; ++s) {
          fq[s] = frag_rows<D>(qt, 32 * dh, pt * KSP + s, ln, g);
          fg[s] = frag_rows<D>(gt, 32 * dh, pt * KSP + s, ln, g);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < KSP; ++s) {
          sacc = mfma_qk<BF16>(fq[s], kfr[pt * KSP + s], sacc);
          dpacc = mfma_qk<BF16>(fg[s], vfr[pt * KSP + s], dpacc);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (PIECES) {
        sacc = mfma_qk<BF16>(lse_slice, ones_frag, sacc);
        dpacc = mfma_qk<BF16>(dlt_slice, ones_frag, dpacc);
      }
    }
    if constexpr (EW && D == 256) mask_scores(sacc, mw);
    else if constexpr (EW) mask_partly(sacc, mw);
    if (tail_step) mask_scores(sacc, (unsigned)(tail_word(valid, g) >> (32 * dh)));
    // (the fragments of the own block's second products are on their way while the vector ALU works)
    uintx4 fgt_own[2][DBW], fqt_own[2][DBW];
    read_cols(qt, gt, dh, fgt_own, fqt_own);
    __builtin_amdgcn_sched_barrier(0);
    // ---- P and dS (rows of the results are queries: register i <-> query 32dh + 8(i/4) + 4g + i%4), packed as
    // the operand slices of the second products, and handed to the partner ----
    uintx4 pm[2], dm[2];             // [16-query slice of this wavefront's query block]
#pragma unroll
    for (int t2 = 0; t2 < 2; ++t2) {
#pragma unroll
      for (int jh = 0; jh < 2; ++jh) {
        const int i0 = 8 * t2 + 4 * jh;
        float p[4], ds[4];
        floatx4 l4, d4;
        if constexpr (!PIECES) {
          const float* st = reinterpret_cast<const float*>(lds + STAT_OFF + stage * 512) + 32 * dh + 8 * (i0 >> 2) + 4 * g;
          l4 = *reinterpret_cast<const floatx4*>(st);
          d4 = *reinterpret_cast<const floatx4*>(st + 64);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if constexpr (PIECES) {
            p[e] = __builtin_amdgcn_exp2f(sacc[i0 + e] * qk_scale);
            ds[e] = p[e] * dpacc[i0 + e];
          } else {   // (a query without any unmasked key has lse = -inf: its P must come out as 0)
            const float nl = EW && l4[e] == -INFINITY ? -INFINITY : -l4[e] * kLog2e;
            p[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(sacc[i0 + e], qk_scale, nl));
            ds[e] = p[e] * (dpacc[i0 + e] - d4[e]);
          }
        }
        pm[t2][2 * jh] = pack2<PB>(p[0], p[1]);   pm[t2][2 * jh + 1] = pack2<PB>(p[2], p[3]);
        dm[t2][2 * jh] = pack2<PB>(ds[0], ds[1]); dm[t2][2 * jh + 1] = pack2<PB>(ds[2], ds[3]);
      }
    }
    // ---- exchange, the second products of the own query block in between ----
#pragma unroll
    for (int t2 = 0; t2 < 2; ++t2) { exch_mine[(2 * t2) * 64 + lane] = pm[t2]; exch_mine[(2 * t2 + 1) * 64 + lane] = dm[t2]; }
    uintx4 fgt_oth[2][DBW], fqt_oth[2][DBW];
    read_cols(qt, gt, 1 - dh, fgt_oth, fqt_oth);
    __builtin_amdgcn_sched_barrier(0);
    second(fgt_own, fqt_own, pm, dm);
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();
    uintx4 pp[2], dp[2];
#pragma unroll
    for (int t2 = 0; t2 < 2; ++t2) { pp[t2] = exch_partner[(2 * t2) * 64 + lane]; dp[t2] = exch_partner[(2 * t2 + 1) * 64 + lane]; }
    second(fgt_oth, fqt_oth, pp, dp);
  }

  if (G == 2 && u1 - u0 < rounds) {  // the first group has one more step: its two barriers
    __syncthreads();
    __syncthreads();
  }
  if constexpr (G == 2) {            // the two groups' sums: the first adds up dK, the second dV
    static_assert(D == 128, "fits");
    __syncthreads();                 // everybody has left the last step
    // (the lane index as a value the compiler cannot trace back, as below)
    int lane_out = lane;
    asm volatile("" : "+v"(lane_out));
    floatx4* give = reinterpret_cast<floatx4*>(lds + wv * DBW * 4096);
    const floatx4* take = reinterpret_cast<const floatx4*>(lds_all + (1 - grp) * dkdv4_lds_bytes<D>() + wv * DBW * 4096);
    auto quads = [&](floatx16 (&mine_acc)[DBW], const floatx16 (&given)[DBW]) {
#pragma unroll
      for (int db = 0; db < DBW; ++db)
#pragma unroll
        for (int i4 = 0; i4 < 4; ++i4) {
          const floatx4 x = {given[db][4 * i4], given[db][4 * i4 + 1], given[db][4 * i4 + 2], given[db][4 * i4 + 3]};
          give[(4 * db + i4) * 64 + lane_out] = x;
        }
      __syncthreads();
#pragma unroll
      for (int db = 0; db < DBW; ++db)
#pragma unroll
        for (int i4 = 0; i4 < 4; ++i4) {
          const floatx4 x = take[(4 * db + i4) * 64 + lane_out];
#pragma unroll
          for (int e = 0; e < 4; ++e) mine_acc[db][4 * i4 + e] += x[e];
        }
    };
    const int64_t r0 = (int64_t)n * 64 + 32 * kh;
    constexpr int OUT_BYTES = rows_out_bytes(32 * DBW, true);
    static_assert(4 * (DBW * 4096 + OUT_BYTES) <= dkdv4_lds_bytes<D>(), "room for the sums and for the results of four wavefronts");
    unsigned char* mine = lds + 4 * DBW * 4096 + wv * OUT_BYTES;
    auto put = [&](const floatx16 (&acc)[DBW], void* out, const int64_t* st, float sc) {
      rows_out<BF16, 32 * DBW>(mine, out, b * st[0] + h * st[1] + r0 * st[2] + 32 * DBW * dh, st[2], prm.out_f32, lane_out,
                               TAIL ? prm.N - (int)r0 : 32, [&](int db, int i) { return acc[db][i] * sc; });
    };
    if (grp == 0) { quads(dkacc, dvacc); put(dkacc, prm.dk, prm.dks, prm.sm_scale); }
    else { quads(dvacc, dkacc); put(dvacc, prm.dv, prm.dvs, 1.0f); }
    return;
  }
  if (split > 1) {   // unscaled fp32 parts; sum_parts_kernel adds them up
    if (!exists) return;
    const int64_t poff = ((int64_t)chunk * prm.B * prm.H + bh) * prm.N * D;
#pragma unroll
    for (int db = 0; db < DBW; ++db)
#pragma unroll
      for (int i4 = 0; i4 < 4; ++i4) {
        const int64_t off = krow * D + 32 * (DBW * dh + db) + 8 * i4 + 4 * g;
        store_out4<BF16>(prm.part_dk + poff, off, true, dkacc[db][4 * i4], dkacc[db][4 * i4 + 1], dkacc[db][4 * i4 + 2],
                         dkacc[db][4 * i4 + 3]);
        store_out4<BF16>(prm.part_dv + poff, off, true, dvacc[db][4 * i4], dvacc[db][4 * i4 + 1], dvacc[db][4 * i4 + 2],
                         dvacc[db][4 * i4 + 3]);
      }
    return;
  }
  // the wavefront's 32 x 64 blocks of dK and dV leave through a stretch of the (now idle) tile stages and exchange area
  constexpr int OUT_BYTES = rows_out_bytes(32 * DBW, true);
  static_assert(4 * 2 * OUT_BYTES <= dkdv4_lds_bytes<D>(), "room for dK and dV of four wavefronts");
  __syncthreads();           // everybody has left the last step
  // (the lane index as a value the compiler cannot trace back: the per-lane addresses of the stores below would
  // otherwise be computed before the walk and held, or spilled, through it)
  int lane_out = lane;
  asm volatile("" : "+v"(lane_out));
  unsigned char* mine = lds + wv * 2 * OUT_BYTES;
  const int64_t r0 = (int64_t)n * 64 + 32 * kh;
  const float sc = prm.sm_scale;
  const int rows_here = TAIL ? prm.N - (int)r0 : 32;
  rows_out<BF16, 32 * DBW>(mine, prm.dk, b * prm.dks[0] + h * prm.dks[1] + r0 * prm.dks[2] + 32 * DBW * dh, prm.dks[2],
                           prm.out_f32, lane_out, rows_here, [&](int db, int i) { return dkacc[db][i] * sc; });
  rows_out<BF16, 32 * DBW>(mine + OUT_BYTES, prm.dv, b * prm.dvs[0] + h * prm.dvs[1] + r0 * prm.dvs[2] + 32 * DBW * dh, prm.dvs[2],
                           prm.out_f32, lane_out, rows_here, [&](int db, int i) { return dvacc[db][i]; });
}

// ---------------------------------------------------------------------------------------
// split > 1: out = scale * sum of the fp32 parts, rounded to the result type.  blockIdx.y: 0 dQ, 1 dK, 2 dV.  A workgroup
// takes 256 quads (4 consecutive values); where lists that are not shared are written already (whole >= 0) a quarter of a
// list's rows, most of which it leaves at once (D = 128, 16 heads N = 2176, keep 0.3, the whole backward: 256 quads 93 us,
// a quarter 88, a list 87; 8 heads N = 4096 dense 276 / 276 / 285).
// ---------------------------------------------------------------------------------------
constexpr int SUM_ROWS = 16;
template <bool BF16>
__global__ __launch_bounds__(256) void sum_parts_kernel(const BwdParams prm, int64_t quads, int D) {
  const int what = blockIdx.y + prm.first_sum;
  const int qpr = D / 4;                                   // quads per row
  int64_t first = (int64_t)blockIdx.x * 256, last = quads < first + 256 ? quads : first + 256;
  if (prm.whole >= 0) {
    const int list = blockIdx.x / (64 / SUM_ROWS), unit = list / prm.nb, blk = list - unit * prm.nb;
    const int b = unit / prm.H, h = unit - b * prm.H, mh = (prm.Bm > 1 ? b : 0) * prm.Hm + (prm.Hm > 1 ? h : 0);
    const cint_ptr_t lp = (cint_ptr_t)(uintptr_t)((what == 0 ? prm.row_ptr : prm.col_ptr) + (int64_t)mh * prm.nb);
    if (lp[blk + 1] - lp[blk] <= prm.whole) return;
    const int row0 = 64 * blk + SUM_ROWS * (blockIdx.x % (64 / SUM_ROWS)), rows = prm.N - row0 < SUM_ROWS ? prm.N - row0 : SUM_ROWS;
    first = ((int64_t)unit * prm.N + row0) * qpr;
    last = first + rows * qpr;
  }
  const float* part = what == 0 ? prm.part_dq : (what == 1 ? prm.part_dk : prm.part_dv);
  void* out = what == 0 ? prm.dq : (what == 1 ? prm.dk : prm.dv);
  const int64_t* st = what == 0 ? prm.dqs : (what == 1 ? prm.dks : prm.dvs);
  const float scale = what == 2 ? 1.0f : prm.sm_scale;
#pragma unroll 2
  for (int64_t i = first + threadIdx.x; i < last; i += 256) {
    floatx4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int c = 0; c < prm.split; ++c) acc += reinterpret_cast<const floatx4*>(part)[c * quads + i];
    // the parts are [B*H][N][D] without gaps; the result has its own strides
    const int64_t row_all = i / qpr;
    const int col = (int)(i - row_all * qpr) * 4;
    const int bh = (int)(row_all / prm.N), row = (int)(row_all - (int64_t)bh * prm.N);
    const int b = bh / prm.H, h = bh - b * prm.H;
    store_out4<BF16>(out, b * st[0] + h * st[1] + row * st[2] + col, prm.out_f32, acc[0] * scale, acc[1] * scale,
                     acc[2] * scale, acc[3] * scale);
  }
}

// ---------------------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------------------
// Workgroups per row / column list.  A single long head would otherwise walk its lists on a fraction of the GPU; every
// further share costs a write and a read of fp32 parts of dQ, dK and dV and, once, the launch that adds them up.
// us of a backward, N(0,1) bf16, 1 / 2 / 3 / 4 / 6 / 8 shares (256 compute units):
//   D = 64    8 heads N = 4096, keep 0.3    88 /  78 /  87 /  90 / 101 / 115     block-causal  149 / 123 / 109 / 115 / 122 / 135
//             8 heads N = 777,  keep 0.6    35 /  31 /  33 /  32 /  34 /  38
//             2 heads N = 1000, causal 0.8  38 /  28 /  29 /  26 /  26 /  28
//   D = 128   8 heads N = 4096, keep 0.3   119 / 131 / 148 / 160 / 217 / 264     block-causal  197 / 184 / 189 / 199 / 249 / 297
//            16 heads N = 1500, keep 0.3    58 /  77 /  90 / 101 / 131 / 179
//             2 heads N = 4096, keep 0.25   79 /  65 /  59 /  60 /  68 /  71     block-causal  178 / 116 /  99 /  93 /  92 /  90
//             4 heads N = 8192, keep 0.2   150 / 169 / 173 / 188 / 240 / 288     block-causal  386 / 334 / 333 / 333 / 366 / 410
//   D = 256   8 heads N = 4000, window     174 / 251 / 305 / 363 / 472 / 578     token-causal  402 / 404 / 480 / 514 / 618 / 715
//            16 heads N = 1500, keep 0.3   113 / 151 / 189 / 233 / 325 / 399
//             2 heads N = 4096, keep 0.25  140 / 101 / 107 / 103 / 127 / 146     block-causal  322 / 191 / 170 / 161 / 181 / 195
//             8 heads N = 777,  keep 0.6    76 /  69 /  77 /  74 /  93 / 110
// D = 64 fills four workgroups per compute unit.  The larger head dimensions have one or two in dkdv4_kernel and parts two
// and four times as large: two per compute unit, rounded to the nearest, but at D = 128 four where rows are long (the
// imbalance of a causal mask then weighs more than the parts).  A share keeps at least 8 tiles of a dense list; 5 in a
// launch of few short lists (at D = 128 that was slower), where the walk's latency is all, except that lists of 16 or 17
// tiles keep two shares (8 heads N = 1024: 35 with two, 39 with three) and shorter ones one from 112 lists on (12 heads
// N = 640, keep 0.3: 24 with one, 28 with two).
// At D = 128, block masks with about one to two lists per compute unit: the longest lists of a causal mask are what a launch
// takes, and the shares of a sparse mask's cost more than they give.  So only lists longer than a share of a dense list are
// shared there (`whole`).  One share for all / as many as here for all / this:
//             4 heads N = 4096, keep 0.3    86 /  92 /  86     block-causal  183 / 132 / 122     dense  185 / 164 / 164
//             6 heads N = 4096             108 / 120 / 111                   192 / 167 / 160            260 / 225 / 226
//             8 heads N = 4096             113 / 136 / 119                   199 / 195 / 187            280 / 274 / 276
//            16 heads N = 2176              86 / 109 /  88                   144 / 138 / 125            195 / 208 / 206
//            12 heads N = 2048              70 /  84 /  73                   135 / 117 / 105            138 / 134 / 134
//            14 heads N = 1792              60 /  -  /  68                   105 /  -  /  92            121 /  -  / 135   (one share there)
// (Elementwise masks, 8 heads N = 4000, a training step: window of 1000 135 / 156 / 140, of 2000 212 / 218 / 226,
// token-causal 316 / 291 / 287: one share from 1.33 lists per compute unit on.)
// (D = 64: what bwd_short_kernel does not take, D = 128: what two groups do not; the workspace has room for these shares all the same.)
struct BwdShares { int split, whole; };
static BwdShares bwd_shares(int B, int H, int N, int D, bool elementwise) {
  const int64_t lists = (int64_t)B * H * ((N + 63) / 64), cus = compute_units();
  const int nb = (N + 63) / 64;
  if (D == 128 && !elementwise && nb < 96 && 3 * lists >= 2 * cus && 4 * lists <= 9 * cus) {
    const int split = 4 * lists <= 5 * cus ? 3 : 2;
    if (nb > (split == 2 ? 28 : 24)) return {split, nb / split};
  }
  int64_t s;
  if (D == 64 || (D == 128 && nb >= 96)) s = (4 * cus + lists - 1) / lists;
  else s = (2 * cus + lists / 2) / lists;
  int cap = nb / 8;
  if (D != 128 && nb <= 32 && 2 * lists <= cus && (nb >= 18 || (nb < 16 && 16 * lists <= 7 * cus))) cap = nb / 5;
  if (s > cap) s = cap;
  return {(int)(s > 8 ? 8 : s < 1 ? 1 : s), -1};
}

// Which launches bwd_short_kernel (D = 64) takes: pairs of wavefronts per workgroup (0: none) and shares of a list.  us of a backward,
// the two kernels with their shares and sums / 2 pairs / 4 pairs / 2 pairs, 2 shares / 4 pairs, 2 shares; fp16, keep 0.1, 0.3, 1, causal:
//    4 heads N = 512 (32 lists)     15 /  9 / 10 / 11 / 14     18 /  9 / 10 / 12 / 13     26 / 13 / 12 / 13 / 14     25 / 13 / 12 / 13 / 13
//    1 head  N = 3072 (48)          23 / 15 / 14 /  - / 14     28 / 24 / 21 /  - / 18     44 / 46 / 38 /  - / 28     36 / 46 / 37 /  - / 26
//    8 heads N = 1024 (128)         23 / 11 / 11 / 20 / 24     29 / 15 / 14 / 22 / 26     36 / 22 / 19 / 26 / 30     35 / 21 / 18 / 25 / 28
//    1 head  N = 8192 (128)         40 / 30 / 25 / 28 / 31     56 / 52 / 43 / 41 / 46     95 /128 /100 / 89 / 92     82 /118 / 91 / 78 / 72
//    8 heads N = 2048 (256)         38 / 16 / 21 / 29 / 39     43 / 21 / 25 / 34 / 44     65 / 46 / 51 / 58 / 68     57 / 40 / 35 / 42 / 51
//    2 heads N = 8192 (256)         50 / 35 / 36 / 41 / 53     76 / 63 / 67 / 72 / 82    162 /158 /160 /163 /174    134 /135 / 99 /106 /109
//    1 head  N = 17536 (274)        76 / 56 / 62 / 60 /  -    159 /137 /140 /130 /  -    427 /403 /425 /373 /  -    253 /276 /227 /212 /  -    (bf16)
//    4 heads N = 8192 (512)         68 / 53 / 65 / 71         121 /111 /123 /126         295 /302 /314 /316         237 /159 /175 /190
//   14 heads N = 4096 (896)         79 / 55 / 76              133 /103 /129              283 /269 /298              188 /153 /174
//   16 heads N = 4096 (1024)        55 / 60 / 85              121 /119 /146              279 /303 /334              197 /171 /191    (bf16; not there)
//    8 heads N = 12032 (1504)      167 /156 /204              437 /407 /449             1303/1274/1343              641 /644 /699    (bf16)
//    2 heads N = 32000 (1000)      266 /258 /286              680 /711 /750             2070/2239/2320             1073/1116/1168    (bf16; not there)
struct BwdShort { int pairs, split; };
static BwdShort bwd_short(int64_t lists_, int nb) {
  const int64_t lists = lists_ * 256 / compute_units();        // (as if there were 256 compute units)
  if (nb > BWD_SHORT_MAX_BLOCKS) return {0, 1};
  if (lists <= 128) return {4, nb >= 90 || (lists <= 64 && nb >= 48) ? 2 : 1};
  if (lists <= 288 && nb >= 150) return {2, 2};
  if (lists <= 256 && nb >= 64) return {4, 1};
  const int64_t most = nb > 300 ? 640 : nb > 128 ? 1536 : 1023;
  return {lists <= most ? 2 : 0, 1};
}

// D = 128, few lists: dq_pairs_kernel with `dq_pairs` pairs of wavefronts per row block (0: dq_kernel), dkdv4_kernel with `groups`
// groups of wavefronts per column block.  Two groups have the compute unit that two shares of a list would have, but add up in LDS: no
// parts, no launch that adds them up.  `split`: the shares there would be (1: nothing to merge, one group).
// us of a backward, bf16, as before / 2 pairs for dQ / 2 pairs, 2 groups / 4 pairs, 2 groups; keep 0.1, 0.3, 1, causal:
//   12 heads N = 768  (144 lists)     22 / 22 / 23 / 24     30 / 28 / 29 / 30      43 / 38 / 37 / 37      43 / 38 / 37 / 37
//    4 heads N = 1024 (64)            26 / 27 / 23 / 25     33 / 35 / 31 / 33      42 / 44 / 43 / 42      39 / 41 / 42 / 41
//   16 heads N = 1024 (256)           43 / 38 / 25 / 26     52 / 47 / 33 / 34      67 / 61 / 47 / 47      64 / 57 / 44 / 44
//    3 heads N = 2048 (96)            37 / 37 / 28 / 29     42 / 44 / 37 / 37      62 / 69 / 70 / 66      55 / 64 / 69 / 65     (not there)
//    8 heads N = 2048 (256)           35 / 32 / 30 / 32     54 / 51 / 40 / 40     102 / 97 / 77 / 75      82 / 78 / 71 / 68
//   10 heads N = 2048 (320)           44 / 41 / 44 / 52     76 / 71 / 65 / 72     122 /124 /126 /138      96 /102 / 93 / 87     (not there)
//   14 heads N = 2048 (448)           48 / 46 / 47 / 54     79 / 69 / 70 / 76     154 /146 /130 /137     113 /112 / 97 / 93
//    2 heads N = 4096 (128)           46 / 46 / 39 / 39     61 / 68 / 66 / 62      98 /114 /125 /115      94 /109 /123 /113     (not there)
//    4 heads N = 4096 (256)           52 / 45 / 40 / 41     84 / 81 / 69 / 66     163 /157 /137 /131     125 /125 /125 /115
//    5 heads N = 4096 (320)           64 / 57 / 57 / 64    108 /100 /109 /116     199 /208 /230 /246     137 /142 /132 /121     (not there)
//    8 heads N = 4096 (512)           64 / 58 / 62 / 70    139 /125 /117 /125     277 /270 /251 /258     188 /175 /152 /145
//   10 heads N = 4096 (640)           68 / 72 / 77 / 88    145 /144 /142 /152     372 /370 /369 /375     240 /215 /234 /235     (dQ only)
//    2 heads N = 6144 (192)           77 / 72 / 51 / 50    104 /107 / 88 / 82     202 /203 /183 /169     140 /168 /178 /162     (not there)
//    4 heads N = 8192 (512)          112 /104 / 90 / 95    200 /192 /176 /186     508 /501 /482 /488     335 /303 /278 /260
//    6 heads N = 8192 (768)          152 /145 /125 /134    300 /294 /271 /274     815 /770 /747 /754     448 /419 /404 /420
//    1 head  N = 16384 (256)         107 /105 / 88 / 85    209 /216 /200 /189     525 /542 /521 /497     366 /413 /472 /428     (not there)
//    2 heads N = 16384 (512)         168 /161 /145 /155    361 /355 /348 /357    1002 /993 /977 /987     639 /584 /563 /520
//    8 heads N = 8192 (1024)         140 /147 /162 /177    336 /337 /343 /362     943 /944 /952 /970     558 /520 /509 /515     (not there)
// So: enough lists that nobody needs more than two streams of a long one, and not a bit more than one list per compute unit, which
// would be a second round of workgroups that fill it.  Token masks, 8 heads N = 4000: window of 1000 84 / 80 / 86 / 94, causal 301 / 263 / 242 / 236.
struct BwdPairs { int dq_pairs, groups; };
static BwdPairs bwd_pairs_128(int64_t lists_, int nb, int split) {
  const int64_t lists = lists_ * 256 / compute_units();        // (as if there were 256 compute units)
  if (nb < 12 || nb > BWD_SHORT_MAX_BLOCKS) return {0, 1};
  if (split > 1) {
    const int64_t least = nb <= 64 ? std::min(4 * nb, 192) : nb <= 128 ? 256 : 2 * nb, most = nb >= 96 && nb <= 128 ? 768 : 512;
    if (lists >= least && lists <= most && (nb < 32 || lists <= 256 || lists >= 384)) return {lists <= 256 && nb >= 32 ? 4 : 2, 2};
    if (lists <= most) return {0, 1};
  }
  return {lists <= 800 ? 2 : 0, 1};
}

// floats in front of the parts (the parts are accessed 16 bytes at a time)
static size_t delta_floats(int B, int H, int N) { return ((size_t)B * H * N + 63) & ~(size_t)63; }

size_t bwd_workspace_bytes(int B, int H, int N, int D) {
  const size_t delta = delta_floats(B, H, N) * sizeof(float);
  const int block = bwd_shares(B, H, N, D, false).split, words = bwd_shares(B, H, N, D, true).split;
  int split = block > words ? block : words;                 // one size for both kinds of masks
  if (const int nb = (N + 63) / 64; D == 64) split = std::max(split, bwd_short((int64_t)B * H * nb, nb).split);
  return delta + (split > 1 ? (size_t)3 * split * B * H * N * D * sizeof(float) : 0);   // + parts of dQ, dK, dV
}

template <bool BF16>
static void launch_sum_parts(const BwdParams& prm, int D, hipStream_t st) {
  const int BH = prm.B * prm.H;
  const int64_t quads = (int64_t)BH * prm.N * D / 4;
  const unsigned blocks = prm.whole >= 0 ? (unsigned)(BH * prm.nb * (64 / SUM_ROWS)) : (unsigned)((quads + 255) / 256);
  hipLaunchKernelGGL((sum_parts_kernel<BF16>), dim3(blocks, 3 - prm.first_sum), dim3(256), 0, st, prm, quads, D);
}

template <int D, bool BF16, bool EW, bool PB, bool TAIL>
static void launch_bwd_t(const BwdParams& prm, int groups, hipStream_t st) {
  using C = BwdCfg<D, EW>;
  constexpr int KB = D >= 128 ? 1 : 2;          // dq_kernel walks D >= 128 tiles in two halves (no gain at D = 64: two wavefronts per SIMD anyway)
  using CQ = BwdCfg<D, EW, 32 * KB>;
  // dkdv_kernel walks halves (191 instead of 318 registers: two wavefronts per SIMD; B*H = 32 N = 8192 dense block-causal
  // backward 1417 -> 1167 us)
  using CK = BwdCfg<D, EW, 32>;
  static std::atomic<unsigned long long> configured{0};   // raising the dynamic LDS limit is idempotent
  once_per_device(configured, [] {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&dq_kernel<D, BF16, EW, PB, KB, TAIL>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, CQ::LDS_BYTES);
    if constexpr (D == 64) {
      (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&dkdv_kernel<D, BF16, EW, PB, TAIL>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, CK::LDS_BYTES);
    } else {
      (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&dkdv4_kernel<D, BF16, PB, EW, TAIL>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, dkdv4_lds_bytes<D>());
      if constexpr (D == 128)
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&dkdv4_kernel<D, BF16, PB, EW, TAIL, 2>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, 2 * dkdv4_lds_bytes<D>());
    }
  });
  const int grid = prm.place.per_share * prm.split;
  if (prm.first_sum == 0) hipLaunchKernelGGL((dq_kernel<D, BF16, EW, PB, KB, TAIL>), dim3(grid), dim3(128), CQ::LDS_BYTES, st, prm);
  if constexpr (D == 128) {
    if (groups == 2) {
      hipLaunchKernelGGL((dkdv4_kernel<D, BF16, PB, EW, TAIL, 2>), dim3(grid), dim3(512), 2 * dkdv4_lds_bytes<D>(), st, prm);
      return;                                   // (one share of a list)
    }
  }
  if constexpr (D == 64) hipLaunchKernelGGL((dkdv_kernel<D, BF16, EW, PB, TAIL>), dim3(grid), dim3(128), CK::LDS_BYTES, st, prm);
  else hipLaunchKernelGGL((dkdv4_kernel<D, BF16, PB, EW, TAIL>), dim3(grid), dim3(256), dkdv4_lds_bytes<D>(), st, prm);
  if (prm.split > 1) launch_sum_parts<BF16>(prm, D, st);
}

void launch_bwd_short(const BwdParams& prm, int pairs, bool bf16, bool pb, hipStream_t st);   // attn_bwd_short.hip
void launch_dq_pairs(const BwdParams& prm, int pairs, bool bf16, bool pb, hipStream_t st);

int launch_bwd(const void* q, const void* k, const void* v, const void* o, const void* d_o,
               const float* lse, void* dq, void* dk, void* dv, const int32_t* row_ptr,
               const int32_t* col_idx, const int32_t* col_ptr, const int32_t* row_idx,
               const uint64_t* bits_rows, const uint64_t* bits_cols,
               const AttnShape& s, void* ws, hipStream_t st) {
  BwdParams prm;
  prm.q = q; prm.k = k; prm.v = v; prm.o = o; prm.d_o = d_o; prm.lse = lse; prm.delta = (float*)ws;
  prm.dq = dq; prm.dk = dk; prm.dv = dv;
  prm.row_ptr = row_ptr; prm.col_idx = col_idx; prm.col_ptr = col_ptr; prm.row_idx = row_idx;
  prm.bits_rows = (const unsigned long long*)bits_rows; prm.bits_cols = (const unsigned long long*)bits_cols;
  prm.B = s.B; prm.H = s.H; prm.N = s.N; prm.nb = (s.N + 63) / 64; prm.Bm = s.Bm; prm.Hm = s.Hm;
  prm.out_f32 = s.out_dtype == BSATTN_F32;
  const BwdShares shares = bwd_shares(s.B, s.H, s.N, s.D, bits_rows != nullptr);
  const BwdShort plan = s.D == 64 ? bwd_short((int64_t)s.B * s.H * prm.nb, prm.nb) : BwdShort{0, 1};
  const BwdPairs pairs = s.D == 128 ? bwd_pairs_128((int64_t)s.B * s.H * prm.nb, prm.nb, shares.split) : BwdPairs{0, 1};
  prm.split = plan.pairs > 0 ? plan.split : pairs.groups > 1 ? 1 : shares.split;
  prm.whole = plan.pairs > 0 || pairs.groups > 1 ? -1 : shares.whole;
  const Groups group = groups_of_heads(s.B * s.H, s.N, s.D);
  prm.place = place_of_eight(s.B * s.H, prm.nb, plan.pairs > 0 ? 2 * prm.split : prm.split, group);
  prm.place_dq = place_of_eight(s.B * s.H, prm.nb, 1, group);
  prm.first_sum = pairs.dq_pairs > 0 ? 1 : 0;
  prm.per_batch = divisor((unsigned)s.H, (uint64_t)s.B * s.H);
  {
    const size_t one = (size_t)prm.split * s.B * s.H * s.N * s.D;
    prm.part_dq = (float*)ws + delta_floats(s.B, s.H, s.N);
    prm.part_dk = prm.part_dq + one;
    prm.part_dv = prm.part_dk + one;
  }
  prm.sm_scale = s.sm_scale;
  prm.qk_scale = s.sm_scale * kLog2e;
  for (int i = 0; i < 3; ++i) {
    prm.qs[i] = s.qs[i]; prm.ks[i] = s.ks[i]; prm.vs[i] = s.vs[i]; prm.os[i] = s.os[i]; prm.dos[i] = s.dos[i];
    prm.dqs[i] = s.dqs[i]; prm.dks[i] = s.dks[i]; prm.dvs[i] = s.dvs[i];
  }
  const bool bf = s.dtype == BSATTN_BF16;
  // bf16 gradients are rounded to 8 bits anyway: P and dS are then rounded to bf16 as well (what the
  // reference's forward does with P, fa2_fwd.py:189) and no tile needs converting; fp32 gradients of
  // bf16 inputs keep P and dS in fp16.
  const bool pb = bf && !prm.out_f32;
  const bool ew = bits_rows != nullptr;
  if (plan.pairs > 0) {
    launch_bwd_short(prm, plan.pairs, bf, pb, st);
    if (prm.split > 1) { if (bf) launch_sum_parts<true>(prm, s.D, st); else launch_sum_parts<false>(prm, s.D, st); }
    return launch_status();
  }
  if (pairs.dq_pairs > 0) launch_dq_pairs(prm, pairs.dq_pairs, bf, pb, st);
  auto pick = [&](auto dc, auto tail) {
    constexpr int DD = decltype(dc)::value;
    constexpr bool TL = decltype(tail)::value;
    if (!ew) {
      if (!bf) launch_bwd_t<DD, false, false, false, TL>(prm, pairs.groups, st);
      else if (pb) launch_bwd_t<DD, true, false, true, TL>(prm, pairs.groups, st);
      else launch_bwd_t<DD, true, false, false, TL>(prm, pairs.groups, st);
    } else {   // elementwise mask
      if (!bf) launch_bwd_t<DD, false, true, false, TL>(prm, pairs.groups, st);
      else if (pb) launch_bwd_t<DD, true, true, true, TL>(prm, pairs.groups, st);
      else launch_bwd_t<DD, true, true, false, TL>(prm, pairs.groups, st);
    }
  };
  auto pick_tail = [&](auto dc) {
    if (s.N % 64 == 0) pick(dc, std::false_type{});
    else pick(dc, std::true_type{});
  };
  if (s.D == 64) pick_tail(std::integral_constant<int, 64>{});
  else if (s.D == 128) pick_tail(std::integral_constant<int, 128>{});
  else pick_tail(std::integral_constant<int, 256>{});
  return launch_status();
}

}  // namespace bsattn
