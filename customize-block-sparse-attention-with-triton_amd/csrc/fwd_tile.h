// Pieces shared by the forward kernels: launch parameters, the softmax of one tile, the rare
// re-centring path.
#pragma once
#include "common.h"
#include "kernel_util.h"
#include "own_rows.h"
#include "place.h"
#include "quad_shares.h"

namespace bsattn {

constexpr int MASK_MAX_BLOCKS = 512;    // ... up to which a kernel takes the columns of a row block from the block mask
constexpr int SHORT_MAX_BLOCKS = 128;   // row blocks of a head up to which fwd_short_kernel takes a launch

struct FwdParams {
  const void* q; const void* k; const void* v; void* o; float* lse;
  const int32_t* row_ptr; const int32_t* col_idx;
  const unsigned char* mask;       // the block mask itself in place of the lists (kernels whose workgroups have a row block each), or null
  int64_t ms[4];                   // its strides
  unsigned char* mask_copy;        // the mask as this launch saw it, [Bm][Hm][nb][nb] of 0 and 1, or null (columns_of_row)
  const unsigned char* tile_partial;        // elementwise masks: per kept tile, 1 = only partly set
  const unsigned long long* tile_bits;      // ... and its 64 row words (bit c = column c)
  float* ws;                       // partial slots of row blocks shared between workgroups (two per workgroup)
  unsigned long long* flags;       // one per row block: parts counted in so far, tagged with `epoch`
  unsigned long long epoch;        // distinguishes this launch's counters from stale contents
  int deterministic;               // tiles go to the wavefronts of a workgroup in a fixed pattern
  int split;                       // pair and short kernel: workgroups per row block (1: results written directly)
  int share_shift;                 // short kernel, split > 1: a share has at least 2^share_shift tiles
  // split > 1: unnormalised fp32 O parts and their (m, l).  Pair kernel: [split][B*H][N][D] and [split][B*H][N][2], and the length of every
  // row block's list [B*H][nb]; short kernel: [B*H][nb][split][64][D] and [B*H][nb][split][64][2]
  float* part_o; float* part_ml;
  int* part_len;
  int B, H, N, nb, Bm, Hm, W;   // W: workgroups per head (ROWS: those for long row blocks)
  int first_ids;                // workgroups with a linear id below this are the first on their compute unit (ROWS: fill the GPU)
  int place_fast, place_quot, place_rest;   // SPREAD: place_range's arguments
  int group;                    // ROWS: heads whose row blocks go out together
  int out_f32;
  float qk_scale;  // sm_scale * log2(e)
  int64_t qs[3], ks[3], vs[3], os[3];
  PlaceOfEight place;              // kernels whose workgroups have a row block each
  Divisor per_batch;               // H
};

constexpr int QUAD_MAX_BLOCKS = 1024;      // row blocks of a head that fwd_quad_kernel takes, at most

// fwd_quad_kernel's and fwd_wide_kernel's: what quad_shares asks for, and
struct FwdShareParams : FwdParams {
  int tail_from, tail_shares, tail_len, load, most, share_least;
  int exact;      // hundredths of a tile whose numerators have no rounding error, of a row, at least
};

// fwd_kernel's
struct FwdRangeParams : FwdParams {
  // fwd_kernel: which range of its head workgroup wg takes, for heads with at least perm_min_tiles kept tiles that
  // are cut into exactly perm_n ranges, the first perm_fast of them with the larger weight (perm_n = 0: none; see
  // range_permutation)
  int perm_n, perm_fast, perm_min_tiles;
  OwnLines own;                    // fwd_kernel, ranges of workgroups: heads that go a row block to a workgroup
  unsigned short perm[512];        // (RANGE_PERM_MAX of range_perm.h)
  unsigned short perm_causal[512]; // the same for heads whose mask is the dense block-causal one
};

// P = exp2(score - m) for the 2 x 16 scores one lane holds of one query (key blocks s0, s1),
// rounded to fp16 and packed as the operand fragments pf[0..3][qb] of the second product.
// Returns l + the row sum of the rounded P over this lane's keys.  With FOLD the scores
// already are "scaled score - m".  PB: P is rounded to bf16 instead of fp16.
template <bool FOLD, bool PB = false>
__device__ __forceinline__ float softmax_tile(const floatx16& s0, const floatx16& s1, float qk_scale, float m,
                                              float l, uintx4 (&pf)[4][2], int qb) {
#pragma unroll
  for (int ts = 0; ts < 4; ++ts) {
#pragma unroll
    for (int jj = 0; jj < 4; ++jj) {
      const int i = 8 * (ts & 1) + 2 * jj;
      const float x0 = ts < 2 ? s0[i] : s1[i], x1 = ts < 2 ? s0[i + 1] : s1[i + 1];
      const float p0 = __builtin_amdgcn_exp2f(FOLD ? x0 : __builtin_fmaf(x0, qk_scale, -m));
      const float p1 = __builtin_amdgcn_exp2f(FOLD ? x1 : __builtin_fmaf(x1, qk_scale, -m));
      const unsigned int hp = pack2<PB>(p0, p1);
      l = add_packed2<PB>(hp, l);
      pf[ts][qb][jj] = hp;
    }
  }
  return l;
}

// The same for one block of 32 keys.
template <bool FOLD, bool PB>
__device__ __forceinline__ float softmax_block(const floatx16& s, float qk_scale, float m, float l, uintx4 (&pf)[2]) {
#pragma unroll
  for (int ts = 0; ts < 2; ++ts) {
#pragma unroll
    for (int jj = 0; jj < 4; ++jj) {
      const int i = 8 * ts + 2 * jj;
      const float p0 = __builtin_amdgcn_exp2f(FOLD ? s[i] : __builtin_fmaf(s[i], qk_scale, -m));
      const float p1 = __builtin_amdgcn_exp2f(FOLD ? s[i + 1] : __builtin_fmaf(s[i + 1], qk_scale, -m));
      const unsigned int hp = pack2<PB>(p0, p1);
      l = add_packed2<PB>(hp, l);
      pf[ts][jj] = hp;
    }
  }
  return l;
}

// The same in two parts of 16 bits, pf and rest, which the second product takes one after the other: numerators to 22 bits (PB: 16).  For the
// first block of a list: what the rounding of P costs a row falls by that block's share of it, more than half for the short lists that weigh
// most in a result's norm.  pf is cut and not rounded and rest is never 0 where the numerator is not, so that a value of V
// that is not finite counts with one sign in both.
template <bool FOLD, bool PB>
__device__ __forceinline__ float softmax_block_parts(floatx16& s, float qk_scale, float m, float l, uintx4 (&pf)[2], uintx4 (&rest)[2]) {
  constexpr float LEAST = 0x1p-24f;       // smallest fp16
  if constexpr (FOLD) asm volatile("" : "+v"(s));      // (or the exponentials of softmax_block in front of it are kept for here, in 16 registers)
  else asm volatile("" : "+v"(m));
#pragma unroll
  for (int ts = 0; ts < 2; ++ts) {
#pragma unroll
    for (int jj = 0; jj < 4; ++jj) {
      const int i = 8 * ts + 2 * jj;
      const float p0 = __builtin_amdgcn_exp2f(FOLD ? s[i] : __builtin_fmaf(s[i], qk_scale, -m));
      const float p1 = __builtin_amdgcn_exp2f(FOLD ? s[i + 1] : __builtin_fmaf(s[i + 1], qk_scale, -m));
      unsigned int hp;
      float h0, h1;
      if constexpr (PB) {
        const unsigned int b0 = __builtin_bit_cast(unsigned int, p0), b1 = __builtin_bit_cast(unsigned int, p1) & 0xffff0000u;
        hp = b1 | (b0 >> 16);
        h0 = __builtin_bit_cast(float, b0 & 0xffff0000u);
        h1 = __builtin_bit_cast(float, b1);
      } else {
        hp = __builtin_bit_cast(unsigned int, __builtin_amdgcn_cvt_pkrtz(p0, p1));
        const half2v h = __builtin_bit_cast(half2v, hp);
        h0 = (float)h[0]; h1 = (float)h[1];
      }
      const unsigned int lp = pack2<PB>(__builtin_amdgcn_fmed3f(p0 - h0, LEAST, p0), __builtin_amdgcn_fmed3f(p1 - h1, LEAST, p1));
      l = add_packed2<PB>(lp, add_packed2<PB>(hp, l));
      pf[ts][jj] = hp;
      rest[ts][jj] = lp;
    }
  }
  return l;
}

// The kept columns of row block m, ascending, from the block mask into cols (LDS), by every wavefront of the workgroup by
// itself (all write the same): no list kernels in front of the launch, and one dependent access instead of two (row
// pointer, then column).  Returns their number, at most nb <= MAX.
// writer: the one wavefront of the head's workgroups for this row block that also writes mask_copy, if the heads that share the
// row have it written by the first of them (a store per 64 columns, against 5 us for a launch that copies the mask).
template <int MAX>
__device__ __forceinline__ int columns_of_row(const FwdParams& prm, int b, int h, int m, int lane, int* cols, bool writer) {
  const int mb = prm.Bm > 1 ? b : 0, mhd = prm.Hm > 1 ? h : 0;
  unsigned char* copy = writer && prm.mask_copy != nullptr && mb == b && mhd == h ? prm.mask_copy + ((int64_t)(mb * prm.Hm + mhd) * prm.nb + m) * prm.nb : nullptr;
  const unsigned char* row = prm.mask + (prm.Bm > 1 ? b : 0) * prm.ms[0] + (prm.Hm > 1 ? h : 0) * prm.ms[1] + m * prm.ms[2];
  constexpr int AHEAD = MAX < 256 ? MAX / 64 : 4;      // accesses on their way at once
  int n = 0;
  for (int c0 = 0; c0 < prm.nb; c0 += 64 * AHEAD) {
    bool keep[AHEAD];
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) {
      const int c = c0 + 64 * i + lane;
      keep[i] = c < prm.nb && row[(int64_t)c * prm.ms[3]] != 0;
    }
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) {
      const unsigned long long bal = __ballot(keep[i]);
      if (keep[i]) cols[n + __popcll(bal & ((1ull << lane) - 1ull))] = c0 + 64 * i + lane;
      if (copy != nullptr && c0 + 64 * i + lane < prm.nb) copy[c0 + 64 * i + lane] = keep[i];
      n += __popcll(bal);
    }
  }
  __builtin_amdgcn_wave_barrier();
  return n;
}

// The kept tiles of SHARE_SAMPLE rows of the block mask, from row m on.
__device__ __forceinline__ int length_of_rows(const FwdParams& prm, int b, int h, int m, int lane) {
  const unsigned char* row = prm.mask + (prm.Bm > 1 ? b : 0) * prm.ms[0] + (prm.Hm > 1 ? h : 0) * prm.ms[1] + m * prm.ms[2];
  int n = 0;
  for (int c = lane; c < prm.nb; c += 64)
#pragma unroll
    for (int i = 0; i < SHARE_SAMPLE; ++i) n += row[i * prm.ms[2] + (int64_t)c * prm.ms[3]] != 0;
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) n += __shfl_xor(n, d);
  return __builtin_amdgcn_readfirstlane(n);
}

// Shares of the list of len tiles of the row block of workgroup `linear` (of the workgroups that come first on their lists).
__device__ __forceinline__ int shares_of_list(const FwdShareParams& prm, cint_ptr_t rp, int b, int h, int len, int linear, bool listed, int lane) {
  if (len < 2 * prm.share_least) return 1;
  const int tail = linear >= prm.tail_from && len >= prm.tail_len ? prm.tail_shares : 1;
  int mid = 0, end = 0;
  if (tail < prm.most) {
    const int nb = prm.nb;
    if (listed) { mid = rp[nb / 2 + SHARE_SAMPLE / 2] - rp[nb / 2 - SHARE_SAMPLE / 2]; end = rp[nb] - rp[nb - SHARE_SAMPLE]; }
    else { mid = length_of_rows(prm, b, h, nb / 2 - SHARE_SAMPLE / 2, lane); end = length_of_rows(prm, b, h, nb - SHARE_SAMPLE, lane); }
  }
  return quad_shares(len, mid, end, tail, prm.load, prm.most, prm.share_least);
}

// Tiles at the front of a walk whose numerators are kept in two parts (softmax_block_parts), for a list that `walks` of them take on: without
// any the largest numerator of a walk is exact, which counts 48 hundredths (FOLD: the reference stays at 0, and none is).
template <bool FOLD>
constexpr int first_tiles(int exact, int walks) { return exact <= (FOLD ? 0 : 48) * walks ? 0 : exact <= 100 * walks ? 1 : 2; }

// Counts a share of a list in, by one thread, when all accesses of its workgroup to its part have been acknowledged; returns how many
// are in.  The counter holds (launch mark << 16 | shares counted); stale contents carry another mark.  seen: a first guess of it.
__device__ __forceinline__ int count_in(unsigned long long* arrivals, unsigned long long epoch, unsigned long long seen) {
  for (;;) {     // (ends: the counter only changes when another share is counted, at most as often as the list has shares)
    const unsigned long long want = (seen >> 16) == epoch ? seen + 1 : ((epoch << 16) | 1ull);
    if (__hip_atomic_compare_exchange_strong(arrivals, &seen, want, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
      return (int)(want & 0xffffull);
  }
}

__device__ __forceinline__ void* out_base(const FwdParams& prm, int b, int h) {
  const int64_t off = b * prm.os[0] + h * prm.os[1];
  return prm.out_f32 ? (void*)((float*)prm.o + off) : (void*)((unsigned short*)prm.o + off);
}

// Natural logarithm of the sum of exponentials of a row with reference exponent m and sum l of its numerators: -inf
// for a row without mass (l = 0: no key, or no score above -inf), NaN where a score is not a number.  (The largest of the references of
// several parts leaves out those that are not numbers, and may be -inf then: the sum says what the row is.)
__device__ __forceinline__ float row_lse(float m, float l) {
  return l == 0.f ? -INFINITY : (m + __builtin_amdgcn_logf(l)) * 0.6931471805599453f;
}

// 1 / l for a row with at least one kept tile.  Elementwise masks (EW) may leave a query without a key, whose row of O is 0; with a
// block mask a sum of 0 says that all scores are -inf, and 0 times infinity gives what softmax gives there: not a number.
template <bool EW>
__device__ __forceinline__ float row_inverse(float l) { return EW && !(l > 0.f) ? 0.f : 1.0f / l; }

// Which queries of the wavefront have no mass yet: bit q (and q + 32, its other lane) is set if both lanes' sums are 0.
__device__ __forceinline__ unsigned long long no_mass(float l) {
  const unsigned long long zero = __ballot(l == 0.f);
  return zero & (zero >> 32 | zero << 32);
}

// A lane whose sum grows by this in a tile calls for a new reference exponent: some P left the safe fp16 range.
constexpr float SUM_LIMIT = 16384.0f;
// The limit after a tile that got one: 0, which every tile reaches, while some query has no mass.  (EW: the lanes look at their sums.)
template <bool EW>
__device__ __forceinline__ float sum_limit(float l) {
  if constexpr (EW) return SUM_LIMIT;
  return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(no_mass(l) != 0ull ? 0 : __builtin_bit_cast(int, SUM_LIMIT)));
}

// Rare path of the softmax: re-centre the reference exponent of one query block on the row
// maximum of the current tile and redo the tile's numerators.
// A query may have had nothing but masked keys (EW) or scores of -inf so far (l == 0, or the whole tile: maximum -inf, which is no
// reference: -inf less -inf is not a number).  Such a lane takes the first finite maximum as its reference; until every query has
// one, block masks' kernels come here in each tile (sum_limit), as with EW they do for every lane whose own sum is 0.
// recentre_on: the reference, l and the accumulators, from the lane's maximum; returns what the scores are to be lowered by (FOLD).
template <int DB, int NQ, bool FOLD, bool EW>
__device__ __forceinline__ float recentre_on(float mx, floatx16 (&oacc)[DB][NQ], int qb, float qk_scale, float& m, float& l,
                                             uintx4& mfrag, bool fresh, int g) {
  mx = xhalf_max(mx);
  // exponent of the largest entry relative to the current reference
  const float smax = FOLD ? mx : __builtin_fmaf(mx, qk_scale, -m);
  // (a query's keys are split over two lanes, which must keep one common reference: the mass is
  // the sum of both halves, or a lane whose own keys were all masked would drift away)
  const bool nomass = (EW && fresh) || __builtin_amdgcn_inverse_ballot_w64(no_mass(l));
  float delta = nomass ? smax : fmaxf(smax, 0.f);
  if (smax == -INFINITY) delta = 0.f;
  m += delta;
  if (EW ? !fresh : __any(!nomass)) {
    const float alpha = nomass ? 1.0f : __builtin_amdgcn_exp2f(-delta);
    l *= alpha;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int i = 0; i < 16; ++i) oacc[db][qb][i] *= alpha;
  }
  if constexpr (FOLD) {
    const _Float16 hi = (_Float16)(-m);
    const _Float16 lo = (_Float16)(-m - (float)hi);
    const half2v hl = {hi, lo};
    mfrag[0] = g == 0 ? __builtin_bit_cast(unsigned int, hl) : 0u;
  }
  return delta;
}

template <int DB, bool FOLD, bool EW>
__device__ __forceinline__ void recentre(floatx16& s0, floatx16& s1, floatx16 (&oacc)[DB][2], int qb, float qk_scale,
                                      float& m, float& l, uintx4& mfrag, bool fresh, int g) {
  float mx = max3f(s0[0], s0[1], s0[2]);
#pragma unroll
  for (int i = 3; i < 15; i += 2) mx = max3f(mx, s0[i], s0[i + 1]);
  mx = max3f(mx, s0[15], s1[0]);
#pragma unroll
  for (int i = 1; i < 15; i += 2) mx = max3f(mx, s1[i], s1[i + 1]);
  const float delta = recentre_on<DB, 2, FOLD, EW>(fmaxf(mx, s1[15]), oacc, qb, qk_scale, m, l, mfrag, fresh, g);
  if constexpr (FOLD) {
#pragma unroll
    for (int i = 0; i < 16; ++i) { s0[i] -= delta; s1[i] -= delta; }
  }
}

// The same for one block of 32 keys.
template <int DB, bool FOLD>
__device__ __forceinline__ void recentre_block(floatx16& s, floatx16 (&oacc)[DB][1], float qk_scale, float& m, float& l,
                                               uintx4& mfrag, bool fresh, int g) {
  float mx = max3f(s[0], s[1], s[2]);
#pragma unroll
  for (int i = 3; i < 15; i += 2) mx = max3f(mx, s[i], s[i + 1]);
  const float delta = recentre_on<DB, 1, FOLD, false>(fmaxf(mx, s[15]), oacc, 0, qk_scale, m, l, mfrag, fresh, g);
  if constexpr (FOLD) {
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] -= delta;
  }
}


}  // namespace bsattn
