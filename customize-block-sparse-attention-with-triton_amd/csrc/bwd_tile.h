// Pieces shared by the backward kernels: launch parameters, tile copies and operand fragments.
#pragma once
#include "common.h"
#include "kernel_util.h"
#include "place.h"
#include <type_traits>

namespace bsattn {

constexpr int BWD_SHORT_MAX_BLOCKS = 512;   // row blocks of a head up to which bwd_short_kernel takes a launch

struct BwdParams {
  const void* q; const void* k; const void* v; const void* o; const void* d_o;
  const float* lse; float* delta;
  void* dq; void* dk; void* dv;
  const int32_t* row_ptr; const int32_t* col_idx; const int32_t* col_ptr; const int32_t* row_idx;
  // elementwise masks: 64 words per entry of the row lists (bit = key) / of the column lists (bit = query)
  const unsigned long long* bits_rows; const unsigned long long* bits_cols;
  int B, H, N, nb, Bm, Hm;
  int out_f32;
  int split;                  // workgroups per row / column list (1: results written directly)
  int whole;                  // split > 1: lists of up to this many tiles are one workgroup's all the same (-1: none)
  float* part_dq; float* part_dk; float* part_dv;   // split > 1: fp32 partial results [split][B*H][N][D]
  float sm_scale, qk_scale;   // qk_scale = sm_scale * log2(e)
  int64_t qs[3], ks[3], vs[3], os[3], dos[3];
  int64_t dqs[3], dks[3], dvs[3];   // batch, head, row strides of the results (elements)
  PlaceOfEight place;         // workgroup -> (head, list, share)
  PlaceOfEight place_dq;      // dq_pairs_kernel's (one share)
  int first_sum;              // parts are added up of: 0 dQ, dK and dV, 1 dK and dV (dQ is dq_pairs_kernel's)
  Divisor per_batch;          // H
};

constexpr float kLog2e = 1.4426950408889634f;

// sum of the products of the eight 16-bit elements of a and b
template <bool BF16>
__device__ __forceinline__ float dot8(const uintx4& a, const uintx4& b, float acc) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float a0, a1, b0, b1;
    const unsigned int au = a[i], bu = b[i];   // by value: bit_cast of a vector element lvalue miscompiles
    if constexpr (BF16) {
      a0 = __builtin_bit_cast(float, au << 16); a1 = __builtin_bit_cast(float, au & 0xffff0000u);
      b0 = __builtin_bit_cast(float, bu << 16); b1 = __builtin_bit_cast(float, bu & 0xffff0000u);
    } else {
      const half2v ah = __builtin_bit_cast(half2v, au), bhh = __builtin_bit_cast(half2v, bu);
      a0 = (float)ah[0]; a1 = (float)ah[1]; b0 = (float)bhh[0]; b1 = (float)bhh[1];
    }
    acc += a0 * b0 + a1 * b1;
  }
  return acc;
}

// ---------------------------------------------------------------------------------------
// helpers of the two walking kernels
// ---------------------------------------------------------------------------------------
// ROWS: rows of a tile staged per step (64, or 32 when a tile is walked in two halves)
template <int D, bool EW, int ROWS = 64> struct BwdCfg {
  static constexpr int TILE_BYTES = ROWS * 2 * D;
  static constexpr int STAT_BYTES = 2 * 64 * 4;                    // lse2[64] + delta[64] of a row block
  static constexpr int BITS_BYTES = EW ? 64 * 8 : 0;               // mask words of the tile (elementwise masks)
  static constexpr int STAGE_BYTES = 2 * TILE_BYTES + STAT_BYTES + BITS_BYTES;  // two tiles, row statistics, mask words
  static constexpr int LDS_BYTES = 2 * STAGE_BYTES;                // double buffer
};

// This wavefront's half of the asynchronous copy of a ROWS x D tile (rows `stride` elements apart)
// into LDS with the u_swz chunk swizzle: wavefront wv issues half of the ROWS*D/512 instructions.
template <int D, int ROWS = 64>
__device__ __forceinline__ void half_tile_load_async(const unsigned short* tile, int64_t stride, int wv, int lane,
                                                     unsigned lds_addr) {
  constexpr int CPR = D / 8, PER_WAVE = ROWS * CPR / 128;
#pragma unroll
  for (int jj = 0; jj < PER_WAVE; ++jj) {
    const int j = wv * PER_WAVE + jj;
    const int c = j * 64 + lane, row = c / CPR, ch = c % CPR;
    const unsigned off = 2u * (unsigned)(row * (int)stride + ((ch ^ u_swz<D>(row)) * 8));
    tile_load_async_one(tile, off, lds_addr + j * 1024);
  }
}

// The same for rows first .. first + ROWS - 1 of a tile of which only `valid` rows exist (N is not a multiple of 64):
// the last one is repeated in place of the others, so that no address lies beyond the tensor.  tile: row 0 of it.
// (The lane index as a value the compiler cannot trace back: the offsets would otherwise be computed before the
// walk and held through it.)
template <int NWV, int D, int ROWS>
__device__ __forceinline__ void tail_tile_load_async(const unsigned short* tile, int64_t stride, int first, int valid, int wv,
                                                     int lane, unsigned lds_addr) {
  constexpr int CPR = D / 8, PER_WAVE = ROWS * CPR / (64 * NWV);
  asm volatile("" : "+v"(lane));
#pragma unroll 1
  for (int j = wv * PER_WAVE; j < (wv + 1) * PER_WAVE; ++j) {
    const int c = j * 64 + lane, row = c / CPR, ch = c % CPR, src = first + row < valid ? first + row : valid - 1;
    tile_load_async_one(tile, 2u * (unsigned)(src * (int)stride + ((ch ^ u_swz<D>(row)) * 8)), lds_addr + j * 1024);
  }
}

// Mask word of a lane in such a tile, shifted for mask_scores: bit = row or column of the tile, set for the first
// `valid` < 64.  (From a value the compiler cannot trace back, or its tests are made before the walk and held.)
__device__ __forceinline__ unsigned long long tail_word(int valid, int g) {
  asm volatile("" : "+s"(valid));
  return ((1ull << valid) - 1ull) >> (4 * g);
}

// asynchronous copy of 64 consecutive floats (one per lane)
__device__ __forceinline__ void stat_load_async(const float* src, int lane, unsigned lds_addr) {
  words_load_async(src, 4u * (unsigned)lane, lds_addr);
}

// operand fragment (32 rows x 16 columns slice s) of a swizzled LDS tile: row r0 + ln, chunk 2s + g
template <int D>
__device__ __forceinline__ uintx4 frag_rows(const unsigned char* tile, int r0, int s, int ln, int g) {
  const int row = r0 + ln;
  return *reinterpret_cast<const uintx4*>(tile + row * 2 * D + (((2 * s + g) ^ u_swz<D>(row)) * 16));
}

// transposed operand fragment: columns 32db + ln of the tile along the lanes, contraction slots j
// of slice ts <-> tile rows 16ts + 8(j/4) + 4g + (j%4) (the order in which a 32x32 MFMA result
// holds its rows), by two LDS transpose reads
template <int D, bool BF16>
__device__ __forceinline__ uintx4 frag_cols(const unsigned char* tile, int db, int ts, int lane) {
  const int blk = lane >> 4, s16 = lane & 15;
  uintx4 a;
#pragma unroll
  for (int jh = 0; jh < 2; ++jh) {
    const int row = 16 * ts + 8 * jh + 4 * (blk >> 1) + (s16 >> 2);
    const int col = 32 * db + 16 * (blk & 1) + 4 * (s16 & 3);
    const int addr = row * 2 * D + (((col >> 3) ^ u_swz<D>(row)) * 16) + (col & 7) * 2;
    const short4v rr = __builtin_amdgcn_ds_read_tr16_b64_v4i16((short4v __attribute__((address_space(3)))*)(tile + addr));
    const uintx2 r2 = __builtin_bit_cast(uintx2, rr);
    a[2 * jh] = r2[0]; a[2 * jh + 1] = r2[1];
  }
  if constexpr (BF16) a = bf16x8_to_f16x8(a);
  return a;
}

// scores of unset mask elements become -inf; mw: the 64 mask bits of this lane's row, already
// shifted right by 4 g, so that bit 8(i/4) + i%4 (+ 32 for the second block) belongs to register i
__device__ __forceinline__ void mask_scores(floatx16& s0, floatx16& s1, unsigned long long mw) {
  const unsigned lo = (unsigned)mw, hi = (unsigned)(mw >> 32);
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const unsigned bit = 1u << (8 * (i / 4) + (i % 4));
    s0[i] = (lo & bit) ? s0[i] : -INFINITY;
    s1[i] = (hi & bit) ? s1[i] : -INFINITY;
  }
}

// the same for one block of 32 keys (bits 0..31 of the shifted word)
__device__ __forceinline__ void mask_scores(floatx16& s0, unsigned lo) {
#pragma unroll
  for (int i = 0; i < 16; ++i) s0[i] = (lo & (1u << (8 * (i / 4) + (i % 4)))) ? s0[i] : -INFINITY;
}

// The same for elementwise masks, where most tiles of a window or a causal mask are kept entirely: one test for the wavefront in front of
// the 16 or 32.  us of a backward, before / with it, token windows of N / 4, N / 2, token-causal: D = 64, 10 heads N = 8127 270 / 242, 352 / 324, 526 / 492;
// 16 heads N = 4000 116 / 114, 167 / 159, 212 / 198; D = 128, 16 heads N = 6000 310 / 304, 464 / 449, 617 / 590.  (Not at D = 256, where the matrix cores
// wait for LDS: 8 heads N = 4000 182 / 185, 308 / 310, 404 / 418.)
constexpr unsigned MASK_BITS = 0x0f0f0f0fu;      // the bits of a word that belong to registers
__device__ __forceinline__ void mask_partly(floatx16& s0, floatx16& s1, unsigned long long mw) {
  if (__any(((unsigned)mw & (unsigned)(mw >> 32) & MASK_BITS) != MASK_BITS)) mask_scores(s0, s1, mw);
}
__device__ __forceinline__ void mask_partly(floatx16& s0, unsigned lo) {
  if (__any((lo & MASK_BITS) != MASK_BITS)) mask_scores(s0, lo);
}

__device__ __forceinline__ floatx16 zero16() {
  floatx16 z;
#pragma unroll
  for (int i = 0; i < 16; ++i) z[i] = 0.f;
  return z;
}


// Values that live in registers through a walking loop (fragments of the stationary operand, row statistics) are
// passed through here once they have been asked for: the compiler waits for their loads at this point.  Left to
// itself it moves the loads next to the loop and plants its waits at their first uses inside it, where, being
// counted waits, they also wait for the tile copies of the next step that have just been issued, in every step.
__device__ __forceinline__ void settle(uintx4& x) { asm volatile("" : "+v"(x)); }
__device__ __forceinline__ void settle(float& x) { asm volatile("" : "+v"(x)); }

}  // namespace bsattn
