// Block-sparse FlashAttention-2 forward for gfx950, head dimension 64 (attn_fwd_short.hip has its launches with few row blocks,
// attn_fwd_pair.hip the larger head dimensions), and what the host decides about a forward launch.
//
// Work decomposition.  The kept tiles of one head form a list in row-major order; it is cut
// into W contiguous ranges, one per workgroup, regardless of row boundaries (W depends on
// shapes only, so no host synchronisation on the mask content is needed; where two workgroups
// share a compute unit the first-comer's range is longer, see fwd_split.h).  A workgroup walks
// its range row block by row block; the kept tiles of the current row block that fall inside
// the range are handed to the workgroup's wavefronts one at a time, each wavefront runs the
// online softmax over the tiles it gets with private LDS tile buffers, and the per-wavefront
// results (acc, m, l) are merged through LDS.  A row block that lies completely inside the
// range is normalised and written straight to O.  A row block cut by range boundaries is
// finished by the workgroup that holds its first tiles: the others publish unnormalised parts
// in the workspace (device-scope stores, then a flag), and it pulls them when it gets there.
// That is the way of launches with few row blocks (COOP).  With about as many as wavefronts fit the GPU, a range
// belongs to a single wavefront (WAVE); with more a wavefront takes a whole row block, or a part of a long one (ROWS).
//
// Per tile a wavefront computes S^T = K Q^T (keys along MFMA rows, queries along lanes), so
// that one lane owns one query: softmax statistics are in-lane reductions plus a single
// cross-half exchange, and P^T leaves the accumulators already in the operand layout of the
// second product O^T += V^T P^T.
//
// Recurrence as the reference kernel, fa2_custom_mask/fa2_fwd.py:146-196 (exp2 domain, fp32
// statistics, P rounded to 16 bits for the second product), with two changes that keep the
// vector ALU out of the way of the matrix cores: the softmax scale is folded into Q, and the
// running maximum is replaced by a reference exponent that is only moved when needed.
#include <algorithm>
#include <atomic>
#include <mutex>
#include <map>
#include <array>
#include <chrono>
#include <cstdlib>
#include "common.h"
#include "fwd_split.h"
#include "fwd_tile.h"
#include "kernel_util.h"
#include "range_perm.h"
#include "row_parts.h"

namespace bsattn {

// A workgroup is four wavefronts, one per SIMD.  A wavefront needs 256 registers and two workgroups share a compute unit
// (while one merges or waits for its first tiles the other computes).
// (At D = 128 a wavefront that owns 64 queries needs all 512 registers of its SIMD and spills beside them: every launch was
// slower here than with the pairs of attn_fwd_pair.hip.)
template <int D> struct FwdCfg {
  static constexpr int NW = 4;
  static constexpr int WG_PER_CU = 2;
  static constexpr int TILE_BYTES = 64 * 2 * D;             // one K or V tile in LDS
  static constexpr int WAVE_LDS = 2 * TILE_BYTES;           // K buffer + V buffer
  static constexpr int ML_BYTES = NW * 2 * 64 * 4 + 64;     // exchange of (m, l) per query + the tile counter
  static constexpr int COLS_CAP = 2048;                     // column indices of the range kept in LDS
  static constexpr int BITS_OFF = NW * WAVE_LDS + ML_BYTES + COLS_CAP * 4;   // mask words of the current tile, 512 bytes per wavefront
  static constexpr int LDS_BYTES = BITS_OFF + NW * 512;
  // one wavefront per workgroup (ROWS): eight workgroups share the 160 KB of a compute unit
  static constexpr int ROWS_COLS_CAP = 896;
  static constexpr int ROWS_BITS_OFF = WAVE_LDS + ROWS_COLS_CAP * 4;
  static constexpr int ROWS_LDS_BYTES = ROWS_BITS_OFF + 512;
  static constexpr int R = WAVE_LDS / 256;                  // accumulator registers exchanged per round (K and V buffer)
  static constexpr int ROUNDS = D / R;
  static constexpr int QPW = (R / 4) / NW;                  // output quads per wavefront and round
  static constexpr int SHORT_ROW = 6 * NW;                  // row blocks up to this many tiles may go to one wavefront
  static constexpr int SNAP = 16;                           // short ranges: a boundary at least this close to an end of its row block moves there
};

// DT: 0 fp16; 1 bf16 with P rounded to fp16 (V fragments converted); 2 bf16 with P rounded to bf16.
// MODE.  COOP: the ranges of four-wavefront workgroups described above (launches with few row blocks).  ROWS: a workgroup
// is one wavefront and takes one row block, or parts of long ones (many row blocks: next to nothing to merge, the
// dispatcher balances the load).
// WAVE: a workgroup is one wavefront and takes one range of its head's list (in between: about as many row blocks as
// wavefronts fit the GPU, which whole row blocks would leave half idle in a second round).
// LAYOUT: GENERAL any strides, any number of tokens; CONTIG_WHOLE the rows of K and of V follow each other without gaps
// (row stride = D) and N is a multiple of 64; CONTIG_TAIL without gaps, any N.
// Where N is not a multiple of 64 the last tile of a row list holds `valid` < 64 keys: its copy repeats the last
// key (no address lies beyond the tensor) and its scores beyond `valid` are set to -inf; the query rows of the last
// row block beyond N repeat the last query and are not written.
enum { GENERAL = 0, CONTIG_WHOLE = 1, CONTIG_TAIL = 2 };
enum { COOP = 0, ROWS_MODE = 1, WAVE = 2 };
// SPREAD: COOP and WAVE with a number of heads that does not divide 8 (place_range).  A variant of its own: the code of the other
// way in the prologue, even where it is jumped over, costs a launch of one head 0.3 us and eight heads 0.7 %.
template <int D, int DT, int MODE, bool EW, int LAYOUT, bool SPREAD>
__global__ __launch_bounds__(MODE != COOP ? 64 : FwdCfg<D>::NW * 64, FwdCfg<D>::WG_PER_CU)
void fwd_kernel(const FwdRangeParams prm) {
  constexpr bool BF16 = DT != 0, PB = DT == 2;
  constexpr bool CONTIG = LAYOUT == CONTIG_WHOLE || LAYOUT == CONTIG_TAIL, TAIL = LAYOUT == GENERAL || LAYOUT == CONTIG_TAIL;
  using C = FwdCfg<D>;
  constexpr bool ROWS = MODE == ROWS_MODE, ONE = MODE != COOP;     // ONE: one wavefront per workgroup
  constexpr int NW = ONE ? 1 : C::NW;
  constexpr bool FOLD = !BF16;     // fp16: scale folded into Q, reference exponent via an extra MFMA slice
  constexpr int KS = D / 16;       // k-slices of the first product
  constexpr int DB = D / 32;       // 32-wide blocks of the head dimension
  constexpr int CPR = D / 8;       // 16-byte chunks per row
  constexpr int ROWB = 2 * D;      // bytes per LDS row
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];

  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ln = lane & 31, g = lane >> 5;
  // linear id -> (head, range): every head gets its share of the workgroups that are first on their compute unit, and an
  // XCD as few heads as possible (place_range; 1, 2, 4 or 8 heads are interleaved, which is the same and what the range
  // permutations below are made for)
  const int BH = prm.B * prm.H, nb = prm.nb;
  int bh, wg;
  if constexpr (ROWS) {
    // (head, row block): heads in groups of `group` (place.h), so that the row blocks at work on an XCD share the K and V of
    // few heads in its L2 (rows_group); in a group the last row blocks of all heads, the long ones of block-causal masks,
    // first.  Behind the first `first_ids` of them, which fill the GPU, W workgroups per head for the long row blocks
    // (wg >= nb; see below).
    const PlaceOfRows at = place_rows(blockIdx.x, BH, prm.group, nb, prm.W, prm.first_ids);
    if (at.p.item >= at.per) return;             // padding of the last group
    bh = at.p.head;
    wg = at.per - 1 - at.p.item + (at.extra ? nb : 0);
  } else if constexpr (SPREAD) {
    const Place p = place_range(blockIdx.x, BH, prm.W, prm.place_fast, prm.place_quot, prm.place_rest);
    bh = p.head;
    wg = p.item;
  } else {      // (1, 2, 4 or 8 heads)
    bh = blockIdx.x & (BH - 1);
    wg = blockIdx.x >> __builtin_ctz(BH);
  }
  const int b = (int)prm.per_batch.of((unsigned)bh), h = bh - b * prm.H;
  const int mh = (prm.Bm > 1 ? b : 0) * prm.Hm + (prm.Hm > 1 ? h : 0);
  // keys of the last tile column; its column block (-1: every tile is whole)
  const int valid = TAIL ? prm.N - (nb - 1) * 64 : 64;
  const int tail_cb = TAIL && valid < 64 ? nb - 1 : -1;
  // the lists are read-only for the whole launch: constant address space => scalar loads
  const cint_ptr_t rp = (cint_ptr_t)(uintptr_t)(prm.row_ptr + (int64_t)mh * nb);
  const cint_ptr_t cols = (cint_ptr_t)(uintptr_t)prm.col_idx;
  HeadSplit hs;
  int snap = 0;
  int64_t x0 = 0, x1 = 0;
  int own_first = 0, own_parts_n = 0;  // a workgroup takes a row block or a part of it: where its parts begin, how many they are
  int r = 0, g0 = 0, g1 = 0;         // COOP: first row block and tiles of the range, g0 < g1 where they are known already
  if constexpr (!ROWS) {
    // (where the head's lists begin, for the choice below: every wavefront asks for all of them now, beside the head's ends, and does
    // not wait; as atomics, which the compiler does not move to their use)
    constexpr int OWN_LOADS = OWN_ROWS_MOST / 64 + 1;
    int begins[OWN_LOADS] = {};
    if constexpr (MODE == COOP && CONTIG) {
      const int32_t* p = prm.row_ptr + (int64_t)mh * nb;
#pragma unroll
      for (int j = 0; j < OWN_LOADS; ++j)
        begins[j] = __hip_atomic_load(p + (64 * j + lane < nb ? 64 * j + lane : nb), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
    }
    hs = head_split(rp, nb, prm.W, /*min_tiles=*/ONE ? 4 : NW, prm.first_ids > bh ? (prm.first_ids - bh + BH - 1) / BH : 0, 0);
    // Long ranges (the regime of the weighted shares) are cut on the axis with gaps and boundaries move to a row
    // block's end only from very close; short ranges are cut on the plain tile axis and their boundaries move to
    // the nearer end of a row block from up to half a range (and at least SNAP tiles) away: a row block is shared
    // only where a boundary falls into its middle, row blocks of up to a range's length or 2 SNAP tiles never (N = 17536,
    // one head, against 8 tiles for every head: keep 0.15 36.0 -> 31.4 us, keep 0.2 40.0 -> 34.6, keep 0.25 43.2 -> 39.8,
    // keep 0.05 21.8 -> 20.2, keep 0.1 25.8 -> 25.1; keep 0.35 and above, other sizes: +-1 %).
    constexpr int LONG_GAP = MODE == WAVE ? 2 : 12, LONG_SNAP = 2;
    const bool long_ranges = MODE == WAVE || ((int64_t)hs.T >= (int64_t)EQUAL_SPLIT_BELOW * hs.Peff || hs.Peff >= 3 * nb);   // (or row blocks much longer than the ranges)
    const int half_range = hs.T / (2 * (hs.Peff > 0 ? hs.Peff : 1)) + 1;
    // (long ranges over short row blocks, up to 32 tiles on average: a boundary moves to the nearer end of its row block
    // from up to half such a row block away, so that next to no row block is shared; against 2 tiles: 8 heads of
    // N = 17536 at keep 0.05 67.9 -> 62 us, 4 heads at keep 0.1 57.9 -> 54.6 us; with longer row blocks the imbalance
    // costs more than the sharing: keep 0.35, one head, 48.0 -> 50.4 us with 12 tiles)
    const int avg_row = hs.T / (nb > 0 ? nb : 1);
    const int long_snap = MODE != WAVE && avg_row <= 32 ? avg_row / 2 + 1 : LONG_SNAP;
    snap = long_ranges ? long_snap : (half_range > C::SNAP ? half_range : C::SNAP);
    // (ranges that are long only against the row blocks they lie in, several to a row block: 24 positions; N = 6400
    // dense 31.2 -> 29.0 us, where 12 are best for N = 17536 dense, 102.1 against 104.0 us)
    const int long_gap = MODE == WAVE || (int64_t)hs.T >= (int64_t)EQUAL_SPLIT_BELOW * hs.Peff ? LONG_GAP : 2 * LONG_GAP;
    if (long_ranges) { hs.gap = long_gap; hs.X = (int64_t)hs.T + (int64_t)long_gap * nb; }
    const int own_row = wg;          // (the first workgroups on their compute units are the first row blocks')
    // Which range this workgroup takes (launches with few heads and long ranges): the ranges of a head start at
    // all phases of a row, and workgroups that share an XCD, hence an L2, get ranges of like phase, so that they
    // walk the same column blocks at the same time (dense N = 17536, one head: 42 instead of 196 MB fetched from
    // HBM per launch, 104.5 instead of 106.6 us).  The phases are those of rows of equal length: heads that keep less
    // than three quarters of their tiles are left alone (keep 0.5 measured 2 % slower with the permutation), except
    // the dense block-causal mask, which has a table of its own (N = 32000: 185 instead of 193 us).
    if (MODE == COOP && prm.perm_n > 0 && prm.perm_n == hs.Peff && prm.perm_fast == hs.fast) {
      if (hs.T >= prm.perm_min_tiles) wg = prm.perm[wg];
      // the dense block-causal mask (by its number of kept tiles and the length of one row in the middle; a mask
      // taken for it by mistake merely gets its ranges in another order): ranges sorted by their first column block
      else if ((int64_t)hs.T * 2 == (int64_t)nb * (nb + 1) && rp[nb / 2 + 1] - rp[nb / 2] == nb / 2 + 1) wg = prm.perm_causal[wg];
    }
    // Heads cut into equal shares: the two workgroups of a compute unit (linear ids L and L + first_ids: the
    // dispatcher places them in the same order in both rounds) take neighbouring ranges 2k and 2k + 1.  A boundary that
    // moves to a row block's end moves tiles from one range to its neighbour; between the two workgroups of a compute
    // unit that changes nothing in what the compute unit has to do, and only every other boundary unbalances the
    // compute units (keep 0.1, N = 17536: 26.2 -> 24.8 us; keep 0.25: 42.2 -> 41.6 us).  (All boundaries move by the
    // same rule: one that may move further than its neighbours can overtake them.)
    {
      const int Fh = prm.first_ids > bh ? (prm.first_ids - bh + BH - 1) / BH : 0;
      if (MODE == COOP && hs.fast == 0 && hs.Peff == prm.W && prm.W == 2 * Fh) wg = wg < Fh ? 2 * wg : 2 * (wg - Fh) + 1;
    }
    // Row blocks without kept tiles belong to no range: they are dealt round-robin over all workgroups
    // of the head, which write O = 0, lse = -inf for their share.
    {
      for (int r0 = wg; r0 < nb; r0 += prm.W) {
        if (rp[r0 + 1] > rp[r0]) continue;
        void* ob = out_base(prm, b, h);
        for (int i = threadIdx.x; i < 64 * (D / 4); i += NW * 64) {
          const int64_t qrow = (int64_t)r0 * 64 + i / (D / 4);
          if (TAIL && qrow >= prm.N) break;
          store_out4<BF16>(ob, qrow * prm.os[2] + 4 * (i % (D / 4)), prm.out_f32, 0.f, 0.f, 0.f, 0.f);
        }
        if (prm.lse != nullptr && threadIdx.x < 64 && (!TAIL || r0 * 64 + (int)threadIdx.x < prm.N)) prm.lse[(int64_t)bh * prm.N + (int64_t)r0 * 64 + threadIdx.x] = -INFINITY;
      }
    }
    if (hs.T == 0) return;
    // Short lists of about the same length (own_rows.h): the first workgroups on their compute units take a row block each, the second ones the row
    // blocks that are left, in as many parts of 8 tiles or more as there are workgroups for.  Nothing has to be searched for and little meets in the
    // workspace, 3 to 8 us of a launch, and no compute unit has two whole row blocks beside others that have none (where ranges snap to row
    // blocks).  The ranges balance the work of uneven lists and long lists by what the first-comers on a compute unit are faster: a causal mask's,
    // told by its first half of rows; heads with a list longer than the rest saves (lists of about 26 tiles and one of 42, 50, 74, 1 head N = 17536:
    // 23.1 / 22.0, 22.9 / 24.7, 23.3 / 30.9; of 42, 58, 74 where every compute unit has two row blocks, 2 heads N = 16064: 34.2 / 28.0, 33.5 / 31.8, 33.7 / 36.3), as row
    // blocks kept whole are (0-3 and column blocks 0-3, ranges / so / as it is: N = 17536 keep 0.1 34.6 / 90 / 35.0, N = 12032 31.4 / 62 / 31.7, N = 32000
    // keep 0.05 41 / 161 / 42, 3 heads N = 10048 keep 0.1 33.6 / 57 / 34.0); and, where compute units have more than one row block, heads of which more than a
    // quarter of the lists are much longer than the mean (every other row at keep 0.1, the others at 0.01: N = 30000 38.5 / 47.8 / 39.0; taken: 3 heads N = 10048
    // 24.6 / 21.9 / 22.3, and with a row block per compute unit N = 10048 19.8 / 16.8 / 17.2).  Looking at all lists costs 0.1 to 0.5 us.  (Not with strided K or V,
    // where the variant for a number of heads that does not divide 8 would spill
    // registers.)  Ranges / so, fp16, us; tiles of a row block, about 3, 8, 16, 26, 32, 48, 64:
    //   1 head  N = 10048 (157 row blocks, 256 first workgroups)  13.0/10.7   15.9/13.1   18.9/16.0   20.7/18.4   22.1/22.1   25.2/26.9   27.8/30.7
    //   1 head  N = 16384 (256)                                   12.1/11.2   15.1/14.0   18.2/16.7   22.5/20.0   25.1/23.1   29.7/28.9   35.5/35.1
    //   1 head  N = 17536 (274, parts; 8 masks each)              14.5/12.9   16.1/16.5   18.3/18.7   23.6/21.8   26.8/24.8   30.0/29.1   35.8/35.8
    //   1 head  N = 20032 (313)                                   15.8/14.5   16.6/17.7   19.3/19.5   25.2/22.8   28.5/26.3   32.6/31.3   38.9/37.3
    //   2 heads N = 9024 (141 of 128, parts)                      14.4/12.8   15.7/16.0   17.7/18.2   23.1/21.1   26.2/24.2   29.8/28.3   35.3/34.0
    //   1 head  N = 24000 (375, parts)                            15.7/15.2   19.8/17.5   21.7/20.8   26.4/24.4   29.3/27.9   37.5/34.4   45.9/40.2
    //   1 head  N = 27008 (422, whole)                                 -      20.7/18.0   25.6/22.7   30.5/27.2   35.9/30.7   39.6/40.5   47.9/53.2
    //   1 head  N = 32000 (500, whole)                            16.0/13.9   23.8/19.1   29.3/24.9   35.4/29.1   41.3/35.0   54.4/43.1   56.0/53.1    (causal, 25: 34 / 38)
    //   3 heads N = 10048 (157 of 85, whole)                      15.9/13.9   22.1/17.7   29.0/23.4   33.9/26.9   39.3/31.1   49.3/41.2   51.6/50.0
    auto of_like_length = [&]() {
      const int longest = own_rows_longest(prm.own, hs.T), even = own_rows_even(prm.own, hs.T);
      int most = 0, uneven = 0, middle = 0;
#pragma unroll
      for (int j = 0; j + 1 < OWN_LOADS; ++j) {
        if (64 * j >= nb) break;
        // (a list ends where the next lane's begins; behind the last one all begin at the head's end)
        const int next = __builtin_amdgcn_update_dpp(__builtin_amdgcn_readfirstlane(begins[j + 1]), begins[j], /*wave_shl:1*/ 0x130, 0xf, 0xf, false);
        const int end = 64 * j + lane < nb ? next : begins[j], len = end - begins[j];
        most = len > most ? len : most;
        uneven += __builtin_popcountll(__ballot(len > even));
        if (nb / 128 == j) middle = __builtin_amdgcn_readlane(begins[j], nb / 2 % 64) - hs.lo;
      }
      return own_rows_by_middle(hs.T, middle) && !__any(most > longest) && 4 * uneven <= nb;
    };
    if (MODE == COOP && CONTIG && own_rows_by_tiles(prm.own, hs.T, nb) && of_like_length()) {
      const OwnItem it = own_item(own_row, nb, prm.W, prm.first_ids > bh ? (prm.first_ids - bh + BH - 1) / BH : 0);
      r = it.row;
      if (r >= nb) return;
      const int row_s = rp[r], len = rp[r + 1] - row_s, parts = own_parts(len, it.most);
      if (it.part >= parts || len == 0) return;
      g0 = row_s + len * it.part / parts;
      g1 = row_s + len * (it.part + 1) / parts;
      wg = own_row;
      own_first = own_row - it.part;
      own_parts_n = parts;
    } else {
      if (wg >= hs.Peff) return;
      // where the range begins and ends on the cutting axis
      x0 = split_pos(hs, wg); x1 = split_pos(hs, wg + 1);
      if (x0 >= x1) return;
    }
  }

  unsigned char* lds_k = lds + w * C::WAVE_LDS;
  unsigned char* lds_v = lds_k + C::TILE_BYTES;
  float* ml = reinterpret_cast<float*>(lds + NW * C::WAVE_LDS);     // [NW][2][64]
  const unsigned lds_k_addr = (unsigned)(uintptr_t)(lds_ptr_t)lds + w * C::WAVE_LDS;
  const unsigned lds_v_addr = lds_k_addr + C::TILE_BYTES;

  const unsigned short* qg = (const unsigned short*)prm.q + b * prm.qs[0] + h * prm.qs[1];
  const unsigned short* kg = (const unsigned short*)prm.k + b * prm.ks[0] + h * prm.ks[1];
  const unsigned short* vg = (const unsigned short*)prm.v + b * prm.vs[0] + h * prm.vs[1];
  const float qk_scale = prm.qk_scale;

  // Per-lane source byte offsets of the asynchronous tile loads (loop invariant).  Copy
  // instruction j covers rows [64j/CPR, 64(j+1)/CPR) of the tile; the row part of the offset is
  // added to the (scalar) tile pointer, the per-lane part only depends on j through the chunk
  // swizzle, whose pattern repeats with period KPER in j (K) or not at all (V).
  constexpr int RPI = 64 / CPR;                 // tile rows per copy instruction
  constexpr int KPER = 2;                       // period of the K swizzle in copy instructions
  unsigned koff[KPER], voff[1];
  {
    const int row0 = lane / CPR, ch = lane % CPR;
#pragma unroll
    for (int par = 0; par < KPER; ++par)
      koff[par] = 2u * (unsigned)(row0 * (int)prm.ks[2] + ((ch ^ k_swz<D>(par * RPI + row0)) * 8));
    voff[0] = 2u * (unsigned)(row0 * (int)prm.vs[2] + ((ch ^ v_swz<D>(row0)) * 8));
  }
  static_assert(D == 64, "swizzle period");
  auto k_copy = [&](const unsigned short* tile, int j) {
    tile_load_async_one(tile + (int64_t)j * RPI * prm.ks[2], koff[j % KPER], lds_k_addr + j * 1024);
  };
  auto v_copy = [&](const unsigned short* tile, int j) {
    tile_load_async_one(tile + (int64_t)j * RPI * prm.vs[2], voff[0], lds_v_addr + j * 1024);
  };
  constexpr int BITS_OFF = ONE ? C::ROWS_BITS_OFF : C::BITS_OFF, COLS_CAP = ONE ? C::ROWS_COLS_CAP : C::COLS_CAP;
  const unsigned lds_bits_addr = (unsigned)(uintptr_t)(lds_ptr_t)lds + BITS_OFF + w * 512;
  const unsigned long long* lds_bits = reinterpret_cast<const unsigned long long*>(lds + BITS_OFF + w * 512);
  constexpr int KOPS = CPR + (EW ? 2 : 0);      // instructions of one K copy
  // copy of the K tile `tile` = entry t of the kept-tile list (EW: with its 512 bytes of mask words)
  // CONTIG (rows that follow each other without gaps, the usual case): copy instruction j reads at
  // byte offset 1024 j from the tile and writes at 1024 j from the buffer, and the instruction's immediate
  // offset applies to both, so four instructions share one scalar base and one m0 (6 instead of 24 scalar
  // instructions per tile copy at D = 64).
  constexpr bool k_contig = CONTIG, v_contig = CONTIG;
  const int64_t k_rs = CONTIG ? (int64_t)D : prm.ks[2], v_rs = CONTIG ? (int64_t)D : prm.vs[2];   // row strides (a constant: a tile's address is a shift)
  // copy of a tile whose last rows do not exist (`valid` of them do): every instruction's rows are bounded
  // (the lane index as a value the compiler cannot trace back: the offsets would otherwise be computed before the
  // tile loop and occupy registers throughout it)
  auto tail_copy = [&](const unsigned short* tile, int64_t rs, unsigned lds_addr, auto&& swz) {
    int lane_t = lane;
    asm volatile("" : "+v"(lane_t));
#pragma unroll 1
    for (int j = 0; j < CPR; ++j) {
      const int row = j * RPI + lane_t / CPR, src = row < valid ? row : valid - 1;
      tile_load_async_one(tile, 2u * (unsigned)(src * (int)rs + (((lane_t % CPR) ^ swz(row)) * 8)), lds_addr + j * 1024);
    }
  };
  auto k_copy_all = [&](int cb, int t) {
    const unsigned short* tile = kg + (int64_t)cb * 64 * k_rs;
    if (TAIL && cb == tail_cb) {
      tail_copy(tile, k_rs, lds_k_addr, [](int row) { return k_swz<D>(row); });
    } else if constexpr (k_contig) {
#pragma unroll
      for (int jb = 0; jb < CPR; jb += 4)
        tile_load_async_four(tile + jb * RPI * D, koff[jb % KPER], koff[(jb + 1) % KPER], koff[(jb + 2) % KPER], koff[(jb + 3) % KPER],
              lds_k_addr + jb * 1024);
    } else {
#pragma unroll
      for (int j = 0; j < CPR; ++j) k_copy(tile, j);
    }
    if constexpr (EW) {
      const unsigned long long* src = prm.tile_bits + (int64_t)t * 64;
#pragma unroll
      for (int j = 0; j < 2; ++j)
        words_load_async(src, 4u * (unsigned)lane + 256u * j, lds_bits_addr + j * 256);
    }
  };
  auto v_copy_all = [&](int cb) {
    const unsigned short* tile = vg + (int64_t)cb * 64 * v_rs;
    if (TAIL && cb == tail_cb) {
      tail_copy(tile, v_rs, lds_v_addr, [](int row) { return v_swz<D>(row); });
    } else if constexpr (v_contig) {
#pragma unroll
      for (int jb = 0; jb < CPR; jb += 4)
        tile_load_async_four(tile + jb * RPI * D, voff[0], voff[0], voff[0], voff[0], lds_v_addr + jb * 1024);
    } else {
#pragma unroll
      for (int j = 0; j < CPR; ++j) v_copy(tile, j);
    }
  };
  // per-lane LDS byte offsets of the operand reads.  K fragment (kb, s): row 32kb+ln, chunk 2s+g
  int kaddr[2][KS];
#pragma unroll
  for (int kb = 0; kb < 2; ++kb)
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const int row = 32 * kb + ln;
      kaddr[kb][s] = row * ROWB + (((2 * s + g) ^ k_swz<D>(row)) * 16);
    }
  // V^T fragment via transpose reads: lane (16-lane block blk, s) supplies 4 halfs of key row
  // 4*(blk/2) + s/4 (+ 16ts + 8jh) at column 16*(blk%2) + 4*(s%4) (+ 32db)
  const int vblk = lane >> 4, vs_ = lane & 15;
  const int vkey0 = 4 * (vblk >> 1) + (vs_ >> 2), vcol0 = 16 * (vblk & 1) + 4 * (vs_ & 3);

  const uintx4 ones_frag = {g == 0 ? 0x3c003c00u : 0u, 0u, 0u, 0u};

  // ---- state of the row block a wavefront is working on, and the steps both drivers share ----
  uintx4 qf[2][KS];          // Q fragments (second operand of S^T = K Q^T): lane owns query ln (+32 qb)
  floatx16 oacc[DB][2];
  // m_i: reference exponent of the row (exp2 domain), l_i: per-lane partial sum of P (this lane's
  // half of the keys), both relative to m_i.  m_i starts at 0 and is re-centred on the first tile
  // and whenever a tile produces a P above 2^14.
  float m_i[2], l_i[2];
  // FOLD: "-m_i" enters the scores through one extra contraction slice, ones x (-m_hi, -m_lo)
  uintx4 mfrag[2];
  bool fresh = true;
  float limit[2] = {SUM_LIMIT, SUM_LIMIT};
  int any_m = 0;     // (wave-uniform) some lane's reference exponent is not zero: the extra contraction slice is needed

  auto reset_acc = [&]() {
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int qb = 0; qb < 2; ++qb)
#pragma unroll
        for (int i = 0; i < 16; ++i) oacc[db][qb][i] = 0.f;
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) { m_i[qb] = 0.f; l_i[qb] = 0.f; mfrag[qb] = uintx4{0u, 0u, 0u, 0u}; limit[qb] = FOLD || EW ? SUM_LIMIT : 0.f; }
    fresh = true;
    any_m = 0;
  };
  // One wavefront: per-lane addresses that do not change from row block to row block are not to be held through the tile
  // loops: the lane index as a value the compiler cannot trace back
  auto fresh_lane = [&](int x) {
    if constexpr (ONE) asm volatile("" : "+v"(x));
    return x;
  };
  auto load_q = [&](int r) {
    const int lane_q = fresh_lane(lane), ln = lane_q & 31, g = lane_q >> 5;
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) {
      int row = r * 64 + qb * 32 + ln;
      if (TAIL && row >= prm.N) {
        row = prm.N - 1;
        if constexpr (EW) l_i[qb] = 1e-30f;      // (a query that has no mass yet is recentred in every tile; this one never will)
      }
      const unsigned short* qrow = qg + (int64_t)row * prm.qs[2];
#pragma unroll
      for (int s = 0; s < KS; ++s) qf[qb][s] = *reinterpret_cast<const uintx4*>(qrow + 16 * s + 8 * g);
    }
    // vmcnt(0), visible to the compiler: Q is complete here, so that no vector-memory waits of
    // its own end up inside the tile loop (they would also wait for the tile prefetches)
    __builtin_amdgcn_s_waitcnt(0x0F70);
    if constexpr (FOLD) {
      // fold sm_scale*log2(e) into Q once per row block: the scores leave the MFMA already in
      // the exp2 domain (fp16 rounding of the scaled Q perturbs an exponent by ~1e-4)
#pragma unroll
      for (int qb = 0; qb < 2; ++qb)
#pragma unroll
        for (int s = 0; s < KS; ++s) {
          const uintx4 raw = qf[qb][s];
          const uintx4 scaled = {scale_half2(raw[0], qk_scale), scale_half2(raw[1], qk_scale),
                                 scale_half2(raw[2], qk_scale), scale_half2(raw[3], qk_scale)};
          qf[qb][s] = scaled;
        }
    }
  };

  // One 64 x 64 tile whose K and V copies have been issued (K first).  has1: the wavefront has a
  // next tile, in column block cbn, whose K copy is issued as soon as this tile's K fragments sit
  // in registers; copy_v: its V copy may be issued too, as soon as this tile's V fragments sit in
  // registers.  Copies are therefore issued in the order K(cur), V(cur), K(nxt), V(nxt), ..., and
  // every wait allows exactly the one younger copy (CPR instructions) in flight.  `mid` runs once
  // the first LDS wait of the tile has passed (the place to pick up earlier LDS results).
  // The tile is processed as four blocks so that the matrix cores and the vector ALU of this
  // wavefront overlap: [1] scores of query block 0, [2] scores of query block 1 interleaved with
  // the softmax numerators of block 0, [3] second product of block 0 interleaved with the
  // numerators of block 1, [4] second product of block 1.  Operand fragments are read from LDS
  // once, all at once (the read latency is a multiple of an MFMA's issue interval), and serve
  // both query blocks.
  auto tile = [&](bool has1, int cbn, int tn, bool copy_v, bool partial, auto&& mid) {
    uintx4 kfr[2][KS], vfr[4][DB];
    uintx4 pf[4][2];  // P^T operand fragments: [16-key slice][qb]
    auto scores = [&](int qb, floatx16& s0, floatx16& s1) {   // S^T[.][qb] = K Q[qb]^T (- m_i when FOLD)
#pragma unroll
      for (int i = 0; i < 16; ++i) { s0[i] = 0.f; s1[i] = 0.f; }
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        s0 = mfma_qk<BF16>(kfr[0][s], qf[qb][s], s0);
        s1 = mfma_qk<BF16>(kfr[1][s], qf[qb][s], s1);
      }
    };
    // FOLD: "- m_i" through the extra slice, only while some lane of the wavefront has moved its reference
    auto mslice = [&](int qb, floatx16& s0, floatx16& s1) {
      if constexpr (FOLD) {
        if (any_m) {
          s0 = mfma_qk<BF16>(ones_frag, mfrag[qb], s0);
          s1 = mfma_qk<BF16>(ones_frag, mfrag[qb], s1);
        }
      }
    };
    auto read_v = [&]() {
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
    auto second = [&](int qb) {        // O^T[.][qb] += V^T P^T[qb]
#pragma unroll
      for (int ts = 0; ts < 4; ++ts)
#pragma unroll
        for (int db = 0; db < DB; ++db)
          oacc[db][qb] = mfma_qk<PB>(vfr[ts][db], pf[ts][qb], oacc[db][qb]);
    };
    // Softmax numerators, one query per lane.  Fast path: P = exp2(score - m_i) with the
    // reference m_i left alone; the row sum of the fp16-rounded P (what the second product
    // consumes) is accumulated with dot2.  If a lane's sum grows by 2^14 or more (or is not
    // finite), some P left the safe fp16 range: recentre() moves m_i to the tile's row maximum
    // and the numerators are redone from the scores, which are still live.
    auto settle = [&](int qb, floatx16& s0, floatx16& s1, float lnew) {
      // (FOLD: the first tile of a row block keeps the reference at 0 when its sums are of moderate size)
      const bool first = FOLD ? fresh && !(lnew >= 0.25f) : EW && fresh;
      if (__any(first || (EW && l_i[qb] == 0.f) || !(lnew - l_i[qb] < limit[qb]))) {
        recentre<DB, FOLD, EW>(s0, s1, oacc, qb, qk_scale, m_i[qb], l_i[qb], mfrag[qb], fresh, g);
        any_m = 1;
        lnew = softmax_tile<FOLD, PB>(s0, s1, qk_scale, m_i[qb], l_i[qb], pf, qb);
        limit[qb] = sum_limit<EW>(lnew);
      }
      l_i[qb] = lnew;
    };

    floatx16 sa0, sa1, sb0, sb1;
    wait_vm<CPR>();  // K(cur) has landed (V(cur), issued after it, may still be in flight)
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int s = 0; s < KS; ++s) kfr[kb][s] = *reinterpret_cast<const uintx4*>(lds_k + kaddr[kb][s]);
    // EW: the 64 mask bits of this lane's two queries, shifted so that bit 8(i/4) + i%4 (+ 32 for
    // the second key block) is the key of score register i; without EW only a tile with missing keys is `partial`
    unsigned long long mw0 = 0ull, mw1 = 0ull;
    if constexpr (EW) {
      if (partial) { mw0 = lds_bits[ln] >> (4 * g); mw1 = lds_bits[32 + ln] >> (4 * g); }
    }
    // (the count as a value the compiler cannot trace back, or the 32 tests of the word are made before the tile loop
    // and held; made where it is used, so that it occupies no registers in between)
    auto tail_word = [&]() {
      int v = valid;                                              // < 64 here
      asm volatile("" : "+s"(v));
      return ((1ull << v) - 1ull) >> (4 * g);
    };
    lds_wait();      // the K fragments have arrived: the K buffer is free
    mid();
    if (has1) k_copy_all(cbn, tn);
    auto mask_scores = [&](floatx16& s0, floatx16& s1, unsigned long long mw) {
      const unsigned lo = (unsigned)mw, hi = (unsigned)(mw >> 32);
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const unsigned bit = 1u << (8 * (i / 4) + (i % 4));
        s0[i] = (lo & bit) ? s0[i] : -INFINITY;
        s1[i] = (hi & bit) ? s1[i] : -INFINITY;
      }
    };
    // [1]
    scores(0, sa0, sa1);
    mslice(0, sa0, sa1);
    if constexpr (EW || TAIL) { if (partial) mask_scores(sa0, sa1, EW ? mw0 : tail_word()); }
    __builtin_amdgcn_sched_barrier(0);
    // [2]
    scores(1, sb0, sb1);
    float lnew0 = softmax_tile<FOLD, PB>(sa0, sa1, qk_scale, m_i[0], l_i[0], pf, 0);
    constexpr int NSC = 2 * KS;
#pragma unroll
    for (int it = 0; it < NSC; ++it) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);   // one MFMA
      __builtin_amdgcn_sched_group_barrier(0x002, 64 / NSC + 1, 0);   // its share of the VALU work
    }
    __builtin_amdgcn_sched_barrier(0);
    mslice(1, sb0, sb1);
    if constexpr (EW || TAIL) { if (partial) mask_scores(sb0, sb1, EW ? mw1 : tail_word()); }
    settle(0, sa0, sa1, lnew0);
    if (has1) wait_vm<KOPS>(); else wait_vm<0>();  // V(cur) has landed (K(nxt) may be in flight)
    read_v();
    lds_wait();      // the V fragments have arrived: the V buffer is free
    if (copy_v) v_copy_all(cbn);
    // [3]
    second(0);
    float lnew1 = softmax_tile<FOLD, PB>(sb0, sb1, qk_scale, m_i[1], l_i[1], pf, 1);
#pragma unroll
    for (int it = 0; it < 4 * DB; ++it) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, 64 / (4 * DB) + 1, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    settle(1, sb0, sb1, lnew1);
    fresh = false;
    // [4]
    second(1);
    __builtin_amdgcn_sched_barrier(0);
  };

  // Number of entries r in [0, nb] with rp[r] <= x, for two values of x at once.  The row pointers
  // ascend, so this is a search; it is done in two rounds of one load per lane (64 evenly spaced
  // entries, then the entries between two of them) instead of a chain of dependent scalar loads.
  // Also returns the entries around x: s = rp[c - 1] (the last one <= x) and e = rp[c] (c <= nb).
  // (The entries are compared as rp[r] + gap * r, their positions on the axis the ranges are cut on, moved by
  // the head's first tile; gap = 0: plain tile offsets.)
  auto count_le2 = [&](int64_t x0, int64_t x1, int gap, int& c0, int& c1, int& s0, int& e0, int& s1, int& e1) {
    const int32_t* rpg_ = prm.row_ptr + (int64_t)mh * nb;
    const int step = (nb + 64) / 64;
    auto key = [&](int i, int v) { return (int64_t)v + (int64_t)gap * i; };
    if (step >= 64) {     // very long sequences: plain binary searches
      int lo = -1, hi = nb + 1;
      while (hi - lo > 1) { const int mid = (lo + hi) >> 1; if (key(mid, rp[mid]) <= x0) lo = mid; else hi = mid; }
      c0 = hi;
      lo = -1; hi = nb + 1;
      while (hi - lo > 1) { const int mid = (lo + hi) >> 1; if (key(mid, rp[mid]) <= x1) lo = mid; else hi = mid; }
      c1 = hi;
      s0 = c0 > 0 ? rp[c0 - 1] : 0; e0 = c0 <= nb ? rp[c0] : 0x7fffffff;
      s1 = c1 > 0 ? rp[c1 - 1] : 0; e1 = c1 <= nb ? rp[c1] : 0x7fffffff;
      return;
    }
    const int i1 = lane * step;
    const bool in1 = i1 <= nb;
    const int v1 = in1 ? rpg_[i1] : 0x7fffffff;
    const int a0 = __builtin_popcountll(__ballot(in1 && key(i1, v1) <= x0)), a1 = __builtin_popcountll(__ballot(in1 && key(i1, v1) <= x1));
    const int b0 = (a0 > 0 ? a0 - 1 : 0) * step, b1 = (a1 > 0 ? a1 - 1 : 0) * step;
    const int j0 = b0 + lane, j1 = b1 + lane;
    // (lane `step` holds the next evenly spaced entry, which is > x: it does not count, but may be e)
    const bool in_w0 = lane <= step && j0 <= nb, in_w1 = lane <= step && j1 <= nb;
    const int w0 = in_w0 ? rpg_[j0] : 0x7fffffff;
    const int w1 = in_w1 ? rpg_[j1] : 0x7fffffff;
    const int k0 = a0 > 0 ? __builtin_popcountll(__ballot(in_w0 && key(j0, w0) <= x0)) : 0;
    const int k1 = a1 > 0 ? __builtin_popcountll(__ballot(in_w1 && key(j1, w1) <= x1)) : 0;
    c0 = b0 + k0;
    c1 = b1 + k1;
    s0 = __builtin_amdgcn_readfirstlane(__shfl(w0, k0 > 0 ? k0 - 1 : 0)); e0 = __builtin_amdgcn_readfirstlane(__shfl(w0, k0));
    s1 = __builtin_amdgcn_readfirstlane(__shfl(w1, k1 > 0 ? k1 - 1 : 0)); e1 = __builtin_amdgcn_readfirstlane(__shfl(w1, k1));
  };

  int* ctr = reinterpret_cast<int*>(ml + NW * 2 * 64);
  int* lcols = ONE ? reinterpret_cast<int*>(lds + C::WAVE_LDS) : ctr + 16;
  // The column indices of the range are staged in LDS: a scalar load per tile would put its whole
  // latency in front of the tile's first LDS wait (scalar loads return out of order, so any wait
  // on the shared counter becomes a wait for all of them).
  typedef const unsigned char __attribute__((address_space(4)))* cbyte_ptr_t;
  // entry t of the column list as staged: column block in the low bits, "partly set" in bit 30
  auto flagged_col = [&](int t) {
    int c = cols[t];
    if constexpr (EW) c |= (int)((cbyte_ptr_t)(uintptr_t)prm.tile_partial)[t] << 30;
    return c;
  };
  constexpr int COL_MASK = 0x3fffffff;
  auto is_partial = [&](int c) { return EW ? (c >> 30) != 0 : TAIL && c == tail_cb; };
  auto stage_cols = [&](int t_lo, int t_hi) {
    for (int i = threadIdx.x; i < t_hi - t_lo && i < COLS_CAP; i += NW * 64) {
      int c = prm.col_idx[t_lo + i];
      if constexpr (EW) c |= (int)prm.tile_partial[t_lo + i] << 30;     // EW: "partly set" rides in bit 30
      lcols[i] = c;
    }
  };

  void* obase = out_base(prm, b, h);
  auto exists = [&](int64_t qrow) { return !TAIL || qrow < prm.N; };
  // normalise and write a row block that this wavefront has run alone
  auto write_row = [&](int row) {
    const int lane_o = fresh_lane(lane), ln = lane_o & 31, g = lane_o >> 5;
    float lsum[2];
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) lsum[qb] = l_i[qb] + __shfl_xor(l_i[qb], 32);
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) {
      const float inv = row_inverse<EW>(lsum[qb]);
      const int64_t qrow = (int64_t)(row * 64 + qb * 32 + ln);
      if (!exists(qrow)) continue;
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int i4 = 0; i4 < 4; ++i4)
          store_out4<BF16>(obase, qrow * prm.os[2] + 32 * db + 8 * i4 + 4 * g, prm.out_f32,
                           oacc[db][qb][4 * i4] * inv, oacc[db][qb][4 * i4 + 1] * inv,
                           oacc[db][qb][4 * i4 + 2] * inv, oacc[db][qb][4 * i4 + 3] * inv);
      if (prm.lse != nullptr && g == 0)
        prm.lse[((int64_t)bh * prm.N) + qrow] = row_lse(m_i[qb], lsum[qb]);
    }
  };
  // row block without kept tiles: O = 0, lse = -inf
  auto write_empty_row = [&](int row) {
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) {
      const int64_t qrow = (int64_t)(row * 64 + qb * 32 + ln);
      if (!exists(qrow)) continue;
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int i4 = 0; i4 < 4; ++i4)
          store_out4<BF16>(obase, qrow * prm.os[2] + 32 * db + 8 * i4 + 4 * g, prm.out_f32, 0.f, 0.f, 0.f, 0.f);
      if (prm.lse != nullptr && g == 0) prm.lse[((int64_t)bh * prm.N) + qrow] = -INFINITY;
    }
  };

  // Whole row blocks [r_lo, r_hi), one wavefront each: handed out through the LDS counter *rctr
  // (set to r_lo + 2 NW beforehand), written directly, nothing to merge.
  auto run_rows = [&](int r_lo, int r_hi, int* rctr, auto&& col_of) {
    // Tickets r_lo, r_lo + 1, ... stand for the row blocks r_hi - 1, r_hi - 2, ...: with block-causal
    // masks the late row blocks are the long ones, and the long ones should not come last.
    int tick = r_lo + w, tick_next = r_lo + NW + w;   // the first two rounds are fixed
    int kdone = -1;                                    // tile whose K and V copies were issued ahead
    while (tick < r_hi) {
      int drawn = 0;
      if (lane == 0) drawn = atomicAdd(rctr, 1);       // the row block after next
      const int row = r_lo + r_hi - 1 - tick, row_next = r_lo + r_hi - 1 - tick_next;
      const int ta = rp[row], tb = rp[row + 1];
      // first tile of the next row block of this wavefront (prefetched under the last tile)
      const int tn = tick_next < r_hi ? rp[row_next] : 0;
      const bool next_has = tick_next < r_hi && rp[row_next + 1] > tn;
      if (ta < tb) {
        int cx = __builtin_amdgcn_readfirstlane(col_of(ta));      // current tile: column block | flag
        if (kdone != ta) {
          k_copy_all(cx & COL_MASK, ta);
          v_copy_all(cx & COL_MASK);
        }
        reset_acc();
        load_q(row);
        for (int j = ta; j < tb; ++j) {
          const bool last = j + 1 == tb;
          const bool has1 = !last || next_has;
          const int cxn = has1 ? __builtin_amdgcn_readfirstlane(col_of(last ? tn : j + 1)) : 0;
          tile(has1, cxn & COL_MASK, last ? tn : j + 1, has1, is_partial(cx), [] {});
          cx = cxn;
        }
        kdone = next_has ? tn : -1;
        write_row(row);
      } else {
        write_empty_row(row);
      }
      tick = tick_next;
      tick_next = __builtin_amdgcn_readfirstlane(drawn);
    }
  };

  // One wavefront: a part of a row block that several workgroups share is published and counted in as in the other mode
  // below; the last one in reads all parts (its own as well) and sums them in their order.  own: this part's slot;
  // parts(first, count): the number of parts and where they begin; slot_of(i, first): part i.
  auto share_row = [&](int row, float* own, auto&& parts, auto&& slot_of) {
    float lsum[2], M[2];
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) {
      lsum[qb] = l_i[qb] + __shfl_xor(l_i[qb], 32);
      M[qb] = lsum[qb] == 0.f ? -INFINITY : m_i[qb];      // (a sum that is not a number stays in)
    }
    const int lane_p = fresh_lane(lane), ln = lane_p & 31, g = lane_p >> 5;
    unsigned long long* arrivals = prm.flags + (int64_t)bh * nb + row;
    unsigned long long seen = __hip_atomic_load(arrivals, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    static_assert(DB == 2, "four accumulators");
    matrix_wait(oacc[0][0], oacc[0][1], oacc[1][0], oacc[1][1]);
#pragma unroll
    for (int quad = 0; quad < D / 4; ++quad) {
      const int idx = 4 * quad;
      const floatx16& o = oacc[idx / 32][(idx / 16) & 1];
      coherent_store4(own + idx * 64 + lane_p * 4, o[idx & 15], o[(idx & 15) + 1], o[(idx & 15) + 2], o[(idx & 15) + 3]);
    }
    if (g == 0) {
#pragma unroll
      for (int qb = 0; qb < 2; ++qb) {
        coherent_store(own + 64 * D + qb * 32 + ln, M[qb]);
        coherent_store(own + 64 * D + 64 + qb * 32 + ln, lsum[qb]);
      }
    }
    int first = 0, nparts = 0;
    parts(first, nparts);
    wait_vm<0>();                             // every store of the part has been acknowledged
    int counted_v = 0;
    if (lane == 0) {
      unsigned long long old = seen;
      for (;;) {     // (ends: the counter only changes when another part is counted, at most nparts times)
        const unsigned long long want = (old >> 16) == prm.epoch ? old + 1 : ((prm.epoch << 16) | 1ull);
        if (__hip_atomic_compare_exchange_strong(arrivals, &old, want, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT)) {
          counted_v = (int)(want & 0xffffull);
          break;
        }
      }
    }
    if (__builtin_amdgcn_readfirstlane(counted_v) != nparts) return;
    float Ms[2] = {-INFINITY, -INFINITY}, Ls[2] = {0.f, 0.f};
    reset_acc();
    for (int p = first; p < first + nparts; ++p) {
      const float* sp = slot_of(p, first);
      float sc_own[2], sc_p[2];
#pragma unroll
      for (int qb = 0; qb < 2; ++qb) {
        const float mp = coherent_load(sp + 64 * D + qb * 32 + ln), lp = coherent_load(sp + 64 * D + 64 + qb * 32 + ln);
        const float mn = fmaxf(Ms[qb], mp);     // a side without mass has maximum -inf and weight 0
        sc_own[qb] = Ms[qb] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(Ms[qb] - mn);
        sc_p[qb] = mp == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mp - mn);
        Ls[qb] = Ls[qb] * sc_own[qb] + lp * sc_p[qb];
        Ms[qb] = mn;
      }
      // The whole part at once, 16 KB, in one round trip, where nearly every row block is shared (four of them, two parts a row block: 8 heads
      // N = 17536 keep 0.1 93.4 -> 90.1 us, 16 heads N = 8192 keep 0.1 51.1 -> 48.4, 24 heads N = 4096 dense 132.7 -> 127.3); a quarter per
      // round trip where it is rare, or spills registers (elementwise masks).
      constexpr int PER = MODE == WAVE && !EW ? D / 4 : 4;
#pragma unroll
      for (int q4 = 0; q4 < D / 4; q4 += PER) {
        floatx4 ld[PER];
        if constexpr (PER == 4) coherent_load4x4(sp + q4 * 256 + lane_p * 4, ld[0], ld[1], ld[2], ld[3]);
        else coherent_load4x16(sp + lane_p * 4, ld);
#pragma unroll
        for (int e = 0; e < 4 * PER; ++e) {
          const int idx = 4 * q4 + e, qb = (idx / 16) & 1;
          oacc[idx / 32][qb][idx & 15] = oacc[idx / 32][qb][idx & 15] * sc_own[qb] + sc_p[qb] * ld[e / 4][e & 3];
        }
      }
    }
    // (write_row sums the two halves of a query)
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) { m_i[qb] = Ms[qb]; l_i[qb] = g == 0 ? Ls[qb] : 0.f; }
    write_row(row);
    // back to zero, so that a replay of this launch (same mark) starts from a clean counter
    if (lane == 0) __hip_atomic_store(arrivals, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };

  if constexpr (ROWS) {
    // ================= one wavefront, one row block =================
    // Row blocks much longer than the others (the rows of text tokens in front of a video, kept whole) would still be
    // walked when all others are done: those above 2.5 times the head's mean length are left to W workgroups per head
    // (wg = nb + p), which cut them into parts (row_parts.h).  Such a workgroup takes the parts p, p + W, ...; the parts of a
    // row block that is cut meet as those of ranges do, in one of W slots each.
    // The W workgroups come when the first row blocks have filled the GPU: in front of them they made a causal launch slower (48
    // heads N = 4096 152 -> 168 us: row blocks then go where a workgroup without work has just ended, long ones side by
    // side), behind all others the parts of a small launch are a tail (24 heads, below: 114 us).
    // bf16, us before / after, and the ranges of workgroups (MODE 0) that this mode replaced:
    //   48 heads N = 17792, keep 0.05, row blocks 0-3 and columns 0-3 kept whole   735 / 415   643     keep 0.2  1238 / 1008   1639
    //   24 heads N = 8192,  keep 0.1,  the same rows and columns                   251 / 101   116     12 heads N = 17792  525 / 172   193
    //   without long row blocks: 48 heads keep 0.05 295 / 285, keep 0.2 913 / 913; 24 heads keep 0.1 75 / 75, causal 299 / 293
    int row = wg, ta, tb, parts = 1, slot0 = 0, slot_own = 0, item = wg - nb, part_len = 0, T = 0;
    auto is_long = [&](int len) { return is_long_row(len, T, nb); };
    // (the head's tiles; the pointer as a value the compiler cannot trace back: looked up only where needed)
    auto total = [&]() {
      cint_ptr_t p = rp;
      asm volatile("" : "+s"(p));
      return p[nb] - p[0];
    };
    auto find = [&]() {       // the row block, tiles and slots of `item`; false if there is no such item
      const int32_t* rpg = prm.row_ptr + (int64_t)mh * nb;
      int items = 0, slots = 0;
      for (int r0 = 0; r0 < nb; r0 += 64) {
        const int r = r0 + fresh_lane(lane), len = r < nb ? rpg[r + 1] - rpg[r] : 0;
        for (unsigned long long left = __ballot(is_long(len)); left != 0ull; left &= left - 1ull) {
          const int at = __builtin_ctzll(left), row_len = __builtin_amdgcn_readlane(len, at);
          const int n = parts_of_row(row_len, part_len);
          if (item < items + n) {
            const int part = item - items;
            row = r0 + at;
            ta = rp[row] + part_begin(row_len, n, part);
            tb = rp[row] + part_begin(row_len, n, part + 1);
            parts = n;
            slot0 = slots;
            slot_own = slots + part;
            return true;
          }
          items += n;
          if (n > 1) slots += n;
        }
      }
      return false;
    };
    if (wg < nb) {
      ta = rp[wg]; tb = rp[wg + 1];
      if (ta == tb) { write_empty_row(wg); return; }
      if (prm.W > 0 && tb - ta > LONG_ROW_MIN) {
        T = total();
        if (is_long(tb - ta)) return;
      }
    } else {
      T = total();
      const int32_t* rpg = prm.row_ptr + (int64_t)mh * nb;
      int sum = 0, count = 0;
      for (int r = lane; r < nb; r += 64) {
        const int len = rpg[r + 1] - rpg[r];
        if (is_long(len)) { sum += len; ++count; }
      }
      if (!__any(count > 0)) return;
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) { sum += __shfl_xor(sum, off); count += __shfl_xor(count, off); }
      part_len = long_part_tiles(__builtin_amdgcn_readfirstlane(sum), __builtin_amdgcn_readfirstlane(count), prm.W, T / nb);
      if (!find()) return;
    }
    for (;;) {
      int cx = flagged_col(ta);                                // current tile: column block | flag
      k_copy_all(cx & COL_MASK, ta);
      v_copy_all(cx & COL_MASK);
      stage_cols(ta, tb);
      auto col_of = [&](int t) { return t - ta < COLS_CAP ? lcols[t - ta] : flagged_col(t); };
      reset_acc();
      load_q(row);
      for (int j = ta; j < tb; ++j) {
        const bool has1 = j + 1 < tb;
        const int cxn = has1 ? __builtin_amdgcn_readfirstlane(col_of(j + 1)) : 0;
        tile(has1, cxn & COL_MASK, j + 1, has1, is_partial(cx), [] {});
        cx = cxn;
      }
      if (parts == 1) {
        write_row(row);
      } else {
        auto slot_at = [&](int i) { return prm.ws + ((int64_t)bh * prm.W + i) * partial_floats(D); };
        share_row(row, slot_at(slot_own), [&](int& first, int& count) { first = slot0; count = parts; },
                  [&](int p, int) { return slot_at(p); });
      }
      if (wg < nb) return;
      item += prm.W;
      if (!find()) return;
    }
  } else if constexpr (MODE == WAVE) {
    // ================= one wavefront, one range =================
    // The range's last row block is walked first, then the others from the range's beginning: what is kept of the last row block begins
    // in an early column, and the rest of the first one goes on about where that has ended (row blocks of equal length: a range is one of
    // them and a bit).  So all wavefronts of an XCD walk the columns from the first to the last at the same time, whatever row block their range
    // begins in, and the tiles at work at once fit its L2, which K and V of a long head do not.  In list order / so, us:
    //   8 heads N = 17536 dense 718 / 695, N = 24000 dense 1381 / 1287, keep 0.1 161 / 154; 5 heads N = 32000 keep 0.5 915 / 745, keep 0.1 209 / 171;
    //   6 heads N = 17536 keep 0.1 80 / 74; 9 heads N = 20032 keep 0.5 555 / 531; within the L2: 10 heads N = 12000 dense 456 / 427, 16 heads
    //   N = 12032 dense 663 / 655, N = 8192 keep 0.1 54 / 51, causal keep 0.2 91 / 93 and 54 / 54, 24 heads N = 4096 keep 0.1 29.6 / 29.7.
    // first row block of the range: largest r with rp[r] <= g0 < rp[r+1]
    // A range boundary within `snap` tiles of an end of the row block it falls in moves to that end
    // (the nearer one): sharing a row block costs a merge, a published part and a pull, several
    // tiles' worth each, and row blocks of up to 2 `snap` tiles are never shared.  Every workgroup
    // applies the same rule with the same distance to both of its boundaries, so the ranges still tile the list.
    int r, g0, g1, start, r_first = 0, r_last = 0;      // start: the first tile walked
    {
      // the row blocks in which the two ends of the range lie (positions behind a row block's tiles count as
      // its end), then the tiles themselves
      int c0, c1, s0, e0, s1, e1;
      count_le2(x0 + hs.lo, x1 + hs.lo, hs.gap, c0, c1, s0, e0, s1, e1);
      r = c0 - 1;
      g0 = tile_of_pos(hs, x0, r, s0, e0);
      const int n0 = snap_boundary(snap, g0, s0, e0);
      if (n0 >= e0) ++r;
      g0 = n0;
      if (x1 < hs.X) {
        g1 = tile_of_pos(hs, x1, c1 - 1, s1, e1);
        g1 = snap_boundary(snap, g1, s1, e1);
      } else {
        g1 = hs.lo + hs.T;
      }
      if (g0 >= g1) return;
      start = g0;
      if (x1 < hs.X && s1 > g0 && s1 < g1) { start = s1; r_last = c1 - 1; }
    }
    // two slots per workgroup: a range can end inside one row block (that part goes to slot 1: it holds the row
    // block's first tiles) after having begun inside another (slot 0)
    auto wg_slot = [&](int p, bool head) { return prm.ws + (((int64_t)bh * prm.W + p) * 2 + (head ? 1 : 0)) * partial_floats(D); };
    int cx = flagged_col(start);                               // current tile: column block | flag
    k_copy_all(cx & COL_MASK, start);
    v_copy_all(cx & COL_MASK);
    stage_cols(g0, g1);
    auto col_of = [&](int t) { return t - g0 < COLS_CAP ? lcols[t - g0] : flagged_col(t); };
    int t = start, end = g1;
    bool wrapped = start == g0;
    if (!wrapped) { r_first = r; r = r_last; }
    for (;;) {
      if (t >= end) {
        if (wrapped) break;
        wrapped = true;
        t = g0;
        end = start;
        r = r_first;
      }
      const int row_s = rp[r], row_e = rp[r + 1];
      if (row_e <= t) { ++r; continue; }          // row block without kept tiles in the range
      const int seg_b = row_e < end ? row_e : end;
      reset_acc();
      load_q(r);
      for (int j = t; j < seg_b; ++j) {           // (the next tile is prefetched across the end of the row block)
        const bool has1 = j + 1 < end || !wrapped;
        const int nxt = j + 1 < end ? j + 1 : g0;
        const int cxn = has1 ? __builtin_amdgcn_readfirstlane(col_of(nxt)) : 0;
        tile(has1, cxn & COL_MASK, nxt, has1, is_partial(cx), [] {});
        cx = cxn;
      }
      if (t == row_s && seg_b == row_e) {
        write_row(r);
      } else {
        share_row(r, wg_slot(wg, t == row_s), [&](int& first, int& count) {
          const int64_t xrow = row_pos(hs, r, row_s);
          int pl_ = split_of_pos(hs, xrow + (row_e - 1 - row_s)), pf_ = split_of_pos(hs, xrow);
          while (pl_ > pf_ && snap_boundary(snap, tile_of_pos(hs, split_pos(hs, pl_), r, row_s, row_e), row_s, row_e) >= row_e) --pl_;
          while (pf_ < pl_ && snap_boundary(snap, tile_of_pos(hs, split_pos(hs, pf_ + 1), r, row_s, row_e), row_s, row_e) <= row_s) ++pf_;
          first = pf_;
          count = pl_ - pf_ + 1;
        }, [&](int p, int first) { return wg_slot(p, p == first); });
      }
      t = seg_b;
      ++r;
    }
  } else {
    // ================= all wavefronts on one row block at a time =================
    // Tiles of the range are handed out to the wavefronts dynamically (the LDS counter), because
    // the two wavefronts of a SIMD do not progress at the same rate: each wavefront owns a current
    // tile `cur` and has already drawn its next one `nxt`, so that it can prefetch it.  Tiles are
    // drawn in list order, so a wavefront's tiles increase, and `cur >= seg_b` means "nothing left
    // for me in this row block".  kdone / vdone name the tile whose copy into this wavefront's
    // K / V buffer has been issued; no copy is issued across the merge of a row block, which
    // borrows both buffers of every wavefront (one exchange round for the whole accumulator).
    // first row block of the range: largest r with rp[r] <= g0 < rp[r+1]
    // A range boundary within `snap` tiles of an end of the row block it falls in moves to that end
    // (the nearer one): sharing a row block costs a merge, a published part and a pull, several
    // tiles' worth each, and row blocks of up to 2 `snap` tiles are never shared.  Every workgroup
    // applies the same rule with the same distance to both of its boundaries, so the ranges still tile the list.
    if (g0 == g1) {
      // the row blocks in which the two ends of the range lie (positions behind a row block's tiles count as
      // its end), then the tiles themselves
      int c0, c1, s0, e0, s1, e1;
      count_le2(x0 + hs.lo, x1 + hs.lo, hs.gap, c0, c1, s0, e0, s1, e1);
      r = c0 - 1;
      g0 = tile_of_pos(hs, x0, r, s0, e0);
      const int n0 = snap_boundary(snap, g0, s0, e0);
      if (n0 >= e0) ++r;
      g0 = n0;
      if (x1 < hs.X) {
        g1 = tile_of_pos(hs, x1, c1 - 1, s1, e1);
        g1 = snap_boundary(snap, g1, s1, e1);
      } else {
        g1 = hs.lo + hs.T;
      }
      if (g0 >= g1) return;
    }
    int kdone = -1, vdone = -1;
    // The copies of this wavefront's first tile are asked for before anything else (its column index by one
    // scalar load), so that they travel while the column list is staged and Q is read.
    if (g0 + w < g1) {
      const int c0 = flagged_col(g0 + w) & COL_MASK;
      k_copy_all(c0, g0 + w);
      v_copy_all(c0);
      kdone = vdone = g0 + w;
    }
    stage_cols(g0, g1);
    if (threadIdx.x == 0) { ctr[0] = g0 + 2 * NW; ctr[3] = 0; }
    __syncthreads();
    auto col_of = [&](int t) { return t - g0 < COLS_CAP ? lcols[t - g0] : flagged_col(t); };
    int cur = g0 + w, nxt = g0 + NW + w;      // the first two rounds are fixed
    int cb_nxt = nxt < g1 ? __builtin_amdgcn_readfirstlane(col_of(nxt)) : 0;   // column block of tile nxt
    int t = g0;
    const int32_t* rpg = prm.row_ptr + (int64_t)mh * nb;
    while (t < g1) {
      const int row_s = rp[r], row_e = rp[r + 1];
      if (row_e <= t) { ++r; continue; }          // row block without kept tiles in the range
      // A run of short row blocks that lie completely inside the range is not worth a merge per
      // row block: such a run is done one row block per wavefront.  Every wavefront looks at the
      // next 64 row blocks (one per lane) and comes to the same decision.
      if (t == row_s && row_e <= g1 && row_e - row_s <= C::SHORT_ROW) {
        const int idx = r + lane;
        const int rs_i = idx < nb ? rpg[idx] : 0, re_i = idx < nb ? rpg[idx + 1] : 0x7fffffff;
        const bool ok_i = idx < nb && re_i <= g1 && re_i - rs_i <= C::SHORT_ROW;
        const unsigned long long okm = __ballot(ok_i);
        const int cnt = ~okm == 0ull ? 64 : __builtin_ctzll(~okm);        // leading run of short inner row blocks
        const bool in_run = lane < cnt;
        const int bn = __builtin_popcountll(__ballot(in_run && re_i > rs_i));   // ... with kept tiles
        int maxlen = in_run ? re_i - rs_i : 0;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) { const int o = __shfl_xor(maxlen, off); maxlen = o > maxlen ? o : maxlen; }
        maxlen = __builtin_amdgcn_readfirstlane(maxlen);
        // worth it when the run keeps the wavefronts busy, or when its row blocks are short
        // against the cost of a merge (about three tiles per wavefront)
        const bool batch = bn >= NW || (bn == 3) || (bn == 2 && maxlen < 3 * NW) || (bn == 1 && maxlen < NW);
        if (batch) {
          const int r2 = r + cnt, t2 = __builtin_amdgcn_readfirstlane(__shfl(re_i, cnt - 1));
          wait_vm<0>();                 // prefetches of the tile hand-out below are abandoned
          __syncthreads();              // everybody has left the previous run and the previous merge
          if (threadIdx.x == 0) { ctr[2] = r + 2 * NW; ctr[0] = t2 + 2 * NW; }
          __syncthreads();
          run_rows(r, r2, ctr + 2, col_of);
          cur = t2 + w; nxt = t2 + NW + w;
          cb_nxt = nxt < g1 ? __builtin_amdgcn_readfirstlane(col_of(nxt)) : 0;
          kdone = -1; vdone = -1;
          t = t2; r = r2;
          continue;
        }
      }
      const int seg_a = t, seg_b = row_e < g1 ? row_e : g1;
      const bool mine = cur < seg_b;      // this wavefront processes at least one tile of the row block
      reset_acc();
      if (mine) {
        int cx = __builtin_amdgcn_readfirstlane(col_of(cur));     // current tile: column block | flag
        if (kdone != cur) { k_copy_all(cx & COL_MASK, cur); kdone = cur; }
        if (vdone != cur) { v_copy_all(cx & COL_MASK); vdone = cur; }
        load_q(r);
        while (cur < seg_b) {
          // draw the tile after next; the value is picked up inside the tile
          int drawn = 0;
          if (lane == 0) drawn = atomicAdd(ctr, 1);
          // the next tile is only prefetched inside the row block: the merge at its end borrows both buffers
          const bool has1 = nxt < seg_b, copy_v = has1;
          int nn = 0, cb_nn_v = 0;
          tile(has1, cb_nxt & COL_MASK, nxt, copy_v, is_partial(cx), [&] {
            // (deterministic: every wavefront takes every NW-th tile, whatever its pace)
            nn = prm.deterministic ? nxt + NW : __builtin_amdgcn_readfirstlane(drawn);
            cb_nn_v = nn < g1 ? col_of(nn) : 0;     // looked up now, needed at the end of the tile
          });
          if (has1) kdone = nxt;
          if (copy_v) vdone = nxt;
          cur = nxt;
          cx = cb_nxt;
          nxt = nn;
          cb_nxt = __builtin_amdgcn_readfirstlane(cb_nn_v);
        }  // tiles of this wavefront
      }
      // ---- merge the wavefronts' results of this row block through LDS ----
      // Each wavefront publishes (m, l) per query and, round by round, R accumulator registers in
      // its own V buffer ([register][lane] floats); in every round each wavefront reduces QPW
      // groups of 4 registers (4 consecutive head-dimension values of one query per lane) over all
      // contributing wavefronts and writes them out.
      {
        // (a wavefront without tiles in the range's first row block may still have its first tile's copies in
        // flight: the merge borrows the tile buffers, so they are waited for and asked for again afterwards)
        if (!mine) { wait_vm<0>(); kdone = -1; vdone = -1; }
        float lsum[2];
#pragma unroll
        for (int qb = 0; qb < 2; ++qb) lsum[qb] = l_i[qb] + __shfl_xor(l_i[qb], 32);
        if (g == 0) {
#pragma unroll
          for (int qb = 0; qb < 2; ++qb) {
            const bool mass = mine && lsum[qb] != 0.f;      // (a sum that is not a number stays in)
            ml[(w * 2 + 0) * 64 + qb * 32 + ln] = mass ? m_i[qb] : -INFINITY;
            ml[(w * 2 + 1) * 64 + qb * 32 + ln] = mass ? lsum[qb] : 0.f;
          }
        }
        // A row block cut by range boundaries has one part per workgroup that holds tiles of it.  Every
        // such workgroup publishes its part and then counts itself in; the one that finds all the
        // others counted merges the parts and writes the row block.  Nobody waits for anybody, so
        // the result does not depend on which workgroups are resident at the same time.
        const bool has_head = seg_a == row_s, has_tail = seg_b == row_e;
        const bool full = has_head && has_tail;
        float wgt[NW][2];   // weight of wavefront p's partial for this lane's query of block qb
        float M[2], L[2];
        float keep[C::ROUNDS][C::QPW][4];   // this wavefront's share of the workgroup's part
        // (parts travel 16 bytes per lane and access: N = 17536, one head, against 4 bytes: dense 101.6 -> 101.0 us, keep 0.25
        // 41.8 -> 41.1, keep 0.05 20.6 -> 20.0)
        // A zero the compiler cannot see through (ctr[3] stays 0): the per-lane addresses into the
        // workspace do not change from row block to row block and would otherwise be computed
        // once, up front, and occupy registers throughout the tile loops.
        typedef volatile int __attribute__((address_space(3)))* lds_vint_ptr_t;
        const int zero = *(lds_vint_ptr_t)(lds_ptr_t)(ctr + 3);
        // two slots per workgroup: a range can end inside one row block (that part goes to slot 1: it
        // holds the row block's first tiles) after having begun inside another (slot 0)
        auto slot_of = [&](int p, bool head) {
          return prm.ws + (((int64_t)bh * prm.W + p) * 2 + (head ? 1 : 0)) * partial_floats(D) + zero;
        };
        float* slot = slot_of(wg, has_head);
        // A part's holder looks at the arrival counter now: the value is only the first guess of the
        // compare-and-swap below, and its round trip runs beside the merge instead of behind it.
        unsigned long long* arrivals = prm.flags + (int64_t)bh * nb + r;
        unsigned long long seen = 0;
        if (!full && threadIdx.x == 0) seen = __hip_atomic_load(arrivals, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (int rd = 0; rd < C::ROUNDS; ++rd) {
          {
            // every wavefront writes (one without tiles of this row block holds zeros), 4 bytes per
            // lane and instruction: wider LDS writes are much slower per byte on this hardware
            float* own = reinterpret_cast<float*>(lds_k);
#pragma unroll
            for (int e = 0; e < C::R; ++e) {
              const int idx = rd * C::R + e;
              own[e * 64 + lane] = oacc[idx / 32][(idx / 16) & 1][idx & 15];
            }
          }
          __syncthreads();
          if (rd == 0) {
#pragma unroll
            for (int qb = 0; qb < 2; ++qb) {
              float mm = -INFINITY;
#pragma unroll
              for (int pw = 0; pw < NW; ++pw) mm = fmaxf(mm, ml[(pw * 2 + 0) * 64 + qb * 32 + ln]);
              float ll = 0.f;
#pragma unroll
              for (int pw = 0; pw < NW; ++pw) {
                const float mp = ml[(pw * 2 + 0) * 64 + qb * 32 + ln];
                const float wp = mp == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mp - mm);
                wgt[pw][qb] = wp;
                ll += wp * ml[(pw * 2 + 1) * 64 + qb * 32 + ln];
              }
              M[qb] = mm; L[qb] = ll;
            }
          }
#pragma unroll
          for (int tq = 0; tq < C::QPW; ++tq) {
            const int quad = w * C::QPW + tq;              // group of 4 registers within this round
            const int idx0 = rd * C::R + 4 * quad;         // accumulator register index (db, qb, i16)
            const int db = idx0 / 32, qb = (idx0 / 16) & 1, i4 = (idx0 & 15) / 4;
            float x[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int pw = 0; pw < NW; ++pw) {
              const float* src = reinterpret_cast<const float*>(lds + pw * C::WAVE_LDS);
#pragma unroll
              for (int e = 0; e < 4; ++e) x[e] += wgt[pw][qb] * src[(4 * quad + e) * 64 + lane];
            }
            if (full) {
              const float inv = row_inverse<EW>(L[qb]);
              const int64_t qrow = (int64_t)(r * 64 + qb * 32 + ln);
              if (exists(qrow))
                store_out4<BF16>(obase, qrow * prm.os[2] + 32 * db + 8 * i4 + 4 * g, prm.out_f32, x[0] * inv, x[1] * inv,
                               x[2] * inv, x[3] * inv);
            } else {
              coherent_store4(slot + idx0 * 64 + lane * 4, x[0], x[1], x[2], x[3]);   // (a part is laid out [quad][lane][4])
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) keep[rd][tq][e] = x[e];
          }
          __syncthreads();
        }
        if (full) {
          if (w == 0 && g == 0 && prm.lse != nullptr) {
#pragma unroll
            for (int qb = 0; qb < 2; ++qb)
              if (exists((int64_t)(r * 64 + qb * 32 + ln))) prm.lse[((int64_t)bh * prm.N) + (int64_t)(r * 64 + qb * 32 + ln)] =
                  row_lse(M[qb], L[qb]);
          }
        } else {
          if (w == 0 && g == 0) {
#pragma unroll
            for (int qb = 0; qb < 2; ++qb) {
              coherent_store(slot + 64 * D + qb * 32 + ln, M[qb]);
              coherent_store(slot + 64 * D + 64 + qb * 32 + ln, L[qb]);
            }
          }
          // The workgroups pf .. pl hold the parts of this row block: pf is the one before the first range
          // boundary that stays inside the row block (boundaries close to an end move there), pl the one
          // after the last.  Every holder computes the same two numbers.
          int pl_, pf_;
          if (own_parts_n > 0) {
            pf_ = own_first;
            pl_ = own_first + own_parts_n - 1;
          } else {
            const int64_t xrow = row_pos(hs, r, row_s);
            pl_ = split_of_pos(hs, xrow + (row_e - 1 - row_s)); pf_ = split_of_pos(hs, xrow);
            while (pl_ > pf_ && snap_boundary(snap, tile_of_pos(hs, split_pos(hs, pl_), r, row_s, row_e), row_s, row_e) >= row_e) --pl_;
            while (pf_ < pl_ && snap_boundary(snap, tile_of_pos(hs, split_pos(hs, pf_ + 1), r, row_s, row_e), row_s, row_e) <= row_s) ++pf_;
          }
          const int nparts = pl_ - pf_ + 1;
          // The part is counted in once every wavefront's stores have been acknowledged (vmcnt 0, then the
          // barrier).  Every access to a part, stores here and loads below, is itself an access at device
          // scope: it is served by the memory all compute units share, never by a cache that only
          // some of them see.  The counter update is therefore relaxed: release / acquire order on it
          // would add a write-back and an invalidation of this die's whole L2, measured at 9 us per
          // launch (keep 0.1, N = 17536: 31 -> 41 us), to order accesses that are already ordered.
          // The counter holds (launch mark << 16 | parts counted); stale contents carry another mark.
          wait_vm<0>();
          __syncthreads();
          if (threadIdx.x == 0) {
            unsigned long long old = seen;
            for (;;) {     // (ends: the counter only changes when another part is counted, at most nparts times)
              const unsigned long long want = (old >> 16) == prm.epoch ? old + 1 : ((prm.epoch << 16) | 1ull);
              if (__hip_atomic_compare_exchange_strong(arrivals, &old, want, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                       __HIP_MEMORY_SCOPE_AGENT)) {
                ctr[4] = (int)(want & 0xffffull);
                break;
              }
            }
          }
          __syncthreads();
          const int counted = __builtin_amdgcn_readfirstlane(*(lds_vint_ptr_t)(lds_ptr_t)(ctr + 4));
          if (counted == nparts) {
            // last one in: every part is in memory.  They are summed in the order of the ranges, whoever
            // does it, so the result does not depend on the order of arrival.
            float Ms[2] = {-INFINITY, -INFINITY}, Ls[2] = {0.f, 0.f}, acc[C::ROUNDS][C::QPW][4];
#pragma unroll
            for (int rd = 0; rd < C::ROUNDS; ++rd)
#pragma unroll
              for (int tq = 0; tq < C::QPW; ++tq)
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[rd][tq][e] = 0.f;
            for (int p = pf_; p <= pl_; ++p) {
              float mp[2], lp[2], dat[C::ROUNDS][C::QPW][4];
              if (p == wg) {
#pragma unroll
                for (int qb = 0; qb < 2; ++qb) { mp[qb] = M[qb]; lp[qb] = L[qb]; }
#pragma unroll
                for (int rd = 0; rd < C::ROUNDS; ++rd)
#pragma unroll
                  for (int tq = 0; tq < C::QPW; ++tq)
#pragma unroll
                    for (int e = 0; e < 4; ++e) dat[rd][tq][e] = keep[rd][tq][e];
              } else {
                const float* sp = slot_of(p, p == pf_);
                // all loads of the part are issued before the first one is waited for (a round trip
                // to the point of coherence costs about a microsecond)
#pragma unroll
                for (int qb = 0; qb < 2; ++qb) {
                  mp[qb] = coherent_load(sp + 64 * D + qb * 32 + ln);
                  lp[qb] = coherent_load(sp + 64 * D + 64 + qb * 32 + ln);
                }
                static_assert(C::ROUNDS == 1 && C::QPW == 4, "four 16-byte loads per lane and part");
                floatx4 ld[4];
                coherent_load4x4(sp + 4 * (w * C::QPW) * 64 + lane * 4, ld[0], ld[1], ld[2], ld[3]);   // ([quad][lane][4]: a quad is 1 KB)
#pragma unroll
                for (int rd = 0; rd < C::ROUNDS; ++rd)
#pragma unroll
                  for (int tq = 0; tq < C::QPW; ++tq)
#pragma unroll
                    for (int e = 0; e < 4; ++e) dat[rd][tq][e] = ld[rd * C::QPW + tq][e];
              }
              float sc_own[2], sc_p[2];
#pragma unroll
              for (int qb = 0; qb < 2; ++qb) {
                const float mn = fmaxf(Ms[qb], mp[qb]);     // a side without mass has maximum -inf and weight 0
                sc_own[qb] = Ms[qb] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(Ms[qb] - mn);
                sc_p[qb] = mp[qb] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mp[qb] - mn);
                Ls[qb] = Ls[qb] * sc_own[qb] + lp[qb] * sc_p[qb];
                Ms[qb] = mn;
              }
#pragma unroll
              for (int rd = 0; rd < C::ROUNDS; ++rd)
#pragma unroll
                for (int tq = 0; tq < C::QPW; ++tq) {
                  const int qb = ((rd * C::R + 4 * (w * C::QPW + tq)) / 16) & 1;
#pragma unroll
                  for (int e = 0; e < 4; ++e) acc[rd][tq][e] = acc[rd][tq][e] * sc_own[qb] + sc_p[qb] * dat[rd][tq][e];
                }
            }
#pragma unroll
            for (int rd = 0; rd < C::ROUNDS; ++rd)
#pragma unroll
              for (int tq = 0; tq < C::QPW; ++tq) {
                const int idx0 = rd * C::R + 4 * (w * C::QPW + tq);
                const int db = idx0 / 32, qb = (idx0 / 16) & 1, i4 = (idx0 & 15) / 4;
                const float inv = row_inverse<EW>(Ls[qb]);
                const int64_t qrow = (int64_t)(r * 64 + qb * 32 + ln);
                if (exists(qrow)) store_out4<BF16>(obase, qrow * prm.os[2] + 32 * db + 8 * i4 + 4 * g, prm.out_f32,
                                 acc[rd][tq][0] * inv, acc[rd][tq][1] * inv, acc[rd][tq][2] * inv, acc[rd][tq][3] * inv);
              }
            if (w == 0 && g == 0 && prm.lse != nullptr) {
#pragma unroll
              for (int qb = 0; qb < 2; ++qb)
                if (exists((int64_t)(r * 64 + qb * 32 + ln))) prm.lse[((int64_t)bh * prm.N) + (int64_t)(r * 64 + qb * 32 + ln)] =
                    row_lse(Ms[qb], Ls[qb]);
            }
            // back to zero, so that a replay of this launch (same mark) starts from a clean counter
            if (threadIdx.x == 0) __hip_atomic_store(arrivals, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          }
        }
      }
      t = seg_b;
      ++r;
    }
  }
}

// A 48-bit number that differs from launch to launch (and, through its start value, from process
// to process); never zero.
unsigned long long next_epoch() {
  static std::atomic<unsigned long long> counter{
      (unsigned long long)std::chrono::steady_clock::now().time_since_epoch().count() * 0x9E3779B97F4A7C15ull};
  unsigned long long e;
  do { e = counter.fetch_add(1) & 0xffffffffffffull; } while (e == 0);
  return e;
}

// Process-wide switch: results that do not depend on the pace of the wavefronts (bsattn_set_deterministic).
static std::atomic<int> deterministic_mode{0};
int set_deterministic(int on) { return deterministic_mode.exchange(on != 0 ? 1 : 0); }
int get_deterministic() { return deterministic_mode.load(); }

int compute_units() {
  static int cached[64] = {0};   // per device; the value never changes, so a race only repeats the query
  int dev = 0, cus = 256;
  if (hipGetDevice(&dev) != hipSuccess) return cus;
  if (dev >= 0 && dev < 64 && cached[dev] > 0) return cached[dev];
  int v = 0;
  if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && v > 0) cus = v;
  if (dev >= 0 && dev < 64) cached[dev] = cus;
  return cus;
}

// How a launch is split at D = 64, by its row blocks against the wavefronts that are resident at once (8 per compute unit).
// From half as many more on a wavefront takes a row block (48 heads of N = 17776, keep 0.3: 2127 -> 1298 us; 24 heads of
// N = 8192 dense 493 -> 425, causal 16 heads of N = 8192, one row block per wavefront, 172 -> 231: not there).  From three
// quarters as many on a wavefront takes a range of the list, with fewer the ranges of whole workgroups are the faster
// ones: they share a row block's merge.  bf16, us, ranges of workgroups / of wavefronts, keep 0.1, 0.3, 1 and block-causal:
//   12 heads N = 8192 (0.75)   53 /  47    92 /  90   247 / 250   137 / 138      8 heads N = 8192 (0.5)   36 / 41   65 / 72   167 / 162    98 / 105
//    9 heads N = 12000 (0.83)  71 /  65   139 / 138   398 / 404   211 / 208      6 heads N = 12000 (0.55) 53 / 52   96 / 98   265 / 270   153 / 153
//   24 heads N = 4096 (0.75)   33 /  31    61 /  55   137 / 135    86 /  77     17 heads N = 4096 (0.53)  30 / 28   47 / 45    99 / 101    66 /  67
//   48 heads N = 2048 (0.75)   26 /  24    40 /  38    85 /  79    54 /  58     56 heads N = 2048 (0.88)  28 / 25   41 / 42    94 /  86    61 /  60
//    5 heads N = 24064 (0.92) 115 / 116   273 / 288   889 / 902   435 / 445    (above 300 row blocks per head: from one per wavefront on)
// With the ranges walked from their last row block on more sizes gain by them, but not with every mask and not in bf16, whose rows have
// fewer first tiles with an exact largest numerator in ranges of wavefronts (20 heads N = 4096 keep 0.5, 6 heads N = 20032 keep 0.15: 2.024e-4 -> 2.036e-4
// and 2.031e-4 -> 2.045e-4 from 64 bits).  fp16, ranges of workgroups / of wavefronts, keep 0.03, 0.1, 0.3, dense, windows of 0.1 and 0.3, row and column
// blocks 0-3 whole in keep 0.05, 0.02 and a diagonal with two whole row blocks:
//   20 heads N = 4096 (0.62)   22 / 22    30 / 29    50 / 54   119 / 116    27 / 25    48 / 48    38 / 43    28 / 36
//   14 heads N = 6656 (0.71)   29 / 23    38 / 38    77 / 71   185 / 185    33 / 39    73 / 67    42 / 50    32 / 43
//    6 heads N = 20032 (0.92)  50 / 42    96 / 86   228 / 211  701 / 649    91 / 83   210 / 197   79 / 82    57 / 66
//    3 heads N = 32000 (0.73)  51 / 52   111 / 108  296 / 264  935 / 825   105 / 103  262 / 247   85 / 104   55 / 91
// whole row blocks / ranges of wavefronts:
//   24 heads N = 8192 (1.50)   38 / 38    72 / 70   167 / 153  436 / 446    62 / 76   140 / 151   84 / 75    77 / 56
//   14 heads N = 17536 (1.87)  70 / 75   157 / 151  392 / 382 1155 / 1151  132 / 164  353 / 374  138 / 122  113 / 89
//   16 heads N = 16640 (2.03)  68 / 70   156 / 151  439 / 386 1322 / 1178  144 / 180  366 / 388  132 / 129  112 / 88
static int wave_slots() { return FwdCfg<64>::NW * FwdCfg<64>::WG_PER_CU * compute_units(); }    // wavefronts resident at once, D = 64
static int fwd_mode(int B, int H, int nb, bool compact) {
  const int64_t rows = (int64_t)B * H * nb, slots = wave_slots();
  if (2 * rows >= 3 * slots) return ROWS_MODE;
  if (compact) return COOP;                                             // (WAVE has four times as many ranges, hence parts)
  return rows >= slots || (nb >= 32 && nb <= 300 && 20 * rows >= (nb >= 48 ? 15 : 16) * slots) ? WAVE : COOP;
}

// ROWS_MODE: the workgroups per head for long row blocks, and the slots for their parts: as many as are resident at once,
// half of them where the scratch memory is the library's.  None with so many heads that a wavefront has the tiles of an
// eighth of a head to do, or where the library's scratch memory does not hold the counters.
static int long_row_groups(int B, int H, int nb, bool compact);

static int groups_per_head(int B, int H, int nb, int mode, bool compact) {
  if (mode == ROWS_MODE) return long_row_groups(B, H, nb, compact);
  const int cus = compute_units();
  const int per_cu = (mode == COOP ? 1 : FwdCfg<64>::NW) * FwdCfg<64>::WG_PER_CU;
  int64_t W = (int64_t)cus * per_cu / ((int64_t)B * H);   // as many workgroups as are resident at once
  const int64_t cap = (int64_t)nb * nb;
  if (W > cap) W = cap;
  if (W < 1) W = 1;
  return (int)W;
}

// workspace: partial slots [B*H][W][2][partial_floats] (fp32; ROWS_MODE: one per workgroup for long row blocks), then the
// arrival counters [B*H][nb] (64 bit)
static size_t slots_bytes(int B, int H, int W, int mode) {
  return (size_t)B * H * W * (mode == ROWS_MODE ? 1 : 2) * partial_floats(64) * sizeof(float);
}
static size_t parts_bytes(int B, int H, int nb, int W, int mode) {
  return slots_bytes(B, H, W, mode) + (size_t)B * H * nb * sizeof(unsigned long long);
}

// ROWS_MODE: heads whose row blocks go out together, the longest first.  One per XCD keeps one head's K and V in an L2, but a
// group's long row blocks then start when the short ones of the group before end, the last group's last of all; as many as
// are at work at once anyway (their row blocks fill the wavefronts of an XCD) cost little locality, above 8 more (300 heads
// N = 1024, keep 0.5, with 1 / 8 / 13: 72 / 73 / 78 us).  Groups of like size.
// Block-causal, bf16, us with 1 / 2 / 3 / 4 / 6 / 8 / 16 heads per XCD and group, and the ranges of workgroups that this mode
// replaced:       128 heads N = 2048 (8 at once)  118 / 115 / 116 /  98 / 105 /  94 /  94    99     256 heads  200 / 195 / 195 / 189 / 193 / 182 / 172   201
//                  64 heads N = 4096 (4)          214 / 189 / 198 / 174 / 221 / 173 / 173   198      96 heads  286 / 276 / 259 / 265 / 251 / 272 / 246   294
//                  48 heads N = 8192 (2)          537 / 509 / 491 / 526 / 463 / 462 / 461   573      24 heads  291 / 271 / 252 / 252 / 252 / 253 / 255   269
//   keep 0.2:      48 heads N = 8192              221 / 222 / 227 / 226 / 256 / 256 / 257   279     keep 0.5, 256 heads N = 2048  184 / 183 / 186 / 184 / 187 / 186 / 205
//   keep 0.05:     48 heads N = 17792 (1)         307 / 315 / 354 / 356 / 408 / 410 / 409   430
// With little more than one row block per wavefront the last group's long row blocks are all that is left to do in the end,
// on wavefronts each alone with its row of up to nb tiles: all heads go out together there, longest row blocks first (what a
// smaller L2 share costs the sparse uniform masks is less).  8 heads per group / all, block-causal, causal keep 0.2, keep 0.1, 0.5:
//    9 heads N = 24064 (1.65 row blocks per wavefront)  1001 /  794   238 / 185   201 / 194   848 / 849
//   11 heads N = 24064 (2.02)                           1103 /  909   261 / 215   223 / 228  1028 / 1033
//   17 heads N = 12000 (1.56)                            541 /  384   130 / 102   110 / 106   430 / 426
//   20 heads N = 12000 (1.84)                            549 /  456   130 / 112   117 / 117   456 / 464
//   25 heads N = 8192 (1.56)                             295 /  272    90 /  75    78 /  79   293 / 294
//   25 heads N = 12000 (2.29)                            660 /  536   158 / 135   145 / 157   574 / 582    (not there: 8 % on a sparse mask)
//    9 heads N = 32000 (2.20)                              -          384 / 305   311 / 329      -         (nor there)
static int rows_group(int B, int H, int nb) {
  const int heads = B * H, per_xcd = (heads + 7) / 8, at_work = (wave_slots() / 8 + nb / 2) / nb;
  if (nb >= 128 && nb <= 400 && 8 * (int64_t)heads * nb <= 17 * (int64_t)wave_slots()) return 8 * per_xcd;
  const int most = at_work < 1 ? 1 : (at_work > 8 ? 8 : at_work), groups = (per_xcd + most - 1) / most;
  return 8 * ((per_xcd + groups - 1) / groups);
}

static int long_row_groups(int B, int H, int nb, bool compact) {
  const int64_t W = wave_slots() / (compact ? 2 : 1) / ((int64_t)B * H);
  if (W < 8) return 0;
  return compact && parts_bytes(B, H, nb, (int)W, ROWS_MODE) > (size_t)BSATTN_STATIC_SCRATCH_BYTES ? 0 : (int)W;
}

// D = 256: shares of a row block's list, at most (quad_shares.h says how many of them a list has).  fwd_wide_kernel has two workgroups on a
// compute unit, so launches that leave the GPU's 512 short share, and those in little more than a round, whose last lists would run alone.
// us, N(0,1) bf16, a fixed number of shares for all lists and a launch that summed their fp32 parts / the lists that their length
// calls for, summed in the launch; keep 0.1, 0.3, 1, block-causal:
//    1 head  N = 768 (12 row blocks)      15 /  14     16 /  17     18 /  19     18 /  18
//    1 head  N = 1024 (16)                14 /  14     17 /  17     19 /  20     19 /  20
//    2 heads N = 1344 (42)                18 /  16     22 /  19     27 /  23     24 /  22
//    1 head  N = 4096 (64)                23 /  20     29 /  27     42 /  41     39 /  37
//    4 heads N = 2048 (128)               28 /  21     32 /  26     42 /  38     38 /  33
//    2 heads N = 4096 (128)               30 /  26     38 /  33     60 /  55     52 /  47
//    7 heads N = 2048 (224)               31 /  22     39 /  31     57 /  52     50 /  44
//    2 heads N = 6461 (202)               50 /  36     72 /  61    132 / 122     90 /  90
//    3 heads N = 6016 (282)               52 /  37     76 /  76    159 / 151    101 /  93
//    8 heads N = 4096 (512)               59 /  34     87 /  67    180 / 154    110 / 102
//    5 heads N = 8192 (640)              104 /  75    176 / 163    386 / 366    239 / 214
// Elementwise masks (on fwd_pair_kernel before), token window of 0.1 N, 0.25 N, 0.45 N, token-causal:
//    1 head  N = 768 (12)                 12 /  14     14 /  14     16 /  17     18 /  17
//    2 heads N = 1024 (32)                14 /  13     18 /  16     20 /  18     20 /  19
//    8 heads N = 2048 (256)               30 /  20     35 /  25     42 /  33     60 /  45
//    8 heads N = 4000 (504)               75 /  34    100 /  53    131 /  76    138 / 101
//    1 head  N = 8192 (128)               34 /  27     43 /  37     60 /  51     96 /  75
static int pair_split_256(int64_t row_blocks, int nb) {
  const int64_t cus = compute_units(), rows = row_blocks * 256 / cus;       // (as if there were 256 compute units)
  if (rows > 8 * nb || rows >= 1024) return 1;
  const int s = rows >= 320 ? 2 : rows >= 208 ? (nb >= 80 ? 3 : 2) : rows > 128 && nb < 80 ? 3 : 4;
  const int cap = rows <= 64 ? nb / 4 : nb / 6;
  return s < cap ? s : cap > 1 ? cap : 1;
}

// The same at D = 128, by fwd_pair_kernel: for what quad_plan leaves of the launches that do not fill the GPU, and for exact_tiles.  A share
// costs the launch that sums the parts (3 us) and their traffic, so short lists are shared only where few of them are in the launch.
// us, N(0,1), 1 / 2 / 3 / 4 / 6 shares; keep 0.3, dense:
//    1 head  N = 832              12 /  12 /  11 /  10 /  10     20 /  16 /  14 /  13 /  12
//    5 heads N = 832              13 /  14 /  14 /  16 /  16     20 /  18 /  17 /  19 /  20
//   11 heads N = 1344             17 /  23 /  24 /  26 /  30     30 /  31 /  31 /  31 /  37
//    1 head  N = 2048             23 /  17 /  15 /  14 /  16     42 /  27 /  22 /  19 /  18
//    4 heads N = 2048             24 /  22 /  23 /  24 /  25     43 /  32 /  31 /  31 /  32
//    2 heads N = 4096             36 /  27 /  27 /  26 /  26     81 /  51 /  44 /  39 /  37
//    1 head  N = 8192             67 /  42 /  35 /  32 /  32    157 /  88 /  69 /  58 /  54
//    3 heads N = 8192             75 /  58 /  68 /  63 /  70    168 / 128 / 159 / 143 / 146
//    2 heads N = 12032            92 /  71 /  83 /  78 /  83    240 / 176 / 223 / 195 / 197
static int pair_split_128(int64_t row_blocks, int nb) {
  const int64_t cus = compute_units(), rows = row_blocks * 256 / cus;       // (as if there were 256 compute units)
  if (nb < 56 && rows > 6 * nb) return 1;
  const int s = rows >= 480 ? 1 : rows >= 320 ? 2 : rows >= 208 ? 3 : 4;
  // a share of a dense list keeps 8 tiles, 4 in a launch of few lists, 12 in one of many short ones
  const int cap = rows <= 64 && nb >= 12 ? nb / 4 : rows > 96 && nb < 48 ? nb / 12 : nb / 8;
  return s < cap ? s : cap > 1 ? cap : 1;
}

// Which launches fwd_quad_kernel (D = 128) takes: groups of four wavefronts per workgroup (0: none) and shares of a list, at most
// (quad_shares.h).  With two groups a row block has a compute unit to itself, with one two share it.  us, fwd_pair_kernel with its shares
// and the launch that summed them / 2 groups, whole lists / 2 groups, up to 2 shares / up to 4 / 1 group, whole / up to 2; N(0,1) bf16;
// keep 0.1, 0.3, 1, block-causal (this kernel without tiles in two parts, which take 0.5 us each, up to two: exact_tiles):
//    1 head  N = 2048 (32 row blocks)  12/13/13/13          15/16/16/16          20/25/21/19          19/25/20/18
//    1 head  N = 4096 (64)             16/15/16/16          20/22/19/18          32/43/30/24          30/43/29/23
//    7 heads N = 1000 (112)            11/10                17/12                28/17                28/16
//    2 heads N = 4096 (128)            22/15/16             26/22/20             40/43/32             35/43/30
//    5 heads N = 256 (20)               - / -                                    9/10 (keep 0.9)                       (not there)
//   11 heads N = 1344 (231)            10/10                17/13                30/20                30/19
//    3 heads N = 4096 (192)            24/16/17             28/23/24             46/44/44             38/43/41
//    2 heads N = 6016 (188)            25/18/19             33/31/32             57/60/61             48/59/45
//    4 heads N = 4096 (256)            25/16/20             31/23/27             55/45/50             49/43/43
//    1 head  N = 16064 (251)           40/32/35             67/61/62            163/160/163          143/147/124
//    1 head  N = 12032 (188)           30/25/27             45/47/49             97/113/115           79/110/70       (not there)
//    8 heads N = 3072 (384)            18/21/25/ - /17/18   33/34/44/ - /28/29   68/67/67/ - /59/59   65/35/51/ - /44/45
//    3 heads N = 8192 (384)            37/36/42/ - /32/38   65/62/68/ - /56/60  139/158/143/ - /143/143  107/79/92/ - /103/84
//    9 heads N = 4096 (576)            28/36/38/ - /29/30   46/57/66/ - /51/52  109/131/127/ - /124/111   94/93/88/ - /75/78     (nor there)
//   24 heads N = 1280 (480)            14/18/28/ - / - /17  20/25/34/ - / - /22  33/37/47/ - / - /32    32/32/38/ - / - /39    (nor there)
//    2 heads N = 12032 (376)           40/42/52/ - /36/38   79/88/87/ - /85/86  191/226/196/ - /202/202  145/113/119/ - /147/108   (nor there)
// Elementwise masks (words), token window of 0.1 N, 0.25 N, 0.45 N, token-causal:
//    2 heads N = 2000 (64)             15/11/ - /11         17/13/ - /13         20/17/ - /16         23/26/ - /17
//    3 heads N = 4000 (189)            23/13/13             26/18/18             31/27/27             44/47/39
//    8 heads N = 4000 (504)            30/24/28/ - /19/19   39/34/37/ - /27/27   52/50/51/ - /41/41   79/55/60/ - /69/59
//    1 head  N = 17000 (266)           40/45/45/ - /37/37   68/65/66/ - /72/72  100/90/90/ - /122/121   191/176/134/ - /256/174
//   10 heads N = 4000 (630)            25/36/36/ - /31/30   41/48/56/ - /41/45   66/63/72/ - /56/60  121/97/94/ - /80/81     (not there)
//   16 heads N = 8000 (2000)           76/115/131/ - /88/88  145/184/202/ - /150/152  217/261/276/ - /217/219  274/345/362/ - /292/294   (nor there)
// Up to 32 row blocks fwd_pair_kernel in four shares is up to 2.4 us faster, and up to 7 % further from 64 bits with fp32 results of
// bf16 (1 head N = 768 keep 0.1 1.63e-4 against 1.54e-4, N = 1536 dense 2.02e-4 and 1.91e-4); with its first tiles in two parts (softmax_block_parts)
// it takes 1.9 to 4 us more.  Pairs / so / this kernel; keep 0.1, 0.3, 1, block-causal:
//    1 head  N = 768  (12)     11/12/11   12/14/12   13/16/15   13/16/15         1 head  N = 1536 (24)     12/13/12   14/16/16   17/21/18   16/20/18
//    1 head  N = 1024 (16)     10/11/11   12/14/14   14/17/17   14/16/16         2 heads N = 1024 (32)     11/12/11   13/15/14   15/18/17   14/17/16
// Whole lists of two groups leave the compute units idle that have none.  Where three shares of every list fit one round of single groups,
// up to 168 row blocks (tail_of), long lists take those (from there on two shares of one head's leave up to a third of the places empty,
// which pairs fill, up to 230 row blocks); a little more than one round of two groups goes to single groups, whose lists
// are cut in three to fill the GPU.  Pairs / two groups / this; keep 0.1, 0.3, 1, block-causal:
//    1 head  N = 8320 (130)    26/25/26  37/43/35   74/ 87/ 66   61/ 52/59       2 heads N = 5120 (160)    25/17/20  33/33/30   55/61/50   46/39/42
//    1 head  N = 9600 (150)    28/26/26  41/48/37   82/ 98/ 75   67/ 57/62       3 heads N = 3392 (159)    23/15/17  28/25/26   43/42/38   37/32/33    (two groups)
//    1 head  N = 10880 (170)   29/ - /28 46/ - /55  93/ - /120   77/ - /66       (pairs)
// Pairs / single groups, whole or by a list's own length / this:
//    3 heads N = 5632 (264)    29/24/26  41/46/47   79/101/ 88   64/ 60/56       3 heads N = 6400 (300)    31/29/28  48/58/50   93/114/103  73/65/64
//    4 heads N = 4352 (272)    26/20/20  36/35/36   66/ 80/ 75   54/ 59/50       4 heads N = 4800 (300)    29/23/23  41/43/44   75/ 86/ 84  59/64/50    (whole)
// (Room for a share that a list never gets costs the launch the workgroups that find so, 1 to 2 us at a full round: 2 x 2 heads N = 3825
// keep 0.63 (240) whole 34.5, with room for two shares 38.9; 3 heads N = 4096 (192) keep 0.3 27.5 and 29.)
//    words: 1 head N = 20000 (313), two groups in place of the whole single ones    57/65/55  94/113/97  134/135/139  236/216/186
//    words: 1 head N = 17920 (280)                                                  43/56/43  74/ 87/77  108/102/117  178/180/143
// From 480 row blocks on a round of single groups is full (one head N = 32000 (500) 105/ - /92  263/ - /218  665/ - /586  636/ - /375).
struct QuadPlan { int groups, split, most; };      // most: shares of a list by its own length; split: that, or what fills the GPU
static QuadPlan quad_plan(int64_t row_blocks, int nb, bool words) {
  const int64_t cus = compute_units(), rows = row_blocks * 256 / cus;       // (as if there were 256 compute units)
  auto plan = [](int groups, int most, int fill = 1) { return QuadPlan{groups, std::max(most, fill), most}; };
  if (rows > 512 || nb > QUAD_MAX_BLOCKS) return plan(0, 1);
  const int fill = nb >= 3 * FILL_GAIN && rows <= 336 ? 3 : 1;      // (more than 256 row blocks: thirds of lists, tail_of)
  if (words) {
    if (rows > 256 && (rows > 272 || nb < 200)) return plan(1, nb >= 28 ? 2 : 1, fill);
    return plan(2, nb < 16 ? 1 : rows <= 64 ? 4 : rows <= 128 || nb >= 28 ? 2 : 1);
  }
  if (rows > 256) {
    if (nb < 28 || (nb >= 150 && rows < 480)) return plan(0, 1);
    return plan(1, nb >= 80 ? 2 : 1, fill);
  }
  if (nb < 6 || (rows > 168 && rows <= 230 && nb >= 150)) return plan(0, 1);
  if (rows > 128 && rows <= 168 && nb >= 64) return plan(1, 3);
  if (rows <= 128) return plan(2, rows <= 64 && nb >= 16 ? 4 : nb >= 24 ? 2 : 1);
  return plan(2, nb >= (rows <= 160 ? 40 : 80) ? 2 : 1);
}
static_assert(SHARE_MIN_BLOCKS <= 16, "heads of launches that share lists have as many row blocks");

// the parts of shared lists and a counter per list
static size_t quad_parts_bytes(int B, int H, int nb, int D, int split) {
  return 256 + (split > 1 ? (size_t)B * H * nb * (split * 64 * (size_t)(D + 2) * sizeof(float) + sizeof(unsigned long long)) : 0);
}

static size_t pair_parts_bytes(int B, int H, int N, int D, int split) {
  return 256 + (split > 1 ? (size_t)B * H * (split * (size_t)N * (D + 2) + (N + 63) / 64) * sizeof(float) : 0);
}

// compact: as many of these shares as the library's scratch memory has room for, two at least (less is refused: 8 heads of N = 1408
// and 1472 at D = 256 have two of three, one head of N = 8192 has three of four; D = 128 has room for all).
static int pair_split(int B, int H, int N, int D, bool compact) {
  const int nb = (N + 63) / 64;
  const int64_t row_blocks = (int64_t)B * H * nb;
  int s = D == 256 ? pair_split_256(row_blocks, nb) : pair_split_128(row_blocks, nb);
  if (compact)
    while (s > 2 && pair_parts_bytes(B, H, N, D, s) > (size_t)BSATTN_STATIC_SCRATCH_BYTES) --s;
  return s;
}

// Which launches fwd_short_kernel (D = 64) takes: pairs of wavefronts per workgroup (0: none) and shares of a row block's list.
// With 4 pairs a row block has a compute unit to itself, with 2 two share it.  us, ranges of workgroups or of wavefronts /
// 2 pairs / 4 pairs / 4 pairs and 2 shares; keep 0.1, 0.3, 1, block-causal (fp16 the first five, bf16 the others):
//    5 heads N = 512 (40 row blocks)   11 /  8 /  8 / 10     11 /  8 /  8 / 10     12 /  8 /  8 / 10     11 /  8 /  8 / 10
//    8 heads N = 2048 (256)            13 /  9 /  9 / 19     16 / 12 / 11 / 21     20 / 19 / 17 / 27     19 / 18 / 16 / 22
//    2 heads N = 8192 (256)            17 / 15 / 14 / 21     27 / 26 / 23 / 30     53 / 55 / 44 / 57     38 / 54 / 44 / 35
//   16 heads N = 3072 (768)            22 / 18 / 21          32 / 28 / 32          59 / 56 / 60          42 / 34 / 40
//   32 heads N = 3072 (1536)           30 / 27 / 40          52 / 47 / 61         101 /103 /126          65 / 62 / 81
//   44 heads N = 3072 (2112)           39 / 37 / 57          57 / 63 / 84         137 /149 /176          81 / 91 /109   (not there)
//   14 heads N = 4096 (896)            29 / 21 / 29          42 / 37 / 47          84 / 87 / 99          53 / 51 / 57
//   24 heads N = 4096 (1536)           31 / 32 / 45          55 / 57 / 70         132 /133 /153          78 / 89 / 93   (nor there)
//    3 heads N = 6400 (300)            20 / 15 / 17          29 / 29 / 30          50 / 65 / 73          37 / 48 / 37   (nor there)
//    5 heads N = 6400 (500)            26 / 16 / 20          41 / 30 / 34          73 / 71 / 75          46 / 51 / 45
//    1 head  N = 10048 (157)           19 / 16 / 13 / 20     26 / 30 / 25 / 30     44 / 72 / 55 / 64     32 / 71 / 53 / 35   (nor there)
// Shares of a list, that meet in the launch (kernel time and launch among others, fp16), of at least 8 tiles: none / 2 / 3 / 4 (and 4 of at
// least one tile); keep 0.1, 0.3, dense, block-causal:
//    1 head  N = 1024 (16)              5.7/ 5.9/ 5.8/ 5.7 ( 8.3)    7.0/ 7.1/ 7.1/ 7.1 ( 9.1)    9.5/10.0/10.0/10.1 ( 9.8)    9.3/ 9.4/ 9.5/ 9.6 ( 9.6)    (not there)
//    1 head  N = 1536 (24)              6.4/ 6.5/ 6.5/ 6.5 ( 8.9)    8.6/ 8.6/ 8.6/ 8.6 ( 9.3)   11.9/11.3/10.5/10.6 (10.5)   11.7/10.8/10.6/10.9 (10.2)
//    1 head  N = 4096 (64)              8.0/ 8.2/ 8.2/ 8.2 ( 9.8)   12.9/11.8/11.2/11.2 (11.0)   24.0/17.7/15.4/14.6 (14.8)   23.6/17.1/14.4/13.2 (13.2)
//    1 head  N = 5120 (80)              9.0/ 9.1/ 9.1/ 9.1 (13.4)   14.8/12.9/11.5/16.7 (16.6)   28.8/20.3/17.4/24.7 (24.7)   28.4/19.4/16.4/17.4 (17.3)
//    5 heads N = 1536 (120)             6.5/ 6.7/ 6.7/ 6.7 (14.7)    9.0/ 9.0/ 9.0/ 9.0 (14.4)   12.0/12.0/17.0/16.9 (16.7)   11.9/11.2/11.3/11.3 (15.2)   (nor there)
//    4 heads N = 2048 (128)             7.1/ 7.3/ 7.3/ 7.3 (14.4)   10.6/10.5/10.6/10.6 (15.0)   14.7/13.6/18.6/18.3 (18.1)   14.5/12.5/15.7/16.9 (16.0)
//    1 head  N = 8192 (128)            11.2/10.9/10.9/10.9 (15.4)   21.4/16.8/22.0/20.8 (21.0)   44.0/29.6/39.1/34.4 (34.3)   42.9/27.2/27.2/27.9 (28.5)
//    3 heads N = 5120 (240)             9.2/10.1/11.4/12.7 (23.5)   17.4/22.3/27.5/31.4 (29.4)   31.0/38.3/43.3/46.9 (47.2)   29.3/25.9/30.2/32.4 (32.6)   (nor there)
// (With bf16 from 56 row blocks on also the shortest lists are shared, as they were when a launch of its own summed four shares of every list there:
// a share's first tiles have exact largest numerators, so that rows of fewer shares would be further from 64 bits than they were.  Lists of fewer
// row blocks never were shared that way.)
struct ShortPlan { int pairs, split; };
static ShortPlan short_plan(int64_t row_blocks, int nb) {
  const int64_t cus = compute_units(), rows = row_blocks * 256 / cus;       // (as if there were 256 compute units)
  if (nb > SHORT_MAX_BLOCKS) return {0, 1};
  // long lists: as many shares as fill the GPU
  if (rows <= 256) {
    const int split = rows > 128 ? 1 : rows > 85 ? 2 : rows > 64 ? 3 : 4;       // (workgroups of 4 pairs are alone on their compute unit)
    return {4, nb < (split == 4 ? 20 : 28) ? 1 : split};
  }
  const bool takes = nb <= 48 ? rows <= 1792 : nb <= 64 ? rows <= 1024 : rows >= 400 && rows <= 512;
  return {takes ? 2 : 0, 1};
}

// compact: as many shares as the library's scratch memory has room for (4 heads of N = 8192 have one of two).
static QuadPlan quad_plan(int B, int H, int nb, bool words, bool compact) {
  QuadPlan plan = quad_plan((int64_t)B * H * nb, nb, words);
  if (compact)
    while (plan.split > 1 && quad_parts_bytes(B, H, nb, 128, plan.split) > (size_t)BSATTN_STATIC_SCRATCH_BYTES) --plan.split;
  plan.most = std::min(plan.most, plan.split);
  return plan;
}

// D = 256: the same by fwd_wide_kernel, at most this many shares of a list ...
static int wide_split(int B, int H, int N, bool compact) {
  const int nb = (N + 63) / 64;
  int s = nb < SHARE_MIN_BLOCKS ? 1 : pair_split(B, H, N, 256, compact);
  if (compact)
    while (s > 1 && quad_parts_bytes(B, H, nb, 256, s) > (size_t)BSATTN_STATIC_SCRATCH_BYTES) --s;
  return s;
}

// Tiles of a share, at least, of a launch that shares lists: a hand-off takes 2.5 us, three or four tiles' time where a workgroup is
// alone on its compute unit, and evens out nothing where the GPU is full.  us, at least 4 / 6 / 8 (16, 24):
//    D = 256   2 heads N = 1024, token-causal (32 row blocks)  20 / 21 / 26         1 head  N = 2048, keep 0.3 (32)  21 / 21 / 26
//              2 heads N = 4096, keep 0.1 (128)                24 / 22 / 26         3 heads N = 4096, token-causal (192)  - / - / 50 (51, 69)
//              8 heads N = 2048, token window of 512 (256)     25 / 21 / 22         5 heads N = 8192, keep 0.1 (640)  75 / 74 / 72 ( - , 66)
//    D = 256, at least 3 / 4 (whole 18, 24, 24, 19, 20, 24, 25): 1 head N = 768, keep 0.3 (12) 17 / 18, dense 19 / 19,
//              block-causal 18 / 20; 1 head N = 1024, keep 0.3 (16) 18 / 19, dense 20 / 20; 4 heads N = 768, block-causal (48) 19 / 20, dense 21 / 20
//    D = 128   3 heads N = 1280, dense (60)                    26 / 17 / 17         2 heads N = 1024, token-causal (32)  14 / 14 / 16
static int share_least(int64_t row_blocks, int D) {
  const int64_t rows = row_blocks * 256 / compute_units();
  if (D == 128) return rows <= 64 ? 6 : 8;
  return rows <= 64 ? 3 : rows <= 256 ? 6 : 24;
}

// How exact a launch's rows are at least, in hundredths of a tile (FwdShareParams::exact): as in a launch of pairs of wavefronts
// (D = 256 with block masks: key halves) that cuts every list into the parts below, whatever its length.  A part's first tile gives the
// reference, so that its largest numerator is exact: of what rounding the numerators of a tile costs a row (their squares), that is
// 38 % with 64 keys of N(0,1) scores, 48 % with 32.  (fp16 with block masks keeps the reference at 0: nothing is exact there.)
// fp32 results of bf16 against 64 bits, without this rule / with it / such a launch: D = 256 2 heads N = 4096 block-causal 1.84e-4 / 1.49e-4 / 1.70e-4,
// 5 heads N = 3648 block-causal keep 0.3 1.78e-4 / 1.48e-4 / 1.71e-4; D = 128 8 heads N = 4000 token window of 1000 1.73e-4 / 1.51e-4 / 1.71e-4.
static int exact_tiles(int64_t row_blocks, int nb, int D, bool words, bool fp16) {
  if (!words) return fp16 ? 0 : D == 256 ? 48 * pair_split_256(row_blocks, nb) : 38 * pair_split_128(row_blocks, nb);
  if (D == 256) return 38 * pair_split_256(row_blocks, nb);
  // about four workgroups per compute unit, at most 4 parts of a row unless it is long
  const int64_t few = nb / 2 < 4 ? nb / 2 : 4, cap = nb / 16 > few ? nb / 16 : few, s = 4 * (int64_t)compute_units() / row_blocks;
  return 38 * (int)std::clamp<int64_t>(std::min(s, cap), 1, 8);
}

// Launches whose workgroups have a row block each need no lists of a block mask: they take its columns from the mask (3 heads
// N = 891, D = 128, a mask per head and call, 21.3 -> 16.2 us; dense mask of N = 6400, D = 64, reduced in the call, 27.1 -> 22.9).
bool launch_fwd_takes_mask(int B, int H, int N, int D) {
  const int nb = (N + 63) / 64;
  return D == 64 ? short_plan((int64_t)B * H * nb, nb).pairs > 0 : nb <= MASK_MAX_BLOCKS;
}

size_t coop_workspace_bytes(int B, int H, int N, int D, bool compact) {
  if (D == 256) {      // (compact: what a launch that sums parts of all lists would take, for which fewer shapes have room)
    return compact ? pair_parts_bytes(B, H, N, D, pair_split(B, H, N, D, true)) : quad_parts_bytes(B, H, (N + 63) / 64, D, wide_split(B, H, N, false));
  }
  if (D == 128) {
    const int nb = (N + 63) / 64;
    auto bytes = [&](bool words) {
      const QuadPlan plan = quad_plan(B, H, nb, words, compact);
      return plan.groups > 0 ? quad_parts_bytes(B, H, nb, 128, plan.split) : pair_parts_bytes(B, H, N, D, pair_split(B, H, N, D, compact));
    };
    return compact ? bytes(false) : std::max(bytes(false), bytes(true));       // (compact launches: block masks only)
  }
  const int nb = (N + 63) / 64;
  if (const ShortPlan plan = short_plan((int64_t)B * H * nb, nb); plan.pairs > 0) return quad_parts_bytes(B, H, nb, 64, plan.split);
  const int mode = fwd_mode(B, H, nb, compact);
  const int W = groups_per_head(B, H, nb, mode, compact);
  return W == 0 ? 256 : parts_bytes(B, H, nb, W, mode);      // (0: nothing is shared)
}

// one size for bsattn_fwd and bsattn_fwd_elementwise
size_t fwd_workspace_bytes(int B, int H, int N, int D) { return coop_workspace_bytes(B, H, N, D); }

void launch_fwd_pair(const FwdParams& prm, int dt, bool elementwise, hipStream_t st);   // attn_fwd_pair.hip
void launch_fwd_short(const FwdParams& prm, int pairs, int dt, bool elementwise, hipStream_t st);   // attn_fwd_short.hip
void launch_fwd_quad(const FwdShareParams& prm, int groups, int dt, bool elementwise, hipStream_t st);   // attn_fwd_quad.hip
void launch_fwd_wide(const FwdShareParams& prm, int dt, bool elementwise, hipStream_t st);   // attn_fwd_wide.hip
template <int D, int DT, int MODE, bool EW, int LAYOUT, bool SPREAD>
static void launch_fwd_s(const FwdRangeParams& prm, int grid, hipStream_t st) {
  using C = FwdCfg<D>;
  constexpr int LDS = MODE != COOP ? C::ROWS_LDS_BYTES : C::LDS_BYTES;
  static std::atomic<unsigned long long> configured{0};   // raising the dynamic LDS limit is idempotent
  once_per_device(configured, [] {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&fwd_kernel<D, DT, MODE, EW, LAYOUT, SPREAD>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
  });
  hipLaunchKernelGGL((fwd_kernel<D, DT, MODE, EW, LAYOUT, SPREAD>), dim3(grid), dim3(MODE != COOP ? 64 : C::NW * 64), LDS, st, prm);
}

template <int D, int DT, int MODE, bool EW, int LAYOUT>
static void launch_fwd_c(const FwdRangeParams& prm, int grid, hipStream_t st) {
  if constexpr (MODE != ROWS_MODE) {
    if (XCDS % (prm.B * prm.H) != 0) { launch_fwd_s<D, DT, MODE, EW, LAYOUT, true>(prm, grid, st); return; }
  }
  launch_fwd_s<D, DT, MODE, EW, LAYOUT, false>(prm, grid, st);
}

// (The copies with immediate offsets are 2-4 % faster.)
template <int DT, int MODE, bool EW>
static void launch_fwd_t(const FwdRangeParams& prm, int grid, hipStream_t st) {
  const bool contig = prm.ks[2] == 64 && prm.vs[2] == 64, whole = prm.N % 64 == 0;
  if (contig && whole) launch_fwd_c<64, DT, MODE, EW, CONTIG_WHOLE>(prm, grid, st);
  else if (contig) launch_fwd_c<64, DT, MODE, EW, CONTIG_TAIL>(prm, grid, st);
  else launch_fwd_c<64, DT, MODE, EW, GENERAL>(prm, grid, st);
}

template <int MODE, bool EW>
static void launch_fwd_m(const FwdRangeParams& prm, int dt, int grid, hipStream_t st) {
  if (dt == 0) launch_fwd_t<0, MODE, EW>(prm, grid, st);
  else if (dt == 1) launch_fwd_t<1, MODE, EW>(prm, grid, st);
  else launch_fwd_t<2, MODE, EW>(prm, grid, st);
}

template <bool EW>
static void launch_fwd_d(const FwdRangeParams& prm, int mode, int dt, hipStream_t st) {
  const int BH = prm.B * prm.H, grid = prm.W * BH;
  if (mode == ROWS_MODE) launch_fwd_m<ROWS_MODE, EW>(prm, dt, placed(BH, prm.group, prm.nb) + placed(BH, prm.group, prm.W), st);
  else if (mode == WAVE) launch_fwd_m<WAVE, EW>(prm, dt, grid, st);
  else launch_fwd_m<COOP, EW>(prm, dt, grid, st);
}

// ---- forward without any allocation by anybody: the scratch memory is part of the library ----
// A file-scope device array stands in for the workspace argument of launch_fwd.  In host code its name
// is only a handle: the address the kernels may use is asked for once per device (each device holds
// its own copy of the array at its own address).
static __device__ __align__(256) unsigned char scratch[BSATTN_STATIC_SCRATCH_BYTES];

int static_scratch(void** ptr) {
  static std::atomic<void*> per_device[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return BSATTN_ERR_LAUNCH;
  void* p = per_device[dev].load(std::memory_order_acquire);
  if (p == nullptr) {
    // (two threads may both ask: they get the same answer)
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || p == nullptr) return BSATTN_ERR_LAUNCH;
    per_device[dev].store(p, std::memory_order_release);
  }
  *ptr = p;
  return BSATTN_OK;
}

// The range permutation of fwd_kernel (range_perm.h) depends on (nb, W, F, heads) only: kept in a small cache.
static bool range_permutation(int nb, int W, int F, int BH, unsigned short* out, unsigned short* out_causal) {
  static std::mutex mu;
  static std::map<std::array<int, 4>, std::array<unsigned short, 2 * RANGE_PERM_MAX>> cache;
  const std::array<int, 4> key = {nb, W, F, BH};
  std::lock_guard<std::mutex> lock(mu);
  auto it = cache.find(key);
  if (it == cache.end()) {
    std::array<unsigned short, 2 * RANGE_PERM_MAX> t{};
    if (!make_range_permutation(nb, W, F, BH, WEIGHT_FAST, WEIGHT_SLOW, false, t.data()) ||
        !make_range_permutation(nb, W, F, BH, WEIGHT_FAST, WEIGHT_SLOW, true, t.data() + RANGE_PERM_MAX)) return false;
    if (cache.size() >= 64) cache.clear();
    it = cache.emplace(key, t).first;
  }
  for (int i = 0; i < W; ++i) { out[i] = it->second[i]; out_causal[i] = it->second[RANGE_PERM_MAX + i]; }
  return true;
}

int launch_fwd(const void* q, const void* k, const void* v, void* o, float* lse,
               const int32_t* row_ptr, const int32_t* col_idx, const uint8_t* tile_partial,
               const uint64_t* tile_bits, const AttnShape& s, void* ws, hipStream_t st) {
  FwdRangeParams prm;
  prm.q = q; prm.k = k; prm.v = v; prm.o = o; prm.lse = lse;
  prm.mask = s.mask;
  prm.mask_copy = s.mask_copy;
  for (int i = 0; i < 4; ++i) prm.ms[i] = s.mask != nullptr ? s.ms[i] : 0;
  prm.row_ptr = row_ptr; prm.col_idx = col_idx; prm.ws = (float*)ws;
  prm.tile_partial = tile_partial; prm.tile_bits = (const unsigned long long*)tile_bits;
  prm.B = s.B; prm.H = s.H; prm.N = s.N; prm.nb = (s.N + 63) / 64; prm.Bm = s.Bm; prm.Hm = s.Hm;
  prm.per_batch = divisor((unsigned)s.H, (uint64_t)s.B * s.H);
  prm.out_f32 = s.out_dtype == BSATTN_F32;
  prm.qk_scale = s.sm_scale * 1.4426950408889634f;
  for (int i = 0; i < 3; ++i) { prm.qs[i] = s.qs[i]; prm.ks[i] = s.ks[i]; prm.vs[i] = s.vs[i]; prm.os[i] = s.os[i]; }
  // bf16 with a bf16-typed result: P is rounded to bf16 as well (the reference rounds P to the type of
  // V, fa2_fwd.py:189) and V is used as it is; an fp32 result keeps P in fp16
  const int dt = s.dtype != BSATTN_BF16 ? 0 : (prm.out_f32 ? 1 : 2), heads = s.B * s.H;
  const ShortPlan plan = s.D == 64 ? short_plan((int64_t)heads * prm.nb, prm.nb) : ShortPlan{0, 1};
  const int wide = s.D == 256 ? wide_split(s.B, s.H, s.N, s.compact) : 1;
  const QuadPlan quads = s.D == 128 ? quad_plan(s.B, s.H, prm.nb, tile_bits != nullptr, s.compact) : QuadPlan{s.D == 256 ? 1 : 0, wide, wide};
  if (quads.groups > 0) {
    const int slots = compute_units() * (quads.groups == 1 ? 2 : 1), rows = heads * prm.nb;
    const size_t parts = (size_t)rows * quads.split * 64;
    FwdShareParams shared;
    static_cast<FwdParams&>(shared) = prm;
    shared.split = quads.split;
    shared.place = place_of_eight(heads, prm.nb, shared.split, groups_of_heads(heads, s.N, s.D));
    shared.load = (int)((int64_t)rows * 4096 / slots);
    shared.most = quads.most;
    const TailShares tail = tail_of(rows, slots, shared.split);
    shared.tail_from = tail.from;
    shared.tail_shares = tail.shares;
    shared.tail_len = tail.len;
    shared.share_least = share_least(rows, s.D);
    shared.exact = exact_tiles(rows, prm.nb, s.D, tile_bits != nullptr, dt == 0);
    shared.part_o = (float*)ws + 64;
    shared.part_ml = shared.part_o + parts * s.D;
    shared.flags = (unsigned long long*)(shared.part_ml + parts * 2);
    shared.epoch = next_epoch();
    if (s.D == 128) launch_fwd_quad(shared, quads.groups, dt, tile_bits != nullptr, st);
    else launch_fwd_wide(shared, dt, tile_bits != nullptr, st);
    return launch_status();
  }
  if (s.D != 64 || plan.pairs > 0) {
    prm.split = s.D == 64 ? plan.split : tile_bits != nullptr ? 1 : pair_split(s.B, s.H, s.N, s.D, s.compact);
    prm.place = place_of_eight(heads, prm.nb, prm.split, groups_of_heads(heads, s.N, s.D));
    const size_t parts = s.D == 64 ? (size_t)heads * prm.nb * prm.split * 64 : (size_t)prm.split * heads * s.N;      // rows of them
    prm.part_o = (float*)ws + 64;
    prm.part_ml = prm.part_o + parts * s.D;
    if (s.D == 64) {
      prm.flags = (unsigned long long*)(prm.part_ml + parts * 2);
      prm.epoch = next_epoch();
      prm.share_shift = dt != 0 && prm.nb >= 56 ? 0 : 3;      // (short_plan)
      launch_fwd_short(prm, plan.pairs, dt, tile_bits != nullptr, st);
      return launch_status();
    }
    prm.part_len = (int*)(prm.part_ml + parts * 2);
    launch_fwd_pair(prm, dt, tile_bits != nullptr, st);
    return launch_status();
  }
  const int mode = fwd_mode(s.B, s.H, prm.nb, s.compact);
  prm.W = groups_per_head(s.B, s.H, prm.nb, mode, s.compact);
  prm.place_fast = mode == COOP ? std::min(compute_units(), prm.W * heads) : 0;
  prm.place_quot = prm.place_fast / heads;
  prm.place_rest = prm.place_fast % heads;
  prm.group = mode == ROWS_MODE ? rows_group(s.B, s.H, prm.nb) : 0;
  // with two workgroups per compute unit the first-comers are faster: tell the kernel which they are.  (Not WAVE: single
  // wavefronts that arrive while another kernel ends do not fill the SIMDs in order, and two with the larger share on one
  // SIMD cost more than the shares gain: 8 heads of N = 17536 dense after a kernel on its inputs 858-933 us against 732-816,
  // after a pause 677 against 707.)
  prm.first_ids = mode == COOP ? compute_units() : mode == ROWS_MODE ? first_ids_of_rows(wave_slots() / 8 * 8, heads, prm.group, prm.nb) : 0;
  prm.own = mode == COOP ? own_lines(prm.nb, prm.W, prm.first_ids / heads) : OwnLines{};
  prm.flags = (unsigned long long*)((char*)ws + slots_bytes(s.B, s.H, prm.W, mode));
  prm.epoch = next_epoch();
  prm.deterministic = get_deterministic();
  {
    const int F = prm.first_ids > 0 && prm.first_ids % heads == 0 ? (prm.first_ids / heads < prm.W ? prm.first_ids / heads : prm.W) : 0;
    const bool ok = mode == COOP && (prm.first_ids == 0 || prm.first_ids % heads == 0) && range_permutation(prm.nb, prm.W, F, heads, prm.perm, prm.perm_causal);
    prm.perm_n = ok ? prm.W : 0;
    prm.perm_fast = F;
    prm.perm_min_tiles = (int)((int64_t)prm.nb * prm.nb * 3 / 4);
  }
  if (tile_bits == nullptr) launch_fwd_d<false>(prm, mode, dt, st);
  else launch_fwd_d<true>(prm, mode, dt, st);
  return launch_status();
}

}  // namespace bsattn
