// Into how many shares the list of a row block is cut (fwd_quad_kernel, fwd_wide_kernel), by its own length.  Plain C++ (constexpr functions are
// usable on the device too).
#pragma once

namespace bsattn {

constexpr int SHARE_SAMPLE = 4;       // lists looked at in the middle and at the end of a head
constexpr int SHARE_MIN_BLOCKS = 16;  // row blocks of a head whose lists may be cut, at least

// len: tiles of the list; mid, end: of SHARE_SAMPLE lists in the middle of the head and of its last ones; tail: shares that a list of
// the last, incomplete round of workgroups is cut into (1: it is in front of it); load: row blocks per resident workgroup, times 4096.
// Where the lists grow along the head (causal masks), those above the mean are cut into shares of about the mean work of a resident
// workgroup, and so are lists of twice the mean in any head, in launches of one round (5 heads N = 8192 block-causal, D = 256, in 1.25
// rounds 217 -> 225 us).  least: tiles of a share, at least.  (Lists of like length in one round of workgroups stay whole: cutting
// some of them by chance of a random mask costs a hand-off and evens out nothing, 6 heads N = 4096 keep 0.3 36 -> 47 us.)
constexpr int quad_shares(int len, int mid, int end, int tail, int load, int most, int least) {
  int n = tail;
  const bool grows = 2 * end > 3 * mid;
  if (load <= 4096 && SHARE_SAMPLE * len > (grows ? mid : 2 * mid)) {
    const long long target = (long long)mid * load;                      // times SHARE_SAMPLE * 4096
    const long long work = (long long)len * SHARE_SAMPLE * 4096;
    const int even = target > 0 ? (int)((work + target / 2) / target < most ? (work + target / 2) / target : most) : most;
    n = n > even ? n : even;
  }
  const int fit = len / least;
  n = n < fit ? n : fit;
  n = n < most ? n : most;
  return n > 1 ? n : 1;
}

}  // namespace bsattn
