// Head-wise token reorder: row t of a head moves to row new_t of the same head, pure data movement bound by HBM.
// Index arithmetic follows fa2_custom_mask/permute.py:20-52 (forward) and :77-120 (inverse); unlike the
// reference's scalar loop over the head dimension (:54-58) a token row is moved with coalesced vector accesses:
// consecutive lanes copy consecutive 16-byte (or 4-byte) pieces of one row.
//
// In place (what the caller around attention wants: the image tokens of q, k and v, rows of a larger tensor, are
// reordered where they are).  Through a buffer every row would cross HBM four times (or more: with contiguous copies
// before and after, 48 heads x 17550 tokens x 64 bf16 of q, k, v and the result took 460 us in 14 launches).  Here the
// rows of a head are spread over the registers of a group of workgroups: each loads its part, counts itself in, waits
// until the whole head is in registers, and stores its rows where they belong: every row crosses HBM twice, 114 us for q, k
// and v and 37 for the result (4.8 TB/s over the five sixths of the heads whose order is not the identity).
// Every wait is bounded: a workgroup that waits too long marks the group as broken, then nobody stores anything of that
// head, and the last one to leave moves the head alone, a column of 4 bytes at a time.  The members of a group have
// neighbouring places in the dispatch order of one XCD, so this happens only where the launch is confined to a few
// compute units.  Heads whose order is the identity are left alone.
#include <mutex>
#include "common.h"

namespace bsattn {

typedef unsigned int uintx4 __attribute__((ext_vector_type(4)));

constexpr int REORDER_TENSORS_MAX = 4;
constexpr int REORDER_UNROLL = 8;                 // out of place: pieces of a thread in flight
// In place: 16-byte pieces held by a thread.  One workgroup of 1024 threads fits a compute unit (at most 128 registers);
// pieces swept for the sizes above: 9 with two workgroups per compute unit 174 us, 12 166, 14 154, 16 156, 18 163, 24 171.
constexpr int GROUP_THREADS = 1024, GROUP_PIECES = 14;
constexpr int GROUP_PARTS_MAX = 32;               // workgroups per head (one per compute unit of an XCD)
constexpr int GROUP_ROWS_MAX = GROUP_THREADS * GROUP_PIECES * 4;     // 4-byte pieces one workgroup can hold
constexpr unsigned long long WAIT_TICKS = 10000;  // of the 100 MHz clock: 100 us
// A group's counter: launch mark << 24 | members that left a broken group << 16 | BROKEN | members counted in.  Counters
// lie 256 bytes apart (8 to a cache line, 8 XCDs polling: 232 instead of 175 us).
constexpr unsigned long long BROKEN = 0x8000ull, COUNT_MASK = 0x7fffull, LEFT_ONE = 0x10000ull;
constexpr int COUNTER_STRIDE = 32;

struct ReorderParams {
  const char* src; char* dst;         // out of place: [BS * NH][T][row_bytes] both
  char* x[REORDER_TENSORS_MAX];       // in place: unit u = (tensor, batch, head)
  int64_t sb[REORDER_TENSORS_MAX], sh[REORDER_TENSORS_MAX], st[REORDER_TENSORS_MAX];     // strides of x in bytes
  int units, BS, NH, F, H, W, row_bytes;
  const int32_t* orders; const int32_t* inv_orders;      // out of place: [NH][3]
  const void* numbers; int number_bytes, inverse;         // in place: permutation number of every head (int32 or int64)
  unsigned* bad_number;               // ... host memory: set to 1 for a number outside the table
  int vshift;                         // log2(pieces per row), -1 if that is not a power of two
  unsigned blocks_per_unit, rows_per_block;         // out of place
  unsigned parts, pieces_per_part;                  // in place
  unsigned long long* counters;
  unsigned long long mark;            // 40 bits
};

// t / d by multiplication, exact for t * d < 2^32 (m = floor(2^32 / d) + 1)
struct Divisor {
  unsigned d, m;
  __device__ __forceinline__ explicit Divisor(unsigned d_) : d(d_), m(d_ > 1 ? 0xffffffffu / d_ + 1u : 0u) {}
  __device__ __forceinline__ unsigned div(unsigned t) const { return d > 1 ? __umulhi(t, m) : t; }
};

// Where a head's tokens go.  new_t = c0 * (e1 e2) + c1 * e2 + c2 with c_i the coordinate p_i and e_i its extent
// (permute.py:45-52): new_t is linear in the three coordinates of t.
struct Order {
  unsigned d12, d2, m0, m1, m2;
  Divisor by12, by2;
  bool small;
  // (inv: NULL, or the order back; t then counts in the dimensions permuted by p, permute.py:77-95)
  template <typename P> __device__ __forceinline__ Order(const ReorderParams& prm, P p, P inv, bool back) : by12(1), by2(1) {
    int p0 = p[0], p1 = p[1], p2 = p[2];
    unsigned d0 = prm.F, d1 = prm.H;
    d2 = prm.W;
    auto extent = [&](int i) { return i == 0 ? d0 : (i == 1 ? d1 : d2); };
    if (back) {
      const unsigned e0 = extent(p0), e1 = extent(p1), e2 = extent(p2);
      d0 = e0; d1 = e1; d2 = e2;
      p0 = inv[0]; p1 = inv[1]; p2 = inv[2];
    }
    const unsigned e1 = extent(p1), e2 = extent(p2);
    auto factor = [&](int c) { return (p0 == c ? e1 * e2 : 0u) + (p1 == c ? e2 : 0u) + (p2 == c ? 1u : 0u); };
    m0 = factor(0); m1 = factor(1); m2 = factor(2);
    d12 = d1 * d2;
    by12 = Divisor(d12); by2 = Divisor(d2);
    small = d0 * d12 < 65536u;          // (then t * d12 < 2^32 and the divisions are multiplications)
  }
  __device__ __forceinline__ unsigned operator()(unsigned t) const {
    const unsigned f = small ? by12.div(t) : t / d12, rest = t - f * d12;
    const unsigned y = small ? by2.div(rest) : rest / d2, w = rest - y * d2;
    return f * m0 + y * m1 + w * m2;
  }
};

template <typename V>
__global__ __launch_bounds__(256) void reorder_kernel(const ReorderParams prm) {
  const unsigned T = (unsigned)(prm.F * prm.H * prm.W);
  const int unit = (int)(blockIdx.x / prm.blocks_per_unit);
  const unsigned row0 = (blockIdx.x - unit * prm.blocks_per_unit) * prm.rows_per_block;
  const int h = unit % prm.NH;
  const Order order(prm, prm.orders + 3 * h, prm.inv_orders + 3 * h, prm.inv_orders != nullptr);
  const int64_t rb = prm.row_bytes;
  const char* src = prm.src + (int64_t)unit * T * rb;
  char* dst = prm.dst + (int64_t)unit * T * rb;
  const unsigned vpr = (unsigned)prm.row_bytes / sizeof(V);
  const unsigned n = (T - row0 < prm.rows_per_block ? T - row0 : prm.rows_per_block) * vpr;     // pieces of this block
  for (unsigned i0 = threadIdx.x; i0 < n; i0 += 256 * REORDER_UNROLL) {
    V val[REORDER_UNROLL];
#pragma unroll
    for (int k = 0; k < REORDER_UNROLL; ++k)
      if (i0 + 256 * k < n) val[k] = *reinterpret_cast<const V*>(src + row0 * rb + (int64_t)(i0 + 256 * k) * sizeof(V));
#pragma unroll
    for (int k = 0; k < REORDER_UNROLL; ++k) {
      const unsigned i = i0 + 256 * k, r = prm.vshift >= 0 ? i >> prm.vshift : i / vpr;
      if (i < n) *reinterpret_cast<V*>(dst + order(row0 + r) * rb + (i - r * vpr) * sizeof(V)) = val[k];
    }
  }
}

// The six orders of the three dimensions and the orders back (fa2_custom_mask/functional.py:23-26, 69-76), by number.
__constant__ signed char ORDERS[6][3] = {{0, 1, 2}, {0, 2, 1}, {1, 2, 0}, {1, 0, 2}, {2, 1, 0}, {2, 0, 1}};
__constant__ signed char ORDERS_BACK[6][3] = {{0, 1, 2}, {0, 2, 1}, {2, 0, 1}, {1, 0, 2}, {2, 1, 0}, {1, 2, 0}};

__global__ __launch_bounds__(GROUP_THREADS, 4) void reorder_group_kernel(const ReorderParams prm) {
  // linear id -> (unit, part): units in groups of 8, one per XCD (workgroups go to the XCDs round-robin), the parts of
  // a unit one after the other
  const unsigned xcd = blockIdx.x & 7, k = blockIdx.x >> 3;
  const int unit = (int)((k / prm.parts) * 8 + xcd);
  const unsigned part = k % prm.parts;
  if (unit >= prm.units) return;
  const int per = prm.BS * prm.NH, ten = unit / per, bh = unit - ten * per, h = bh % prm.NH;
  long long number = prm.number_bytes == 8 ? ((const long long*)prm.numbers)[h] : ((const int*)prm.numbers)[h];
  if (number < 0) number += 6;
  if (number < 0 || number > 5) {                   // no order: the head stays as it is, and the next call says so
    if (part == 0 && threadIdx.x == 0) __hip_atomic_store(prm.bad_number, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    return;
  }
  if (number == 0) return;                          // the identity
  const Order order(prm, ORDERS[number], ORDERS_BACK[number], prm.inverse != 0);
  char* rows = prm.x[ten] + (bh / prm.NH) * prm.sb[ten] + h * prm.sh[ten];
  const int64_t xs = prm.st[ten];
  const unsigned vpr = (unsigned)prm.row_bytes >> 4, T = (unsigned)(prm.F * prm.H * prm.W), total = T * vpr;
  const unsigned begin = part * prm.pieces_per_part;
  const unsigned end = total - begin < prm.pieces_per_part ? total : begin + prm.pieces_per_part;
  auto row_of = [&](unsigned i) { return prm.vshift >= 0 ? i >> prm.vshift : i / vpr; };
  uintx4 val[GROUP_PIECES];
#pragma unroll
  for (int j = 0; j < GROUP_PIECES; ++j) {
    const unsigned i = begin + threadIdx.x + GROUP_THREADS * j;
    if (i < end) {
      const unsigned r = row_of(i);
      val[j] = *reinterpret_cast<const uintx4*>(rows + r * xs + (i - r * vpr) * 16);
    }
  }
  // everything this workgroup asked for has arrived (a wavefront's own loads by its wait, all of them by the barrier)
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (prm.parts > 1) {
    __shared__ int outcome;            // 0: store, 1: the group is broken, 2: ... and this workgroup is the last to leave it
    if (threadIdx.x == 0) {
      unsigned long long* counter = prm.counters + (int64_t)unit * COUNTER_STRIDE;
      const unsigned long long mark = prm.mark << 24;
      // count in; the first of the group replaces what earlier launches left
      unsigned long long v = __hip_atomic_load(counter, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      bool in = false;
      if ((v >> 24) != prm.mark) {
        in = __hip_atomic_compare_exchange_strong(counter, &v, mark | 1ull, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (in) v = mark | 1ull;
      }
      if (!in) v = __hip_atomic_fetch_add(counter, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1ull;
      // the last one in clears the counter for a replay of this launch (same mark); the others see it complete or cleared
      auto complete = [&](unsigned long long u) { return (u >> 24) != prm.mark || (!(u & BROKEN) && (u & COUNT_MASK) == prm.parts); };
      if (complete(v)) __hip_atomic_store(counter, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const unsigned long long t0 = __builtin_readsteadycounter();
      while (!complete(v) && !(v & BROKEN)) {
        if (__builtin_readsteadycounter() - t0 > WAIT_TICKS) {
          // (a failure brings the value another member made of it, at most one per member)
          if (__hip_atomic_compare_exchange_strong(counter, &v, v | BROKEN, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) v |= BROKEN;
        } else {
          __builtin_amdgcn_s_sleep(2);
          v = __hip_atomic_load(counter, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
      }
      outcome = 0;
      if (!complete(v)) {
        const unsigned long long left = __hip_atomic_fetch_add(counter, LEFT_ONE, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        outcome = ((left >> 16) & 0xffull) + 1 == prm.parts ? 2 : 1;
        if (outcome == 2) __hip_atomic_store(counter, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    __syncthreads();
    const int what = outcome;
    if (what == 1) return;
    if (what == 2) {
      for (unsigned c = 0; c < (unsigned)prm.row_bytes; c += 4) {
        unsigned* column = reinterpret_cast<unsigned*>(val);
#pragma unroll
        for (int j = 0; j < 4 * GROUP_PIECES; ++j) {
          const unsigned r = threadIdx.x + GROUP_THREADS * j;
          if (r < T) column[j] = *reinterpret_cast<const unsigned*>(rows + r * xs + c);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
#pragma unroll
        for (int j = 0; j < 4 * GROUP_PIECES; ++j) {
          const unsigned r = threadIdx.x + GROUP_THREADS * j;
          if (r < T) *reinterpret_cast<unsigned*>(rows + order(r) * xs + c) = column[j];
        }
      }
      return;
    }
  }
#pragma unroll
  for (int j = 0; j < GROUP_PIECES; ++j) {
    const unsigned i = begin + threadIdx.x + GROUP_THREADS * j;
    if (i < end) {
      const unsigned r = row_of(i);
      // (non-temporal: 154 against 178 us)
      __builtin_nontemporal_store(val[j], reinterpret_cast<uintx4*>(rows + order(r) * xs + (i - r * vpr) * 16));
    }
  }
}

static void pieces_of_row(ReorderParams& prm, int piece) {
  const unsigned vpr = prm.row_bytes / piece;
  prm.vshift = (vpr & (vpr - 1)) == 0 ? __builtin_ctz(vpr) : -1;
}

int launch_reorder(const void* x, void* out, int BS, int NH, int F, int Hh, int W, int row_bytes,
                   const int32_t* orders, const int32_t* inv_orders, hipStream_t st) {
  ReorderParams prm = {};
  prm.src = (const char*)x; prm.dst = (char*)out;
  prm.BS = BS; prm.NH = NH; prm.F = F; prm.H = Hh; prm.W = W; prm.row_bytes = row_bytes;
  prm.orders = orders; prm.inv_orders = inv_orders;
  const bool v16 = row_bytes % 16 == 0 && ((uintptr_t)x & 15) == 0 && ((uintptr_t)out & 15) == 0;
  const int piece = v16 ? 16 : 4;
  pieces_of_row(prm, piece);
  const unsigned T = (unsigned)(F * Hh * W), rows = 256u * REORDER_UNROLL / (unsigned)(row_bytes / piece);
  prm.rows_per_block = rows < 1 ? 1 : rows;
  prm.blocks_per_unit = (T + prm.rows_per_block - 1) / prm.rows_per_block;
  const int64_t blocks = (int64_t)BS * NH * prm.blocks_per_unit;
  if (blocks > 0x7fffffffLL) return BSATTN_ERR_RANGE;
  if (v16) hipLaunchKernelGGL(reorder_kernel<uintx4>, dim3((unsigned)blocks), dim3(256), 0, st, prm);
  else hipLaunchKernelGGL(reorder_kernel<unsigned>, dim3((unsigned)blocks), dim3(256), 0, st, prm);
  return launch_status();
}

// Workgroups per head of reorder_group_kernel; 0 if the head does not fit a group.
static int group_parts(int F, int Hh, int W, int row_bytes) {
  const int64_t T = (int64_t)F * Hh * W, pieces = T * (row_bytes / 16), most = GROUP_THREADS * GROUP_PIECES;
  const int64_t parts = (pieces + most - 1) / most;
  return T <= GROUP_ROWS_MAX && parts <= GROUP_PARTS_MAX ? (int)parts : 0;
}

// 0: no in-place reorder at this size
size_t reorder_workspace_bytes(int n, int BS, int NH, int F, int Hh, int W, int row_bytes) {
  const int parts = group_parts(F, Hh, W, row_bytes);
  const int64_t units = (int64_t)n * BS * NH;
  if (parts == 0 || (units + 7) / 8 * 8 * parts > 0x7fffffffLL) return 0;
  return (size_t)units * COUNTER_STRIDE * sizeof(unsigned long long);
}

// Where a device's kernels report a permutation number outside the table: a word of host memory per device, allocated by
// the first call on it and kept (a call that is being captured may make that allocation too).
struct BadNumber { unsigned* host; unsigned* device; };
static int bad_number_word(BadNumber& w) {
  static std::mutex mu;
  static BadNumber words[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return BSATTN_ERR_LAUNCH;
  std::lock_guard<std::mutex> lock(mu);
  if (words[dev].host == nullptr) {
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    if (hipThreadExchangeStreamCaptureMode(&mode) != hipSuccess) return BSATTN_ERR_LAUNCH;
    void *host = nullptr, *device = nullptr;
    const bool ok = hipHostMalloc(&host, sizeof(unsigned), hipHostMallocMapped) == hipSuccess &&
                    hipHostGetDevicePointer(&device, host, 0) == hipSuccess;
    (void)hipThreadExchangeStreamCaptureMode(&mode);
    if (!ok) return BSATTN_ERR_LAUNCH;
    *(unsigned*)host = 0;
    words[dev] = {(unsigned*)host, (unsigned*)device};
  }
  w = words[dev];
  return BSATTN_OK;
}

int launch_reorder_inplace(void* const* x, const int64_t* strides, int n, int BS, int NH, int F, int Hh, int W,
                           int row_bytes, const void* numbers, int number_bytes, int inverse, void* ws, hipStream_t st) {
  ReorderParams prm = {};
  for (int i = 0; i < n; ++i) {
    prm.x[i] = (char*)x[i];
    prm.sb[i] = strides[3 * i]; prm.sh[i] = strides[3 * i + 1]; prm.st[i] = strides[3 * i + 2];
  }
  prm.units = n * BS * NH;
  prm.BS = BS; prm.NH = NH; prm.F = F; prm.H = Hh; prm.W = W; prm.row_bytes = row_bytes;
  prm.numbers = numbers; prm.number_bytes = number_bytes; prm.inverse = inverse;
  BadNumber bad;
  if (const int rc = bad_number_word(bad); rc != BSATTN_OK) return rc;
  if (__atomic_load_n(bad.host, __ATOMIC_RELAXED) != 0 && __atomic_exchange_n(bad.host, 0u, __ATOMIC_RELAXED) != 0) return BSATTN_ERR_ORDER;
  prm.bad_number = bad.device;
  prm.counters = (unsigned long long*)ws;
  do { prm.mark = next_epoch() & 0xffffffffffull; } while (prm.mark == 0);
  pieces_of_row(prm, 16);
  const int parts = group_parts(F, Hh, W, row_bytes), pieces = F * Hh * W * (row_bytes / 16);
  prm.parts = (unsigned)parts;
  prm.pieces_per_part = (unsigned)((pieces + parts - 1) / parts);
  hipLaunchKernelGGL(reorder_group_kernel, dim3((unsigned)((prm.units + 7) / 8 * 8 * parts)), dim3(GROUP_THREADS), 0, st, prm);
  return launch_status();
}

}  // namespace bsattn
