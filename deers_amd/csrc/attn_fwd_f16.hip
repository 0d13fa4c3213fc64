// Fused causal attention forward, f16 storage / f32 accumulate, gfx950: launches that the 32-row form
// (attn_split_f16.hip) leaves to 128 rows per workgroup.  The kernel is attn_fwd_f16_bp.h; here are the order of its
// workgroups and its launch.
//
// Replaces the op chain of src/models/gpt.rs:139-144 (matmul, scalar_mul,
// causal_mask + add, log_sum_exp, sub, exp, matmul) with one kernel that never
// materialises the [T,T] score tensor.
//
// Work decomposition
//   grid  = one workgroup per (head, 128-row query tile), dealt to the XCDs so a
//           head stays on one XCD; 256 threads = 4 waves; wave w owns query rows
//           [q0 + 32w, q0 + 32w + 32) of the tile.
//   loop  over key/value blocks of 32 rows, stopping at the diagonal; only the diagonal block is masked.
//   S^T   = K Q^T on v_mfma_f32_32x32x16_f16 (K row-major in LDS as the A operand, the wave's Q rows in registers as
//           the B operand).  In this orientation every lane owns ONE query column of the 32x32 accumulator, so row max /
//           row sum are in-lane reductions plus one exchange with lane+32, and a rescale of O is a per-lane scalar.
//   O^T  += V^T P^T: P^T is taken straight from the S^T accumulator registers as the B operand; V^T fragments come from
//           the row-major V block in LDS through ds_read_b64_tr_b16.
#include <algorithm>
#include <map>
#include <vector>

#include "attn_fwd_f16_bp.h"
#include "common.h"

namespace deers {

// What the device holds of the block-pipelined kernel: CUs of an XCD and workgroups of a CU.
template <int D>
static void resident_capacity(int* n_cu, int* per_cu) {
  static int cus = 0, wgs = 0;  // launches are serialised by the caller
  if (cus == 0) {
    int dev = 0, all = 0;
    (void)hipGetDevice(&dev);
    (void)hipDeviceGetAttribute(&all, hipDeviceAttributeMultiprocessorCount, dev);
    (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&wgs, attn_fwd_f16_bp_kernel<D, false>, 256, BpCfg<D>::kLds);
    cus = std::max(all / 8, 1);
  }
  *n_cu = cus;
  *per_cu = wgs;
}

// Builds the TileOrder of a launch of whole heads per XCD whose workgroups are all resident at once (their
// number does not exceed what the chip holds).  Workgroup position p of an XCD (id / 8)
// lands on CU p % cus_per_xcd when the dispatcher fills an empty chip, so positions p,
// p + cus, p + 2 cus share a CU and its issue ports: tiles are dealt longest first to the
// CU with the smallest total that still has a free slot.  Returns nullptr when the tiles
// do not all fit (then the dispatcher's own longest-first hand-out is the better order).
// Built at the first launch of a geometry and kept on the host for the life of the
// process; no device memory.
template <int D>
static const TileOrder* resident_order(int heads_per_xcd, int T, int n_cu, int per_cu) {
  const int n_qtiles = (T + kFwdBM - 1) / kFwdBM;
  const int n_items = heads_per_xcd * n_qtiles;
  if (n_items > n_cu * per_cu || n_items > kMaxResidentTiles) return nullptr;
  struct Entry {
    bool usable = false;  // the table is filled in
    TileOrder order{};
  };
  static std::map<std::pair<int, int>, Entry> cache;  // launches are serialised by the caller
  const auto found = cache.find({heads_per_xcd, T});
  if (found != cache.end()) return found->second.usable ? &found->second.order : nullptr;
  Entry& entry = cache[{heads_per_xcd, T}];
  std::vector<long> load(n_cu, 0);
  std::vector<int> used(n_cu, 0);
  std::vector<char> filled((size_t)n_items, 0);
  for (int qt = n_qtiles - 1; qt >= 0; --qt) {  // descending cost
    const int cost = std::min(T - 1, qt * kFwdBM + kFwdBM - 1) / 64 + 1;
    for (int h = 0; h < heads_per_xcd; ++h) {
      int best = -1;
      for (int c = 0; c < n_cu; ++c)
        if (used[c] < per_cu && used[c] * n_cu + c < n_items && (best < 0 || load[c] < load[best])) best = c;
      if (best < 0) return nullptr;
      const int pos = used[best] * n_cu + best;
      entry.order.code[pos] = (h << 16) | qt;
      filled[pos] = 1;
      load[best] += cost;
      ++used[best];
    }
  }
  for (int i = 0; i < n_items; ++i)
    if (!filled[i]) return nullptr;
  entry.usable = true;
  return &entry.order;
}

template <int D>
static void launch_fwd_f16_d(const FwdParams& p, int B, bool from_q, hipStream_t stream) {
  const int BH = B * p.H;
  const int n_qtiles = (p.T + kFwdBM - 1) / kFwdBM;
  // heads that the XCDs cannot share out whole (9 x 8192 x 128: 218 us with two heads on one XCD, 163
  // with the ninth head's tiles dealt to all; 25 x 4096 x 64 74 -> 65, 20 x 2048 x 64 30.6 -> 29.8)
  const bool even = BH % 8 != 0;
  const int heads_per_xcd = even ? 0 : (BH + 7) / 8;
  const int grid = even ? map_even_blocks(n_qtiles, BH) : 8 * n_qtiles * heads_per_xcd;
  static bool attr_set = false;  // launches are serialised by the caller
  if (!attr_set) {
    allow_lds(attn_fwd_f16_bp_kernel<D, false>, BpCfg<D>::kLds);
    if constexpr (D > 32) allow_lds(attn_fwd_f16_bp_kernel<D, true>, BpCfg<D>::kLds);
    attr_set = true;
  }
  static const TileOrder kNoTable = [] {
    TileOrder t{};
    t.code[0] = -1;
    return t;
  }();
  LaunchScope scope("attn_fwd_f16", stream);
  // While all workgroups fit (three to a CU at head widths 32 and 64, two at 128) every one of them is resident from the
  // start and they are placed for even CU totals: by a table where an XCD has whole heads, by paired_block where the
  // tiles of some heads are dealt to all XCDs.  Longest first instead, the CUs that have two get the longest ones and
  // others beside them (16 heads x 4096 x 64 in a kernel with 64-row tiles, two workgroups to each CU: 61.5 us, with even
  // totals 58.7).  Beyond that the dispatcher hands out each XCD's list longest first.
  int n_cu, per_cu;
  resident_capacity<D>(&n_cu, &per_cu);
  const bool paired = even && grid / 8 > n_cu && grid / 8 <= per_cu * n_cu;
  const TileOrder* order = even ? nullptr : resident_order<D>(heads_per_xcd, p.T, n_cu, per_cu);
  auto kernel = attn_fwd_f16_bp_kernel<D, false>;
  if constexpr (D > 32)
    if (from_q) kernel = attn_fwd_f16_bp_kernel<D, true>;
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(256), BpCfg<D>::kLds, stream, p, BH, n_qtiles, paired ? -n_cu : heads_per_xcd,
                     order ? *order : kNoTable);
}

bool attn_fwd_f16_split_takes(int64_t BH, int64_t T, int64_t D);  // attn_split_f16.hip
bool attn_bwd_f16_split_takes(int64_t BH, int64_t T, int64_t D);

// Whether a launch's scores are formed from Q itself, or from Q * scale * log2(e) rounded to f16.  Forward and backward
// ask the same question: a probability that is recomputed from another score than it was normalised with is off by
// up to |S| * 2^-11, dV of a peaked row by more than 5e-3.
//   both in the 32-row form       from Q (a product per score costs them nothing)
//   128 rows, D = 64 and 128      from Q up to two workgroups to a CU, beyond that from scaled queries, 6 % faster
//                                 (forward 16 x 4096 x 64 53.1 / 49.2 us; O 2.5e-4 / 3.2e-4 from 64 bits, relative)
//   else                          from scaled queries: the 128-row backward after a 32-row forward, and head width 32
// The 128-row backward starts from -LSE / scale: not for scales whose reciprocal leaves f32.
bool attn_f16_from_q(int64_t BH, int64_t T, int64_t D, float scale) {
  if (attn_fwd_f16_split_takes(BH, T, D)) return attn_bwd_f16_split_takes(BH, T, D);
  return D > 32 && (BH + 7) / 8 * ((T + kFwdBM - 1) / kFwdBM) <= 64 && scale >= 0x1p-60f;
}

void launch_attn_fwd_f16(const FwdParams& p, int B, int D, bool from_q, hipStream_t stream) {
  switch (D) {
    case 32: launch_fwd_f16_d<32>(p, B, from_q, stream); break;
    case 64: launch_fwd_f16_d<64>(p, B, from_q, stream); break;
    case 128: launch_fwd_f16_d<128>(p, B, from_q, stream); break;
  }
}

}  // namespace deers
