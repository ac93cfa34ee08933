// fa_plan.cpp -- host-only half of libfa_mi355x.so: the kernel table's
// metadata, tile planning and the C-ABI calls that make no HIP call
// (fa_validate, fa_query_config, fa_default_kv_splits,
// fa_workspace_kv_splits, fa_split_workspace_bytes, fa_kernel_info, fa_kernel_wg_per_cu, ...).
//
// Plain C++17 with no HIP header: fa_fwd.hip includes this file (the library
// stays one translation unit, and the kernel pointer table there is built
// from kKernelMeta below, entry for entry), and the host sanitizer test
// compiles it on its own with g++ -fsanitize=address,undefined.
//
// Counterparts in the reference (flash_attention_forward.py): argument checks
// of `_validate_inputs` (:1114-1122), the tile resolution of `_default_tiling`
// / `_resolve_tiling` (:221-242, :626-631), the grid of `_build_grid` and
// `_get_persistent_programs` (:616-623, :1125-1127), and `_describe_runtime`
// (:634-644).
#include <math.h>
#include <stdint.h>

#include "fa_fwd.h"

namespace {

// Rows a kernel may address past a tensor's end (a last partial m-tile, or the
// DMAs issued past the last KV tile); >= every BLOCK_M and ring depth * BLOCK_N.
constexpr int kRowMargin = 1024;

constexpr bool is_supported_head_dim(int d) { return d == 16 || d == 32 || d == 64 || d == 128 || d == 256; }
constexpr bool is_valid_dtype(int dt) {
  return dt == FA_DTYPE_FP16 || dt == FA_DTYPE_BF16 || dt == FA_DTYPE_FP16_V_E5M2 || dt == FA_DTYPE_BF16_V_E5M2;
}
constexpr bool v_is_fp8(int dt) { return dt == FA_DTYPE_FP16_V_E5M2 || dt == FA_DTYPE_BF16_V_E5M2; }
constexpr bool out_is_bf16(int dt) { return dt == FA_DTYPE_BF16 || dt == FA_DTYPE_BF16_V_E5M2; }
// Head dims of the fp8-V kernels.
constexpr bool is_supported_fp8v_head_dim(int d) { return is_supported_head_dim(d); }

// ---------------------------------------------------------------------------
// Kernel table metadata.  Two kernel families (fa_fwd.hip):
//  * kDma: fa_fwd_dma_kernel<D, BN, NW, stages, wg_per_cu, bf16, causal, fp8 V>,
//    4 waves (BLOCK_M 128), K/V through a 2-stage LDS ring filled by DMA;
//  * kPingPong: fa_fwd_pp_kernel<D, BN, stages, bf16, causal>, 8 waves
//    (BLOCK_M 256) in two phase-shifted groups, separate K and V rings of
//    `stages` tiles, one workgroup per CU, no split-KV.
enum KernelKind : int32_t { kDma = 0, kPingPong = 1 };

struct KernelMeta {
  int32_t kind;
  int32_t D, dtype, causal, BN, NW;
  int32_t stages;     // LDS stages of the K/V ring (ping-pong: per ring)
  int32_t wg_per_cu;  // resident workgroups per CU (registers and LDS)
  bool splittable;    // supports split-KV (partial outputs + merge)
};

// Dynamic LDS bytes of one workgroup: the Q area of the kernels with one
// workgroup per CU, 16-bit V and fewer 1 KB DMA chunks per wave than 32 Q rows
// fill (BLOCK_M rows of 2 D bytes); 0 for the others.
constexpr int32_t kernel_dyn_lds_bytes(const KernelMeta &m) {
  if (m.kind == kPingPong || m.wg_per_cu != 1 || v_is_fp8(m.dtype)) return 0;
  const int32_t ndma = 2 * (m.BN * 2 * m.D / 1024 / m.NW);  // K and V chunks per wave and tile
  return ndma < m.D / 16 ? 32 * m.NW * 2 * m.D : 0;
}

// LDS bytes of one workgroup (what the kernels' __shared__ arrays and the
// dynamic Q area add up to; fa_fwd.hip checks every entry against its
// kernel's own layout).
constexpr int32_t kernel_lds_bytes(const KernelMeta &m) {
  if (m.kind == kPingPong) return 2 * m.stages * m.BN * 2 * m.D;  // K and V rings
  const int32_t k_tile = m.BN * 2 * m.D;
  const int32_t v_tile = m.BN * (v_is_fp8(m.dtype) ? 1 : 2) * m.D;
  const int32_t v_ipt = v_tile / 1024;  // 1 KB DMA instructions per V tile
  const int32_t v_ipw = v_ipt >= m.NW ? v_ipt / m.NW : 1;
  return m.stages * (k_tile + v_ipw * m.NW * 1024) + kernel_dyn_lds_bytes(m);
}

constexpr KernelMeta dma(int D, int BN, int occ, int dtype, int causal) {
  return KernelMeta{kDma, D, dtype, causal, BN, 4, 2, occ, true};
}
constexpr KernelMeta pp(int D, int BN, int rings, int dtype, int causal) {
  return KernelMeta{kPingPong, D, dtype, causal, BN, 8, rings, 1, false};
}

#define FA_DMA4(D, BN, OCC)                                                                     \
  dma(D, BN, OCC, FA_DTYPE_FP16, 0), dma(D, BN, OCC, FA_DTYPE_FP16, 1), dma(D, BN, OCC, FA_DTYPE_BF16, 0), \
      dma(D, BN, OCC, FA_DTYPE_BF16, 1)
#define FA_PP4(D, BN, NR) \
  pp(D, BN, NR, FA_DTYPE_FP16, 0), pp(D, BN, NR, FA_DTYPE_FP16, 1), pp(D, BN, NR, FA_DTYPE_BF16, 0), pp(D, BN, NR, FA_DTYPE_BF16, 1)
// fp8-e5m2 V with fp16 / bf16 Q, K, O (dtype codes FA_DTYPE_*_V_E5M2).
#define FA_DMA8_4(D, BN, OCC)                                                                             \
  dma(D, BN, OCC, FA_DTYPE_FP16_V_E5M2, 0), dma(D, BN, OCC, FA_DTYPE_FP16_V_E5M2, 1),                   \
      dma(D, BN, OCC, FA_DTYPE_BF16_V_E5M2, 0), dma(D, BN, OCC, FA_DTYPE_BF16_V_E5M2, 1)

// The first entry matching (D, dtype, causal, BLOCK_N, waves) serves a launch.
constexpr KernelMeta kKernelMeta[] = {
    FA_DMA4(128, 64, 2),
    FA_PP4(128, 64, 4),
    // D = 128, 32-key tiles: non-causal at three workgroups per CU (1.5-3.7%
    // faster than two); the causal kernel spills at three and keeps two.
    dma(128, 32, 3, FA_DTYPE_FP16, 0), dma(128, 32, 2, FA_DTYPE_FP16, 1),
    dma(128, 32, 3, FA_DTYPE_BF16, 0), dma(128, 32, 2, FA_DTYPE_BF16, 1),
    // D <= 64 is softmax (VALU) bound, and a single wave issues VALU work
    // well below the SIMD's rate: more resident waves fill the gaps.  D = 64
    // default: 64-key tiles, whose 32 KB of LDS and <= 168 registers let three
    // workgroups share a CU (0.7-7.7% faster than 128-key tiles at two, on
    // every D = 64 workload measured, fp16 and bf16, causal and not).
    FA_DMA4(64, 64, 3),
    FA_PP4(64, 64, 4),
    FA_DMA4(64, 32, 2),
    FA_DMA4(64, 128, 2),
    // D = 256: 512 registers per wave (O^T alone is 128), so one workgroup
    // per CU; 32-key tiles keep S, P and the operand fragments small.  The
    // 64-key kernels are candidates for the tile sweep.
    FA_DMA4(256, 32, 1),
    FA_DMA4(256, 64, 1),
    // D = 32: four workgroups per CU when causal (8-9% faster than two);
    // non-causal measured 1.7% slower at four, so it keeps two.
    dma(32, 64, 2, FA_DTYPE_FP16, 0), dma(32, 64, 4, FA_DTYPE_FP16, 1),
    dma(32, 64, 2, FA_DTYPE_BF16, 0), dma(32, 64, 4, FA_DTYPE_BF16, 1),
    // D = 16: a 64-key tile is only two DMA instructions; 128 keys give each
    // wave one.  Three workgroups per CU (4-10% faster than two).
    FA_DMA4(16, 128, 3),
    FA_DMA8_4(128, 64, 2),
    // fp8 V at D <= 64: three workgroups per CU (causal 6.7-8.4% faster than
    // two, non-causal equal).
    FA_DMA8_4(64, 64, 3),
    FA_DMA8_4(256, 64, 1),
    FA_DMA8_4(32, 64, 3),
    FA_DMA8_4(16, 128, 3),
};
#undef FA_DMA4
#undef FA_PP4
#undef FA_DMA8_4
constexpr int kNumKernels = sizeof(kKernelMeta) / sizeof(kKernelMeta[0]);

constexpr bool table_fits_lds() {
  for (const KernelMeta &m : kKernelMeta)
    if (kernel_lds_bytes(m) * m.wg_per_cu > 160 * 1024) return false;
  return true;
}
static_assert(table_fits_lds(), "LDS budget of one gfx950 CU");

// Default (BLOCK_N, waves); BLOCK_M = 32 * waves.
void default_tiling(const fa_fwd_params *p, int *bn, int *nw) {
  *nw = 4;
  // fp8 V: 64-key tiles (D = 16: 128), one 32x32x64 MFMA per 64 keys and 32
  // head dims.  16-bit V: 64 keys, except D = 16 (128) and D = 256 (32).
  if (v_is_fp8(p->dtype)) {
    *bn = p->D == 16 ? 128 : 64;
    return;
  }
  *bn = p->D == 16 ? 128 : p->D == 256 ? 32 : 64;
  if (p->D != 128 || p->causal) return;
  // Non-causal D = 128: the 64-key kernel (two workgroups per CU, its tile
  // carried as two 32-key blocks) is 1-10% faster than the 32-key one (three per
  // CU) on full grids and 8-30% up to one tile per CU (fp16, us, 32 against 64
  // keys: H16 S2048 44.3 / 37.5, H128 S2048 255 / 250, H16 S1024 23.0 / 18.5).
  // Timed at 16 to 16384 keys and 1 to 32768 tiles, the 32-key kernel is the faster
  //  * up to 48 keys, where half of a 64-key tile is padding (H1024 S32 9.8 / 12.4,
  //    S48 13.5 / 14.6);
  //  * up to 96 keys on grids of more tiles than the 512 workgroups that the
  //    64-key kernel has on the chip: a unit is then mostly prologue and
  //    epilogue, which the third workgroup per CU hides (H1024 S64 15.5 / 16.3,
  //    S96 20.6 / 23.2).  From 4096 tiles on, eight rounds, it no longer pays
  //    (H4096 S96 91.5 / 85.7).
  // At 8192 and 16384 keys with 4096 tiles and more the two are within 2% of each
  // other, either one ahead from run to run.
  const int64_t heads = (int64_t)p->B * p->H;  // < 2^62
  const int64_t tiles = ((int64_t)p->Sq + 127) / 128 * (heads < INT32_MAX ? heads : INT32_MAX);
  if (p->Sk <= 48 || (p->Sk <= 96 && tiles > 512 && tiles < 4096)) *bn = 32;
}

int find_kernel(int D, int dtype, int causal, int BN, int NW) {
  for (int i = 0; i < kNumKernels; ++i) {
    const KernelMeta &e = kKernelMeta[i];
    if (e.D == D && e.dtype == dtype && e.causal == causal && e.BN == BN && e.NW == NW) return i;
  }
  return -1;
}

struct Plan {
  int kernel;
  int BM, BN, NW;
  int n_mtiles;
  int64_t total_tiles;  // (head, m-tile) tiles
  int grid;
  int split_tiles;      // KV tiles per split-KV run (0: no split)
};

constexpr int kMaxKvSplits = 64;

// CUs of an MI355X; fa_fwd asks the device, the host-only calls assume this.
constexpr int kDefaultCuCount = 256;

int make_plan(const fa_fwd_params *p, Plan *out, int cu_count = kDefaultCuCount, int splits = 1) {
  int bn, nw;
  if (p->block_m == 0 && p->block_n == 0) {
    default_tiling(p, &bn, &nw);
  } else {
    if (p->block_m <= 0 || p->block_n <= 0 || p->block_m % 32 != 0) return FA_ERR_TILING;
    bn = p->block_n;
    nw = p->block_m / 32;
  }
  const int kid = find_kernel(p->D, p->dtype, p->causal ? 1 : 0, bn, nw);
  if (kid < 0) return FA_ERR_TILING;
  out->kernel = kid;
  out->BN = bn;
  out->NW = nw;
  out->BM = 32 * nw;
  out->n_mtiles = (int)(((int64_t)p->Sq + out->BM - 1) / out->BM);
  const int64_t heads = (int64_t)p->B * p->H;  // < 2^62: no overflow
  if (heads > INT32_MAX) return FA_ERR_SHAPE;
  out->total_tiles = (int64_t)out->n_mtiles * heads;
  if (out->total_tiles > INT32_MAX) return FA_ERR_SHAPE;
  // Persistent grid: as many workgroups as fit on the GPU at once, pulling
  // tiles from the tile queues; PERSISTENT_PROGRAMS (num_programs) overrides
  // the count.
  const int64_t kv_tiles = ((int64_t)p->Sk + bn - 1) / bn;
  out->split_tiles = splits > 1 ? (int)((kv_tiles + splits - 1) / splits) : 0;
  const int64_t units = out->total_tiles * (splits > 1 ? splits : 1);
  if (units > INT32_MAX) return FA_ERR_SHAPE;
  int64_t grid = (int64_t)kKernelMeta[kid].wg_per_cu * (cu_count > 0 ? cu_count : kDefaultCuCount);
  if (p->num_programs > 0) grid = p->num_programs;
  if (grid > units) grid = units;
  out->grid = (int)grid;
  return FA_OK;
}

// ---------------------------------------------------------------------------
// Order of the persistent grid's work.  A unit is a (head, m-tile, KV run); the
// units are dealt to nq queues (TileQueue in fa_fwd.hip), and ticket t of queue x
// is the t-th unit of its list.  Queue x owns heads x, x + nq, x + 2 nq, ..., so a
// whole head's K/V is read through one queue's L2; it takes them in groups of 8,
// and inside a group KV run by KV run and m-tile by m-tile, heaviest first
// (causal: the largest), each through the group's heads.  The B*H mod nq heads
// left over go with the last group: their tiles are dealt to the queues in turn,
// each m-tile's after the queue's own heads (make_tile_order has one exception).
// So every list stays heaviest first, and the queues' unit counts differ by at
// most one, as the workgroups of a grid of one per unit do.  Dealt before
// everything else, light tiles with heavy ones, the left-over heads made causal
// B*H = 15 S4096 (fp16) 48 us at D = 32 and 201 at D = 256, against 35 and 165
// here and 37 and 173 with whole heads on some of the queues.
//
// The padding groups what the compiler loads together: the default kernels spill
// 54-103 scalar registers with it, up to 25 more without.
struct TileOrder {
  int32_t nq;        // queues
  int32_t n_mtiles;
  int32_t ranks;     // m-tiles * KV runs
  int32_t heads0;    // queue 0's heads: as below, or, with a whole left-over head, heads + nq
  int32_t heads;     // B*H; less the left-over head where queue 0 has it whole
  int32_t pad[2];
  int32_t cols;      // heads of a group but the last: nq * heads per queue and group
  int32_t own;       // where heads are left over: the last group's other heads
  int32_t last;      // index of the last group
  int32_t tickets;   // tickets of a queue in a group but the last
  int32_t pad2;
};

// `grid` workgroups on `cu_count` CUs.
constexpr TileOrder make_tile_order(int heads, int n_mtiles, int splits, int nq, bool causal, int grid, int cu_count) {
  // Groups of 8 heads per queue.  Measured on the benchmark workloads against
  // groups of 2..64 heads: within 1% of the best time on each, with the
  // least HBM traffic or close to it (e.g. B8 H32 S3000 causal: 646 us and
  // 2.5 GB fetched per launch, against 804 us and 6.6 GB for all 32 heads of
  // a queue at once; B16 H16 S1024: 87 us against 101 us).
  const int per_queue = heads / nq;  // >= 1
  const int left = heads % nq;
  const int group = per_queue < 8 ? per_queue : 8;
  TileOrder o = {};
  o.nq = nq;
  o.n_mtiles = n_mtiles;
  o.ranks = n_mtiles * splits;
  o.cols = nq * group;
  o.last = (per_queue - 1) / group;
  o.tickets = group * o.ranks;
  // Non-causal, where tiles are all alike: one left-over head stays whole, one
  // more of queue 0's own, on grids of more units than workgroups where its tiles
  // cost queue 0's CUs no further round.  Dealt, they make every queue start
  // one for a few tiles, 1-7% slower (fp16, us, whole / dealt: B*H = 97 S2048
  // D128 194 / 202, D256 449 / 484, 65 S1024 D128 48 / 50).  Where the whole head
  // costs a round more, dealt is up to 1.45x faster (9 S8192 D32), on grids of
  // one round up to 1.8x, and with two heads and more left over 1-7% on average.
  const int cus = cu_count / nq > 0 ? cu_count / nq : 1;  // of one queue
  const int64_t dealt = ((int64_t)heads * o.ranks + nq - 1) / nq, whole = (int64_t)(per_queue + 1) * o.ranks;
  const bool keep = !causal && left == 1 && (int64_t)heads * o.ranks > grid &&
                    (dealt + cus - 1) / cus == (whole + cus - 1) / cus;
  o.heads = keep ? heads - 1 : heads;
  o.heads0 = keep ? heads - 1 + nq : heads;
  // (With fewer than 8 queues, a program count's, the last group's heads all take turns.)
  o.own = left != 0 && !keep && nq == 8 ? heads - left - o.last * o.cols : 0;
  return o;
}

// Tickets of queue x.
__attribute__((always_inline)) constexpr uint32_t queue_tickets(const TileOrder &o, int x) {
  const uint32_t heads = (uint32_t)(x == 0 ? o.heads0 : o.heads);
  return (heads * (uint32_t)o.ranks - (uint32_t)x + (uint32_t)o.nq - 1) / (uint32_t)o.nq;
}

// Ticket t < queue_tickets(o, x) of queue x -> (head, m-tile, KV run): element
// x + nq * t of the group's list (rank, column), `cols` heads wide.
__attribute__((always_inline)) constexpr void tile_of_ticket(const TileOrder &o, int x, uint32_t t, bool causal, int *bh,
                                                             int *mt, int *split) {
  uint32_t g = t / (uint32_t)o.tickets;
  if (g > (uint32_t)o.last) g = (uint32_t)o.last;
  const uint32_t base = g * (uint32_t)o.cols;  // first head of the group
  const uint32_t cols = g == (uint32_t)o.last ? (uint32_t)(x == 0 ? o.heads0 : o.heads) - base : (uint32_t)o.cols;
  const uint32_t e = (uint32_t)x + (uint32_t)o.nq * (t - g * (uint32_t)o.tickets);
  const uint32_t rank = e / cols;
  uint32_t col = e - rank * cols;
  // Where cols is no multiple of the 8 queues, their turn moves on from rank to
  // rank; of each block of 8 whole heads, this queue's own is the one to take.
  if (col < (uint32_t)o.own) col = (col & ~7u) + (uint32_t)x;
  *bh = (int)(base + col);
  *split = (int)(rank / (uint32_t)o.n_mtiles);
  const int k = (int)(rank - (uint32_t)*split * (uint32_t)o.n_mtiles);
  *mt = causal ? o.n_mtiles - 1 - k : k;
}

bool aligned16(const void *ptr) { return ((uintptr_t)ptr & 15u) == 0; }

// Workspace of a split-KV launch: partial O, then (256-byte aligned) LSE.
// Sizes are formed in 128-bit arithmetic; a workspace of 2^62 bytes or more
// (no device has one) is reported as -1.
constexpr __int128 kMaxWorkspace = (__int128)1 << 62;
int64_t split_part_o_bytes(const fa_fwd_params *p, int splits) {
  const __int128 b = ((__int128)splits * p->B * p->H * p->Sq * p->D * 4 + 255) / 256 * 256;
  return b < kMaxWorkspace ? (int64_t)b : -1;
}
int64_t split_workspace_bytes(const fa_fwd_params *p, int splits) {
  const int64_t po = split_part_o_bytes(p, splits);
  const __int128 b = (__int128)po + (__int128)splits * p->B * p->H * p->Sq * 4;
  return po >= 0 && b < kMaxWorkspace ? (int64_t)b : -1;
}

// The split count that is estimated to be the fastest; with any_workspace false,
// of those that fa_default_kv_splits may return.
//
// A grid of at most one tile per CU takes as long as one workgroup needs for all
// its keys, and splitting them pays what the merge costs: its launch, and one pass
// of the partial O (tiles * splits of them) out and in.  Both are estimated in
// us from timings of 1960 shapes with up to 15 split counts each (6 to 320
// tiles, 300 to 16384 keys, every head dim, fp16, bf16 and e5m2 V):
//  * 5 us and a time per key that grows with D (H16 S1024 D128: 18.5 us, H8 S2048
//    29.4, H1 S4096 D16 31);
//  * the merge: 4.5 us, 0.2 per split and 0.03 per tile and split at D = 128
//    (0.6 of it where causal, as fitted: both masks store every partial O);
//  * a split call takes the host about 14.5 us, whatever its size.
// Tried are the powers of two and the counts that fill the CUs, in runs of at
// least 128 keys, none of them empty (H1 S10240 D32, 80 tiles: 36.5 us at 3
// splits, 47.1 at 2), on at most
//  * one workgroup per CU;
//  * causal, where half of the work is missing: 288 workgroups (H2 S6144 D128, 96
//    tiles: 39 us at 3 splits, 48 at 2), at D = 256 from runs of 1365 keys on (H2
//    S6144 74 / 87); 512 at D <= 128 with up to 128 tiles and such runs (H1 S16384
//    D128: 101 us at 4, 124 at 2); 384 for two runs of 2048 keys (H3 S6144 D256,
//    144 tiles: 99 us, 143 unsplit), not more (H4 S8192 D256, 256 tiles: 235 / 204).
// The picks are 2.2% slower than the fastest count on average.  Against the rule
// of 64K key-columns a run and one workgroup per CU, two if causal, 8.4% slower
// on average, they are up to 2.3x faster, and 3-7% slower on 16 of the shapes (15%
// on one between them: H1 S14000 D16 causal).
int choose_kv_splits(const fa_fwd_params *p, bool any_workspace) {
  // Shape-only (no pointer or stride checks): usable before tensors exist.
  if (p == nullptr || p->B <= 0 || p->H <= 0 || p->Sq <= 0 || p->Sk <= 0) return 1;
  if (!is_supported_head_dim(p->D) || !is_valid_dtype(p->dtype) || p->num_programs < 0) return 1;
  Plan plan;
  if (make_plan(p, &plan) != FA_OK || !kKernelMeta[plan.kernel].splittable) return 1;
  const int64_t tiles = plan.total_tiles, D = p->D;
  if (tiles > kDefaultCuCount) return 1;
  const int64_t kv_tiles = ((int64_t)p->Sk + plan.BN - 1) / plan.BN;
  const int64_t keys = p->causal && p->Sq < p->Sk ? p->Sq : p->Sk;  // of the longest m-tile
  const double key_us = (D == 16 ? 6.5 : D == 32 ? 7.5 : D == 64 ? 9.3 : D == 128 ? 11.7 : 23.0) / 1024;
  const double unit_us = 0.030 * (p->causal ? 0.6 : 1.0) * D / 128;
  // A program count below the tiles makes each program walk several units anyway.
  const int64_t programs = p->num_programs > 0 && p->num_programs < tiles ? p->num_programs : 0;
  auto rounds = [&](int64_t units) { return programs > 0 ? (double)((units + programs - 1) / programs) : 1.0; };
  double best = 0.0;
  int splits = 1;
  for (int s = 2; s <= kMaxKvSplits && p->Sk / s >= 128; ++s) {
    const int64_t run_tiles = (kv_tiles + s - 1) / s, units = tiles * s;
    if ((kv_tiles + run_tiles - 1) / run_tiles < s) continue;  // empty runs at the end
    const int64_t run = run_tiles * plan.BN < keys ? run_tiles * plan.BN : keys;
    int64_t fill = kDefaultCuCount;
    if (p->causal && (D <= 128 || run >= 1365)) fill = 288;
    if ((s & (s - 1)) != 0 && s != kDefaultCuCount / tiles && s != fill / tiles) continue;
    int64_t limit = fill;
    if (p->causal && D <= 128 && tiles <= 128 && run >= 1365) limit = 512;
    if (p->causal && s == 2 && run >= 2048 && limit < 384) limit = 384;
    if (units > limit) continue;
    // Callers of fa_fwd_split_static ask fa_default_kv_splits for their count: what
    // its buffer cannot hold is theirs only where runs keep 64K key-columns.
    if (!any_workspace && (tiles > 128 || s * (int64_t)65536 > p->Sk * D)) {
      const int64_t bytes = split_workspace_bytes(p, s);
      if (bytes < 0 || bytes > (int64_t)FA_STATIC_SCRATCH_BYTES) continue;
    }
    double split_us = run * key_us * rounds(units) + 4.5 + 0.2 * s + unit_us * (double)units;
    if (split_us < 14.5 - 5.0) split_us = 14.5 - 5.0;
    const double gain = keys * key_us * rounds(tiles) - split_us;
    if (gain > best) {
      best = gain;
      splits = s;
    }
  }
  return splits;
}

}  // namespace

#ifndef FA_SOURCE_HASH
#define FA_SOURCE_HASH "unknown"
#endif

extern "C" {

int fa_abi_version(void) { return FA_ABI_VERSION; }

const char *fa_build_id(void) { return FA_SOURCE_HASH; }

const char *fa_error_string(int code) {
  switch (code) {
    case FA_OK: return "ok";
    case FA_ERR_NULL: return "a required tensor pointer is NULL";
    case FA_ERR_SHAPE: return "invalid shape (negative size, Sq>0 with Sk==0, or too many tiles)";
    case FA_ERR_HEAD_DIM: return "HEAD_DIM is not one of 16, 32, 64, 128, 256";
    case FA_ERR_DTYPE: return "dtype must be fp16 or bf16 (optionally with fp8-e5m2 V)";
    case FA_ERR_STRIDE: return "the head-dim stride must be 1 and the other strides multiples of 8 elements (16 for an fp8 V)";
    case FA_ERR_ALIGN: return "tensor base pointers must be 16-byte aligned";
    case FA_ERR_TILING: return "unsupported BLOCK_M/BLOCK_N combination";
    case FA_ERR_SCALE: return "sm_scale must be finite";
    case FA_ERR_GRID: return "the persistent program count must be >= 0";
    case FA_ERR_SCRATCH: return "the split-KV partial results exceed the library's static scratch buffer (FA_STATIC_SCRATCH_BYTES)";
    case FA_ERR_LAUNCH: return "the HIP runtime rejected the kernel launch";
    default: return "unknown fa_fwd status";
  }
}

int fa_validate(const fa_fwd_params *p) {
  if (p == nullptr) return FA_ERR_NULL;
  if (p->B < 0 || p->H < 0 || p->Sq < 0 || p->Sk < 0 || p->D <= 0) return FA_ERR_SHAPE;
  if (p->Sq > 0 && p->Sk == 0 && p->B > 0 && p->H > 0) return FA_ERR_SHAPE;
  if (!is_supported_head_dim(p->D)) return FA_ERR_HEAD_DIM;
  if (!is_valid_dtype(p->dtype)) return FA_ERR_DTYPE;
  if (v_is_fp8(p->dtype) && !is_supported_fp8v_head_dim(p->D)) return FA_ERR_HEAD_DIM;
  if (!(p->sm_scale == p->sm_scale) || isinf(p->sm_scale)) return FA_ERR_SCALE;
  if (p->num_programs < 0) return FA_ERR_GRID;
  if ((p->block_m == 0) != (p->block_n == 0)) return FA_ERR_TILING;
  const bool empty = p->B == 0 || p->H == 0 || p->Sq == 0;
  if (empty) return FA_OK;
  if (p->q == nullptr || p->k == nullptr || p->v == nullptr || p->o == nullptr) return FA_ERR_NULL;
  const int64_t *st[4] = {p->q_stride, p->k_stride, p->v_stride, p->o_stride};
  const int64_t rows[4] = {p->Sq, p->Sk, p->Sk, p->Sq};
  for (int t = 0; t < 4; ++t) {
    // 16-byte rows: strides in multiples of 8 16-bit or 16 fp8 elements.
    const int64_t align = (t == 2 && v_is_fp8(p->dtype)) ? 16 : 8;
    if (st[t][3] != 1) return FA_ERR_STRIDE;
    for (int i = 0; i < 3; ++i)
      if (st[t][i] < 0 || st[t][i] % align != 0) return FA_ERR_STRIDE;
    if (rows[t] > 1 && st[t][2] < p->D) return FA_ERR_STRIDE;
    // Buffer offsets inside one (b, h) slice are 32-bit: keep the slice, plus
    // the rows past its end that a last partial m-tile or the DMAs issued past
    // the last KV tile address, below 2 GiB.  rows < 2^31 and row_stride <
    // 2^31 here, so the product is formed in 128-bit arithmetic (it can
    // exceed int64: e.g. 2^31 rows of a 2^31 - 8 element stride).
    const int64_t row_stride = st[t][2] > p->D ? st[t][2] : p->D;
    if (row_stride >= ((int64_t)1 << 31)) return FA_ERR_SHAPE;
    if ((__int128)(rows[t] + kRowMargin) * row_stride * 2 >= ((__int128)1 << 31)) return FA_ERR_SHAPE;
  }
  if ((int64_t)p->Sq * 4 >= ((int64_t)1 << 31)) return FA_ERR_SHAPE;
  if (!aligned16(p->q) || !aligned16(p->k) || !aligned16(p->v) || !aligned16(p->o)) return FA_ERR_ALIGN;
  if (p->lse != nullptr && ((uintptr_t)p->lse & 3u) != 0) return FA_ERR_ALIGN;
  Plan plan;
  return make_plan(p, &plan);
}

int fa_query_config(const fa_fwd_params *p, int32_t out[FA_CFG_COUNT]) {
  if (p == nullptr || out == nullptr) return FA_ERR_NULL;
  if (p->B < 0 || p->H < 0 || p->Sq < 0 || p->Sk < 0) return FA_ERR_SHAPE;
  if (!is_supported_head_dim(p->D)) return FA_ERR_HEAD_DIM;
  if (!is_valid_dtype(p->dtype)) return FA_ERR_DTYPE;
  if (v_is_fp8(p->dtype) && !is_supported_fp8v_head_dim(p->D)) return FA_ERR_HEAD_DIM;
  if ((p->block_m == 0) != (p->block_n == 0)) return FA_ERR_TILING;
  if (p->num_programs < 0) return FA_ERR_GRID;
  Plan plan;
  const int rc = make_plan(p, &plan);
  if (rc != FA_OK) return rc;
  out[FA_CFG_BLOCK_M] = plan.BM;
  out[FA_CFG_BLOCK_N] = plan.BN;
  out[FA_CFG_WAVES] = plan.NW;
  out[FA_CFG_GRID] = plan.grid;
  out[FA_CFG_TOTAL_TILES] = (int32_t)plan.total_tiles;
  out[FA_CFG_LDS_BYTES] = kernel_lds_bytes(kKernelMeta[plan.kernel]);
  out[FA_CFG_STAGE] = p->causal ? 3 : 1;
  out[FA_CFG_KERNEL_ID] = plan.kernel;
  return FA_OK;
}

int fa_num_kernels(void) { return kNumKernels; }

int fa_params_size(void) { return (int)sizeof(fa_fwd_params); }

int fa_kernel_info(int index, int32_t out[6]) {
  if (out == nullptr) return FA_ERR_NULL;
  if (index < 0 || index >= kNumKernels) return FA_ERR_TILING;
  const KernelMeta &e = kKernelMeta[index];
  out[0] = e.D;
  out[1] = e.dtype;
  out[2] = e.causal;
  out[3] = 32 * e.NW;
  out[4] = e.BN;
  out[5] = e.NW;
  return FA_OK;
}

int fa_kernel_wg_per_cu(int index) {
  if (index < 0 || index >= kNumKernels) return FA_ERR_TILING;
  return kKernelMeta[index].wg_per_cu;
}

int64_t fa_split_workspace_bytes(const fa_fwd_params *p, int32_t kv_splits) {
  if (p == nullptr) return FA_ERR_NULL;
  if (kv_splits < 1 || kv_splits > kMaxKvSplits) return FA_ERR_GRID;
  if (p->B < 0 || p->H < 0 || p->Sq < 0 || p->D <= 0) return FA_ERR_SHAPE;
  if (kv_splits == 1) return 0;
  const int64_t bytes = split_workspace_bytes(p, kv_splits);
  return bytes >= 0 ? bytes : (int64_t)FA_ERR_SHAPE;
}

int32_t fa_default_kv_splits(const fa_fwd_params *p) { return choose_kv_splits(p, false); }

int32_t fa_workspace_kv_splits(const fa_fwd_params *p) { return choose_kv_splits(p, true); }

}  // extern "C"
