// C ABI of the gfx950 grouped quantized matmul backend (see include/msco_gmm.h).
// Host side only: argument checking, kernel-family choice from shapes (never from tensor values),
// workspace sizing and the launches.
#include "msco_gmm.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <string>

#include "gmm_kernels.h"
#include "gmm_tile_times.h"

namespace {

using namespace msco;

enum Family : int { FAM_NONE = 0, FAM_TILE = 1, FAM_SKINNY = 2, FAM_GENERIC = 3, FAM_REGT = 4, FAM_ROWS16 = 5 };

// values of msco_gmm_desc::kernel_override
enum Override : int {
  OV_AUTO = 0, OV_TILE_256 = 1, OV_TILE_128 = 2, OV_TILE_64 = 3, OV_SKINNY = 4, OV_GENERIC = 5,
  OV_TILE_256_W4 = 6,  // persistent four-wave 256 x 256 kernel
  OV_TILE_128x256 = 7,  // four waves side by side, 128 x 256
  OV_TILE_256_W4_MFMA32 = 8,  // the persistent kernel's 32 x 32 x 32 form (never planned)
  OV_ROWS128 = 9,  // packed weights: chunks of up to 128 rows through LDS, weights straight into MFMA operands (other layouts: 128 x 256 tiles)
  OV_ROWS256 = 10,  // the same with chunks of up to 256 rows (other layouts: the persistent kernel)
  OV_ROWS160 = 11,  // ... of up to 160 rows (other layouts: the persistent kernel)
  OV_REGT = 12,     // [E,K,N] weights transposed and converted in registers (other layouts: as planned)
  OV_TILE_4BIT = 13,  // 4-bit weights, int8 x: 64 x 256 or 128 x 256 tiles that read the nibbles (else: as planned)
  OV_ROWS16 = 14,     // weight-only: equal chunks of up to 128 rows x strips of 512 columns (else: as planned)
  OV_ROWS16_256 = 15,  // the same with strips of 256 columns
  OV_ROWS16_256X2 = 16, // ... and two sets of waves that take turns at the K blocks
  OV_TILE_32x128 = 17,  // a few rows on [E,K,N] and [E,N,K] weights (packed: 64 x 128 tiles)
  OV_TILE_32x256 = 18,  // ... on [E,K,N] weights ([E,N,K]: as 17)
  OV_W4_128 = 19, OV_W4_160 = 20, OV_W4_192 = 21, OV_W4_224 = 22, OV_W4_288 = 23,  // the persistent kernel with tiles of that many rows
  OV_W4_128x192 = 24, OV_W4_160x192 = 25
};

constexpr int64_t kSkinnyMaxRows = 64;   // total rows up to which the weight-streaming kernel is planned
constexpr int64_t kSkinnyMaxChunkSlots = 1024;   // (group, 16-row chunk) slots up to which many small groups take the decode kernels
constexpr int kTargetWorkgroups = 512;  // skinny kernels with a K split: aim for this many workgroups (2 per CU)
constexpr int kMaxSplitK = 8;             // keeps the last arriver's reduction to two rounds of loads
constexpr int kDefaultCUs = 256;   // MI355X; the plan uses the count the device reports
constexpr int kTileTargetWorkgroups = 256;   // tile kernels with a K split: aim for this many workgroups (one per CU)
constexpr int kTileSplitMaxTiles = 128;      // ... and only split below this many tiles (measured: beyond it the partial-tile exchange costs more than it hides)
constexpr size_t kTileSplitMaxWorkspace = (size_t)128 << 20;   // bytes of split-K partial tiles a plan may ask the caller for
constexpr int kTileMinSlabs = 4;               // 64-byte K slabs every slice keeps at least

int env_int(const char *name, int fallback) {
  const char *v = std::getenv(name);
  return (v && *v) ? std::atoi(v) : fallback;
}

// MSCO_PRINT_PLAN (the counterpart of the reference's INTERNAL_PRINT_TILING) is read from the environment once per
// process, at the first plan; planning itself reads no environment.  The other fields override plan constants for
// tuning sweeps and exist only in a library built with -DMSCO_TUNING_SWITCHES (build.py --tuning): the shipped
// library has no such switches.
struct Tuning {
  int print_plan, tile_cfg, tile_target_wgs, tile_split_k, stream_max_slots, skinny_wide16, stream_min_wgs, stream_groups,
      skinny_target_wgs, skinny_split_k, tile_wide_k, stream_tch, two_level, regt_cols;
};
const Tuning &tuning() {
#ifdef MSCO_TUNING_SWITCHES
  static thread_local Tuning t;   // read again at every plan: a sweep changes them between plans
  t = Tuning{env_int("MSCO_PRINT_PLAN", 0),        env_int("MSCO_TILE_CFG", -1),
                           env_int("MSCO_TILE_TARGET_WGS", 0),   env_int("MSCO_TILE_SPLIT_K", 0),
                           env_int("MSCO_STREAM_MAX_SLOTS", 0),  env_int("MSCO_SKINNY_WIDE16", -1),
                           env_int("MSCO_STREAM_MIN_WGS", 0),    env_int("MSCO_STREAM_GROUPS", 0),
                           env_int("MSCO_SKINNY_TARGET_WGS", 0), env_int("MSCO_SKINNY_SPLIT_K", 0),
                           env_int("MSCO_TILE_WIDE_K", -1),      env_int("MSCO_STREAM_TCH", 0),
                           env_int("MSCO_TWO_LEVEL", 1),         env_int("MSCO_REGT_COLS", 0)};
#else
  static const Tuning t = {env_int("MSCO_PRINT_PLAN", 0), -1, 0, 0, 0, -1, 0, 0, 0, 0, -1, 0, 1, 0};
#endif
  return t;
}
int or_default(int v, int fallback) { return v > 0 ? v : fallback; }

}  // namespace

struct msco_gmm_op {
  msco_gmm_desc desc{};
  bool planned = false;
  int64_t m = 0, k = 0, n = 0, e = 0;
  int family = FAM_NONE;
  int tile_cfg = 0;
  int tile_shape = 0;        // persistent tile kernel: index into kT4mShape, negative: picked on the device from the groups
  int split_k = 1;
  int skinny_wide16 = 0;
  int skinny_cols = kSkinnyCols;
  int n_strips = 0;
  int strip_groups = 16;
  int stream_tch = 1;        // packed and, weight-only, [E,K,N] weights: 16-row fragments per chunk (1: the 16-row streaming kernels, 2/4/8: the multi-row ones)
  int wide_k_slabs = 0;      // small tile kernels on K-major weights: 128-byte K slabs
  int w_nontemporal = 0;     // small tile kernels on packed weights: non-temporal weight loads
  int small_group_rows = 0;  // > 0: the persistent kernel takes the groups with more rows, a second launch of 64 x 128 tiles the others
  int row_blocks = 1;        // register-transpose kernels: 16-row blocks per chunk
  int strip_cols = 256;      // ... and columns per strip (also of the weight-only 128-row kernel)
  int wave_sets = 1;         // weight-only 128-row kernel: sets of waves that take turns at the K blocks
  bool shallow = false;      // ... and the form with one K step in flight per wave (several workgroups per CU)
  int64_t widen_bytes = 0;   // 4-bit weights without a kernel of their own for the shape: int8 copy of them at the front of the workspace
  size_t workspace_bytes = 0;
  unsigned *counters = nullptr;
  size_t counters_cap = 0, counters_used = 0;   // allocated; of the present plan
  bool counters_recorded = false;               // a recorded graph counts with `counters`: they are never freed
  unsigned *recorded = nullptr;                 // counters of the launches that capture `recorded_id` records
  size_t recorded_cap = 0;
  unsigned long long recorded_id = 0;
  int num_cus = kDefaultCUs;   // compute units of the device that was current at create time
  std::string info;
  std::mutex mu;
};

namespace {

bool is_w8a8(const msco_gmm_desc &d) { return d.x_dtype == MSCO_DT_I8; }
bool is_a16w8(const msco_gmm_desc &d) { return d.x_dtype == MSCO_DT_BF16 || d.x_dtype == MSCO_DT_F16; }
bool is_w4(const msco_gmm_desc &d) { return d.weight_dtype == MSCO_DT_I4; }
bool is_packed(const msco_gmm_desc &d) { return d.weight_layout == MSCO_WL_PACKED; }
// 0 [E,K,N], 1 [E,N,K], 2 packed
int layout_of(const msco_gmm_desc &d) { return is_packed(d) ? 2 : (d.transpose_b ? 1 : 0); }

int check_desc(const msco_gmm_desc &d) {
  if (d.abi_version != MSCO_GMM_ABI_VERSION) return MSCO_ERR_INVALID_ARG;
  if (d.weight_dtype != MSCO_DT_I8 && d.weight_dtype != MSCO_DT_I4) return MSCO_ERR_UNSUPPORTED;
  if (d.weight_dtype == MSCO_DT_I4 && (d.weight_layout != MSCO_WL_ROW_MAJOR || d.transpose_b != 0)) return MSCO_ERR_UNSUPPORTED;
  if (d.group_list_dtype != MSCO_DT_NONE && d.group_list_dtype != MSCO_DT_I32 && d.group_list_dtype != MSCO_DT_I64)
    return MSCO_ERR_UNSUPPORTED;
  if (d.group_list_type != 0 && d.group_list_type != 1) return MSCO_ERR_INVALID_ARG;
  if (d.kernel_override < OV_AUTO || d.kernel_override > OV_W4_160x192) return MSCO_ERR_INVALID_ARG;
  if (d.weight_layout != MSCO_WL_ROW_MAJOR && d.weight_layout != MSCO_WL_PACKED) return MSCO_ERR_INVALID_ARG;
  if (d.force_split_k < 0) return MSCO_ERR_INVALID_ARG;
  if (d.act_type < MSCO_ACT_NONE || d.act_type > MSCO_ACT_SILU) return MSCO_ERR_INVALID_ARG;
  if (d.act_type == MSCO_ACT_GELU_ERF) return MSCO_ERR_UNSUPPORTED;
  if (d.act_type != MSCO_ACT_NONE && d.out_dtype == MSCO_DT_I32) return MSCO_ERR_UNSUPPORTED;
  if (is_w8a8(d)) {
    if (d.out_dtype != MSCO_DT_BF16 && d.out_dtype != MSCO_DT_F16 && d.out_dtype != MSCO_DT_I32)
      return MSCO_ERR_UNSUPPORTED;
    if (d.bias_dtype != MSCO_DT_NONE && d.bias_dtype != MSCO_DT_I32) return MSCO_ERR_UNSUPPORTED;
    if (d.scale_dtype != MSCO_DT_NONE && d.scale_dtype != MSCO_DT_F32 && d.scale_dtype != MSCO_DT_BF16 &&
        d.scale_dtype != MSCO_DT_I64 && d.scale_dtype != MSCO_DT_U64)
      return MSCO_ERR_UNSUPPORTED;
    if (d.per_token_dtype != MSCO_DT_NONE && d.per_token_dtype != MSCO_DT_F32) return MSCO_ERR_UNSUPPORTED;
    if (d.antiquant_dtype != MSCO_DT_NONE) return MSCO_ERR_UNSUPPORTED;
    return MSCO_OK;
  }
  if (is_a16w8(d)) {
    if (d.out_dtype != d.x_dtype) return MSCO_ERR_UNSUPPORTED;       // weight-only output keeps x's dtype
    if (d.antiquant_dtype != d.x_dtype) return MSCO_ERR_UNSUPPORTED; // scale / offset share x's dtype
    if (d.transpose_b && d.weight_layout == MSCO_WL_ROW_MAJOR) return MSCO_ERR_UNSUPPORTED;
    if (d.bias_dtype != MSCO_DT_NONE || d.scale_dtype != MSCO_DT_NONE || d.per_token_dtype != MSCO_DT_NONE)
      return MSCO_ERR_UNSUPPORTED;
    return MSCO_OK;
  }
  return MSCO_ERR_UNSUPPORTED;
}

// Groups that hold rows when m rows go to e groups at random: the mean and one standard deviation, at most min(m, e).
int64_t groups_hit(int64_t m, int64_t e) {
  if (m < 1 || e < 2) return 1;
  const double ed = (double)e, q = std::pow(1.0 - 1.0 / ed, (double)m), r = std::pow(1.0 - 2.0 / ed, (double)m);
  const double var = ed * (ed - 1.0) * r + ed * q - ed * ed * q * q;
  return std::max<int64_t>(1, std::min<int64_t>(std::min(m, e), (int64_t)std::ceil(ed * (1.0 - q) + std::sqrt(std::max(var, 0.0)))));
}

// Mean number of bm-row tiles of a group that holds `avg` rows on average: a random routing scatters them by about the root of that.
double expected_row_tiles(double avg, double bm) {
  const double sd = std::sqrt(std::max(avg, 1e-9));
  const double sure = std::max(0.0, std::floor((avg - 5.0 * sd) / bm));
  double tiles = sure;
  for (double rows = sure * bm + 0.5; rows < avg + 5.0 * sd; rows += bm) tiles += 0.5 * std::erfc((rows - avg) / (sd * std::sqrt(2.0)));
  return std::max(tiles, 1e-3);
}

// 4-bit weights, 16-bit x, several groups of more than 30 rows whose 128-row chunks on strips of 256 columns are at most a quarter of the chip: the
// register-transpose kernels, whose 32-row chunks are four times as many workgroups, take less than the 128-row kernel with its K
// splits.  They convert the weights once per 32 rows in place of 128, which costs more than that with a long K.  642 random
// shapes of 31 to 1000 rows per group, even and skewed, 0.66 of the time, 1.01 at worst (us: 16 experts, 58 rows, 1440 x 576 23.8 -> 16.5; 8 experts,
// 110 rows, 1856 x 784 28.0 -> 18.2; 8 experts, 2000 rows, 1120 x 240 22.1 -> 14.5; the chunks and strips that plan_regt counts for them are part of
// it: 0.72 and 1.32 without).  Beyond, without those: up to three eighths of the chip 0.85 and 1.25, K of 3072 to 4096 0.88 and 1.19.  The error against
// float64 is the same to six digits.
bool few_4bit_chunks(const msco_gmm_op *op) {
  const int64_t m = op->m, e = op->e, cus = op->num_cus > 0 ? op->num_cus : kDefaultCUs, avg = (m + e - 1) / e, rows = avg + avg / 10;
  return is_w4(op->desc) && is_a16w8(op->desc) && e >= 8 && op->k >= 512 && op->k <= 3072 && (op->n + 255) / 256 * std::min(e, m) * ((rows + 127) / 128) * 4 <= cus;
}

// Row-major [E,K,N] weights transposed and converted in registers (gmm_regt.hip).  Called behind choose_plan's own pick:
// takes the plan over where these kernels are the better ones, and sets up the widening where 4-bit weights go to a
// kernel that reads int8.
void plan_regt(msco_gmm_op *op) {
  const msco_gmm_desc &d = op->desc;
  const int64_t m = op->m, k = op->k, n = op->n, e = op->e;
  const int bits = is_w4(d) ? 4 : 8;
  // rows a group is expected to hold (shapes only); real routings are uneven, hence 1.5 x the average
  const int64_t avg = (m + e - 1) / e, rows = e == 1 ? m : avg + avg / 2;
  const int blocks = bits == 8 || rows <= 16 ? 1 : 2;
  // int8 x on 4-bit weights: int32 sums of 16 times the products, K x 2^14 < 2^31.  16-bit x is summed in float32, whatever K.
  // A chunk's x rows and a group's weights are addressed through 32-bit offsets.
  const bool sums_fit = !(is_w8a8(d) && bits == 4) || k < ((int64_t)1 << 17);
  const bool can = layout_of(d) == 0 && k % 16 == 0 && n % 16 == 0 && sums_fit && k * n * bits / 8 < ((int64_t)1 << 31) &&
                   m * k < ((int64_t)1 << 31) && std::min<int64_t>(m, 16 * blocks) * k * (is_w8a8(d) ? 1 : 2) < ((int64_t)1 << 31);
  // 4-bit weights with 16-bit x: widening them first (8 experts, K = 4096, N = 14336: 120 us for the widening alone) costs
  // more than a second and third pass over the nibbles (4 / 32 rows per group: 47 / 95 us in all).
  // Weight-only on 8-bit weights, one 16-row chunk per group: the decode form.
  const bool want = d.kernel_override == OV_REGT ||
                    (d.kernel_override == OV_AUTO && bits == 4 && (rows <= 64 || few_4bit_chunks(op)) && op->family != FAM_ROWS16) ||
                    (op->family == FAM_SKINNY && bits == 8 && is_a16w8(d) && op->stream_tch == 1);
  // 4-bit weights, int8 x, more than one 16-row chunk per group: tiles that read the nibbles through LDS (4 / 16 / 32 rows
  // per group 52 / 53 / 58 us against 44 / 53 / 82 us in 32-row chunks)
  // ... up to some two thousand rows per group, where the persistent kernel, a sixth to an eighth faster, makes up for widening
  // the weights first (3 us and 1 us per 3.9 M weights) by the time that is 11.6 % of the products (2.2 Pop/s).  4-bit tiles
  // against widening, us: 8 experts, K = 4096, N = 14336, 2048 / 3072 / 4096 rows per group 920 / 1367 / 1800 against 937 / 1321 / 1712;
  // one group, N = 11008, 2048 / 3072 / 16384 rows 101 / 152 / 674 against 101 / 144 / 590; K = N = 4096, 4096 / 8192 rows 66 / 126 against
  // 67 / 114; 16 experts, 2048 x 2816, 1792 / 4096 rows 194 / 407 against 204 / 388.  The line is not sharp: 128 experts, 2048 x 768,
  // 2048 rows (14.6 %) 502 against 475, 32 experts, 4096 x 1024, 2048 rows (14.9 %) 297 against 310.
  const bool widen_pays = d.kernel_override == OV_AUTO && op->family == FAM_TILE && op->tile_cfg == TILE_256x256_W4 &&
                          3.0 + (double)(e * k * n) / 3.9e6 <= 0.116 * 2.0 * (double)(m * k) * (double)n / 2.2e9;
  if (can && bits == 4 && is_w8a8(d) && (d.kernel_override == OV_TILE_4BIT || (d.kernel_override == OV_AUTO && rows > 16 && !widen_pays))) {
    const int64_t cus = op->num_cus > 0 ? op->num_cus : kDefaultCUs, groups = std::max<int64_t>(1, std::min<int64_t>(e, m)), n_tiles = (n + 255) / 256;
    // 128-row tiles once 64 rows no longer hold a group and there are tiles for most CUs (64 / 128 rows per group 83 / 114 us
    // with 64-row tiles, 68 / 106 us with 128; one group of 256 rows, N = 11008: 31.7 against 42.7 us)
    const bool tall = rows > 64 && std::max<int64_t>((m + 127) / 128, groups) * n_tiles * 4 >= cus * 3;
    op->family = FAM_TILE;
    op->tile_cfg = tall ? TILE_128x256_W4B : TILE_64x256_W4B;
    if (tuning().tile_cfg >= TILE_64x256_W4B) op->tile_cfg = tuning().tile_cfg;
    op->wide_k_slabs = 0;
    op->small_group_rows = 0;
    const int bm = op->tile_cfg == TILE_128x256_W4B ? 128 : 64;
    op->w_nontemporal = (rows + bm - 1) / bm <= 2 && e * k * n / 2 >= ((int64_t)32 << 20);   // (as for int8 weights)
    // K split of the 64-row tiles up to one workgroup per CU, by the cost in 64-byte K slabs: a slice's slabs, 10 for the
    // workgroup's ends and 5 per slice of the exchange (one group, 32 rows, N = 11008, split 2 / 4 / 5: 21.6 / 18.7 / 19.0 us; 8 x
    // 38 rows, N = 1024, split 2 / 4 / 8: 21.4 / 18.0 / 20.9 us)
    const int64_t tiles = std::max<int64_t>((m + bm - 1) / bm, groups) * n_tiles, slabs = (k + 63) / 64;
    const int64_t most = bm == 64 ? std::min<int64_t>({cus / tiles, kMaxSplitK, std::max<int64_t>(1, slabs / kTileMinSlabs)}) : 1;
    auto cost = [&](int64_t s) { return (slabs + s - 1) / s + (s > 1 ? 5 * s : 0); };
    int64_t split = 1;
    for (int64_t s = 2; s <= most; ++s)
      if (cost(s) < cost(split)) split = s;
    if (d.force_split_k > 0 && bm == 64) split = std::min<int64_t>(d.force_split_k, slabs);
    while (split > 1 && tile_workspace_bytes(op->tile_cfg, m, n, e, (int)split) > kTileSplitMaxWorkspace) --split;
    op->split_k = (int)split;
    op->workspace_bytes = tile_workspace_bytes(op->tile_cfg, m, n, e, op->split_k);
    return;
  }
  if (can && want) {
    GmmParams p{};
    p.m = (int)m;
    p.e = (int)e;
    const int64_t slots = chunk_slots(p, 16 * blocks);
    // 16-bit x on 8-bit weights: a form with one K step in flight per wave and four waves per SIMD, for several workgroups per CU
    const bool can_be_shallow = bits == 8 && is_a16w8(d);
    // Chunks expected to hold rows (an average group's, not one per group: 8 experts, 40 rows each, K = N = 4096, 4-bit weights: a K
    // split for 16 chunks instead of 8 and 45.3 -> 37.0 us).  Few rows over many groups: the groups that a random routing hits where
    // the forms below are chosen by how full the chip is (32 experts, 52 rows, K = 6976, N = 1920, not full: 70.9 -> 65.2 us), as
    // many as there can be elsewhere (the other estimate there: 110 shapes at 0.98 to 1.13 of the time, 1.003 on average).
    // Groups of more than 30 rows (few_4bit_chunks): those that a random routing makes, most groups ending in a chunk of their own.  A chip that an
    // average group's would just fill, with or without a K split, takes a second round for the others (us; 128-row kernel, an average group's, these: 32
    // experts, 54 rows, 3024 x 400 30.2 / 37.4 / 29.5; 32 experts, 174 rows, 560 x 208 15.3 / 17.0 / 12.5).
    const bool few = d.kernel_override == OV_AUTO && m > 30 * e && few_4bit_chunks(op);
    const int64_t active = few ? std::min<int64_t>(slots, (int64_t)std::ceil((double)std::min(m, e) * expected_row_tiles((double)m / (double)std::min(m, e), 16.0 * blocks))) :
      std::max<int64_t>(1, std::min<int64_t>(slots, (can_be_shallow ? groups_hit(m, e) : std::min<int64_t>(m, e)) * ((avg + 16 * blocks - 1) / (16 * blocks))));
    const int64_t cus = op->num_cus > 0 ? op->num_cus : kDefaultCUs;
    // Strips of 512 columns (eight waves, twice as many neighbouring bytes per K row) while they fill most of the CUs
    // without a K split, strips of 256 (four waves) otherwise.  8 experts, K = 4096, N = 14336, 4 rows per group, 4-bit
    // weights: 44 against 51 us (int8 x), 47 against 52 us (bf16).  One group, N = 11008: 20 against 17 us.
    const int64_t wgs512 = ((n + 511) / 512) * active, wgs256 = ((n + 255) / 256) * active;
    // (not for those groups, of which only up to 256 columns would give so many: 64 experts, 116 rows, 1504 x 112 42.3 us with half of the waves
    // without columns, 26.7 with strips of 256)
    int64_t cols = wgs512 * 4 >= cus * 3 && !few ? 512 : 256;
    // 8-bit weights: 512 columns take 0.9 of the time of two strips of 256, but their rounds on the chip are coarser: up to two they are
    // counted whole, the chip full with 31/32 of the CUs (256 columns: with 34/32, four of them fit a CU and fewer groups may be hit); beyond,
    // a half for the last one.  Strips of 512 / 256, us, the weights not in the caches: 48 rows over 32 experts, K = 2624, N = 4624 (more than one round): 96.6 / 72.4; 320 over 32, K = 832, N = 4688: 38.8 / 36.4; 288
    // over 64, K = 1088, N = 4064 (all of two rounds): 73 / 63; 1296 over 128, K = 1248, N = 704 (all of one): 46 / 31; one round: 28 over 8,
    // K = 2944, N = 13840: 65.9 / 73.5; 24 over 32, K = 3168, N = 4016 (152 workgroups): 57 / 66; many: 198 over 64, K = 704, N = 7824: 71.7 / 80.2.
    // Fitted to 620 shapes of 1 to 10 rows per group, K = 512 .. 8192, N = 512 .. 14336, random routings.
    if (can_be_shallow) {
      auto tenths = [&](int64_t w, int64_t full) { return w <= 2 * cus ? 10 * ((32 * w + full * cus - 1) / (full * cus)) : 10 * w / cus + 5; };
      cols = wgs512 * 20 >= cus * 11 && 9 * tenths(wgs512, 31) < 5 * tenths(wgs256, 34) ? 512 : 256;
    }
    if (tuning().regt_cols > 0) cols = tuning().regt_cols;
    const int64_t strips = (n + cols - 1) / cols;
    if (slots <= 65535) {
      op->family = FAM_REGT;
      op->row_blocks = blocks;
      op->strip_cols = (int)cols;
      op->n_strips = (int)strips;
      // K split across workgroups up to one of them per CU: of the splits that leave the fewest K steps to a wave (four
      // waves share them, in rounds of four or two), the smallest.  K = 4096, N = 11008, one row, 8-bit weights, split
      // 1 / 2 / 3 / 4 / 6 / 8: 27 / 20 / 17.4 / 17.0 / 19.6 / 19.9 us -- beyond one workgroup per CU the slower half of a
      // CU's pair and the exchange of partial tiles cost more than the shorter walk saves.
      const int64_t steps = is_w8a8(d) ? (k + 63) / 64 : (k + 31) / 32, round = is_w8a8(d) ? 2 : 4;
      auto per_wave = [&](int64_t s) { return ((((steps + s - 1) / s + 3) / 4 + round - 1) / round) * round; };
      const int64_t most = std::min<int64_t>({std::max<int64_t>(1, cus / std::max<int64_t>(strips * active, 1)), kMaxSplitK, steps});
      int64_t split = 1;
      for (int64_t s = 2; s <= most; ++s)
        if (per_wave(s) + 1 < per_wave(split)) split = s;
      // A chip that is a little more than half full: two slices would start a second round, three make the shallow form's rounds
      // (16 experts, K = 7872, N = 2192, 30 rows: 72.6 -> 65.2 us; K = 6368, 40 rows: 60.9 -> 56.8; 8 experts, K = 2720, N = 5120, 10 rows: 26.6 ->
      // 21; K = 2464, N = 4320, 62 rows: 28.9 -> 29.6; three quarters full, 64 experts, K = 2912, N = 768, 278 rows: 28.5 -> 36.3).
      if (can_be_shallow && cols == 256 && split == 1 && k >= 1536 && strips * active * 8 <= cus * 5) split = 3;
      if (d.force_split_k > 0) split = std::min<int64_t>(d.force_split_k, steps);
      const size_t tile = (size_t)slots * strips * regt_slice_bytes(blocks, (int)cols);
      while (split > 1 && tile * split > kTileSplitMaxWorkspace) --split;
      op->split_k = (int)split;
      op->workspace_bytes = op->split_k > 1 ? tile * op->split_k : 0;
      // One K step in flight per wave and twice the waves where CUs get more than one workgroup: strips of 512 columns (8
      // experts, K = 512, N = 14336, 8 rows per group, 224 workgroups: 18.2 -> 15.7 us) and 256 workgroups of 256 (64 experts, K = 4096,
      // N = 1024: 50.9 -> 47.1 us; 8 experts, K = N = 4096, two slices: 31.1 -> 30.2 us); below that three steps (176 workgroups, 8
      // experts, K = 4096, N = 5632: 35.5 against 42.6 us; 224, N = 7168: 43.2 against 44.3 us).
      op->shallow = can_be_shallow && (cols == 512 || strips * active * split >= cus);
      return;
    }
  }
  if (op->family == FAM_SKINNY && layout_of(d) == 0 && is_a16w8(d) && op->stream_tch == 1) {   // (what the kernels above cannot take)
    op->family = FAM_GENERIC;
    op->split_k = 1;
  }
  if (bits == 4 && op->family != FAM_ROWS16) {   // (the 128-row weight-only kernel reads the nibbles)
    op->widen_bytes = (e * k * n + 255) / 256 * 256;
    op->workspace_bytes += (size_t)op->widen_bytes;
  }
}

// Weight-only on packed or [E,K,N] weights beyond one 16-row chunk per group: the forms of the 128-row kernel
// (gmm_rows_a16w8_kernel.h) -- strips of 512 columns, strips of 256 with two workgroups per CU, strips of 256 whose K blocks two
// sets of waves share, the last two with a K split -- against the 32- and 64-row kernels, by a model of the time in us.  All
// of them take as long as their rounds on the chip are many; a round has ends of its own and a part per K block, larger with more
// rows, and the weights and rows have to be read.  Fitted to 460 random shapes (8 to 128 experts, 10 to 3200 rows per group,
// K = 512 .. 8192, N = 512 .. 14336, random routings), every form measured on all of them: off by 8 .. 10 % (rms), and what it picks takes
// 1.03 of the time of the best form and 0.83 of what the rules before it picked.  us, before -> now: 8 experts, K = 5056,
// N = 3984, 145 rows per group, [E,K,N] 136 -> 71 (two sets; strips of 512: 107, of 256: 81); K = 6176, N = 688, 2485 rows, packed 318 -> 185
// (256; 512: 271); 16 experts, K = 6336, N = 544, 51 rows 78 -> 38 (two sets, two slices; one set, one slice: 63); 64 experts, K = 928,
// N = 2000, 282 rows, [E,K,N] 150 -> 104; 8 experts, K = 4096, N = 14336, 512 rows stays with 512: 437 (256: 445).
struct Rows16Form { int cols, sets, split; };
// fixed, per round, per K block and round, the same per 16 rows, per us of reading; K split: fixed, per slice, 16 rows and round
struct Rows16Cost { double fixed, round, block, rows, stream, split, slice; };
constexpr Rows16Cost kRows16[2][4] = {   // [packed][strips of 512; of 256 alone on their CUs; of 256 two per CU; two sets]
  {{2.6, 8.15, 0.632, 0.075, 0.54, 0, 0}, {8.75, 0, 0.337, 0.063, 0.67, 4.0, 0.74}, {8.75, 1.57, 0.533, 0.100, 0.67, 4.0, 0.74}, {4.73, 6.91, 0.428, 0.103, 0.75, 4.2, 0.20}},
  {{2.4, 5.81, 0.357, 0.095, 0.68, 0, 0}, {7.05, 0, 0.181, 0.068, 0.74, 3.1, 0.74}, {7.05, 1.47, 0.320, 0.101, 0.74, 3.1, 0.74}, {3.11, 6.09, 0.182, 0.123, 0.77, 3.8, 0.22}}};
constexpr Rows16Cost kRowsSmall[2][2] = {   // [packed][32- and 64-row chunks], strips of 256 columns
  {{6.2, 0, 0.665, 0.079, 0.84, 0, 0}, {7.8, 0, 0.803, 0.071, 0.84, 0, 0}}, {{5.9, 0, 0.860, 0.034, 0.50, 0, 0}, {5.8, 0, 0.747, 0.173, 0.50, 0, 0}}};

double chip_rounds(double workgroups, double slots) { return workgroups <= slots ? 1.0 : workgroups / slots + 0.5; }

double rows_stream_us(int64_t m, int64_t k, int64_t n, int64_t e, int bits) {   // at the rate of a read-only launch
  return ((double)std::max<int64_t>(1, std::min(e, m)) * (double)(k * n) * bits / 8 + 2.0 * (double)m * (double)(k + n)) / 6.7e6;
}

double rows16_us(int64_t m, int64_t k, int64_t n, int64_t e, int64_t cus, bool packed, int bits, const Rows16Form &f) {
  const int64_t avg = (m + e - 1) / e, rows = e == 1 ? m : avg + avg / 10;   // (real routings are uneven)
  const int64_t groups = std::max<int64_t>(1, std::min(e, m)), chunks = (rows + 127) / 128;
  const double rb = (double)std::min<int64_t>(8, ((rows + chunks - 1) / chunks + 15) / 16);
  const int depth = rb <= 2 ? 6 : rb <= 4 ? 4 : 3;   // K blocks per unrolled round of the kernel
  const int64_t slice = ((k + 63) / 64 + f.split - 1) / f.split, own = (slice + f.sets - 1) / f.sets;
  const double blocks = (double)((own + depth - 1) / depth * depth);
  const double wgs = (double)((n + f.cols - 1) / f.cols) * (double)(groups * chunks * f.split);
  const bool pairs = f.cols == 256 && f.sets == 1 && wgs > (double)cus;
  const Rows16Cost &c = kRows16[packed][f.cols == 512 ? 0 : f.sets == 2 ? 3 : pairs ? 2 : 1];
  // (packed weights, two sets: a second round is a whole one.  257 .. 351 workgroups at w / CUs + 0.5 rounds were picked over the 32- and 64-row
  // kernels and took 1.1 times as long: 8 experts, 210 rows, 5472 x 8816 88 against 108 us)
  const bool two_rounds = packed && f.sets == 2 && wgs <= 2.0 * (double)cus &&
                          (double)((n + f.cols - 1) / f.cols) * (double)(groups * f.split) * (e == 1 ? (double)chunks : expected_row_tiles((double)m / (double)groups, 128.0)) > (double)cus;
  const double r = two_rounds ? 2.0 : chip_rounds(wgs, pairs ? 2.0 * (double)cus : (double)cus);
  const double us = c.fixed + r * (c.round + blocks * (c.block + c.rows * rb)) + c.stream * rows_stream_us(m, k, n, e, bits) + (f.split > 1 ? c.split + c.slice * rb * r * (f.split - 1) : 0.0);
  return pairs && r > 3 && rb >= 6 ? 1.07 * us : us;   // (what the fit is off by there: x comes in twice per CU)
}

// the kernels with 32- and 64-row chunks (tch = 2, 4)
double rows_small_us(int64_t m, int64_t k, int64_t n, int64_t e, int64_t cus, int tch, bool packed) {
  const int64_t avg = (m + e - 1) / e, chunk = 16 * tch, groups = std::max<int64_t>(1, std::min(e, m)), col_groups = (n + 15) / 16;
  const int64_t active = std::max<int64_t>(1, std::min<int64_t>(e * ((m + chunk - 1) / chunk), groups + m / chunk));
  const int wide = ((col_groups + 15) / 16) * active >= 2 * cus ? 16 : 8;   // column groups per strip (as planned below)
  const double wgs = (double)((col_groups + wide - 1) / wide) * (double)(groups * ((avg + avg / 10 + chunk - 1) / chunk));
  const double live = (double)std::min<int64_t>(tch, (avg + 15) / 16), blocks = (double)((k + 63) / 64) * wide / 16;
  const Rows16Cost &c = kRowsSmall[packed][tch == 4];
  return c.fixed + chip_rounds(wgs, 2.0 * (double)cus) * blocks * (c.block + c.rows * live) + c.stream * rows_stream_us(m, k, n, e, 8);
}

// 4-bit weights: these kernels read the nibbles; the model with their bytes picks forms that take 1.035 of the time of the best one (87
// shapes).  Beyond 30 rows per group on average they beat the 32-row chunks of the register-transpose kernels (us, those -> these: 33 rows, 64
// experts, 1376 x 1120 50 -> 37; 128 experts, 1696 x 1712 132 -> 91; 35 rows, 64 experts, 544 x 6032 93 -> 65; 37 rows, 32 experts, 3424 x
// 2608 112 -> 74; up to there 54 against 62 and 58 against 67, one group at most 128 rows either way), and what they replace beyond: the weights
// widened into the workspace first, then the kernels for int8 weights (64 experts, 6336 x 896, 89 rows 205 -> 113; 128 experts,
// 1536 x 1856, 76 rows 209 -> 98).
// `family_fits`: the kernels planned so far can take the shape (their grids are bounded; the 128-row kernel's is not)
void plan_rows16(msco_gmm_op *op, bool family_fits) {
  const msco_gmm_desc &d = op->desc;
  if ((op->family != FAM_SKINNY && family_fits) || !is_a16w8(d) || layout_of(d) == 1 || op->k >= ((int64_t)1 << 22)) return;   // (128 rows of x through 32-bit offsets)
  const int64_t m = op->m, k = op->k, n = op->n, e = op->e, cus = op->num_cus > 0 ? op->num_cus : kDefaultCUs;
  const int bits = is_w4(d) ? 4 : 8;
  GmmParams p{};
  p.m = (int)m;
  p.e = (int)e;
  auto workspace = [&](const Rows16Form &f) {
    return f.split > 1 ? (size_t)chunk_slots(p, 128) * ((n + f.cols - 1) / f.cols) * f.split * rows_a16w8_slice_bytes() : (size_t)0;
  };
  Rows16Form best{512, 1, 1};
  if (d.kernel_override == OV_ROWS16 || d.kernel_override == OV_ROWS16_256 || d.kernel_override == OV_ROWS16_256X2) {
    if (d.kernel_override != OV_ROWS16) best = Rows16Form{256, d.kernel_override == OV_ROWS16_256X2 ? 2 : 1, (int)std::min<int64_t>(std::max(d.force_split_k, 1), (k + 63) / 64)};
    while (best.split > 1 && workspace(best) > kTileSplitMaxWorkspace) --best.split;
  } else if (d.kernel_override != OV_AUTO || d.force_split_k != 0 || (family_fits && op->stream_tch == 1)) {
    return;
  } else if (bits == 4 && e >= 8 && k >= 512 && (m <= 30 * e || few_4bit_chunks(op))) {
    return;   // (the register-transpose kernels)
  } else if (e < 8 || k < 512) {
    // Outside what the model was fitted to (one group has kernels with a K split of its own): strips of 512 where they fill the chip and
    // a tile has rows enough.  One group, N = 11008, K = 4096, 512 (88 tiles) / 1024 (176) / 4096 rows: 91 -> 113, 158 -> 108, 444 -> 327 us
    // packed, 90 -> 107, 141 -> 116, 464 -> 347 us [E,K,N].
    const int64_t strips = (n + 511) / 512, avg = (m + e - 1) / e, rows = e == 1 ? m : avg + avg / 10;
    const int64_t tiles = strips * std::max<int64_t>(1, std::min<int64_t>(e, m)) * ((rows + 127) / 128), rounds = (tiles + cus - 1) / cus;
    const int64_t k_min = rows <= 128 ? (is_packed(d) ? 1024 : 2048) : is_packed(d) ? 512 : rows <= 256 ? 768 : 1280;
    if (!(k >= k_min && avg >= 48 && (tiles >= 2 * cus || tiles * 100 >= rounds * cus * 65) && n * 100 >= strips * 512 * 85)) return;
  } else {
    const int64_t avg = (m + e - 1) / e, rows = avg + avg / 10;
    // (strips of 512 not where N fills them to less than four fifths: 512 and 256 in one round take equally long by the model, but in 118 shapes of 22 to 2000 rows
    // a group and N = 528 .. 2464 one set on 256 takes 0.87 of the time; from four fifths on 0.97)
    const int64_t wide = (n + 511) / 512 * 512;
    if (n * 5 < wide * 4) best = Rows16Form{256, 1, 1};
    double us = rows16_us(m, k, n, e, cus, is_packed(d), bits, best);
    for (int sets = 1; sets <= 2; ++sets)
      for (int split = 1; split <= 4 && split <= (k + 63) / 64; ++split) {
        const Rows16Form f{256, sets, split};
        if (workspace(f) > (size_t)MSCO_GMM_STATIC_WORKSPACE_BYTES) break;   // (msco_gmm_launch_static takes what it took without a split)
        const double t = rows16_us(m, k, n, e, cus, is_packed(d), bits, f);
        if (t < us) {
          us = t;
          best = f;
        }
      }
    // (two sets of waves hide one another's waits where a CU has one workgroup; in more than a round, counted with a mean routing, one set takes
    // 0.93 of their time: 276 shapes, 8- and 4-bit weights; 5268 rows over 8 experts, 2688 x 4112 165 -> 145 us)
    const int64_t groups = std::min(e, m);
    if (best.sets == 2 && best.split == 1 && (double)((n + 255) / 256 * groups) * expected_row_tiles((double)m / (double)groups, 128.0) > 1.02 * (double)cus) best.sets = 1;
    // (4-bit weights that the register-transpose kernels can take: strips of 256 columns and 32-row chunks there are twice as many workgroups, which
    // counts where these fill no more than half of the chip: 8 experts, 330 rows, 4416 x 4096 39 against 48 us; 8138 random shapes of 30 to 42 rows per
    // group 0.83 of the time of what the model picked, 0.79 with a quarter of the chip, 0.85 with half of it)
    if (bits == 4 && avg + avg / 2 <= 64 && (n + best.cols - 1) / best.cols * std::min(e, m) * ((rows + 127) / 128) * best.split * 2 <= cus) return;
    // (the kernels for smaller chunks keep what is not clearly better here; 128-row chunks are always better off)
    // (nor what the model prices too low: one row block per group on more than two 256-column workgroups per CU, 26 shapes 1.08 of the time of the
    // smaller chunks (16 experts, 179 rows, 1760 x 8640 50.6 -> 59.5 us; two row blocks and more 0.87))
    const int64_t wgs = (n + best.cols - 1) / best.cols * std::min(e, m) * ((rows + 127) / 128) * best.split;
    const bool priced_low = best.cols == 256 && best.sets == 1 && rows <= 16 && wgs > 2 * cus;
    if (bits == 8 && family_fits && op->stream_tch <= 4 && (priced_low || 0.9 * rows_small_us(m, k, n, e, cus, op->stream_tch, is_packed(d)) < us)) return;
  }
  op->family = FAM_ROWS16;
  op->strip_cols = best.cols;
  op->wave_sets = best.sets;
  op->n_strips = (int)((n + best.cols - 1) / best.cols);
  op->split_k = best.split;
  op->workspace_bytes = workspace(best);
}

// 128-column tiles a launch is expected to have when no group has more rows than a tile
int64_t few_row_tiles(int64_t m, int64_t n, int64_t e) { return groups_hit(m, e) * ((n + 127) / 128); }

// int8 x on [E,K,N] or [E,N,K] weights, groups that a 32-row tile holds (gmm_tile_w8a8.hip): all the rows of one group, or 16 a
// group on average -- real routings are uneven.  Everything is us, the plan before -> the 32-row tile, 160 [E,K,N] and 100 [E,N,K] shapes of 1 to
// 800 rows, 1 to 128 experts, K = 512 .. 8192, N = 512 .. 14336, random routings (popularity even or falling as 1 / rank^0.6 or 1 / rank^1.2),
// each form measured on all of them: 0.80 of the time on [E,K,N], 0.93 with one group; four of 122 grouped shapes slower by 4 to 16 %.
//   up to 9/8 tiles of 128 columns per CU: 32 x 128.  16 experts, 18 rows, 3392 x 1168 24.6 -> 14.3; 32 experts, 18 rows, 640 x 2208 13.7 ->
//   9.0; one group, 13 rows, 7968 x 5392 20.2 -> 16.8; 64 experts, 76 rows, 7008 x 720 77.5 -> 55.9.
//   more: 32 x 256 (8 experts, 32 rows, 5632 x 5120 60.4 -> 48.7, 32 x 128: 62.4), or, where K below 1024 leaves its three-slab ring too
//   little to walk, 64 x 128 with 64-byte slabs and three workgroups per CU (16 experts, 162 rows, 864 x 4112 22.7 -> 15.3, 32 x 256: 18.8).
// The decode kernels keep what leaves most CUs idle whatever the tile, because their 16 waves split K inside a workgroup: a handful of
// rows over dozens of experts (64 experts, 1 row, 2272 x 800: 8.3 against 9.9; 5 rows, 800 x 1824: 8.0 against 8.8), one group of ten
// tiles and a long K (1 row, 3744 x 1120: 9.5 against 10.4), and several groups where that is K / 192 tiles, at least ten, of up to two rows for five
// experts (2 rows over 16, 7712 x 656: 13.6 against 16.9; 157 [E,K,N] shapes of up to 0.3 rows per expert 0.93 of the time of 32 x 128 tiles, 64 of three
// rows over eight 1.00; with more rows those have more tiles to share K: up to one row per expert 1.06, one to eleven 1.15; 63 rows over 8, 7680 x
// 528: 20.8 against 15.5).  They also keep K below 512 (not measured).  On [E,N,K] weights several groups take 64 x 128
// tiles already, which are as fast (60 shapes: 0.98), but for more than 32 experts and up to 64 rows (41 rows over 64 experts, 4352 x 688: 27.9 ->
// 20.3; 52 rows, 544 x 10576: 17.2 -> 15.3 with 64 x 128 tiles), where the decode kernels' plan dates from launches with workgroups for experts
// without rows.
void plan_few_rows(msco_gmm_op *op, int &family) {
  const int64_t m = op->m, k = op->k, n = op->n, e = op->e, cus = op->num_cus > 0 ? op->num_cus : kDefaultCUs;
  const bool nk = op->desc.transpose_b != 0;
  if (is_packed(op->desc) || k < 512 || (e == 1 ? m > 32 : m > 16 * e)) return;
  const int64_t tiles = few_row_tiles(m, n, e);
  if (e == 1 && !nk && m <= kSkinnyRows && tiles <= 10 && k >= 2048) return;
  if (e > 1 && ((nk && family != FAM_SKINNY) || tiles <= 10 || (!nk && family == FAM_SKINNY && tiles * 192 <= k && m * 5 <= e * 2) || (e >= 32 && m <= 5))) return;
  family = FAM_TILE;
  op->tile_cfg = tiles * 8 <= cus * 9 ? TILE_32x128 : nk || k < 1024 ? TILE_64x128 : TILE_32x256;
}

// Tiles just too many for one round of the chip.  128 x 128 and 64 x 128 tiles that are one to a CU walk K in 128-byte slabs with nothing
// masked; with more of them than CUs the plan gives them 64-byte slabs and two or three workgroups share a CU's loads, which takes about
// twice as long.  The next shape in one round (or in fewer, larger workgroups) is then the better one.  us, the tile picked above -> this,
// 1200 random shapes, all forms measured on each (one group of 33 to 4096 rows; 8 to 128 groups, even and uneven routings):
//   [E,K,N], 128 x 128 -> 128 x 256 from K = 1024: 45 shapes at 0.84 (0.63 .. 1.00); 8 experts, 165 rows, 7168 x 3696 122 -> 79; one group, 947 rows,
//   4224 x 4704 43 -> 34; not where N leaves a quarter of the wider tiles empty (8 experts, 718 rows, 1792 x 560 14.7 -> 19.6) or K is short
//   (10812 rows, 768 x 640 12.1 -> 15.7).
//   [E,K,N] and [E,N,K], 64 x 128 -> 128 x 128 from K = 2048 where those are one round: 12 shapes at 0.72 (0.59 .. 0.84); 8 experts, 97 rows, 5312 x
//   2368 55 -> 34; one group, 156 rows, 5184 x 13856 51 -> 39; shorter K 0.97 .. 1.11.  [E,N,K] tiles of 128 x 256 gain less (one group 0.94,
//   several 0.99, from 0.77 to 1.58) and are not taken.
//   [E,N,K], several groups, more than two 128 x 128 tiles per CU -> the persistent kernel where its tiles are one round on more than half of the
//   CUs, from K = 2048: 25 shapes at 0.78 (0.54 .. 1.04); 16 experts, 627 rows, 5472 x 1168 146 -> 79; 32 experts, 296 rows, 3520 x 864 71 -> 56.
//   ([E,K,N] from 128 x 256 tiles: 0.83, but up to 1.25.)
//   Packed weights stay (128 x 256 tiles for several groups 0.95, from 0.81 to 1.31; 64 x 128 for one group 0.94, from 0.77 to 1.04).
// 600 other shapes: 21 changed, 0.83 of the time, the worst 1.01.
// Which side of a round a launch of several groups falls is counted with the mean over the routings of its row tiles: "a tenth more rows" jumps by a
// tile per group just below a multiple of the tile (8 experts, 121 rows each: three 64-row tiles, 2.4 on average).
// Shapes between the two counts, us, the wider tile / the other:
// 128 x 256 where 128 x 128 are expected to be 180 .. 250 tiles 1.36 times as long (8 experts, 490 tokens x 4, 4032 x 1776 45.5 / 32.1), 260 and more
// 0.91; 128 x 128 where 64 x 128 are 180 .. 236 1.08 (skewed routings 1.07), 248 .. 256 0.99; a K split of 128 x 128 tiles that fill
// more than half of a round 1.25 (16 experts, 2872 rows, 3168 x 592, [E,N,K] two slices 33.5, 64 x 128 22.8).
bool plan_one_round(msco_gmm_op *op) {   // true: K is not to be split
  const int64_t m = op->m, k = op->k, n = op->n, e = op->e, cus = op->num_cus > 0 ? op->num_cus : kDefaultCUs;
  const bool packed = is_packed(op->desc), kn = !packed && !op->desc.transpose_b;
  auto tiles = [&](int64_t bm, int64_t bn) {   // an average group's and a tenth more rows (real routings are uneven)
    const int64_t groups = std::max<int64_t>(1, std::min(e, m)), rows = e == 1 ? m : (11 * m + 10 * e - 1) / (10 * e);
    return groups * ((rows + bm - 1) / bm) * ((n + bn - 1) / bn);
  };
  auto expected = [&](int64_t bm, int64_t bn) {
    return (e == 1 ? (double)((m + bm - 1) / bm) : (double)std::min(e, m) * expected_row_tiles((double)m / (double)std::min(e, m), (double)bm)) * (double)((n + bn - 1) / bn);
  };
  if (op->tile_cfg == TILE_128x128 && tiles(128, 128) > cus) {
    if (kn && k >= 1024 && n * 4 >= (n + 255) / 256 * 256 * 3 && (e == 1 || expected(128, 128) > (double)cus)) op->tile_cfg = TILE_128x256;
    else if (!packed && !kn && e > 1 && e <= 1024 && k >= 2048 && tiles(128, 128) > 2 * cus && tiles(256, 256) * 2 > cus && tiles(256, 256) <= cus) op->tile_cfg = TILE_256x256_W4;
  } else if (op->tile_cfg == TILE_64x128 && !packed && k >= 2048 && tiles(64, 128) > cus && expected(64, 128) * 16 > (double)(cus * 15) && tiles(128, 128) <= cus) {
    op->tile_cfg = TILE_128x128;
    // (a K split of more than half a round would make two rounds of one)
    return expected(128, 128) * 2 > (double)cus;
  }
  return false;
}

// Mean number of bm-row tiles of a group that holds `avg` rows on average and, in a random routing, scatters by about the root
// of that; and their variance.
struct TileMoments { double mean, var; };
TileMoments row_tile_moments(double avg, double bm) {
  const double sd = std::sqrt(std::max(avg, 1e-9));
  double t = std::max(0.0, std::floor((avg - 5.0 * sd) / bm)), mean = t, square = t * t;
  for (double rows = t * bm + 0.5; rows < avg + 5.0 * sd; rows += bm, t += 1.0) {
    const double p = 0.5 * std::erfc((rows - avg) / (sd * std::sqrt(2.0)));   // P(more than t tiles)
    mean += p;
    square += p * (2.0 * t + 1.0);
  }
  return {std::max(mean, 1e-3), std::max(square - mean * mean, 0.0)};
}

// Rounds that tiles of bm rows x bn columns make, one per CU, and the share of them that the CUs are busy: `busy` is tiles / CUs.
struct TileRounds { double rounds, busy; };
double even_busy(int64_t m, int64_t n, int64_t e, int64_t bm, int64_t bn, int64_t cus) {   // several groups
  const double groups = (double)std::min(e, m);
  return row_tile_moments((double)m / groups, (double)bm).mean * groups * (double)((n + bn - 1) / bn) / (double)cus;
}
TileRounds even_rounds(int64_t m, int64_t n, int64_t e, int64_t bm, int64_t bn, int64_t cus) {
  const double nt = (double)((n + bn - 1) / bn);
  if (e == 1) {
    const int64_t t = (m + bm - 1) / bm * (int64_t)nt;
    return {(double)((t + cus - 1) / cus), (double)t / (double)cus};
  }
  const double groups = (double)std::min(e, m);
  const TileMoments g = row_tile_moments((double)m / groups, (double)bm);
  const double mean = g.mean * groups, sd = std::sqrt(g.var * groups);
  double rounds = 0.0;
  for (double r = 0.0;; r += 1.0) {   // sum of P(more than r rounds): the row tiles are whole ones
    const double need = std::floor((double)cus * r / nt) + 0.5;
    const double p = sd < 1e-6 ? (mean > need ? 1.0 : 0.0) : 0.5 * std::erfc((need - mean) / (sd * std::sqrt(2.0)));
    if (p < 1e-3) break;
    rounds += p;
  }
  return {std::max(rounds, 1.0), mean * nt / (double)cus};
}
// ... with a popularity that falls as 1 / rank^z: a group of `avg` rows has avg / bm + 0.5 tiles where it has half a tile's rows, one below that, and min(avg, 1)
// where it expects less than a row.  The ranks of each kind follow one another, and the sums over them are those of rank^-z, by Euler and
// Maclaurin's formula from the 16th term on (off by less than 1e-7): a plan takes as long for 1024 groups as for 8 (adding them up one by one, for
// every tile shape: 128 groups 69 us on the host, now 5; 1024 groups 536, now 7).
class SkewedRouting {
 public:
  SkewedRouting(int64_t m, int64_t e, double z) : z_(z), e_((double)e) {
    for (int i = 1; i <= kFirst; ++i) first_[i] = first_[i - 1] + std::pow((double)i, -z);
    to_all_ = upto(e_);
    scale_ = (double)m / to_all_;   // rows of the first group
    expected_ = std::clamp(std::floor(std::pow(scale_, 1.0 / z)), 0.0, e_);   // groups of a row or more
    to_expected_ = upto(expected_);
  }
  TileRounds rounds(int64_t n, int64_t bm, int64_t bn, int64_t cus) const {
    const double tall = std::clamp(std::ceil(std::pow(2.0 * scale_ / (double)bm, 1.0 / z_)) - 1.0, 0.0, expected_);   // groups of more than half a tile's rows
    const double row_tiles = scale_ * upto(tall) / (double)bm + 0.5 * tall + (expected_ - tall) + scale_ * (to_all_ - to_expected_);
    const double t = row_tiles * (double)((n + bn - 1) / bn) / (double)cus;
    return {std::max(1.0, t + 0.5), t};
  }

 private:
  static constexpr int kFirst = 16;
  double upto(double i) const {   // sum of rank^-z over the first i ranks
    if (i <= (double)kFirst) return first_[(int)i];
    auto tail = [&](double r) { const double p = std::pow(r, -z_); return p * (r / (1.0 - z_) + 0.5 - z_ / (12.0 * r)); };
    return first_[kFirst] + tail(i) - tail((double)kFirst);
  }
  double z_, e_, first_[kFirst + 1] = {}, to_all_, scale_, expected_, to_expected_;
};

// The persistent kernel on tiles of other shapes than 256 x 256 (kT4mShape), against each other and against the 128 x 256, 128 x 128 and
// 64 x 128 tiles, by a model of the time in us (kTileTimes): rounds of one tile per CU, each a part per 128-byte K slab (more where K rows do not start on
// a line) and a fixed one; CUs without a tile in the last round leave the others more of the clock and of the L2, hence `idle`, and rows that do
// not exist draw less power, hence `empty`; and the weights have to be read (us per MB).  The operand stream of a CU is what 512 rows of
// either side take and the matrix pipe is busy for 64 blocks per wave, so a lower tile is dearer per product but wastes
// less: of a group's last row tile, and of the last round.  Fitted to 1900 random shapes (1 to 128 groups, 14 rows per group to
// 32768 rows, K = 512 .. 8192, N = 512 .. 14336, even and skewed routings, weights from memory), every shape and tile measured on all of them: off by
// 10 .. 16 % (rms), between shapes by less.  One group, picked here: 0.86 of the time of 256 x 256 tiles where those were planned.  Several: the device picks, as
// it alone knows how even they are (t4m_pick).  us, before -> now: one group of 2048 rows, 4096 x 11008, [E,N,K] 94 -> 83 (192 x 256; 344 tiles
// made two rounds on 172 CUs); 8 experts, 256 rows on average, 4096 x 14336, packed 160 -> 130 (288 x 224: 512 tiles for 672).
// The smaller tiles give way where the least time, over even and skewed routings, is 0.93 of theirs ([E,K,N], several groups: 0.88) and the tiles are
// more than 140 of 256 columns' worth (their K splits and second workgroups win below), several groups from 160 rows each on (128 experts, 2576 columns, 108 rows,
// packed 1.03), on [E,N,K] from 20 rows each where K is 2048 or more (64 experts, 46 rows, 768 x 1792 1.19, 14 rows, 1984 x 1008 1.08),
// 128 x 128 and 64 x 128 from K = 1536 (8 experts, 732 rows, 704 x 2608 1.17; one group of 2373 rows, 1120 x 1904 1.04).  1200 other shapes, of the time before: [E,N,K]
// 0.93 with several groups (32 experts, 49 rows, 5824 x 2304 0.71; 8 experts, 109 rows, 1760 x 10656 0.72), 0.99 with one (573 rows, 4928 x 6544 0.66);
// [E,K,N] 0.99 and 0.98 (1643 rows, 4608 x 2480 0.78); packed 0.99.
bool tile_shapes_fit(const msco_gmm_desc &d) {   // shapes other than 256 x 256 are built for these outputs only
  return d.out_dtype != MSCO_DT_I32 && (d.act_type == ACT_NONE || d.act_type == ACT_SILU || d.act_type == ACT_FAST_GELU);
}

void plan_tile_shape(msco_gmm_op *op) {
  const msco_gmm_desc &d = op->desc;
  const int64_t m = op->m, k = op->k, n = op->n, e = op->e, cus = op->num_cus > 0 ? op->num_cus : kDefaultCUs;
  const bool large = op->tile_cfg == TILE_256x256_W4, tall = op->tile_cfg == TILE_128x256, small = op->tile_cfg == TILE_128x128, low = op->tile_cfg == TILE_64x128;
  const bool nk = layout_of(d) == 1;
  if (!(large || tall || small || low) || k < ((small || low) ? 1536 : 512) || e > 1024 || !tile_shapes_fit(d)) return;
  if (e > 1) {
    if (large) {
      // (beyond six rounds the other shapes save nothing -- 19 shapes 0.99 of the time -- and counting them takes a microsecond or two: 64 experts,
      // 49152 rows, 2048 x 2816, [E,K,N], skewed 327.7 / 326.0; not packed groups of just more than 256 rows, of which 256 x 256 tiles make two: choose_plan)
      const int64_t avg_rows = (m + e - 1) / e;
      const bool just_beyond = is_packed(d) && avg_rows > 256 && avg_rows <= 296;
      op->tile_shape = !just_beyond && even_busy(m, n, e, 256, 256, cus) > 6.0 ? 0 : -1;
      return;
    }
    if (m < 160 * e && !(nk && m >= 20 * e && k >= 2048)) return;
  }
  const TileTimes &t = kTileTimes[layout_of(d)];
  T4mPick pick{};
  tile_shape_times(layout_of(d), k, pick);
  const double mb = (double)(std::min(e, m) * k) * (double)n * 1e-6;
  auto both = [](double tiles_us, double read_us) { return std::sqrt(std::sqrt(tiles_us * tiles_us * tiles_us * tiles_us + read_us * read_us * read_us * read_us)); };
  // the least time of the shapes, and that of the tile planned so far, for an even routing (null) or a skewed one
  int best = 0;
  double best_tiles = 0.0;   // for an even routing, in tiles of 256 columns
  auto rounds = [&](int64_t bm, int64_t bn, const SkewedRouting *skewed) {
    return skewed ? skewed->rounds(n, bm, bn, cus) : even_rounds(m, n, e, bm, bn, cus);
  };
  auto least = [&](const SkewedRouting *skewed) {
    double us = 0.0;
    for (int j = 0; j < T4M_SHAPES; ++j) {
      if (pick.us[j] <= 0.0f) continue;
      const int64_t bm = 32 * kT4mShape[j].xb, bn = 32 * kT4mShape[j].wb;
      const TileRounds r = rounds(bm, bn, skewed);
      const double rows = r.busy * (double)cus / (double)((n + bn - 1) / bn) * (double)bm;   // of all tiles, whether they exist or not
      const double u = t.launch + both(((1.0 - t.idle) * r.rounds + t.idle * r.busy) * (double)pick.us[j] * (1.0 - t.empty * std::max(0.0, 1.0 - (double)m / rows)), mb * t.read);
      if (j > 0 && u >= us) continue;
      us = j == 0 && large ? 0.97 * u : u;
      if (!skewed) {
        best = j;
        best_tiles = r.busy * (double)cus * (double)bn / 256.0;
      }
    }
    return us;
  };
  auto now = [&](const SkewedRouting *skewed) {
    const TileTime &o = tall ? t.tall : small ? t.small : t.low;
    const TileRounds r = rounds(low ? 64 : 128, tall ? 256 : 128, skewed);
    return o.launch + both(((1.0 - o.idle) * r.rounds + o.idle * r.busy) * ((double)k / 128.0 * o.slab * (k % 128 != 0 ? 1.0 + o.unaligned : 1.0) + o.fixed), mb * o.read);
  };
  double us = least(nullptr);
  if (!large) {
    double old = now(nullptr);
    if (e > 1) {
      const SkewedRouting some(m, e, 0.6), strong(m, e, 1.2);
      us = 0.5 * us + 0.25 * least(&some) + 0.25 * least(&strong);
      old = 0.5 * old + 0.25 * now(&some) + 0.25 * now(&strong);
    }
    if (best_tiles <= 140.0 || us >= (layout_of(d) == 0 && e > 1 ? 0.88 : 0.93) * old) return;
  }
  op->tile_cfg = TILE_256x256_W4;
  op->tile_shape = e > 1 ? -1 : best;
}

void choose_plan(msco_gmm_op *op) {
  const msco_gmm_desc &d = op->desc;
  const int num_cus = op->num_cus;
  const int64_t m = op->m, k = op->k, n = op->n, e = op->e;
  const bool aligned = (k % 16 == 0) && (n % 16 == 0) && k >= 16 && n >= 16;
  op->split_k = 1;
  op->skinny_wide16 = 0;
  op->skinny_cols = kSkinnyCols;
  op->n_strips = (int)((n + kSkinnyCols - 1) / kSkinnyCols);
  op->workspace_bytes = 0;
  op->tile_cfg = TILE_256x256;
  op->wide_k_slabs = 0;
  op->w_nontemporal = 0;
  op->small_group_rows = 0;
  op->tile_shape = 0;
  op->shallow = false;

  int family;
  // All three W8A8 weight layouts follow the same tile rules: packed weights are K-contiguous per column like [E,N,K],
  // and [E,K,N] weights run the same LDS-direct tile kernels (transpose reads turn them on the way out of LDS; rows of
  // whole 16-column chunks, which the alignment rule guarantees).  Only the decode kernels are per layout.
  // (a group that overflows its 16-row chunk streams its weights twice, so 1.5 x the average has to fit; beyond that
  // the 64 x 128 tile kernel with non-temporal weight loads is the better streamer -- 128 rows over 8 experts, 470 MB
  // of weights: 76 us against 82 us for the 32-row streaming kernel and 105 us for 16-row chunks; row-major [E,N,K]:
  // 111 us against 140 us)
  // row-major [E,N,K] weights at decode sizes: a column's K bytes are contiguous and the columns are K bytes apart, which
  // suits the 64 x 128 tile's LDS-direct loads better than the decode kernel's 64-byte row pieces (K = 4096, N = 11008,
  // 1 / 16 rows: 15.8 / 15.9 us against 16.8 / 17.7 us; 32 rows over 8 experts, N = 14336: 103 against 115 us)
  // (a few rows over hundreds of experts are the decode kernel's again -- 40 rows over 256 experts, K = 512, N = 7168: 41 us
  // against 95 us -- but not a thousand rows over them: K = 2048, N = 7168: 635 against 595 us, K = 7168, N = 4096: 1467
  // against 1244 us)
  const bool nk_rows = is_w8a8(d) && d.transpose_b != 0 && !is_packed(d) && !(e > 32 && m <= kSkinnyMaxRows);
  const int64_t avg_rows = (m + (e > 0 ? e : 1) - 1) / (e > 0 ? e : 1);
  // (the decode kernels' grid enumerates the chunks that hold rows -- at most min(E, M) + M / 16 of them -- so experts
  // without rows cost nothing)
  const bool many_small_groups = e > 1 && avg_rows + avg_rows / 2 <= kSkinnyRows &&
                                 std::min<int64_t>(m, e) + m / kSkinnyRows <= kSkinnyMaxChunkSlots;
  if (!aligned) {
    family = FAM_GENERIC;
  } else if (is_a16w8(d)) {
    family = FAM_SKINNY;  // the weight-only path is a decode path; large M re-streams weights per 16 rows
  } else if (((m <= kSkinnyMaxRows && !(e == 1 && m > kSkinnyRows)) || many_small_groups) && !nk_rows) {
    // decode: few rows in total, or groups of about one 16-row chunk each (the weights stream once per chunk).  The
    // grid enumerates every (group, chunk) a malformed-to-the-limit group_list could fill; beyond a thousand slots
    // the empty workgroups cost more than the tile kernel's partial tiles.  A single group of more than one 16-row
    // chunk takes the small tile kernel with a K split instead (measured on packed weights, K = 4096, N = 11008:
    // 32 / 48 / 64 rows 17.1 / 17.5 / 18.0 us against 18.7 / 24.4 / 26.3 us of the multi-row streaming kernel, which
    // stays for several groups of a few dozen rows each; [E,K,N] weights, same shape, 17 / 32 / 64 rows: 16.5 / 16.9 /
    // 18.3 us).
    family = FAM_SKINNY;
  } else {
    family = FAM_TILE;
    // tile shape from shapes only: average rows per group and how many tiles fill 256 CUs
    const int64_t rows_per_group = m / (e > 0 ? e : 1);
    auto tiles = [&](int bm, int bn) { return ((m + bm - 1) / bm) * ((n + bn - 1) / bn); };
    // several groups, a few dozen to a few hundred rows each: the launch is bound by the weight
    // stream (every group's matrix is read once per m-tile of the group), so the m-tile should hold a whole group --
    // real routings are uneven, hence 1.5 x the average -- as long as there are tiles for most CUs.  Measured (E = 8,
    // K = 4096, N = 14336, packed; 64 x 128 / 128 x 128 / 256 x 256 tiles): 64 rows per group 112 / 97 / 100 us, 128 rows per
    // group 162 / 150 / 109 us (136 us with 128 x 256), 32 rows per group 87.5 us with the first.
    auto group_tiles = [&](int bm, int bn) { return e * ((rows_per_group + bm - 1) / bm) * ((n + bn - 1) / bn); };
    const int64_t cover = rows_per_group + rows_per_group / 2;
    const int64_t busy = (num_cus > 0 ? num_cus : kTileTargetWorkgroups) * 3 / 4;
    // (the persistent four-wave kernel: at least four 128-byte K slabs per tile, a group table that fits in LDS)
    const bool w4_ok = k >= 512 && e <= 1024;
    // (128-row m-tiles while every group fits one: 8 experts, 72 .. 112 rows per group on average, the largest group 80 ..
    // 126 rows: 84 - 92 us with 128 x 256 tiles against 100 - 109 us with 256 x 256; at 120 rows on average the largest
    // group has 131, streams its weights twice and the launch takes 126 against 113 us -- so the 256-row tile takes
    // over at 1.5 x the average = 174 rows, not at 128; at 112 rows on average, the largest group 126, [E,K,N] weights:
    // 104 us with 128 x 256 tiles against 116 us)
    // Packed weights, several groups of up to about 150 rows each and enough columns that 256-column strips give every CU
    // a workgroup: the row-chunk kernels stream a group's weights once, straight into MFMA operands, and multiply only
    // the 16-row blocks that hold rows.  Measured, 8 experts, K = 4096, N = 14336 (470 MB of weights; a launch that only
    // reads them takes 72 us), rows per group 16 / 32 / 64 / 96 / 112: 72.8 / 75.8 / 79.2 / 83.8 / 85.9 us with 128-row
    // chunks against 76.5 / 79.6 / 82.4 / 89.1 / 111.0 us for the tiles picked below.  A group that overflows its chunk
    // takes a second workgroup that streams its weights again (128 rows on average, half of the groups above 128: 131 us),
    // hence 160-row chunks from 116 rows on average (still two workgroups per CU, with room for two K blocks of weights
    // in flight only): 120 / 128 / 136 / 144 rows per group 88.6 / 89.3 / 91.6 / 91.7 us against 100 / 103 / 103 / 105 us
    // with 256-row chunks (one workgroup per CU) and 110 - 112 us for the persistent kernel.  256-row chunks are left with
    // 147 .. 155 rows per group (152 rows, the largest group 164: 107.9 against 118 us); the persistent kernel wins beyond
    // (160 rows: 115 us either way; 192 rows: 125 against 115 us).  Few columns leave CUs idle: N = 1344, K = 5120: 41
    // against 24 us for 64 x 128 tiles with a K split.
    // (narrower strips for fewer columns do not pay: with one or two column groups per wave, strips of 6 / 3 column groups,
    // 8 experts, 1024 rows, K = 5120, N = 2688 / 1344: 55 / 40 us against 46 / 24 us for the 64 x 128 tiles)
    const bool rows_kernel_ok = is_packed(d) && e > 1 && k >= 1024 && ((n + 255) / 256) * std::min<int64_t>(e, m) >= num_cus;
    // The 160-row form again where a group is two or three equal chunks that share its weights through the L2.  All figures are
    // routings by the top-2 of random logits (groups as uneven as real ones), us, former plan -> this.
    //   257 .. 296 rows per group on average: the persistent kernel's 256-row tiles give a group of just more than 256 rows a second m-tile. 8 experts,
    //   K = 4096, N = 14336, 260 / 290 rows: 167 -> 149, 197 -> 160; 64 experts, 2048 x 1408, 260 / 275 / 290: 84 -> 79, 90 -> 82, 90 -> 89; 128 experts, 4096
    //   x 1024, 270: 213 -> 188.  Its other shapes, picked from the groups in any number of rounds, take over where the outputs have them: uneven groups leave
    //   CUs without chunks idle, tiles of 256 columns less so.  615 random shapes of 8 to 256 experts, shapes over chunks for even routings / popularity as 1 /
    //   rank^0.6 / 1 / rank^1.2: up to two chunk workgroups per CU, their one round, 0.93 / 0.79 / 0.87 (at worst 1.13), up to four 1.04 / 0.94 / 0.94 (1.19), more of
    //   them 1.01 / 1.00 / 0.98 from K = 2816 on (1.16) and 1.06 / 1.02 / 1.01 below, where the chunks stay.  (256 x 256 tiles alone 1.20 / 0.97 / 1.00; 8 experts, 4096 x
    //   14336, 257 .. 296 rows: shapes 1.00 / 0.95 / 0.93.)  More than 256 groups, whose every chunk workgroup walks them all: up to 511 columns 0.86 / 0.85 / 0.66,
    //   more columns 0.96 / 0.97 / 0.86 (140 shapes); beyond the persistent kernel's 1024 groups eight-wave tiles up to 511 columns, 0.92 / 0.70 / 0.60, not from
    //   512 on, 1.31 / 0.99 / 1.19 (33 shapes).
    //   297 .. 340 (three chunks): 8 experts, 4096 x 14336, 300 / 335 rows: 205 -> 177, 199 -> 189; 2816 x 5664, 330: 80 -> 72; 16 experts,
    //   4096 x 4096, 320: 112 -> 113; not beyond: 8 experts, 2816 x 5664, 400 rows 70 -> 77.
    //   192 .. 256 where larger tiles than 128 x 128 do not fill the chip but these workgroups do: 8 experts, 7168 x 4096, 200 / 250
    //   rows: 91 -> 73, 120 -> 79; 2816 x 4096, 200 / 250: 38 -> 33, 55 -> 37.  A short K needs the 250: 2048 x 4096, 210 / 250 rows 24.2 ->
    //   28.8, 36.6 -> 33.9; 16 experts, 2048 x 2048, 230 / 250: 29.9 -> 33.8, 36.4 -> 35.4.
    // Popularity falling as 1 / rank^0.6 and 1 / rank^1.2 in place of even: the second band lies between 0.90 and 1.14, the third
    // between 1.0 and 1.5 times the former plan's speed; which it will be only the device knows.
    // Where 256-row tiles fill the chip, 256 rows on average and fewer stay with them: even groups of 240 rows, one m-tile each, take
    // 126 us there (8 experts, 4096 x 14336) and 141 us here; random routings of 256 rows on average 158 and 147 us.
    const int64_t row_wgs = ((n + 255) / 256) * std::min<int64_t>(e, m) * ((avg_rows + avg_rows / 20 + 159) / 160);
    const int64_t cus = num_cus > 0 ? num_cus : kDefaultCUs;
    const bool by_groups = tile_shapes_fit(d) && d.force_split_k == 0 && (e <= 256 ? k >= 2816 || row_wgs <= 4 * cus : e <= 1024 || n < 512);   // (plan_tile_shape follows)
    const bool rows_chunks_ok = is_packed(d) && e > 1 && k >= 2048 &&
                                ((avg_rows > 256 && avg_rows <= 296 && row_wgs >= 172 && !by_groups) || (avg_rows > 296 && avg_rows <= 340 && n >= 4096 && row_wgs >= 256) ||
                                 (avg_rows >= 192 && avg_rows <= 256 && n >= 2048 && (k >= 2816 || avg_rows >= 250) && row_wgs >= 172 && row_wgs <= 256 && group_tiles(256, 256) < busy));
    if (rows_kernel_ok && avg_rows <= 116) {
      op->tile_cfg = TILE_ROWS128;
    } else if (rows_kernel_ok && avg_rows <= 146) {
      op->tile_cfg = TILE_ROWS160;
    } else if (rows_kernel_ok && avg_rows <= 155) {
      op->tile_cfg = TILE_ROWS256;
    } else if (rows_chunks_ok) {
      op->tile_cfg = TILE_ROWS160;
    } else if (e > 1 && w4_ok && cover > 174 && cover <= 384 && group_tiles(256, 256) >= busy) {
      op->tile_cfg = TILE_256x256_W4;
    } else if (e > 1 && cover > 64 && cover <= 192 && group_tiles(128, 128) >= busy) {
      // (128 x 256 tiles re-read x half as often: 64 / 96 rows per group 93 / 99 us against 100 / 111 us)
      op->tile_cfg = group_tiles(128, 256) >= busy ? TILE_128x256 : TILE_128x128;
    } else if (e == 1 && w4_ok && tiles(256, 256) >= busy * 2 / 3 && tiles(128, 256) > busy * 4 / 3) {
      // one group, a few hundred to a thousand rows: the persistent kernel already on half of the CUs
      // when 128 x 256 tiles would no longer run in one round (N = 11008: M = 768 / 1024: 47 / 52 us against 63 / 68 us
      // with 128 x 128 tiles) ...
      op->tile_cfg = TILE_256x256_W4;
    } else if (e == 1 && tiles(128, 256) >= busy * 4 / 5 && tiles(128, 256) <= busy * 4 / 3) {
      // ... and 128 x 256 tiles while they do and fill most of the chip (M = 448 .. 640: 40 - 42 us against 45 - 47 us;
      // M = 384, 129 tiles: 41 us against 35 us with 128 x 128)
      op->tile_cfg = TILE_128x256;
    } else if (rows_per_group >= 192 && tiles(256, 256) >= 256) {
      op->tile_cfg = w4_ok ? TILE_256x256_W4 : TILE_256x256;
    } else if (rows_per_group >= 96 && tiles(128, 128) >= 256) {
      op->tile_cfg = TILE_128x128;
    } else if (tiles(128, 128) >= 512) {
      op->tile_cfg = TILE_128x128;
    } else if (rows_per_group >= 192 && tiles(128, 128) > kTileSplitMaxTiles) {
      // a few hundred rows: 128 x 128 tiles on at least half of the CUs beat twice as many 64 x 128
      // tiles (measured: M = 256, N = 11008: 32 us against 44 us); with fewer tiles the K split of the small tile wins
      op->tile_cfg = TILE_128x128;
    } else {
      op->tile_cfg = TILE_64x128;
    }
  }
  bool one_round = false;
  if (d.kernel_override == OV_AUTO && aligned && is_w8a8(d) && !is_w4(d)) {
    one_round = family == FAM_TILE && plan_one_round(op);
    plan_few_rows(op, family);
    if (family == FAM_TILE && d.force_split_k == 0) plan_tile_shape(op);
  }
  switch (d.kernel_override) {
    case OV_TILE_256: family = FAM_TILE; op->tile_cfg = TILE_256x256; break;
    case OV_TILE_256_W4: family = FAM_TILE; op->tile_cfg = TILE_256x256_W4; break;
    case OV_TILE_256_W4_MFMA32: family = FAM_TILE; op->tile_cfg = TILE_256x256_W4_MFMA32; break;
    case OV_W4_128: case OV_W4_160: case OV_W4_192: case OV_W4_224: case OV_W4_288: case OV_W4_128x192: case OV_W4_160x192:
      family = FAM_TILE;
      op->tile_cfg = TILE_256x256_W4;
      if (!tile_shapes_fit(d)) break;
      op->tile_shape = d.kernel_override >= OV_W4_288 ? 5 + d.kernel_override - OV_W4_288 : OV_W4_224 + 1 - d.kernel_override;
      if (layout_of(d) == 0 && d.kernel_override == OV_W4_288) op->tile_shape = 0;
      break;
    case OV_TILE_128: family = FAM_TILE; op->tile_cfg = TILE_128x128; break;
    case OV_TILE_128x256: family = FAM_TILE; op->tile_cfg = TILE_128x256; break;
    case OV_TILE_64: family = FAM_TILE; op->tile_cfg = TILE_64x128; break;
    case OV_ROWS128: family = FAM_TILE; op->tile_cfg = is_packed(d) ? TILE_ROWS128 : TILE_128x256; break;
    case OV_ROWS256: family = FAM_TILE; op->tile_cfg = is_packed(d) ? TILE_ROWS256 : TILE_256x256_W4; break;
    case OV_ROWS160: family = FAM_TILE; op->tile_cfg = is_packed(d) ? TILE_ROWS160 : TILE_256x256_W4; break;
    case OV_TILE_32x128: family = FAM_TILE; op->tile_cfg = is_packed(d) ? TILE_64x128 : TILE_32x128; break;
    case OV_TILE_32x256: family = FAM_TILE; op->tile_cfg = is_packed(d) ? TILE_64x128 : d.transpose_b ? TILE_32x128 : TILE_32x256; break;
    case OV_SKINNY: family = FAM_SKINNY; break;
    case OV_GENERIC: family = FAM_GENERIC; break;
    default: break;
  }
  // (what the persistent kernel cannot take runs the eight-wave kernel of the same tile shape; the plan says so)
  if (family == FAM_TILE && (op->tile_cfg == TILE_256x256_W4 || op->tile_cfg == TILE_256x256_W4_MFMA32) && !(k >= 512 && e <= 1024))
    op->tile_cfg = TILE_256x256;
  // the MFMA kernels address x and one group's weights through 32-bit buffer offsets
  const bool fits32 = (is_packed(d) ? (int64_t)packed_weight_bytes(k, n) : k * n) < ((int64_t)1 << 31) &&
                      m * k < ((int64_t)1 << 31);
  if ((family == FAM_TILE || family == FAM_SKINNY) && !(aligned && fits32)) family = FAM_GENERIC;
  if (family == FAM_TILE && !is_w8a8(d)) family = FAM_SKINNY;
  if (family == FAM_TILE) {
    const int forced = tuning().tile_cfg;
    if (forced >= 0 && forced < TILE_CFG_COUNT && d.kernel_override == OV_AUTO) op->tile_cfg = forced;
    if ((op->tile_cfg == TILE_ROWS256 || op->tile_cfg == TILE_ROWS160) && !is_packed(d)) op->tile_cfg = TILE_256x256_W4;
    if (op->tile_cfg == TILE_ROWS128 && !is_packed(d)) op->tile_cfg = TILE_128x256;
    // Few tiles (M of a few hundred rows): split K across workgroups until about kTileTargetWorkgroups of them
    // stream operands; every slice keeps at least kTileMinSlabs 64-byte K slabs.  Small tile shapes only.
    const bool few = op->tile_cfg == TILE_32x128;
    if (op->tile_cfg == TILE_128x128 || op->tile_cfg == TILE_64x128 || few || op->tile_cfg == TILE_32x256) {
      int bm, bn;
      tile_cfg_dims(op->tile_cfg, &bm, &bn);
      // tiles the launch is expected to have: every group that holds rows has at least one m-tile
      const int64_t groups_with_rows = std::min<int64_t>(e, m);
      const int64_t t = few ? few_row_tiles(m, n, e) : std::max<int64_t>((m + bm - 1) / bm, groups_with_rows) * ((n + bn - 1) / bn);
      // t tiles x s slices run in ceil(t s / CUs) rounds (the operand ring takes most of a CU's LDS: one workgroup per
      // CU).  In units of one 64-byte K slab of a tile (0.2 us): a round costs its slabs plus 10 (prologue, epilogue),
      // a split adds 8 per slice for 64 x 128 tiles and 12 for 128 x 128 (its partial tile out and in, one round trip of
      // the last arriver), less 2.  The cheapest s wins, the smaller one on a tie.  Fitted to M = 128, K = N = 4096
      // (64 tiles; s = 1 / 2 / 3 / 4 / 6: 18.7 / 15.2 / 14.5 / 15.3 / 21.3 us) and M = 64, K = 4096, N = 11008 (86 tiles;
      // s = 1 / 2 / 3: 20.9 / 18.0 / 24.3 us, the third slice starting a second round).  Of the 32 x 128 tiles two share a CU, in a
      // fifth more time than one alone, and the exchange is half as large: 128 experts, 24 rows, 3264 x 976, s = 1 / 2: 21.7 / 16.9; 16 experts,
      // 18 rows, 3392 x 1168: 16.0 / 14.3; 8 experts, 16 rows, 6400 x 2304: 32.6 / 30.3; 16 experts, 12 rows, 608 x 2096: 7.8 / 9.7.
      // One group (206 random shapes of 1 to 400 rows, every split measured): a slice adds less than that -- 4 and 6 in place of 6 and 8, and 2
      // once -- and two 32 x 128 tiles on a CU take 1.6 times one alone.  32 x 128 0.971 of the time, none slower (7 rows, 6176 x 10464 26.2 ->
      // 21.5; 3 rows, 7552 x 4256 15.4 -> 14.0), 64 x 128 0.991 (41 rows, 2720 x 1200 10.9 -> 9.6).  Its rounds are those of an XCD, which takes an
      // eighth of the tiles, rounded up, with all their slices: three slices of 81 to 85 tiles are 33 workgroups for 32 CUs.  Counted over the
      // chip that was one round.  7778 random shapes that this changes, 0.83 of the time, one slower by more than 0.05: 64 x 128, three
      // slices -> two 0.77 (72 rows, 2688 x 5280, [E,N,K] 15.6 -> 11.3), 32 x 128, 62 to 64 tiles, three -> four 0.95.  Four slices of 57 to
      // 64 32 x 128 tiles leave no CU of an XCD idle, and the exchange is 2 dearer: 260 shapes, four slices against three K = 3000 .. 4000 1.045
      // (23 rows, 3616 x 8048 11.6 / 11.0), to 5000 0.996, to 6500 0.95, beyond 0.93.
      const int cus = or_default(tuning().tile_target_wgs, num_cus > 0 ? num_cus : kTileTargetWorkgroups);
      const int cap = (int)std::max<int64_t>(1, ((k + 63) / 64) / kTileMinSlabs);
      // (several groups, more than 11 and up to 16 rows each on average: all of them hold rows, some of them more than a tile, and a second tile per CU costs what it
      // costs with one group.  2411 such shapes 0.85 of the time of the splits before, none
      // with an even routing slower than 64 x 128 tiles (32 experts, 364 rows, 3616 x 832 28.3 -> 22.1); up to 11 rows a group the 1.2 times stand, as a random routing leaves groups empty)
      const bool full_groups = (m + e - 1) / e * 3 / 2 > kSkinnyRows;
      auto split_cost = [&](int sl) {
        const int64_t slabs = ((k + 63) / 64 + sl - 1) / sl;
        const bool one_small = e == 1 && (few || op->tile_cfg == TILE_64x128);
        const int64_t xcd_cus = std::max(1, cus / kNumXcd);
        const int64_t xcd_tiles = (t + kNumXcd - 1) / kNumXcd;
        const int64_t rounds = e == 1 ? (xcd_tiles * sl + xcd_cus - 1) / xcd_cus : (t * sl + cus - 1) / cus;
        const int64_t fifths = few && rounds > 1 ? (rounds + 1) / 2 * (e == 1 || full_groups ? 8 : 6) : rounds * 5;
        const int64_t full_xcd = e == 1 && few && sl == 4 && xcd_tiles * sl == xcd_cus ? 2 : 0;
        const int64_t exchange = sl <= 1 ? 0 : one_small ? (int64_t)(2 + bm * bn / 2048) * sl + 2 + full_xcd : (int64_t)(4 + bm * bn / 2048) * sl - 2;
        return fifths * (slabs + 10 + exchange);
      };
      int want = 1;
      if (!one_round && t <= (few ? 2 * kTileSplitMaxTiles : kTileSplitMaxTiles)) {
        for (int sl = 2; sl <= std::min(kMaxSplitK, cap); ++sl)
          if (split_cost(sl) < split_cost(want)) want = sl;
      }
      const int forced_split = d.force_split_k > 0 ? d.force_split_k : tuning().tile_split_k;
      if (forced_split > 0) want = std::min(forced_split, cap);
      // the partial tiles of a K split are sized for the worst group_list (one partial m-tile per group): with many
      // groups that bound dwarfs the problem, so the split is halved until the workspace fits under the cap
      // (few rows: no more than a launch without a workspace of the caller's has)
      const size_t most_bytes = few && d.force_split_k <= 0 ? (size_t)MSCO_GMM_STATIC_WORKSPACE_BYTES : kTileSplitMaxWorkspace;
      while (want > 1 && tile_workspace_bytes(op->tile_cfg, m, n, e, want) > most_bytes) want /= 2;
      op->split_k = want;
      op->workspace_bytes = tile_workspace_bytes(op->tile_cfg, m, n, e, op->split_k);
      // 128-byte K slabs (a 4-stage ring of them takes most of a CU's LDS: one workgroup per CU) when the workgroups
      // run in one round; more tiles than CUs keep 64-byte slabs and two workgroups per CU (M = 512, N = 11008: 344
      // tiles, 46.8 us against 50.1 us)
      op->wide_k_slabs = t * want <= (num_cus > 0 ? num_cus : kTileTargetWorkgroups);
      if (tuning().tile_wide_k >= 0) op->wide_k_slabs = tuning().tile_wide_k != 0;
    }
    if (op->tile_cfg == TILE_128x128 || op->tile_cfg == TILE_64x128 || op->tile_cfg == TILE_128x256 || few || op->tile_cfg == TILE_32x256) {
      // Non-temporal weight loads: a weight stream of tens of megabytes that at most two m-tiles read should not push x
      // out of the caches (E = 8 x 32 rows, 470 MB: 87.7 -> 79.4 us; M = 128, 45 MB: 20.8 -> 19.6 us); three m-tiles
      // re-read it from the cache and lose badly without it there (M = 384: 35 -> 47 us), and a weight set the caches
      // hold anyway gains nothing (M = 128, 16.8 MB: 13.8 -> 14.4 us).
      int bm, bn;
      tile_cfg_dims(op->tile_cfg, &bm, &bn);
      const int64_t group_rows = e > 1 ? (m / e) + (m / e) / 2 : m;
      // ([E,K,N] rows: a wave instruction brings whole lines too; 470 MB over 8 experts, 64 / 128 rows in all: 94 -> 84 us
      // and 97 -> 87 us; on 45 MB it loses a little -- 32 rows 16.9 -> 17.3 us -- so the bar is higher there)
      const int64_t nt_bytes = is_packed(d) ? ((int64_t)32 << 20) : ((int64_t)64 << 20);
      op->w_nontemporal = (is_packed(d) || d.transpose_b == 0) && e * k * n >= nt_bytes && (group_rows + bm - 1) / bm <= 2;
    }
    if (op->tile_cfg == TILE_128x256 && tuning().tile_wide_k >= 0) op->wide_k_slabs = tuning().tile_wide_k != 0;   // (measured slower with 128-byte slabs: 99 against 93 us)
  }
  if (family == FAM_TILE && (op->tile_cfg == TILE_ROWS256 || op->tile_cfg == TILE_ROWS128 || op->tile_cfg == TILE_ROWS160)) {
    // Row-chunk kernel: every workgroup streams a strip of up to 16 column groups over all of K plus its chunk's x rows,
    // and the workgroups that share a CU share its operand path.  The strip is as wide as makes the bytes a CU moves
    // least: ceil(workgroups / CUs) x (strip bytes + x bytes of a chunk), one chunk per group expected.  8 experts x 14336
    // columns on 256 CUs: 448 workgroups of 16 column groups cost two per CU as 512 of 14 do (c3_t64 82.2 -> 72.8 us).
    const int64_t cus = num_cus > 0 ? num_cus : kDefaultCUs;
    const int64_t col_groups = (n + 15) / 16, groups = std::max<int64_t>(1, std::min<int64_t>(e, m));
    const int64_t chunk_rows = op->tile_cfg == TILE_ROWS128 ? 128 : op->tile_cfg == TILE_ROWS160 ? 160 : 256;
    const int64_t group_chunks = std::max<int64_t>(1, (avg_rows + chunk_rows - 1) / chunk_rows), x_bytes = (avg_rows + group_chunks - 1) / group_chunks * k;
    int best = 16;
    int64_t best_cost = INT64_MAX;
    for (int sg = 16; sg >= 10; --sg) {
      const int64_t wgs = ((col_groups + sg - 1) / sg) * groups * group_chunks;
      const int64_t cost = ((wgs + cus - 1) / cus) * ((int64_t)sg * 16 * k + x_bytes);
      if (cost < best_cost) { best_cost = cost; best = sg; }
    }
    op->strip_groups = best;
    const int forced_groups = tuning().stream_groups;
    if (forced_groups >= 1 && forced_groups <= 16) op->strip_groups = forced_groups;
    op->n_strips = (int)((col_groups + op->strip_groups - 1) / op->strip_groups);
    op->w_nontemporal = avg_rows <= chunk_rows;   // (the 128- and 256-row forms are planned for one chunk per group and always set the bit)
  }
  // Many experts with uneven loads (a skewed routing): every group of a few rows costs the persistent kernel a whole
  // 256-row m-tile per n-tile.  The groups of at most 64 rows go to a second launch of 64 x 128 tiles instead, which
  // streams their weights once with non-temporal loads.  On the skewed 64-expert workload (49152 rows, K = 2048, N = 2816;
  // 29 groups of at most 64 rows) the persistent kernel's tiles go from 10.2 to 8.9 per workgroup and the pair of launches
  // measures 336 against 348 us on packed weights and 340 against 352 us on [E,K,N]; on [E,N,K] weights (64-byte row
  // pieces, no non-temporal loads) 347 against 350, not worth a launch.  Which groups are small only the device knows;
  // with few experts the second launch would mostly find none.
  if (family == FAM_TILE && op->tile_cfg == TILE_256x256_W4 && (is_packed(d) || d.transpose_b == 0) && e >= 16 &&
      (d.kernel_override == OV_AUTO || d.kernel_override == OV_TILE_256_W4) && tuning().two_level != 0)
    op->small_group_rows = 64;
  op->stream_tch = 1;
  bool rows16_fits = false;   // more (expert, chunk) pairs than the other weight-only kernels' grids hold
  if (family == FAM_SKINNY && is_packed(d) && is_w8a8(d)) {
    // rows a group is expected to hold (shapes only): 16-row chunks up to 16 rows, else chunks of 32 / 64 / 128 rows
    // (several groups: 1.5 x the average, real routings are uneven and a group that overflows its chunk streams its
    // weights twice -- 128 rows over 8 experts: 90.5 us with 32-row chunks against 105 us with 16-row chunks)
    const int64_t avg = (m + e - 1) / e;
    const int64_t rows = e == 1 ? m : avg + avg / 2;
    op->stream_tch = rows <= 16 ? 1 : rows <= 32 ? 2 : rows <= 64 ? 4 : 8;
    // fewer, larger chunks when there would be more chunks than the grid should enumerate
    while (op->stream_tch < 8 && std::min<int64_t>(m, e) + m / (16 * op->stream_tch) > or_default(tuning().stream_max_slots, (int)kSkinnyMaxChunkSlots))
      op->stream_tch = op->stream_tch == 1 ? 2 : op->stream_tch * 2;
    if (tuning().stream_tch == 1 || tuning().stream_tch == 2 || tuning().stream_tch == 4 || tuning().stream_tch == 8) op->stream_tch = tuning().stream_tch;
  } else if (family == FAM_SKINNY && is_a16w8(d) && (is_packed(d) || (d.transpose_b == 0 && n % 16 == 0))) {
    // weight-only on packed or [E,K,N] weights: chunks of 32, 64 or 128 rows by the same estimate; larger groups stream
    // their weights once per chunk (8 experts, K = 4096, N = 14336, 128 / 512 / 2048 rows: 111 / 334 / 1307 us with
    // 16-row chunks)
    const int64_t avg = (m + e - 1) / e;
    const int64_t rows = e == 1 ? m : avg + avg / 2;
    op->stream_tch = rows <= 16 ? 1 : rows <= 32 ? 2 : rows <= 64 ? 4 : 8;
    while (op->stream_tch < 8 && std::min<int64_t>(m, e) + m / (16 * op->stream_tch) > or_default(tuning().stream_max_slots, (int)kSkinnyMaxChunkSlots))
      op->stream_tch *= 2;
    // One group whose column strips do not fill the chip: the multi-row kernels walk all of K in every workgroup (only
    // the 128-row form has a K split, below), and for few rows the 16-row kernels with their K split are faster
    // although they stream the weights once per 16 rows (K = 4096, N = 11008, 32 / 64 rows: packed 24 / 41 us against
    // 49 / 51; [E,K,N] 32 us against 39 at 32 rows -- its 33 to 64 rows go on to the 128-row form, 39 us against 48).
    if (e == 1 && (n + 127) / 128 < num_cus && m <= (is_packed(d) ? 64 : 32)) op->stream_tch = 1;
    if (tuning().stream_tch == 1 || tuning().stream_tch == 2 || tuning().stream_tch == 4 || tuning().stream_tch == 8)
      op->stream_tch = tuning().stream_tch;
  }
  int64_t max_chunks = 1;   // chunks of 16 * stream_tch rows that a group can have
  if (family == FAM_SKINNY) {
    // grid.y enumerates (group, chunk) pairs
    const int64_t chunk_rows = (int64_t)kSkinnyRows * op->stream_tch;
    max_chunks = std::max<int64_t>(1, (m + chunk_rows - 1) / chunk_rows);
    if (e * max_chunks > 65535) {
      family = FAM_GENERIC;
      rows16_fits = is_a16w8(d);
    }
  }
  if (family == FAM_SKINNY) {
    // Only shapes enter: the number of (group, chunk) pairs that can hold rows is estimated from M and E.
    const int64_t active = std::max<int64_t>(
      1, std::min<int64_t>(e * max_chunks, std::min<int64_t>(m, e) + m / (kSkinnyRows * op->stream_tch)));
    const int64_t tiles128 = ((n + 127) / 128) * active;
    int wide16 = is_w8a8(d) && tiles128 <= num_cus && !is_packed(d);
    const int forced_variant = tuning().skinny_wide16;
    if (forced_variant >= 0 && is_w8a8(d)) wide16 = forced_variant != 0;
    op->skinny_wide16 = wide16;
    int want, cap;
    if (op->stream_tch > 1 && !is_w8a8(d)) {
      // multi-row weight-only kernels: strips of 16 column groups (256 columns) when they still give every CU two
      // workgroups, else of 8; every workgroup walks all of K (one exception below).
      const int64_t col_groups = (n + 15) / 16;
      op->strip_groups = ((col_groups + 15) / 16) * active >= 2 * (int64_t)num_cus ? 16 : 8;
      op->n_strips = (int)((col_groups + op->strip_groups - 1) / op->strip_groups);
      op->skinny_cols = op->strip_groups * 16;
      want = cap = 1;
      // One group whose strips leave most CUs idle: 128-row chunks with a K split (slices of at least 8 blocks) up to
      // about two workgroups per CU.  K = 4096, N = 11008, 128 / 256 / 512 rows without it: 59 / 61 / 83 us.
      const int64_t base = (int64_t)op->n_strips * active, k_blocks = (k + 63) / 64;
      if (e == 1 && base < num_cus && tuning().stream_tch == 0) {
        op->stream_tch = 8;
        max_chunks = (m + 127) / 128;
        want = (int)std::min<int64_t>(kTargetWorkgroups / std::max<int64_t>((int64_t)op->n_strips * max_chunks, 1), kMaxSplitK);
        cap = std::max<int>(1, (int)(k_blocks / 8));
      }
    } else if (is_packed(d) && op->stream_tch > 1) {
      // multi-row kernel: strips of four column groups, K split until about two workgroups per CU stream operands
      const int64_t col_groups = (n + 15) / 16, k_blocks = (k + 63) / 64;
      op->strip_groups = 4;
      op->n_strips = (int)((col_groups + 3) / 4);
      op->skinny_cols = 64;
      const int64_t base = (int64_t)op->n_strips * active;
      want = (int)(kTargetWorkgroups / std::max<int64_t>(base, 1));
      cap = std::max<int>(1, (int)(k_blocks / 16));      // a slice keeps at least 16 blocks
      want = std::max(1, std::min(std::min(want, kMaxSplitK), cap));
    } else if (is_packed(d)) {
      // Packed weights: strips as wide as still give every CU a workgroup.  With int8 x, where one workgroup walks all of K, those are counted over the
      // groups that a random routing hits (16 experts, 16 rows, 800 x 4176: 14.6 -> 11.1 us with the strips that follow; 329 int8
      // shapes of 8 to 128 experts 0.988 of the time that one workgroup per group that can be hit gives; 16-bit x gains 0.4 % over 449 shapes and loses 5 %
      // on some of them: 100 rows over 16 experts, 3776 x 1440 19.6 -> 20.6).
      // A slice of K holds 128 blocks of 64 bytes, with 16-bit x 64.  Beyond 64 the 16-bit kernel would take two slices of 9 to 16 blocks
      // per wave in the code for 16, most requests of a shorter one masked: slices of at most 32 blocks, eight per wave, instead (us, two
      // slices -> three, random routings: 18 rows over 16 experts, 4288 x 2320 44.1 -> 28.8; 14 rows, one group, 4288 x 8288 21.7 -> 14.4; 4 rows over 16
      // experts, 4352 x 1136 12.0 -> 11.1; 96 rows over 16, 6016 x 1792 48.8 -> 38.7).  Up to 64 blocks one slice is as good.  (Where the two slices are
      // one workgroup per CU they are 3 % faster on 38 grouped shapes, but slower on others: 140 where that rule applied 1.03 of the time, one group 1.02.)
      const int64_t col_groups = (n + 15) / 16, k_blocks = (k + 63) / 64;
      const int slice_blocks = is_w8a8(d) ? 128 : 64, fewest = (int)((k_blocks + slice_blocks - 1) / slice_blocks);
      const bool short_slices = !is_w8a8(d) && fewest > 1 && k_blocks <= 32 * kMaxSplitK;
      const int floor_split = short_slices ? (int)((k_blocks + 31) / 32) : fewest;
      const int64_t hit = floor_split > 1 || !is_w8a8(d) ? active : std::min(active, groups_hit(m, e) * std::max<int64_t>(1, (m / e + kSkinnyRows - 1) / kSkinnyRows));
      int groups = 16;
      const int min_wgs = or_default(tuning().stream_min_wgs, num_cus);
      while (groups > 1 && ((col_groups + groups - 1) / groups) * hit * floor_split < min_wgs) groups /= 2;
      const int forced_groups = tuning().stream_groups;
      if (forced_groups >= 1 && forced_groups <= 16) groups = forced_groups;
      op->strip_groups = groups;
      op->n_strips = (int)((col_groups + groups - 1) / groups);
      op->skinny_cols = groups * 16;
      // No split beyond that: a strip of one column group is a walk of K / 256 requests per wave, and the exchange costs more than any
      // of it saves (us, two workgroups per CU through a split -> none: one row, 2688 x 2800 8.1 -> 5.1; 13 rows, 8128 x 1568 13.0 -> 7.9; 5 rows
      // over 32 experts, 5536 x 576 8.9 -> 6.7; 16-bit x, one row, 3520 x 3920 9.9 -> 6.9; up to 1024 columns and K from 4096, where two slices stayed
      // longest: 8336 shapes, two slices 1.14 of the time of one, K = 4096 1.15 to 1.19, K = 8192 1.07 to 1.17).
      // (short slices only where msco_gmm_launch_static takes their partial tiles too)
      want = floor_split;
      if (short_slices && decode_tiles(m, n, e, kSkinnyRows, op->skinny_cols) * (size_t)want * stream_a16w8_tile_bytes() > (size_t)MSCO_GMM_STATIC_WORKSPACE_BYTES) want = fewest;
      cap = kMaxSplitK * 64;
    } else if (wide16) {
      // at most one 16-wave workgroup per CU, every wave keeps at least one block
      want = (int)(num_cus / std::max<int64_t>(tiles128, 1));
      cap = std::max<int>(1, (int)(d.transpose_b ? (k + 63) / 64 : (k + 31) / 32) / 16);
      want = std::min(want, 8);
    } else {
      // K is split across workgroups until about kTargetWorkgroups of them stream weights
      const int64_t base = (int64_t)op->n_strips * active;
      const int target = or_default(tuning().skinny_target_wgs, 2 * num_cus);
      want = (int)((target + base / 2) / base);
      cap = std::max<int>(1, (int)(d.transpose_b ? (k + 63) / 64 : (k + 31) / 32) / 4);
      want = std::min(want, kMaxSplitK);
    }
    want = std::max(1, std::min(want, cap));
    const int forced = d.force_split_k > 0 ? d.force_split_k : tuning().skinny_split_k;
    if (forced > 0) want = std::min(forced, cap);
    if (is_packed(d) && op->stream_tch == 1) {   // also under a forced split
      const int slice_blocks = is_w8a8(d) ? 128 : 64;
      want = std::max(want, (int)(((k + 63) / 64 + slice_blocks - 1) / slice_blocks));
    }
    if (op->stream_tch > 1 && !is_w8a8(d) && !(e == 1 && op->stream_tch == 8)) want = 1;   // the multi-row weight-only kernels walk all of K, but for one group in 128-row chunks
    op->split_k = want;
    if (!is_packed(d) && !(op->stream_tch > 1 && !is_w8a8(d))) op->skinny_cols = wide16 ? 128 : kSkinnyCols;
    size_t slice_bytes = (size_t)kSkinnyRows * op->skinny_cols * 4;
    if (op->stream_tch > 1 && !is_w8a8(d)) slice_bytes = rows32_a16w8_slice_bytes(op->strip_groups);
    else if (is_packed(d))   // (the packed-layout kernels keep a full 16 x 256 partial tile per (strip, K slice) whatever the strip's width)
      slice_bytes = !is_w8a8(d) ? stream_a16w8_tile_bytes() : op->stream_tch > 1 ? streamm_tile_bytes(op->stream_tch) : (size_t)kSkinnyRows * kSkinnyCols * 4;
    else if (!is_w8a8(d)) slice_bytes = 0;   // (plan_regt's)
    op->workspace_bytes = op->split_k > 1 ? decode_tiles(m, n, e, kSkinnyRows * op->stream_tch, op->skinny_cols) * (size_t)op->split_k * slice_bytes : 0;
  }
  op->family = family;
  op->widen_bytes = 0;
  plan_rows16(op, !rows16_fits);
  plan_regt(op);

  family = op->family;
  char buf[320];
  const char *fam = family == FAM_REGT ? (op->shallow ? "skinny_regt_shallow" : "skinny_regt") : family == FAM_ROWS16 ? (op->strip_cols == 512 ? "rows128" : op->wave_sets == 2 ? "rows128x256_2" : "rows128x256") : family == FAM_TILE ? (op->tile_cfg >= TILE_32x128 ? "skinny_tile" : "tile") : family == FAM_SKINNY ? "skinny" : "generic";
  std::snprintf(buf, sizeof(buf),
                "msco_gmm plan: kernel=%s%s%s%s layout=%s m=%lld k=%lld n=%lld e=%lld split_k=%d strips=%d "
                "workspace=%zu%s%s",
                is_w4(d) ? (op->widen_bytes > 0 ? (is_w8a8(d) ? "a8w4_widened_" : "a16w4_widened_") : (is_w8a8(d) ? "a8w4_" : "a16w4_"))
                         : is_w8a8(d) ? "w8a8_" : "a16w8_", (family == FAM_SKINNY && is_packed(d)) ? (op->stream_tch > 1 ? "stream_rows" : "stream")
                : (family == FAM_SKINNY && op->stream_tch > 1)    ? "skinny_rows" : fam,
                family == FAM_TILE ? (std::string("_") + tile_cfg_name(op->tile_cfg)).c_str() : "",
                (family == FAM_SKINNY && op->skinny_wide16) ? "_16w" : "",
                is_packed(d) ? "packed" : d.transpose_b ? "[E,N,K]" : "[E,K,N]", (long long)m, (long long)k, (long long)n, (long long)e,
                op->split_k, op->n_strips, op->workspace_bytes,
                op->small_group_rows > 0 ? (" small_groups=" + std::to_string(op->small_group_rows) + ":tile_64x128").c_str() : "",
                family == FAM_TILE && op->tile_cfg == TILE_256x256_W4 && op->tile_shape != 0
                    ? (op->tile_shape < 0 ? std::string(" tile_rows=by_groups") : " tile_rows=" + std::to_string(32 * kT4mShape[op->tile_shape].xb) + (kT4mShape[op->tile_shape].wb == 6 ? "x192" : "")).c_str() : "");
  op->info = buf;
}

}  // namespace

extern "C" {

int msco_gmm_abi_version(void) { return MSCO_GMM_ABI_VERSION; }

const char *msco_status_string(int status) {
  switch (status) {
    case MSCO_OK: return "ok";
    case MSCO_ERR_INVALID_ARG: return "invalid argument";
    case MSCO_ERR_UNSUPPORTED: return "unsupported dtype or layout";
    case MSCO_ERR_SHAPE: return "shape rule violated";
    case MSCO_ERR_NOT_PLANNED: return "launch before plan";
    case MSCO_ERR_WORKSPACE: return "workspace missing or too small";
    case MSCO_ERR_DEVICE: return "HIP runtime error";
    default: return "unknown status";
  }
}

int msco_gmm_create(const msco_gmm_desc *desc, msco_gmm_handle *out_handle) {
  if (desc == nullptr || out_handle == nullptr) return MSCO_ERR_INVALID_ARG;
  const int rc = check_desc(*desc);
  if (rc != MSCO_OK) return rc;
  msco_gmm_op *op = new (std::nothrow) msco_gmm_op();
  if (op == nullptr) return MSCO_ERR_DEVICE;
  op->desc = *desc;
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) == hipSuccess && hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess &&
      cus > 0) {
    op->num_cus = cus;
  } else {
    (void)hipGetLastError();   // no device yet: planning falls back to the MI355X count, launch reports the error
  }
  *out_handle = op;
  return MSCO_OK;
}

// Planning allocates, clears and frees counters, also while a stream of this thread is being captured (the first call of a shape under
// capture plans there): the runtime refuses these calls in the default capture mode and spoils the capture.  Relaxed, it takes
// them, as none of them belongs to the captured stream -- but nothing on the null stream, so clearing has a stream of its own.
namespace {
constexpr int kMaxDevices = 64;
struct RelaxedCapture {
  hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
  RelaxedCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
  ~RelaxedCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
  RelaxedCapture(const RelaxedCapture &) = delete;
};

std::mutex g_clear_mu;
hipStream_t g_clear_stream[kMaxDevices] = {};

bool clear_counters(unsigned *counters, size_t count) {   // and wait for it
  int dev = -1;
  hipStream_t stream = nullptr;
  {
    std::lock_guard<std::mutex> lock(g_clear_mu);
    if (hipGetDevice(&dev) == hipSuccess && dev >= 0 && dev < kMaxDevices &&
        (g_clear_stream[dev] != nullptr || hipStreamCreateWithFlags(&g_clear_stream[dev], hipStreamNonBlocking) == hipSuccess))
      stream = g_clear_stream[dev];
  }
  if (stream != nullptr && hipMemsetAsync(counters, 0, count * sizeof(unsigned), stream) == hipSuccess && hipStreamSynchronize(stream) == hipSuccess) return true;
  (void)hipGetLastError();
  return false;
}

void free_counters(msco_gmm_op *h) {
  if (h->counters != nullptr && !h->counters_recorded) (void)hipFree(h->counters);
  h->counters = nullptr;
  h->counters_cap = 0;
  h->counters_recorded = false;
}

// A recorded launch is replayed whenever its graph is: after the handle is gone or re-planned, and beside eager launches and other graphs.
// So the launches that one capture records through one handle (they are ordered) count in a range of this array that is handed
// out once.  It is zero when the library is loaded, counters reset themselves at the end of a launch, nothing is
// allocated under capture.  Once it is used up, a recorded launch counts with its handle's own counters, which then stay allocated.
constexpr size_t kRecordedCounters = (size_t)4 << 20;
static __device__ unsigned recorded_counters[kRecordedCounters];
std::mutex g_recorded_mu;
unsigned *g_recorded_ptr[kMaxDevices] = {};
size_t g_recorded_used[kMaxDevices] = {};

unsigned *take_recorded_counters(size_t count) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) {
    (void)hipGetLastError();
    return nullptr;
  }
  std::lock_guard<std::mutex> lock(g_recorded_mu);
  if (g_recorded_ptr[dev] == nullptr) {
    void *ptr = nullptr;
    if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(recorded_counters)) != hipSuccess || ptr == nullptr) {
      (void)hipGetLastError();
      return nullptr;
    }
    g_recorded_ptr[dev] = static_cast<unsigned *>(ptr);
  }
  count = (count + 15) / 16 * 16;   // (ranges of different captures share no 64-byte piece)
  if (count > kRecordedCounters - g_recorded_used[dev]) return nullptr;
  unsigned *at = g_recorded_ptr[dev] + g_recorded_used[dev];
  g_recorded_used[dev] += count;
  return at;
}

// the arrival counters of a launch on `stream`
unsigned *launch_counters(msco_gmm_op *h, hipStream_t stream) {
  if (h->split_k <= 1 || h->counters == nullptr || stream == nullptr) return h->counters;   // (the null stream is not captured)
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  unsigned long long id = 0;
  if (hipStreamGetCaptureInfo(stream, &status, &id) != hipSuccess) {
    (void)hipGetLastError();
    return h->counters;
  }
  if (status != hipStreamCaptureStatusActive) return h->counters;
  std::lock_guard<std::mutex> lock(h->mu);
  if (h->recorded == nullptr || h->recorded_id != id || h->recorded_cap < h->counters_used) {
    h->recorded = take_recorded_counters(h->counters_used);
    h->recorded_cap = h->recorded != nullptr ? h->counters_used : 0;
    h->recorded_id = id;
  }
  if (h->recorded != nullptr) return h->recorded;
  h->counters_recorded = true;
  return h->counters;
}
}  // namespace

int msco_gmm_plan(msco_gmm_handle h, int64_t m, int64_t k, int64_t n, int64_t e, size_t *workspace_bytes) {
  if (h == nullptr) return MSCO_ERR_INVALID_ARG;
  if (m < 0 || k <= 0 || n <= 0 || e <= 0) return MSCO_ERR_SHAPE;
  if (m > INT32_MAX || k > INT32_MAX || n > INT32_MAX || e > 65535 || m * n > ((int64_t)1 << 40)) return MSCO_ERR_SHAPE;
  if (h->desc.group_list_dtype == MSCO_DT_NONE && m % e != 0) return MSCO_ERR_SHAPE;
  if (is_w4(h->desc) && n % 2 != 0) return MSCO_ERR_SHAPE;   // [E,K,N/2] bytes hold pairs of columns
  std::lock_guard<std::mutex> lock(h->mu);
  h->m = m; h->k = k; h->n = n; h->e = e;
  choose_plan(h);
  if (h->family != FAM_GENERIC && h->split_k > 1) {
    GmmParams p{};
    p.m = (int)m;
    p.e = (int)e;
    const size_t need = h->family == FAM_ROWS16 ? (size_t)chunk_slots(p, 128) * h->n_strips
                        : h->family == FAM_REGT ? (size_t)chunk_slots(p, 16 * h->row_blocks) * h->n_strips
                        : h->family == FAM_TILE ? tile_count_bound(h->tile_cfg, m, n, e)
                                              : decode_tiles(m, n, e, kSkinnyRows * h->stream_tch, h->skinny_cols);
    const RelaxedCapture relaxed;
    h->counters_used = need;
    if (need > h->counters_cap) {
      free_counters(h);
      if (hipMalloc(reinterpret_cast<void **>(&h->counters), need * sizeof(unsigned)) != hipSuccess) {
        (void)hipGetLastError();
        return MSCO_ERR_DEVICE;
      }
      if (!clear_counters(h->counters, need)) return MSCO_ERR_DEVICE;
      h->counters_cap = need;
    } else if (h->counters != nullptr) {
      // the counters reset themselves at the end of a launch; one that was abandoned half-way (a failed launch, a
      // destroyed stream) may have left tickets behind, so a new plan starts from zero again
      if (!clear_counters(h->counters, h->counters_cap)) return MSCO_ERR_DEVICE;
    }
  }
  h->planned = true;
  if (workspace_bytes) *workspace_bytes = h->workspace_bytes;
  if (tuning().print_plan) std::fprintf(stderr, "%s\n", h->info.c_str());
  return MSCO_OK;
}

int msco_gmm_plan_info(msco_gmm_handle h, char *buf, size_t buf_len) {
  if (h == nullptr) return -1;
  std::lock_guard<std::mutex> lock(h->mu);
  if (buf && buf_len) {
    std::strncpy(buf, h->info.c_str(), buf_len - 1);
    buf[buf_len - 1] = '\0';
  }
  return (int)h->info.size();
}

int msco_gmm_launch(msco_gmm_handle h, const void *const *inputs, void *out, void *workspace, size_t workspace_bytes,
                    void *stream) {
  if (h == nullptr || inputs == nullptr) return MSCO_ERR_INVALID_ARG;
  if (!h->planned) return MSCO_ERR_NOT_PLANNED;
  const msco_gmm_desc &d = h->desc;
  if (h->m == 0) return MSCO_OK;
  if (out == nullptr || inputs[MSCO_IN_X] == nullptr || inputs[MSCO_IN_WEIGHT] == nullptr) return MSCO_ERR_INVALID_ARG;
  // a present dtype needs a pointer, an absent one must not get one
  auto need = [&](int slot, int dtype) { return (dtype != MSCO_DT_NONE) == (inputs[slot] != nullptr); };
  if (!need(MSCO_IN_BIAS, d.bias_dtype) || !need(MSCO_IN_SCALE, d.scale_dtype) ||
      !need(MSCO_IN_GROUP_LIST, d.group_list_dtype) || !need(MSCO_IN_PER_TOKEN_SCALE, d.per_token_dtype) ||
      !need(MSCO_IN_ANTIQUANT_SCALE, d.antiquant_dtype))
    return MSCO_ERR_INVALID_ARG;
  if ((d.has_antiquant_offset != 0) != (inputs[MSCO_IN_ANTIQUANT_OFFSET] != nullptr)) return MSCO_ERR_INVALID_ARG;
  if (h->workspace_bytes > 0 && (workspace == nullptr || workspace_bytes < h->workspace_bytes))
    return MSCO_ERR_WORKSPACE;

  GmmParams p{};
  p.x = inputs[MSCO_IN_X];
  p.w = static_cast<const int8_t *>(inputs[MSCO_IN_WEIGHT]);
  p.bias = static_cast<const int32_t *>(inputs[MSCO_IN_BIAS]);
  p.scale = inputs[MSCO_IN_SCALE];
  p.group_list = inputs[MSCO_IN_GROUP_LIST];
  p.per_token = static_cast<const float *>(inputs[MSCO_IN_PER_TOKEN_SCALE]);
  p.aq_scale = inputs[MSCO_IN_ANTIQUANT_SCALE];
  p.aq_offset = inputs[MSCO_IN_ANTIQUANT_OFFSET];
  p.out = out;
  p.partial = static_cast<int32_t *>(workspace);
  if (is_w4(d) && (reinterpret_cast<uintptr_t>(p.w) & 15) != 0) return MSCO_ERR_INVALID_ARG;
  if (h->widen_bytes > 0) {
    // 4-bit weights on their way to a kernel that reads int8: the int8 copy sits at the front of the workspace
    if (launch_unpack_int4(p.w, workspace, h->e * h->k * h->n / 2, static_cast<hipStream_t>(stream)) != hipSuccess) return MSCO_ERR_DEVICE;
    p.w = static_cast<const int8_t *>(workspace);
    p.partial = reinterpret_cast<int32_t *>(static_cast<char *>(workspace) + h->widen_bytes);
  }
  p.counters = launch_counters(h, static_cast<hipStream_t>(stream));
  p.m = (int)h->m; p.k = (int)h->k; p.n = (int)h->n; p.e = (int)h->e;
  p.gl_dtype = d.group_list_dtype;
  p.gl_type = d.group_list_type;
  p.scale_dtype = d.scale_dtype;
  p.scale_per_group = d.scale_per_group;
  p.scale_is_scalar = d.scale_is_scalar;
  p.out_dtype = d.out_dtype;
  p.x_dtype = d.x_dtype;
  p.split_k = h->split_k;
  p.n_strips = h->n_strips;
  p.strip_groups = h->strip_groups;
  p.act_type = d.act_type;
  // rows a 16-row chunk is expected to hold (shapes only): measured on the dense 45 MB decode, 16 rows 13.1 -> 12.35 us with
  // the x rows staged through LDS, one row 11.85 -> 12.2 us, four rows per chunk (8 experts x 32 rows) 70.1 -> 70.4 us
  p.x_via_lds = (h->e > 0 ? (h->m + h->e - 1) / h->e : h->m) >= 8;
  p.wide_k_slabs = h->wide_k_slabs;
  p.w_nontemporal = h->w_nontemporal;
  p.rows_lo = 0;
  p.rows_hi = 0x7FFFFFFF;

  hipStream_t s = static_cast<hipStream_t>(stream);
  hipError_t err = hipSuccess;
  const bool nk = d.transpose_b != 0;
  const int layout = layout_of(d);
  T4mPick pick{h->tile_shape};
  if (h->tile_shape < 0) tile_shape_times(layout, h->k, pick);
  if (h->family == FAM_REGT) {
    err = launch_regt(p, is_w4(d) ? 4 : 8, h->row_blocks, h->strip_cols, h->shallow, s);
  } else if (h->family == FAM_ROWS16) {
    err = launch_rows_a16w8(p, layout == 2, is_w4(d), h->strip_cols, h->wave_sets, s);
  } else if (is_w8a8(d)) {
    if (h->family == FAM_TILE && h->small_group_rows > 0) {
      GmmParams big = p, small = p;
      big.rows_lo = h->small_group_rows;
      small.rows_hi = h->small_group_rows;
      small.split_k = 1;
      small.wide_k_slabs = 0;              // (128-byte slabs measured slower here: 340 against 336 us)
      small.w_nontemporal = layout == 2 || !nk;   // each small group's weights are read by one m-tile (packed, [E,K,N])
      err = launch_tile_w8a8(big, h->tile_cfg, nk, layout == 2, pick, s);
      if (err == hipSuccess) err = launch_tile_w8a8(small, TILE_64x128, nk, layout == 2, pick, s);
    } else if (h->family == FAM_TILE && is_w4(d) && h->widen_bytes == 0) err = launch_tile_a8w4(p, h->tile_cfg, s);
    else if (h->family == FAM_TILE) err = launch_tile_w8a8(p, h->tile_cfg, nk, layout == 2, pick, s);
    else if (h->family == FAM_SKINNY && layout == 2) err = h->stream_tch > 1 ? launch_streamm_w8a8(p, h->stream_tch, s) : launch_stream_w8a8(p, s);
    else if (h->family == FAM_SKINNY) err = launch_skinny_w8a8(p, nk, h->skinny_wide16 != 0, s);
    else err = launch_generic_w8a8(p, layout, s);
  } else {
    if (h->family == FAM_SKINNY && h->stream_tch > 1) err = launch_streamm_a16w8(p, h->stream_tch, layout == 2, s);
    else if (h->family == FAM_SKINNY && layout == 2) err = launch_stream_a16w8(p, s);
    else err = launch_generic_a16w8(p, layout, s);
  }
  return err == hipSuccess ? MSCO_OK : MSCO_ERR_DEVICE;
}

// ---- launch without a caller workspace ----------------------------------------------------------------------------
// The split-K partial tiles go to a fixed device array instead of a caller buffer.  Host code never passes the array's
// name to a kernel or a runtime call (on the host it is a stand-in, not a device address): the address on each device
// is looked up once with hipGetSymbolAddress, with that device current, and kept.
namespace {
static __device__ __align__(256) unsigned char scratch[MSCO_GMM_STATIC_WORKSPACE_BYTES];
std::mutex g_scratch_mu;
void *g_scratch_ptr[kMaxDevices] = {};

// the current device's copy of `scratch`; nullptr (and *status set) on failure
void *scratch_of_current_device(int *status) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) {
    (void)hipGetLastError();
    *status = MSCO_ERR_DEVICE;
    return nullptr;
  }
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_ptr[dev] == nullptr) {
    void *ptr = nullptr;
    if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess || ptr == nullptr) {
      (void)hipGetLastError();
      *status = MSCO_ERR_DEVICE;
      return nullptr;
    }
    g_scratch_ptr[dev] = ptr;
  }
  return g_scratch_ptr[dev];
}
}  // namespace

int msco_gmm_launch_static(msco_gmm_handle h, const void *const *inputs, void *out, void *stream) {
  if (h == nullptr || inputs == nullptr) return MSCO_ERR_INVALID_ARG;
  if (!h->planned) return MSCO_ERR_NOT_PLANNED;
  if (h->workspace_bytes > (size_t)MSCO_GMM_STATIC_WORKSPACE_BYTES) {
    std::fprintf(stderr, "msco_gmm_launch_static: the plan needs %zu bytes of workspace, the static one holds %zu\n",
                 h->workspace_bytes, (size_t)MSCO_GMM_STATIC_WORKSPACE_BYTES);
    return MSCO_ERR_WORKSPACE;
  }
  int status = MSCO_OK;
  void *ws = scratch_of_current_device(&status);
  if (ws == nullptr) return status;
  // nothing in the array has to start at zero: every K slice writes its whole partial tile before it takes a ticket,
  // and the tickets live in the handle
  return msco_gmm_launch(h, inputs, out, ws, (size_t)MSCO_GMM_STATIC_WORKSPACE_BYTES, stream);
}

int msco_transpose_2d(const void *src, void *dst, int64_t batch, int64_t rows, int64_t cols, int32_t elem_bytes,
                      void *stream) {
  if (batch < 0 || rows < 0 || cols < 0 || batch > 65535) return MSCO_ERR_SHAPE;
  if (batch * rows * cols == 0) return MSCO_OK;
  if (src == nullptr || dst == nullptr) return MSCO_ERR_INVALID_ARG;
  if (elem_bytes != 1 && elem_bytes != 2 && elem_bytes != 4) return MSCO_ERR_UNSUPPORTED;
  const hipError_t err =
    launch_transpose_2d(src, dst, batch, rows, cols, elem_bytes, static_cast<hipStream_t>(stream));
  return err == hipSuccess ? MSCO_OK : MSCO_ERR_DEVICE;
}

size_t msco_packed_weight_bytes(int64_t k, int64_t n) {
  if (k <= 0 || n <= 0) return 0;
  return packed_weight_bytes(k, n);
}

int msco_pack_weight(const void *src, void *dst, int64_t e, int64_t k, int64_t n, int32_t src_transposed, void *stream) {
  if (e < 0 || k < 0 || n < 0 || k > INT32_MAX || n > INT32_MAX) return MSCO_ERR_SHAPE;
  if (e * k * n == 0) return MSCO_OK;
  if (src == nullptr || dst == nullptr) return MSCO_ERR_INVALID_ARG;
  if ((e * (int64_t)(packed_weight_bytes(k, n) / 16) + 255) / 256 > 0x7FFFFFFFll) return MSCO_ERR_SHAPE;
  const hipError_t err = launch_pack_weight(src, dst, e, k, n, src_transposed != 0, static_cast<hipStream_t>(stream));
  return err == hipSuccess ? MSCO_OK : MSCO_ERR_DEVICE;
}

int msco_gmm_destroy(msco_gmm_handle h) {
  if (h == nullptr) return MSCO_ERR_INVALID_ARG;
  {
    const RelaxedCapture relaxed;
    free_counters(h);
  }
  delete h;
  return MSCO_OK;
}

}  // extern "C"
