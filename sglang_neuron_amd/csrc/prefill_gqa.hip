// Segmented prefill attention over the paged pool (GQA, FP8 K/V with per-KV-head scales): a chunk's queries attend
// to their request's prior and, causally, to the chunk itself, all read from the pool (the chunk's K/V are stored
// before the attention runs), optionally inside a sliding window and with a sink logit per head.
//   reference: segmented_attention / _torch_segmented_attention (ops/attention/attention_segmented_cte.py:21-75)
//
// Work: one workgroup of 4 waves per (request, block of query tokens, KV head), dealt to the XCDs in contiguous runs
// so the blocks that read one request's keys of a KV head share an L2 (the DMAs keep the default cache policy for
// those rereads). Its 128 query rows are (token, head) pairs, token-major (row = t * group + j for the group's query
// head j); wave w owns rows 32 w .. 32 w + 31, one 32-column MFMA tile. Keys run in tiles of 64 positions from the
// window's first key to the block's last query, two sub-tiles of 32 each. A tile's K and V rows are DMA'd into a 2-slot
// LDS ring shared by the 4 waves, wave w loading the tile's 16-key group w (a group lies in one page, so its address is
// scalar work). The block-table entries of the key range are staged in LDS first.
//
// Where the query blocks alone leave CUs idle (a short chunk after a long prior) the keys are split on the device
// (prefill_item) and a second launch merges the partials: two turns of 150 and 251 tokens after 9000 and 17000 (32 / 8
// heads, bf16) 322 us whole, 116 split (512 workgroups; with 384 and 256 a fifth and four fifths longer); 16 tokens after
// 30000 (FP8) 469 and 47; 64 after 3000, 56 and 26. The search and the merge launch cost 5-6 us where the device's
// lengths leave nothing to split (8 requests of 100 tokens after 4000, bf16: 84 us unsplit, 90 here).
//
// Lane roles (lane = 32 g2 + i), per sub-tile of 32 keys:
//   QK  S^T[key, row] = K[key, :] . Q[row, :]: lane (g2, i) feeds A row i, the key whose index swaps bits 2 and 3 of i.
//       FP8: 32 of its bytes per 64 dims straight from LDS into v_mfma_scale_f32_32x32x64_f8f6f4 against the query's two
//       exact e4m3fn parts (below); bf16: 8 elements per 16 dims into v_mfma_f32_32x32x16_bf16. The result hands lane
//       (g2, i) keys 16 s + 8 g2 + j (s < 2, j < 8) of row i: with that key order, exactly the PV operand of its row.
//   PV  O^T[dim, row] += V^T[dim, key] . P^T[key, row] per 32-dim tile c and 16 keys (v_mfma_f32_32x32x16_bf16): lane
//       (g2, i) supplies its own probabilities and V^T's values of keys 8 g2 .. + 7 at dim 32 c + i through transposing
//       LDS reads of the ring's V rows: FP8, one ds_read_b64_tr_b8 converted in registers; bf16, two ds_read_b64_tr_b16.
//   acc lane (g2, i) holds row i at dims 32 c + 8 q + 4 g2 + r.
// Online softmax in the log2 domain with a lazily moved reference maximum (as the decode kernels). Keys that no row
// of the block may see (past the chunk, or on an invalid page) have their V rows zeroed in LDS, so stale pool bytes
// cannot reach the output through p = 0.
//
// What bounds it: the matrix cores under the card's power limit. On four requests of 2048 tokens after 2048 (32 / 8
// heads of 128, FP8) the clock settles near 1.87 GHz and the matrix pipe is busy 57% of the cycles; without the QK
// products the launch took 278 us, without PV's 316, without the exponentials 348, against 380 us then; alone in graph
// replays it takes 350-380 us (1.09-1.18 PFLOP/s; a large bf16 GEMM reaches 1.38 on the same card). Steps of this form,
// from 432 us: whole-row swizzled DMAs and masks only in boundary tiles (VALU per tile and wave 307 -> 205) 388; the 32
// x 32 shapes 388 (half the matrix instructions, the same time); the next tile's QK beside this tile's softmax 380. bf16
// pools, the same batch: 571 -> 418 us (now 400-417), V^T straight from the ring instead of through a shared bf16 copy.
// Head dim 64 (8 heads on one, FP8, sinks): 112 -> 93 us.

#include <algorithm>
#include <type_traits>

#include "sna_device.h"
#include "sna_host.h"

namespace sna {

struct PrefillArgs {
  const uint16_t* q;       // [T, H, D] bf16
  const uint8_t* k_cache;  // [num_blocks, G, P, D] e4m3fn
  const uint8_t* v_cache;
  const float* k_scale;  // [G] dequantization scales, or (mul_scale) GPT-OSS multipliers m: a byte is worth byte / m
  const float* v_scale;
  bool mul_scale;
  const int32_t* table;  // [R, table_width] (row stride table_stride)
  int64_t table_stride;
  int32_t table_width;
  const int32_t* q_start;  // [R + 1] the requests' first rows in q
  const int32_t* prior;    // [R] prior tokens of each request
  const float* sinks;      // [H] natural-log sink logits, or null
  uint16_t* out;           // [T, H, D] bf16
  int32_t R, H, G, P, group, bq;  // bq: query tokens per workgroup (128 / group)
  int32_t group_magic;            // ceil(2^16 / group): row / group = row * magic >> 16 for a block's rows (< 128)
  int64_t num_blocks;
  float sm_scale;
  int32_t window;
  // a launch that splits the keys (SPLIT): see prefill_item
  int32_t qblocks;   // query blocks of the longest chunk (max_q_len)
  int32_t slots;     // workgroups of the launch: the items it may run
  int32_t min_tiles; // least key tiles of a split
  float* ws_o;       // [slots, 128, D] unnormalized partials
  float* ws_ml;      // [slots, 128, 2] reference max (log2 domain) and softmax sum
  int2* ws_item;     // [G, R, qblocks] a query block's first item and its split count
};

constexpr int kPrefillTile = 64;   // keys per tile
constexpr int kPrefillRows = 128;  // query rows of a workgroup
// the most (request, query block) pairs of a split launch: 4 a lane of one wave
constexpr int kPrefillSplitPairs = 256;

// A split launch's workgroups (two a CU), the most query blocks of a launch that splits (one a CU), the least tiles a
// split takes, and the most tiles of a block that is never split (less than its partials and the merge pass cost).
constexpr int kPrefillSlots = 512;
constexpr int kPrefillSplitBlocks = 256;
constexpr int kPrefillMinSplit = 8;
constexpr int kPrefillNoSplit = 16;
// The most tiles of a query block of a launch that splits (prefill_item's exact divisions hold below 2^17): a table that
// can name more keys runs unsplit, which reads any length.
constexpr int kPrefillSplitMaxTiles = (1 << 17) - 1;

template <int D, int ESZ>  // ESZ: bytes per K/V element (1: e4m3fn, 2: bf16)
struct PrefillGeo {
  static constexpr int TK = kPrefillTile;        // keys per tile: NSUB sub-tiles of 32
  static constexpr int NSUB = TK / 32;
  static constexpr int ROWB = D * ESZ;           // bytes of a K or V row
  static constexpr int CH = ROWB / 16;           // 16-byte chunks of a row
  static constexpr int HALF = TK * ROWB;         // the K (or V) rows of a tile
  static constexpr int SLOT = 2 * HALF;          // one ring slot: K then V
  static constexpr int RPD = 1024 / ROWB;        // rows one wave-wide DMA fills
  static constexpr int MW = 16 / RPD;            // a wave's DMAs of K (and of V) per tile: its 16-key group
  static constexpr int PAGES = 2048;             // block-table entries staged in LDS at a time
  // A row's chunks sit XOR-swizzled in LDS (chunk c of tile row r at position c ^ swz(r)), so that the QK reads (16 keys
  // differing in row bits 0-3, one chunk) and the transposing PV reads (a half wave: FP8 8 rows x 2 chunks, bf16 4 rows
  // x 4 chunks) each touch every bank once, without padding: a DMA then fills whole rows of one 16-key group.
  static __device__ __forceinline__ int swz(int r) {
    const int b0 = r & 1, b1 = r >> 1 & 1, b2 = r >> 2 & 1, b3 = r >> 3 & 1;
    if (CH == 16) return b0 << 2 | b1 << 3 | b2 | b3 << 1;
    if (CH == 8 && ESZ == 2) return b1 << 2 | b2 | b3 << 1;
    if (CH == 8) return b1 << 1 | b2 << 2 | b3;
    return b3 | b2 << 1;
  }
};

constexpr float kPrefillRescaleSlack = 8.0f;

// One query block's keys: its queries are q0 .. q0 + nq - 1 of the request's chunk, at positions pos0 .. hi - 1, and it
// reads keys [lo, hi) in tiles [t0, t1). nq = 0: no such block (bx past the chunk).
struct PrefillBlock {
  int32_t q0, nq, pos0, lo, hi, t0, t1;
};
__device__ __forceinline__ PrefillBlock prefill_block(const PrefillArgs& a, int32_t S, int32_t prior, int32_t bx) {
  PrefillBlock b;
  const int32_t nqb = (S + a.bq - 1) / a.bq;
  b.q0 = (nqb - 1 - bx) * a.bq;  // the blocks with the most keys start first
  b.nq = bx < nqb ? min(a.bq, S - b.q0) : 0;
  b.pos0 = prior + b.q0;
  b.hi = b.pos0 + b.nq;
  b.lo = a.window > 0 ? max(0, b.pos0 - a.window + 1) : 0;
  b.t0 = b.lo / kPrefillTile;
  b.t1 = (b.hi + kPrefillTile - 1) / kPrefillTile;
  return b;
}

// The item w of a workgroup of a launch that splits the keys. Every (request, query block, KV head) is cut into splits
// of st tiles, st the least size (at least min_tiles) whose items fit the launch's workgroups; the pairs' tile counts
// come from the device's lengths, 4 a lane in registers, and every wave computes the same st and item. The split is
// dropped (st the longest block) where it would not pay (fitted at head dim 128 and 256 CUs): a tile takes about 1.3 us
// up to one workgroup a CU and 2 us with two (the card's power limit holds the chip to some 270 tiles a microsecond),
// the partials of 32 items 1 us of the launch and the merge pass 5 us. w numbers the items KV head by KV head, then pair
// by pair (request-major), a pair's splits in order. Every lane gets the same values; false past the last item.
__device__ bool prefill_item(const PrefillArgs& a, int32_t& w, int32_t& g, int32_t& r, int32_t& bx, int32_t& split,
                             int32_t& st_out, int32_t& ns) {
  constexpr int N = kPrefillSplitPairs / 64;
  const int lane = threadIdx.x & 63;
  const int32_t pairs = a.R * a.qblocks;
  const float rq = 1.0f / (float)a.qblocks;
  int32_t tiles[N];
  int32_t lane_total = 0, lane_max = 0;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    tiles[i] = 0;
    if (64 * i < pairs) {  // uniform
      const int32_t p = lane + 64 * i;
      if (p < pairs) {
        const int32_t rr = div_small(p, a.qblocks, rq);
        const int32_t S = a.q_start[rr + 1] - a.q_start[rr];
        const PrefillBlock b = prefill_block(a, S, a.prior[rr], p - rr * a.qblocks);
        // A block with queries has an item, and no length the device may hold makes more than the workspace's: its tiles
        // are held to the launch's bound (past the table's keys all are invalid) and, for a negative prior, from below
        // (such a block's item runs no tile, as the unsplit kernel's).
        tiles[i] = b.nq > 0 ? max(1, min(b.t1 - b.t0, kPrefillSplitMaxTiles)) : 0;
      }
      lane_total += tiles[i];
      lane_max = max(lane_max, tiles[i]);
    }
  }
  int32_t total;
  wave_incl_scan_i32(lane_total, &total);
  const int32_t mx = wave_max_nonneg_i32(lane_max);
  const int32_t items = a.slots / a.G;  // per KV head
  int32_t lo = max(a.min_tiles, (total + items - 1) / items), hi = max(lo, mx);
  while (lo < hi) {  // uniform
    const uint32_t mid = (uint32_t)((lo + hi) >> 1);
    const float rmid = 1.0f / (float)mid;
    int32_t lane_n = 0;
#pragma unroll
    for (int i = 0; i < N; ++i)
      if (64 * i < pairs) lane_n += (int32_t)ceil_div_small(tiles[i], mid, rmid);
    int32_t n;
    wave_incl_scan_i32(lane_n, &n);
    if (n <= items) hi = (int32_t)mid;
    else lo = (int32_t)mid + 1;
  }
  uint32_t st = (uint32_t)__builtin_amdgcn_readfirstlane(lo);
  float rst = 1.0f / (float)st;
  int32_t per_head = 0, blocks = 0;
#pragma unroll
  for (int i = 0; i < N; ++i)
    if (64 * i < pairs) {
      int32_t part;
      wave_incl_scan_i32((int32_t)ceil_div_small(tiles[i], st, rst), &part);
      per_head += part;
      blocks += __popcll(__ballot(tiles[i] > 0));
    }
  // tenths of a microsecond, in 64 bits
  const int64_t whole = (int64_t)mx * 13;  // (at most one block a CU)
  const int64_t cut = (int64_t)st * (per_head * a.G > kPrefillSlots / 2 ? 20 : 13) + 50 + per_head * a.G * 10 / 32;
  if (cut >= whole) {
    st = (uint32_t)max(mx, 1), rst = 1.0f / (float)st;
    per_head = blocks;
  }
  st_out = (int32_t)st;
  const int32_t n_items = per_head * a.G;
  if ((int32_t)blockIdx.x >= n_items) return false;
  // XCD-aware order over the items there are, so they spread over the XCDs whatever the grid
  w = (int32_t)xcd_order(blockIdx.x, n_items);
  g = w / per_head;
  const int32_t v = w - g * per_head;
  int32_t base = 0;
  bool found = false;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    if (64 * i < pairs && !found) {  // uniform
      const int32_t n = (int32_t)ceil_div_small(tiles[i], st, rst);
      int32_t part;
      const int32_t incl = wave_incl_scan_i32(n, &part);
      if (v < base + part) {
        const int32_t excl = incl - n;
        const uint64_t mine = __ballot(v >= base + excl && v < base + incl);
        const int32_t src = (int32_t)__builtin_amdgcn_readfirstlane(__ffsll((long long)mine) - 1);
        const int32_t p = 64 * i + src;
        r = p / a.qblocks;
        bx = p - r * a.qblocks;
        split = v - base - __builtin_amdgcn_readlane(excl, src);
        ns = __builtin_amdgcn_readlane(n, src);
        found = true;
      }
      base += part;
    }
  }
  return found;
}

// kOneTile and kHalfTile: the launch's tables name at most one tile of keys, or 32 of them (prompts of up to 64 or 32
// tokens with no prior), so the loop's next tile, whose products it computes whether there is one or not, and the tile's
// second sub-tile are left out (32 / 8 heads of 128, FP8 / bf16, us: 16 tokens 8.2 / 7.6 through the loop, 6.9 / 6.2 so;
// 60 tokens 9.0 / 8.4 and 8.7 / 8.0; as runtime branches of one kernel 7.8 / 7.4 and 9.1 / 9.0).
enum PrefillMode { kWhole, kSplit, kOneTile, kHalfTile };
template <int D, int ESZ, PrefillMode MODE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2)))
void prefill_gqa_kernel(PrefillArgs a) {
  using Geo = PrefillGeo<D, ESZ>;
  constexpr int ROWB = Geo::ROWB, CH = Geo::CH, HALF = Geo::HALF, SLOT = Geo::SLOT;
  constexpr bool ONE = MODE == kOneTile || MODE == kHalfTile;
  constexpr int TK = MODE == kHalfTile ? Geo::TK / 2 : Geo::TK, NSUB = TK / 32;
  constexpr int MW = Geo::MW, RPD = Geo::RPD;
  constexpr bool FP8 = ESZ == 1, SPLIT = MODE == kSplit;
  constexpr int NS = FP8 ? D / 64 : D / 16;  // QK steps
  constexpr int NC = D / 32;                 // PV dim tiles
  typedef __attribute__((address_space(3))) void lds_void;
  typedef __attribute__((address_space(3))) uint8_t lds_u8;
  __shared__ __attribute__((aligned(1024))) uint8_t sm_ring[2 * SLOT];
  __shared__ int32_t sm_pages[Geo::PAGES];

  const int tid = threadIdx.x, lane = tid & 63, g2 = lane >> 5, i32 = lane & 31, li = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int32_t bx, r, g, split = 0, split_tiles = 0, ns = 1, item = 0, note = -1;
  if constexpr (SPLIT) {
    // the same in every lane: made scalar, so what is addressed with them stays in scalar registers
    if (!__builtin_amdgcn_readfirstlane((int)prefill_item(a, item, g, r, bx, split, split_tiles, ns))) return;
    g = __builtin_amdgcn_readfirstlane(g), r = __builtin_amdgcn_readfirstlane(r);
    bx = __builtin_amdgcn_readfirstlane(bx), split = __builtin_amdgcn_readfirstlane(split);
    split_tiles = __builtin_amdgcn_readfirstlane(split_tiles), ns = __builtin_amdgcn_readfirstlane(ns);
    if (split == 0) note = (g * a.R + r) * a.qblocks + bx;  // (ws_item's entry of the block)
  } else {
    // XCD-aware order: each XCD takes a contiguous run of the (query block, request, KV head) order, so the query
    // blocks that read the same request's keys of one KV head share that XCD's L2
    const uint32_t lin = xcd_order(blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z),
                                   gridDim.x * gridDim.y * gridDim.z);
    bx = (int32_t)(lin % gridDim.x);
    r = (int32_t)((lin / gridDim.x) % gridDim.y), g = (int32_t)(lin / (gridDim.x * gridDim.y));
  }
  const int32_t qa = a.q_start[r];
  const PrefillBlock blk = prefill_block(a, a.q_start[r + 1] - qa, a.prior[r], bx);
  if (blk.nq <= 0) return;
  const int32_t nq = blk.nq, pos0 = blk.pos0, hi = blk.hi;

  // ---- this lane's row: token, head, position, and the query operand ----
  // (a row past the block computes as its last token and is not written)
  auto token_of = [&](int32_t row) -> int32_t { return row * a.group_magic >> 16; };
  auto head_of = [&](int32_t row) -> int32_t { return g * a.group + row - token_of(row) * a.group; };
  auto q_offset = [&](int32_t row) -> int64_t {
    return ((int64_t)(qa + blk.q0 + min(token_of(row), nq - 1)) * a.H + head_of(row)) * D;
  };
  const int32_t qpos = pos0 + min(token_of(32 * wave + i32), nq - 1);
  // The query operand of the FP8 QK: in step s lane (g2, i) supplies dims 64 s + 32 g2 .. + 31 of row i, the bf16 values
  // scaled by a power of two sc (the row's absolute maximum into [128, 256)) and split exactly into two e4m3fn parts,
  // hi + lo / 16 (hi keeps the top 4 significant bits, lo the next 4). The MFMA's E8M0 B scales undo sc (and the 1/16 of
  // lo), so K . Q is the exact bf16 dot product accumulated in fp32.
  // A bf16 pool instead takes the bf16 query elements 16 s + 8 g2 .. + 7 for v_mfma_f32_32x32x16_bf16 (qf).
  uint32_t qhi[FP8 ? NS : 1][8], qlo[FP8 ? NS : 1][8];
  int32_t qsc_hi = 0, qsc_lo = 0;
  uint32_t qf[FP8 ? 1 : NS][4];
  const uint16_t* qrow = a.q + q_offset(32 * wave + i32);
  if constexpr (!FP8) {
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const uint4 w = ld16(qrow + 16 * s + 8 * g2);
      qf[s][0] = w.x, qf[s][1] = w.y, qf[s][2] = w.z, qf[s][3] = w.w;
    }
  } else {
    float v[NS][32];
    float amax = 0.0f;
#pragma unroll
    for (int s = 0; s < NS; ++s)
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const uint4 w = ld16(qrow + 64 * s + 32 * g2 + 8 * c);
        const uint32_t ww[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          v[s][8 * c + 2 * e] = bf16_bits_to_f32(ww[e] & 0xffffu);
          v[s][8 * c + 2 * e + 1] = bf16_bits_to_f32(ww[e] >> 16);
        }
      }
#pragma unroll
    for (int s = 0; s < NS; ++s)
#pragma unroll
      for (int e = 0; e < 32; ++e) amax = fmaxf(amax, fabsf(v[s][e]));
    amax = xor32_partner_max(amax);
    // sc = 2^(7 - floor(log2 amax)): amax * sc in [128, 256); E8M0 scale of hi = 127 - log2 sc, of lo 4 less
    // (the exponent is held to [-116, 127], where sc and both E8M0 scales are representable; a row that small only
    // loses bits far below the tolerance)
    const int32_t ex = amax > 0.0f ? max((int32_t)((__float_as_uint(amax) >> 23) & 0xff) - 127, -116) : -7;
    const float sc = __uint_as_float((uint32_t)(127 + 7 - ex) << 23);
    qsc_hi = 127 + ex - 7;
    qsc_lo = 127 + ex - 7 - 4;
#pragma unroll
    for (int s = 0; s < NS; ++s)
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        float h4[4], l4[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) split_q(v[s][4 * k + e] * sc, h4[e], l4[e]);
        qhi[s][k] = pack_e4m3fn_x4(h4[0], h4[1], h4[2], h4[3]);
        qlo[s][k] = pack_e4m3fn_x4(l4[0], l4[1], l4[2], l4[3]);
      }
  }
  const float k_deq = FP8 ? (a.mul_scale ? 1.0f / a.k_scale[g] : a.k_scale[g]) : 1.0f;
  const float qk_scale = a.sm_scale * kLog2e * k_deq;
  const float v_scale = FP8 ? (a.mul_scale ? 1.0f / a.v_scale[g] : a.v_scale[g]) : 1.0f;

  float m_ref = 0.0f, l_run = 0.0f;
  f32x16_t acc[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[c][e] = 0.0f;

  const uint32_t ring = lds_address((lds_void*)(lds_u8*)&sm_ring[0]);
  const int64_t head_stride = (int64_t)a.P * ROWB;  // bytes between KV heads of one page
  const int64_t page_stride = head_stride * a.G;
  const uint8_t* kg = a.k_cache + g * head_stride;
  const uint8_t* vg = a.v_cache + g * head_stride;

  int32_t p0 = 0;  // first page index staged in sm_pages
  const bool p_pow2 = (a.P & (a.P - 1)) == 0;  // uniform: the page column of a key is a shift
  const int p_shift = __builtin_ctz((uint32_t)a.P);
  // A tile is four 16-key groups, each inside one page; wave w loads group w, RPD rows a DMA: DMA m's lane fills chunk
  // position lane % CH of group row RPD m + lane / CH, with the row's chunk that the swizzle puts there.
  uint32_t dma_off[MW];
#pragma unroll
  for (int m = 0; m < MW; ++m) {
    const int grow = RPD * m + lane / CH;
    dma_off[m] = (uint32_t)(grow * ROWB + 16 * ((lane % CH) ^ Geo::swz(grow)));
  }
  auto column = [&](int32_t key) -> int32_t { return p_pow2 ? key >> p_shift : key / a.P; };
  // lane u's 16-key group's page of tile t (-1: invalid), lanes past the tile's groups repeating its last
  auto page_of = [&](int32_t t) -> int32_t { return sm_pages[column(TK * t + 16 * min(lane, TK / 16 - 1)) - p0]; };
  // Whether each group's page is valid (bit u; pg: page_of(t)), and this wave's group's byte offset in the caches.
  auto pages_ok = [&](int32_t pg) -> uint32_t { return (uint32_t)__ballot(pg >= 0) & ((1u << (TK / 16)) - 1u); };
  auto group_off = [&](int32_t t, int32_t pg) -> int64_t {
    const int32_t mypg = max((int32_t)__builtin_amdgcn_readlane(pg, wave), 0);
    const int32_t key = TK * t + 16 * wave;
    return (int64_t)mypg * page_stride + (int64_t)(key - column(key) * a.P) * ROWB;
  };
  auto load = [&](const uint8_t* base, uint32_t lds) {
#pragma unroll
    for (int m = 0; m < MW; ++m) dma_saddr16_cached(base, dma_off[m], lds + wave * 16 * ROWB + 1024 * m);
  };

  // LDS read addresses in a slot. QK: lane i feeds A row i, the key whose row swaps bits 2 and 3 of i (+ 32 u by the
  // immediate offset); step s XORs the chunk.
  const int k_row = (i32 & 19) | (i32 >> 1 & 4) | (i32 << 1 & 8);
  const uint32_t k_at = (uint32_t)(k_row * ROWB + 16 * ((FP8 ? 2 * g2 : g2) ^ Geo::swz(k_row)));
  // PV: FP8 row 8 g2 + li / 2, its 8 bytes li % 2 of the 16-byte half (lane / 16) % 2 of a 32-byte dim tile; bf16 rows
  // 8 g2 + li / 4 and + 4, the 8 bytes li % 4 of the 32-byte half of a 64-byte dim tile. Dim tile c XORs 32 c (64 c).
  uint32_t v_at[FP8 ? 1 : 2];
#pragma unroll
  for (int hh = 0; hh < (FP8 ? 1 : 2); ++hh) {
    const int v_row = 8 * g2 + (FP8 ? li >> 1 : 4 * hh + (li >> 2)), dh = lane >> 4 & 1;
    const int ch = FP8 ? dh : 2 * dh + (li >> 1 & 1);
    v_at[hh] = (uint32_t)(HALF + v_row * ROWB + 16 * (ch ^ Geo::swz(v_row)) + 8 * (li & 1));
  }

  // S^T of a slot's keys, in sub-tiles of 32: element 8 s + j is key k0 + 32 u + 16 s + 8 g2 + j of the lane's row
  auto qk = [&](const uint8_t* S0, f32x16_t (&st)[NSUB]) {
#pragma unroll
    for (int u = 0; u < NSUB; ++u)
#pragma unroll
      for (int e = 0; e < 16; ++e) st[u][e] = 0.0f;
    if constexpr (!FP8) {
#pragma unroll
      for (int s = 0; s < NS; ++s)
#pragma unroll
        for (int u = 0; u < NSUB; ++u) {
          const uint4 w = *reinterpret_cast<const uint4*>(S0 + 32 * u * ROWB + (k_at ^ (32 * s)));
          const uint32_t kop[4] = {w.x, w.y, w.z, w.w};
          st[u] = mfma_32x32x16_bf16(kop, qf[s], st[u]);
        }
    } else {
      // the K bytes of the lane's key and dims straight from LDS (e4m3fn, no conversion)
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        uint32_t kop[NSUB][8];
#pragma unroll
        for (int u = 0; u < NSUB; ++u) {
          const uint4 w0 = *reinterpret_cast<const uint4*>(S0 + 32 * u * ROWB + (k_at ^ (64 * s)));
          const uint4 w1 = *reinterpret_cast<const uint4*>(S0 + 32 * u * ROWB + (k_at ^ (64 * s + 16)));
          kop[u][0] = w0.x, kop[u][1] = w0.y, kop[u][2] = w0.z, kop[u][3] = w0.w;
          kop[u][4] = w1.x, kop[u][5] = w1.y, kop[u][6] = w1.z, kop[u][7] = w1.w;
        }
#pragma unroll
        for (int u = 0; u < NSUB; ++u) st[u] = mfma_32x32x64_fp8(kop[u], qhi[s], st[u], qsc_hi);
#pragma unroll
        for (int u = 0; u < NSUB; ++u) st[u] = mfma_32x32x64_fp8(kop[u], qlo[s], st[u], qsc_lo);
      }
    }
  };
  // The exponents of a tile's raw scores relative to the row's reference maximum (log2 domain), in place, and the lane's
  // largest.
  float mx = -INFINITY;
  auto exponents = [&](f32x16_t (&y)[NSUB]) {
    mx = -INFINITY;
#pragma unroll
    for (int u = 0; u < NSUB; ++u)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        y[u][e] = fmaf(y[u][e], qk_scale, -m_ref);
        mx = fmaxf(mx, y[u][e]);
      }
  };
  auto mask = [&](int32_t k0, uint32_t pg_ok, f32x16_t (&y)[NSUB]) {
    // (no position is below 0, so neither is a window's first key: `first` does not leave 32 bits for any window)
    const int32_t last = qpos - 8 * g2, first = a.window > 0 ? max(qpos - a.window + 1, 0) - 8 * g2 : INT32_MIN;
    mx = -INFINITY;
#pragma unroll
    for (int u = 0; u < NSUB; ++u)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const bool page_ok = (pg_ok >> (2 * u + e / 8)) & 1u;  // uniform
        const int32_t key = k0 + 32 * u + 16 * (e / 8) + e % 8;  // less 8 g2
        y[u][e] = (page_ok & (key <= last) & (key >= first)) ? y[u][e] : -INFINITY;
        mx = fmaxf(mx, y[u][e]);
      }
  };
  // The reference moves to the row's maximum when that passes it by the slack; a row that has seen no key yet (its
  // reference 0 stands for none) takes its first maximum, whatever it is.
  bool unset = true, any_unset = true;  // this lane's row; any row of the wave (uniform)
  auto move_reference = [&](f32x16_t (&y)[NSUB]) {
    const float tmax = xor32_partner_max(mx);
    const float d = tmax > (unset ? -INFINITY : kPrefillRescaleSlack) ? tmax : 0.0f;
    const float alpha = unset ? 1.0f : __builtin_amdgcn_exp2f(-d);
    m_ref += d;
    unset = unset && !(tmax > -INFINITY);
    any_unset = __any(unset);
    l_run *= alpha;
#pragma unroll
    for (int c = 0; c < NC; ++c) acc[c] *= alpha;
#pragma unroll
    for (int u = 0; u < NSUB; ++u)
#pragma unroll
      for (int e = 0; e < 16; ++e) y[u][e] -= d;
  };
  // The probabilities, packed as the PV operand, and their sum (of the bf16 values the numerator weighs: v_dot2 with a
  // pair of ones).
  uint32_t pop[NSUB][2][4];
  auto probabilities = [&](const f32x16_t (&y)[NSUB]) {
#pragma unroll
    for (int u = 0; u < NSUB; ++u)
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const uint32_t w = pack_bf16x2(__builtin_amdgcn_exp2f(y[u][2 * k]), __builtin_amdgcn_exp2f(y[u][2 * k + 1]));
        pop[u][k / 4][k % 4] = w;
        l_run = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, w),
                                                __builtin_bit_cast(bf16x2_t, 0x3f803f80u), l_run, false);
      }
  };
  auto pv = [&](const uint8_t* S0) {
#pragma unroll
    for (int u = 0; u < NSUB; ++u)
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const uint8_t* V0 = S0 + (32 * u + 16 * s) * ROWB;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          uint32_t vop[4];
          if constexpr (FP8) {
            const uint2 w = lds_read_tr8(V0 + (v_at[0] ^ (32 * c)));
            fp8x4_to_bf16x4(w.x, vop[0], vop[1]);
            fp8x4_to_bf16x4(w.y, vop[2], vop[3]);
          } else {
            const uint2 w0 = lds_read_tr16(V0 + (v_at[0] ^ (64 * c)));
            const uint2 w1 = lds_read_tr16(V0 + (v_at[FP8 ? 0 : 1] ^ (64 * c)));
            vop[0] = w0.x, vop[1] = w0.y, vop[2] = w1.x, vop[3] = w1.y;
          }
          acc[c] = mfma_32x32x16_bf16(vop, pop[u][s], acc[c]);
        }
      }
  };

  // The compiler's own loads (the query operand) complete here, in a wait it sees, before any DMA is in flight.
  __builtin_amdgcn_s_waitcnt(0x0f70);

  const int32_t t_first = blk.t0 + (SPLIT ? split * split_tiles : 0);
  // (ONE: a length past the table has only invalid keys in its other tiles)
  const int32_t t_end = SPLIT ? min(blk.t1, t_first + split_tiles) : ONE ? min(blk.t1, t_first + 1) : blk.t1;
  const int32_t chunk_tiles = (Geo::PAGES - 1) * a.P / TK;  // (a chunk may start mid-page: PAGES - 1 whole pages)
  for (int32_t c0 = t_first; c0 < t_end; c0 += chunk_tiles) {
    const int32_t c1 = min(c0 + chunk_tiles, t_end);
    // stage the table entries of pages [p0, p1) (ring and pages are free: the previous chunk drained)
    __syncthreads();
    p0 = TK * c0 / a.P;
    const int32_t p1 = (TK * c1 - 1) / a.P + 1;
    const int32_t* trow = a.table + (int64_t)r * a.table_stride;
    for (int32_t i = tid; i < p1 - p0; i += 256) {
      const int32_t col = p0 + i;
      const int32_t e = col < a.table_width ? trow[col] : -1;
      sm_pages[i] = (e >= 0 && (int64_t)e < a.num_blocks) ? e : -1;
    }
    __syncthreads();
    const int32_t n = c1 - c0;
    // The loop over tiles holds tile i's scores and computes tile i + 1's beside tile i's probabilities (the matrix
    // products of one, the vector work of the other, in one stretch of code), so K runs a tile ahead of V in the ring:
    // K of tile i + 2 loads into tile i's slot, V of tile i + 1 into its own, while tile i computes.
    int32_t pg = page_of(c0);
    uint32_t ok_cur = pages_ok(pg), ok_next;
    int64_t off = group_off(c0, pg);
    if (TK / 16 == 4 || wave < TK / 16) {
      load(kg + off, ring);
      load(vg + off, ring + HALF);
    }
    pg = page_of(min(c0 + 1, c1 - 1));
    ok_next = pages_ok(pg);
    off = group_off(min(c0 + 1, c1 - 1), pg);  // of tile i + 1
    if (n > 1) load(kg + off, ring + SLOT);
    pg = page_of(min(c0 + 2, c1 - 1));  // of tile i + 2, looked up a tile ahead
    wait_vmcnt<0>();
    __syncthreads();
    f32x16_t sa[NSUB], sb[NSUB];
    qk(&sm_ring[0], sa);
    exponents(sa);
    // tile i (in ring slot P) up to its exponents under the reference maximum: V cleaned, scores masked
    auto settle = [&](int32_t i, int P, f32x16_t (&cur)[NSUB]) {
      const int32_t k0 = TK * (c0 + i);
      const bool valid = ok_cur == (1u << (TK / 16)) - 1;
      if (!valid || k0 + TK > hi) {
        // keys no row of the block may see (past the chunk, or on an invalid page): their V rows are zeroed, so that
        // stale pool bytes (a NaN among them) cannot reach the output through p = 0
        for (int32_t o = tid; o < TK * CH; o += 256) {
          const int32_t vr = o / CH;
          if (k0 + vr >= hi || !((ok_cur >> (vr >> 4)) & 1u))
            *reinterpret_cast<uint4*>(&sm_ring[P * SLOT + HALF + 16 * o]) = make_uint4(0, 0, 0, 0);
        }
        __syncthreads();
      }
      // a tile that is not full (a key invalid or not visible to every row of the block) masks its scores
      if (!valid || k0 + TK - 1 > pos0 || (a.window != 0 && k0 <= hi - 1 - a.window)) mask(k0, ok_cur, cur);
      if (any_unset || __any(mx > kPrefillRescaleSlack)) move_reference(cur);
    };
    if constexpr (ONE) {
      settle(0, 0, sa);
      probabilities(sa);
      pv(&sm_ring[0]);
    } else {
      auto step = [&](int32_t i, auto parity, f32x16_t (&cur)[NSUB], f32x16_t (&next)[NSUB]) {
        constexpr int P = decltype(parity)::value;  // i % 2
        wait_vmcnt<0>();  // this wave's K of tile i + 1 and V of tile i have landed
        // every wave's have; every wave is done with K of tile i and V of tile i - 1 (their slots are free)
        __syncthreads();
        if (i + 1 < n) load(vg + off, ring + (1 - P) * SLOT + HALF);
        const uint32_t ok2 = pages_ok(pg);
        if (i + 2 < n) {
          off = group_off(c0 + i + 2, pg);
          load(kg + off, ring + P * SLOT);
          pg = page_of(min(c0 + i + 3, c1 - 1));
        }
        settle(i, P, cur);
        qk(&sm_ring[(1 - P) * SLOT], next);  // (past the last tile: whatever the slot holds, not used)
        probabilities(cur);
        pv(&sm_ring[P * SLOT]);
        exponents(next);
        // (a use here, so the compiler does not move the next tile's products past the loop's exit test)
        asm volatile("" : "+v"(mx), "+v"(next[0]), "+v"(next[1]));
        ok_cur = ok_next;
        ok_next = ok2;
      };
      for (int32_t i = 0;;) {
        step(i, std::integral_constant<int, 0>{}, sa, sb);
        if (++i >= n) break;
        step(i, std::integral_constant<int, 1>{}, sb, sa);
        if (++i >= n) break;
      }
    }
  }

  if (unset) m_ref = kNegBig;  // no key seen
  float L = xor32_partner_sum(l_run);
  // the row again, from a lane index the compiler takes for a new one, so that nothing of it is held over the loop
  int32_t row = 32 * wave + i32;
  asm volatile("" : "+v"(row));
  const bool row_ok = token_of(row) < nq;
  // Of a launch that splits, a block's first item and split count, written by the thread of its first row (always valid).
  // Last, and by an index made at the head: with a store to memory before the loop the compiler no longer takes the
  // lengths, scales and tables for unchanging, and with the block's three indices held over the loop it runs out of
  // registers; either way the loop waits for every LDS read by itself (a turn of 128-dim rows 1.1 times the unsplit
  // kernel's with FP8 and 1.35 times with bf16 pools: 8 requests of 100 tokens after 4000, 32 / 8 heads, 86 and 113 us,
  // so 80 and 90).
  auto note_item = [&]() {
    if (SPLIT && note >= 0 && tid == 0) a.ws_item[note] = make_int2(item, ns);
  };
  if (SPLIT && ns > 1) {  // this split's partial: the combine pass merges the block's splits
    if (!row_ok) return;
    float* wo = a.ws_o + ((int64_t)item * kPrefillRows + row) * D + 4 * g2;
    if (g2 == 0)
      *reinterpret_cast<float2*>(a.ws_ml + ((int64_t)item * kPrefillRows + row) * 2) = make_float2(m_ref, L);
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *reinterpret_cast<f32x4_t*>(wo + 32 * c + 8 * q) =
            f32x4_t{acc[c][4 * q], acc[c][4 * q + 1], acc[c][4 * q + 2], acc[c][4 * q + 3]};
    note_item();
    return;
  }
  // ---- epilogue: normalize (sinks join the denominator), scale by v_scale, write the valid rows ----
  if (a.sinks) L += __builtin_amdgcn_exp2f(a.sinks[head_of(row)] * kLog2e - m_ref);
  const float inv = v_scale / L;
  if (!row_ok) return;
  uint16_t* dst = a.out + q_offset(row) + 4 * g2;
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int q = 0; q < 4; ++q)
      *reinterpret_cast<uint2*>(dst + 32 * c + 8 * q) =
          make_uint2(pack_bf16x2(acc[c][4 * q] * inv, acc[c][4 * q + 1] * inv),
                     pack_bf16x2(acc[c][4 * q + 2] * inv, acc[c][4 * q + 3] * inv));
  note_item();
}

// Merge of the split query blocks, 1024 / D of a block's rows a workgroup: out = sum_s e_s o_s / (sum_s e_s l_s +
// e_sink) with e_s = exp2(m_s - M), M the largest m_s. D / 4 lanes a row, the loads of four splits in flight together.
template <int D>
__global__ __launch_bounds__(256) void prefill_combine_kernel(PrefillArgs a, bool fp8) {
  constexpr int LR = D / 4;  // lanes a row
  const int tid = threadIdx.x;
  constexpr int NP = kPrefillRows * LR / 256;  // workgroups a block
  const int32_t bx = blockIdx.x / NP, r = blockIdx.y, g = blockIdx.z;
  const int2 it = a.ws_item[((int64_t)g * a.R + r) * a.qblocks + bx];
  const int32_t qa = a.q_start[r];
  const PrefillBlock blk = prefill_block(a, a.q_start[r + 1] - qa, a.prior[r], bx);
  if (blk.nq <= 0 || it.y <= 1) return;  // no such block, or its one split wrote the output
  const float v_scale = fp8 ? (a.mul_scale ? 1.0f / a.v_scale[g] : a.v_scale[g]) : 1.0f;
  const int col = 4 * (tid % LR);
  const int row = 256 / LR * (blockIdx.x % NP) + tid / LR;
  const int32_t t = row * a.group_magic >> 16;
  if (t >= blk.nq) return;
  const int32_t head = g * a.group + row - t * a.group;
  const float* ml = a.ws_ml + ((int64_t)it.x * kPrefillRows + row) * 2;
  const float* wo = a.ws_o + ((int64_t)it.x * kPrefillRows + row) * D + col;
  float M = kNegBig;
  for (int32_t s = 0; s < it.y; ++s) M = fmaxf(M, ml[(int64_t)s * kPrefillRows * 2]);
  float den = a.sinks ? __builtin_amdgcn_exp2f(a.sinks[head] * kLog2e - M) : 0.0f;
  f32x4_t o = {0.f, 0.f, 0.f, 0.f};
  for (int32_t s0 = 0; s0 < it.y; s0 += 4) {
    f32x4_t x[4];
    float2 w[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int64_t s = min(s0 + k, it.y - 1);
      x[k] = *reinterpret_cast<const f32x4_t*>(wo + s * kPrefillRows * D);
      w[k] = *reinterpret_cast<const float2*>(ml + s * kPrefillRows * 2);
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float e = s0 + k < it.y ? __builtin_amdgcn_exp2f(w[k].x - M) : 0.0f;
      den += e * w[k].y;
      o += e * x[k];
    }
  }
  const float inv = v_scale / den;
  uint16_t* dst = a.out + ((int64_t)(qa + blk.q0 + t) * a.H + head) * D + col;
  *reinterpret_cast<uint2*>(dst) = make_uint2(pack_bf16x2(o[0] * inv, o[1] * inv), pack_bf16x2(o[2] * inv, o[3] * inv));
}

// The workgroups of a split launch: 0 where the launch's own query blocks are more than one a CU (they reach the rate
// that the power limit allows by themselves: 352 blocks of up to 136 tiles took 201 us whole, 206 in a split launch; 376
// of up to 24 tiles 36 and 42; requests of unequal lengths would gain, which the host does not know), too short (the
// search and the merge launch), or past what the split counts.
static int32_t prefill_split_slots(int64_t qblocks, int32_t R, int32_t G, int64_t bound_tiles) {
  const int64_t base = qblocks * R * G;
  if (base > kPrefillSplitBlocks || bound_tiles <= kPrefillNoSplit || bound_tiles > kPrefillSplitMaxTiles) return 0;
  static_assert(kPrefillSplitPairs >= kPrefillSplitBlocks, "a split launch's pairs fit a wave");
  return (int32_t)std::min<int64_t>(kPrefillSlots, base * ((bound_tiles + kPrefillMinSplit - 1) / kPrefillMinSplit));
}

}  // namespace sna

using namespace sna;

namespace {

// The key tiles a query block can span: its table's keys, inside a window the window's and the block's own.
int64_t prefill_bound_tiles(int32_t table_width, int32_t page_size, int32_t window, int32_t bq) {
  const int64_t keys = (int64_t)table_width * page_size;
  const int64_t span = window > 0 ? std::min<int64_t>(keys, (int64_t)window + bq + kPrefillTile) : keys;
  return (span + kPrefillTile - 1) / kPrefillTile;
}

int32_t split_slots_of(int32_t R, int32_t max_q_len, int32_t num_q_heads, int32_t num_kv_heads, int32_t page_size,
                       int32_t table_width, int32_t window) {
  const int32_t bq = kPrefillRows / (num_q_heads / num_kv_heads);
  const int64_t qblocks = ((int64_t)max_q_len + bq - 1) / bq;
  return prefill_split_slots(qblocks, R, num_kv_heads, prefill_bound_tiles(table_width, page_size, window, bq));
}

int64_t split_workspace_bytes(int32_t slots, int32_t R, int32_t max_q_len, int32_t num_q_heads, int32_t num_kv_heads,
                              int32_t head_dim) {
  const int32_t bq = kPrefillRows / (num_q_heads / num_kv_heads);
  const int64_t qblocks = ((int64_t)max_q_len + bq - 1) / bq;
  return (int64_t)slots * kPrefillRows * (head_dim + 2) * (int64_t)sizeof(float) +
         qblocks * R * num_kv_heads * (int64_t)sizeof(int2);
}

template <int D, int ESZ>
void launch_prefill(const PrefillArgs& a, hipStream_t s) {
  if (a.slots > 0) {
    hipLaunchKernelGGL((prefill_gqa_kernel<D, ESZ, kSplit>), dim3(a.slots), dim3(256), 0, s, a);
    hipLaunchKernelGGL((prefill_combine_kernel<D>), dim3(kPrefillRows * D / 1024 * a.qblocks, a.R, a.G),
                       dim3(256), 0, s, a, ESZ == 1);
  } else if ((int64_t)a.table_width * a.P <= kPrefillTile / 2) {
    hipLaunchKernelGGL((prefill_gqa_kernel<D, ESZ, kHalfTile>), dim3(a.qblocks, a.R, a.G), dim3(256), 0, s, a);
  } else if ((int64_t)a.table_width * a.P <= kPrefillTile) {
    hipLaunchKernelGGL((prefill_gqa_kernel<D, ESZ, kOneTile>), dim3(a.qblocks, a.R, a.G), dim3(256), 0, s, a);
  } else {
    hipLaunchKernelGGL((prefill_gqa_kernel<D, ESZ, kWhole>), dim3(a.qblocks, a.R, a.G), dim3(256), 0, s, a);
  }
}

}  // namespace

static int prefill_attention(const void* q, const void* k_cache, const void* v_cache, const float* k_scale,
                                     const float* v_scale, const int32_t* block_table, int64_t table_stride,
                                     int32_t table_width, const int32_t* q_start, const int32_t* prior_lens,
                                     int32_t R, int32_t max_q_len, const float* sinks, float sm_scale, int32_t window,
                                     void* out, int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim,
                                     int32_t page_size, int64_t num_blocks, int32_t kv_dtype, void* workspace,
                                     int64_t workspace_bytes, void* stream) {
  if (R < 0 || max_q_len < 0 || num_q_heads < 1 || num_kv_heads < 1 || num_q_heads % num_kv_heads != 0 ||
      window < 0 || num_blocks < 1 || table_width < 1 || table_stride < table_width)
    return fail(SNA_ERR_INVALID_ARGUMENT,
                "prefill_attention: bad sizes (R %d, max_q_len %d, heads %d / %d, window %d, blocks %lld, table %d "
                "wide, stride %lld)",
                R, max_q_len, num_q_heads, num_kv_heads, window, (long long)num_blocks, table_width,
                (long long)table_stride);
  const int32_t group = num_q_heads / num_kv_heads;
  if (group > 128) return fail(SNA_ERR_UNSUPPORTED, "prefill_attention: %d query heads per KV head (at most 128)", group);
  if (head_dim != 64 && head_dim != 128)
    return fail(SNA_ERR_UNSUPPORTED, "prefill_attention: head_dim %d (64 or 128)", head_dim);
  if (page_size < 16 || page_size % 16 != 0)
    return fail(SNA_ERR_UNSUPPORTED, "prefill_attention: page_size %d (a multiple of 16)", page_size);
  if (kv_dtype != SNA_DTYPE_FP8_E4M3FN && kv_dtype != SNA_DTYPE_FP8_E4M3FN_MUL && kv_dtype != SNA_DTYPE_BF16)
    return fail(SNA_ERR_UNSUPPORTED, "prefill_attention: KV dtype %d (FP8 e4m3fn or bf16)", kv_dtype);
  if (R == 0 || max_q_len == 0) return SNA_OK;
  if (!q || !k_cache || !v_cache || (kv_dtype != SNA_DTYPE_BF16 && (!k_scale || !v_scale)) || !block_table ||
      !q_start || !prior_lens || !out)
    return fail(SNA_ERR_INVALID_ARGUMENT, "prefill_attention: null pointer");
  if (!aligned(q, 16) || !aligned(out, 16) || !aligned(k_cache, 16) || !aligned(v_cache, 16))
    return fail(SNA_ERR_INVALID_ARGUMENT, "prefill_attention: q, out and the caches must be 16-byte aligned");
  if (R > 65535 || num_kv_heads > 65535)
    return fail(SNA_ERR_INVALID_ARGUMENT, "prefill_attention: %d requests x %d KV heads exceed the grid", R,
                num_kv_heads);
  PrefillArgs a;
  a.q = (const uint16_t*)q;
  a.k_cache = (const uint8_t*)k_cache;
  a.v_cache = (const uint8_t*)v_cache;
  a.k_scale = k_scale;
  a.v_scale = v_scale;
  a.mul_scale = kv_dtype == SNA_DTYPE_FP8_E4M3FN_MUL;
  a.table = block_table;
  a.table_stride = table_stride;
  a.table_width = table_width;
  a.q_start = q_start;
  a.prior = prior_lens;
  a.sinks = sinks;
  a.out = (uint16_t*)out;
  a.R = R;
  a.H = num_q_heads;
  a.G = num_kv_heads;
  a.P = page_size;
  a.group = group;
  a.bq = kPrefillRows / group;
  a.group_magic = (65536 + group - 1) / group;
  a.num_blocks = num_blocks;
  a.sm_scale = sm_scale;
  a.window = window;
  const int64_t qblocks = ((int64_t)max_q_len + a.bq - 1) / a.bq;
  if (qblocks * R * num_kv_heads > (int64_t)UINT32_MAX)  // the kernel's XCD-aware order numbers them in 32 bits
    return fail(SNA_ERR_INVALID_ARGUMENT, "prefill_attention: %lld query blocks x %d requests x %d KV heads exceed "
                "the grid (split the batch)", (long long)qblocks, R, num_kv_heads);
  a.qblocks = (int32_t)qblocks;
  a.min_tiles = kPrefillMinSplit;
  a.slots = 0;
  a.ws_o = a.ws_ml = nullptr;
  a.ws_item = nullptr;
  const int32_t slots = workspace ? split_slots_of(R, max_q_len, num_q_heads, num_kv_heads, page_size, table_width,
                                                   window) : 0;
  if (slots > 0) {
    const int64_t need = split_workspace_bytes(slots, R, max_q_len, num_q_heads, num_kv_heads, head_dim);
    if (workspace_bytes < need)
      return fail(SNA_ERR_WORKSPACE, "prefill_attention: workspace of %lld bytes, the split needs %lld",
                  (long long)workspace_bytes, (long long)need);
    if (!aligned(workspace, 16))
      return fail(SNA_ERR_INVALID_ARGUMENT, "prefill_attention: the workspace must be 16-byte aligned");
    a.slots = slots;
    a.ws_o = (float*)workspace;
    a.ws_ml = a.ws_o + (int64_t)slots * kPrefillRows * head_dim;
    a.ws_item = (int2*)(a.ws_ml + (int64_t)slots * kPrefillRows * 2);
  }
  const hipStream_t s = (hipStream_t)stream;
  if (kv_dtype != SNA_DTYPE_BF16) {
    if (head_dim == 128) launch_prefill<128, 1>(a, s); else launch_prefill<64, 1>(a, s);
  } else {
    if (head_dim == 128) launch_prefill<128, 2>(a, s); else launch_prefill<64, 2>(a, s);
  }
  return check_launch("prefill_attention");
}

extern "C" int sna_prefill_attention(const void* q, const void* k_cache, const void* v_cache, const float* k_scale,
                                     const float* v_scale, const int32_t* block_table, int64_t table_stride,
                                     int32_t table_width, const int32_t* q_start, const int32_t* prior_lens,
                                     int32_t R, int32_t max_q_len, const float* sinks, float sm_scale, int32_t window,
                                     void* out, int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim,
                                     int32_t page_size, int64_t num_blocks, int32_t kv_dtype, void* stream) {
  ApiGuard guard;
  return prefill_attention(q, k_cache, v_cache, k_scale, v_scale, block_table, table_stride, table_width, q_start,
                           prior_lens, R, max_q_len, sinks, sm_scale, window, out, num_q_heads, num_kv_heads, head_dim,
                           page_size, num_blocks, kv_dtype, nullptr, 0, stream);
}

extern "C" int64_t sna_prefill_workspace_bytes(int32_t R, int32_t max_q_len, int32_t num_q_heads, int32_t num_kv_heads,
                                               int32_t head_dim, int32_t page_size, int32_t table_width,
                                               int32_t window) {
  if (R < 1 || max_q_len < 1 || num_q_heads < 1 || num_kv_heads < 1 || num_q_heads % num_kv_heads != 0 ||
      num_q_heads / num_kv_heads > kPrefillRows || head_dim < 1 || page_size < 1 || table_width < 1 || window < 0)
    return 0;
  const int32_t slots = split_slots_of(R, max_q_len, num_q_heads, num_kv_heads, page_size, table_width, window);
  return slots > 0 ? split_workspace_bytes(slots, R, max_q_len, num_q_heads, num_kv_heads, head_dim) : 0;
}

extern "C" int sna_prefill_attention_split(const void* q, const void* k_cache, const void* v_cache,
                                           const float* k_scale, const float* v_scale, const int32_t* block_table,
                                           int64_t table_stride, int32_t table_width, const int32_t* q_start,
                                           const int32_t* prior_lens, int32_t R, int32_t max_q_len, const float* sinks,
                                           float sm_scale, int32_t window, void* out, int32_t num_q_heads,
                                           int32_t num_kv_heads, int32_t head_dim, int32_t page_size,
                                           int64_t num_blocks, int32_t kv_dtype, void* workspace,
                                           int64_t workspace_bytes, void* stream) {
  ApiGuard guard;
  return prefill_attention(q, k_cache, v_cache, k_scale, v_scale, block_table, table_stride, table_width, q_start,
                           prior_lens, R, max_q_len, sinks, sm_scale, window, out, num_q_heads, num_kv_heads, head_dim,
                           page_size, num_blocks, kv_dtype, workspace, workspace_bytes, stream);
}
