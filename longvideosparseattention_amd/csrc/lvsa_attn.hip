// Block-sparse flash-attention forward for LVSA on gfx950 (MI355X): the C ABI
// entry point (lvsa_attn_fwd), its argument checks and the dispatch by head
// size.  The kernels are in lvsa_attn_kernels.h, instantiated per head size
// in lvsa_attn_d64.hip, lvsa_attn_d96.hip, lvsa_attn_d128.hip,
// lvsa_attn_d192.hip and lvsa_attn_d256.hip.
#include "lvsa_attn_kernels.h"

#include <cstdlib>
#include <cstring>
#include <mutex>

using namespace lvsa;

namespace {

// Compute units of the current device (the persistent grid of the
// single-stream kernel), cached per device.
int cu_count() {
  static std::mutex mu;
  static int cached[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
  std::lock_guard<std::mutex> lock(mu);
  if (cached[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && n > 0) cached[dev] = n;
  }
  return cached[dev];
}

// Key blocks of a video tile of `rows` rows, guessed (the plan's counts are on
// the device): about six frames of anchors and window and a keyframe in eight,
// one more for each further query frame of the tile, and the extra rows.  Only
// balance depends on it.
int64_t guessed_tile_blocks(const lvsa_attn_args* a, int rows) {
  const int64_t C = a->C > 0 ? a->C : 1, R = a->R > 0 ? a->R : 1, frames = ceil_div(a->n_k, C);
  const int64_t more = rows % R == 0 || R % rows == 0 ? ceil_div(rows, R) - 1 : ceil_div(rows - 1, R);
  const int64_t attended = 6 + ceil_div(frames, 8) + more;
  const int64_t all = ceil_div(a->n_k, kBN);
  const int64_t b = attended < frames ? ceil_div(attended * C, kBN) : all;
  return (b < all ? b : all) + ceil_div(a->n_x, kBN);
}

// Key blocks (of 64 keys) per text chunk when a text tile is split: about a
// third of a Wan / HunyuanVideo video tile and below a CogVideoX one, so the
// chunks fill the launch's last round at a granularity finer than a tile
// (64 measured the same at CogVideoX and 0.3% slower at HunyuanVideo).
// Text tiles of one such chunk beside shorter video tiles may run in chunks as
// long as those (at least kMinTextChunkBlocks, wanted_text_chunks), where
// split_of finds that to end the launch sooner and they take at most
// kMaxSmallText of scratch and the caller's.
constexpr int kTextChunkBlocks = 128, kMinTextChunkBlocks = 16;
constexpr int kMaxTextChunks = 64;
constexpr int64_t kMaxSmallText = 16LL << 20;

int64_t text_ws_bytes(const lvsa_attn_args* a, int chunks) {
  if (a->n_tq == 0 || chunks <= 1) return 0;
  return 4 * (text_ws_o_elems(chunks, a->B, a->H, a->n_tq, a->D) + 2LL * chunks * a->B * a->H * a->n_tq);
}

// Most text chunks per text tile (1 = no split).
int wanted_text_chunks(const lvsa_attn_args* a) {
  if (a->n_tq == 0) return 1;
  const int64_t blocks = ceil_div(a->n_k, kBN) + ceil_div(a->n_x, kBN);
  const int64_t c = ceil_div(blocks, kTextChunkBlocks);
  if (c <= 1 && a->n_q > 0) {
    const int64_t tile = guessed_tile_blocks(a, 1);
    const int f = (int)ceil_div(blocks, tile > kMinTextChunkBlocks ? tile : kMinTextChunkBlocks);
    if (text_ws_bytes(a, f) <= kMaxSmallText) return f < 1 ? 1 : f;
  }
  return (int)(c < 1 ? 1 : (c > kMaxTextChunks ? kMaxTextChunks : c));
}

// Chunks that every workspace has to hold the partials of: those of long text
// tiles in 16 bit.
int text_chunks_least(const lvsa_attn_args* a) {
  const int64_t blocks = ceil_div(a->n_k, kBN) + ceil_div(a->n_x, kBN);
  return a->dtype == LVSA_FP32 || blocks <= kTextChunkBlocks ? 1 : wanted_text_chunks(a);
}

// The video split of a call: `tiles` tiles of `rows` rows per queue in `parts`
// parts each.
struct VideoSplit {
  int tiles = 0, parts = 0, rows = 0;
};

// Partials of the video split (O, then the (running max, row sum) pairs).
int64_t video_ws_bytes(const lvsa_attn_args* a, VideoSplit v) {
  if (v.tiles <= 0) return 0;
  return 4 * (video_ws_o_elems(v.tiles, v.parts, v.rows, a->D) + 2LL * kXcds * v.tiles * v.parts * v.rows);
}

int64_t align256(int64_t x) { return (x + 255) & ~int64_t(255); }

// fp32: blocks of K and V as fp16 pairs (lvsa_attn_f32.hip).  0 where that
// scratch would pass kMaxSplitBytes (as much as K and V themselves: 2.3 GB for
// 121 frames of 1560 tokens, 12 heads, D = 128) or the grid's 2^31: such a
// call runs the fp32 kernel.
constexpr int64_t kMaxSplitBytes = 16LL << 30;
int64_t f32_split_slots(const lvsa_attn_args* a) {
  if (a->dtype != LVSA_FP32) return 0;
  const int64_t slots = 2LL * a->B * a->Hkv * (ceil_div(a->n_k, kBN) + ceil_div(a->n_x, kBN));
  return slots >= (int64_t)INT32_MAX || f32_split_bytes(slots, a->D) > kMaxSplitBytes ? 0 : slots;
}

// Workspace of a call: the text-split partials at offset 0, the video-split
// partials, the work-queue counters (kQueueBytes) and the fp32 pairs after
// them, each at a 256-byte boundary.
struct Scratch {
  int chunks;
  VideoSplit v;
  int64_t slots, video, queue, split, bytes;
};
Scratch scratch_of(const lvsa_attn_args* a, int chunks, VideoSplit v, int64_t slots) {
  Scratch s{chunks, v, slots, 0, 0, 0, 0};
  s.video = align256(text_ws_bytes(a, chunks));
  s.queue = align256(s.video + video_ws_bytes(a, v));
  s.bytes = s.queue + kQueueBytes;
  s.split = align256(s.bytes);
  if (slots) s.bytes = s.split + f32_split_bytes(slots, a->D);
  return s;
}
Scratch scratch_least(const lvsa_attn_args* a) { return scratch_of(a, text_chunks_least(a), VideoSplit{}, 0); }
Scratch scratch_full(const lvsa_attn_args* a, bool video_split = true);

// Zero the work-queue counters (a kernel, not a memset, so the call can be
// captured in a HIP graph and replayed).
__global__ __launch_bounds__(64) void queue_reset_kernel(uint32_t* q) {
  if (threadIdx.x < 8) q[threadIdx.x * (kQueueStride / 4)] = 0u;
}

// Whether the short last key block of the frame-structured source crosses a
// frame boundary: it holds the t = n_k - 64 floor((n_k - 1) / 64) < 64 last
// keys, tokens [k_tok0 + n_k - t, k_tok0 + n_k), and the last boundary at or
// below its end lies e = (k_tok0 + n_k) mod C tokens before that end.  The
// plan builder describes such a block as "generic" (two frames and the rows
// past the end of the source).
bool stream_tail_crosses_frame(int64_t n_q, int64_t n_k, int64_t k_tok0, int C) {
  if (n_q == 0 || n_k <= 0 || C <= 0) return false;
  const int64_t t = n_k - kBN * ((n_k - 1) / kBN);
  const int64_t e = (k_tok0 + n_k) % C;
  return t < kBN && e > 0 && e < t;
}

// LVSA_VIDEO_SPLIT=0: no video tile's keys are split (comparisons).
bool no_key_split() {
  const char* e = getenv("LVSA_VIDEO_SPLIT");
  return e && strcmp(e, "0") == 0;
}

// Items of the longest queue (XCD) of a launch with tiles of `rows` rows, video
// tiles whole.
int64_t queue_fill(const lvsa_attn_args* a, int rows) {
  return ceil_div(ceil_div(a->n_q, rows) * a->H * a->B, kXcds) +
         ceil_div(ceil_div(a->n_tq, rows) * wanted_text_chunks(a) * a->H * a->B, kXcds);
}

// Which kernel a call runs, and on tiles of how many rows.
struct Route {
  bool stream, dual, half;   // the single-stream kernel, and its map
  bool pairs;                // the half map with two key groups
  int shift;                 // two tiles per plan tile
  int rows;                  // query rows per tile
  int per_cu;                // work-groups per CU
  bool src32, tail_cross;
};
Route route_of(const lvsa_attn_args* a) {
  const bool fp32 = a->dtype == LVSA_FP32;
  const int R = a->R > 0 ? a->R : 1, C = a->C > 0 ? a->C : 1;
  Route r{false, false, false, false, 0, a->block_q, 1, false, false};
  // The single-stream kernel (every 16-bit head size) serves plans without
  // generic descriptors: 256-row tiles touch at most two query frames when
  // frames have >= 255 rows (128-row tiles: 127), and 64-key blocks (even
  // short last ones) at most two key frames when frames have >= 64 keys.
  // LVSA_ATTN_KERNEL=pp selects the compiler-built kernels instead
  // (comparisons).
  const char* kenv = getenv("LVSA_ATTN_KERNEL");
  const bool force_pp = kenv != nullptr && strcmp(kenv, "pp") == 0;
  // Its copies address a whole key source through one buffer resource with
  // 32-bit byte offsets; at D = 96 and 192 the lanes of the unused chunks of
  // a row add 0x7FFF0000 to theirs, which must lie past the end of the
  // source (zeros, no access) or inside it (a harmless read into chunks no
  // read touches): the rows must stay below 2^31 bytes there.
  const int64_t lim = (a->D == 96 || a->D == 192) ? (1LL << 31) : (1LL << 32);
  auto fits32 = [lim](int64_t rows, int64_t row_elems) { return (rows + kBN) * row_elems * 2 < lim; };
  r.src32 = fits32(a->n_k, a->k_str[1]) && fits32(a->n_k, a->v_str[1]) &&
            (a->n_x == 0 || (fits32(a->n_x, a->kx_str[1]) && fits32(a->n_x, a->vx_str[1])));
  // Its lane copy offsets are 24-bit products (row x row stride in bytes).
  auto fits24 = [](int64_t row_elems) { return row_elems * 2 < (1LL << 24); };
  const bool str24 = fits24(a->k_str[1]) && fits24(a->v_str[1]) &&
                     (a->n_x == 0 || (fits24(a->kx_str[1]) && fits24(a->vx_str[1])));
  // Its loop masks "two-part" descriptors only.  A short last key block of
  // the frame source that crosses a frame boundary (a source starting
  // mid-frame, as on a context-parallel shard) has three parts (two frames
  // and the rows past the end) and is planned "generic".
  r.tail_cross = stream_tail_crosses_frame(a->n_q, a->n_k, a->k_tok0, C);
  if (fp32 || force_pp || !r.src32 || !str24 || r.tail_cross) return r;
  if (a->n_q > 0 && (R < a->block_q - 1 || C < kBN)) return r;
  // 12-wave tiles of 384 rows (D = 64); 256-row tiles of D <= 128 and, on the
  // dual-wide map, 192; the wide map's 128-row tiles of D = 192 and 256
  r.stream = true;
  if (a->D > 128 || a->block_q == kStream12BM) return r;
  // D = 64 on 256-row tiles: the dual map (64 rows per wave, 4 waves, two
  // work-groups per CU); LVSA_D64_WAVES=8 selects 8 waves of 32 rows instead
  // (comparisons).
  const char* w = getenv("LVSA_D64_WAVES");
  const bool waves8 = a->D == 64 && w && strcmp(w, "8") == 0;
  if (a->block_q == kBM) {
    r.half = a->D != 96;
  } else if (a->D != 96 && !waves8) {
    // A plan of few 256-row tiles runs as twice as many 128-row ones: while
    // each has a CU of its own at D = 128 (108 plan tiles: 51 -> 39 us, 124
    // with text 151 -> 106; 143 to 176 within -2% to +8%), two at D = 64 (108:
    // 42 -> 35 us, 256: 60 -> 52; 336 with text 103 -> 114).
    r.half = queue_fill(a, kBM) * kXcds <= cu_count() * (a->D == 128 ? 1 : 2);
    r.shift = r.half ? 1 : 0;
  }
  r.dual = a->D == 64 && !r.half && !waves8;
  if (r.half) {
    r.rows = kBM;
    // Two key groups while every item has a CU of its own: a single group's
    // four waves are one per SIMD there, which hides little of the softmax
    // (D = 64, 108 plan tiles: 36 -> 26 us; D = 128, 84 items 43 -> 33 us, 192
    // 42 -> 39, 216 42 -> 44: two groups read K and V twice as fast, and at
    // D = 128 that many of them run into the L2).  Like the video split, off
    // with LVSA_VIDEO_SPLIT=0.
    r.pairs = queue_fill(a, kBM) * kXcds <= cu_count() * (a->D == 128 ? 3 : 4) / 4 && !no_key_split();
  }
  if (r.half || r.dual) r.per_cu = r.pairs ? 1 : 2;
  return r;
}

// Launches of this many rounds of work-groups gain nothing from a finer last
// round, nor from short text tiles in chunks.
constexpr int kSplitRounds = 5;
constexpr int kMaxParts = 8;
constexpr int64_t kMaxVideoSplitBytes = 48LL << 20;

// What a call splits.
struct Split {
  int chunks;
  VideoSplit v;
};

// Work-groups per CU of the call's kernel for that many items.  fp32: one
// with two key groups for at most an item per CU (launch_f32).
int groups_per_cu(const lvsa_attn_args* a, const Route& r, int64_t items, int64_t cus) {
  if (items <= cus) return 1;
  if (a->dtype == LVSA_FP32) return a->D == 64 ? 3 : a->D <= 128 ? 2 : 1;
  return !r.stream && r.rows == kBM && a->D <= 128 ? 2 : r.per_cu;
}

// Work-groups of a CU that launch_us lets run side by side.  The single-stream
// kernel's, alone on a CU, are nearly as much faster (D = 128, 128 rows: 0.9
// and 1.7 us per block), so they count as one after the other; the 4-wave and
// the fp32 kernel's are not (1.6 and 2.0; 4 and 5.2).
int side_by_side(const lvsa_attn_args* a, const Route& r, int per_cu) {
  return a->dtype == LVSA_FP32 || (!r.stream && r.rows == kBM) ? per_cu : 1;
}

// Microseconds per key block of an item with per_cu items on its CU, as
// measured on launches of one round, tiles of 128 and 256 rows (with x = 1 for
// 256 rows of D = 128): the single-stream kernel 0.53 to 2.24 (two key groups:
// 0.54 at D = 128), the 4-wave kernel with masks in every block 1.35 to 2.49,
// fp32 1.6 to 5.8.
double block_us(const lvsa_attn_args* a, const Route& r, int per_cu) {
  const double x = r.rows * a->D / 32768.0;
  if (a->dtype == LVSA_FP32) return (0.15 + 5.3 * x) * per_cu;
  if (!r.stream && r.rows == kBM) return per_cu == 1 ? 0.55 + 2.0 * x : 0.73 + 2.5 * x;
  return (0.2 + 1.4 * x) * per_cu * (r.pairs ? 0.62 : 1.0);
}

// Estimated microseconds of a launch with the split s: the longest queue's
// items in their order, each taken by the first work-group that is free
// (without the work queues an XCD runs its own items too: 124 tiles in two
// parts and 8 text chunks, 33 on an XCD of 32 CUs: 151 us); the longest item
// takes its time beside another one.  8 us to start and end a launch and 5 per
// item; a merge 3, and its partials once each way at 4.6 TB/s.
double launch_us(const lvsa_attn_args* a, const Route& r, int64_t cus, const Split& s) {
  const int64_t all = ceil_div(a->n_k, kBN) + ceil_div(a->n_x, kBN), tile = guessed_tile_blocks(a, r.rows);
  const int64_t videos = ceil_div(ceil_div(a->n_q, r.rows) * a->H * a->B, kXcds);
  const int64_t texts = ceil_div(ceil_div(a->n_tq, r.rows) * s.chunks * a->H * a->B, kXcds);
  const int64_t split = s.v.tiles < videos ? s.v.tiles : videos;
  struct Items {
    int64_t n, blocks;
  } items[4] = {{s.chunks == 1 ? texts : 0, all},
                {videos - split, tile},
                {split * s.v.parts, s.v.parts ? ceil_div(tile, s.v.parts) : 0},
                {s.chunks == 1 ? 0 : texts, ceil_div(all, s.chunks)}};
  const int per_cu = groups_per_cu(a, r, kXcds * (texts + videos + split * (s.v.parts - 1)), cus);
  const int side = side_by_side(a, r, per_cu);
  const double share = (double)side / per_cu, per_item = 5.0 * share, per_block = block_us(a, r, per_cu) * share;
  // work-groups by the time at which they are free, ascending: a class of
  // equal items adds one time at most
  struct Free {
    double t;
    int64_t n;
  } free[6] = {{0.0, cus * side / kXcds > 0 ? cus * side / kXcds : 1}};
  int nf = 1;
  double end = 0.0;
  for (const Items& it : items) {
    const double us = per_item + it.blocks * per_block;
    if (it.n > 0 && us > end * share) end = us / share;
    for (int64_t left = it.n; left > 0;) {
      const int64_t x = left < free[0].n ? left : free[0].n;
      const double t = free[0].t + us;
      left -= x;
      end = t > end ? t : end;
      if (x == free[0].n) {
        for (int i = 1; i < nf; ++i) free[i - 1] = free[i];
        --nf;
      } else {
        free[0].n -= x;
      }
      int at = nf;
      while (at > 0 && free[at - 1].t > t) --at;
      if (at > 0 && free[at - 1].t == t) {
        free[at - 1].n += x;
        continue;
      }
      for (int i = nf; i > at; --i) free[i] = free[i - 1];
      free[at] = {t, x};
      ++nf;
    }
  }
  return 8.0 + end + (s.v.tiles > 0 ? 3.0 + video_ws_bytes(a, s.v) / 2.3e6 : 0.0) +
         (s.chunks > 1 ? 3.0 + text_ws_bytes(a, s.chunks) / 2.3e6 : 0.0);
}

// The split of a call: text chunks, and video tiles that run as parts of their
// key ranges at the end of the launch (none with LVSA_VIDEO_SPLIT=0), so that
// its last round is finer than whole tiles.
// - Long text tiles always run in chunks.
// - The dual map over the work queues: its two work-groups per CU take whole
//   tiles at half the CU's rate, so a last round of whole tiles leaves CUs
//   idle for longer.  As many tiles per queue as the queue has work-groups on
//   its XCD, halved (32), in two parts (CogVideoX 0.9% faster).
// - Otherwise launches of fewer than kSplitRounds rounds: the tiles of a last
//   round that is not full in the number of parts, and short text tiles in
//   chunks, that end the launch soonest (launch_us), where parts save 6 us and
//   6% of it (chunks alone 3 us and 4%).  33 frames of 390 tokens, 12 heads,
//   D = 128 (612 tiles, 2.4 rounds): 383 -> 338 us and 10 for the merge; 9
//   frames of 256 (108 tiles, one round): 46 -> 36 + 10, so whole; 33 frames
//   of 400, 6 heads, 40 text tokens: 247 us whole and 272 in parts, beside
//   which the text chunks are the longest items.  24 frames of 130, 12 heads,
//   D = 128, 37 text tokens ran its one 50-block text tile per head whole,
//   three times as long as its video tiles (69.6 us, 59.1 in chunks); 13
//   frames of 600, 24 heads, D = 64, 226 text tokens take 261 us with whole
//   text tiles, first in the launch, and 295 with chunks at its end.  Longer
//   launches gain little from their last round and pay the same merge (Wan 4x
//   and HunyuanVideo, 24 and 20 rounds, within +-0.5%).
Split split_of(const lvsa_attn_args* a, const Route& r, bool video) {
  const int want = wanted_text_chunks(a);
  const bool long_text = ceil_div(a->n_k, kBN) + ceil_div(a->n_x, kBN) > kTextChunkBlocks || a->n_q == 0;
  Split best{long_text ? want : 1, VideoSplit{}};
  const int64_t cus = cu_count();
  if (a->n_q == 0 || cus <= 0) return best;
  const int64_t vwork = ceil_div(a->n_q, r.rows) * a->H * a->B;
  const int64_t twork = ceil_div(a->n_tq, r.rows) * a->H * a->B;
  const int per_cu = groups_per_cu(a, r, vwork + twork * want, cus);
  const int64_t groups = cus * per_cu;
  video = video && !no_key_split() && a->block_q != kStream12BM;
  const bool dual = video && r.dual && vwork + twork > groups;
  if (dual) {
    const int64_t s = groups / (2 * kXcds), per_queue = ceil_div(vwork, kXcds);
    best.v = VideoSplit{(int)(s < per_queue ? s : per_queue), 2, r.rows};
  }
  const int64_t blocks = guessed_tile_blocks(a, r.rows);
  const int64_t rest = vwork % (cus * side_by_side(a, r, per_cu));
  const int most = dual || !video || rest == 0 ? 1 : (int)(blocks / 6 < kMaxParts ? blocks / 6 : kMaxParts);
  if (vwork >= kSplitRounds * groups || (most < 2 && (long_text || want == 1))) return best;
  const double whole = launch_us(a, r, cus, best);
  auto margin = [whole](double us, double share) { return us > share * whole ? us : share * whole; };
  double least = whole;
  for (int chunks = best.chunks, more = 1; more; chunks = want) {
    more = !long_text && chunks < want;
    for (int k = 1; k <= most || k == 1; ++k) {
      Split s{chunks, dual ? best.v : VideoSplit{}};
      if (k > 1) s.v = VideoSplit{(int)ceil_div(rest, kXcds), k, r.rows};
      if (k > 1 && video_ws_bytes(a, s.v) > kMaxVideoSplitBytes) break;
      double t = launch_us(a, r, cus, s);
      if (k > 1) t += margin(6.0, 0.06);
      else if (chunks > 1 && !long_text) t += margin(3.0, 0.04);
      if (t < least) {
        least = t;
        best = s;
      }
    }
  }
  return best;
}

Scratch scratch_full(const lvsa_attn_args* a, bool video_split) {
  const int64_t slots = f32_split_slots(a);
  if (a->dtype == LVSA_FP32 && slots == 0) return scratch_least(a);
  if (a->block_q <= 0) return scratch_of(a, text_chunks_least(a), VideoSplit{}, slots);
  const Split s = split_of(a, route_of(a), video_split);
  return scratch_of(a, s.chunks, s.v, slots);
}

// Exact log-sum-exp merge of the text chunks (lvsa-vllm-omni/lvsa_vllm_omni/
// flashinfer_runner.py:184-197 merges two key sets the same way): with m_c the
// running max (log2 units), l_c the row sum and o_c the unnormalised O of
// chunk c, O = sum_c 2^(m_c - M) o_c / sum_c 2^(m_c - M) l_c, M = max_c m_c.
// One thread per 4 consecutive d of one (batch, head, text row).
template <typename E>
__global__ __launch_bounds__(256) void attn_text_merge_kernel(const float* ws, int chunks, int B, int H, int n_tq,
                                                              int D, char* ot, int64_t s0, int64_t s1, int64_t s2,
                                                              float* lse_t) {
  const int g4 = D / 4;
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t per_bh = (int64_t)n_tq * g4;
  if (t >= per_bh * B * H) return;
  const int64_t bh = t / per_bh;
  const int row = (int)((t % per_bh) / g4), dq = (int)(t % g4);
  const int head = (int)(bh % H), batch = (int)(bh / H);
  const int64_t stride_c = (int64_t)B * H * n_tq;  // slots per chunk
  const int64_t slot0 = bh * n_tq + row;
  const float2* ml = reinterpret_cast<const float2*>(ws + text_ws_o_elems(chunks, B, H, n_tq, D));
  float M = -INFINITY;
  for (int c = 0; c < chunks; ++c) M = fmaxf(M, ml[c * stride_c + slot0].x);
  float L = 0.f;
  float4 acc = float4{0.f, 0.f, 0.f, 0.f};
  for (int c = 0; c < chunks; ++c) {
    const float2 mc = ml[c * stride_c + slot0];
    const float w = __builtin_amdgcn_exp2f(mc.x - M);
    const float4 o = *reinterpret_cast<const float4*>(ws + (c * stride_c + slot0) * D + 4 * dq);
    L += w * mc.y;
    acc.x += w * o.x;
    acc.y += w * o.y;
    acc.z += w * o.z;
    acc.w += w * o.w;
  }
  const float inv = L > 0.f ? 1.0f / L : 0.f;
  E* op = reinterpret_cast<E*>(ot + sizeof(E) * (batch * s0 + row * s1 + head * s2)) + 4 * dq;
  op[0] = (E)(acc.x * inv);
  op[1] = (E)(acc.y * inv);
  op[2] = (E)(acc.z * inv);
  op[3] = (E)(acc.w * inv);
  if (lse_t && dq == 0)
    lse_t[bh * n_tq + row] = L > 0.f ? (M + __log2f(L)) * 0.69314718055994530942f : -INFINITY;
}

// Merge of the parts of the split video tiles (vsplit slots per queue): one
// thread per (slot, row, 4 columns), the exact log-sum-exp combination of
// attn_text_merge_kernel, written where the unsplit tile writes O and LSE.
// Bound by the partials it reads.
template <typename E>
__global__ __launch_bounds__(256) void attn_video_merge_kernel(AttnParams p, int block_q, int D) {
  const int g4 = D / 4;
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t per_slot = (int64_t)block_q * g4;
  const int64_t slot = t / per_slot;   // x * vsplit + s
  if (slot >= (int64_t)kXcds * p.vsplit) return;
  const int x = (int)(slot / p.vsplit), sx = (int)(slot % p.vsplit);
  const QueueShape q = queue_shape(p, x);
  if (sx >= q.n_split) return;
  const int w = q.v0 + q.n_video - q.n_split + sx;
  const int tile = w % p.n_vt, rest = w / p.n_vt, head = rest % p.H, batch = rest / p.H;
  const int r = (int)((t % per_slot) / g4), dq = (int)(t % g4);
  const int64_t row = (int64_t)tile * block_q + r;
  if (row >= p.n_q) return;
  const float2* ml = reinterpret_cast<const float2*>(p.vws + video_ws_o_elems(p.vsplit, q.parts, block_q, D));
  const int64_t i0 = (q.parts * slot) * block_q + r;
  float M = -INFINITY;
  for (int c = 0; c < q.parts; ++c) M = fmaxf(M, ml[i0 + (int64_t)c * block_q].x);
  float L = 0.f;
  float4 acc = float4{0.f, 0.f, 0.f, 0.f};
  for (int c = 0; c < q.parts; ++c) {
    const int64_t i = i0 + (int64_t)c * block_q;
    const float2 mc = ml[i];
    const float wt = __builtin_amdgcn_exp2f(mc.x - M);
    const float4 o = *reinterpret_cast<const float4*>(p.vws + i * D + 4 * dq);
    L += wt * mc.y;
    acc.x += wt * o.x;
    acc.y += wt * o.y;
    acc.z += wt * o.z;
    acc.w += wt * o.w;
  }
  const float inv = L > 0.f ? 1.0f / L : 0.f;
  E* op = reinterpret_cast<E*>(p.o + sizeof(E) * (batch * p.o_str[0] + row * p.o_str[1] + head * p.o_str[2])) + 4 * dq;
  op[0] = (E)(acc.x * inv);
  op[1] = (E)(acc.y * inv);
  op[2] = (E)(acc.z * inv);
  op[3] = (E)(acc.w * inv);
  if (p.lse && dq == 0)
    p.lse[((int64_t)batch * p.H + head) * p.n_q + row] =
        L > 0.f ? (M + __log2f(L)) * 0.69314718055994530942f : -INFINITY;
}

bool aligned16(const void* ptr, const int64_t* str, int n, int elem_bytes) {
  if (((uintptr_t)ptr) % 16) return false;
  for (int i = 0; i < n; ++i)
    if ((str[i] * elem_bytes) % 16) return false;
  return true;
}

}  // namespace

extern "C" int lvsa_attn_fwd(const lvsa_attn_args* a, hipStream_t stream) {
  clear_error();
  LVSA_REQUIRE(a != nullptr, LVSA_ERR_INVALID_ARG, "lvsa_attn_fwd: null args");
  LVSA_REQUIRE(a->D == 64 || a->D == 96 || a->D == 128 || a->D == 192 || a->D == 256, LVSA_ERR_UNSUPPORTED,
               "lvsa_attn_fwd: head_dim %d not supported (64, 96, 128, 192, 256)", a->D);
  LVSA_REQUIRE(a->D < 192 || a->block_q == kBM || (a->D == 192 && a->block_q == kPPBM), LVSA_ERR_UNSUPPORTED,
               "lvsa_attn_fwd: head_dim %d runs 128-row tiles (192 also 256-row ones; block_q %d)", a->D,
               a->block_q);
  LVSA_REQUIRE(a->dtype == LVSA_BF16 || a->dtype == LVSA_FP16 || a->dtype == LVSA_FP32, LVSA_ERR_UNSUPPORTED,
               "lvsa_attn_fwd: dtype %d", a->dtype);
  const bool fp32 = a->dtype == LVSA_FP32;
  const int es = fp32 ? 4 : 2;   // bytes per element
  LVSA_REQUIRE(fp32 || a->D != 96 || a->block_q == kPPBM, LVSA_ERR_UNSUPPORTED,
               "lvsa_attn_fwd: head_dim 96 runs 256-row tiles (block_q %d)", a->block_q);
  LVSA_REQUIRE(!fp32 || a->block_q == kBM, LVSA_ERR_UNSUPPORTED,
               "lvsa_attn_fwd: fp32 runs 128-row tiles (block_q %d)", a->block_q);
  LVSA_REQUIRE(a->B >= 1 && a->H >= 1 && a->Hkv >= 1 && a->H % a->Hkv == 0, LVSA_ERR_INVALID_ARG,
               "lvsa_attn_fwd: B=%d H=%d Hkv=%d (H must be a multiple of Hkv)", a->B, a->H, a->Hkv);
  LVSA_REQUIRE(a->n_q >= 0 && a->n_k >= 0 && a->n_x >= 0 && a->n_tq >= 0, LVSA_ERR_INVALID_ARG,
               "lvsa_attn_fwd: negative length");
  LVSA_REQUIRE(a->tile_indptr && a->entries, LVSA_ERR_INVALID_ARG, "lvsa_attn_fwd: missing plan");
  LVSA_REQUIRE(a->block_q == kBM || a->block_q == kPPBM || a->block_q == kStream12BM, LVSA_ERR_UNSUPPORTED,
               "lvsa_attn_fwd: block_q %d (the kernels tile 128, 256 or 384 query rows)", a->block_q);
  // 384-row tiles: the 12-wave single-stream kernel, head size 64 in 16 bit;
  // its loop handles descriptors "none" and "two-part" only, which is all a
  // plan holds when a tile touches at most two query frames (frames of at
  // least 383 rows) and a key block at most two key frames (at least 64).
  LVSA_REQUIRE(a->block_q != kStream12BM ||
                   (a->D == 64 && !fp32 && (a->n_q == 0 || (a->R >= kStream12BM - 1 && a->C >= kBN))),
               LVSA_ERR_UNSUPPORTED,
               "lvsa_attn_fwd: 384-row tiles need head_dim 64 in bf16/fp16 and frames of >= 383 query and >= 64 "
               "key rows (head_dim %d, R %d, C %d); build the plan with block_q 256", a->D, a->R, a->C);
  const int plan_vt = (int)ceil_div(a->n_q, a->block_q), plan_tt = (int)ceil_div(a->n_tq, a->block_q);
  LVSA_REQUIRE(a->n_video_tiles == plan_vt && a->n_tiles == plan_vt + plan_tt, LVSA_ERR_INVALID_ARG,
               "lvsa_attn_fwd: plan has %d/%d tiles, expected %d/%d for block_q %d", a->n_video_tiles,
               a->n_tiles, plan_vt, plan_vt + plan_tt, a->block_q);
  LVSA_REQUIRE(a->n_q == 0 || (a->q && a->o), LVSA_ERR_INVALID_ARG, "lvsa_attn_fwd: null q/o");
  LVSA_REQUIRE(a->n_tq == 0 || (a->qt && a->ot), LVSA_ERR_INVALID_ARG, "lvsa_attn_fwd: null text q/o");
  LVSA_REQUIRE(a->n_k == 0 || (a->k && a->v), LVSA_ERR_INVALID_ARG, "lvsa_attn_fwd: null k/v");
  LVSA_REQUIRE(a->n_x == 0 || (a->kx && a->vx), LVSA_ERR_INVALID_ARG, "lvsa_attn_fwd: null extra k/v");
  LVSA_REQUIRE(a->n_k + a->n_x > 0 || a->n_tiles == 0, LVSA_ERR_INVALID_ARG, "lvsa_attn_fwd: no keys");
  bool ok = true;
  if (a->n_q) ok = ok && aligned16(a->q, a->q_str, 3, es) && aligned16(a->o, a->o_str, 3, es);
  if (a->n_tq) ok = ok && aligned16(a->qt, a->qt_str, 3, es) && aligned16(a->ot, a->ot_str, 3, es);
  if (a->n_k) ok = ok && aligned16(a->k, a->k_str, 3, es) && aligned16(a->v, a->v_str, 3, es);
  if (a->n_x) ok = ok && aligned16(a->kx, a->kx_str, 3, es) && aligned16(a->vx, a->vx_str, 3, es);
  LVSA_REQUIRE(ok, LVSA_ERR_UNSUPPORTED, "lvsa_attn_fwd: tensors must be 16-byte aligned with 16-byte row strides");
  // per-lane DMA offsets within a 64-row key block are 32-bit
  auto fits = [&](int64_t row_elems) { return row_elems >= 0 && row_elems * es * (kBN - 1) + es * (int64_t)a->D <= 0xFFFFFFFFLL; };
  LVSA_REQUIRE(fits(a->k_str[1]) && fits(a->v_str[1]) && (a->n_x == 0 || (fits(a->kx_str[1]) && fits(a->vx_str[1]))),
               LVSA_ERR_UNSUPPORTED, "lvsa_attn_fwd: key/value row stride too large");
  // the 256-row kernel forms per-lane row offsets with 24-bit multiplies
  auto fits24 = [&](int64_t row_elems) { return row_elems * 2 < (1LL << 24); };
  LVSA_REQUIRE(a->block_q == kBM || (fits24(a->k_str[1]) && fits24(a->v_str[1]) &&
                                       (a->n_x == 0 || (fits24(a->kx_str[1]) && fits24(a->vx_str[1])))),
               LVSA_ERR_UNSUPPORTED, "lvsa_attn_fwd: key/value row stride of 16 MiB or more (block_q %d)",
               a->block_q);
  // Every query row must have a relation row (generic blocks read it).
  if (a->n_q > 0) {
    const int64_t R = a->R > 0 ? a->R : 1;
    const int64_t first = a->q_tok0 / R - a->q_frame0, last = (a->q_tok0 + a->n_q - 1) / R - a->q_frame0;
    LVSA_REQUIRE(a->q_tok0 >= 0 && a->k_tok0 >= 0 && first >= 0 && last < a->rel_rows && a->rel && a->words >= 1,
                 LVSA_ERR_INVALID_ARG,
                 "lvsa_attn_fwd: query rows map to relation rows [%lld, %lld], the relation has %d rows",
                 (long long)first, (long long)last, a->rel_rows);
  }
  // As much of the scratch as the workspace holds: all, without the video
  // split, or the least.
  Scratch ws{1, VideoSplit{}, 0, 0, 0, 0, 0};
  int64_t ws_need = 0;
  if (a->workspace) {
    const Scratch least = scratch_least(a);
    ws_need = least.bytes;
    ws = scratch_full(a);
    if (ws.bytes > a->workspace_bytes) ws = scratch_full(a, false);
    if (ws.bytes > a->workspace_bytes) ws = least;
  }
  const int chunks = ws.chunks;
  const Route route = route_of(a);
  const int n_vt = (int)ceil_div(a->n_q, route.rows), n_tt = (int)ceil_div(a->n_tq, route.rows);
  LVSA_REQUIRE(a->workspace_bytes >= ws_need, LVSA_ERR_CAPACITY,
               "lvsa_attn_fwd: workspace of %lld bytes < %lld needed (lvsa_attn_workspace_query)",
               (long long)a->workspace_bytes, (long long)ws_need);
  LVSA_REQUIRE(ws_need == 0 || ((uintptr_t)a->workspace) % 16 == 0, LVSA_ERR_INVALID_ARG,
               "lvsa_attn_fwd: workspace must be 16-byte aligned");
  const int64_t vwork = (int64_t)n_vt * a->H * a->B, twork = (int64_t)n_tt * chunks * a->H * a->B;
  const int64_t work = vwork + twork;
  LVSA_REQUIRE(work < (int64_t)INT32_MAX, LVSA_ERR_INVALID_ARG, "lvsa_attn_fwd: too much work");
  if (work == 0) return LVSA_OK;

  AttnParams p;
  p.q = (const char*)a->q;
  p.k = (const char*)a->k;
  p.v = (const char*)a->v;
  p.kx = (const char*)a->kx;
  p.vx = (const char*)a->vx;
  p.qt = (const char*)a->qt;
  p.o = (char*)a->o;
  p.ot = (char*)a->ot;
  p.lse = a->lse;
  p.lse_t = a->lse_t;
  for (int i = 0; i < 3; ++i) {
    p.q_str[i] = a->q_str[i];
    p.k_str[i] = a->k_str[i];
    p.v_str[i] = a->v_str[i];
    p.kx_str[i] = a->kx_str[i];
    p.vx_str[i] = a->vx_str[i];
    p.qt_str[i] = a->qt_str[i];
    p.o_str[i] = a->o_str[i];
    p.ot_str[i] = a->ot_str[i];
  }
  p.B = a->B;
  p.H = a->H;
  p.Hkv = a->Hkv;
  p.group = a->H / a->Hkv;
  p.n_q = a->n_q;
  p.n_k = a->n_k;
  p.n_x = a->n_x;
  p.n_tq = a->n_tq;
  p.scale_log2 = a->scale * 1.4426950408889634f;
  p.tile_indptr = a->tile_indptr;
  p.entries = reinterpret_cast<const uint2*>(a->entries);
  p.n_tiles = a->n_tiles;
  p.n_vt = n_vt;
  p.n_tt = n_tt;
  p.rel = a->rel;
  p.words = a->words;
  p.R = a->R > 0 ? a->R : 1;
  p.C = a->C > 0 ? a->C : 1;
  p.qo = (uint32_t)(a->q_tok0 % p.R);
  p.ko = (uint32_t)(a->k_tok0 % p.C);
  p.qf0 = (int)(a->q_tok0 / p.R - a->q_frame0);
  p.kf0 = (int)(a->k_tok0 / p.C);
  p.total_work = (int)work;
  p.n_vwork = (int)vwork;
  p.n_twork = (int)twork;
  p.text_chunks = chunks;
  p.text_first = chunks == 1 ? 1 : 0;
  p.ws = chunks > 1 ? (float*)a->workspace : nullptr;
  p.split = nullptr;
  p.split_exp = nullptr;
  p.split_slots = (int)ws.slots;
  if (ws.slots) {
    p.split = (char*)a->workspace + ws.split;
    p.split_exp = (int32_t*)(p.split + ws.slots * 4LL * kBN * a->D);
  }
  // Calls without text rows and of fewer query rows than keys (per K/V head)
  // may leave most of K and V unattended.  Each work-group of the split then
  // reads the relation rows first (at most 16 KiB of them).
  const int64_t rel_words = a->n_q > 0 ? ((a->q_tok0 % p.R + a->n_q - 1) / p.R + 1) * (int64_t)a->words : 0;
  p.split_seen = ws.slots && a->n_tq == 0 && a->n_q > 0 && (int64_t)a->n_q * p.group < a->n_k &&
                 a->words <= kSeenWords && rel_words <= 4096;
  p.vsplit = ws.v.tiles;
  p.vparts = ws.v.parts;
  p.vws = ws.v.tiles > 0 ? (float*)((char*)a->workspace + ws.video) : nullptr;
  // A plan holds generic blocks only where a tile touches more than two query
  // frames or a key block more than two parts.
  const bool generic = a->n_q > 0 && (p.R < a->block_q - 1 || p.C < kBN || route.tail_cross);
  p.rel_lds = generic && p.words <= kRelWords;
  // D = 192 on 256-row tiles: the loop's dual-wide map, the only kernel for
  // them (frames of >= 255 query rows).
  LVSA_REQUIRE(a->D != 192 || a->block_q != kPPBM || route.stream, LVSA_ERR_UNSUPPORTED,
               "lvsa_attn_fwd: head_dim 192 on 256-row tiles needs frames of >= 255 query and >= 64 key rows, "
               "key sources below 2^31 bytes with row strides below 16 MiB, the last key block of the frame "
               "source inside one frame, and no LVSA_ATTN_KERNEL=pp (R %d, C %d); build the plan with block_q 128",
               p.R, p.C);
  if (a->block_q == kStream12BM) {
    LVSA_REQUIRE(route.src32, LVSA_ERR_UNSUPPORTED,
                 "lvsa_attn_fwd: 384-row tiles address each key source with 32-bit byte offsets (source too large); "
                 "build the plan with block_q 256");
    LVSA_REQUIRE(!route.tail_cross, LVSA_ERR_UNSUPPORTED,
                 "lvsa_attn_fwd: 384-row tiles need the last key block of the frame source inside one frame "
                 "(n_k %lld, k_tok0 %lld, C %d); build the plan with block_q 256",
                 (long long)a->n_k, (long long)a->k_tok0, p.C);
  }
  p.use_stream = route.stream || a->block_q == kStream12BM;
  p.dual = route.dual;
  p.half = route.pairs ? 2 : route.half ? 1 : 0;
  p.plan_shift = route.shift;
  // With a workspace, the single-stream kernel runs one persistent
  // work-group per CU (two with the dual and the half map) over the work
  // queues (counters zeroed first).
  p.queues = nullptr;
  p.grid = static_grid(p);
  const int cus = cu_count();
  const int per_cu = route.per_cu;
  if (p.use_stream && a->workspace && cus > 0 && work > per_cu * cus) {
    p.queues = (uint32_t*)((char*)a->workspace + ws.queue);
    p.grid = per_cu * cus;
    hipLaunchKernelGGL(queue_reset_kernel, dim3(1), dim3(64), 0, stream, p.queues);
    const int qrc = launch_status("lvsa_attn_fwd (queue reset)");
    if (qrc != LVSA_OK) return qrc;
  }
  const int bq = a->block_q;
  const bool bf16 = a->dtype == LVSA_BF16;
  int rc;
  if (fp32) rc = launch_f32(p, a->D, cus, stream);
  else if (a->D == 256) rc = launch_d256(p, bq, bf16, stream);
  else if (a->D == 128) rc = launch_d128(p, bq, bf16, stream);
  else if (a->D == 96) rc = launch_d96(p, bq, bf16, stream);
  else if (a->D == 192) rc = launch_d192(p, bq, bf16, stream);
  else rc = launch_d64(p, bq, bf16, stream);
  if (rc != LVSA_OK) return rc;
  if (p.vsplit > 0) {
    const int64_t threads = (int64_t)kXcds * p.vsplit * route.rows * (a->D / 4);
    const dim3 grid((unsigned)ceil_div(threads, 256));
    if (fp32) hipLaunchKernelGGL(attn_video_merge_kernel<float>, grid, dim3(256), 0, stream, p, route.rows, a->D);
    else if (bf16) hipLaunchKernelGGL(attn_video_merge_kernel<__bf16>, grid, dim3(256), 0, stream, p, route.rows, a->D);
    else hipLaunchKernelGGL(attn_video_merge_kernel<_Float16>, grid, dim3(256), 0, stream, p, route.rows, a->D);
    rc = launch_status("lvsa_attn_fwd (video merge)");
    if (rc != LVSA_OK) return rc;
  }
  if (chunks == 1) return rc;
  const int64_t threads = (int64_t)a->B * a->H * a->n_tq * (a->D / 4);
  const dim3 grid((unsigned)ceil_div(threads, 256));
  if (fp32) {
    hipLaunchKernelGGL(attn_text_merge_kernel<float>, grid, dim3(256), 0, stream, (const float*)a->workspace,
                       chunks, a->B, a->H, a->n_tq, a->D, (char*)a->ot, a->ot_str[0], a->ot_str[1], a->ot_str[2],
                       a->lse_t);
  } else if (bf16) {
    hipLaunchKernelGGL(attn_text_merge_kernel<__bf16>, grid, dim3(256), 0, stream, (const float*)a->workspace,
                       chunks, a->B, a->H, a->n_tq, a->D, (char*)a->ot, a->ot_str[0], a->ot_str[1], a->ot_str[2],
                       a->lse_t);
  } else {
    hipLaunchKernelGGL(attn_text_merge_kernel<_Float16>, grid, dim3(256), 0, stream, (const float*)a->workspace,
                       chunks, a->B, a->H, a->n_tq, a->D, (char*)a->ot, a->ot_str[0], a->ot_str[1], a->ot_str[2],
                       a->lse_t);
  }
  return launch_status("lvsa_attn_fwd (text merge)");
}

namespace lvsa {
int64_t attn_workspace_min_bytes(const lvsa_attn_args* a) { return scratch_least(a).bytes; }
}  // namespace lvsa

extern "C" int lvsa_attn_workspace_query(const lvsa_attn_args* a, int64_t* bytes) {
  clear_error();
  LVSA_REQUIRE(a != nullptr && bytes != nullptr, LVSA_ERR_INVALID_ARG, "lvsa_attn_workspace_query: null pointer");
  LVSA_REQUIRE(a->n_k >= 0 && a->n_x >= 0 && a->n_tq >= 0 && a->B >= 1 && a->H >= 1, LVSA_ERR_INVALID_ARG,
               "lvsa_attn_workspace_query: bad sizes");
  LVSA_REQUIRE(a->D == 64 || a->D == 96 || a->D == 128 || a->D == 192 || a->D == 256, LVSA_ERR_UNSUPPORTED,
               "lvsa_attn_workspace_query: head_dim %d not supported", a->D);
  *bytes = scratch_full(a).bytes;
  return LVSA_OK;
}
