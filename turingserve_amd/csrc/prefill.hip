// Paged chunked-prefill attention for gfx950 (ops/triton_prefill_attention.py:17-79).
// Host entry points; the kernels and their launch plans are in prefill_kernels.h (head_dim < 128,
// and the 4-wavefront tile kernel) and prefill_pair.h (head_dim 128).
#include <type_traits>

#include "prefill_pair.h"

using namespace ts;

namespace {

// head_dim 64: which kernel, and the tile kernel's key groups and split plan, from host bounds
// alone. Measured on MI355X (H 14 unless said, KVH 2, us per call: stream kernel / tile kernel with
// one key group and 128-row tiles / with two and 64-row tiles):
//  * the stream kernel keeps short contexts whose 32-row tiles fit one per CU, where a call is
//    launch and first-load latency and no split pays: 2 rows on 0 4.1 / 4.7 / 5.8, 256 on 0 7.6 / 8.7
//    / 7.2, 512 on 0 9.7 / 12.6 / 9.8, 300 on 700 13.3 and 15.0 with two groups, 512 on 1000 17.6 and
//    17.9 (past one per CU: six chunks of 300 on 0 14.5 / 9.6 / 9.5); a batch of a few tiles, whose
//    keys split well, leaves it at 640 keys (30 rows on 700 11.1 and 10.1, 16 on 500 9.2 and 9.9), a
//    single chunk whose 64-row tiles give most CUs work, which a split can only double, later than
//    others (two layers, stream and split tiles: 700 on 900 on 8 heads 42.1 / 43.8, 1024 on 596 42.0 /
//    44.9, on 736 44.1 / 45.8 and on 926 47.5 / 46.6, 500 on 1080 on 14 heads 39.2 / 40.2; three of 240
//    on 1340 on 8 heads 44.9 / 39.2);
//  * two key groups halve a workgroup's chain of key steps and give a short batch twice the
//    workgroups: 1024 on 0 19.3 / 18.2 / 15.2, 2048 on 0 43.8 / 32.2 / 30.0, 2000-token prefix with
//    16 rows 19.5 / 11.5 / 11.0, five ragged chunks 35.7 / 31.8 / 23.8;
//  * one key group (three workgroups per CU, each staged step read by four wavefronts) where the
//    key ranges are long enough to split (2048 on 4096 131.8 / 70.9 / 82.0, 1000 on 6000 88.0 / 52.0 /
//    58.5) or the tiles fill the device anyway (H 28: six of 300 on 0 22.6 / 12.3 / 17.2).
// A split costs its partials' traffic and the merge launch, about 4.5 us, so with two key groups
// only a batch of a few tiles splits below 16 steps (16 rows on 2000: 11.0 us at 4 steps, 16.7 at
// 16; 512 on 1000: 19.9 and 17.9), and one whose tiles reach half the CUs splits from 28 steps on
// (1115 on 94, 19 steps: 18.3 unsplit, 19.8 split; 400 on 1500, 30 steps: 23.8 and 20.0; three of 120
// on 1600, few tiles: 22.1 and 18.4).
enum { kStream64 = 0 };                            // Plan64::ks of the stream kernel
struct Plan64 {
  int ks;                                          // key groups of the tile kernel
  TilePlan tile;
};
constexpr int kStream64Keys = 1536, kStream64KeysFew = 640;
constexpr int kStream64KeysThird = 1664, kStream64KeysMost = 1760;   // a single chunk
constexpr int kLong64Steps = 64, kFew64 = 8, kSplit64Steps = 16, kSplit64From = 28;

TilePlan tile_plan64(int ks, int min_steps, int P, int H, int max_query_len, int max_seq_len,
                     int cus, bool split) {
  const int per_cu = ks == 2 ? kTilePerCu<64, 2> : kTilePerCu<64, 1>;
  return tile_plan(P, H, 64, max_query_len, max_seq_len, cus, split, (int64_t)per_cu * cus,
                   tile_rows(ks), min_steps);
}

// num_tokens bounds the tiles of a batch of unequal chunks better than P of the longest.
Plan64 plan64(int P, int H, int64_t num_tokens, int max_query_len, int max_seq_len, int cus,
              bool split) {
  const int seq = max_seq_len > max_query_len ? max_seq_len : max_query_len;
  auto tiles = [&](int rows) {
    const int64_t a = (int64_t)cdiv(max_query_len, rows) * P, b = num_tokens / rows + P;
    return (a < b ? a : b) * H;
  };
  const int64_t t2 = tiles(tile_rows(2));
  const bool few = t2 * kFew64 <= cus;
  int stream_keys = few ? kStream64KeysFew : kStream64Keys;
  if (P == 1 && t2 * 3 > cus) stream_keys = t2 * 16 >= 7LL * cus ? kStream64KeysMost : kStream64KeysThird;
  if (tiles(kPsRows) <= cus && seq <= stream_keys) return {kStream64, {}};
  const int ks = cdiv(seq, kTileKeys) >= kLong64Steps || tiles(kTileRows) * 4 > 7LL * cus ? 1 : 2;
  const int min_steps = ks == 1 || few ? kPrefillMinSteps : kSplit64Steps;
  const bool pays =
      ks == 1 || t2 * 2 <= cus || cdiv(seq, kTileKeys) >= kSplit64From;
  return {ks, tile_plan64(ks, min_steps, P, H, max_query_len, max_seq_len, cus, split && pays)};
}

// Partials of whichever plan the launch takes.
size_t workspace64(int P, int H, int max_query_len, int max_seq_len, int cu_count) {
  const int cus = cu_count > 0 ? cu_count : 256;
  size_t most = 0;
  for (int ks = 1; ks <= 2; ++ks)
    for (int steps : {kPrefillMinSteps, kSplit64Steps}) {
      const size_t b =
          tile_plan64(ks, steps, P, H, max_query_len, max_seq_len, cus, true).ws_bytes;
      most = b > most ? b : most;
    }
  return most;
}

// head_dim 128 runs one of two kernels. The paired kernel (two 128-row units per 512-thread
// workgroup, one workgroup per CU, stream-K key-range slots) wins when each launch slot has many
// key steps; with few steps per slot its per-segment prologue, partials and merge dominate and
// the 4-wavefront tile kernel (two workgroups per CU, split plan sized for one resident round)
// is faster. Measured on MI355X (H 12, KVH 2; us per call, tile / paired, and the host-bound
// steps per paired slot): 512 rows on a 1037 prefix 28.0 / 34.0 (2.4), 2048 on 0 39.6 / 43.3
// (12.2), 1024 on 0 21.8 / 28.9 (3.0), 2048 on 2048 67.8 / 65.7 (24.4), 2048 on 4096 99.6 / 89.7
// (36.6), 1856 on 6144 125.5 / 106.2 (44.6).
constexpr int kPairMinSlotSteps = 16;

bool pair_pays(const PairPlan& pl, int num_heads, int num_kv_heads, int max_query_len,
               int max_seq_len) {
  if (pl.seg_cap == 0) return true;                // no split: the paired kernel as is
  const int tr = pair_heads(num_heads, num_kv_heads) ? kTileRows : 2 * kTileRows;
  const int seq = max_seq_len > max_query_len ? max_seq_len : max_query_len;
  const int64_t bound = (int64_t)cdiv(max_query_len, tr) * cdiv(seq, kTileKeys);
  return bound >= (int64_t)kPairMinSlotSteps * pl.slots;
}

// Shared body of the prefill entry points. With `workspace` the head_dim 128 kernels may split
// long key ranges; a workspace smaller than the plan needs runs the paired kernel unsplit.
int prefill_launch(const void* q, int64_t q_stride_t, int64_t q_stride_h, void* out,
                   int64_t out_stride_t, int64_t num_tokens, const void* k_cache,
                   const void* v_cache, int64_t num_blocks, const int32_t* block_tables,
                   int64_t bt_stride, int32_t max_blocks_per_seq, const int32_t* seq_lens,
                   const int32_t* query_start_loc, int32_t num_seqs, int32_t num_decode,
                   int32_t max_query_len, int32_t max_seq_len, int32_t num_heads,
                   int32_t num_kv_heads, int32_t head_dim, float scale, void* workspace,
                   size_t workspace_bytes, void* stream) {
  TS_REQUIRE(num_seqs >= 0 && num_decode >= 0 && num_decode <= num_seqs, TS_ERR_INVALID_ARG,
             "prefill_attention: num_decode=%d num_seqs=%d", num_decode, num_seqs);
  const int P = num_seqs - num_decode;
  if (P == 0 || max_query_len <= 0) return TS_OK;
  TS_REQUIRE(q && out && k_cache && v_cache && block_tables && seq_lens && query_start_loc,
             TS_ERR_INVALID_ARG, "prefill_attention: null pointer argument");
  TS_REQUIRE(num_heads > 0 && num_kv_heads > 0 && num_heads % num_kv_heads == 0,
             TS_ERR_INVALID_ARG, "prefill_attention: num_heads=%d not a multiple of num_kv_heads=%d",
             num_heads, num_kv_heads);
  TS_REQUIRE(head_dim == 16 || head_dim == 32 || head_dim == 64 || head_dim == 128,
             TS_ERR_UNSUPPORTED, "prefill_attention: head_dim %d not in {16, 32, 64, 128}", head_dim);
  TS_REQUIRE(num_blocks > 0 && max_blocks_per_seq > 0 && bt_stride >= max_blocks_per_seq,
             TS_ERR_INVALID_ARG, "prefill_attention: bad block table");
  TS_REQUIRE(num_tokens > 0, TS_ERR_INVALID_ARG, "prefill_attention: num_tokens %lld",
             (long long)num_tokens);
  const int vec = head_dim >= 32 ? 8 : 4;
  TS_REQUIRE(q_stride_t % vec == 0 && q_stride_h % vec == 0 && out_stride_t % 4 == 0 &&
                 aligned(q, 2 * vec) && aligned(out, 8) && aligned(k_cache, 16) &&
                 aligned(v_cache, 16),
             TS_ERR_INVALID_ARG, "prefill_attention: misaligned q / out / caches");
  const hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const float sl2 = scale * kLog2eP;
  // The 4-wavefront tile kernel on a split plan, with its merge where the plan splits.
  auto launch_tiles = [&](auto dim, auto groups, TilePlan tp) {
    constexpr int D = decltype(dim)::value, KS = decltype(groups)::value;
    // head_dim 64 computes rows from 0 up to max_query_len rounded to the stream kernel's tiles
    // and any seq_len, whichever kernel runs; head_dim 128 the longest tiles of the launch
    const PrefillCaps caps =
        D == 64 ? PrefillCaps{cdiv(max_query_len, kPsRows) * kPsRows,
                              max_seq_len > max_query_len ? max_seq_len : max_query_len}
                : kNoCaps;
    if (tp.ws_bytes == 0) tp.smax = kUnsplit;         // unsplit: no tile leaves partials
    const int per_kvh = tp.slots * P * (num_heads / num_kv_heads);
    const int n_launch = 8 % num_kv_heads == 0 ? 8 * cdiv(per_kvh, 8 / num_kv_heads)
                                                : per_kvh * num_kv_heads;
    prefill_tile_kernel<D, KS><<<n_launch, kTileThreads, 0, s>>>(
        static_cast<const half_t*>(q), q_stride_t, q_stride_h, static_cast<half_t*>(out),
        out_stride_t, num_tokens, static_cast<const half_t*>(k_cache),
        static_cast<const half_t*>(v_cache), num_blocks, block_tables, bt_stride,
        max_blocks_per_seq, seq_lens, query_start_loc, num_decode, num_heads, num_kv_heads, sl2,
        tp.smax, tp.slots, P, caps, static_cast<float*>(workspace));
    if (tp.ws_bytes > 0)
      prefill_merge_kernel<D, KS><<<dim3(kMergeParts<D, KS> * cdiv(max_query_len, tile_rows(KS)), P,
                                          num_heads),
                                kTileThreads, 0, s>>>(
          static_cast<const float*>(workspace), static_cast<half_t*>(out), out_stride_t,
          num_tokens, max_blocks_per_seq, seq_lens, query_start_loc, num_decode, num_heads,
          tp.smax, tp.slots, caps);
  };
  if (head_dim == 64) {
    int cus = 0;
    if (device_cu_count(stream, &cus) != TS_OK) return TS_ERR_DEVICE;
    Plan64 pl = plan64(P, num_heads, num_tokens, max_query_len, max_seq_len, cus,
                       workspace != nullptr);
    if (pl.tile.ws_bytes > workspace_bytes || (pl.tile.ws_bytes > 0 && !aligned(workspace, 16)))
      pl = plan64(P, num_heads, num_tokens, max_query_len, max_seq_len, cus, false);
    const std::integral_constant<int, 64> d64;
    if (pl.ks != kStream64) {
      if (pl.ks == 2)
        launch_tiles(d64, std::integral_constant<int, 2>{}, pl.tile);
      else
        launch_tiles(d64, std::integral_constant<int, 1>{}, pl.tile);
      return check_launch("prefill_attention");
    }
  }
  if (head_dim == 128) {
    int cus = 0;
    if (workspace != nullptr && device_cu_count(stream, &cus) != TS_OK) return TS_ERR_DEVICE;
    PairPlan pl = pair_plan(P, num_heads, num_kv_heads, max_query_len, max_seq_len, cus,
                            workspace != nullptr);
    if (!pair_pays(pl, num_heads, num_kv_heads, max_query_len, max_seq_len)) {
      TilePlan tp = tile_plan(P, num_heads, head_dim, max_query_len, max_seq_len, cus, true);
      if (tp.ws_bytes <= workspace_bytes && (tp.ws_bytes == 0 || aligned(workspace, 16))) {
        launch_tiles(std::integral_constant<int, 128>{}, std::integral_constant<int, 1>{}, tp);
        return check_launch("prefill_attention");
      }
    }
    if (pl.ws_bytes > workspace_bytes || (pl.ws_bytes > 0 && !aligned(workspace, 16)))
      pl = pair_plan(P, num_heads, num_kv_heads, max_query_len, max_seq_len, cus, false);
    const bool heads = pair_heads(num_heads, num_kv_heads);
    const int per_kvh = pl.slots * P * (num_heads / num_kv_heads / (heads ? 2 : 1));
    const int n_launch = 8 % num_kv_heads == 0 ? 8 * cdiv(per_kvh, 8 / num_kv_heads)
                                                : per_kvh * num_kv_heads;
    prefill_pair_kernel<<<n_launch, kPairThreads, 0, s>>>(
        static_cast<const half_t*>(q), q_stride_t, q_stride_h, static_cast<half_t*>(out),
        out_stride_t, num_tokens, static_cast<const half_t*>(k_cache),
        static_cast<const half_t*>(v_cache), num_blocks, block_tables, bt_stride,
        max_blocks_per_seq, seq_lens, query_start_loc, num_decode, num_heads, num_kv_heads, sl2,
        pl.slots, pl.seg_cap, P, static_cast<float*>(workspace));
    if (pl.seg_cap > 0)
      prefill_pair_merge_kernel<<<dim3(4 * cdiv(max_query_len, kTileRows), P, num_heads),
                                  kTileThreads, 0, s>>>(
          static_cast<const float*>(workspace), static_cast<half_t*>(out), out_stride_t,
          num_tokens, max_blocks_per_seq, seq_lens, query_start_loc, num_decode, num_heads,
          num_kv_heads, pl.slots, pl.seg_cap);
    return check_launch("prefill_attention");
  }
  const dim3 grid((max_query_len + kPsRows - 1) / kPsRows, P, num_heads);
#define TS_PF_CASE(DD)                                                                            \
  case DD:                                                                                        \
    prefill_stream_kernel<DD, kPsWaves><<<grid, kPsWaves * 64, 0, s>>>(                           \
        static_cast<const half_t*>(q), q_stride_t, q_stride_h, static_cast<half_t*>(out),        \
        out_stride_t, num_tokens, static_cast<const half_t*>(k_cache),                           \
        static_cast<const half_t*>(v_cache), num_blocks, block_tables, bt_stride,                \
        max_blocks_per_seq, seq_lens, query_start_loc, num_decode, num_heads, num_kv_heads, sl2); \
    break;
  switch (head_dim) {
    TS_PF_CASE(16)
    TS_PF_CASE(32)
    TS_PF_CASE(64)
  }
#undef TS_PF_CASE
  return check_launch("prefill_attention");
}

}  // namespace

extern "C" size_t ts_prefill_workspace_bytes(int32_t num_prefill, int32_t num_heads,
                                             int32_t head_dim, int32_t max_query_len,
                                             int32_t max_seq_len, int32_t cu_count) {
  if (num_prefill <= 0 || num_heads <= 0 || max_query_len <= 0) return 0;
  if (head_dim == 64)
    return workspace64(num_prefill, num_heads, max_query_len, max_seq_len, cu_count);
  if (head_dim != 128) return 0;
  // The paired plan depends on whether the GQA group size is even (not an argument here), and
  // short splits take the tile plan instead: enough for every form.
  const size_t a = pair_plan(num_prefill, num_heads, 1, max_query_len, max_seq_len, cu_count,
                             true).ws_bytes;
  const size_t b = pair_plan(num_prefill, num_heads, num_heads, max_query_len, max_seq_len,
                             cu_count, true).ws_bytes;
  const size_t c = tile_plan(num_prefill, num_heads, head_dim, max_query_len, max_seq_len,
                             cu_count, true).ws_bytes;
  const size_t ab = a > b ? a : b;
  return ab > c ? ab : c;
}

extern "C" int ts_prefill_attention(const void* q, int64_t q_stride_t, int64_t q_stride_h,
                                    void* out, int64_t out_stride_t, int64_t num_tokens,
                                    const void* k_cache, const void* v_cache, int64_t num_blocks,
                                    const int32_t* block_tables, int64_t bt_stride,
                                    int32_t max_blocks_per_seq, const int32_t* seq_lens,
                                    const int32_t* query_start_loc, int32_t num_seqs,
                                    int32_t num_decode, int32_t max_query_len, int32_t num_heads,
                                    int32_t num_kv_heads, int32_t head_dim, float scale,
                                    void* stream) {
  ts::clear_error();
  return prefill_launch(q, q_stride_t, q_stride_h, out, out_stride_t, num_tokens, k_cache,
                        v_cache, num_blocks, block_tables, bt_stride, max_blocks_per_seq, seq_lens,
                        query_start_loc, num_seqs, num_decode, max_query_len, max_query_len,
                        num_heads, num_kv_heads, head_dim, scale, nullptr, 0, stream);
}

extern "C" int ts_prefill_attention_ws(const void* q, int64_t q_stride_t, int64_t q_stride_h,
                                       void* out, int64_t out_stride_t, int64_t num_tokens,
                                       const void* k_cache, const void* v_cache,
                                       int64_t num_blocks, const int32_t* block_tables,
                                       int64_t bt_stride, int32_t max_blocks_per_seq,
                                       const int32_t* seq_lens, const int32_t* query_start_loc,
                                       int32_t num_seqs, int32_t num_decode,
                                       int32_t max_query_len, int32_t max_seq_len,
                                       int32_t num_heads, int32_t num_kv_heads, int32_t head_dim,
                                       float scale, void* workspace, size_t workspace_bytes,
                                       void* stream) {
  ts::clear_error();
  return prefill_launch(q, q_stride_t, q_stride_h, out, out_stride_t, num_tokens, k_cache,
                        v_cache, num_blocks, block_tables, bt_stride, max_blocks_per_seq, seq_lens,
                        query_start_loc, num_seqs, num_decode, max_query_len, max_seq_len,
                        num_heads, num_kv_heads, head_dim, scale, workspace, workspace_bytes,
                        stream);
}
