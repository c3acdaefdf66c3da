// Attention tile planner: which (tree, row tile, cached-key range) units a pass
// runs and how split ranges merge. Host code, no device calls.
//
// Two rules share one implementation:
//   * reference rule  -- PlanOptions::reference(): the records are identical,
//     field for field, to what the reference's planner emits
//     (plan_tiles, src/model/impl/forest.h:1378-1433 without the sparse branch;
//      g4_plan_tiles, src/model/impl/gemma.h:77-116): 8-row tiles, every tree
//     gets the same split budget 256 / (groups * tiles), 32-key boundaries.
//   * balanced rule   -- PlanOptions::mi355x(): one chunk size for the whole
//     pass, derived from the pass's total key count, so every workgroup
//     streams about the same number of KV bytes whatever its sequence length
//     (the reference rule gives a 512-token and an 8192-token sequence the same
//     number of splits, which leaves most of 256 CUs idle while the longest
//     sequence finishes). Boundaries stay on page multiples.
// Only the algebra is contractual: the cached ranges of a tile group partition
// [k0, P), its batch ranges partition the batch keys from b0 on (one range - the
// last part's - unless the balanced rule cuts the batch keys too: `last` = e + 2
// ends a part's batch keys at row e of the tree, `last` = 1 leaves them open),
// parts merge in range order.
#pragma once

#include <algorithm>
#include <climits>
#include <cstdint>
#include <functional>
#include <limits>
#include <queue>
#include <vector>

#include "../../include/espetero_attn.h"
#include "../csrc/launch_shape.hpp"

namespace espetero::engine {

struct PlanOptions {
  int rows_per_tile = 8;    // query rows per tile
  int groups_target = 256;  // workgroups a few-tile pass is split up to
  int split = 512;          // reference rule: largest chunk a split tile is sized to; 0: never split
  int min_chunk = 32;       // fewest cached keys a split tile takes
  int granule = 32;         // split boundaries are multiples of this
  int max_splits = 64;      // parts per tile group
  int min_span = 64;        // shorter cached ranges are not split
  bool balanced = false;    // false: reference rule; true: equal keys per workgroup
  // Balanced rule on the tiled kernel (rows_per_tile > 32): groups_target is the number of workgroups
  // resident at once, and the chunk is the one whose workgroups, handed to those slots in the kernel's
  // dispatch order, finish earliest. item_steps: what a workgroup costs beside its key steps (set-up,
  // epilogue), in steps of `granule` keys.
  int item_steps = 0;
  int part_steps = 0;  // what a split part costs on top: its partial record written, read again and merged
  // Tiled kernel, balanced rule: a tile's batch keys are cut like its cached keys (a pass of fewer workgroups than
  // slots - one prompt's first chunk - is otherwise as long as its last tile, which scans every row of the chunk).
  // Off in mi355x(): measured on one 2048-row first chunk, 16 heads, the attention kernel gets shorter (head dim 256:
  // 80 -> 72 us, head dim 128: 42.5 -> 36.4 us) and the step with the merge of the partial records behind it does not
  // (79.5 -> 82.9 us, 42.0 -> 43.3 us).
  bool cut_batch = false;

  static PlanOptions reference() { return PlanOptions{}; }
  // rows: query rows per tile (decode 1..8 -> 8-row budget is irrelevant; prefill 64/128).
  static PlanOptions mi355x(int rows, int workgroups) {
    PlanOptions o;
    o.rows_per_tile = rows;
    o.groups_target = workgroups;
    o.split = 0;
    o.min_chunk = 64;
    o.granule = 32;
    o.max_splits = 256;
    o.min_span = 128;
    o.balanced = true;
    if (rows > 32) {  // tiled kernel: 64-key steps, and a split part must amortise its partial record
      o.granule = 64;
      o.min_chunk = 512;
      o.min_span = 1024;
      o.item_steps = 6;
      o.part_steps = 6;  // (8 before the merge of tiled passes got its own instantiation: config 3's four chunks 738.9 -> 736.2 us)
    }
    return o;
  }
};

struct AttnPlan {
  std::vector<esp_tree> trees;
  std::vector<esp_tile> tiles;
  std::vector<esp_combine> combine;
  int parts = 0;
  int rows_per_tile = 8;
};

// The kernel a pass is planned for, as far as a plan depends on it. family 0: not known.
struct PlanShape {
  int family = 0;      // kernel_family()
  int head_dim = 0;
  int Hkv = 0, G = 0;  // KV heads, query heads per KV head
};

// Of the layer's parameters; not known (also) where `groups` is not that kernel's count of workgroups per tile.
inline PlanShape plan_shape(const esp_attn_params* p, int groups, int rows_per_tile) {
  if (!p || p->Hkv <= 0 || p->H <= 0 || p->H % p->Hkv) return {};
  if (p->head_dim != 128 && p->head_dim != 256 && p->head_dim != 512) return {};  // no kernel serves it
  const int G = p->H / p->Hkv, family = esp::kernel_family(p->head_dim, rows_per_tile, G);
  if (groups != (family > 0 ? p->Hkv : p->H)) return {};
  return {family, p->head_dim, p->Hkv, G};
}

struct RowTile {
  int tree, r, k0, b0, span;
  int batch;  // batch keys the tile scans after its cached range (balanced rule: part of its work)
};

// Streaming kernel, balanced rule: the parts of every row tile of a pass. `room`: tiles resident at once (all the KV
// heads of a tile run side by side, so a tile stands for one workgroup on each of `groups` shares of the chip). `most_parts`:
// what esp_attn_forward_static has room for.
//
// What a split costs is worked out by running it: the tiles go to the compute units in the order the hardware will
// start them, two workgroups on one compute unit share what it can pull (36 GB/s, whether one or two ask), all of them
// together what memory gives (0.75 of that per unit), every workgroup has a fixed set-up and end, and a pass with any
// split tile a merge behind it: 60 KB and 4.6 us at 36 GB/s, here in keys. Against 61
// measured passes (16 to 96 ragged sequences, head dims 128 and 256, 24 to 258 tiles) this is right within 10 %. A pass
// that fills more than half of the chip with whole sequences gains from a split too: 48 sequences of 60 .. 3000 keys on
// 8 KV heads 72.5 us whole, 62.6 at 74 tiles.
// Where the kernel is not known neither is what a key costs: a pass that whole sequences fill less than half is then cut
// as evenly as fits, without weighing, and for the others the split target has to stand for the key. A target below what the
// chip holds of the kernel asks for so many tiles: such a pass is cut without weighing too.
template <typename PartsOf>
inline std::vector<int> stream_split(const std::vector<RowTile>& rts, const PlanOptions& o, const PlanShape& shape, int room,
                                     long long most_parts, const PartsOf& parts_of) {
  const int n = int(rts.size());
  const bool known = shape.family != 0;
  const int per_cu = !known              ? (o.groups_target >= 512 ? 2 : 1)
                     : shape.family > 0 ? esp::stream_workgroups_per_cu(shape.head_dim, shape.family)
                                        : esp::tiled_workgroups_per_cu(shape.head_dim);
  const bool even = !known || o.groups_target < esp::kComputeUnits * per_cu;
  const int cus = std::max(1, room / per_cu);
  // Two column tiles of 128 dims: a key takes its workgroup about twice as long as its bytes do. (One sequence of 300 keys,
  // 4 rows at 32 / 4 heads: 11.3 us in five parts, which keys of 512 bytes would refuse, 11.8 whole.)
  const int key_bytes = !known ? (per_cu == 2 ? 512 : 1024) : 4 * shape.head_dim * (shape.head_dim == 128 && shape.family == 2 ? 2 : 1);
  const double kFixed = 60000 / key_bytes, kMerge = 165600 / key_bytes;
  // Wavefront pairs of 512 dims reach less of memory together, and a record of theirs is four times a 128-dim one's: no
  // halves of a resident tile's share. (16 / 2 heads of 512: 130 sequences of 1000 .. 1500 keys 138 us at 255 tiles, 137 at
  // 385, 141 at 580; 100 of 60 .. 3000 111 us at 247 tiles, 126 at 369; 200 of them 238 us at 256, 285 whole.)
  const bool wide = known && shape.head_dim == 512;
  const double kMemory = wide ? 0.6 : 0.75;
  long long total = 0;
  for (const RowTile& rt : rts) total += rt.span + rt.batch;
  std::vector<int> ns(size_t(n), 1), best(size_t(n), 1);
  struct Item {
    bool last;
    int keys;
  };
  std::vector<Item> items;
  auto count_at = [&](long long chunk) {
    long long k = 0;
    for (const RowTile& rt : rts) k += parts_of(rt, chunk);
    return k;
  };
  struct Cu {
    double rem[2], since;
    int running;
  };
  std::vector<Cu> cu;
  std::vector<double> idle;
  constexpr double kNever = std::numeric_limits<double>::infinity();
  double least = kNever;
  // kNever for a split that is the best so far once more, or cannot end early enough by its keys or by its longest part alone.
  auto time_at = [&](long long chunk, double win) {
    items.clear();
    bool split = false;
    for (int i = 0; i < n; ++i) {
      const RowTile& rt = rts[size_t(i)];
      const int k = int(parts_of(rt, chunk));
      ns[size_t(i)] = k;
      split = split || k > 1;
      const int work = rt.span + rt.batch, step = ((work + k - 1) / k + o.granule - 1) / o.granule * o.granule;
      for (int p = 0; p + 1 < k && p * step < rt.span; ++p) items.push_back({false, std::min(step, rt.span - p * step)});
      items.push_back({true, std::max(0, work - (k - 1) * step)});
    }
    long long keys = 0, most = 0;
    for (const Item& x : items) keys += x.keys, most = std::max<long long>(most, x.keys);
    const double bound = std::max((double(keys) + kFixed * double(items.size())) / (kMemory * cus), double(most) + kFixed) + (split ? kMerge : 0);
    if (bound >= win * least || (least < kNever && ns == best)) return kNever;
    const bool one_round = int(items.size()) <= room;
    std::stable_sort(items.begin(), items.end(), [&](const Item& x, const Item& y) {
      if (one_round && x.last != y.last) return x.last;
      return x.keys > y.keys;
    });
    // Every compute unit's own clock advances with the bytes it may pull; the real time follows from how many pull. (Units
    // beyond the number of tiles get none: a target of any size is planned in the memory of the tiles.)
    const int used = int(std::min(size_t(cus), items.size()));
    cu.assign(size_t(used), Cu{{0, 0}, 0, 0});
    size_t next = 0;
    for (int s = 0; s < per_cu; ++s)
      for (int c = 0; c < used && next < items.size(); ++c) cu[size_t(c)].rem[cu[size_t(c)].running++] = items[next++].keys + kFixed;
    using Event = std::pair<double, int>;
    std::priority_queue<Event, std::vector<Event>, std::greater<Event>> q;
    auto next_end = [&](const Cu& x) { return x.since + (x.running == 2 ? 2 * std::min(x.rem[0], x.rem[1]) : x.rem[0]); };
    for (int c = 0; c < used; ++c)
      if (cu[size_t(c)].running) q.push({next_end(cu[size_t(c)]), c});
    idle.clear();
    while (!q.empty()) {
      const auto [at, c] = q.top();
      q.pop();
      Cu& x = cu[size_t(c)];
      if (x.running == 2) {
        const double d = std::min(x.rem[0], x.rem[1]);
        x.rem[0] = std::max(x.rem[0], x.rem[1]) - d;
      }
      --x.running;
      x.since = at;
      if (next < items.size()) x.rem[x.running++] = items[next++].keys + kFixed;
      if (x.running) q.push({next_end(x), c});
      else idle.push_back(at);
    }
    double t = 0, was = 0;
    size_t pulling = idle.size();
    for (double at : idle) {  // ascending: the queue hands events out in time order
      t += (at - was) / std::min(1.0, kMemory * cus / double(pulling--));
      was = at;
    }
    return t + (split ? kMerge : 0);
  };
  // The smallest chunk whose tiles are all resident at once (a pass that overshoots that by a few tiles pays a second
  // round for them), or no split where whole sequences already overfill the chip; any other candidate has to win by 5 %,
  // a margin for kernels whose workgroups pull less alone than the model's (two column tiles, wavefront pairs): no
  // split, and chunks of one and a half, three quarters and half of the pass's keys per resident tile.
  auto consider = [&](long long chunk, double win) {
    chunk = std::max<long long>(chunk, std::max(1, o.min_chunk));
    chunk = (chunk + o.granule - 1) / o.granule * o.granule;
    // Sequences that fill less than half of the chip are cut into as many tiles as are resident whatever their records take;
    // any other split (134 sequences at 16 / 2 heads of 512, 4 rows: 268 parts, 34 MB) stays within the library's own array.
    long long tiles = 0, parts = 0;
    for (const RowTile& rt : rts) {
      const long long k = parts_of(rt, chunk);
      tiles += k;
      parts += k > 1 ? k : 0;
    }
    if ((n > room / 2 || tiles > room) && parts > most_parts) return;
    const double t = time_at(chunk, win);
    if (t < win * least) least = t, best = ns;
  };
  const long long whole = total + o.min_chunk;
  if (n <= room) {
    long long lo = std::max(1, o.min_chunk / o.granule), hi = std::max<long long>(lo, (total + o.granule - 1) / o.granule + 1);
    while (lo < hi) {
      const long long mid = (lo + hi) / 2;
      if (count_at(mid * o.granule) <= room) hi = mid;
      else lo = mid + 1;
    }
    consider(lo * o.granule, 1);
    if (even && n <= room / 2) return best;
    consider(whole, 0.95);
  } else {
    // Handed out one by one, whole sequences end at most a full unit's last ones after an even share: often near enough as it is.
    long long most = 0;
    for (const RowTile& rt : rts) most = std::max<long long>(most, rt.span + rt.batch);
    const double even_share = (double(total) + kFixed * n) / cus;
    if (even_share + per_cu * (double(most) + kFixed) <= 1.1 * (even_share + kMemory * kMerge)) return best;
    consider(whole, 1);
  }
  // Where the compute units end together no other split does better; within 10 % of that none is tried.
  long long n_best = 0;
  for (int k : best) n_best += k;
  if (least > 1.1 * ((double(total) + kFixed * double(n_best)) / (kMemory * cus) + kMerge))
    for (const double share : {1.5, 0.75, 0.5})
      if (!wide || share > 0.5) consider((long long)(double(total) / room * share), 0.95);
  return best;
}

// groups: workgroups per tile (KV heads, or KV heads x head splits).
// window > 0 needs pos (4 ints per row, pos[4 * row] = position).
// params: the layer the pass is planned for (may be null: a plan that holds for any).
inline void plan_tiles(AttnPlan& A, int groups, int window, const int32_t* pos, const PlanOptions& o, const esp_attn_params* params = nullptr) {
  const PlanShape shape = plan_shape(params, groups, o.rows_per_tile);
  A.tiles.clear();
  A.combine.clear();
  A.parts = 0;
  A.rows_per_tile = o.rows_per_tile;
  const int R = o.rows_per_tile;
  std::vector<RowTile> rts;
  for (int ti = 0; ti < int(A.trees.size()); ++ti) {
    const esp_tree& t = A.trees[size_t(ti)];
    for (int r = 0; r < t.M; r += R) {
      int k0 = 0, b0 = 0;
      if (window > 0) {
        // The tile's earliest row bounds what any of its rows can still see:
        // cached key j sits at position j, root row j at P + j (gemma.h:88-94).
        int minpos = INT32_MAX;
        for (int i = r; i < std::min(t.M, r + R); ++i) minpos = std::min(minpos, pos[4 * (t.base + i)]);
        k0 = std::clamp(minpos - window + 1, 0, t.P);
        b0 = std::max(0, minpos - window + 1 - t.P);
      }
      // A causal tile scans the batch rows up to its own last row; one split part takes them all.
      const int batch = o.balanced ? std::max(0, std::min(t.M, r + R) - b0) : 0;
      rts.push_back({ti, r, k0, b0, t.P - k0, batch});
    }
  }
  const int n_tiles = int(rts.size());
  int budget = std::max(1, o.groups_target / std::max(1, groups * n_tiles));
  auto cuttable = [&](const RowTile& rt) { return rt.span + (o.cut_batch ? rt.batch : 0) >= o.min_span; };
  auto parts_of = [&](const RowTile& rt, long long chunk) {
    // (at least one: with min_span <= 0 a tile that sees no key at all may be asked for)
    return cuttable(rt) ? std::clamp<long long>((rt.span + rt.batch + chunk - 1) / chunk, 1, o.max_splits) : 1;
  };
  // Parts whose records fit esp_attn_forward_static's array beside what else such a pass keeps there. Where the layer is not
  // known (only the streaming rule asks then): of the largest records there are, 32 columns of 512 dims on every KV head.
  auto most_static_parts = [&] {
    int n_rows = 0;
    for (const esp_tree& t : A.trees) n_rows = std::max(n_rows, t.base + t.M);
    if (!shape.family) return (long long)(ESP_STATIC_SCRATCH_BYTES) / (32LL * 514 * 4 * std::max(1, groups));
    auto fits = [&](long long parts) {
      return esp::carve_workspace(shape.G * shape.Hkv, shape.Hkv, shape.head_dim, R, n_rows, parts).total <= ESP_STATIC_SCRATCH_BYTES;
    };
    long long lo = 0, hi = 1 << 20;
    while (lo < hi) {
      const long long mid = (lo + hi + 1) / 2;
      if (fits(mid)) lo = mid;
      else hi = mid - 1;
    }
    return lo;
  };
  // Balanced rule: the batch keys count as work of the last part, so the cached range is
  // cut into parts of (cached + batch) / ns keys and the last part keeps what is left.
  auto step_of = [&](const RowTile& rt, int ns) {
    const int per = (rt.span + rt.batch + ns - 1) / ns;
    return (per + o.granule - 1) / o.granule * o.granule;
  };
  // A tile's ns parts, batch keys uncut: all but the last are `step` cached keys on page multiples; the last keeps the
  // rest of the cached range (possibly nothing) and the batch keys.
  auto for_cached_parts = [&](const RowTile& rt, int ns, auto&& part) {
    const int P = A.trees[size_t(rt.tree)].P, step = step_of(rt, ns);
    int k = rt.k0;
    for (int p = 0; p < ns; ++p) {
      const bool is_last = p + 1 == ns;
      int k1 = P;
      if (!is_last) {
        k1 = std::min(P, k + step);
        if (k1 < P) k1 = std::min(P, std::max(k + o.granule, k1 / o.granule * o.granule));
        if (k1 == k) continue;  // the cached range ran out: the batch keys alone fill the last part
      }
      part(k, k1, is_last);
      k = k1;
    }
  };
  std::vector<int> ns_of;  // balanced rule: parts of every row tile, once chosen
  std::vector<int> emit(size_t(n_tiles), 0);  // row tiles in the order their records are written
  for (int i = 0; i < n_tiles; ++i) emit[size_t(i)] = i;
  if (o.balanced && o.item_steps > 0) {
    // Tiled kernel. A pass is tiles x groups workgroups of unequal length (a causal chunk's later tiles
    // see more keys) on groups_target slots; the hardware hands the next workgroup to the first free slot,
    // in the kernel's dispatch order (tile records last to first, the groups of a record together). The
    // time of the pass is when the last slot finishes, so the split is chosen by running that hand-out
    // for every candidate: a few long workgroups leave slots idle at the end, many short ones pay their
    // set-up, partial records and merge more often.
    const int slots = std::max(1, o.groups_target);
    long long max_work = 1;
    for (const RowTile& rt : rts) max_work = std::max<long long>(max_work, rt.span + rt.batch);
    const long long c_lo = std::max(1, o.min_chunk / o.granule), c_hi = (max_work + o.granule - 1) / o.granule;
    // A mixed pass: decoding sequences or drafts ride with prompt chunks, in a grid that fills the slots or whose short tiles
    // the kernel packs. It is run as the kernel runs it: workgroups by the kernel's own rule (the others of a packed tile end at
    // once), records in an order of their own, and each part at what the merge dispatch costs for its record, 0.6 steps
    // (passes of chunks alone have few). Of 19 such passes on 4 to 32 KV heads, each timed whole and in up to 21 cuts, this picks
    // one that takes 5 % longer than the best that fits the library's own array, in geometric mean, 21 % at worst (it does not
    // know that two workgroups slow each other on a compute unit). 512 rows over 2048 keys beside 12 sequences of 200 .. 6000,
    // attention and merge: 90 us whole -> 60 (32 / 4 heads), 90 -> 61 (40 / 8; 56 in 20 parts, which do not fit), 130 -> 79
    // (32 / 32, where nothing is packed). Passes below that fill the chip less
    // than once and are cut for that already (322 and 124 rows beside 13 sequences, 8 / 2 heads of 256: 56 us, 63 as mixed), and
    // a chunk's short remainder counted as packed was 2 % slower (eight chunks of 1032 rows over 15360 keys at 16 / 8 heads of
    // 256: 2577 -> 2630 us): everything else is planned as if nothing were packed, as is every pass whose layer is not known.
    const long long grid = 1LL * n_tiles * groups;
    auto live_rows = [&](const RowTile& rt) { return std::min(R, A.trees[size_t(rt.tree)].M - rt.r); };
    auto is_short = [&](const RowTile& rt) { return live_rows(rt) <= 16 && esp::tiled_packs(shape.head_dim, live_rows(rt), shape.G, LLONG_MAX); };
    const bool fills = shape.family < 0 && (grid >= slots || grid > esp::kComputeUnits);
    const bool by_tree = fills && std::any_of(rts.begin(), rts.end(), is_short);
    bool mixed = fills && std::any_of(rts.begin(), rts.end(), [&](const RowTile& rt) { return rt.r == 0 && is_short(rt); });
    // Workgroups that work on one part of a tile in a pass of so many records.
    auto groups_of = [&](const RowTile& rt, long long records) {
      return mixed && esp::tiled_packs(shape.head_dim, live_rows(rt), shape.G, records * groups) ? shape.Hkv : groups;
    };
    // Records are handed out last to first, and trees in the order of the pass put a long chunk's parts behind those of
    // decoding sequences, beside which they end alone. In a pass with short tiles trees go by their longest part, longest last;
    // the tiles of a tree stay together in their order, since those that run side by side share the tree's keys. (Those three
    // passes, in 20 parts, by tree and in the pass's order: 60 and 70, 52 and 55, 85 and 98 us. Chunks of 445, 453 and 396 rows on a
    // period of five sliding layers and a full one, 24 / 4 heads of 256: 609 and 633 us. Records sorted one by one, in a pass of
    // the eight chunks: 2577 -> 2943 us.)
    std::vector<int> longest(A.trees.size(), 0);
    auto order_records = [&](const std::vector<int>& ns_v) {
      for (int i = 0; i < n_tiles; ++i) emit[size_t(i)] = i;
      if (!by_tree) return;
      std::fill(longest.begin(), longest.end(), 0);
      for (int i = 0; i < n_tiles; ++i) {
        int& part = longest[size_t(rts[size_t(i)].tree)];
        part = std::max(part, (rts[size_t(i)].span + rts[size_t(i)].batch) / ns_v[size_t(i)]);
      }
      std::stable_sort(emit.begin(), emit.end(), [&](int x, int y) {
        const int tx = rts[size_t(x)].tree, ty = rts[size_t(y)].tree;
        return longest[size_t(tx)] != longest[size_t(ty)] ? longest[size_t(tx)] < longest[size_t(ty)] : tx < ty;
      });
    };
    auto parts_in = [](const std::vector<int>& ns_v) {
      long long k = 0;
      for (int ns : ns_v) k += ns > 1 ? ns : 0;
      return k;
    };
    // In tenths of a step.
    auto finish_time = [&](const std::vector<int>& ns_v) {
      order_records(ns_v);
      long long records = 0;
      for (int ns : ns_v) records += ns;
      // (when, how many slots): the workgroups of a record are alike and mostly take slots that are.
      using Free = std::pair<long long, int>;
      std::priority_queue<Free, std::vector<Free>, std::greater<Free>> free_at;
      free_at.push({0, slots});
      long long end = 0;
      for (int i = n_tiles - 1; i >= 0; --i) {
        const int at = emit[size_t(i)];
        const RowTile& rt = rts[size_t(at)];
        const long long work = rt.span + rt.batch;
        const long long ns = ns_v[size_t(at)];
        const long long per = (work + ns - 1) / ns;
        const int workgroups = groups_of(rt, records);
        for (long long p = ns - 1; p >= 0; --p) {  // a record's parts in reverse too
          const long long keys = std::min(per, work - p * per);
          const long long cost = o.item_steps + (ns > 1 ? o.part_steps : 0) + (std::max<long long>(keys, 0) + o.granule - 1) / o.granule;
          for (int left = workgroups; left > 0;) {
            const Free f = free_at.top();
            const int take = std::min(left, f.second);
            free_at.pop();
            if (f.second > take) free_at.push({f.first, f.second - take});
            free_at.push({f.first + cost, take});
            end = std::max(end, f.first + cost);
            left -= take;
          }
        }
      }
      return 10 * end + (mixed ? 6 * parts_in(ns_v) : 0);
    };
    // The split that finishes first, of those with no more than `most` parts.
    std::vector<int> cand;
    auto choose = [&](long long most) {
      cand.assign(size_t(n_tiles), 1);
      ns_of = cand;
      long long best = finish_time(cand);
      auto consider = [&] {
        if (parts_in(cand) > most) return;
        const long long t = finish_time(cand);
        if (t < best) best = t, ns_of = cand;
      };
      long long items = 0;
      for (const RowTile& rt : rts) items += groups_of(rt, n_tiles);
      const long long rounds = items / slots;
      // Fewer workgroups than slots (with cut_batch: no more than slots): one chunk for every tile, the chunks that cut the longest tile into 2 .. 8
      // parts (fewer parts first: ties keep them). With a round or more of whole workgroups such a split was
      // measured slower than none (two workgroups share a compute unit and the older one is served first, so the
      // slots are less alike than this hand-out takes them to be).
      auto cut_at = [&](long long c) {
        for (int i = 0; i < n_tiles; ++i) cand[size_t(i)] = int(parts_of(rts[size_t(i)], std::max(c_lo, c) * o.granule));
        consider();
      };
      for (int parts = 2; parts <= 8 && !mixed && (rounds == 0 || (o.cut_batch && items <= slots)); ++parts) cut_at((c_hi + parts - 1) / parts);
      // A mixed pass may end on one long sequence whatever the rounds, and between two of those chunks lie many cuts of it.
      for (int part = 15; part >= 2 && mixed; --part) cut_at((c_hi * part + 15) / 16);
      // A round or more, and some workgroups over (640 on 512 slots): those would run nearly alone at the end.
      // Only the tiles with the least work are split, just enough of them that the whole ones fill whole rounds,
      // and their parts fill the slots beside and behind those; the tile dispatched last gets the most parts, so
      // that the pass ends on short workgroups. (Measured on 2048-row causal chunks over 2048 .. 6144 cached keys:
      // 5 to 8 % faster than unsplit; splitting fewer tiles than that, so that some whole ones still spill into
      // another round, was 3 to 6 % slower.)
      if (rounds >= 1 && items % slots != 0) {
        std::vector<int> order(size_t(n_tiles), 0);  // tiles by work, least first (ties: dispatched last first)
        for (int i = 0; i < n_tiles; ++i) order[size_t(i)] = i;
        std::stable_sort(order.begin(), order.end(), [&](int x, int y) {
          return rts[size_t(x)].span + rts[size_t(x)].batch < rts[size_t(y)].span + rts[size_t(y)].batch;
        });
        int n_tail = 0;
        for (long long over = items - rounds * slots; over > 0; ++n_tail) over -= groups_of(rts[size_t(order[size_t(n_tail)])], n_tiles);
        for (int most = 3; most <= 6; ++most) {  // parts of the tile with the least work; the others one fewer each, down to 2
          std::fill(cand.begin(), cand.end(), 1);
          bool any = false;
          for (int j = 0; j < n_tail; ++j) {
            const RowTile& rt = rts[size_t(order[size_t(j)])];
            const long long cap = std::min<long long>((rt.span + rt.batch) / std::max(1, o.min_chunk), o.max_splits);
            const int want = std::max(2, most - j);
            const int ns = rt.span >= o.min_span ? int(std::min<long long>(want, cap)) : 1;
            cand[size_t(order[size_t(j)])] = std::max(1, ns);
            any = any || ns > 1;
          }
          if (!any) break;
          consider();
        }
      }
    };
    choose(LLONG_MAX);
    // A mixed pass leaves slots for more parts than it would be cut into with nothing packed, and a part's record has room for a
    // whole tile (22 parts at 32 / 4 heads: 47 MB). What esp_attn_forward_static took that way it still takes.
    if (const long long room = most_static_parts(); mixed && parts_in(ns_of) > room) {
      mixed = false;
      choose(LLONG_MAX);
      mixed = true;
      choose(std::max(room, parts_in(ns_of)));
    }
    // A pass of few workgroups, at most one for two compute units, that nothing has cut so far - behind a window, or behind few keys - ends
    // with its longest tile while the rest of the chip stands idle: its tiles are cut until the parts fill the chip once, as long as
    // that is shorter with the merge's dispatch and the records there and back. In steps of 64 keys of the longest part, of the parts as they
    // are emitted: 2.5 for the merge and 0.6 for each MB of records at 128 dims (where a step behind a window counts 1.4), 4.5 and 0.15 at
    // 256, 2 and 0.15 at 512. Fitted to 217 passes of 40 .. 1900 rows timed whole and in every even cut, 1295 plans: what it picks takes
    // 1.6 % longer than the best of them in geometric mean, 18 % at worst, never more than 2.5 % longer than the whole pass, which takes
    // 24 % more than the best. The last part of a tile may hold its batch keys alone: 960 keys + 100 rows, 16 / 8 heads of 256, 37.1 us
    // whole, 26.0 in five parts and those, 27.6 in the most parts that all have cached keys. No tile in more than eight: nine cost the merge
    // another 12 us there. Not beyond what the rule above has cut (100 rows over 6871 keys 40.3 in its eight parts, 42.8 in fourteen).
    // Passes with decoding rows are left to the rules above, and whatever is planned fits esp_attn_forward_static.
    if (shape.family < 0 && !o.cut_batch && parts_in(ns_of) == 0 && grid * 2 <= esp::kComputeUnits && slots >= esp::kComputeUnits && o.part_steps > 0 &&
        std::none_of(rts.begin(), rts.end(), [&](const RowTile& rt) { return rt.r == 0 && live_rows(rt) <= 16; })) {
      const double merge = shape.head_dim == 128 ? 2.5 : shape.head_dim == 256 ? 4.5 : 2.0;
      const double per_mb = shape.head_dim == 128 ? 0.6 : 0.15;
      const long long room = most_static_parts();
      long long parts = 0, tiles = 0;  // of the plan priced last
      auto price = [&](const std::vector<int>& ns_v) {
        long long steps = 0, rows = 0;
        parts = 0, tiles = n_tiles;
        for (int i = 0; i < n_tiles; ++i) {
          const RowTile& rt = rts[size_t(i)];
          int used = 0;
          for_cached_parts(rt, ns_v[size_t(i)], [&](int k, int k1, bool last) {
            steps = std::max(steps, (long long)(k1 - k + (last ? rt.batch : 0) + o.granule - 1) / o.granule);
            ++used;
          });
          if (ns_v[size_t(i)] <= 1) continue;
          parts += used, tiles += used - 1, rows += used * live_rows(rt);
        }
        return double(steps) * (shape.head_dim == 128 && window > 0 ? 1.4 : 1.0) + (parts ? merge + per_mb * 4e-6 * double(rows) * groups * shape.head_dim : 0);
      };
      double best = price(ns_of);
      // The limits a caller sets bind here at a quarter: parts of 128 keys and ranges of 256 with the tuned ones.
      const int min_step = std::max(2 * o.granule, o.min_chunk / 4), min_span = std::max(1, o.min_span / 4);
      for (long long c = c_hi - 1; c >= 2; c -= std::max<long long>(1, c_hi / 32)) {
        const long long chunk = c * o.granule;
        for (int i = 0; i < n_tiles; ++i) {
          const RowTile& rt = rts[size_t(i)];
          int ns = int(std::clamp<long long>((rt.span + rt.batch + chunk - 1) / chunk, 1, rt.span >= min_span ? std::min(o.max_splits, 8) : 1));
          while (ns > 1 && step_of(rt, ns) < min_step) --ns;
          cand[size_t(i)] = ns;
        }
        const double t = price(cand);
        if (tiles * groups > esp::kComputeUnits || parts > room) break;
        if (t < best) best = t, ns_of = cand;
      }
    }
    order_records(ns_of);
  } else if (o.balanced && n_tiles > 0) {
    ns_of = stream_split(rts, o, shape, std::max(1, o.groups_target / std::max(1, groups)), most_static_parts(), parts_of);
  }
  for (const int index : emit) {
    const RowTile& rt = rts[size_t(index)];
    const esp_tree& t = A.trees[size_t(rt.tree)];
    const int span = rt.span;
    int ns = 1;
    if (!ns_of.empty()) {
      ns = ns_of[size_t(index)];
    } else if (!o.balanced && budget > 1 && span >= o.min_span) {
      if (o.split > 0) {
        const int chunk =
            std::max(std::max(32, o.min_chunk),
                     std::min(o.split, ((span + budget - 1) / budget + o.granule - 1) / o.granule * o.granule));
        ns = std::min({(span + chunk - 1) / chunk, budget, o.max_splits});
      }
    }
    // Balanced rule: the tile carries its tree's block-list offset (pad = table + 1), which
    // saves the kernels a dependent load; the reference rule leaves pad 0 as the reference does.
    const int pad = o.balanced ? t.table + 1 : 0;
    if (ns <= 1) {
      A.tiles.push_back({rt.tree, t.base + rt.r, rt.k0, t.P, -1, 1, rt.b0, pad});
      continue;
    }
    const int step = step_of(rt, ns);
    const int part0 = A.parts;
    int used = 0;
    if (o.balanced && o.cut_batch && span < (ns - 1) * step) {
      // Some cut falls among the batch keys: walk cached keys [k0, P) and then batch rows [b0, b0 + batch) in parts of
      // `step`, cached cuts on page multiples, batch cuts on multiples of the granule in the tree's rows. A part that
      // ends among the batch rows says where (`last` = its last row + 2); the last part's batch range stays open, so
      // rows that see beyond their own tile (ancestors, image spans) find those keys there.
      const int b_end = rt.b0 + rt.batch;  // one past the tile's last row
      int k = rt.k0, b = rt.b0;
      for (int p = 0; p < ns && (k < t.P || b < b_end); ++p) {
        const bool is_last = p + 1 == ns;
        int k1 = t.P, b1 = b_end;
        if (!is_last) {
          int room = step;
          if (k < t.P) {
            k1 = std::min(t.P, k + room);
            if (k1 < t.P) k1 = std::min(t.P, std::max(k + o.granule, k1 / o.granule * o.granule));
            room -= k1 - k;
          }
          if (k1 < t.P) {
            b1 = b;  // all of it cached keys
          } else {
            b1 = std::min(b_end, b + std::max(room, 0));
            if (b1 < b_end) b1 = std::min(b_end, std::max(b + (k1 > k ? 0 : o.granule), b1 / o.granule * o.granule));
            if (b1 < b) b1 = b;
          }
        }
        if (k1 == k && b1 == b) continue;
        const bool rest = b1 >= b_end;  // nothing left for a later part: this one is the group's last
        const int last = b1 > b ? (rest ? 1 : b1 + 1) : (rest && k1 >= t.P ? 1 : 0);
        A.tiles.push_back({rt.tree, t.base + rt.r, k, k1, A.parts++, last, b, pad});
        k = k1;
        b = b1;
        ++used;
        if (rest && k >= t.P) break;
      }
      if (used == 1) {  // nothing was cut after all
        A.tiles.back().part = -1;
        --A.parts;
        continue;
      }
    } else if (o.balanced) {
      for_cached_parts(rt, ns, [&](int k, int k1, bool last) {
        A.tiles.push_back({rt.tree, t.base + rt.r, k, k1, A.parts++, last ? 1 : 0, rt.b0, pad});
        ++used;
      });
    } else {
      for (int k = rt.k0; k < t.P; k += step, ++used) {
        const int k1 = std::min(t.P, k + step);
        A.tiles.push_back({rt.tree, t.base + rt.r, k, k1, A.parts++, k1 >= t.P ? 1 : 0, rt.b0, pad});
      }
    }
    A.combine.push_back({t.base + rt.r, std::min(R, t.M - rt.r), part0, used});
  }
  // Streaming kernel, balanced rule: the hardware starts the workgroups in record order over a few microseconds. Where
  // all of them are resident at once the tiles that own their tree's batch keys go first - behind their stream of
  // cached keys they have a serial tail (the batch rows through the masked path) that the others' streaming then
  // covers - and the rest follow by cached range, longest first. (Measured on the batched decode of 16 ragged
  // sequences: 26.6 -> 25.8 us; with the owners of the batch keys last instead, 26.9 us.) Where there are more, the
  // longest go first whatever they own, so that the pass ends on short ones (48 ragged sequences, 74 tiles of 64
  // resident: 67.3 -> 62.6 us). The records' partial-record indices stay as assigned, so the merge order does not change.
  if (o.balanced && o.item_steps == 0) {
    const bool one_round = int(A.tiles.size()) <= std::max(1, o.groups_target / std::max(1, groups));
    std::stable_sort(A.tiles.begin(), A.tiles.end(), [&](const esp_tile& x, const esp_tile& y) {
      if (one_round && x.last != y.last) return x.last > y.last;
      return (x.k1 - x.k0) > (y.k1 - y.k0);
    });
  }
}

}  // namespace espetero::engine
