// Host-side work planning of the forward launches (no device code): the
// block height the launcher picks, the split-KV plan and the XCD placement
// table (declared in fa_fwd_kernel.h).  Pure host C++ so it can be built and
// checked on the CPU, including under AddressSanitizer.
//
// The reference launches one workgroup per q-tile
// (python/flash_attention_runtime/_ext.cu:96-102); these plans have no
// counterpart there.
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <functional>

#include "fa_fwd_kernel.h"

namespace fa {

int block_rows(const KernelArgs& a) {
  // The choice launch_causal makes.  Causal bf16 takes 8-wave workgroups on
  // long rows only where the 4-wave grid would be split: same box, against
  // 4 waves, B1 H2 N8192 +33 % (its split plan); but B1 H4 N8192 D64 (pair
  // mode) -4.9 %, B1 H8 N8192 (placement table) -2.9 %, B2 H32 N8192 (C4)
  // -0.7...0 %, and +1...+2 % for B2 H8 N8192 and B1 H16 N16384.
  if (a.causal) {
    if (a.seq_len < kWideCausalMinSeq) return 128;
    const int64_t tiles128 = (int64_t)a.batch * a.heads * ((a.seq_len + 127) / 128);
    return (!a.bf16 || tiles128 < kWideCausalBf16MaxTiles) ? 256 : 128;
  }
  return a.seq_len >= kWideMinSeq ? 256 : 128;
}

namespace {

constexpr int kKeyTile = 64;  // keys per K/V tile (Tile<D>::BN)
constexpr int kMaxTiles = kMaxSplitItems * 256 / kKeyTile;  // key tiles of a row that may be split
constexpr int kMaxCusPerXcd = 128;  // modelled (ChunkCost); an MI355X has 32

// Key tiles of q-tile qb.
int q_tile_tiles(const KernelArgs& a, int BM, int qb) {
  const int kv = a.causal ? std::min(a.seq_len, (qb + 1) * BM) : a.seq_len;
  return (kv + kKeyTile - 1) / kKeyTile;
}

// Workgroup slots of the machine: two 4-wave workgroups or one 8-wave
// workgroup per CU.
int64_t workgroup_slots(int BM, int compute_units) {
  return (int64_t)compute_units * (BM == 128 ? 2 : 1);
}

// Whether splitting key ranges pays on the grid of block_rows(a)-row q-tiles;
// *total_tiles is its number of key tiles over all q-tiles.
bool split_pays(const KernelArgs& a, int compute_units, double* total_tiles) {
  const int BM = block_rows(a);
  const int nq = (a.seq_len + BM - 1) / BM;
  if (nq > kMaxSplitItems) return false;
  // The unsplit grid finishes no earlier than its longest q-tile (t_max key
  // tiles) and no earlier than the total load over the machine's throughput.
  // A CU running one 4-wave workgroup alone already reaches ~90 % of its
  // two-workgroup throughput (measured: 1.14 us per 128x64 tile alone, 2.1 us
  // each for two), so the throughput bound counts 1.1 workgroups per CU for
  // 4-wave kernels.  Split only when the longest q-tile clearly dominates
  // that bound: the partials cost an fp32 write and read of O per chunk,
  // which ate the whole gain at B1 H16 N3000 causal (bound ratio 1.4) and
  // left +11 % at H8 (2.8) and +50 % at B1 H4 N8192 causal (3.9).
  int64_t sum = 0;
  int t_max = 0;
  for (int qb = 0; qb < nq; ++qb) {
    const int t = q_tile_tiles(a, BM, qb);
    sum += t;
    t_max = std::max(t_max, t);
  }
  *total_tiles = (double)sum * a.batch * a.heads;
  const double bound = *total_tiles / ((double)compute_units * (BM == 128 ? 1.1 : 1.0));
  return t_max > 1.5 * bound + 8.0;
}

// Chunks of a split: at most S key tiles each (S = 0: no split).
struct Chunks {
  bool pays = false;  // split_pays
  int average = 0;    // key tiles per workgroup slot
  int S = 0;
  int64_t bytes = 0;  // of the partials
};

// Chunks of q-tile qb.
int q_tile_chunks(const KernelArgs& a, int BM, int qb, int S) {
  return std::min(255, (q_tile_tiles(a, BM, qb) + S - 1) / S);
}

// Key tiles of chunk c of nch of a q-tile of T tiles (the kernel's t_begin and t_end).
int chunk_tiles(int c, int nch, int T) {
  return (int)((int64_t)(c + 1) * T / nch) - (int)((int64_t)c * T / nch);
}

// Items per (batch, head) with chunks of at most S tiles; *n_slots of them
// leave partials.  Neither rises with S.
int count_items(const KernelArgs& a, int BM, int nq, int S, int* n_slots) {
  if (!a.causal) {  // every q-tile alike
    const int nch = q_tile_chunks(a, BM, 0, S);
    *n_slots = nch > 1 ? nq * nch : 0;
    return nq * nch;
  }
  int items = 0;
  *n_slots = 0;
  for (int qb = 0; qb < nq; ++qb) {
    const int nch = q_tile_chunks(a, BM, qb, S);
    items += nch;
    if (nch > 1) *n_slots += nch;
  }
  return items;
}

int64_t partial_bytes(const KernelArgs& a, int BM, int64_t n_slots) {
  // Partial O (fp32) then (m, l, lr, unused) per row of every slot.
  return (int64_t)a.batch * a.heads * n_slots * BM * (a.head_dim * 4 + 16);
}

// Modelled time of a split launch and its merge, in key tiles of a workgroup:
// the last CU's load when each XCD hands out its run of items (head after
// head, each longest first) to its CUs in order, + 10 per partial slot per CU
// (written, read and merged) + 3/4 per four chunks of a row (the merge reads
// four at a time).  Two 4-wave workgroups of a CU run at 1.1 times the rate of
// one.  The constants are a fit to both rules' times on 1555 plans (H = 1...40,
// N = 500...32700, both head dims and types): of the two it picks the slower
// one by more than 2 % on 23 of them, by more than 5 % on 2 (both within the
// spread of their own runs).
struct ChunkCost {
  const KernelArgs& a;
  int compute_units, BM;
  int lens[kMaxSplitItems], n = 0;  // items of a head, longest first
  double partials;                  // the cost of the partials and the merge

  ChunkCost(const KernelArgs& args, int cus, int bm, int nq, int S)
      : a(args), compute_units(cus), BM(bm) {
    // T tiles in nch chunks: T % nch of T / nch + 1 tiles, the rest of T / nch.
    int count[kMaxTiles + 2] = {}, longest = 0, n_slots = 0;
    const int distinct = a.causal ? nq : 1, alike = a.causal ? 1 : nq;
    for (int qb = 0; qb < distinct; ++qb) {
      const int T = q_tile_tiles(a, BM, qb), nch = q_tile_chunks(a, BM, qb, S);
      const int len = T / nch, more = T - len * nch;
      count[len + 1] += alike * more;
      count[len] += alike * (nch - more);
      longest = std::max(longest, len + (more > 0));
      if (nch > 1) n_slots += alike * nch;
    }
    for (int l = longest; l > 0; --l)
      for (int i = 0; i < count[l]; ++i) lens[n++] = l;
    const int chunks = (q_tile_tiles(a, BM, nq - 1) + S - 1) / S;
    partials = 10.0 * (double)n_slots * a.batch * a.heads / compute_units +
               0.75 * ((chunks + 3) / 4);
  }
  int64_t items() const { return (int64_t)a.batch * a.heads * n; }
  double rate() const { return BM == 128 && items() > compute_units ? 1.1 : 1.0; }
  // No less than this, and exactly this with a CU for each item.
  double least() const {
    int64_t sum = 0;
    for (int i = 0; i < n; ++i) sum += lens[i];
    const double mean = (double)sum * a.batch * a.heads / compute_units / rate();
    return partials + (items() <= compute_units ? lens[0] : std::max((double)lens[0], mean));
  }
  // The cost, or any value above `limit` once it is known to exceed that.
  double cost(double limit = INFINITY) const {
    if (items() <= compute_units || least() > limit) return least();
    const int cpx = std::max(1, std::min(compute_units / 8, kMaxCusPerXcd));
    const int64_t per = items() / 8, more = items() % 8;
    int worst = 0, starts[8];
    int64_t first = 0;
    for (int x = 0; x < 8 && partials + worst / rate() <= limit; ++x) {
      const int64_t count = per + (x < more ? 1 : 0);
      int at = starts[x] = (int)(first % n);
      first += count;
      // XCDs whose run starts at the same item do alike (the first `more`
      // XCDs, with an item more each, and the others apart).
      const int* same = starts + (x < more ? 0 : more);
      if (std::find(same, (const int*)starts + x, at) != starts + x) continue;
      int cu[kMaxCusPerXcd];  // a heap of the CUs' loads, the least loaded first
      for (int64_t i = 0; i < count; ++i) {
        const int len = lens[at];
        if (++at == n) at = 0;
        if (i < cpx) {
          cu[i] = len;
          if (i == cpx - 1) std::make_heap(cu, cu + cpx, std::greater<int>());
          worst = std::max(worst, len);
          continue;
        }
        const int v = cu[0] + len;
        int k = 0;  // v sinks from the root
        for (int c = 1; c < cpx; c = 2 * k + 1) {
          if (c + 1 < cpx && cu[c + 1] < cu[c]) ++c;
          if (cu[c] >= v) break;
          cu[k] = cu[c];
          k = c;
        }
        cu[k] = v;
        worst = std::max(worst, v);
      }
    }
    return partials + std::max((double)lens[0], worst / rate());
  }
};

// A split's chunks by the first rule of choose_chunks.
Chunks average_chunks(const KernelArgs& a, int compute_units) {
  Chunks ch;
  double total = 0.0;
  ch.pays = split_pays(a, compute_units, &total);
  if (!ch.pays) return ch;
  const int BM = block_rows(a);
  const int nq = (a.seq_len + BM - 1) / BM;
  ch.average = (int)std::ceil(total / (double)workgroup_slots(BM, compute_units));
  int S = std::max(8, ch.average), n_slots = 0;
  while (count_items(a, BM, nq, S, &n_slots) > kMaxSplitItems) S *= 2;
  if (n_slots == 0) return ch;  // every q-tile whole
  ch.S = S;
  ch.bytes = partial_bytes(a, BM, n_slots);
  return ch;
}

// The chunk length of a split, the better of two by ChunkCost:
//  * about the average load of a workgroup slot (8 tiles at least), doubled
//    while the items exceed their table (average_chunks);
//  * the shortest (from 4 tiles on) with which all items run at once, one per
//    slot: the launch takes one chunk's time, and no second round of a few
//    items follows a full one.
// us, first rule / second: causal B1 H2 N8192 D128 bf16 56.2 / 46.1 (34 tiles
// a chunk on 156 of 256 CUs; 19 on 254), H1 N16384 169 / 119, H1 N8192 D64
// 42.2 / 29.0.  But with nearly as many q-tiles as slots the second's chunks
// are nearly whole q-tiles: fp16 D64 H5 N12000 146 / 166 (88 tiles, 172), H6
// N10000 133 / 148; and where the first's items already run at once, one to a
// CU, it only adds partials: H4 N2048 D128 20.9 / 23.4, H20 N1000 D64 16.7 /
// 19.2.
void choose_chunks(const KernelArgs& a, int compute_units, Chunks* ch) {
  // Problems whose partials exceed the static scratch under the first rule
  // keep its plan, and no other may exceed it: fa_fwd_scratch refuses them.
  // So do grids of more q-tiles than slots, which no S runs at once.
  const int BM = block_rows(a);
  const int nq = (a.seq_len + BM - 1) / BM;
  const int64_t bh = (int64_t)a.batch * a.heads;
  const int64_t slots = workgroup_slots(BM, compute_units);
  if (ch->bytes > (int64_t)kScratchBytes || nq * bh > slots) return;
  // The items, the slots and so the bytes fall as S rises: bisection.
  const int t_max = q_tile_tiles(a, BM, nq - 1);
  int lo = std::max(4, ch->average), hi = t_max, n_slots = 0;
  auto fits = [&](int S) {
    const int items = count_items(a, BM, nq, S, &n_slots);
    return items <= kMaxSplitItems && items * bh <= slots &&
           partial_bytes(a, BM, n_slots) <= (int64_t)kScratchBytes;
  };
  while (lo < hi) {
    const int mid = (lo + hi) / 2;
    if (fits(mid)) hi = mid; else lo = mid + 1;
  }
  if (lo == t_max || lo == ch->S) return;
  const ChunkCost c0(a, compute_units, BM, nq, ch->S), c1(a, compute_units, BM, nq, lo);
  // The one with a CU for each item first: its cost needs no simulation.
  const bool c0_first = c0.items() <= compute_units;
  const double known = c0_first ? c0.cost() : c1.cost();
  if (c0_first ? c1.cost(known) >= known : c0.cost(known) <= known) return;
  count_items(a, BM, nq, lo, &n_slots);
  ch->S = lo;
  ch->bytes = partial_bytes(a, BM, n_slots);
}

// Fills the split-KV plan of chunks of at most S tiles.
void plan_chunks(const KernelArgs& a, int S, SplitPlan* plan) {
  const int BM = block_rows(a);
  const int nq = (a.seq_len + BM - 1) / BM;
  // Items, longest first (the dispatch order of the grid).
  struct Item { int len, qb, c, nch; };
  Item list[kMaxSplitItems];
  int n = 0, slot_base[kMaxSplitItems], n_slots = 0, n_merge = 0;
  for (int qb = 0; qb < nq; ++qb) {
    const int nch = q_tile_chunks(a, BM, qb, S), T = q_tile_tiles(a, BM, qb);
    slot_base[qb] = n_slots;
    if (nch > 1) {
      plan->merge[n_merge] = (uint32_t)qb | ((uint32_t)nch << 16);
      plan->merge_slot[n_merge] = (uint32_t)n_slots;
      ++n_merge;
      n_slots += nch;
    }
    for (int c = 0; c < nch; ++c) list[n++] = Item{chunk_tiles(c, nch, T), qb, c, nch};
  }
  std::stable_sort(list, list + n, [](const Item& x, const Item& y) {
    return x.len != y.len ? x.len > y.len : x.qb > y.qb;
  });
  for (int i = 0; i < n; ++i) {
    plan->item[i] = (uint32_t)list[i].qb | ((uint32_t)list[i].c << 16) |
                    ((uint32_t)list[i].nch << 24);
    plan->slot[i] = (uint32_t)(list[i].nch > 1 ? slot_base[list[i].qb] : 0);
  }
  plan->n_items = n;
  plan->n_slots = n_slots;
  plan->n_merge = n_merge;
}

// XCD placement table for a causal 4-wave grid of exactly two q-tiles per CU
// (below that the grid runs in pair mode): each XCD (cpx CUs) receives 2 cpx
// workgroups, whole heads.  Measured dispatch (per-workgroup hardware CU ids):
// an XCD's k-th workgroup goes to CU slot k mod cpx, so positions k and
// k + cpx share a CU.  Longest first (the default order) pairs the longest
// q-tile with the (cpx + 1)-th longest; the table pairs long with short: the
// first half runs longest first, heads interleaved, the second half backwards.
// No q-tile is split and the kernel's arithmetic is that of the plain grid
// (only the order changes).  The kernels of the product compute this order
// (work_item); the table itself is for fa_fwd_plan and the test builds.
void plan_xcd_table(const KernelArgs& a, int compute_units, SplitPlan* plan) {
  const int BM = block_rows(a);
  if (!a.causal || BM != 128 || compute_units % 8 != 0) return;
  const int64_t bh = (int64_t)a.batch * a.heads;
  if (bh % 8 != 0) return;
  const int nq = (a.seq_len + BM - 1) / BM;
  const int64_t hpx = bh / 8;
  const int64_t cpx = compute_units / 8;
  if (hpx * nq != 2 * cpx || hpx * nq > kMaxSplitItems) return;
  const int n = (int)(hpx * nq);
  for (int i = 0; i < n; ++i) {
    const int w = i < n / 2 ? i : n + n / 2 - 1 - i;
    plan->item[i] = (uint32_t)(nq - 1 - w / (int)hpx) | (1u << 24);
    plan->slot[i] = (uint32_t)(w % (int)hpx);
  }
  plan->n_items = n;
  plan->xcd_heads = (int)hpx;
}

}  // namespace

// Pair mode for causal 4-wave grids of 0.75 to 2 q-tiles (128 rows) per CU:
// one 8-wave workgroup per q-tile, its halves on alternate key tiles, one
// workgroup per CU, dispatched longest first.  Such grids are bound by
// their longest q-tiles, which a 4-wave workgroup runs alone on its CU
// once its partner is done (1.55 us per key tile alone against 2.1 us for
// each of two sharing it, at B1 H16 N3000); a pair workgroup keeps two waves
// on every SIMD.  Measured against the 4-wave kernel with its plans: +7..8 %
// at B1 H16 N3000 (Q, K ~ N(0, 3^2)), +8..27 % at H8..H16 N2048..6000
// (bf16 and D = 64 included); -6..-12 % at H24 and H32 N3000 (2.25 and 3 per
// CU) and -20..-49 % below 0.75 per CU (H4, H6), where split-KV spreads the
// few long q-tiles over more CUs.
namespace {
bool pair_mode(const KernelArgs& a, int compute_units) {
  if (!a.causal || block_rows(a) != 128) return false;
  const int64_t items = (int64_t)a.batch * a.heads * ((a.seq_len + 127) / 128);
  return 4 * items >= 3 * (int64_t)compute_units && items < 2 * (int64_t)compute_units;
}
}  // namespace

// Heads per dispatch group of an XCD for a causal grid in plain order (the
// kernel interleaves the q-tiles of a group's heads, longest first, and
// runs the groups one after the other).  Interleaving keeps a head's long
// q-tiles from starting late (+1.5 % at B2 H32 N8192 and B1 H16 N16384,
// +2.7 % at B1 H16 N8192 over head after head); smaller groups shrink the
// XCD's K/V working set.  Groups of 4 instead of all 8 heads of B2 H32
// N8192 measured +2.3…3 %, and groups of 2 another +0.4…1.3 % there (HBM
// reads 1.23 GB with groups of 4), but -1.5…1.8 % at B4 H32 N4096, where a
// group of 2 heads is a single round of workgroups: a group is kept at two
// or more rounds.
namespace {
int causal_head_group(const KernelArgs& a, int compute_units, bool pair) {
  const int64_t bh = (int64_t)a.batch * a.heads;
  if (!a.causal || bh % 8 != 0) return 0;
  const int hpx = (int)(bh / 8);  // heads per XCD
  int g = hpx % 4 == 0 ? 4 : hpx;
  const int bm = pair ? 128 : block_rows(a);
  const int64_t nq = (a.seq_len + bm - 1) / bm;
  const int64_t slots_per_xcd = (int64_t)(compute_units / 8) * (bm == 128 && !pair ? 2 : 1);
  if (g > 2 && hpx % 2 == 0 && 2 * nq >= 2 * slots_per_xcd) g = 2;
  return g;
}

// Key groups (fa_kg_kernel) for grids that leave CUs idle or with one wave per
// SIMD: four groups on 64-row q-tiles while those fit one per CU, two on
// 128-row q-tiles of non-causal problems while those do (causal ones are in
// pair mode from 0.75 per CU on).  One workgroup of 8 waves then holds each
// CU and a row's keys take a quarter (half) of the steps.  Past one
// workgroup per CU the second round costs more than it saves (1.1 to 1.5
// 128-row q-tiles per CU: 0.70...0.79 x).
//
// Measured us before -> after, fp16: four groups, B1 H8 N512 D64 8.7 -> 6.4,
// H32 N512 D128 13.6 -> 9.4, H16 N1024 D64 14.1 -> 8.8, causal 16.3 -> 9.7,
// H8 N2048 D64 25.6 -> 13.5, causal D128 27.1 -> 21.1; two groups, B2 H12
// N1024 D128 22.0 -> 18.2, B1 H12 N2048 D64 39.5 -> 19.9, H6 N4096 D128
// 85.2 -> 55.7.  Short rows: two key tiles gain from 4 groups on causal rows
// (D = 64 6.7 -> 5.8, D = 128 8.3 -> 6.7) but not on D = 64 non-causal ones
// (4.7 -> 5.0; four tiles 6.0 -> 5.2, ragged ones 6.3 -> 5.2); at D = 128 they gain as well (7.4 ->
// 6.4), but N = 128 non-causal is held to one 128-row q-tile per head by the
// plan's tests, so the line is three tiles.  Two groups need 4 tiles at
// D = 128 (10.4 -> 9.7) and 6 at D = 64 (4 tiles: 6.9 -> 7.1).
//
// Where split-KV would run (split_pays), its time is about constant plus the
// work W per CU (128-row q-tiles x key tiles), that of four groups about
// constant plus the row's T key tiles; the lines below cross where the
// measured times do (e.g. D128 N2048: H2 and H3 non-causal T = 32 at the
// line, causal H4 equal; N4096: H2 split 34.4 against 35.8 us, H4 four
// groups 40.6 against 45.7).  Grids of at most an eighth (causal: a quarter)
// of the CUs in 64-row q-tiles keep split-KV: the plan's tests hold shapes
// of one or two heads there to it (B1 H2 N1000 D64 non-causal 12.4 us split,
// 9.2 with four groups).  So do the few whose partials exceed the static
// scratch (D = 128, about 5 heads of N = 6000): fa_fwd_scratch refuses those,
// with or without key groups for their neighbours.  Two groups give way to a
// split that is clearly faster (split_beats_two_groups).
// ch: average_chunks.
int key_groups(const KernelArgs& a, int compute_units, const Chunks& ch) {
  const int64_t bh = (int64_t)a.batch * a.heads;
  const int T = (a.seq_len + kKeyTile - 1) / kKeyTile;
  const int nq128 = (a.seq_len + 127) / 128;
  const int64_t w64 = bh * T, w128 = bh * nq128;
  const bool d64 = a.head_dim == 64, causal = a.causal != 0;
  if (w64 > compute_units && (causal || w128 > compute_units)) return 0;
  int groups = 0;
  if (w64 <= compute_units) {
    if (!ch.pays) return T >= (causal ? 2 : d64 ? 4 : 3) ? 4 : 0;
    if (w64 <= compute_units / (causal ? 4 : 8)) return 0;
    const double W = causal ? (double)bh * nq128 * (nq128 + 1) : (double)w128 * T;
    const double t0 = causal ? (d64 ? 29.0 : 20.0) : (d64 ? 34.0 : 25.0);
    const double per_w = causal ? 2.56 : (d64 ? 2.3 : 1.46);
    groups = T < t0 + per_w * W / compute_units ? 4 : 0;
  } else {
    groups = T >= (d64 ? 6 : 4) ? 2 : 0;
  }
  if (ch.pays && groups != 0 && ch.bytes > (int64_t)kScratchBytes) return 0;
  return groups;
}

// Whether a split with chunks of at most S tiles beats two key groups, whose
// launch is T / 2 steps of the same work as a 256-row tile.  The line is where
// the measured times cross: of 138 grids below 0.92 the split is 3...18 % faster
// on those below 0.9 (us, two groups / split: B1 H2 N9032 D64 fp16 69.4 / 60.0,
// D128 103.1 / 90.4, H3 N7092 D64 bf16 56.2 / 51.7) and 3...5 % slower at 0.919
// (H4 N5341 D64 43.3 / 45.3).
bool split_beats_two_groups(const KernelArgs& a, int compute_units, int S) {
  const int BM = block_rows(a);
  const ChunkCost split(a, compute_units, BM, (a.seq_len + BM - 1) / BM, S);
  const int T = (a.seq_len + kKeyTile - 1) / kKeyTile;
  return split.cost() < 0.9 * 0.5 * T;
}

// Whether waves whose rows all lie past N compute like the others instead of
// only staging (D = 64 non-causal 4-wave grids).  Only staging frees their SIMD
// and is 1...2 % faster on most ragged grids, but a CU whose workgroups end
// early takes two of the remaining ones where each CU should get one.  Grids
// with 2.375 to 3 workgroups per CU of at least 800 rows show it: on 102 such
// grids staging takes 0.98 to 1.11 times as long as computing.  us, staging /
// computing: bf16 B1 H48 N2016 62.3 / 57.8, H50 N1856 57.2 / 54.3, fp16 H50
// N1856 61.1 / 57.9.  Below 2.375, above 3 and at shorter rows staging is the
// faster one, and at D = 128 within 1 %.
bool all_rows(const KernelArgs& a, int compute_units) {
  if (a.causal || a.head_dim != 64 || block_rows(a) != 128 || a.seq_len < 800) return false;
  const int64_t w = (int64_t)a.batch * a.heads * ((a.seq_len + 127) / 128);
  return 8 * w > 19 * (int64_t)compute_units && w <= 3 * (int64_t)compute_units;
}

}  // namespace

size_t plan_split(const KernelArgs& a, int compute_units, bool allow_split, SplitPlan* plan) {
  plan->n_items = plan->n_slots = plan->n_merge = plan->xcd_heads = plan->pair = 0;
  plan->head_group = plan->key_groups = plan->all_rows = 0;
  if (compute_units < 1) return 0;
  if (pair_mode(a, compute_units)) {
    plan->pair = 1;
    plan->head_group = causal_head_group(a, compute_units, true);
    return 0;
  }
  Chunks ch = average_chunks(a, compute_units);
  plan->key_groups = key_groups(a, compute_units, ch);
  if (allow_split && ch.S > 0 && plan->key_groups != 4) {
    choose_chunks(a, compute_units, &ch);
    if (plan->key_groups == 0 || split_beats_two_groups(a, compute_units, ch.S)) {
      plan->key_groups = 0;
      plan_chunks(a, ch.S, plan);
      return (size_t)ch.bytes;
    }
  }
  if (plan->key_groups != 0) return 0;
  plan_xcd_table(a, compute_units, plan);
  if (plan->n_items == 0) {
    plan->head_group = causal_head_group(a, compute_units, false);
    plan->all_rows = all_rows(a, compute_units);
  }
  return 0;
}

}  // namespace fa
