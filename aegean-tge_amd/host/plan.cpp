// Host-side planning of one step: see plan.hpp.
#include "plan.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>

#include "tge_kv.h"

namespace tge::plan {

namespace {
std::size_t align256(std::size_t x) { return (x + 255) & ~std::size_t(255); }
}  // namespace

int Staged::upload(MemOps& m, std::size_t bytes, void* stream,
                   const std::function<void(char*)>& fill) {
  bytes = std::max<std::size_t>(bytes, 256);
  if (staged) {
    const int s = m.wait_event(staged);
    if (s != TGE_OK) return s;
  }
  if (bytes > host_bytes) {
    if (host) m.host_free(host);
    host = nullptr;
    host_bytes = 0;
    const int s = m.host_alloc(&host, bytes);
    if (s != TGE_OK) {
      host = nullptr;
      return s;
    }
    host_bytes = bytes;
  }
  if (bytes > dev_bytes) {
    if (dev) {
      const int s = m.wait_stream(stream);  // queued kernels may still read it
      if (s != TGE_OK) return s;
      m.dev_free(dev);
    }
    dev = nullptr;
    dev_bytes = 0;
    const int s = m.dev_alloc(&dev, bytes);
    if (s != TGE_OK) {
      dev = nullptr;
      return s;
    }
    dev_bytes = bytes;
  }
  fill(host);
  int s = m.copy_to_device(dev, host, bytes, stream);
  if (s == TGE_OK) s = m.record(&staged, stream);
  return s;
}

void Staged::release(MemOps& m) {
  if (dev) m.dev_free(dev);
  if (host) m.host_free(host);
  if (staged) m.event_free(staged);
  dev = host = nullptr;
  staged = nullptr;
  dev_bytes = host_bytes = 0;
}

int Scratch::reserve(MemOps& m, std::size_t need, void* stream) {
  if (need <= bytes) return TGE_OK;
  if (dev) {
    const int s = m.wait_stream(stream);
    if (s != TGE_OK) return s;
    m.dev_free(dev);
  }
  dev = nullptr;
  bytes = 0;
  const int s = m.dev_alloc(&dev, need);
  if (s != TGE_OK) {
    dev = nullptr;
    return s;
  }
  bytes = need;
  return TGE_OK;
}

void Scratch::release(MemOps& m) {
  if (dev) m.dev_free(dev);
  dev = nullptr;
  bytes = 0;
}

int build_step(Step& step, int ns, const int* ctx, const int* n_new, const int* table_offsets,
               const int* page_ids, int q_heads, int kv_heads, int head_dim, int pool_pages,
               const char** message) {
  auto bad = [&](const char* m) {
    if (message) *message = m;
    return TGE_ERR_INVALID;
  };
  if (ns <= 0 || !ctx || !n_new || !table_offsets || !page_ids)
    return bad("batch_plan: empty or incomplete description");
  if (q_heads <= 0 || kv_heads <= 0 || q_heads % kv_heads != 0)
    return bad("batch_plan: q_heads must be a multiple of kv_heads");
  const int group = q_heads / kv_heads;
  if (group > prefill_tile_rows(head_dim <= 128 ? 128 : 256))
    return bad("batch_plan: more than 128 query heads per KV head (64 at head_dim > 128)");
  if (table_offsets[0] != 0) return bad("batch_plan: table_offsets[0] must be 0");
  const int n_entries = table_offsets[ns];
  if (n_entries < 0) return bad("batch_plan: negative table size");

  // Validate first: a failed plan leaves the step untouched.
  int max_rows = 0;
  for (int s = 0; s < ns; ++s) {
    const int c = ctx[s], nn = n_new[s];
    const int lo = table_offsets[s], hi = table_offsets[s + 1];
    if (c < 0 || nn < 1) return bad("batch_plan: ctx must be >= 0 and n_new >= 1");
    if (hi < lo || hi > n_entries) return bad("batch_plan: table_offsets must not decrease");
    const long need = ((long)c + nn + 15) / 16;
    if (hi - lo < need) return bad("batch_plan: block table shorter than the context");
    for (long i = 0; i < need; ++i) {
      const int id = page_ids[lo + i];
      if (id < 0 || id >= pool_pages) return bad("batch_plan: page id outside the pool");
    }
    if ((long)nn * group > (1L << 30)) return bad("batch_plan: too many rows");
    max_rows = std::max(max_rows, nn * group);
  }

  step.sessions.assign((std::size_t)ns, {});
  step.rows.clear();
  step.tables.assign(page_ids, page_ids + n_entries);
  int q_row = 0;
  for (int s = 0; s < ns; ++s) {
    const int c = ctx[s], nn = n_new[s], lo = table_offsets[s];
    step.sessions[(std::size_t)s] = SessionRec{c, nn, q_row, lo};
    for (int j = 0; j < nn; ++j) {
      const int pos = c + j;
      step.rows.push_back(RowRec{page_ids[lo + pos / 16], pos % 16, pos});
    }
    q_row += nn;
  }
  step.kv_heads = kv_heads;
  step.head_dim = head_dim;
  step.block_dims = head_dim <= 64 ? 64 : head_dim <= 128 ? 128 : 256;
  step.q_heads = q_heads;
  step.group = group;
  step.pages = pool_pages;
  step.max_rows = max_rows;
  return TGE_OK;
}

void build_append_tiles(const Step& s, std::vector<TileRec>& tiles, bool i8) {
  tiles.clear();
  const long values = (long)s.rows.size() * 2 * s.kv_heads * s.block_dims;
  const int width = s.kv_heads * s.head_dim;  // dims of a row of K
  const bool wide = width >= 1024;
  const long line = i8 ? (wide ? 3L << 20 : 9L << 19) : (wide ? 1L << 20 : 2L << 20);
  if (s.block_dims <= 64 || values < line || (i8 && width < 256)) return;
  for (const auto& sr : s.sessions) {
    for (int j = 0; j < sr.n_new;) {
      const int slot = (sr.ctx + j) % kPageTokens;
      const int n = std::min(kPageTokens - slot, sr.n_new - j);
      tiles.push_back(TileRec{s.rows[(std::size_t)(sr.q_row + j)].page, sr.q_row + j, slot, n});
      j += n;
    }
  }
  if (s.rows.size() < 12 * tiles.size()) tiles.clear();
}

bool decode_session(const Step& s, const SessionRec& r) {
  return r.n_new * s.group <= max_unit_rows(s.block_dims);
}

bool take_session(const Step& s, const SessionRec& r, int only) {
  return only == 0 || (only == 1) == decode_session(s, r);
}

// Relative speed of the k-th workgroup that lands on a CU. Workgroups are
// dispatched one per CU before a CU gets a second, and on a shared SIMD the
// older wave wins issue, so equal page shares finish far apart. Measured
// pages per microsecond of the c5 decode kernel by dispatch rank: 1 : 0.79
// with two workgroups per CU (1 : 0.75 before page loads read whole KiB
// runs), 1 : 0.775 : 0.54 with three (per-workgroup timestamps over whole
// launches); more ranks fall off by TGE_DECODE_RANK_WEIGHT.
#ifndef TGE_DECODE_RANK_WEIGHT
#define TGE_DECODE_RANK_WEIGHT 0.76
#endif

namespace {
double rank_weight(int rank, int per_cu) {
  if (per_cu == 2 && rank < 2) return rank == 0 ? 1.0 : 0.79;
  if (per_cu == 3 && rank < 3) return rank == 0 ? 1.0 : rank == 1 ? 0.775 : 0.54;
  return std::pow(TGE_DECODE_RANK_WEIGHT, (double)rank);
}
}  // namespace
// Fixed cost of one unit of a share (start-up and merge), in pages.
#ifndef TGE_DECODE_UNIT_COST
#define TGE_DECODE_UNIT_COST 22
#endif
// At least 8 pages per workgroup: on small steps (one to four sessions
// of 1k-8k positions) shorter chains win over fewer split merges down to
// 8 pages (c1-c3: 5-7 % per layer-step against 16; 4 is slower again).
#ifndef TGE_DECODE_MIN_PAGES
#define TGE_DECODE_MIN_PAGES 8
#endif

void build_decode(const Step& b, Residency res, AttnLists& pl, int only) {
  pl.work.clear();
  pl.reduce.clear();
  pl.wg_first.clear();
  pl.app_first.clear();
  pl.app_recs.clear();
  pl.app_waves = 0;
  pl.parts = pl.max_splits = 0;
  int max_rows = 0;
  for (const auto& sr : b.sessions)
    if (take_session(b, sr, only)) max_rows = std::max(max_rows, sr.n_new * b.group);
  pl.row_groups = std::max(1, std::min(4, (max_rows + 15) / 16));

  struct Seg {
    int session, head, pages;
  };
  std::vector<Seg> segs;
  long total = 0;
  for (int s = 0; s < (int)b.sessions.size(); ++s) {
    const SessionRec& sr = b.sessions[(std::size_t)s];
    if (!take_session(b, sr, only)) continue;
    const int pages = (sr.ctx + sr.n_new + 15) / 16;
    for (int h = 0; h < b.kv_heads; ++h) segs.push_back(Seg{s, h, pages});
    total += (long)pages * b.kv_heads;
  }
  const long g_eff = std::max<long>(
      1, std::min<long>(res.groups, (total + TGE_DECODE_MIN_PAGES - 1) / TGE_DECODE_MIN_PAGES));
  std::vector<double> w((std::size_t)g_eff);
  double wrem = 0.0;
  for (long g = 0; g < g_eff; ++g) {
    const int cus = std::max(1, res.cus);
    w[(std::size_t)g] = rank_weight((int)(g / cus), (res.groups + cus - 1) / cus);
    wrem += w[(std::size_t)g];
  }

  // Cut the segments, end to end, into one share per workgroup. A share's
  // cost is its pages plus TGE_DECODE_UNIT_COST per piece (the fixed cost
  // of starting and merging a unit); each share gets the remaining cost in
  // proportion to its rank weight, the last one takes what is left.
  const double unit_cost = TGE_DECODE_UNIT_COST;
  std::vector<int> seg_of;  // segment of each work item
  long pages_rem = total, segs_rem = (long)segs.size();
  std::size_t si = 0;
  int pos = 0;
  pl.wg_first.push_back(0);
  for (long g = 0; g < g_eff && si < segs.size(); ++g) {
    const bool last_wg = g + 1 == g_eff;
    double target =
        ((double)pages_rem + unit_cost * (double)(segs_rem + (g_eff - g))) * w[(std::size_t)g] / wrem;
    wrem -= w[(std::size_t)g];
    bool started = false;
    while (si < segs.size()) {
      const Seg& sg = segs[si];
      const int left = sg.pages - pos;
      int take = left;
      if (!last_wg) {
        const double room = target - unit_cost;
        if (started && room < 1.0) break;
        take = (int)std::min<double>(left, std::max(1.0, std::floor(room)));
      }
      const SessionRec& sr = b.sessions[(std::size_t)sg.session];
      WorkRec it{};
      it.session = sg.session;
      it.kv_head = sg.head;
      it.page_begin = pos;
      it.page_end = pos + take;
      it.part = -1;
      it.row_begin = 0;
      it.rows = sr.n_new * b.group;
      it.rows_per_query = b.group;
      it.head_base = sg.head * b.group;
      it.ctx = sr.ctx;
      it.q_row = sr.q_row;
      it.table_off = sr.table_off;
      it.red = -1;
      pl.work.push_back(it);
      seg_of.push_back((int)si);
      started = true;
      target -= take + unit_cost;
      pos += take;
      pages_rem -= take;
      if (pos == sg.pages) {
        ++si;
        pos = 0;
        --segs_rem;
      }
      if (!last_wg && target < unit_cost + 1.0) break;
    }
    pl.wg_first.push_back((int)pl.work.size());
  }

  // Segments cut into several items are merged by the split reduction.
  for (std::size_t i = 0; i < pl.work.size();) {
    std::size_t j = i + 1;
    while (j < pl.work.size() && seg_of[j] == seg_of[i]) ++j;
    const int n = (int)(j - i);
    pl.max_splits = std::max(pl.max_splits, n);
    if (n > 1) {
      const WorkRec& w0 = pl.work[i];
      ReduceRec r{};
      r.session = w0.session;
      r.row_begin = w0.row_begin;
      r.rows = w0.rows;
      r.rows_per_query = w0.rows_per_query;
      r.head_base = w0.head_base;
      r.first_part = pl.parts;
      r.q_row = w0.q_row;
      r.n_parts = n;
      for (std::size_t k = i; k < j; ++k) {
        pl.work[k].part = pl.parts++;
        pl.work[k].red = (int)pl.reduce.size();
      }
      pl.reduce.push_back(r);
    }
    i = j;
  }
  pl.groups = (int)pl.wg_first.size() - 1;
}

namespace {

// Splits [0, pages) into n ranges that differ by at most a page, one unit
// each; a unit of len pages goes to work[at[len]++].
void add_units(std::vector<WorkRec>& work, std::vector<int>& at, std::vector<ReduceRec>& red, int& parts,
               int& max_splits, WorkRec w, int pages, int n) {
  max_splits = std::max(max_splits, n);
  w.part = w.red = -1;
  if (n == 1) {
    w.page_begin = 0;
    w.page_end = pages;
    work[(std::size_t)at[(std::size_t)pages]++] = w;
    return;
  }
  ReduceRec r{};
  r.session = w.session;
  r.row_begin = w.row_begin;
  r.rows = w.rows;
  r.rows_per_query = w.rows_per_query;
  r.head_base = w.head_base;
  r.first_part = parts;
  r.q_row = w.q_row;
  r.n_parts = n;
  w.red = (int)red.size();
  w.page_end = 0;
  for (int k = 0; k < n; ++k) {
    w.page_begin = w.page_end;
    w.page_end = (int)((long)pages * (k + 1) / n);
    w.part = parts++;
    work[(std::size_t)at[(std::size_t)(w.page_end - w.page_begin)]++] = w;
  }
  red.push_back(r);
}

#ifndef TGE_PREFILL_MIN_SPLIT
#define TGE_PREFILL_MIN_SPLIT 32
#endif

// What a block-prefill launch of its own costs on an MI355X, microseconds,
// by kernel: the launch, an item's start and end, and a page of an item.
// Where a compute unit holds three workgroups (64 dims), `page` is that of
// an item alone there, and `two` and `three` times as much is a page of each
// of two or three that share it. Fitted to 1,636 launches (12 to 2,826
// items, 28/4, 12/2, 16/4 x 96, 14/2 x 64 and 16/8 x 256 heads, contexts up
// to 24,000): 5 to 6 % rms off at 128 and 256 dims, 8 to 9 % at 64.
struct PrefillCost {
  double launch, item, page;
  int per_cu;
  double two, three;
};
PrefillCost prefill_cost(int block_dims, int tile_rows, bool i8) {
  if (block_dims <= 64)
    return i8 ? PrefillCost{8.0, 2.0, 0.327, 3, 1.57, 2.19} : PrefillCost{7.5, 2.9, 0.194, 3, 1.47, 2.17};
  if (block_dims > 128) return i8 ? PrefillCost{3.0, 9.9, 0.899, 1, 1, 1} : PrefillCost{2.6, 9.6, 0.447, 1, 1, 1};
  if (tile_rows == 64) return i8 ? PrefillCost{3.6, 6.1, 0.333, 1, 1, 1} : PrefillCost{3.3, 6.1, 0.167, 1, 1, 1};
  return i8 ? PrefillCost{3.5, 9.9, 0.422, 1, 1, 1} : PrefillCost{3.2, 10.0, 0.230, 1, 1, 1};
}
// The merge launch behind it, and 64 KiB of partials through it (1,368
// launches, 0.9 us rms off).
constexpr double kMergeLaunch = 5.6, kMergePart = 0.0100;

// A way to cut a step's tiles: tiles of tile_rows rows (tq queries), of
// lens[i] pages once per KV head, in cuts[i] pieces.
struct TileCuts {
  int tile_rows = 0, tq = 1;
  std::vector<int> lens, cuts;
};

// The number of pieces of each length (0 to the longest) of one KV head.
void piece_lengths(const TileCuts& c, std::vector<int>& count) {
  int longest = 0;
  for (std::size_t i = 0; i < c.lens.size(); ++i)
    longest = std::max(longest, c.cuts[i] == 1 ? c.lens[i] : (c.lens[i] - 1) / c.cuts[i] + 1);
  count.assign((std::size_t)longest + 1, 0);
  for (std::size_t i = 0; i < c.lens.size(); ++i) {
    if (c.cuts[i] == 1) {
      count[(std::size_t)c.lens[i]]++;
      continue;
    }
    const int len = c.lens[i] / c.cuts[i], more = c.lens[i] % c.cuts[i];
    count[(std::size_t)len] += c.cuts[i] - more;
    if (more) count[(std::size_t)len + 1] += more;
  }
}

// Microseconds of the launch that `c` gives. The pieces go out longest
// first: with L(i) the length of the i-th and S workgroups at once, the end
// is past k + 1 pieces of length L(k * S) for every k, and past all pages
// divided by S. (`count`: scratch.)
double launch_time(const TileCuts& c, const PrefillCost& cost, int heads, int cus, int block_dims,
                   std::vector<int>& count) {
  piece_lengths(c, count);
  const long slots = (long)cus * cost.per_cu;
  long rank = 0, next = 0, round = 0, pages = 0, parts = 0;
  double t = 0.0, shared[3] = {0, 0, 0};
  for (int len = (int)count.size() - 1; len > 0; --len) {
    if (!count[(std::size_t)len]) continue;
    const long n = (long)count[(std::size_t)len] * heads;
    rank += n;
    pages += n * len;
    for (; next < rank; next += cus, ++round) {
      if (cost.per_cu == 1)
        t = std::max(t, (double)(round + 1) * (cost.item + cost.page * len));
      else if (round < 3)
        shared[round] = len;
    }
  }
  if (cost.per_cu > 1)  // the first compute unit's: three, then two, then one at work
    t = cost.item + cost.page * (shared[2] * cost.three + (shared[1] - shared[2]) * cost.two + (shared[0] - shared[1]));
  if (rank > slots)
    t = std::max(t, (cost.page * (double)pages + cost.item * (double)rank) * cost.three / (double)slots);
  for (int cuts : c.cuts) parts += cuts > 1 ? cuts : 0;
  if (parts)
    t += kMergeLaunch + kMergePart * (double)(parts * heads) * prefill_tile_rows(block_dims) * block_dims / 16384.0;
  return cost.launch + t;
}

}  // namespace

void build_prefill(const Step& b, int cus, AttnLists& pl, int only, int halves, bool i8) {
  pl.work.clear();
  pl.reduce.clear();
  pl.wg_first.clear();
  pl.groups = 0;
  pl.parts = pl.max_splits = 0;
  pl.row_groups = kPrefillRows / 16;
  cus = std::max(1, cus);
  halves = halves == 2 ? 2 : 1;
  const int min_pages = TGE_PREFILL_MIN_SPLIT * halves;
  // Tiles of tile_rows rows in pieces of about equal length: enough for two
  // rounds of two four-wave workgroups on each compute unit (of one
  // eight-wave workgroup with two halves). A tile is cut when it is longer
  // than min_pages.
  const auto equal_pieces = [&](int tile_rows) {
    TileCuts c;
    c.tile_rows = tile_rows;
    c.tq = std::max(1, tile_rows / b.group);
    long total = 0;
    for (const auto& sr : b.sessions) {
      if (!take_session(b, sr, only)) continue;
      for (int a = 0; a < sr.n_new; a += c.tq) {
        c.lens.push_back((sr.ctx + a + std::min(c.tq, sr.n_new - a) + 15) / 16);
        total += (long)c.lens.back() * b.kv_heads;
      }
    }
    const long units = 2L * cus * (halves == 2 ? 1 : 2);
    const int pps = (int)std::max<long>(min_pages, ((total + units - 1) / units + 3) / 4 * 4);
    c.cuts.resize(c.lens.size());
    for (std::size_t i = 0; i < c.lens.size(); ++i)
      c.cuts[i] = (c.lens[i] + pps - 1) / pps;
    return c;
  };
  TileCuts best = equal_pieces(prefill_tile_rows(b.block_dims));
  std::vector<int> count;
  // A launch of its own takes the shortest of a few ways: those pieces, whole
  // tiles, every tile in as many pieces as one, two or three rounds hold, or
  // whole tiles for the full rounds and only the shortest, those of the
  // last, partial round, in pieces that fill it; at 128 dims with two halves
  // each of these for 128-row tiles and for 64-row ones (one 16-row group
  // per wave), whose items are twice as many and cost less than half as
  // much more a page. Ways with a merge launch have to be 5 % shorter than
  // whole tiles. No piece is shorter than half of min_pages. (Tiles beside a
  // decode role, or in two workgroups of 128 dims per unit, keep equal
  // pieces: neither has been fitted.)
  if (only == 0 && !best.lens.empty() && (halves == 2 || b.block_dims != 128)) {
    double best_time = 1e30;
    const int widths = b.block_dims == 128 && b.group <= 64 ? 2 : 1;
    TileCuts ways[2] = {std::move(best), widths > 1 ? equal_pieces(64) : TileCuts{}};
    for (int w = 0; w < widths; ++w) {
      TileCuts& c = ways[w];
      const PrefillCost cost = prefill_cost(b.block_dims, c.tile_rows, i8);
      const long n = (long)c.lens.size() * b.kv_heads, slots = (long)cus * cost.per_cu;
      const auto take = [&] {
        const bool whole = std::all_of(c.cuts.begin(), c.cuts.end(), [](int x) { return x == 1; });
        const double t = launch_time(c, cost, b.kv_heads, cus, b.block_dims, count) * (whole ? 0.95 : 1.0);
        if (t >= best_time) return;
        best_time = t;
        best = c;
      };
      take();
      long last = 0;
      for (long pieces : {1L, slots / n, 2 * slots / n, 3 * slots / n}) {
        if (pieces <= last) continue;
        last = pieces;
        for (std::size_t i = 0; i < c.lens.size(); ++i)
          c.cuts[i] = (int)std::max<long>(1, std::min<long>(pieces, c.lens[i] / min_pages));
        take();
      }
      const long rest = n % slots;
      if (n < slots || rest == 0) continue;
      std::vector<std::size_t> order(c.lens.size());
      for (std::size_t i = 0; i < order.size(); ++i) order[i] = i;
      const std::size_t tail = (std::size_t)((rest + b.kv_heads - 1) / b.kv_heads);  // tiles of one head
      std::nth_element(order.begin(), order.begin() + (std::ptrdiff_t)tail - 1, order.end(),
                       [&](std::size_t x, std::size_t y) { return c.lens[x] != c.lens[y] ? c.lens[x] < c.lens[y] : x < y; });
      const long most = slots / ((long)tail * b.kv_heads);
      for (long pieces : {most, most + 1}) {
        if (pieces < 2) continue;
        std::fill(c.cuts.begin(), c.cuts.end(), 1);
        for (std::size_t k = 0; k < tail; ++k)
          c.cuts[order[k]] = (int)std::max<long>(1, std::min<long>(pieces, c.lens[order[k]] / min_pages));
        take();
      }
    }
  }
  pl.tile_rows = best.tile_rows;
  // Longest items first (partial slots are fixed per item, so order is free):
  // the place of the first item of each length.
  piece_lengths(best, count);
  int items = 0;
  for (std::size_t len = count.size(); len-- > 0;) {
    const int n = count[len] * b.kv_heads;
    count[len] = items;
    items += n;
  }
  pl.work.resize((std::size_t)items);
  std::size_t tile = 0;
  for (int s = 0; s < (int)b.sessions.size(); ++s) {
    const SessionRec& sr = b.sessions[(std::size_t)s];
    if (!take_session(b, sr, only)) continue;
    const std::size_t tile0 = tile;
    for (int h = 0; h < b.kv_heads; ++h) {
      tile = tile0;
      for (int a = 0; a < sr.n_new; a += best.tq, ++tile) {
        WorkRec w{};
        w.session = s;
        w.kv_head = h;
        w.ctx = sr.ctx;
        w.q_row = sr.q_row;
        w.table_off = sr.table_off;
        w.row_begin = a;
        w.rows = std::min(best.tq, sr.n_new - a) * b.group;
        w.rows_per_query = b.group;
        w.head_base = h * b.group;
        add_units(pl.work, count, pl.reduce, pl.parts, pl.max_splits, w, best.lens[tile], best.cuts[tile]);
      }
    }
  }
  pl.groups = (int)pl.work.size();
}

// When every context of the step fits this many batches, each is one piece:
// a batch more per wave (about a microsecond) costs less than the split
// merge it saves (the partials' coherent stores, the arrival counter and
// the last piece's reads, 3-4 microseconds), and no piece waits for another.
constexpr int kStepUnsplitBatches = 3;

bool build_step_lists(const Step& b, bool i8, bool scale_f32, StepLists& out) {
  out = StepLists{};
  if (b.max_rows > max_unit_rows(b.block_dims) || b.sessions.empty()) return false;
  long blocks = 0;
  int max_pages = 0;
  for (const auto& sr : b.sessions) {
    const int pages = (sr.ctx + sr.n_new + 15) / 16;
    blocks += (long)pages * b.kv_heads;
    max_pages = std::max(max_pages, pages);
  }
  if (blocks > kStepMaxBlocks) return false;
  // 64 rows at head_dim 128 (48 with int8 K/V and fp32 scales) do not fit
  // the step kernel's registers beside its page images (it would spill);
  // those steps take the decode kernel
  if (!step_fits(i8, scale_f32, b.block_dims, b.max_rows)) return false;
  out.row_groups = std::max(1, std::min(4, (b.max_rows + 15) / 16));
  // A piece is a whole number of batches (every wave of the workgroup loads
  // one batch of pages at once), as few as keep every context within
  // kStepMaxParts pieces.
  const int batch = kStepWaves * step_batch_pages(i8, scale_f32, b.block_dims, out.row_groups);
  const int heads = kStepMaxParts - 1;  // pieces before the appending one
  const int piece = batch * std::max(1, (max_pages + batch * heads - 1) / (batch * heads));
  out.piece_pages = piece;
  const bool unsplit = max_pages <= kStepUnsplitBatches * batch;
  for (int s = 0; s < (int)b.sessions.size(); ++s) {
    const SessionRec& sr = b.sessions[(std::size_t)s];
    const int pages = (sr.ctx + sr.n_new + 15) / 16;
    // A context of more than one piece: the pages before the first new
    // position in pieces of `piece` pages cut from the end (the first takes
    // the remainder), then one piece of the pages the new positions fall in
    // (at most 5: n_new <= 64), which stores the new rows first.
    const int written = sr.ctx / 16;
    const int head = unsplit || pages <= piece ? 0 : (written + piece - 1) / piece;
    const int n = head + 1;
    out.max_pieces = std::max(out.max_pieces, n);
    for (int h = 0; h < b.kv_heads; ++h) {
      const int seg = out.segments++;
      const int first = n > 1 ? out.parts : -1;
      if (n > 1) out.parts += n;
      for (int k = 0; k < n; ++k) {
        StepRec r{};
        if (k < head) {
          const int end = written - (head - 1 - k) * piece;
          r.page_begin = std::max(0, end - piece);
          r.page_end = end;
        } else {
          r.page_begin = head > 0 ? written : 0;
          r.page_end = pages;
        }
        r.session = s;
        r.kv_head = h;
        r.part = n > 1 ? first + k : -1;
        r.seg = seg;
        r.seg_parts = n;
        r.seg_first = first;
        r.append = k == n - 1;
        r.ctx = sr.ctx;
        r.n_new = sr.n_new;
        r.q_row = sr.q_row;
        r.table_off = sr.table_off;
        out.recs.push_back(r);
        const int pb = batch / kStepWaves;
        for (int i = 0; i < kStepFirstIds / kStepWaves; ++i)
          for (int w = 0; w < kStepWaves; ++w) {
            const int pg = std::min(r.page_begin + w + i * kStepWaves, r.page_end - 1);
            out.first_ids.push_back(i < pb && pg >= 0
                                        ? b.tables[(std::size_t)(r.table_off + pg)]
                                        : 0);
          }
      }
    }
  }
  return true;
}

std::size_t image_layout(const AttnLists& pl, std::size_t* off_reduce, std::size_t* off_first,
                         std::size_t* off_app) {
  const std::size_t wbytes = pl.work.size() * sizeof(WorkRec);
  *off_reduce = align256(wbytes);
  *off_first = align256(*off_reduce + pl.reduce.size() * sizeof(ReduceRec));
  const std::size_t end = *off_first + pl.wg_first.size() * sizeof(int);
  if (!off_app) return end;
  *off_app = align256(end);
  return *off_app + (pl.app_first.size() + pl.app_recs.size()) * sizeof(int);
}

void write_image(const AttnLists& pl, std::size_t off_reduce, std::size_t off_first, char* h,
                 std::size_t off_app) {
  if (!pl.work.empty()) std::memcpy(h, pl.work.data(), pl.work.size() * sizeof(WorkRec));
  if (!pl.reduce.empty())
    std::memcpy(h + off_reduce, pl.reduce.data(), pl.reduce.size() * sizeof(ReduceRec));
  if (!pl.wg_first.empty())
    std::memcpy(h + off_first, pl.wg_first.data(), pl.wg_first.size() * sizeof(int));
  if (off_app && !pl.app_first.empty()) {
    std::memcpy(h + off_app, pl.app_first.data(), pl.app_first.size() * sizeof(int));
    std::memcpy(h + off_app + pl.app_first.size() * sizeof(int), pl.app_recs.data(),
                pl.app_recs.size() * sizeof(int));
  }
}

void build_decode_appends(const Step& b, AttnLists& pl, int waves, int max_rows) {
  pl.app_first.clear();
  pl.app_recs.clear();
  pl.app_waves = 0;
  // (the kernel keys a row by its work item, below 2^15)
  if (waves <= 0 || pl.work.size() >= (std::size_t)1 << 15) return;
  const int groups = (int)pl.wg_first.size() - 1;
  std::vector<std::vector<int>> per((std::size_t)waves);
  for (int g = 0; g < groups; ++g) {
    for (auto& v : per) v.clear();
    for (int it = pl.wg_first[(std::size_t)g]; it < pl.wg_first[(std::size_t)g + 1]; ++it) {
      const WorkRec& u = pl.work[(std::size_t)it];
      const SessionRec& sr = b.sessions[(std::size_t)u.session];
      const int j0 = std::max(0, 16 * u.page_begin - sr.ctx);
      const int j1 = std::min(sr.n_new, 16 * u.page_end - sr.ctx);
      for (int j = j0; j < j1; ++j) {
        const int pos = sr.ctx + j;
        auto& v = per[(std::size_t)((pos / 16 - u.page_begin + it) % waves)];
        v.push_back(b.tables[(std::size_t)sr.table_off + (std::size_t)(pos / 16)]);
        v.push_back(pos);
        v.push_back((sr.q_row + j) * b.kv_heads + u.kv_head);
        v.push_back(it);
      }
    }
    for (const auto& v : per) {
      if ((int)(v.size() / kAppRecInts) > max_rows) {  // more than a wave holds: no lists
        pl.app_first.clear();
        pl.app_recs.clear();
        return;
      }
      pl.app_first.push_back((int)(pl.app_recs.size() / kAppRecInts));
      pl.app_recs.insert(pl.app_recs.end(), v.begin(), v.end());
    }
  }
  pl.app_first.push_back((int)(pl.app_recs.size() / kAppRecInts));
  pl.app_recs.resize(pl.app_recs.size() + (std::size_t)kAppPad * kAppRecInts, 0);
  pl.app_waves = waves;
}

}  // namespace tge::plan
