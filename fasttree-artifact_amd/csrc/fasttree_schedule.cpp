// Launch schedule of the first decode stage: vnode lists re-cut into block programs for a device.
// Declarations and array layouts: include/fasttree_schedule.h.
//
// A launch holds two kinds of work.  *Wide* vnodes (more than 16 query rows) are served by blocks of
// four waves and are bound by the matrix instructions; *narrow* ones by a wave each, bound by memory.
// A block program is a list of wide vnodes that one block serves one after the other for one KV
// head.  Blocks are handed out in index order, two per compute unit, and with 256 of them a round
// goes once around the machine: block b and block b + (number of units) share a unit.  The schedule
// therefore places programs on units in pairs, a first row of programs and a second one, and
// chooses the cut of the runs -- into row chunks and, along the tokens, into pieces -- whose modelled
// duration is the shortest:
//
//  * a unit with programs of TA >= TB (each alone) is done after TA + kPairing * TB: two blocks step
//    about 1.5 times slower each than one alone (measured: kStep below);
//  * the narrow vnodes follow in index order and fill the block slots that programs leave or never
//    had, so short second programs are not idle slots but room for them;
//  * every piece costs its start-up and wind-down and, per query row, a partial result that the
//    second stage reads back.

#include "fasttree_schedule.h"
#include "fasttree_hip.h"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <memory>
#include <numeric>
#include <queue>
#include <unordered_map>
#include <vector>

namespace {

constexpr int kTile = 32;              // tokens of a step
constexpr int kCut = 64;               // pieces start at multiples of this many tokens
constexpr int kMinPiece = 128;         // and are not made shorter than this
constexpr int kWaveRows = 32;          // query rows a wave of the narrow path serves per pass
constexpr int kNarrowChunk = 1024;     // tokens one wave walks at most
constexpr int kJoined = 256;           // and the most of short vnodes that are made one
constexpr int kBlocksPerCu = 2;
constexpr int kWavesPerBlock = 4;
constexpr int kXcds = 8;

// ---- the model (microseconds; measured on the shapes of the kernel's own loop, rows resident in L2)

// One 32-token step of a block that has its compute unit to itself, by 16-row groups of the piece.
// head_dim 128, rows in L2: 20 and 32 rows .35, 48 and 64 rows .42, 80 and 96 rows .52, 128 rows .67, 192 rows .86
// (.36, .43, .53, .69 and .88 on the kernel that the table was set with).  The
// entries for 32 and 48 rows are those of a kernel that split their tokens four ways (.42 and .51): with the
// figures measured since in their place trees of 64/8 heads are cut finer and took 3 to 4 % longer (26.3 -> 27.5, 35.2 ->
// 36.2 and 132 -> 136 us), so short pieces of few rows cost more than their steps.  The entries above 128 rows are
// an eighth longer than a block alone takes: beside another block pieces of 192 rows fall behind.  In calls one at a
// time two such blocks on a unit took 1.71 times one's time a step, two of 128 rows 1.51 (1.39 and .96 us; .81 and .64
// alone), 1.44 times as long as 128 rows as in this table; in a queue of calls, on the present kernel, 1.54 and 1.44
// (1.34 and 1.03 us; .87 and .72 alone).  Other head sizes: measured on full chunks.
// The blocks of a run lie on one XCD and share it in its L2 where the KV heads divide evenly over the
// XCDs; otherwise every XCD reads it, and a step of few rows lasts as long as its loads.
double step_us(int groups, int head_dim, int heads) {
  static const double at128[13] = {0, .35, .42, .51, .44, .53, .53, .69, .69, .97, .98, .99, .99};
  static const double at64[13] = {0, .25, .30, .36, .31, .38, .38, .49, .49, .61, .62, .63, .63};
  static const double at256[9] = {0, .91, .91, .92, .92, 1.42, 1.42, 1.42, 1.42};
  if (head_dim > 128) return at256[std::min(groups, 8)];
  const int g = std::min(groups, 12);
  const double at = head_dim == 128 ? at128[g] : head_dim == 64 ? at64[g] : 0.85 * at64[g];
  return heads % kXcds ? std::max(at, .005 * head_dim) : at;
}
constexpr double kPairing = 0.55;      // see above
constexpr double kYounger = 1.67;      // a second program as long as the first ends this much later than alone: its waves issue second
constexpr double kNarrowPairing = 0.28;  // the same for narrow vnodes beside a program
constexpr double kNarrowBeside = 1.4;    // a narrow vnode takes this much longer where programs run
constexpr double kVnode = 5.5;         // start-up and wind-down of a wide vnode
constexpr double kChained = 1.0;       // and what one costs more as a later vnode of a program: no other block covers for it
constexpr double kNarrowStart = 4.5, kNarrowStep = 1.0, kNarrowShare = 0.6;   // a narrow vnode; its waves' merge
constexpr double kBytesPerUs = 5.6e6;  // rows at random slots, the whole part
constexpr double kScratchPerUs = 4.0e6;  // partial results, written and read back
constexpr double kNoOverlap = 0.35;
constexpr double kLaunch = 1.5;
// K/V rows of a small launch (see arrange), for 256 units: about what they read while a wide vnode starts and ends
// twice.  With half of it 15 of the 18 drawn trees that it concerns take longer (24.6 -> 29.7 us the most), with
// twice 9 of 17 get shorter, by up to a tenth, others longer (30.0 -> 38.1).
constexpr double kSmallLaunchBytes = 64e6;

// Of two decisions on what attends what, a launch is clearly better that is modelled shorter by a twentieth and by this
// many microseconds: below that the model chose wrongly as often as not (12.0 us instead of 10.5, 12.6 instead of 11.9).
constexpr double kClearlyBetter = 0.95, kClearlyUs = 1.5;

// A launch of whole paths, both launches of any other plan in one: its start and end, and a round of tiles (as many as a
// block has waves, 128 KB at 256-byte rows, which a unit takes in at 64 bytes a cycle), longer by kPathShared of it where every
// unit has a block.  Whole calls of head_dim 128, whole paths and otherwise, us: 4 requests of 32/8 heads with 80 tokens each
// 4.3 and 6.5, 408 tokens 6.4 and 7.5, 924 tokens 8.4 and 7.7 (not taken), 1524 tokens 10.5 and 8.4; 31 with 300 tokens 6.5 and
// 9.6, with 1100 11.4 and 11.2; 240 of 16/1 heads with 288 tokens 7.0 and 9.4, with 1100 12.1 and 17.3.
//
// A block has its unit to itself at 256- and 512-byte rows, so past a block per unit a second round begins there: 33 requests of 300
// tokens 9.6 and 8.5, of 408 tokens 11.1 and 8.6, 9 of 32/32 heads 9.5 and 7.9, 65 of 16/4 heads of 256 17.3 and 14.0, 257 of 16/1
// heads 10.4 and 10.2.  The rule is drawn one block short of that: just a block per unit (32 of 32/8 heads) would still be
// shorter, 6.0 and 8.5 (408 tokens 6.8 and 8.2, 8 of 32/32 5.7 and 7.8, 256 of 16/1 of 256 11.6 and 18.9).  Of rows of 128 bytes a unit
// holds two blocks, and whole paths would go on being shorter: 33 of 64-dim heads 5.5 and 7.4, 64 5.9 and 8.0, 96 8.0 and 9.9.
constexpr double kPathStart = 3.8, kPathRound = 1.1, kPathShared = 0.43;

struct Run {
  int64_t start;                 // into the flat slot list
  std::vector<int32_t> lens;     // the chunks it came in
  int64_t tokens;
  const int32_t* reqs;
  int n;                         // requests
};

struct Piece {
  int64_t start;
  int32_t tokens;
  const int32_t* reqs;
  int n;
  double us;                     // alone on a unit, start-up included
};

struct Narrow {
  int64_t start;
  int32_t tokens;
  const int32_t* reqs;
  int n;
};

struct Machine {
  int cus, heads, group, head_dim;
  int units() const { return std::max(1, cus / heads); }   // compute units per KV head
  int block_slots() const { return (head_dim <= 128 ? kBlocksPerCu : 1) * cus; }   // blocks the device holds at a time
  int64_t wave_slots() const { return (int64_t)block_slots() * kWavesPerBlock; }
};

int rows_per_block(int head_dim) { return head_dim <= 128 ? 192 : 128; }
int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

// The (KV run, request list) pairs behind vnode lists: vnodes over one KV slice whose scratch rows
// adjoin are the query tiles of one chunk; chunks whose slices adjoin and whose requests are equal are
// the KV splits of one node.
std::vector<Run> runs_of(int64_t n, const int32_t* ko, const int32_t* kl, const int32_t* qo, const int32_t* ql, const int32_t* q_entries) {
  std::vector<int64_t> order(n);
  for (int64_t i = 0; i < n; ++i) order[i] = i;
  std::sort(order.begin(), order.end(), [&](int64_t a, int64_t b) {
    if (ko[a] != ko[b]) return ko[a] < ko[b];
    if (kl[a] != kl[b]) return kl[a] < kl[b];
    return qo[a] < qo[b];
  });
  struct Chunk { int64_t off; int32_t len; const int32_t* reqs; int n; uint64_t key; };
  std::vector<Chunk> chunks;
  for (int64_t i = 0; i < n;) {
    const int64_t v = order[i];
    int64_t end = (int64_t)qo[v] + ql[v], j = i + 1;
    for (; j < n; ++j) {
      const int64_t w = order[j];
      if (ko[w] != ko[v] || kl[w] != kl[v] || qo[w] != end) break;
      end += ql[w];
    }
    const int32_t* reqs = q_entries + qo[v];
    const int count = (int)(end - qo[v]);
    uint64_t key = 1469598103934665603ull;
    for (int r = 0; r < count; ++r) key = (key ^ (uint32_t)reqs[r]) * 1099511628211ull;
    chunks.push_back({ko[v], kl[v], reqs, count, key});
    i = j;
  }
  auto same = [](const Chunk& a, const Chunk& b) { return a.n == b.n && a.key == b.key && std::equal(a.reqs, a.reqs + a.n, b.reqs); };
  std::unordered_multimap<int64_t, int> by_start;
  by_start.reserve(chunks.size() * 2);
  for (int i = (int)chunks.size() - 1; i >= 0; --i) by_start.emplace(chunks[i].off, i);
  std::vector<int> follower(chunks.size(), -1);
  std::vector<char> led(chunks.size(), 0);
  for (int i = 0; i < (int)chunks.size(); ++i) {
    if (chunks[i].len == 0) continue;
    auto range = by_start.equal_range(chunks[i].off + chunks[i].len);
    int found = -1;
    for (auto it = range.first; it != range.second; ++it)
      if (it->second != i && !led[it->second] && same(chunks[i], chunks[it->second]) && (found < 0 || it->second < found)) found = it->second;
    if (found >= 0) {
      follower[i] = found;
      led[found] = 1;
    }
  }
  std::vector<Run> runs;
  for (int i = 0; i < (int)chunks.size(); ++i) {
    if (led[i]) continue;
    Run r{chunks[i].off, {}, 0, chunks[i].reqs, chunks[i].n};
    for (int c = i; c >= 0; c = follower[c]) {
      r.lens.push_back(chunks[c].len);
      r.tokens += chunks[c].len;
    }
    runs.push_back(std::move(r));
  }
  return runs;
}

// A tree as its arrays (arguments as in ft_schedule_tree).
struct Tree {
  int n;
  const int32_t *parent, *seqlen, *num_children;
  const int64_t* req_offs;
  const int32_t* req_ids;
  const int64_t* kv_ptrs;
  const int32_t* slot_map;
  int64_t slot_map_len;
  int64_t requests(int v) const { return req_offs[v + 1] - req_offs[v]; }
};

// Which nodes attend their parent's run together with their own tokens.  Top down as the reference's
// greedy splitter goes (kernel_bench/fasttree.py:64-96), with its padding costs replaced by bytes: a child that
// stays a vnode of its own adds a partial result (head_dim + 1 floats, written and read) per query head of its
// requests; one that takes along the run its parent attends reads that run's rows again, unless nobody else is
// left on it.  (A 256-token prompt of 4 samples at one KV head of 16 query heads: the samples stay apart, 33 KB of
// partials each against 262 KB of rows.)
std::vector<int32_t> taken_along(const Tree& t, const Machine& m) {
  std::vector<int> first(t.n, -1), next(t.n, -1), last(t.n, -1);     // children in ascending id
  for (int v = 1; v < t.n; ++v) {
    const int up = t.parent[v];
    if (last[up] < 0) first[up] = v;
    else next[last[up]] = v;
    last[up] = v;
  }
  const double row_bytes = 2.0 * 4.0 * m.group * m.heads * (m.head_dim + 1), token_bytes = 4.0 * m.head_dim * m.heads;
  std::vector<int64_t> run(t.seqlen, t.seqlen + t.n);
  std::vector<int32_t> along(t.n, 0);
  std::vector<int> queue{0};
  for (size_t at = 0; at < queue.size(); ++at) {
    const int v = queue[at];
    int64_t attached = t.requests(v);
    for (int l = first[v]; l >= 0; l = next[l]) {
      const int64_t rows = t.requests(l);
      const bool rest = rows < attached;
      if ((rest ? token_bytes * run[v] : 0.0) < row_bytes * rows) {
        along[l] = 1;
        attached -= rows;
        run[l] = t.seqlen[l] + run[v];
      }
      queue.push_back(l);
    }
  }
  return along;
}

// The tree's runs under such a decision.
struct TreeRuns {
  std::vector<Run> runs;
  std::vector<std::vector<int32_t>> served;
  std::vector<int32_t> kv_entries;
  std::vector<int32_t> along;    // per node, 1: attends its parent's run together with its own tokens
};
int tree_runs(const Tree& tree, std::vector<int32_t> decided, TreeRuns& t) {
  const int n = tree.n;
  t.along = std::move(decided);
  // which requests every node's own vnodes serve (kernel_bench/fasttree.py:126-141)
  t.served.resize(n);
  std::vector<int> fifo;
  std::vector<int64_t> waiting(tree.num_children, tree.num_children + n);
  for (int v = 0; v < n; ++v)
    if (tree.num_children[v] == 0) {
      fifo.push_back(v);
      t.served[v].assign(tree.req_ids + tree.req_offs[v], tree.req_ids + tree.req_offs[v + 1]);
    }
  for (size_t at = 0; at < fifo.size(); ++at) {
    const int v = fifo[at], up = tree.parent[v];
    if (v == 0 || up < 0) continue;
    if (!t.along[v]) t.served[up].insert(t.served[up].end(), tree.req_ids + tree.req_offs[v], tree.req_ids + tree.req_offs[v + 1]);
    if (--waiting[up] == 0) fifo.push_back(up);
  }
  std::vector<int> chain;
  t.kv_entries.reserve((size_t)std::min<int64_t>(std::max<int64_t>(tree.kv_ptrs[n], 0), 1 << 26) + 32);
  for (int v = 0; v < n; ++v) {
    if (t.served[v].empty()) continue;
    chain.assign(1, v);
    while (t.along[chain.back()]) chain.push_back(tree.parent[chain.back()]);
    const int64_t start = (int64_t)t.kv_entries.size();
    for (auto it = chain.rbegin(); it != chain.rend(); ++it) {
      const int64_t lo = tree.kv_ptrs[*it], hi = tree.kv_ptrs[*it + 1];
      if (lo < 0 || hi < lo || hi > INT32_MAX || (tree.slot_map && hi > tree.slot_map_len) || start + hi - lo > INT32_MAX - 64) return FT_SCHEDULE_ERR_ARGUMENT;
      if (tree.slot_map) {
        t.kv_entries.insert(t.kv_entries.end(), tree.slot_map + lo, tree.slot_map + hi);
      } else {
        t.kv_entries.resize(t.kv_entries.size() + hi - lo);
        std::iota(t.kv_entries.end() - (hi - lo), t.kv_entries.end(), (int32_t)lo);
      }
    }
    const int64_t tokens = (int64_t)t.kv_entries.size() - start;
    Run r{start, {}, tokens, t.served[v].data(), (int)t.served[v].size()};
    // (chunks for the narrow path: a wave should not walk much more than its neighbours)
    const int64_t parts = std::max<int64_t>(1, ceil_div(tokens, kNarrowChunk)), tiles = ceil_div(tokens, kTile);
    int64_t done = 0;
    for (int64_t i = 0; i < parts; ++i) {
      const int64_t take = std::min((tiles / parts + (i < tiles % parts ? 1 : 0)) * kTile, tokens - done);
      if (take > 0 || parts == 1) r.lens.push_back((int32_t)take);
      done += take;
    }
    t.runs.push_back(std::move(r));
  }
  t.kv_entries.insert(t.kv_entries.end(), 32, -1);
  return FT_SCHEDULE_OK;
}

// Narrow vnodes with the longest runs halved while the waves they take fill less than three quarters
// of the wave slots: a wave walks its run tile by tile, one memory round trip each, so a launch of a
// few long runs lasts as long as its longest walk.
std::vector<Narrow> cut_long(std::vector<Narrow> in, int group, int heads, int64_t wave_slots) {
  auto waves = [&](const Narrow& v) { return ceil_div((int64_t)v.n * group, kWaveRows) * heads; };
  int64_t total = 0;
  for (const Narrow& v : in) total += waves(v);
  auto shorter = [&](int a, int b) { return in[a].tokens != in[b].tokens ? in[a].tokens < in[b].tokens : a > b; };
  std::vector<int> order(in.size());
  for (size_t i = 0; i < in.size(); ++i) order[i] = (int)i;
  std::priority_queue<int, std::vector<int>, decltype(shorter)> heap(shorter, std::move(order));
  while (!heap.empty() && 4 * total < 3 * wave_slots && in[heap.top()].tokens >= 2 * kMinPiece) {
    const int i = heap.top();
    heap.pop();
    const int32_t first = (int32_t)(ceil_div(in[i].tokens / 2, kTile) * kTile);
    if (in[i].tokens - first < kMinPiece) continue;
    Narrow rest{in[i].start + first, in[i].tokens - first, in[i].reqs, in[i].n};
    in[i].tokens = first;
    in.push_back(rest);
    heap.push(i);
    heap.push((int)in.size() - 1);
    total += waves(rest);
  }
  return in;
}

// Narrow vnodes of one run that lie side by side, made one where one of them is short (a serving batch's requests come with
// their prompt and their generated tokens apart): where they are more waves than there is room for beside the programs, and
// so made fit in.  The second round costs more than the longer walk of the first, and a partial result per request goes.
// First stage, us: 128 requests of 128 + 58 tokens beside 32 programs per KV head 30.5 -> 29.3, 128 of 100 + 60 beside as many
// 27.3 -> 24.4, 120 of 30 + 70 21.0 -> 18.5.  Not taken where all fit in as they are (64 of 160 + 140 + 90 beside 12 programs 23.2
// -> 25.4), nor where not all of them do even so (192 of 120 + 18 32.6 either way).
// Around the last wave slot the gain is a matter of a few hundredths either way.  Whole calls of eight groups on 2560 tokens beside
// 24 programs, apart and as one: of 128 + 58 tokens 128 requests 36.1 and 35.1, 144 40.1 and 39.9, 160 (the slots are just filled)
// 41.6 and 40.8, and past the line 168 42.0 and 41.4, 192 45.7 and 43.7; of 100 + 60 tokens 128 33.9 and 33.3, 144 36.6 and 37.5,
// 160 38.0 and 38.6, past it 176 39.4 and 40.0, 192 42.7 and 41.4.
std::vector<Narrow> join_short(const std::vector<Narrow>& in, int64_t programs, int heads, int64_t wave_slots) {
  auto fit = [&](const std::vector<Narrow>& v) { return ((int64_t)v.size() + programs * kWavesPerBlock) * heads <= wave_slots; };
  if (fit(in)) return in;
  std::vector<int> order(in.size());
  std::iota(order.begin(), order.end(), 0);
  std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return in[a].start < in[b].start; });
  std::vector<Narrow> out = in;
  int last = -1;
  for (int i : order) {
    if (out[i].tokens == 0) continue;
    if (last >= 0 && out[last].start + out[last].tokens == out[i].start && out[last].reqs == out[i].reqs && out[last].n == out[i].n &&
        std::min(out[last].tokens, out[i].tokens) < kMinPiece && out[last].tokens + out[i].tokens <= kJoined) {
      out[last].tokens += out[i].tokens;
      out[i].n = 0;
    } else {
      last = i;
    }
  }
  out.erase(std::remove_if(out.begin(), out.end(), [](const Narrow& v) { return v.n == 0; }), out.end());
  // (longest walk first, as they were)
  std::stable_sort(out.begin(), out.end(), [](const Narrow& a, const Narrow& b) { return ceil_div(a.tokens, kTile) > ceil_div(b.tokens, kTile); });
  return fit(out) ? out : in;
}

// How a launch's wide runs are cut and placed.
struct Cut {
  int rows_cap;      // requests per row chunk
  double piece_us;   // pieces are made about this long
  int row_slots;     // program slots per unit: 1 or 2
  double last;       // the last piece of a run relative to the others (two slots: the second program of a unit is the slower)
};

struct Layout {
  std::vector<Piece> pieces;
  std::vector<std::vector<int>> programs;   // pieces of every program, in launch order
  double wide_us = 0, total_us = 1e30;
};

struct NarrowLoad {
  double block_us;    // time the narrow vnodes take of block slots, all heads
  double longest_us;  // the longest of them
  double bytes_us;    // at the memory's rate
};

// Passes over its run that a narrow vnode takes (one of a 16-row group costs less than one of two: at 512-byte rows about half).
double passes(const Narrow& v, const Machine& m) {
  const int64_t rows = (int64_t)v.n * m.group;
  return rows <= 16 ? (m.head_dim <= 128 ? 0.8 : 0.55) : (double)ceil_div(rows, kWaveRows);
}

NarrowLoad narrow_load(const std::vector<Narrow>& narrow, const Machine& m, double bytes_us) {
  NarrowLoad load{0, 0, bytes_us};
  // the launcher lets 2 or 4 waves share a vnode while that leaves a quarter of the wave slots free
  const int64_t items = (int64_t)narrow.size() * m.heads;
  int share = 1;
  while (share < kWavesPerBlock && 4 * items * 2 * share <= 3 * m.wave_slots()) share *= 2;
  for (const Narrow& v : narrow) {
    const double us = kNarrowStart + kNarrowStep * std::max(0.6, m.head_dim / 128.0) * ceil_div(ceil_div(v.tokens, kTile), share) * passes(v, m) + (share > 1 ? kNarrowShare : 0.0);
    load.block_us += us * m.heads * share / kWavesPerBlock;
    load.longest_us = std::max(load.longest_us, us);
  }
  return load;
}

// The time that reading the runs' rows takes.
double read_us(const std::vector<Run>& runs, const Machine& m) {
  double bytes = 0;
  for (const Run& r : runs) bytes += 4.0 * m.head_dim * r.tokens * m.heads;
  return bytes / kBytesPerUs * 256 / m.cus;
}

std::vector<Piece> cut_runs(const std::vector<Run>& wide, const Machine& m, const Cut& cut) {
  std::vector<Piece> pieces;
  for (const Run& r : wide) {
    const int chunks = (int)std::max<int64_t>(1, ceil_div(r.n, cut.rows_cap));
    const int groups = (int)ceil_div((int64_t)ceil_div(r.n, chunks) * m.group, 16);
    const double step = step_us(groups, m.head_dim, m.heads);
    const int64_t units = ceil_div(r.tokens, kCut);
    const double run_us = step * ceil_div(r.tokens, kTile);
    int64_t n = (int64_t)std::ceil(run_us / std::max(1.0, cut.piece_us - kVnode) - 1e-9);
    n = std::max<int64_t>(1, std::min(n, r.tokens / kMinPiece));
    for (int c = 0; c < chunks; ++c) {
      const int base = r.n / chunks, extra = r.n % chunks;
      const int lo = c * base + std::min(c, extra), size = base + (c < extra ? 1 : 0);
      int64_t done = 0;
      const int64_t short_units = n > 1 && cut.last < 1.0 ? std::max<int64_t>(kMinPiece / kCut, std::llround(units * cut.last / (n - 1 + cut.last))) : 0;
      const int64_t evens = short_units ? n - 1 : n, even_units = units - short_units;
      for (int64_t i = 0; i < n && done < r.tokens; ++i) {
        const int64_t share = i == evens ? short_units : even_units / evens + (i < even_units % evens ? 1 : 0);
        const int64_t take = std::min(share * kCut, r.tokens - done);
        pieces.push_back({r.start + done, (int32_t)take, r.reqs + lo, size, step * ceil_div(take, kTile) + kVnode});
        done += take;
      }
    }
  }
  return pieces;
}

// Reading and computing overlap, but a launch that needs both for long overlaps them only in part.
double overlapped(double a, double b) { return std::max(a, b) + kNoOverlap * std::min(a, b); }

// Longest piece first, each to the unit that is done first with it, into that unit's emptier slot.
void place(Layout& l, const Machine& m, const Cut& cut, const NarrowLoad& narrow) {
  const int units = m.units();
  std::vector<int> order(l.pieces.size());
  for (size_t i = 0; i < order.size(); ++i) order[i] = (int)i;
  std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return l.pieces[a].us > l.pieces[b].us; });
  struct Unit { double t[2] = {0, 0}; std::vector<int> in[2]; };
  std::vector<Unit> unit(units);
  auto done = [&](const Unit& u) {
    const double longer = std::max(u.t[0], u.t[1]), shorter = std::min(u.t[0], u.t[1]);
    return std::max(longer + kPairing * shorter, kYounger * shorter);
  };
  typedef std::pair<double, int> Entry;
  std::priority_queue<Entry, std::vector<Entry>, std::greater<Entry>> next;
  for (int i = 0; i < units; ++i) next.push({0.0, i});
  for (int i : order) {
    const int u = next.top().second;
    next.pop();
    const int slot = cut.row_slots == 2 && unit[u].t[1] < unit[u].t[0] ? 1 : 0;
    unit[u].t[slot] += l.pieces[i].us + (unit[u].in[slot].empty() ? 0.0 : kChained);
    unit[u].in[slot].push_back(i);
    next.push({done(unit[u]), u});
  }
  // units with two programs first, so that the second row's programs land beside the first ones
  std::vector<int> by(units);
  for (int i = 0; i < units; ++i) by[i] = i;
  for (Unit& u : unit)
    if (u.t[1] > u.t[0]) {
      std::swap(u.t[0], u.t[1]);
      std::swap(u.in[0], u.in[1]);
    }
  std::stable_sort(by.begin(), by.end(), [&](int a, int b) {
    const bool pa = !unit[a].in[1].empty(), pb = !unit[b].in[1].empty();
    return pa != pb ? pa : unit[a].t[0] > unit[b].t[0];
  });
  l.programs.clear();
  for (int row = 0; row < 2; ++row)
    for (int i : by)
      if (!unit[i].in[row].empty()) l.programs.push_back(std::move(unit[i].in[row]));
  // ---- duration: the narrow vnodes take the slots as they become free and slow the programs beside them
  l.wide_us = 0;
  for (const Unit& u : unit) l.wide_us = std::max(l.wide_us, done(u));
  double total = l.wide_us;
  if (narrow.block_us > 0) {
    const double work = narrow.block_us / m.heads;
    double end = 0;
    auto enough = [&](double t) {   // whether the narrow vnodes fit by time t; `end`: when the programs are done then
      double have = 0;
      end = 0;
      for (const Unit& u : unit) {
        const double second = u.t[1] > 0 ? u.t[1] * (1 + kPairing) : 0.0;
        const double beside = std::max(0.0, std::min(t, done(u)) - second);
        const double last = u.t[0] > 0 ? done(u) + kNarrowPairing * beside : 0.0;
        have += beside / kNarrowBeside + (kBlocksPerCu == 2 ? std::max(0.0, t - std::max(second, last)) : 0.0) + std::max(0.0, t - last);
        end = std::max(end, last);
      }
      return have >= work;
    };
    double lo = 0, hi = l.wide_us + work + 1.0;
    for (int i = 0; i < 14; ++i) {
      const double mid = 0.5 * (lo + hi);
      (enough(mid) ? hi : lo) = mid;
    }
    enough(hi);
    total = std::max({hi, end, narrow.longest_us});
  }
  l.total_us = overlapped(total, narrow.bytes_us);
}

}  // namespace

struct ft_schedule {
  std::vector<int32_t> arrays[FT_SCHEDULE_ARRAYS];
};

namespace {

void build(const Machine& m, int batch, Layout& l, std::vector<Narrow>& narrow, const int32_t* kv_entries, ft_schedule& s) {
  auto& A = s.arrays;
  std::vector<int32_t>&ko = A[FT_SCHEDULE_KV_OFFS], &kl = A[FT_SCHEDULE_KV_LENS], &qe = A[FT_SCHEDULE_Q_ENTRIES], &qo = A[FT_SCHEDULE_Q_OFFS],
                      &ql = A[FT_SCHEDULE_Q_LENS], &table = A[FT_SCHEDULE_PROG_TABLE];
  auto emit = [&](int64_t start, int32_t tokens, const int32_t* reqs, int n) {
    ko.push_back((int32_t)start);
    kl.push_back(tokens);
    qo.push_back((int32_t)qe.size());
    ql.push_back(n);
    qe.insert(qe.end(), reqs, reqs + n);
  };
  for (const std::vector<int>& program : l.programs) {
    table.push_back((int32_t)ko.size());
    for (int i : program) emit(l.pieces[i].start, l.pieces[i].tokens, l.pieces[i].reqs, l.pieces[i].n);
    table.push_back((int32_t)ko.size());
    table.push_back(0);
    table.push_back(0);
  }
  const int32_t wide = (int32_t)ko.size();
  for (const Narrow& v : narrow) emit(v.start, v.tokens, v.reqs, v.n);
  // scratch rows of every request, in row order
  std::vector<int32_t>&re = A[FT_SCHEDULE_REQ_ENTRIES], &ro = A[FT_SCHEDULE_REQ_OFFS], &rl = A[FT_SCHEDULE_REQ_LENS];
  rl.assign(batch, 0);
  ro.assign(batch, 0);
  for (int32_t r : qe) rl[r] += 1;
  for (int r = 1; r < batch; ++r) ro[r] = ro[r - 1] + rl[r - 1];
  re.assign(qe.size() + 32, -1);
  std::vector<int32_t> cursor(ro);
  for (size_t row = 0; row < qe.size(); ++row) re[cursor[qe[row]]++] = (int32_t)row;
  const int32_t programs = (int32_t)l.programs.size(), narrows = (int32_t)ko.size() - wide;
  A[FT_SCHEDULE_COUNTS] = {wide, narrows, programs, 0, 0};
  // ---- records (layouts: include/fasttree_hip.h)
  std::vector<int32_t>& req_table = A[FT_SCHEDULE_REQ_TABLE];
  req_table.assign((size_t)batch * 16, 0);
  for (int r = 0; r < batch; ++r) {
    int32_t* rec = &req_table[(size_t)r * 16];
    rec[0] = rl[r];
    rec[1] = ro[r];
    for (int i = 0; i < std::min(rl[r], 14); ++i) rec[2 + i] = re[ro[r] + i];
  }
  if (!kv_entries) return;
  std::vector<int32_t>& nt = A[FT_SCHEDULE_NARROW_TABLE];
  nt.assign((size_t)narrows * 64, 0);
  for (int32_t i = 0; i < narrows; ++i) {
    const int32_t v = wide + i;
    int32_t* rec = &nt[(size_t)i * 64];
    rec[0] = ko[v]; rec[1] = kl[v]; rec[2] = qo[v]; rec[3] = ql[v];
    if (ql[v] > 0)
      for (int r = 0; r < 16; ++r) rec[4 + r] = qe[qo[v] + std::min(r, ql[v] - 1)];
    if (kl[v] > 0)
      for (int t = 0; t < 32; ++t) rec[20 + t] = kv_entries[ko[v] + std::min(t, kl[v] - 1)];
  }
  std::vector<int32_t>& pr = A[FT_SCHEDULE_PROG_RECORDS];
  pr.assign((size_t)programs * 256, 0);
  for (int32_t p = 0; p < programs; ++p) {
    const int32_t v = table[4 * p];
    int32_t* rec = &pr[(size_t)p * 256];
    rec[0] = ko[v]; rec[1] = kl[v]; rec[2] = qo[v]; rec[3] = ql[v];
    // (the record holds 128 requests, and what one pass of a block serves)
    if (ql[v] < 1 || ql[v] > 128 || (int64_t)ql[v] * m.group > rows_per_block(m.head_dim)) continue;
    rec[4] = 1;
    for (int r = 0; r < 128; ++r) rec[8 + r] = qe[qo[v] + std::min(r, ql[v] - 1)];
    if (kl[v] > 0)
      for (int t = 0; t < 64; ++t) rec[136 + t] = kv_entries[ko[v] + std::min(t, kl[v] - 1)];
  }
}

// A record per wave of every narrow vnode, of a plan of whole paths.
void wave_records(const Machine& m, const int32_t* kv_entries, ft_schedule& s) {
  const std::vector<int32_t>& nt = s.arrays[FT_SCHEDULE_NARROW_TABLE];
  std::vector<int32_t>& wr = s.arrays[FT_SCHEDULE_WAVE_RECORDS];
  const int waves = FT_PATH_WAVES(m.head_dim);
  wr.reserve(nt.size() * waves);
  for (size_t at = 0; at < nt.size(); at += 64)
    for (int w = 0; w < waves; ++w) {
      int32_t* rec = &*wr.insert(wr.end(), nt.begin() + at, nt.begin() + at + 64);
      for (int i = 0; i < kTile; ++i) rec[20 + i] = kv_entries[rec[0] + std::min(w * kTile + i, rec[1] - 1)];
    }
}

// A launch: its programs, its narrow vnodes, and what the model expects of both stages.
struct Launch {
  Layout layout;
  std::vector<Narrow> narrow;
  Cut chosen{1, 0, 1, 1.0};
  bool programs = false;
  double score = 1e30;   // modelled: the first stage, and the partials of both
};

// The launch with runs of up to narrow_rows query rows served by waves of their own, wave_rows of them each.
// `bound`: a launch with a score of this or more is of no use (it comes back with the score kNone).
constexpr double kNone = 1e30;
Launch solve(const std::vector<Run>& runs, const Machine& m, int narrow_rows, int wave_rows, double bound = kNone) {
  const int block_rows = rows_per_block(m.head_dim);
  const int slots = m.block_slots();
  const double bytes_us = read_us(runs, m);
  std::vector<Run> wide;
  Launch out;
  std::vector<Narrow>& narrow = out.narrow;
  auto go_narrow = [&](const Run& r) {
    // a wave serves up to kWaveRows rows per pass; row chunks lie side by side, so that the second one finds the rows in L2
    const int cap = std::max(1, wave_rows / m.group), chunks = (int)std::max<int64_t>(1, ceil_div(r.n, cap));
    int64_t off = r.start;
    for (int32_t len : r.lens) {
      for (int c = 0; c < chunks; ++c) {
        const int base = r.n / chunks, extra = r.n % chunks, lo = c * base + std::min(c, extra);
        narrow.push_back({off, len, r.reqs + lo, base + (c < extra ? 1 : 0)});
      }
      off += len;
    }
  };
  int64_t wide_blocks = 0;
  for (const Run& r : runs) {
    // (a run without tokens has no steps to place: a wave writes its empty partial results)
    if ((int64_t)r.n * m.group <= narrow_rows || r.tokens == 0) go_narrow(r);
    else {
      wide.push_back(r);
      wide_blocks += (int64_t)r.lens.size() * ceil_div((int64_t)r.n * m.group, block_rows) * m.heads;
    }
  }
  // Short runs of a few dozen rows are bound by memory latency: where the wide blocks overfill the
  // machine they go with the narrow vnodes, eight of which a compute unit has in flight.
  if (wide_blocks > slots) {
    std::vector<Run> kept;
    for (Run& r : wide) {
      const int64_t rows = (int64_t)r.n * m.group;
      if (rows <= 64 && rows * *std::max_element(r.lens.begin(), r.lens.end()) <= 4096) go_narrow(r);
      else kept.push_back(std::move(r));
    }
    wide.swap(kept);
  }
  narrow = cut_long(std::move(narrow), m.group, m.heads, m.wave_slots());
  std::stable_sort(narrow.begin(), narrow.end(), [&](const Narrow& a, const Narrow& b) {
    return ceil_div(a.tokens, kTile) * passes(a, m) > ceil_div(b.tokens, kTile) * passes(b, m);
  });
  const NarrowLoad load = narrow_load(narrow, m, bytes_us);
  Layout& best = out.layout;
  Cut& chosen = out.chosen;
  double& score = out.score;
  out.programs = !wide.empty();
  double narrow_out = 0;
  for (const Narrow& v : narrow) narrow_out += v.n;
  const double narrow_scratch = 8.0 * narrow_out * m.group * m.heads * (m.head_dim + 1) / kScratchPerUs;
  const bool bounded = bound < kNone;
  if (bounded) score = bound - narrow_scratch;
  if (wide.empty()) {
    score = best.total_us = std::max({load.bytes_us, load.longest_us, load.block_us / slots});
  } else {
    for (int rows : {block_rows, 128, 64}) {
      if (rows > block_rows) continue;
      Cut cut{std::max(1, rows / m.group), 0, 0, 1.0};
      double whole = 0;
      for (const Run& r : wide) {
        const int chunks = (int)ceil_div(r.n, cut.rows_cap);
        whole = std::max(whole, kVnode + step_us((int)ceil_div((int64_t)ceil_div(r.n, chunks) * m.group, 16), m.head_dim, m.heads) * ceil_div(r.tokens, kTile));
      }
      double wide_sum = 0;
      for (const Piece& p : cut_runs(wide, m, Cut{cut.rows_cap, whole, 1, 1.0})) wide_sum += p.us;
      // A launch bound by reading keeps its wide vnodes on one slot per unit and in chunks of 128 rows, so
      // that every unit streams beside them all along (2048 requests with 1024 tokens each, 32/8 heads:
      // 1549 us, on both slots 1562, in chunks of 192 rows 1557; a 512-document tree 274 / 282 / 280).
      // With less than twice as much to read as to compute the second slot pays (1089 requests in 95 groups
      // of 869 tokens, 24/8 heads: 200 us, on one slot 212).
      const bool reading = bytes_us > 2 * wide_sum / m.units();
      if (reading && rows > 128) continue;
      const int row_slots = m.head_dim > 128 || reading ? 1 : 2;
      for (cut.row_slots = 1; cut.row_slots <= row_slots; ++cut.row_slots) {
        size_t last = 0;
        for (double us = whole; us == whole || us > kVnode + 1.0; us = kVnode + (us - kVnode) * 0.8) {
          cut.piece_us = us;
          cut.last = 1.0;
          std::vector<Piece> pieces = cut_runs(wide, m, cut);
          if (pieces.size() == last) continue;
          last = pieces.size();
          double rows_out = 0, sum = 0, longest = 0;
          for (const Piece& p : pieces) {
            rows_out += p.n;
            sum += p.us;
            longest = std::max(longest, p.us);
          }
          const double scratch = 8.0 * rows_out * m.group * m.heads * (m.head_dim + 1) / kScratchPerUs;
          // (the first layout of all is taken as it is: runs that are many pieces uncut have to be placed too)
          const bool taken = bounded || !best.programs.empty();
          if (taken && (last > 4096 || scratch > score)) break;
          // (what no placement goes below)
          const double least = std::max(longest, sum / m.units() * (cut.row_slots == 2 ? 0.5 * (1 + kPairing) : 1.0));
          if (taken && overlapped(least, load.bytes_us) + scratch >= score) continue;
          double even_us = 0;
          // Even pieces, and a shorter last one: 425 requests of 32/8 heads on 4289 tokens 62.4 us, with even pieces only
          // 66.9, with 0.8 66.9; the 400-request tree 57.4, 60.0 and 57.3; 507 requests of 64-dim heads 49.8, 52.7 and
          // 49.3; 608 of 24/8 heads 35.3, 34.2 and 35.4.
          for (double ratio : {1.0, 0.87}) {
            if (ratio < 1.0) {
              // (it gains a tenth at most)
              if (cut.row_slots == 1 || even_us > 1.1 * score) break;
              cut.last = ratio;
              pieces = cut_runs(wide, m, cut);
            }
            Layout l;
            l.pieces = std::move(pieces);
            place(l, m, cut, load);
            even_us = l.total_us + scratch;
            if ((!bounded && best.programs.empty()) || l.total_us + scratch < score) {
              score = l.total_us + scratch;
              best = std::move(l);
              chosen = cut;
            }
          }
        }
      }
    }
  }
  score += narrow_scratch;
  if (bounded && (score >= bound || (out.programs && best.programs.empty()))) score = kNone;
  return out;
}

// The launch of a list of runs.
Launch best_launch(const std::vector<Run>& runs, const Machine& m, double bound = kNone) {
  Launch best = solve(runs, m, kWaveRows, kWaveRows, bound);
  // In a small launch a wide vnode's start-up is most of it, and runs of a few more rows than a wave's are
  // sooner done by several waves of one 16-row group each (whole calls: 3 requests of 16/1 heads of 256 on an
  // 881-token run 18.6 us wide, 14.8 narrow; 50 requests of 32/8 heads of 256 in six groups of 611 tokens
  // 30.9 and 24.9; 25 requests of 32/8 heads in two groups of 352 tokens 17.9 and 12.3; 188 requests of 16/1 heads
  // in 19 groups of 160 rows and 259 tokens 17.8 and 14.5, 46 of 24/8 heads on 236 tokens 13.7 and 11.8).  A larger
  // one would read their rows twice.
  double bytes = 0;
  for (const Run& r : runs) bytes += 4.0 * m.head_dim * r.tokens * m.heads;
  if (bytes * 256 / m.cus < kSmallLaunchBytes) {
    int tried = 16;
    for (int limit : {kWaveRows, 64, 128, 256}) {
      bool any = false;
      for (const Run& r : runs) any = any || ((int64_t)r.n * m.group > tried && (int64_t)r.n * m.group <= limit && r.tokens > 0);
      tried = limit;
      if (!any) continue;
      Launch other = solve(runs, m, limit, 16, std::min(bound, best.score));
      if (other.score < best.score) best = std::move(other);
    }
  }
  return best;
}

// What a launch of whole paths is modelled to take: `paths` vnodes, the longest of `longest` tokens.
double whole_paths_us(int64_t paths, int64_t longest, const Machine& m) {
  const int64_t rounds = ceil_div(ceil_div(longest, kTile), FT_PATH_WAVES(m.head_dim));
  return kPathStart + kPathRound * (1 + kPathShared * paths * m.heads / m.cus) * std::min(1.5, m.head_dim / 128.0) * rounds;
}

// A tree's whole paths, one vnode per leaf, where they are a launch of less than a block per unit that takes less than
// `bound` (`taken`).
int whole_paths(const Tree& tree, const Machine& m, int batch, double bound, TreeRuns& t, double& us, bool& taken) {
  taken = false;
  std::vector<int64_t> path(tree.n);
  int64_t leaves = 0, longest = 0;
  for (int v = 0; v < tree.n; ++v) {
    path[v] = tree.seqlen[v] + (v > 0 ? path[tree.parent[v]] : 0);
    if (tree.num_children[v] > 0) continue;
    longest = std::max(longest, path[v]);
    ++leaves;
    if (path[v] < 1 || tree.requests(v) * m.group > kWaveRows) return FT_SCHEDULE_OK;
  }
  us = whole_paths_us(leaves, longest, m);
  if (m.head_dim < 32 || leaves * m.heads >= m.cus || us >= bound) return FT_SCHEDULE_OK;
  std::vector<int32_t> all(tree.n, 1);
  all[0] = 0;
  if (int rc = tree_runs(tree, std::move(all), t)) return rc;
  int64_t requests = 0;
  for (const Run& r : t.runs) requests += r.n;
  // (every request in one vnode, whatever the arguments say of inner nodes)
  std::vector<char> seen(batch, 0);
  for (const Run& r : t.runs)
    for (int i = 0; i < r.n; ++i) {
      if (seen[r.reqs[i]]) return FT_SCHEDULE_OK;
      seen[r.reqs[i]] = 1;
    }
  taken = requests == batch && (int64_t)t.runs.size() == leaves;
  return FT_SCHEDULE_OK;
}

// (request, token) pairs of a list of runs, pieces or narrow vnodes.
template <typename List, typename Tokens>
double pairs(const List& list, Tokens tokens) {
  double sum = 0;
  for (const auto& x : list) sum += (double)x.n * tokens(x);
  return sum;
}

// Writes the schedule.
int finish(Launch& best, const std::vector<Run>& runs, const Machine& m, int batch, const int32_t* kv_entries, ft_schedule& s, double* modelled_us) {
  // A schedule attends what its runs attend, whatever the search did: anything less is an error, not a result.
  // (whole numbers below 2^53 in doubles: exact)
  double placed = pairs(best.narrow, [](const Narrow& v) { return v.tokens; });
  for (const std::vector<int>& program : best.layout.programs)
    for (int i : program) placed += (double)best.layout.pieces[i].n * best.layout.pieces[i].tokens;
  if (placed != pairs(runs, [](const Run& r) { return r.tokens; })) return FT_SCHEDULE_ERR_INCOMPLETE;
  build(m, batch, best.layout, best.narrow, kv_entries, s);
  s.arrays[FT_SCHEDULE_COUNTS][3] = best.programs ? best.chosen.row_slots * m.cus : m.block_slots();
  if (modelled_us) *modelled_us = best.layout.total_us + kLaunch;
  return FT_SCHEDULE_OK;
}

}  // namespace

extern "C" {

int ft_schedule_create(int64_t num_vnodes, const int32_t* kv_offs, const int32_t* kv_lens, const int32_t* q_offs, const int32_t* q_lens,
                       int64_t num_rows, const int32_t* q_entries, int64_t num_kv_entries, const int32_t* kv_entries, int batch_size,
                       int group, int num_kv_heads, int head_dim, int num_cus, double* modelled_us, ft_schedule** out) {
  if (!out || (num_vnodes > 0 && (!kv_offs || !kv_lens || !q_offs || !q_lens)) || (num_rows > 0 && !q_entries)) return FT_SCHEDULE_ERR_NULL_POINTER;
  if (num_vnodes < 0 || num_rows < 0 || batch_size < 0 || group < 1 || num_kv_heads < 1 || head_dim < 1 || num_cus < 1) return FT_SCHEDULE_ERR_ARGUMENT;
  for (int64_t v = 0; v < num_vnodes; ++v) {
    if (kv_offs[v] < 0 || kv_lens[v] < 0 || q_offs[v] < 0 || q_lens[v] < 0 || (int64_t)q_offs[v] + q_lens[v] > num_rows) return FT_SCHEDULE_ERR_ARGUMENT;
    if (kv_entries && (int64_t)kv_offs[v] + kv_lens[v] > num_kv_entries) return FT_SCHEDULE_ERR_ARGUMENT;
  }
  for (int64_t i = 0; i < num_rows; ++i)
    if (q_entries[i] < 0 || q_entries[i] >= batch_size) return FT_SCHEDULE_ERR_ARGUMENT;
  try {
    const Machine m{num_cus, num_kv_heads, group, head_dim};
    auto s = std::make_unique<ft_schedule>();
    const std::vector<Run> runs = runs_of(num_vnodes, kv_offs, kv_lens, q_offs, q_lens, q_entries);
    Launch launch = best_launch(runs, m);
    // (records of narrow vnodes are made where the slots are known; without them the kernel of programs contracts what rounding leaves
    // over.  Head_dim 16 has no such kernel, and vnodes that are joined would round more: 2.044e-4 of P where 2.036e-4.)
    if (!kv_entries && m.head_dim >= 32 && !launch.layout.programs.empty()) {
      std::vector<Narrow> joined = join_short(launch.narrow, (int64_t)launch.layout.programs.size(), m.heads, m.wave_slots());
      if (joined.size() < launch.narrow.size()) {
        launch.narrow = std::move(joined);
        place(launch.layout, m, launch.chosen, narrow_load(launch.narrow, m, read_us(runs, m)));   // (the same programs, and what they take beside these)
      }
    }
    if (int rc = finish(launch, runs, m, batch_size, kv_entries, *s, modelled_us)) return rc;
    *out = s.release();
    return FT_SCHEDULE_OK;
  } catch (const std::exception&) {   // bad_alloc, length_error
    return FT_SCHEDULE_ERR_MEMORY;
  }
}

int ft_schedule_tree(int num_nodes, const int32_t* parent, const int32_t* seqlen, const int32_t* num_children, const int64_t* req_offs,
                     const int32_t* req_ids, const int64_t* kv_ptrs, const int32_t* kv_slot_map, int64_t kv_slot_map_len, int batch_size,
                     int group, int num_kv_heads, int head_dim, int num_cus, double* modelled_us, ft_schedule** out) {
  return ft_schedule_tree_weighed(num_nodes, parent, seqlen, num_children, req_offs, req_ids, kv_ptrs, kv_slot_map, kv_slot_map_len, nullptr,
                                  batch_size, group, num_kv_heads, head_dim, num_cus, modelled_us, out);
}

int ft_schedule_tree_weighed(int num_nodes, const int32_t* parent, const int32_t* seqlen, const int32_t* num_children, const int64_t* req_offs,
                             const int32_t* req_ids, const int64_t* kv_ptrs, const int32_t* kv_slot_map, int64_t kv_slot_map_len,
                             const int32_t* decided, int batch_size, int group, int num_kv_heads, int head_dim, int num_cus,
                             double* modelled_us, ft_schedule** out) {
  return ft_schedule_tree_within(num_nodes, parent, seqlen, num_children, req_offs, req_ids, kv_ptrs, kv_slot_map, kv_slot_map_len, decided, -1,
                                 batch_size, group, num_kv_heads, head_dim, num_cus, modelled_us, out);
}

int ft_schedule_tree_within(int num_nodes, const int32_t* parent, const int32_t* seqlen, const int32_t* num_children, const int64_t* req_offs,
                            const int32_t* req_ids, const int64_t* kv_ptrs, const int32_t* kv_slot_map, int64_t kv_slot_map_len,
                            const int32_t* decided, int64_t most_kv_entries, int batch_size, int group, int num_kv_heads, int head_dim,
                            int num_cus, double* modelled_us, ft_schedule** out) {
  if (!parent || !seqlen || !num_children || !req_offs || !kv_ptrs || !out) return FT_SCHEDULE_ERR_NULL_POINTER;
  if (num_nodes < 1 || batch_size < 0 || group < 1 || num_kv_heads < 1 || head_dim < 1 || num_cus < 1) return FT_SCHEDULE_ERR_ARGUMENT;
  for (int v = 0; v < num_nodes; ++v) {
    if ((v > 0 && (parent[v] < 0 || parent[v] >= v)) || seqlen[v] < 0 || req_offs[v + 1] < req_offs[v]) return FT_SCHEDULE_ERR_ARGUMENT;
    if (decided && (decided[v] < 0 || decided[v] > (v > 0 ? 1 : 0))) return FT_SCHEDULE_ERR_ARGUMENT;
  }
  if (req_offs[num_nodes] > 0 && !req_ids) return FT_SCHEDULE_ERR_NULL_POINTER;
  for (int64_t i = 0; i < req_offs[num_nodes]; ++i)
    if (req_ids[i] < 0 || req_ids[i] >= batch_size) return FT_SCHEDULE_ERR_ARGUMENT;
  try {
    const Machine m{num_cus, num_kv_heads, group, head_dim};
    const Tree tree{num_nodes, parent, seqlen, num_children, req_offs, req_ids, kv_ptrs, kv_slot_map, kv_slot_map_len};
    TreeRuns t;
    std::vector<int32_t> along = taken_along(tree, m), other_along;
    if (decided) other_along.assign(decided, decided + num_nodes);
    const bool differ = decided && other_along != along;
    if (int rc = tree_runs(tree, std::move(along), t)) return rc;
    Launch launch = best_launch(t.runs, m);
    if (differ) {
      // The bytes leave out what a vnode of its own costs besides its partials, a start-up on a wave or a block, and
      // trees of many short nodes were slower by them than by the planner's padding costs: 1024 leaves of 16 tokens
      // under five levels, 32/32 heads, 172.6 us and 155.4; 256 leaves of 32 tokens on a prompt of 256, 16/1 heads,
      // 14.9 and 12.2.  Others are the other way round (143 against 121 us), so the modelled launches decide.
      TreeRuns u;
      if (int rc = tree_runs(tree, std::move(other_along), u)) return rc;
      Launch other = best_launch(u.runs, m, std::min(kClearlyBetter * launch.score, launch.score - kClearlyUs));
      if (other.score < kNone) {
        launch = std::move(other);
        t = std::move(u);
      }
    }
    auto s = std::make_unique<ft_schedule>();
    TreeRuns u;
    double us = 0;
    bool whole;
    if (int rc = whole_paths(tree, m, batch_size, kClearlyBetter * (launch.score + kLaunch), u, us, whole)) return rc;
    // (a path's tokens stand in the slot list once per leaf)
    if (most_kv_entries >= 0 && (int64_t)u.kv_entries.size() > most_kv_entries) whole = false;
    if (whole) {
      launch = Launch{};
      for (const Run& r : u.runs) launch.narrow.push_back({r.start, (int32_t)r.tokens, r.reqs, r.n});
      std::stable_sort(launch.narrow.begin(), launch.narrow.end(), [](const Narrow& a, const Narrow& b) { return a.tokens > b.tokens; });
      launch.layout.total_us = us - kLaunch;
      t = std::move(u);
    }
    if (int rc = finish(launch, t.runs, m, batch_size, t.kv_entries.data(), *s, modelled_us)) return rc;
    if (whole) wave_records(m, t.kv_entries.data(), *s);
    s->arrays[FT_SCHEDULE_KV_ENTRIES] = std::move(t.kv_entries);
    s->arrays[FT_SCHEDULE_NODE_ASSIGNMENTS] = std::move(t.along);
    *out = s.release();
    return FT_SCHEDULE_OK;
  } catch (const std::exception&) {   // bad_alloc, length_error
    return FT_SCHEDULE_ERR_MEMORY;
  }
}

int64_t ft_schedule_size(const ft_schedule* s, int which) {
  return s && which >= 0 && which < FT_SCHEDULE_ARRAYS ? (int64_t)s->arrays[which].size() : -1;
}

int ft_schedule_pack(const ft_schedule* s, int32_t* dst, int64_t capacity, int64_t offsets[FT_SCHEDULE_ARRAYS], int64_t* total) {
  if (!s || !offsets || !total) return FT_SCHEDULE_ERR_NULL_POINTER;
  int64_t at = 0;
  for (int i = 0; i < FT_SCHEDULE_ARRAYS; ++i) {
    offsets[i] = at;
    at += ceil_div((int64_t)s->arrays[i].size(), 64) * 64;
  }
  *total = at;
  if (!dst) return FT_SCHEDULE_OK;
  if (at > capacity) return FT_SCHEDULE_ERR_ARGUMENT;
  for (int i = 0; i < FT_SCHEDULE_ARRAYS; ++i)
    if (!s->arrays[i].empty()) std::memcpy(dst + offsets[i], s->arrays[i].data(), s->arrays[i].size() * sizeof(int32_t));
  return FT_SCHEDULE_OK;
}

void ft_schedule_destroy(ft_schedule* s) { delete s; }

}  // extern "C"
