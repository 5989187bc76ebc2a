// Checks the runs of split prefill launches (bnr::plan_prefill_runs) over
// seeded shapes (1 to 5000 tokens, 0 to 9000 cached rows, 1 to 8 kv heads of
// 2, 4 or 8 query heads, 80 and 256 CUs, few and many states), decoding every
// run's words the way the kernel does: the key tiles 0 .. nk - 1 of every query
// unit are covered once, in order; the pieces of a unit are numbered 0 .. nch -
// 1 in key order and share one slot base; slots of different units are
// disjoint and within n_slots <= max_slots; the grid's numbering reaches every
// (kv head, run) once; no run is empty.  Then measured shapes on both sides of the
// line between split and fp32 launches (bnr::prefill_split_pays).  Prints "ok <plans>" or the first
// failing case.
#include <cstdio>
#include <random>
#include <vector>

#include "bnr_internal.h"

using namespace bnr;

static bool check(const PrefillRunsArgs &a, int group, long long max_slots) {
  const int uq = split_unit(group);
  const int rows = a.start_pos + a.n_tokens;
  auto nk = [&](int u) { return (std::min(a.start_pos + (u + 1) * uq, rows) + 31) / 32; };
  if (a.n_units != (a.n_tokens + uq - 1) / uq) return false;
  std::vector<std::vector<int>> pieces((size_t)a.n_units);  // (ch, nch, base) of each unit's pieces
  int u = 0, kt = 0;
  for (int r = 0; r < a.n_runs; ++r) {
    const unsigned w0 = a.run[r][0], w1 = a.run[r][1], w2 = a.run[r][2];
    if ((int)(w0 & 0xffff) != u || (int)(w0 >> 16) != kt) return false;
    int left = (int)(w1 & 0xffff);
    if (left < 1) return false;
    bool first = true;
    while (left > 0) {
      if (u >= a.n_units) return false;
      const int take = std::min(left, nk(u) - kt);
      left -= take;
      kt += take;
      const bool last = left == 0;
      pieces[(size_t)u].insert(pieces[(size_t)u].end(),
                               {first ? (int)(w1 >> 24) : 0,
                                first ? (int)(w1 >> 16 & 255) : last ? (int)(w2 >> 20) : 1,
                                (int)(first ? w2 & 1023 : w2 >> 10 & 1023)});
      if (!first && !last && kt != nk(u)) return false;
      if (kt == nk(u)) {
        ++u;
        kt = 0;
      }
      first = false;
    }
  }
  if (u != a.n_units || kt != 0) return false;
  std::vector<char> used((size_t)std::max(a.n_slots, 1), 0);
  for (const auto &p : pieces) {
    const int n = (int)p.size() / 3;
    for (int c = 0; c < n; ++c) {
      if (p[3 * c] != c || p[3 * c + 1] != n) return false;
      if (n == 1) continue;
      const int slot = p[3 * c + 2] + c;
      if (p[3 * c + 2] != p[2] || slot >= a.n_slots || used[(size_t)slot]++) return false;
    }
  }
  if (a.n_slots > max_slots) return false;
  // the kernel's numbering of the grid
  std::vector<char> seen((size_t)(a.n_kv * a.n_runs), 0);
  if (a.grid % 16) return false;
  for (int i = 0; i < a.grid; ++i) {
    const int per_xcd = a.grid >> 3, j8 = i >> 3, half = split_waves(group) == 4 ? per_xcd >> 1 : per_xcd;
    const int id = (i & 7) * per_xcd + (split_waves(group) == 4 ? (j8 % half) * 2 + j8 / half : j8);
    if (id / a.n_runs >= a.n_kv) continue;
    if (seen[(size_t)id]++) return false;
  }
  for (char c : seen)
    if (!c) return false;
  return true;
}

// Shapes on both sides of the line between split and fp32 launches, each at
// least 8 % faster (MI355X) with the launch named: tokens, cached rows, heads, kv heads.
struct Line {
  int n, start, heads, kv;
  bool split;
};
constexpr Line kLine[] = {
    {256, 0, 20, 5, false},  {1024, 0, 20, 5, true},  {333, 1207, 20, 5, true}, {256, 2000, 20, 5, true},
    {64, 2000, 20, 5, false}, {16, 32000, 20, 5, false}, {128, 8000, 20, 5, true}, {96, 0, 4, 1, false},
    {1024, 0, 4, 1, true},   {512, 0, 2, 1, false},   {192, 2000, 2, 1, false}, {640, 0, 4, 2, false},
    {512, 0, 16, 2, false},  {768, 0, 16, 2, true},   {96, 8000, 8, 1, false},  {384, 8000, 8, 1, true}};

int main() {
  for (const Line &l : kLine)
    if (prefill_split_pays(l.n, l.start, l.heads, l.kv) != l.split) {
      std::printf("FAIL line: n %d start %d heads %d/%d\n", l.n, l.start, l.heads, l.kv);
      return 1;
    }
  std::mt19937 rng(20261204);
  int plans = 0;
  for (int it = 0; it < 4000; ++it) {
    const int groups[] = {2, 4, 8}, kvs[] = {1, 2, 3, 5, 8};
    const int group = groups[rng() % 3], n_cu = rng() % 4 ? 256 : 80;
    PrefillRunsArgs a{};
    a.n_kv = kvs[rng() % 5];
    a.n_tokens = 1 + (int)(rng() % (it % 2 ? 5000u : 200u));
    a.start_pos = rng() % 3 ? (int)(rng() % 9000u) : 0;
    a.n_heads = a.n_kv * group;
    const long long max_slots = it % 5 ? 1000 : 3 + (long long)(rng() % 60u);
    if (!plan_prefill_runs(a, group, n_cu, max_slots) || !check(a, group, max_slots)) {
      std::printf("FAIL n %d start %d n_kv %d group %d cu %d slots %lld\n", a.n_tokens, a.start_pos,
                  a.n_kv, group, n_cu, max_slots);
      return 1;
    }
    ++plans;
  }
  std::printf("ok %d\n", plans);
  return 0;
}
