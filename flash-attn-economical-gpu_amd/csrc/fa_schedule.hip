// Host side: how long an attention grid takes, in steps of its kernel, by following the blocks through
// the chip's dispatch. The tile choice compares kernels with it (gfx950_configs.py holds each kernel's
// step time): in C++ because a new sequence length pays for it once, 10-40 us for four kernels where the
// same simulation in Python took 0.2-0.6 ms.
#include <algorithm>
#include <cstdint>
#include <exception>
#include <functional>  // std::greater
#include <set>
#include <vector>

#include "../../include/fa_gfx950.h"

namespace {

constexpr int kXcds = 8, kEngines = 4, kCusPerEngine = 8;  // MI355X: 32 CUs per XCD, in shader engines of 8
constexpr int kCusPerXcd = kEngines * kCusPerEngine;
constexpr int64_t kMaxBlocks = 4096;  // beyond, rounds are many and the schedule matters little
// A block with at most half its rows costs this much of block_steps: half its waves load no Q and store no O.
constexpr double kHalfBlock = 0.7;
// A CU shared by m blocks of a four-wave kernel: a step of each takes kShared[m] times its step beside
// one other; alone it takes `alone` times that.
constexpr double kShared3 = 1.4, kShared4 = 1.8;

struct Grid {
  int blocks_per_head;
  int64_t total;
  std::vector<double> cost;  // steps of time by query block of a head
};

// One block to a CU: the XCD hands its blocks out in order, to its engines in turn; a block waits for a
// CU of its engine, and all later blocks with it. (at(k): query block of the XCD's k-th.)
template <class BlockAt>
double end_exclusive(int64_t n, const BlockAt& at, const Grid& g) {
  std::vector<double> busy[kEngines];
  double start = 0, end = 0;
  for (int64_t k = 0; k < n; ++k) {
    std::vector<double>& cus = busy[k % kEngines];  // min-heap of the engine's end times
    double free_at = 0;
    if ((int)cus.size() >= kCusPerEngine) {
      std::pop_heap(cus.begin(), cus.end(), std::greater<double>());
      free_at = cus.back();
      cus.pop_back();
    }
    start = std::max(start, free_at);
    cus.push_back(start + g.cost[at(k)]);
    std::push_heap(cus.begin(), cus.end(), std::greater<double>());
    end = std::max(end, start + g.cost[at(k)]);
  }
  return end;
}

// Several blocks to a CU, each the slower the more share it. Equal blocks (spread) do not end at once as
// they would here: CUs free up one after the other, and the last blocks start before the round is over.
template <class BlockAt>
double end_shared(int64_t n, const BlockAt& at, const Grid& g, int per_cu, double alone, bool spread) {
  const double pace[5] = {0, alone, 1, kShared3, kShared4};
  constexpr double kIdle = 1e300;
  double left[kCusPerXcd][4], now[kCusPerXcd] = {}, done[kCusPerXcd];  // done: when the CU's next block ends
  int count[kCusPerXcd] = {};
  std::fill(done, done + kCusPerXcd, kIdle);
  auto advance = [&](int c, double t) {
    for (int i = 0; i < count[c]; ++i) left[c][i] -= (t - now[c]) / pace[count[c]];
    now[c] = t;
  };
  auto update = [&](int c) {
    done[c] = count[c] == 0 ? kIdle : now[c] + *std::min_element(left[c], left[c] + count[c]) * pace[count[c]];
  };
  int64_t k = 0;
  auto dispatch = [&](double t) {
    while (k < n) {
      const int first = (int)(k % kEngines) * kCusPerEngine;
      const int c = (int)(std::min_element(count + first, count + first + kCusPerEngine) - count);
      if (count[c] == per_cu) return;
      advance(c, t);
      left[c][count[c]++] = g.cost[at(k)] * (spread ? 0.95 + 0.1 * (double)(k * 37 % 101) / 100 : 1.0);
      ++k;
      update(c);
    }
  };
  dispatch(0);
  for (double t = 0;;) {
    const int c = (int)(std::min_element(done, done + kCusPerXcd) - done);
    if (done[c] == kIdle) return t;
    t = done[c];
    advance(c, t);
    double* const ended = std::min_element(left[c], left[c] + count[c]);
    *ended = left[c][--count[c]];
    update(c);
    dispatch(t);
  }
}

// The persistent kernel's sequences: rounds over the workgroups, every second one backwards.
template <class BlockAt>
double end_persistent(int64_t n, int workgroups, const BlockAt& at, const Grid& g) {
  std::vector<double> end(workgroups, 0.0);
  for (int64_t k = 0; k < n; ++k) {
    const int64_t round = k / workgroups;
    const int slot = (int)(k % workgroups);
    end[round & 1 ? workgroups - 1 - slot : slot] += g.cost[at(k)];
  }
  return *std::max_element(end.begin(), end.end());
}

double grid_steps(int rows, int tiles_per_step, int order, int per_cu, double block_steps, double alone, int BH, int M,
                  int N, bool causal) {
  if (rows <= 0 || tiles_per_step <= 0 || per_cu < 1 || per_cu > 4 || BH <= 0 || M <= 0 || N < 0) return -1;
  Grid g;
  g.blocks_per_head = (int)(((int64_t)M + rows - 1) / rows);
  g.total = (int64_t)g.blocks_per_head * BH;
  if (g.total > kMaxBlocks) return -1;
  for (int i = 0; i < g.blocks_per_head; ++i) {
    const int64_t keys = causal ? std::min<int64_t>(N, (int64_t)(i + 1) * rows) : N;
    const int64_t tiles = (keys + 63) / 64;
    const bool half = M - (int64_t)i * rows <= rows / 2;
    g.cost.push_back(block_steps * (half ? kHalfBlock : 1.0) + (double)((tiles + tiles_per_step - 1) / tiles_per_step));
  }
  const int nb = g.blocks_per_head;
  auto query_block = [&](int64_t pid) { return causal ? nb - 1 - (int)(pid % nb) : (int)(pid % nb); };
  const bool by_xcd = g.total % kXcds == 0;  // each XCD has a run of its own (xcd_remap, item_pid)
  const int64_t per = by_xcd ? g.total / kXcds : (g.total + kXcds - 1) / kXcds;
  if (order == FA_GRID_PERSISTENT && !by_xcd)
    return end_persistent(g.total, (int)std::min<int64_t>(g.total, kXcds * kCusPerXcd), query_block, g);
  const bool by_weight = order == FA_GRID_HEAVIEST_FIRST && causal;
  double end = 0;
  std::set<int64_t> seen;  // XCDs whose runs start at the same query block take the same time
  // shared CUs even long runs out (and take longest to follow): a few of the XCDs will do
  const int stride = per_cu > 1 && per > 2 * kCusPerXcd ? 3 : 1;
  for (int x = 0; x < std::min<int64_t>(kXcds, g.total); x += stride) {
    if (!by_weight && !seen.insert(causal ? (by_xcd ? x * per : x) % nb : 0).second) continue;
    const auto at = [&](int64_t k) {
      return by_weight ? nb - 1 - (int)((x + kXcds * k) / BH) : query_block(by_xcd ? x * per + k : x + kXcds * k);
    };
    const int64_t n = by_xcd ? per : (g.total - x + kXcds - 1) / kXcds;
    if (order == FA_GRID_PERSISTENT)
      end = std::max(end, end_persistent(n, (int)std::min<int64_t>(n, kCusPerXcd), at, g));
    else if (per_cu > 1)
      end = std::max(end, end_shared(n, at, g, per_cu, alone, !causal));
    else
      end = std::max(end, end_exclusive(n, at, g));
  }
  return end;
}

}  // namespace

extern "C" double fa_grid_steps(int32_t rows, int32_t tiles_per_step, int32_t order, int32_t per_cu, double block_steps,
                                double alone, int32_t BH, int32_t M, int32_t N, int32_t causal) {
  try {
    return grid_steps(rows, tiles_per_step, order, per_cu, block_steps, alone, BH, M, N, causal != 0);
  } catch (const std::exception&) {  // out of memory: the caller's other rule
    return -1;
  }
}
