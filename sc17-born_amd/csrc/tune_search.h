// tune_search.h -- the autotuner's search over tile shapes and z chunks.
//
// z chunks split the nzi interior planes evenly (ceil(nzi / k) for k chunks,
// two planes or more): no block marches more planes than the others, and the
// number of blocks can match what the CUs hold at once.  Which k is best
// depends on the tile and the grid: a launch wants some hundreds of blocks at
// least (with 64^3 cells, chunks of 2 planes: 7.4 us per FP32 forward step; of
// 19 planes, 23.6 us) and few planes read twice (304^3: chunks of 74 planes,
// 164 us; of 37, 172 us).  So each shape (with one plane of lookahead) is first
// timed with the chunks that come nearest to five numbers of blocks, then the
// best five shapes with every chunk that gives from half to twice as many
// blocks as their best, and with two planes of lookahead; the four fastest of
// all are timed again, round-robin.  Grids of so many tiles that even chunks of
// 64 planes give more blocks than that are also timed with these (8 windows of
// 256-336 x 352, 24-bit forward: 1.43 ms with the 5120 blocks that chunks were
// cut at, 1.40 with chunks of 32 planes).
#ifndef BORN_TUNE_SEARCH_H
#define BORN_TUNE_SEARCH_H

#include <algorithm>
#include <vector>

namespace born {

struct TuneChoice {
  int shape, zchunk;
  float ms;  // per launch
};

// The fastest of the n shapes (cells per lane vx, which must divide xdiv;
// lookahead la; ry, wy and lx) and z chunks, or of the shapes with chunk zfixed
// (> 0).  tiles(shape) is the number of xy tiles; time(shape, zchunk, untimed,
// reps, &ms) runs that many launches, the last `reps` of them timed together,
// and returns 0, or an error that ends the search.
template <class Shape, class Tiles, class Time>
int tune_search(const Shape *shapes, int n, int xdiv, int nzi, int zfixed, Tiles tiles,
                Time time, TuneChoice *out) {
  constexpr int kMinBlocks = 128, kMaxBlocks = 5120, kManyBlocks = 3450, kManyPlanes = 64;
  constexpr float kShort = .03f;  // ms: launches of a few us
  std::vector<TuneChoice> cand;
  float single = 1e30f;  // the fastest lone launch
  auto try_one = [&](int sh, int zc) -> int {
    for (const TuneChoice &c : cand)
      if (c.shape == sh && c.zchunk == zc) return 0;
    TuneChoice c{sh, zc, 0.f};
    // One launch tells the hopeless ones.  A lone launch takes about 2 us more
    // than one of a row, so it is held against lone launches, and more closely
    // where these us weigh (held against the fastest of a row, a launch of
    // 4.3 us was dropped for the 6.6 us that it took alone).  The very first
    // one loads the kernels' code (2.4 to 3.7 ms) and is not timed.
    const float limit = (single < kShort ? 1.1f : 1.4f) * single;
    if (const int e = time(sh, zc, cand.empty() ? 1 : 0, 1, &c.ms)) return e;
    const bool fair = c.ms < limit;
    single = std::min(single, c.ms);
    // launches of a few us are timed over more of them
    if (fair)
      if (const int e = time(sh, zc, 1, c.ms < kShort ? 10 : 3, &c.ms)) return e;
    cand.push_back(c);
    return 0;
  };
  auto faster = [](const TuneChoice &a, const TuneChoice &b) { return a.ms < b.ms; };
  // the z chunks of a shape with lo to hi blocks, coarse to fine; if none,
  // the one nearest to that
  auto chunks = [&](int sh, double lo, double hi) {
    std::vector<int> zcs;
    const int nt = std::max(1, tiles(sh)), kmax = std::max(1, nzi / 2);
    int near = 1;
    for (int k = 1; k <= kmax; k++) {
      if ((double)nt * k < lo) near = k;
      if ((double)nt * k < lo || (double)nt * k > hi) continue;
      const int zc = (nzi + k - 1) / k;
      if (zcs.empty() || zcs.back() != zc) zcs.push_back(zc);
    }
    if (zcs.empty()) zcs.push_back((nzi + near - 1) / near);
    return zcs;
  };
  for (int sh = 0; sh < n; sh++) {
    if (xdiv % shapes[sh].vx || shapes[sh].la != 1) continue;
    if (zfixed > 0) {
      if (const int e = try_one(sh, zfixed)) return e;
      continue;
    }
    const int nt = std::max(1, tiles(sh));
    std::vector<double> targets = {256., 512., 768., 1280., 2300.};
    const double many = (double)nt * ((nzi + kManyPlanes - 1) / kManyPlanes);
    if (many > kManyBlocks) targets.push_back(many);
    const std::vector<int> zcs = chunks(sh, kMinBlocks, std::max<double>(kMaxBlocks, many));
    for (double target : targets) {
      int best = zcs[0];
      double off = 1e30;
      for (int zc : zcs) {
        const double nb = (double)nt * ((nzi + zc - 1) / zc);
        const double d = nb > target ? nb / target : target / nb;
        if (d < off) {
          off = d;
          best = zc;
        }
      }
      if (const int e = try_one(sh, best)) return e;
    }
  }
  std::vector<TuneChoice> order = cand;
  std::sort(order.begin(), order.end(), faster);
  std::vector<int> done;
  for (size_t i = 0; i < order.size() && done.size() < 5; i++) {
    const int sh = order[i].shape, zc = order[i].zchunk;
    if (std::find(done.begin(), done.end(), sh) != done.end()) continue;
    done.push_back(sh);
    const Shape &ts = shapes[sh];
    for (int l = 0; l < n; l++) {
      const Shape &o = shapes[l];
      if (o.la == 2 && o.ry == ts.ry && o.wy == ts.wy && o.vx == ts.vx && o.lx == ts.lx)
        if (const int e = try_one(l, zc)) return e;
    }
    if (zfixed > 0) continue;
    const double nb = (double)std::max(1, tiles(sh)) * ((nzi + zc - 1) / zc);
    for (int z : chunks(sh, nb / 2, nb * 2))
      if (const int e = try_one(sh, z)) return e;
  }
  if (cand.empty()) return 0;
  std::sort(cand.begin(), cand.end(), faster);
  // the four fastest again, round-robin over three rounds of about 2 ms, 8 to
  // 30 launches (a drift of the clocks during the search then favours none)
  const size_t top = std::min<size_t>(cand.size(), 4);
  const int reps = (int)std::min(30.f, std::max(8.f, 2.f / std::max(cand[0].ms, 1e-3f)));
  float sum[4] = {0.f, 0.f, 0.f, 0.f};
  for (int round = 0; round < 3; round++)
    for (size_t i = 0; i < top; i++) {
      float ms = 0.f;
      if (const int e = time(cand[i].shape, cand[i].zchunk, 1, reps, &ms)) return e;
      sum[i] += ms / 3.f;
    }
  const size_t best = std::min_element(sum, sum + top) - sum;
  *out = {cand[best].shape, cand[best].zchunk, sum[best]};
  return 0;
}

}  // namespace born

#endif
