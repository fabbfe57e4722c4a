// Checks the threshold rounds' decision of picks on the host: the rounds are restated on one
// list of points, with the bounds and steps that the kernels take (fps_rounds_bound.hpp), and
// compared with the loop that takes one pick per pass.  Clouds of one to 125 points, where a
// round can hold every point: wide scales, duplicates, lattices, special values, both tie
// rules, whole runs and runs in parts.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <limits>
#include <random>
#include <vector>

#include "fps_rounds_bound.hpp"

using fpsx::make_key;

struct Cloud {
  uint32_t n, dim;
  std::vector<float> x;  // row-major
};

static float sqdist(const Cloud &c, uint32_t a, uint32_t b) {
  float d = 0.0f;
  for (uint32_t j = 0; j < c.dim; ++j) {
    const float t = c.x[a * c.dim + j] - c.x[b * c.dim + j];
    d = d + t * t;
  }
  return d;
}

static int bits_of(float v) {
  int b;
  std::memcpy(&b, &v, 4);
  return b;
}

static uint64_t key_of(float v, uint32_t i, bool lowest) {
  return make_key(bits_of(v), lowest ? ~i : i);
}

// One pick per pass.
static std::vector<uint32_t> plain(const Cloud &c, uint32_t m, uint32_t start, bool lowest,
                                   float init) {
  std::vector<float> dm(c.n, init);
  std::vector<uint32_t> out(1, start);
  while (out.size() < m) {
    uint64_t best = 0;
    uint32_t at = 0;
    for (uint32_t i = 0; i < c.n; ++i) {
      const float d = sqdist(c, i, out.back());
      if (d < dm[i]) dm[i] = d;
      const uint64_t k = key_of(dm[i], i, lowest);
      if (k > best) {
        best = k;
        at = i;
      }
    }
    out.push_back(at);
  }
  return out;
}

// In rounds: at most `cap` candidates are decided on, rounds of more than `list` are lost; in
// parts of `part` picks.
static std::vector<uint32_t> rounds(const Cloud &c, uint32_t m, uint32_t start, bool lowest,
                                    float init, uint32_t cap, uint32_t list, uint32_t target,
                                    uint32_t part) {
  std::vector<float> dm(c.n, init);
  std::vector<uint32_t> out(1, start), np(1, start);
  uint64_t T = ~0ull, Tg = ~0ull, step = (uint64_t)1 << 51;
  uint32_t end = std::min(m, 1 + part);
  bool stuck = false;
  uint64_t last = ~0ull;
  bool empty = false;
  for (;;) {
    if (out.size() >= m) return out;
    const bool cut = out.size() >= end;
    if (stuck && !cut) {
      while (out.size() < end) out.push_back(out.back());
      if (out.size() >= m) return out;
    }
    // update
    for (uint32_t p : np)
      for (uint32_t i = 0; i < c.n; ++i) {
        const float d = sqdist(c, i, p);
        if (d < dm[i]) dm[i] = d;
      }
    np.clear();
    if (cut || stuck) {  // the next part takes the run up again
      T = cut ? last : ~0ull;
      Tg = fpsx::round_bound(T, step);
      end = std::min<uint64_t>(m, out.size() + part);
      stuck = false;
    }
    std::vector<std::pair<uint64_t, uint32_t>> ck;
    uint64_t U = 0;
    for (uint32_t i = 0; i < c.n; ++i) {
      const uint64_t k = key_of(dm[i], i, lowest);
      U = std::max(U, k);
      if (k > Tg) ck.push_back({k, i});
    }
    const uint32_t C = (uint32_t)ck.size();
    if (C == 0 || C > list) {
      // the best point alone
      const uint32_t i = lowest ? ~(uint32_t)U : (uint32_t)U;
      stuck = !(sqdist(c, i, i) < dm[i]);
      out.push_back(i);
      np.push_back(i);
      last = U;
      if (C)
        step = fpsx::less_step(step, target, C);
      else if (empty)
        step = fpsx::next_step(step, target, 1);
      empty = C == 0;
      T = U;
      Tg = fpsx::round_bound(T, step);
      continue;
    }
    empty = false;
    std::sort(ck.rbegin(), ck.rend());
    const uint32_t F = std::min(C, cap);
    uint64_t te = C > cap ? ck[cap].first : 0;
    uint32_t stop = ~0u;
    std::vector<std::pair<uint64_t, uint32_t>> acc;
    for (uint32_t i = 0; i < F; ++i) {
      const float v = dm[ck[i].second];
      bool taken = true;
      for (auto &p : acc) {
        const float d = sqdist(c, ck[i].second, p.second);
        if (d < v) {
          te = std::max(te, make_key(bits_of(d), (uint32_t)ck[i].first));
          taken = false;
          break;
        }
      }
      if (!taken) continue;
      if (!(sqdist(c, ck[i].second, ck[i].second) < v)) stop = std::min(stop, (uint32_t)acc.size());
      acc.push_back(ck[i]);
    }
    T = std::max(te, Tg);
    uint32_t keep = 0;
    while (keep < acc.size() && keep <= stop && acc[keep].first > T) ++keep;
    stuck = stop < keep;
    keep = std::min<uint32_t>(keep, end - (uint32_t)out.size());
    for (uint32_t i = 0; i < keep; ++i) {
      out.push_back(acc[i].second);
      np.push_back(acc[i].second);
      last = acc[i].first;
    }
    step = fpsx::next_step(step, target, C);
    Tg = fpsx::round_bound(T, step);
  }
}

static int bad = 0;

static void check(const Cloud &c, uint32_t m, uint32_t start, const char *name) {
  const struct {
    uint32_t cap, list, target, part;
  } forms[] = {{256, 256, 64, ~0u >> 1}, {256, 512, 160, ~0u >> 1}, {256, 256, 64, 5},
               {128, 128, 64, ~0u >> 1}, {16, 32, 8, ~0u >> 1},     {16, 16, 8, 3}};
  for (int lowest = 0; lowest < 2; ++lowest) {
    const float init = lowest ? std::numeric_limits<float>::max()
                              : std::numeric_limits<float>::infinity();
    const std::vector<uint32_t> want = plain(c, m, start, lowest != 0, init);
    for (auto &f : forms)
      if (rounds(c, m, start, lowest != 0, init, f.cap, f.list, f.target, f.part) != want) {
        if (bad++ < 5)
          std::printf("FAIL %s n=%u dim=%u m=%u start=%u lowest=%d cap=%u list=%u part=%u\n", name,
                      c.n, c.dim, m, start, lowest, f.cap, f.list, f.part);
      }
  }
}

int main() {
  std::mt19937 rng(5);
  auto uni = [&](double a, double b) { return std::uniform_real_distribution<double>(a, b)(rng); };
  {
    // Duplicates of the start and points ever nearer to it.
    Cloud c{80, 3, std::vector<float>(240, 0.0f)};
    for (int k = 0; k < 40; ++k) c.x[(40 + k) * 3] = std::ldexp(1.0f, -k);
    check(c, 60, 0, "ladder");
    check({3, 3, {0, 0, 0, 0, 0, 0, 1e-20f, 0, 0}}, 3, 0, "three");
  }
  for (int t = 0; t < 1500; ++t) {
    Cloud c;
    c.n = 1 + rng() % 125;
    c.dim = 1 + rng() % 4;
    c.x.resize((size_t)c.n * c.dim);
    const int kind = t % 4;
    for (uint32_t i = 0; i < c.n; ++i) {
      const double scale = kind == 0 ? std::pow(10.0, uni(-12, 0)) : 1.0;
      for (uint32_t j = 0; j < c.dim; ++j)
        c.x[i * c.dim + j] = kind == 1 ? (float)(rng() % 4) : (float)(scale * uni(-1, 1));
      if (kind == 3 && rng() % 9 == 0)
        c.x[i * c.dim + rng() % c.dim] = rng() % 2 ? NAN : (rng() % 2 ? INFINITY : 3e19f);
    }
    for (uint32_t q = rng() % 30; q > 0; --q) {  // copies
      const uint32_t a = rng() % c.n, b = rng() % c.n;
      for (uint32_t j = 0; j < c.dim; ++j) c.x[a * c.dim + j] = c.x[b * c.dim + j];
    }
    check(c, c.n, rng() % c.n, "random");
  }
  if (bad) {
    std::printf("%d runs differ\n", bad);
    return 1;
  }
  std::printf("OK\n");
  return 0;
}
