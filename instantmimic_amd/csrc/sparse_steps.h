// Sparse plans on a wavefront per world: what its lanes do in a level, settled on the host (WaveSteps), and where a launch
// keeps it.  Host code without the runtime, checked on its own.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <vector>

#include "sparse_plan.h"

#ifdef __HIPCC__
#define IM_BOTH __host__ __device__
#else
#define IM_BOTH
#endif

namespace im {

constexpr int kStepTerms = 4;  // terms' operands read ahead of their products
// (the factor's steps read up to 3 * 64 words past an operand's last term, which they leave out)
constexpr int kStepSlack = (kStepTerms - 1) * 64;

// A plan's levels as the steps of a wavefront's 64 lanes (factor_steps, backward_steps).
struct WaveSteps {
  std::vector<uint32_t> words;  // the factor's, an empty one, the backward solve's, an empty one
  std::vector<uint16_t> pairs;
  int nfactor = 0, nbackward = 0;
};
inline WaveSteps wave_steps(const im_sparse_plan &pl) {
  WaveSteps out;
  std::vector<uint32_t> factor, backward;
  const auto &T = pl.table;
  for (int l = 0; l < pl.nlevels; ++l) {
    const int width = T[LT][l], teams = 64 / width;
    int log2 = 0;
    while ((1 << log2) < width) ++log2;
    for (int e0 = T[LP][l]; e0 < T[LP][l + 1]; e0 += teams) {
      int runs = 1;
      for (int e = e0; e < std::min(e0 + teams, T[LP][l + 1]); ++e) runs = std::max(runs, T[RP][e + 1] - T[RP][e]);
      for (int r = 0; r < runs; ++r) {
        int most = 0;  // terms of a lane
        for (int e = e0; e < std::min(e0 + teams, T[LP][l + 1]); ++e)
          if (r < T[RP][e + 1] - T[RP][e]) most = std::max(most, (int)(((uint32_t)T[RKL][T[RP][e] + r] >> 16) + width - 1) / width);
        for (int lane = 0; lane < 64; ++lane) {
          const int e = e0 + lane / width, tl = lane % width;
          uint32_t x = 0, y = (uint32_t)(most < 2) << 25 | (uint32_t)log2 << 26 | (uint32_t)(r == 0) << 29 | (uint32_t)(r == runs - 1) << 30 | (uint32_t)(most == 2) << 31;
          if (e < T[LP][l + 1]) {
            if (r < T[RP][e + 1] - T[RP][e]) {
              const uint32_t ab = (uint32_t)T[RAB][T[RP][e] + r], kl = (uint32_t)T[RKL][T[RP][e] + r];
              const int terms = ((int)(kl >> 16) - tl + width - 1) / width;
              if ((int)(kl >> 16) > tl) {
                x = ((ab & 0xFFFFu) + tl) | ((ab >> 16) + tl) << 12;
                y |= ((kl & 0xFFFFu) + tl) | (uint32_t)terms << 6;
              }
            }
            if (r == runs - 1 && tl == 0) {
              y |= (uint32_t)(T[ES][e] + 1) << 13;
              x |= (uint32_t)(T[EC][e] + 1) << 24;
            }
          }
          factor.push_back(x);
          factor.push_back(y);
        }
      }
    }
    for (int p0 = T[BL][l]; p0 < T[BL][l + 1]; p0 += 64)
      for (int lane = 0; lane < 64; ++lane) {
        const int p = p0 + lane;
        backward.push_back(p < T[BL][l + 1] ? (uint32_t)T[BS][p] | (uint32_t)T[BI][p] << 12 | (uint32_t)T[BJ][p] << 18 | 1u << 31 : 0u);
      }
  }
  out.nfactor = (int)(factor.size() / 128), out.nbackward = (int)(backward.size() / 64);
  factor.resize(factor.size() + 128, 0);
  backward.resize(backward.size() + 64, 0);
  out.words = std::move(factor);
  out.words.insert(out.words.end(), backward.begin(), backward.end());
  for (int c = 0; c < 64; ++c)
    for (int r = 0; r <= c; ++r) out.pairs.push_back((uint16_t)(r | c << 8));
  return out;
}

// ---- words of LDS ------------------------------------------------------------------------------

// What a plan asks of a launch: its own sizes, the words of its steps and of the tables that the update stage's worlds
// share (the forward solve's and the dofs' order behind them).
struct SparseSizes {
  int nv, nslots, step_words, shared_words;
};

// First factor, four worlds a workgroup: a world's factor and the list of its contributing rows.
IM_BOTH inline int init_world_words(int nslots, int n, int njmax) { return ((nslots + n + 3) & ~3) + 2 * ((njmax + 3) & ~3); }
// (behind the last world's factor lie at least the slack's words)
inline size_t init_lds_bytes(const SparseSizes &s, int njmax) {
  return 4 * (4 * (size_t)init_world_words(s.nslots, s.nv, njmax) + std::max(0, kStepSlack - 2 * ((njmax + 3) & ~3)));
}

IM_BOTH inline int update_world_words(int nslots, int n, int staged_rows) {
  const int factor = nslots + n + 2 * n + (staged_rows + 1) * n + staged_rows, reach = nslots + n + kStepSlack;
  return ((factor > reach ? factor : reach) + 3) & ~3;
}
// Update stage: worlds per workgroup, staged rows of a world, bytes (waves = 0: the wavefront kernel does not take the plan).
struct SparseUpdate {
  int waves = 0, staged_rows = 0;
  size_t lds = 0;
};
inline SparseUpdate sparse_update_layout(const SparseSizes &s, int nworld, int ncu) {
  constexpr size_t kCuLds = 160 * 1024;
  SparseUpdate u;
  // 32 staged rows where a CU still holds sixteen worlds with them, else 16
  u.staged_rows = 4 * (s.shared_words + 16 * (size_t)update_world_words(s.nslots, s.nv, 32)) <= kCuLds ? 32 : 16;
  const size_t per_world = (size_t)update_world_words(s.nslots, s.nv, u.staged_rows);
  auto bytes = [&](int waves) { return 4 * (s.shared_words + waves * per_world); };
  if (bytes(4) > 64 * 1024) return u;
  // Worlds per workgroup: every workgroup stages the tables for itself, so larger workgroups
  // leave more of a CU's 160 KB to the worlds.  The count that keeps the most worlds on a CU
  // (at most 32 wavefronts) is taken, the smallest on a tie and where four
  // per workgroup already hold the whole batch.
  int64_t best = 0;
  for (int cand = 4; cand <= 16; cand *= 2) {
    const int64_t held = std::min<int64_t>((int64_t)(kCuLds / bytes(cand)) * cand, 32);
    if (held > best && (cand == 4 || (int64_t)nworld > best * ncu)) best = held, u.waves = cand;
  }
  u.lds = bytes(u.waves);
  return u;
}

// Resident loop: the stage's area, which a tile of J and the gradient's lists also use, and what a world keeps beside it.
IM_BOTH inline int resident_area_words(int nslots, int n, int njmax, int staged_rows) {
  int words = update_world_words(nslots, n, staged_rows);
  const int tile = 64 * 17, grad = 2 * njmax + n;
  words = words > tile ? words : tile;
  words = words > grad ? words : grad;
  return (words + 3) & ~3;
}
struct SparseResident {
  int waves = 0, staged_rows = 0, step_words = 0;  // step_words: of the steps in LDS, all or none
  size_t lds = 0;
  int per_cu = 0;  // workgroups that a CU holds: by LDS, and sixteen wavefronts of up to 128 registers
};
// `waves` (nwaves): the worlds per workgroup that there are kernels for, most first; `table_words`: of the loop's shared row tables;
// `kept_words`: what a world keeps beside the area.
// The most worlds per workgroup (one workgroup per CU) that 158 KB of LDS admit, with 32 staged rows where they still
// fit (they cost a CU no world then; snu: 32 rows with eight worlds per CU instead of twelve was measured slower, 1344
// against 1283 us per loop), else 16.  The steps lie in LDS unless they cost a CU worlds and the batch does not fit the
// chip at once with them there.  Whole solves, us, steps in LDS / in memory: 16 worlds instead of 12 in memory: a forest of 54
// dofs (29 KB of steps), 96 rows x 4096 worlds 503 / 463, x 1000 376 / 378, one of 57 (34 KB) 522 / 496 and 393 / 394; as many worlds:
// 35 dofs (13 KB) x 8192 436 / 445, x 1000 296 / 302, a forest of 40 dofs (31 KB; 32 staged rows instead of 16 in memory) x 8192
// 468 / 483.
inline SparseResident sparse_resident_layout(const SparseSizes &s, int njmax, int table_words, size_t kept_words, const int *waves, int nwaves,
                                             int nworld, int ncu) {
  auto layout = [&](int step_words) {
    SparseResident r;
    const size_t shared = (size_t)step_words + s.shared_words + table_words;
    for (int i = 0; i < nwaves; ++i) {
      const int w = waves[i];
      auto bytes = [&](int rows) { return 4 * (shared + w * (resident_area_words(s.nslots, s.nv, njmax, rows) + kept_words)); };
      const int rows = bytes(32) <= 158 * 1024 ? 32 : 16;
      if (bytes(rows) > 158 * 1024) continue;
      r.waves = w, r.staged_rows = rows, r.step_words = step_words, r.lds = bytes(rows);
      r.per_cu = std::max(1, std::min((int)(160 * 1024 / r.lds), 16 / w));
      break;
    }
    return r;
  };
  const SparseResident near = layout(s.step_words), far = layout(0);
  if (near.waves == 0) return far;
  const int held = near.waves * near.per_cu;
  return far.waves * far.per_cu > held && (int64_t)nworld > (int64_t)held * ncu ? far : near;
}

}  // namespace im

#undef IM_BOTH
