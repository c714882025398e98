// Forward-path work plan (host only): the degree-skew bins of the forward
// counting kernels (k_forward.hip) and the planner that fills them.  Plain
// C++ with no HIP dependency, so that the CPU tests compile the same planner
// (tests/test_pack_plan.py) and check its bounds against an emulation of the
// wave-pack kernel's index arithmetic.
#pragma once

#include <algorithm>
#include <cstdint>
#include <thread>
#include <utility>
#include <vector>

namespace accfwd {
constexpr int kWG = 512;                              // threads per workgroup (8 waves)
constexpr int kWaves = kWG / 64;
constexpr int kTableBits = 12;                        // workgroup LDS hash table of 4096 keys
constexpr uint32_t kLdsCap = 1u << (kTableBits - 1);  // |N<(b)| up to 2048 stays in LDS
constexpr uint32_t kChunk = 512;                      // upper slots per workgroup unit
constexpr uint32_t kBitmapIds = 32u << kTableBits;    // b - min N(b) <= 2^17: N<(b) as an LDS bitmap of [min N(b), b)
constexpr uint32_t kBitmapMaxLow = 65535;             // word prefixes are 16-bit
constexpr int kWaveTableBits = 9;                     // wave-private table of 512 keys
constexpr uint32_t kWaveCap = 1u << (kWaveTableBits - 1);  // |N<(b)| up to 256 in a wave unit
constexpr uint32_t kWaveSlots = 64;                   // upper slots of a wave unit
constexpr int kBigWG = 256;
}  // namespace accfwd

// One forward-path work unit: source b, its upper slots [j0, j1), nlow = |N<(b)|.
struct FwdUnit {
  int32_t b;
  uint32_t j0;
  uint32_t j1;
  uint32_t nlow;
};

// Forward plan, binned by degree skew: a source b with upper slots (neighbors
// > b) is a small source when it has at most wave_slots upper slots and
// |N<(b)| <= wave_low; runs of consecutive small sources form wave packs
// (FwdUnit {b0, b1, upper slots, lower entries}: at most 64 sources, 64
// upper slots, 256 lower entries and 512 hash-table entries, each source's
// table being the smallest power of two >= 2 |N<(b)|, at least 16).  Other
// sources become workgroup units of at most `chunk` upper slots (N<(b) as an
// LDS bitmap when b - lo[b] <= kBitmapIds, else an LDS hash table); sources
// whose N<(b) fits neither go to the global-memory variant.  hs[b] is the
// first upper slot of b, lo[b] its smallest neighbor.
inline void build_forward_range(uint32_t b_lo, uint32_t b_hi, const uint32_t *off, const uint32_t *hs,
                                const int32_t *lo, uint32_t wave_slots, uint32_t wave_low, uint32_t chunk,
                                uint32_t max_sources, std::vector<FwdUnit> &wave, std::vector<FwdUnit> &block,
                                std::vector<FwdUnit> &big) {
  auto table = [](uint32_t nl) -> uint32_t {
    if (!nl) return 0;
    uint32_t t = 16;
    while (t < 2 * nl) t *= 2;
    return t;
  };
  FwdUnit pack{0, 0, 0, 0};
  uint32_t pack_tbl = 0, pack_sources = 0;
  bool open = false;
  auto close = [&]() {
    if (open) wave.push_back(pack);
    open = false;
  };
  for (uint32_t b = b_lo; b < b_hi; b++) {
    const uint32_t nl = hs[b] - off[b];
    const uint32_t nup = off[b + 1] - hs[b];
    if (nup == 0) continue;
    if (nup <= wave_slots && nl <= wave_low) {
      const uint32_t t = table(nl);
      if (open && (b + 1 - static_cast<uint32_t>(pack.b) > 64 || pack_sources == max_sources || pack.j1 + nup > 64 ||
                   pack.nlow + nl > accfwd::kWaveCap || pack_tbl + t > (1u << accfwd::kWaveTableBits)))
        close();
      if (!open) {
        pack = FwdUnit{static_cast<int32_t>(b), b + 1, 0, 0};
        pack_tbl = 0;
        pack_sources = 0;
        open = true;
      }
      pack_sources++;
      pack.j0 = b + 1;
      pack.j1 += nup;
      pack.nlow += nl;
      pack_tbl += t;
      continue;
    }
    close();
    for (uint32_t j0 = hs[b]; j0 < off[b + 1]; j0 += chunk) {
      FwdUnit u{static_cast<int32_t>(b), j0, std::min(j0 + chunk, off[b + 1]), nl};
      const uint32_t span = b - static_cast<uint32_t>(lo[b]);
      const bool lds = nl <= accfwd::kLdsCap || (span <= accfwd::kBitmapIds && nl <= accfwd::kBitmapMaxLow);
      (lds ? block : big).push_back(u);
    }
  }
  close();
}

// Runs fn(0) .. fn(pieces - 1), on host threads of their own where there are threads to spare.
template <class F>
inline void run_pieces(uint32_t pieces, F &&fn) {
  std::vector<std::thread> th;
  uint32_t t = 1;
  try {
    for (; t < pieces; t++) th.emplace_back(fn, t);
  } catch (...) {  // no thread to spare: the rest run here
  }
  fn(0);
  for (uint32_t r = t; r < pieces; r++) fn(r);
  for (auto &x : th) x.join();
}

// Builds the plan of the sources in `ranges` (ascending, disjoint) in
// kPlanThreads contiguous pieces on as many host threads (packs cross neither
// a range nor a piece boundary) and joins the pieces' lists in order.
// Sources per pack: just enough packs to give every wave slot of the device
// one (a small graph keeps one source per wave), at most 64.
constexpr uint32_t kPlanThreads = 8;
using SourceRange = std::pair<uint32_t, uint32_t>;
inline void build_forward_plan(const std::vector<SourceRange> &ranges, const uint32_t *off, const uint32_t *hs,
                               const int32_t *lo, uint32_t wave_slots, uint32_t wave_low, uint32_t chunk,
                               uint32_t wave_slots_on_device, std::vector<FwdUnit> &wave, std::vector<FwdUnit> &block,
                               std::vector<FwdUnit> &big) {
  uint64_t span = 0;
  for (const SourceRange &r : ranges) span += r.second - r.first;
  const uint32_t pieces = span < (1u << 16) ? 1 : kPlanThreads;
  std::vector<uint64_t> small(pieces, 0);
  std::vector<std::vector<FwdUnit>> w(pieces), bl(pieces), bg(pieces);
  // the parts of the ranges holding the span's sources [span t / pieces, span (t + 1) / pieces)
  auto each = [&](uint32_t t, auto &&fn) {
    const uint64_t s0 = span * t / pieces, s1 = span * (t + 1) / pieces;
    uint64_t at = 0;
    for (const SourceRange &r : ranges) {
      const uint64_t len = r.second - r.first;
      const uint64_t a = std::max(s0, at), e = std::min(s1, at + len);
      if (a < e) fn(r.first + static_cast<uint32_t>(a - at), r.first + static_cast<uint32_t>(e - at));
      at += len;
    }
  };
  run_pieces(pieces, [&](uint32_t t) {
    uint64_t c = 0;
    each(t, [&](uint32_t a, uint32_t e) {
      for (uint32_t b = a; b < e; b++) {
        const uint32_t nl = hs[b] - off[b], nup = off[b + 1] - hs[b];
        c += nup && nup <= wave_slots && nl <= wave_low;
      }
    });
    small[t] = c;
  });
  uint64_t n_small = 0;
  for (uint64_t c : small) n_small += c;
  const uint64_t per = (n_small + wave_slots_on_device - 1) / std::max<uint32_t>(wave_slots_on_device, 1);
  const uint32_t max_sources = static_cast<uint32_t>(std::min<uint64_t>(64, std::max<uint64_t>(1, per)));
  run_pieces(pieces, [&](uint32_t t) {
    each(t, [&](uint32_t a, uint32_t e) {
      build_forward_range(a, e, off, hs, lo, wave_slots, wave_low, chunk, max_sources, w[t], bl[t], bg[t]);
    });
  });
  for (uint32_t t = 0; t < pieces; t++) {
    wave.insert(wave.end(), w[t].begin(), w[t].end());
    block.insert(block.end(), bl[t].begin(), bl[t].end());
    big.insert(big.end(), bg[t].begin(), bg[t].end());
  }
}

// The plan of the sources [b_lo, b_hi).
inline void build_forward_plan(uint32_t b_lo, uint32_t b_hi, const uint32_t *off, const uint32_t *hs,
                               const int32_t *lo, uint32_t wave_slots, uint32_t wave_low, uint32_t chunk,
                               uint32_t wave_slots_on_device, std::vector<FwdUnit> &wave, std::vector<FwdUnit> &block,
                               std::vector<FwdUnit> &big) {
  build_forward_plan(std::vector<SourceRange>{{b_lo, b_hi}}, off, hs, lo, wave_slots, wave_low, chunk,
                     wave_slots_on_device, wave, block, big);
}

// Dense sources (k_dense.hip): the first sources of a graph whose vertices
// are [v0, v1), as many as keep many upper slots.  Blocks of kDenseBlock
// sources are taken while a block's sources have at least kDenseUpper upper
// slots on average; ids relative to v0 stay below kDenseIds (16-bit lists
// with one padding value).  Returns the number of dense sources and adds
// their upper slots to *upper.  The pass's time hardly depends on where the
// sources stop (24 to 96 upper slots on average: within 2% at R-MAT scale 20
// and 17); with fewer than kDenseMin upper slots of dense sources in all the
// two more launches cost what they save (per-slot pass, Chung-Lu, average
// degree 32: 99 against 101 us at 32,000 vertices, 152 against 124 us at
// 64,000).
constexpr uint32_t kDenseIds = 65535;
constexpr uint32_t kDenseBlock = 64;
constexpr uint32_t kDenseUpper = 48;
constexpr uint64_t kDenseMin = 1ull << 18;
inline uint32_t dense_sources(uint32_t v0, uint32_t v1, const uint32_t *off, const uint32_t *hs, uint64_t *upper) {
  const uint32_t most = std::min(v1 - v0, kDenseIds);
  uint32_t d = 0;
  while (d < most) {
    const uint32_t k = std::min(kDenseBlock, most - d);
    uint64_t up = 0;
    for (uint32_t b = v0 + d; b < v0 + d + k; b++) up += off[b + 1] - hs[b];
    if (up < static_cast<uint64_t>(kDenseUpper) * k) break;
    d += k;
    *upper += up;
  }
  return d;
}
