// The tile width of a launch, and the sizes of the launches it makes.
#include "fa_launch.h"

#include <math.h>

#include <type_traits>

#include "fa_device.h"

namespace fa {
namespace {

constexpr int kFwdRows = 64;   // query rows of the forward's smallest tile
// Lanes per row of the backward's preprocess at a width (256 threads per workgroup).
constexpr int pre_lanes(int width) { return width <= 64 ? 8 : width <= 128 ? 16 : 32; }

template <class Args, class Launch>
hipError_t by_width(const Args& a, bool bf, const Launch& launch) {
  auto at = [&](auto w) {
    return bf ? launch(w, std::true_type{}, a) : launch(w, std::false_type{}, a);
  };
  switch (padded_head_dim(a.D)) {
    case 32: return at(std::integral_constant<int, 32>{});
    case 64: return at(std::integral_constant<int, 64>{});
    case 96: return at(std::integral_constant<int, 96>{});
    case 128: return at(std::integral_constant<int, 128>{});
    default: return at(std::integral_constant<int, 256>{});
  }
}

}  // namespace

// The plan with the least estimated time. Units: one product of a 128 x 128
// score block with 128 columns on one CU (0.53 us); phase 1 takes four per
// block, phase 2 three. With one item per tile (both phases, balanced under
// causal masking by the split in bwd_kernel) the items are equal and long: 384
// of them on 256 CUs (B=2 H=32/8 N=3001 D=128 dense) need two full rounds, and
// fewer than 256 leave CUs idle. Phases apart, the hardware fills the CUs with
// the short phase-2 items as the long phase-1 ones end; under causal masking
// the longest phase-1 item then bounds a grid of one round (B=1 H=8 N=4096
// D=128: 136 us against 132 together). Parts cut that item, which with few kv
// heads or rows is most of the time, for the price of writing and summing the
// partials. The constants were fitted to 7638 timed plans of 1183 random shapes
// (64 <= D <= 256, 100 <= N <= 8192, B <= 16, 1 to 64 heads): the plan taken is
// 1.4% slower than the best one on average, one item per tile 46% slower.
// Backward, same box, together -> apart: 1042 -> 948 us (the ragged dense shape
// above); 180 -> 131 at B=2 H=8 N=2663 D=128 causal; with parts 737 -> 113 (8
// parts) at B=1 H=16/1 N=2048 D=128 causal, 512 -> 396 (4) at B=1 H=32/4 N=4608
// D=64 causal, 321 -> 146 (4) at B=3 H=16/4 N=896 D=256 causal.
namespace {

constexpr int kPartsTried[] = {1, 2, 3, 4, 6, 8, 12, 16, 24};

struct BwdCost {
  int W, G;
  double nk, nq, n1, n2, total;  // tiles of a head, items of the phases, all units
  bool causal;

  BwdCost(int B, int Hq, int Hkv, int N, int NK, int D, bool causal) : causal(causal) {
    W = padded_head_dim(D);
    G = Hq / Hkv;
    nk = (NK + kBwdTile - 1) / kBwdTile;
    nq = (N + kBwdTile - 1) / kBwdTile;
    n1 = (double)B * Hkv * nk;
    n2 = (double)B * Hq * nq;
    const double half = 0.5 * nq * (nq + 1);  // causal, the last rows aligned
    const double blocks = !causal ? nk * nq : nk >= nq ? nq * (nk - nq) + half : 0.5 * nk * (nk + 1);
    total = 7.0 * B * Hq * blocks;
  }
  // Units of a block's product and of an item's start and end, at this width;
  // w4: for each of two workgroups per CU.
  double unit(bool w4) const {
    return w4 ? 0.71 : W <= 64 ? 0.46 : W <= 96 ? 0.88 : W <= 128 ? 1.0 : 8.5;
  }
  double fixed(bool w4) const {
    return w4 || W <= 64 ? 10.0 : W <= 96 ? 13.0 : W <= 128 ? 16.0 : 9.0;
  }
  static constexpr double kSolo = 0.8;  // a workgroup alone on its CU, of unit(true)

  double together(bool w4) const {
    const double n = nk > nq ? n1 : n1 * nq / nk;
    // (width 256 and unequal sides run without the causal split)
    const double item =
        unit(w4) * (causal && (W > 128 || nk != nq) ? G * (4.0 * nq + 3.0) : total / n);
    const double ends = fixed(w4) * (1.0 + 0.46 * G);
    if (!w4) return ceil(n / kCUs) * (item + ends);
    const double full = floor(n / (2 * kCUs)), rest = n - full * 2 * kCUs;
    const double last = rest <= 0 ? 0.0 : item * (rest > kCUs ? 1.0 : kSolo) + ends;
    return full * (item + ends) + last;
  }
  double apart(int parts, bool w4) const {
    const double items = n1 * parts + n2, u = unit(w4), slots = w4 ? 2 * kCUs : kCUs;
    const double ends = 0.77 * fixed(w4), work = total * u + items * ends;
    const bool few = w4 && items < slots;
    double t = fmax(work / slots, 4.0 * G * nq * u / parts * (few ? kSolo : 1.0) + ends);
    if (few) t = fmax(t, work / kCUs * kSolo);
    if (items > slots) t += 0.36 * 3.0 * (causal ? 0.5 * nk : nk) * u;  // the uneven end
    if (parts > 1) t += 1.0 + 0.17 * n1 * parts * (W / 128.0);
    return 1.03 * t;  // (one item per tile where the two are about equal)
  }
  bool allows(int parts, int N) const {
    return parts == 1 || (n1 < 500 && n1 * parts < 1200 && (double)G * N >= 128.0 * parts);
  }
};

}  // namespace

BwdPlan bwd_plan(int B, int Hq, int Hkv, int N, int NK, int D, bool causal, bool has_w4,
                 bool slots) {
  const BwdCost cost(B, Hq, Hkv, N, NK, D, causal);
  BwdPlan best{false, 1, false};
  double least = HUGE_VAL;
  auto consider = [&](BwdPlan p, double t) {
    if (t < least) {
      least = t;
      best = p;
    }
  };
  // (a launch counts its work-items in 32 bits: one item per tile always fits)
  const double threads = cost.W > 128 ? 256.0 : 512.0;
  auto search = [&](bool w4, bool may_share) {
    consider({false, 1, w4}, cost.together(w4));
    for (const int parts : kPartsTried) {
      if (parts > 1 && (!may_share || NK != N)) break;
      if (!cost.allows(parts, N) || (cost.n1 * parts + cost.n2 + 16) * threads > 4294967295.0) break;
      consider({true, parts, w4}, cost.apart(parts, w4));
    }
  };
  search(false, true);
  if (has_w4) search(true, true);
  if (!slots && best.parts > 1) {  // (the same workgroups, so that dQ is the same)
    least = HUGE_VAL;
    search(best.w4, false);
  }
  return best;
}

int bwd_max_parts(int B, int Hq, int Hkv, int N, int D) {
  int most = 1;
  for (const bool causal : {false, true})
    for (const bool w4 : {false, true}) {
      if (w4 && padded_head_dim(D) != 64) continue;
      const BwdPlan p = bwd_plan(B, Hq, Hkv, N, N, D, causal, w4, true);
      if (p.parts > most) most = p.parts;
    }
  return most;
}

// Estimated microseconds, fitted to 20 shapes (1 to 512 query rows, 1000 to
// 32768 keys): a workgroup of fa_dec.hip takes 1.2 us for a round of its waves
// (256 keys; 128 at width 256) while it waits for memory and 1.5 where every CU
// has one, 2 us to start and end; the keys and values come at 5.4 TB/s; parts
// cost a second launch (2 us on the GPU, 3 on the host, which small calls wait
// for) and 0.019 us for each partial O (width 128) to write and
// combine. A step (128 keys) of fa_fwd.hip takes 1 us.
// Same box, fa_fwd.hip -> here: 220 -> 99 us at B=16 H=32/8 N=1 against 8192
// keys, D=128 (2 parts); 238 -> 29 at B=1 H=32/8 N=1, 32768 keys, D=128 (16
// parts); 225 -> 18 at B=1 H=16/2 N=4, 8000 keys, D=256 (16 parts); 55 -> 23 at
// B=32 H=32/8 N=1, 1000 keys, D=128 (1 part); 68 -> 23 at B=1 H=32/8 N=128, 4096
// keys, D=128 (2 parts); 71 -> 76 at B=4 H=32/4 N=321, 1506 keys, D=128, which
// stays there. Only with more keys than query rows: the square shapes' results
// do not change.
DecPlan dec_plan(const FwdArgs& a) {
  constexpr int kTried[] = {1, 2, 3, 4, 6, 8, 12, 16, 24, 32, 48, 64};
  const DecPlan none{0, 0, 1};
  const int NK = key_rows(a.N, a.Nkv), W = padded_head_dim(a.D);
  if (NK <= a.N || a.mask || a.drop || a.bias || a.block_rows || a.seg_start) return none;
  const double tiles = ceil((double)(a.Hq / a.Hkv) * a.N / 32), items = tiles * a.B * a.Hkv;
  if (items * 512 > 4294967295.0 || items * (W / 32) * 256 > 4294967295.0) return none;
  const int wave_keys = W > 128 ? 128 : 256;
  const double seen = a.window > 0 ? fmin(NK, (double)a.window + a.N) : NK;
  const double read = 4.0 * a.B * a.Hkv * seen * a.D / 5.4e6;
  double least = HUGE_VAL;
  int best = 1;
  for (const int parts : kTried) {
    if (parts > 1 && (seen < parts * 128.0 || items * parts > 4096)) break;
    const double rounds = ceil(items * parts / kCUs);
    const double each = ceil(seen / parts / wave_keys) * (items * parts >= kCUs ? 1.5 : 1.2) + 2.0;
    const double t = fmax(rounds * each, read) + (parts > 1 ? 5.0 + 0.019 * items * parts * W / 128 : 0.0);
    if (t < least) {
      least = t;
      best = parts;
    }
  }
  const double q_tiles = (a.N + 63) / 64, per_wg = a.causal && q_tiles > 1 ? 2 : 1;
  const double wgs = ceil(q_tiles / per_wg) * a.B * a.Hq;
  const double there = ceil(wgs / kCUs) * per_wg * (seen / (W > 128 ? 64 : 128) + 2.0);
  return least < there ? DecPlan{(int)tiles, (int)items, best} : none;
}

hipError_t launch_fwd(const FwdArgs& a, void* workspace) {
  DecPlan plan = dec_plan(a);
  if (plan.items > 0) {
    if (!workspace) plan.parts = 1;
    return by_width(a, a.dtype == kBF16, [&](auto w, auto bf, const FwdArgs& a) {
      return launch_dec_w<decltype(w)::value, decltype(bf)::value>(a, plan, workspace);
    });
  }
  return by_width(a, a.dtype == kBF16, [](auto w, auto bf, const FwdArgs& a) {
    return launch_fwd_w<decltype(w)::value, decltype(bf)::value>(a);
  });
}

hipError_t launch_bwd_preprocess(const BwdArgs& a) {
  return by_width(a, a.dtype == kBF16, [](auto w, auto bf, const BwdArgs& a) {
    return launch_bwd_pre_w<decltype(w)::value, decltype(bf)::value>(a);
  });
}

hipError_t launch_bwd_main(const BwdArgs& a) {
  return by_width(a, a.dtype == kBF16, [](auto w, auto bf, const BwdArgs& a) {
    return launch_bwd_main_w<decltype(w)::value, decltype(bf)::value>(a);
  });
}

unsigned long long fwd_launch_items(int B, int Hq, int N, int D) {
  const unsigned long long tiles = ((unsigned long long)N + kFwdRows - 1) / kFwdRows;
  const unsigned long long wgs = tiles * (unsigned long long)B * (unsigned long long)Hq;
  return (wgs + kXcds - 1) / kXcds * kXcds * (padded_head_dim(D) > 128 ? 256 : 512);
}

unsigned long long bwd_launch_items(int B, int Hq, int Hkv, int N, int D, int Nkv) {
  const unsigned long long rows = (unsigned long long)B * Hq * N;
  const unsigned long long rows_per_block = 256 / pre_lanes(padded_head_dim(D));
  const unsigned long long pre = (rows + rows_per_block - 1) / rows_per_block * 256;
  const unsigned long long NK = (unsigned long long)key_rows(N, Nkv);
  const unsigned long long kt = (NK + kBwdTile - 1) / kBwdTile;
  const unsigned long long qt = ((unsigned long long)N + kBwdTile - 1) / kBwdTile;
  const unsigned long long wgs = (kt > qt ? kt : qt) * (unsigned long long)B * Hkv;
  const unsigned long long threads = padded_head_dim(D) > 128 ? 256 : 512;
  const unsigned long long main = (wgs + kXcds - 1) / kXcds * kXcds * threads;
  return pre > main ? pre : main;
}

}  // namespace fa
