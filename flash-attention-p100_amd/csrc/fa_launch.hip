// The tile width of a launch, and the sizes of the launches it makes.
#include "fa_launch.h"

#include <limits.h>
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
// partials. The constants were fitted to 7638 timed plans of 1183 random square
// shapes (64 <= D <= 256, 100 <= N <= 8192, B <= 16, 1 to 64 heads) without a
// window: the plan taken is 1.4% slower than the best one on average, one item per
// tile 46% slower. Over 1400 random calls each, the plan taken is 1.3% slower than
// the best with a window and 0.6% with unequal sides (3.9% and 2.3% before they
// were priced); 2% of the calls are more than 5% slower than one item per tile.
// Key lengths and packed sequences are on the device, so the plan does not see
// them (1.7% and 3.6%); a mask's, dropout's and a bias's cost is not in it either
// (a bias: 2.9%). Backward, same box, one item per tile -> the plan's: 1102 -> 974
// us (the ragged dense shape above, apart); 162 -> 126 at B=2 H=8 N=2663 D=128
// causal (apart); 720 -> 110 at B=1 H=16/1 N=2048 D=128 causal (16 parts), 529 ->
// 403 at B=1 H=32/4 N=4608 D=64 causal (4), 312 -> 154 at B=3 H=16/4 N=896 D=256
// causal (3); 32 -> 22 at B=3 H=1 N=3801 D=128, window 107 (39 with the 3 parts
// that the whole triangle would get); 184 -> 144 at B=5 H=4/2 N=3581, 807 keys,
// D=64 (290 on two workgroups per CU).
namespace {

constexpr int kPartsTried[] = {1, 2, 3, 4, 6, 8, 12, 16, 24};

struct BwdCost {
  int W, G;
  double nk, nq, n1, n2, total;  // tiles of a head, items of the phases, all units
  double q_reach, k_reach;       // most query tiles a key tile is seen by, key tiles one sees
  bool causal, window;

  BwdCost(int B, int Hq, int Hkv, int N, int NK, int D, bool causal, int window)
      : causal(causal), window(window > 0) {
    W = padded_head_dim(D);
    G = Hq / Hkv;
    nk = (NK + kBwdTile - 1) / kBwdTile;
    nq = (N + kBwdTile - 1) / kBwdTile;
    n1 = (double)B * Hkv * nk;
    n2 = (double)B * Hq * nq;
    const double half = 0.5 * nq * (nq + 1);  // causal, the last rows aligned
    double blocks = !causal ? nk * nq : nk >= nq ? nq * (nk - nq) + half : 0.5 * nk * (nk + 1);
    q_reach = causal ? fmin(nq, nk) : nq;
    k_reach = nk;
    if (window > 0) {  // (in streamed tiles of 64 rows, half a tile each)
      const double reach = (ceil((window - 1) / 64.0) + 2) / 2;
      q_reach = fmin(q_reach, reach);
      k_reach = fmin(k_reach, reach);
      // Query tiles see lo .. nk key tiles, at most `reach` of them.
      const double lo = fmax(1.0, nk - nq + 1), below = fmax(lo - 1, floor(fmin(reach, nk)));
      blocks = 0.5 * (lo + below) * (below - lo + 1) + (nk - below) * reach;
    }
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
    const double n = nk > nq ? n1 : n1 * nq / nk, slots = w4 ? 2 * kCUs : kCUs;
    const double ends = fixed(w4) * (1.0 + 0.46 * G);
    if (nk != nq) {  // workgroups with both phases beside workgroups with one
      const double item = G * (4.0 * q_reach + 3.0 * k_reach) * unit(w4);
      return fmax(total * unit(w4) / fmin(slots, n), item * (w4 && n <= kCUs ? kSolo : 1.0)) +
             ends * ceil(n / slots) + (n > slots ? 0.5 * item : 0.0);
    }
    // (width 256 and windows run without the causal split)
    const double item =
        unit(w4) * (window ? G * (4.0 * q_reach + 3.0 * fmin(fmax(nk - q_reach + 1, 1.0), k_reach))
                    : causal && W > 128 ? G * (4.0 * nq + 3.0)
                                        : total / n);
    if (!w4) return ceil(n / kCUs) * (item + ends);
    const double full = floor(n / slots), rest = n - full * slots;
    const double last = rest <= 0 ? 0.0 : item * (rest > kCUs ? 1.0 : kSolo) + ends;
    return full * (item + ends) + last;
  }
  double apart(int parts, bool w4) const {
    const double items = n1 * parts + n2, u = unit(w4), slots = w4 ? 2 * kCUs : kCUs;
    const double ends = 0.77 * fixed(w4), work = total * u + items * ends;
    const bool few = w4 && items < slots;
    double t = fmax(work / slots, 4.0 * G * q_reach * u / parts * (few ? kSolo : 1.0) + ends);
    if (few) t = fmax(t, work / kCUs * kSolo);
    if (items > slots)  // the uneven end
      t += 0.36 * 3.0 * (window ? k_reach : causal ? 0.5 * nk : nk) * u;
    if (parts > 1) t += 1.0 + 0.17 * n1 * parts * (W / 128.0);
    return 1.03 * t;  // (one item per tile where the two are about equal)
  }
  bool allows(int parts, int N) const {
    return parts == 1 || (n1 < 500 && n1 * parts < 1200 && (double)G * N >= 128.0 * parts);
  }
};

}  // namespace

BwdPlan bwd_plan(int B, int Hq, int Hkv, int N, int NK, int D, bool causal, int window,
                 bool has_w4, BwdShare share) {
  const BwdCost cost(B, Hq, Hkv, N, NK, D, causal, window);
  // One item per tile, two workgroups per CU where the grid fills both.
  const BwdPlan plain{false, 1,
                      has_w4 && fmax(cost.nk, cost.nq) * (double)B * Hkv >= 2.0 * kCUs};
  BwdPlan best{false, 1, false};
  double least = HUGE_VAL;
  auto consider = [&](BwdPlan p, double t) {
    if (t < least) {
      least = t;
      best = p;
    }
  };
  // (windows' shared tiles stay within the workspace, which is sized without one)
  const int most = window > 0 ? bwd_max_parts(B, Hq, Hkv, N, D) : INT_MAX;
  // (a launch counts its work-items in 32 bits: one item per tile always fits)
  const double threads = cost.W > 128 ? 256.0 : 512.0;
  auto search = [&](bool w4, bool may_share) {
    // Windows and unequal sides: another plan only for a clear gain.
    if ((window > 0 || cost.nk != cost.nq) && w4 == plain.w4) consider(plain, 0.95 * cost.together(w4));
    consider({false, 1, w4}, cost.together(w4));
    for (const int parts : kPartsTried) {
      if (parts > 1 && (!may_share || NK != N || parts > most)) break;
      if (!cost.allows(parts, N) || (cost.n1 * parts + cost.n2 + 16) * threads > 4294967295.0) break;
      consider({true, parts, w4}, cost.apart(parts, w4));
    }
  };
  search(false, share != BwdShare::kNone);
  if (has_w4) search(true, share != BwdShare::kNone);
  if (share == BwdShare::kSameDq && best.parts > 1) {
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
      const BwdPlan p = bwd_plan(B, Hq, Hkv, N, N, D, causal, 0, w4, BwdShare::kShare);
      if (p.parts > most) most = p.parts;
    }
  return most;
}

// Estimated microseconds of a forward on each kernel, fitted per width to 6110
// random square shapes (100 <= N <= 8192, B <= 16, 1 to 64 heads) and 1359 with
// up to 16384 more keys than query rows, every candidate timed for each. Over
// 1400 random calls each the plan taken is 2.4% slower than the best candidate on
// average (key lengths, ALiBi and dropout 2%, a bias 0.9%, packed sequences, which
// it does not see, 5.5%), fa_fwd.hip alone 31% (24% with dropout, 89% with a
// window). Same box, fa_fwd.hip -> the plan's: 358 -> 312 us at B=2 H=32/8 N=3001
// D=128 dense (fa_rows.hip, 4 waves), 312 -> 293 at B=1 H=16 N=8192 D=128 causal
// (4 waves, paired), 248 -> 164 at B=9 H=12 N=2145 D=128 causal (the same), 21 ->
// 8.0 at B=14 H=12 N=189 D=64 causal (8 waves); fa_fwd.hip stays where few rows
// leave CUs idle (B=1 H=8 N=4096 D=128 causal: 48 us, 73 with 4 waves). More keys
// than rows: 222 -> 100 at B=16 H=32/8 N=1, 8192 keys, D=128 (fa_dec.hip, 2 parts);
// 240 -> 30 at B=1 H=32/8 N=1, 32768 keys (24 parts); 225 -> 19 at B=1 H=16/2 N=4,
// 8000 keys, D=256 (32 parts); 134 -> 86 at B=1 H=32/8 N=512, 8192 keys
// (fa_rows.hip, 8 waves, 3 parts).
namespace {

// One kernel's times at a width.
struct FwdTimes {
  double solo, full;  // a step of a workgroup, alone on its CU and with it full
  double ends;        // a tile's start and end
  double uneven;      // (causal fa_rows.hip) the end of the grid, in longest tiles
  int per_cu;         // workgroups that share a CU
};
enum { kW32, kW64, kW96, kW128, kW256 };
constexpr FwdTimes kTilesTimes[] = {{0.60, 0.70, 4.2, 0, 1}, {0.60, 0.70, 4.2, 0, 1},
                                    {0.80, 0.95, 4.2, 0, 1}, {0.98, 1.12, 7.0, 0, 1},
                                    {1.38, 1.38, 20.2, 0, 1}};
constexpr FwdTimes kRows4Times[] = {{0.69, 2.38, 4.6, 0.25, 4}, {0.69, 2.38, 4.6, 0.25, 4},
                                    {0.86, 2.28, 4.9, 0.31, 3}, {1.02, 1.93, 5.6, 0.41, 2},
                                    {2.06, 2.54, 8.7, 0.39, 1}};
constexpr FwdTimes kRows8Times[] = {{1.03, 2.49, 4.8, 0.25, 2}, {1.03, 2.49, 4.8, 0.25, 2},
                                    {1.21, 1.63, 4.9, 0.32, 1}, {1.46, 2.11, 6.0, 0.27, 1},
                                    {2.72, 4.12, 9.5, 0.20, 1}};
constexpr FwdTimes kPairTimes[] = {{0.80, 2.67, 3.4, 0, 4}, {0.80, 2.67, 3.4, 0, 4},
                                   {1.21, 2.66, 3.8, 0, 3}, {1.49, 2.24, 4.2, 0, 2},
                                   {2.96, 3.08, 6.2, 0, 1}};
// (a round of fa_dec.hip: 256 keys, 128 at width 256)
constexpr double kDecTimes[] = {0.9, 0.9, 1.3, 1.6, 1.5};
// Two workgroups per CU of fa_fwd.hip (FwdShape W4): a step on a full chip.
constexpr double kTilesW4[] = {0, 1.27, 0, 2.2, 0};

double step_time(const FwdTimes& t, double per_cu) {
  if (t.per_cu == 1) return t.full;
  const double r = fmin(fmax(per_cu, 1.0), t.per_cu);
  return t.solo + (t.full - t.solo) * (r - 1) / (t.per_cu - 1);
}
// n equal workgroups of `steps` steps and `tiles` tiles.
double equal_time(const FwdTimes& t, double n, double steps, double tiles) {
  const double slots = (double)kCUs * t.per_cu, full = floor(n / slots), rest = n - full * slots;
  double us = full * (steps * t.full + tiles * t.ends);
  if (rest > 0) us += steps * step_time(t, ceil(rest / kCUs)) + tiles * t.ends;
  return us;
}
// n causal tiles of `total` steps in all, the longest first.
double uneven_time(const FwdTimes& t, double n, double total, double longest) {
  const double slots = (double)kCUs * t.per_cu;
  return fmax(total * t.full / slots + n / slots * t.ends + t.uneven * longest * t.full,
              longest * step_time(t, ceil(n / kCUs)) + t.ends);
}
double ceil_div(double a, double b) { return ceil(a / b); }

}  // namespace

FwdPlan fwd_plan(const FwdArgs& a, bool workspace) {
  FwdPlan best{FwdPlan::kTiles, 0, false, 1, 0, 0};
  // fa_rows.hip takes dropout, a bias (whose rows load 16 bytes at a time) or
  // ALiBi alone, the first two at widths up to 128; the other per-score inputs
  // stay on fa_fwd.hip.
  const bool feat = a.drop || a.bias || a.alibi;
  if (a.mask || a.block_rows || (a.drop && a.bias) || ((a.drop || a.bias) && (a.alibi || a.D > 128)))
    return best;
  if (a.bias && ((a.N | a.bias_sb | a.bias_sh) % 4 != 0 ||
                 (reinterpret_cast<uintptr_t>(a.bias) & 15) != 0))
    return best;
  const int NK = key_rows(a.N, a.Nkv), W = padded_head_dim(a.D);
  const int wi = W <= 32 ? kW32 : W <= 64 ? kW64 : W <= 96 ? kW96 : W <= 128 ? kW128 : kW256;
  const double BH = (double)a.B * a.Hq, kofs = NK - a.N;
  // Keys seen by the rows of a tile that ends before row i1, a window's start rounded down.
  auto keys = [&](double rows, double i1) {
    const double hi = a.causal ? fmax(1, fmin(NK, i1 + kofs)) : NK;
    return a.window > 0 ? fmin(hi, rows + a.window) : hi;
  };
  double least, wgs;  // fa_fwd.hip's time and workgroups
  {  // fa_fwd.hip
    const double n = ceil_div(a.N, 64), stage = W > 128 ? 64 : 128;
    const bool pairs = a.causal && n > 1;
    wgs = (pairs ? ceil_div(n, 2) : n) * BH;
    const double first = ceil_div(keys(64, 64), stage), last = ceil_div(keys(64, 64 * n), stage);
    const double steps = 0.5 * (first + last) * n * BH / wgs, tiles = pairs ? 2 : 1;
    const FwdTimes& t = kTilesTimes[wi];
    const bool masked = a.N % 64 || a.kv_len || a.window > 0 || a.alibi || a.seg_start || NK != a.N;
    least = 1 + (kTilesW4[wi] > 0 && wgs >= 2 * kCUs && !(a.causal && masked)
                     ? wgs / (2 * kCUs) * (steps * kTilesW4[wi] + tiles * t.ends)
                     : equal_time(t, wgs, steps, tiles));
  }
  // These inputs cost the two kernels differently: a bias takes fa_fwd.hip 2.6
  // times as long as none and fa_rows.hip 1.6 times (B=4 H=8 N=1024 D=64 dense:
  // 51 -> 28 us, B=1 H=16 N=4096 D=64 causal: 217 -> 127, B=2 H=32 N=1500 D=128
  // causal: 185 -> 120); dropout costs fa_rows.hip more than fa_fwd.hip's unmasked
  // copies (79 us there and 82 here at B=1 H=16 N=4096 D=64 causal) and as much as
  // its masked ones, which a ragged N takes (96 -> 72 us at B=2 H=32 N=1500 D=128).
  // Dense grids of at most one tile per CU gain nothing from waves of 32 rows at
  // the widths from 128 on, whose estimate there is 15-20% high, nor with a bias
  // (up to width 64: on half as many tiles): 28.7 us against 37.0 at B=1 H=2 N=1396
  // D=96, 14.7 against 17.9 at B=2 H=4 N=400 D=128 with one, 17.0 against 20.4 at
  // B=4 H=4 N=260 D=256 without. Of 1400 random calls with a bias 99 ran more than
  // 5% slower than on fa_fwd.hip without this rule, 4 with it.
  // On causal grids of as few workgroups the estimates' errors decide, so another
  // kernel is taken for a clear gain only: at most half a workgroup per CU, 7%, and
  // with ALiBi, which costs fa_rows.hip more, 10% on up to one (14.1 us against 16.1
  // at B=1 H=1 N=896 D=64): of 1400 random calls 46 without per-score inputs and 29
  // with ALiBi were more than 5% slower than on fa_fwd.hip before, 35 and 3 now.
  // (Not at width 256, where fa_fwd.hip's estimate errs the other way: 88 us
  // there and 63 on fa_rows.hip at B=3 H=2 N=1727.)
  const bool square = NK == a.N && !a.seg_start && a.window == 0;
  const double few = a.bias && W <= 64 ? kCUs / 2 : kCUs;
  if (square && !a.causal && wgs <= few)
    least *= a.bias ? (W <= 64 ? 1.0 : W <= 96 ? 0.9 : 0.8) : (W <= 96 ? 1.0 : W <= 128 ? 0.85 : 0.8);
  else if (a.bias)
    least *= 1.6;
  else if (square && a.causal && W <= 128)
    least *= a.alibi && wgs <= kCUs ? 0.9 : wgs <= kCUs / 2 ? 0.93 : 1.0;
  if (a.drop && a.N % 128 == 0) least *= 0.85;
  // A launch's work-items and the row blocks' indices stay within 32 bits.
  constexpr double kMostItems = 4294967295.0;
  auto consider = [&](FwdPlan p, double us) {
    if (us >= least) return;
    least = us;
    best = p;
  };
  // What parts cost: a second launch (3 us, and 2 on the host, which small calls
  // wait for) and the partial results to write and combine.
  auto merge = [&](double items, int parts) {
    return parts == 1 ? 0.0 : 5.0 + 0.0137 * items * parts * W / 128;
  };
  const bool split = NK > a.N && !a.seg_start;  // square calls' results do not depend on a workspace
  // Without a workspace the search is over one part only: a kernel that is the
  // best one with several parts can be far from it with one (B=1 H=32/8 N=512,
  // 8192 keys, D=128 causal: 182 us on 8 waves of fa_rows.hip, 111 on
  // fa_dec.hip, 138 on fa_fwd.hip).
  const bool shared = split && workspace;
  constexpr int kTried[] = {1, 2, 3, 4, 6, 8, 12, 16, 24, 32, 48, 64};
  {  // fa_rows.hip
    for (const int waves : {4, 8}) {
      if (feat && waves == 8) continue;
      const double rows = 32.0 * waves, n = ceil_div(a.N, rows);
      const double first = ceil_div(keys(rows, rows), 64), last = ceil_div(keys(rows, rows * n), 64);
      const double total = 0.5 * (first + last) * n * BH, items = n * waves * BH;
      const FwdTimes& t = waves == 4 ? kRows4Times[wi] : kRows8Times[wi];
      if (n * BH * 512 > kMostItems) continue;
      for (const int parts : kTried) {
        if (parts > 16 || (parts > 1 && (!shared || last < 2 * parts || items * parts > 8192))) break;
        const double us = a.causal && n > 1 ? uneven_time(t, n * BH * parts, total, last / parts)
                                            : equal_time(t, n * BH * parts, ceil(last / parts), 1);
        consider({FwdPlan::kRows, waves, false, parts, (int)(n * waves), (int)items},
                 us + merge(items, parts));
      }
      if (waves == 4 && a.causal && n > 1) {
        const double wgs = ceil_div(n, 2) * BH;
        consider({FwdPlan::kRows, 4, true, 1, (int)(n * waves), (int)items},
                 equal_time(kPairTimes[wi], wgs, total / wgs, 2));
      }
    }
  }
  if (split) {  // fa_dec.hip
    // (K and V come at 6 TB/s from 170 workgroups on, fewer cannot keep enough
    // loads in flight: B=4 H=32/8 N=1, 32000 keys, D=128 takes 309, 173, 106 and
    // 95 us with 1, 2, 4 and 8 parts of 32 workgroups)
    const double tiles = ceil_div((double)(a.Hq / a.Hkv) * a.N, 32), items = tiles * a.B * a.Hkv;
    const double seen = keys(a.N, a.N), read = 4.0 * a.B * a.Hkv * seen * a.D / 6.0e6;
    if (items * (W / 32) * 512 <= kMostItems) {
      for (const int parts : kTried) {
        if (parts > 1 && (!shared || seen < 128.0 * parts || items * parts > 8192)) break;
        const double rounds = ceil_div(ceil_div(seen, parts), W > 128 ? 128 : 256) * kDecTimes[wi];
        const double n = items * parts, full = floor(n / kCUs), rest = n - full * kCUs;
        double us = full * (rounds * 1.36 + 1.3);
        if (rest > 0) us += rounds * (rest < kCUs / 2 ? 1.0 : 1.36) + 1.3;
        consider({FwdPlan::kDec, 0, false, parts, (int)tiles, (int)items},
                 2 + fmax(us, read * fmax(1.0, pow(170.0 / n, 0.6))) + merge(items, parts));
      }
    }
  }
  return best;
}

hipError_t launch_fwd(const FwdArgs& a, const FwdPlan& plan, void* workspace) {
  const bool bf = a.dtype == kBF16;
  const hipError_t e = by_width(a, bf, [&](auto w, auto bf, const FwdArgs& a) {
    constexpr int W = decltype(w)::value;
    constexpr bool BF = decltype(bf)::value;
    switch (plan.kind) {
      case FwdPlan::kRows: return launch_rows_w<W, BF>(a, plan, workspace);
      case FwdPlan::kDec: return launch_dec_w<W, BF>(a, plan, workspace);
      default: return launch_fwd_w<W, BF>(a);
    }
  });
  if (e != hipSuccess || plan.parts <= 1) return e;
  return by_width(a, bf, [&](auto w, auto bf, const FwdArgs& a) {
    return launch_merge_w<decltype(w)::value, decltype(bf)::value>(a, plan, workspace);
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
