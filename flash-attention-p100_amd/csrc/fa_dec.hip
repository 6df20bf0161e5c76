// Forward over few query rows and many keys: KV-cache decoding (one row per
// sequence) and short chunks behind a long cache. No counterpart in the
// reference, which has one row count for q, k and v (fa_p100.py:48-55).
//
// Bound: HBM, each K/V row is read once per 32 query rows. fa_fwd.hip gives
// every query head a 64-row tile of its own and one workgroup all its keys:
// at one row per head that reads K/V once per query head of a group (through
// L2) and leaves the CUs idle that have no (b, head). Here
//   * a row tile is 32 rows of one kv head: the rows of all the query heads of
//     its group, head after head (row r of the tile's kv head is query head
//     r / N of the group, row r % N), so K/V are read once per group;
//   * the keys are cut into `parts` runs, a workgroup each, whose partial
//     (max, sum, O) dec_merge_kernel combines;
//   * in a workgroup every wave takes 32-key blocks of its own (block kWaves *
//     i + wave of the run) through its own LDS tiles, so that no barrier ties
//     the waves' loads together; K's next block loads while V's is used and
//     the other way round. The waves' partials meet in LDS at the end.
// The products, the softmax and the operand layouts are fa_fwd.hip's (S^T =
// K Q^T, lazy rescaling, O^T += V^T P^T on v_mfma_f32_32x32x16).
#include <type_traits>

#include "fa_device.h"
#include "fa_launch.h"

namespace fa {
namespace {

constexpr int kRows = 32;             // query rows of a tile
constexpr int kKeys = 32;             // keys of a wave's block

template <int D>
struct Dec {
  // (width 256: a wave's K and V tiles take 34 KB of LDS)
  static constexpr int kWaves = D > 128 ? 4 : 8;
  static constexpr int kThreads = 64 * kWaves;
  static constexpr int kTileHalves = Tile<D>::template halves<kKeys>();  // of one wave
  static constexpr int kFloats = kRows * D;  // a partial O (one row tile)
  static_assert(kWaves / 2 * kFloats * 4 <= kWaves * kTileHalves * 2, "merge area exceeds the tiles");
};

// A wave's LDS reads so far are done: its tile may be loaded again.
__device__ __forceinline__ void wait_lds() {
  __builtin_amdgcn_s_waitcnt(0xC07F);
  __builtin_amdgcn_sched_barrier(0);
}

struct DecArgs {
  const half_t* q;
  const half_t* k;
  const half_t* v;
  half_t* o;
  float* lse;
  float* part_o;   // (item, part) x kFloats: unscaled partial O^T, in accumulator order
  float2* part_ml; // (item, part) x kRows: running max (log2 units), row sum
  int N, NK, Hq, group, n_tiles, items, parts, causal, window, dr;
  float scale_log2;
  const int* kv_len;
  const float* alibi;
  Strides stq, stk;
};

// Partial O^T of one lane in accumulator order: entry (cb * 4 + g) * 64 + lane
// holds columns 32cb + 8g + 4(lane / 32) .. +3 of row lane % 32.
template <int D, bool BF>
__global__ __launch_bounds__((Dec<D>::kThreads)) void dec_kernel(const DecArgs a) {
  using T = Dec<D>;
  constexpr int kWaves = T::kWaves;
  __shared__ __align__(16) half_t kt[kWaves * T::kTileHalves];
  __shared__ __align__(16) half_t vt[kWaves * T::kTileHalves];
  __shared__ float2 ml[kWaves * 64];
  const int w = xcd_work_index(a.items * a.parts);
  if (w < 0) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  __builtin_assume(wave >= 0 && wave < kWaves);
  const int h = lane >> 5, l32 = lane & 31;
  // Work item: row tile `tile` of (b, kv head) bkv, key run `part`; a kv
  // head's tiles of one run are neighbours, so that they share K/V in L2.
  const int tile = w % a.n_tiles, part = w / a.n_tiles % a.parts, bkv = w / (a.n_tiles * a.parts);
  const int Hkv = a.Hq / a.group, b = bkv / Hkv, hkv = bkv % Hkv;
  const int rows = a.group * a.N;
  const int r = tile * kRows + l32;  // this lane's row of the kv head
  const bool row_ok = r < rows;
  const int rc = min(r, rows - 1);
  const int hq = hkv * a.group + rc / a.N, n = rc % a.N;
  const half_t* qrow = a.q + b * a.stq.b + hq * a.stq.h + (size_t)n * a.stq.n;
  half8 qb[D / 16];
#pragma unroll
  for (int kk = 0; kk < D / 16; ++kk)
    qb[kk] = as_half8(load16(qrow + kk * 16 + h * 8, kk * 16 + h * 8 < a.dr));

  // Keys [lo, hi) of this lane's row (the diagonal aligned at the bottom
  // right), and the tile's: rows of one tile may belong to several heads, so
  // the bounds are over its rows' n.
  const int kofs = a.NK - a.N;
  const int Nk = a.kv_len ? min(max(a.kv_len[b], 1), a.NK) : a.NK;
  auto lower = [&](int i) { return a.window > 0 ? max(0, i + kofs - a.window + 1) : 0; };
  auto upper = [&](int i) { return a.causal ? min(Nk, i + kofs + 1) : Nk; };
  const int lo = lower(n), hi = upper(n);
  const int r0 = tile * kRows, r1 = min(r0 + kRows, rows) - 1;
  const bool wraps = r0 / a.N != r1 / a.N;  // rows of several heads: any n
  const int n0 = wraps ? 0 : r0 % a.N, n1 = wraps ? a.N - 1 : r1 % a.N;
  const int t_lo = lower(n0), t_hi = upper(n1);    // some row sees these keys
  const int all_lo = lower(n1), all_hi = upper(n0);  // every row sees these
  const int first = t_lo / kKeys, n_blocks = max(0, (t_hi + kKeys - 1) / kKeys - first);
  const int per = (n_blocks + a.parts - 1) / a.parts;
  const int j0 = first + part * per, j1 = min(j0 + per, first + n_blocks);

  const float c = a.scale_log2, thr_raw = kRescaleLog2 / c;
  const float alibi_raw = a.alibi ? a.alibi[hq] * kLog2e / c : 0.f;
  const int roff = row_lane_off<D>(lane), troff = tr_lane_off<D>(lane);
  const size_t kv_off = (size_t)(b * a.stk.b + hkv * a.stk.h);
  // Rows from the key length on read as zeros: a masked key's P is zero, but
  // zero times a NaN or an infinity that the padding holds would be NaN.
  const rsrc_t rk = rows_rsrc(a.k + kv_off, Nk, a.stk.n, a.dr);
  const rsrc_t rv = rows_rsrc(a.v + kv_off, Nk, a.stk.n, a.dr);
  TilePlan<D, kKeys, 1, false> plan;
  plan.init(0, lane, a.stk.n, a.dr);
  half_t* const my_k = kt + wave * T::kTileHalves;
  half_t* const my_v = vt + wave * T::kTileHalves;
  // The loads take the array and a byte offset (lds_direct_buf).
  auto load = [&](half_t* array, rsrc_t rs, int block) {
#pragma unroll
    for (int u = 0; u < decltype(plan)::kParts; ++u)
      lds_direct_buf<16>(array, rs, plan.off[u], (uint32_t)(block * kKeys) * plan.row_bytes,
                         (uint32_t)(wave * T::kTileHalves * 2 + u * 1024));
  };

  floatx16 oacc[D / 32];
#pragma unroll
  for (int cb = 0; cb < D / 32; ++cb) oacc[cb] = zero16();
  float m_raw = -INFINITY, l = 0.f;
  constexpr int kLoads = decltype(plan)::kParts;
  // s_waitcnt for all but the last kLoads vector memory operations
  constexpr int kWaitOlder = 0x0F70 | (kLoads & 15) | ((kLoads >> 4) << 14);
  int j = j0 + wave;
  if (j < j1) {
    load(kt, rk, j);
    load(vt, rv, j);
  }
  for (; j < j1; j += kWaves) {
    const int jn = min(j + kWaves, j1 - 1);  // (past the end: loaded, not used)
    __builtin_amdgcn_s_waitcnt(kWaitOlder);  // K's block is here, V's may be under way
    floatx16 s = zero16();
#pragma unroll
    for (int kk = 0; kk < D / 16; ++kk)
      s = mfma16<BF>(tile_read16<D>(my_k, 0, kk, roff), qb[kk], s);
    wait_lds();
    load(kt, rk, jn);
    const int base = j * kKeys + 4 * h;
    if (alibi_raw != 0.f) {
      const float d0 = (float)(n + kofs - base);
#pragma unroll
      for (int e = 0; e < 16; ++e)
        s[e] = fmaf(-alibi_raw, fabsf(d0 - (float)(8 * (e >> 2) + (e & 3))), s[e]);
    }
    if (j * kKeys < all_lo || (j + 1) * kKeys > all_hi) {
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int key = base + 8 * (e >> 2) + (e & 3);
        if (key < lo || key >= hi) s[e] = -INFINITY;
      }
    }
    float mloc = s[0];
#pragma unroll
    for (int e = 1; e < 16; ++e) mloc = fmaxf(mloc, s[e]);
    mloc = max_halves(mloc);
    if (__any(mloc > m_raw + thr_raw)) {
      const float m_new = fmaxf(m_raw, mloc);
      const float corr = m_raw == -INFINITY ? 0.f : fast_exp2((m_raw - m_new) * c);
      l *= corr;
#pragma unroll
      for (int cb = 0; cb < D / 32; ++cb)
#pragma unroll
        for (int e = 0; e < 16; ++e) oacc[cb][e] *= corr;
      m_raw = m_new;
    }
    const float neg = m_raw == -INFINITY ? 0.f : -m_raw * c;
    half8 pb[2];
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const float p = fast_exp2(fmaf(s[e], c, neg));
      l += p;
      pb[e >> 3][e & 7] = to16<BF>(p);
    }
    __builtin_amdgcn_s_waitcnt(kWaitOlder);  // V's block is here, K's next may be under way
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int cb = 0; cb < D / 32; ++cb)
        oacc[cb] = mfma16<BF>(tile_tr_operand<D>(my_v, 16 * q, 32 * cb, troff), pb[q], oacc[cb]);
    wait_lds();
    load(vt, rv, jn);
  }
  wait_vmem();
  __syncthreads();  // every wave's loads have landed: the tiles hold the merge area

  auto part_of = [&](int src) {
    return reinterpret_cast<float*>(src < kWaves / 2 ? kt : vt) + src % (kWaves / 2) * T::kFloats;
  };
#pragma unroll
  for (int cb = 0; cb < D / 32; ++cb)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const floatx4 v = {oacc[cb][4 * g], oacc[cb][4 * g + 1], oacc[cb][4 * g + 2],
                         oacc[cb][4 * g + 3]};
      *reinterpret_cast<floatx4*>(part_of(wave) + ((cb * 4 + g) * 64 + lane) * 4) = v;
    }
  ml[wave * 64 + lane] = make_float2(m_raw, l);
  __syncthreads();
  float m_star = -INFINITY, l_star = 0.f, wk[kWaves];
#pragma unroll
  for (int k = 0; k < kWaves; ++k) m_star = fmaxf(m_star, ml[k * 64 + lane].x);
#pragma unroll
  for (int k = 0; k < kWaves; ++k) {
    const float2 x = ml[k * 64 + lane];
    wk[k] = x.x == -INFINITY ? 0.f : fast_exp2((x.x - m_star) * c);
    l_star += wk[k] * (x.y + ml[k * 64 + (lane ^ 32)].y);
  }
  const bool whole = a.parts == 1;
  const float inv_l = l_star > 0.f ? 1.f / l_star : 0.f;  // a row without keys: O = 0
  const size_t slot = (size_t)(bkv * a.n_tiles + tile) * a.parts + part;
  half_t* orow = a.o + b * a.stq.b + hq * a.stq.h + (size_t)n * a.stq.n;
  constexpr int kRuns = D / 8;  // float4 runs per lane, dealt to the waves
#pragma unroll
  for (int i = 0; i < (kRuns + kWaves - 1) / kWaves; ++i) {
    const int run = i * kWaves + wave;
    if (run >= kRuns) break;
    floatx4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < kWaves; ++k)
      acc += *reinterpret_cast<const floatx4*>(part_of(k) + (run * 64 + lane) * 4) * wk[k];
    if (!whole) {
      *reinterpret_cast<floatx4*>(a.part_o + slot * T::kFloats + (run * 64 + lane) * 4) = acc;
    } else if (row_ok && 8 * run + 4 * h < a.dr) {
      half4 o4;
#pragma unroll
      for (int e = 0; e < 4; ++e) o4[e] = to16<BF>(acc[e] * inv_l);
      *reinterpret_cast<half4*>(orow + 8 * run + 4 * h) = o4;
    }
  }
  if (wave == 0 && h == 0) {
    if (!whole) a.part_ml[slot * kRows + l32] = make_float2(m_star * c, l_star);
    else if (row_ok)
      a.lse[((size_t)b * a.Hq + hq) * a.N + n] =
          l_star > 0.f ? (m_star * c + __log2f(l_star)) * kLn2 : INFINITY;
  }
}

// Combines the parts of each row tile: one float4 of a partial O per thread.
template <int D, bool BF>
__global__ __launch_bounds__(256) void dec_merge_kernel(const DecArgs a) {
  constexpr int kBlocks = D / 32;  // workgroups per row tile
  const int item = blockIdx.x / kBlocks, f = blockIdx.x % kBlocks * 256 + threadIdx.x;
  const int tile = item % a.n_tiles, bkv = item / a.n_tiles;
  const int lane = f % 64, run = f / 64, l32 = lane & 31, h = lane >> 5;
  const int Hkv = a.Hq / a.group, b = bkv / Hkv, hkv = bkv % Hkv;
  const int r = tile * kRows + l32;
  if (r >= a.group * a.N) return;
  const int hq = hkv * a.group + r / a.N, n = r % a.N;
  const float2* ml = a.part_ml + (size_t)item * a.parts * kRows + l32;
  const float* po = a.part_o + (size_t)item * a.parts * Dec<D>::kFloats + 4 * f;
  float m = -INFINITY;
#pragma unroll 4
  for (int p = 0; p < a.parts; ++p) m = fmaxf(m, ml[p * kRows].x);
  floatx4 acc = {0.f, 0.f, 0.f, 0.f};
  float l = 0.f;
#pragma unroll 4
  for (int p = 0; p < a.parts; ++p) {
    const float2 x = ml[p * kRows];
    const float w = x.x == -INFINITY ? 0.f : fast_exp2(x.x - m);  // (no key: zeros)
    l += w * x.y;
    acc += *reinterpret_cast<const floatx4*>(po + (size_t)p * Dec<D>::kFloats) * w;
  }
  const float inv_l = l > 0.f ? 1.f / l : 0.f;
  if (8 * run + 4 * h < a.dr) {
    half4 o4;
#pragma unroll
    for (int e = 0; e < 4; ++e) o4[e] = to16<BF>(acc[e] * inv_l);
    *reinterpret_cast<half4*>(a.o + b * a.stq.b + hq * a.stq.h + (size_t)n * a.stq.n + 8 * run +
                              4 * h) = o4;
  }
  if (run == 0 && h == 0)
    a.lse[((size_t)b * a.Hq + hq) * a.N + n] = l > 0.f ? (m + __log2f(l)) * kLn2 : INFINITY;
}

}  // namespace

static DecArgs dec_args(const FwdArgs& a, const FwdPlan& plan, void* workspace) {
  DecArgs d{};
  d.q = (const half_t*)a.q;
  d.k = (const half_t*)a.k;
  d.v = (const half_t*)a.v;
  d.o = (half_t*)a.o;
  d.lse = a.lse;
  d.N = a.N;
  d.NK = key_rows(a.N, a.Nkv);
  d.Hq = a.Hq;
  d.group = a.Hq / a.Hkv;
  d.n_tiles = plan.tiles;
  d.items = plan.items;
  d.parts = plan.parts;
  d.causal = a.causal;
  d.window = a.window;
  d.dr = a.D;
  d.scale_log2 = kLog2e * (a.scale > 0.f ? a.scale : 1.f / sqrtf((float)a.D));
  d.kv_len = a.kv_len;
  d.alibi = a.alibi;
  d.stq = make_strides(a.layout, a.Hq, a.N, a.D);
  d.stk = make_strides(a.layout, a.Hkv, d.NK, a.D);
  if (plan.parts > 1) {
    d.part_ml = (float2*)workspace;
    d.part_o = (float*)((char*)workspace + part_ml_bytes(plan));
  }
  return d;
}

template <>
hipError_t launch_dec_w<FA_WIDTH, FA_BF>(const FwdArgs& a, const FwdPlan& plan, void* workspace) {
  constexpr int D = FA_WIDTH;
  const DecArgs d = dec_args(a, plan, workspace);
  hipLaunchKernelGGL((dec_kernel<D, FA_BF>), dim3((unsigned)xcd_grid(plan.items * plan.parts)),
                     dim3(Dec<D>::kThreads), 0, (hipStream_t)a.stream, d);
  return hipGetLastError();
}

// Combines the parts of fa_rows.hip's row blocks (each a head's own: group 1)
// or of this file's row tiles.
template <>
hipError_t launch_merge_w<FA_WIDTH, FA_BF>(const FwdArgs& a, const FwdPlan& plan, void* workspace) {
  constexpr int D = FA_WIDTH;
  DecArgs d = dec_args(a, plan, workspace);
  if (plan.kind == FwdPlan::kRows) d.group = 1;
  hipLaunchKernelGGL((dec_merge_kernel<D, FA_BF>), dim3((unsigned)plan.items * (D / 32)), dim3(256),
                     0, (hipStream_t)a.stream, d);
  return hipGetLastError();
}

}  // namespace fa
