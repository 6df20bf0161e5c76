// Forward over grids that fill the chip: a wave owns 32 query rows and every
// key its rows see (the counterpart of fa_fwd.hip, whose waves share their rows
// and split the keys; fa_launch.hip picks). No counterpart in the reference
// beyond flash::fwd_kernel (flash_fwd.cuh:68-340).
//
// Bound: in fa_fwd.hip a 64-row tile loads every K/V row it sees, so at two
// workgroups per CU the direct loads (21.75 cycles per KB per CU) take 1392
// cycles per 1024 of MFMA. Here 4 waves share each stage over 128 rows (two
// workgroups per CU) or 8 over 256 (one): 0.33 or 0.17 of that, no partial
// results to merge at the end and one barrier per 64 keys. What is left is LDS
// reads (about 1350 of 2048 cycles per stage and CU) beside the products and
// the softmax, which the other waves of a SIMD overlap. Measured and not kept:
// S of the next stage, or that and P V of the last, in flight during the
// softmax (3-5% slower, 251 registers); two row blocks per wave, which halves
// the LDS reads (one wave per SIMD: 8-12% slower); 32- and 128-key stages
// (within 3%, slower); wave priorities (1-2% slower).
//
// Row i sees the keys [lower(i), upper(i)): causal masking aligned at the
// bottom right, windows, key lengths and packed sequences all come down to
// these bounds, of which neither decreases with i; only the stages at the ends
// of a wave's bounds test them, and stages outside them are skipped.
//
// Dropout (FEAT kFeatDrop): a lane's keep bits of the next stage (two words of
// its row) load during this one. Bias (kFeatBias): each wave's 32 x 64 values of
// the next stage load into LDS of its own as soon as this stage's are in
// registers (fa_fwd.hip reads them per lane from rows N floats apart, 32 cache
// lines per load).
#include <type_traits>

#include "fa_device.h"
#include "fa_launch.h"

namespace fa {
namespace {

constexpr int kFeatAlibi = 64;  // (a FEAT bit beside Feat's)

template <int D, int NW>
struct Rows {
  static constexpr int kThreads = 64 * NW;
  static constexpr int kRows = 32 * NW;  // query rows of a workgroup
  static constexpr int kKeys = 64;       // keys of a stage
  static constexpr int kTileHalves = TileLoad<D, kKeys, NW>::kHalves;
};

struct RowsArgs {
  const half_t* q;
  const half_t* k;
  const half_t* v;
  half_t* o;
  float* lse;
  float* part_o;    // partial O^T and (max, sum) of each 32-row block and part
  float2* part_ml;  // (parts > 1; DecArgs' layout)
  int N, NK, Hq, group, n_tiles, BH, parts, causal, window, dr;
  float scale_log2;
  const uint32_t* drop;  // as FwdArgs (kFeatDrop, kFeatBias instantiations)
  float drop_scale;
  const float* alibi;  // (kFeatAlibi)
  const float* bias;
  long long bias_sb, bias_sh;
  float bias_raw;  // 1 / softmax scale
  const int* kv_len;
  const int* seg_start;
  const int* seg_end;
  Strides stq, stk;
};

// PAIR (causal): a workgroup takes query tile T-1-x, then x, so that all do the
// same work; without it the tiles start longest first.
template <int D, int NW, bool PAIR, int FEAT, bool BF>
__global__ __launch_bounds__((Rows<D, NW>::kThreads)) __attribute__((amdgpu_waves_per_eu(2, 2)))
void rows_kernel(const RowsArgs a) {
  using R = Rows<D, NW>;
  constexpr int kKeys = R::kKeys;
  // K and V of two stages as distinct LDS objects, so that the compiler can
  // tell a stage's reads from the other one's loads.
  __shared__ __align__(16) half_t kt0[R::kTileHalves];
  __shared__ __align__(16) half_t vt0[R::kTileHalves];
  __shared__ __align__(16) half_t kt1[R::kTileHalves];
  __shared__ __align__(16) half_t vt1[R::kTileHalves];
  constexpr bool DROP = FEAT == kFeatDrop, BIAS = FEAT == kFeatBias, ALIBI = FEAT == kFeatAlibi;
  // Bias rows of a wave: 64 floats, 16-byte chunk c of row r at position c ^
  // (r % 16), so that 16 rows' reads of one chunk hit 16 bank groups.
  __shared__ __align__(16) float bt[BIAS ? NW * 32 * kKeys : 4];
  const int gx = PAIR ? (a.n_tiles + 1) / 2 : a.n_tiles;
  const int w = xcd_work_index(gx * a.parts * a.BH);
  if (w < 0) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  __builtin_assume(wave >= 0 && wave < NW);
  const int h = lane >> 5, l32 = lane & 31;
  const int x = w % gx, part = w / gx % a.parts, bh = w / (gx * a.parts);
  const int b = bh / a.Hq, hq = bh % a.Hq, hkv = hq / a.group;

  const int kofs = a.NK - a.N;
  const int Nk = a.kv_len ? min(max(a.kv_len[b], 1), a.NK) : a.NK;
  const int* const sst = a.seg_start ? a.seg_start + (size_t)b * a.N : nullptr;
  const int* const sen = a.seg_end ? a.seg_end + (size_t)b * a.N : nullptr;
  auto lower = [&](int i) {
    i = min(i, a.N - 1);
    int lo = a.window > 0 ? i + kofs - a.window + 1 : 0;
    if (sst) lo = max(lo, min(sst[i], i));
    return max(lo, 0);
  };
  auto upper = [&](int i) {
    i = min(i, a.N - 1);
    if (a.causal) return min(Nk, i + kofs + 1);
    return sen ? min(Nk, max(sen[i], i + 1)) : Nk;
  };

  const float c = a.scale_log2, thr_raw = kRescaleLog2 / c;
  // ALiBi slope of this head in raw-score units.
  const float slope = ALIBI ? a.alibi[hq] * kLog2e / c : 0.f;
  const int roff = row_lane_off<D>(lane), troff = tr_lane_off<D>(lane);
  const size_t kv_off = (size_t)(b * a.stk.b + hkv * a.stk.h);
  // Rows from the key length on read as zeros: a masked key's P is zero, but
  // zero times a NaN or an infinity that the padding holds would be NaN.
  const rsrc_t rk = rows_rsrc(a.k + kv_off, Nk, a.stk.n, a.dr);
  const rsrc_t rv = rows_rsrc(a.v + kv_off, Nk, a.stk.n, a.dr);
  TilePlan<D, kKeys, NW, false> plan;
  plan.init(wave, lane, a.stk.n, a.dr);
  constexpr int kParts = decltype(plan)::kParts;

  const int n_mine = PAIR && a.n_tiles - 1 - x != x ? 2 : 1;
  for (int turn = 0; turn < n_mine; ++turn) {
    const int tile = turn ? x : a.n_tiles - 1 - x;
    const int q0 = tile * R::kRows, i_base = q0 + wave * 32, i_row = i_base + l32;
    const half_t* qrow =
        a.q + b * a.stq.b + hq * a.stq.h + (size_t)min(i_row, a.N - 1) * a.stq.n;
    half8 qb[D / 16];
#pragma unroll
    for (int kk = 0; kk < D / 16; ++kk)
      qb[kk] = as_half8(load16(qrow + kk * 16 + h * 8, kk * 16 + h * 8 < a.dr));
    // This lane's row, the wave's rows (some see [w_lo, w_hi), all of them
    // [all_lo, all_hi)) and the stages the tile's rows reach, of which this
    // workgroup runs its part (at least one stage: with no key in reach every
    // score is masked).
    const int lo = lower(i_row), hi = upper(i_row);
    const int w_lo = lower(i_base), w_hi = upper(i_base + 31);
    const int all_lo = lower(i_base + 31), all_hi = upper(i_base);
    const int s_lo = lower(q0) / kKeys;
    const int s_hi = max(s_lo + 1, (upper(q0 + R::kRows - 1) + kKeys - 1) / kKeys);
    const int per = (s_hi - s_lo + a.parts - 1) / a.parts;
    const int first = min(s_lo + part * per, s_hi - 1);
    const int last = max(first + 1, min(s_lo + (part + 1) * per, s_hi));
    const bool none = s_lo + part * per >= s_hi;  // (a part without stages)

    floatx16 oacc[D / 32];
#pragma unroll
    for (int cb = 0; cb < D / 32; ++cb) oacc[cb] = zero16();
    float m_raw = -INFINITY, l = 0.f;
    if (PAIR && turn) __syncthreads();  // the last tile's stages have been read
    const int W32 = (a.N + 31) >> 5;
    const uint32_t* zrow =
        DROP ? a.drop + ((size_t)bh * a.N + min(i_row, a.N - 1)) * W32 : nullptr;
    auto zword = [&](int j, int t) { return DROP ? zrow[min(2 * j + t, W32 - 1)] : ~0u; };
    uint32_t zw[2] = {zword(first, 0), zword(first, 1)};
    const rsrc_t rb = bias_rows_rsrc(BIAS ? a.bias + b * a.bias_sb + hq * a.bias_sh : nullptr,
                                     i_base, a.N);
    // Instruction u covers the wave's rows 4u .. 4u+3.
    auto bload = [&](int j) {
      if constexpr (BIAS) {
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int r = 4 * u + (lane >> 4);
          lds_direct_buf<16>(bt, rb, (uint32_t)(r * a.N) * 4u + ((lane ^ r) & 15) * 16u,
                             (uint32_t)(j * kKeys) * 4u, (uint32_t)(wave * 32 * kKeys + u * 256) * 4u);
        }
      }
    };
    bload(first);
#pragma unroll
    for (int u = 0; u < kParts; ++u) {
      plan.part(kt0, rk, first * kKeys, wave, u);
      plan.part(vt0, rv, first * kKeys, wave, u);
    }
    // Stage j in the buffers of parity P, while the next one loads.
    auto step = [&](int j, auto par) {
      constexpr int P = decltype(par)::value;
      const half_t* Ks = P ? kt1 : kt0;
      const half_t* Vs = P ? vt1 : vt0;
      wait_vmem();
      __syncthreads();
      const int jn = min(j + 1, last - 1) * kKeys;
      auto issue = [&](int s) {  // the next stage's loads leave between the products
        if (s < 2 * kParts) {
          if (s & 1) plan.part(P ? vt0 : vt1, rv, jn, wave, s >> 1);
          else plan.part(P ? kt0 : kt1, rk, jn, wave, s >> 1);
        }
      };
      const int base = j * kKeys;
      const uint32_t zc[2] = {zw[0], zw[1]};
      if constexpr (DROP) {
        zw[0] = zword(min(j + 1, last - 1), 0);
        zw[1] = zword(min(j + 1, last - 1), 1);
      }
      if (none || base >= w_hi || base + kKeys <= w_lo) {  // no key for any row of the wave
#pragma unroll
        for (int u = 0; u < 2 * kParts; ++u) issue(u);
        if constexpr (BIAS) bload(min(j + 1, last - 1));
        return;
      }
      floatx16 s[2] = {zero16(), zero16()}, bv[2];
      // The bias is added to the finished products (kept in the accumulators from
      // the start, every product would round at its magnitude). Up to width 64
      // there are registers to read it before them.
      auto bread = [&] {
        const float* brow = bt + wave * 32 * kKeys + l32 * kKeys;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const floatx4 x =
                *reinterpret_cast<const floatx4*>(brow + (((8 * t + 2 * g + h) ^ l32) & 15) * 4);
#pragma unroll
            for (int e = 0; e < 4; ++e) bv[t][4 * g + e] = x[e];
          }
        __builtin_amdgcn_s_waitcnt(0xC07F);  // the reads are done before the loads below
        __builtin_amdgcn_sched_barrier(0);
        bload(min(j + 1, last - 1));
      };
      if constexpr (BIAS && D <= 64) bread();
#pragma unroll
      for (int t = 0; t < 2; ++t) {
#pragma unroll
        for (int kk = 0; kk < D / 16; ++kk) {
          s[t] = mfma16<BF>(tile_read16<D>(Ks, 32 * t, kk, roff), qb[kk], s[t]);
          issue(t * (D / 16) + kk);
        }
      }
#pragma unroll
      for (int u = 2 * (D / 16); u < 2 * kParts; ++u) issue(u);
      if constexpr (BIAS) {
        if constexpr (D > 64) bread();
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int e = 0; e < 16; ++e) s[t][e] = fmaf(bv[t][e], a.bias_raw, s[t][e]);
      }
      if constexpr (ALIBI) {  // -slope |i - j|, distances exact in fp32
        const float d0 = (float)(i_row + kofs - base - 4 * h);
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int e = 0; e < 16; ++e)
            s[t][e] = fmaf(-slope, fabsf(d0 - (float)(32 * t + 8 * (e >> 2) + (e & 3))), s[t][e]);
      }
      if (base < all_lo || base + kKeys > all_hi) {
        const int d = base + 4 * h;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            const int key = d + 32 * t + 8 * (e >> 2) + (e & 3);
            if (key < lo || key >= hi) s[t][e] = -INFINITY;
          }
      }
      float mloc = s[0][0];
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) mloc = fmaxf(mloc, s[t][e]);
      mloc = max_halves(mloc);
      if (__builtin_expect(__any(mloc > m_raw + thr_raw), 0)) {
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
      half8 pb[4];
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const float p = fast_exp2(fmaf(s[t][e], c, neg));
          l += p;
          // Dropout: the row sum keeps every key, P V only the kept ones.
          const bool keep = !DROP || ((zc[t] >> (4 * h)) >> (8 * (e >> 2) + (e & 3))) & 1u;
          pb[2 * t + (e >> 3)][e & 7] = to16<BF>(keep ? p : 0.f);
        }
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int cb = 0; cb < D / 32; ++cb)
          oacc[cb] = mfma16<BF>(tile_tr_operand<D>(Vs, 16 * q, 32 * cb, troff), pb[q], oacc[cb]);
    };
    int j = first;
    for (; j + 2 <= last; j += 2) {
      step(j, std::integral_constant<int, 0>{});
      step(j + 1, std::integral_constant<int, 1>{});
    }
    if (j < last) step(j, std::integral_constant<int, 0>{});

    const float l_all = l + xor32(l);
    if (a.parts > 1) {  // for dec_merge_kernel: row blocks of 32, fa_dec.hip's layout
      const size_t slot = ((size_t)bh * (a.n_tiles * NW) + tile * NW + wave) * a.parts + part;
      float* po = a.part_o + slot * (32 * D);
#pragma unroll
      for (int cb = 0; cb < D / 32; ++cb)
#pragma unroll
        for (int g = 0; g < 4; ++g)
          *reinterpret_cast<floatx4*>(po + ((cb * 4 + g) * 64 + lane) * 4) =
              floatx4{oacc[cb][4 * g], oacc[cb][4 * g + 1], oacc[cb][4 * g + 2], oacc[cb][4 * g + 3]};
      if (h == 0) a.part_ml[slot * 32 + l32] = make_float2(m_raw * c, l_all);
    } else if (i_row < a.N) {
      // (a row without keys: O = 0; dropout scales the kept keys)
      const float inv_l = l_all > 0.f ? (DROP ? a.drop_scale : 1.f) / l_all : 0.f;
      half_t* orow = a.o + b * a.stq.b + hq * a.stq.h + (size_t)i_row * a.stq.n;
#pragma unroll
      for (int cb = 0; cb < D / 32; ++cb)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          half4 o4;
#pragma unroll
          for (int e = 0; e < 4; ++e) o4[e] = to16<BF>(oacc[cb][4 * g + e] * inv_l);
          if (cb * 32 + 8 * g + 4 * h < a.dr)
            *reinterpret_cast<half4*>(orow + cb * 32 + 8 * g + 4 * h) = o4;
        }
      if (h == 0)
        a.lse[(size_t)bh * a.N + i_row] =
            l_all > 0.f ? (m_raw * c + __log2f(l_all)) * kLn2 : INFINITY;
    }
  }
}

template <int D, int NW, bool PAIR, int FEAT, bool BF>
hipError_t launch_rows_t(const RowsArgs& a, hipStream_t stream) {
  const int gx = PAIR ? (a.n_tiles + 1) / 2 : a.n_tiles;
  hipLaunchKernelGGL((rows_kernel<D, NW, PAIR, FEAT, BF>),
                     dim3((unsigned)xcd_grid(gx * a.parts * a.BH)), dim3(Rows<D, NW>::kThreads), 0,
                     stream, a);
  return hipGetLastError();
}

}  // namespace

template <>
hipError_t launch_rows_w<FA_WIDTH, FA_BF>(const FwdArgs& a, const FwdPlan& plan, void* workspace) {
  constexpr int D = FA_WIDTH;
  RowsArgs d{};
  d.q = (const half_t*)a.q;
  d.k = (const half_t*)a.k;
  d.v = (const half_t*)a.v;
  d.o = (half_t*)a.o;
  d.lse = a.lse;
  d.N = a.N;
  d.NK = key_rows(a.N, a.Nkv);
  d.Hq = a.Hq;
  d.group = a.Hq / a.Hkv;
  d.n_tiles = (a.N + 32 * plan.waves - 1) / (32 * plan.waves);
  d.BH = a.B * a.Hq;
  d.parts = plan.parts;
  d.causal = a.causal;
  d.window = a.window;
  d.dr = a.D;
  d.scale_log2 = kLog2e * (a.scale > 0.f ? a.scale : 1.f / sqrtf((float)a.D));
  d.kv_len = a.kv_len;
  d.seg_start = a.seg_start;
  d.seg_end = a.seg_end;
  d.stq = make_strides(a.layout, a.Hq, a.N, a.D);
  d.stk = make_strides(a.layout, a.Hkv, d.NK, a.D);
  if (plan.parts > 1) {
    d.part_ml = (float2*)workspace;
    d.part_o = (float*)((char*)workspace + part_ml_bytes(plan));
  }
  const hipStream_t stream = (hipStream_t)a.stream;
  d.drop = a.drop;
  d.drop_scale = a.drop_scale;
  d.bias = a.bias;
  d.bias_sb = a.bias_sb;
  d.bias_sh = a.bias_sh;
  d.bias_raw = 1.f / (a.scale > 0.f ? a.scale : 1.f / sqrtf((float)a.D));
  if constexpr (D <= 128) {  // (the plan keeps width 256 with these two on fa_fwd.hip)
    if (a.drop)
      return plan.pair ? launch_rows_t<D, 4, true, kFeatDrop, FA_BF>(d, stream)
                       : launch_rows_t<D, 4, false, kFeatDrop, FA_BF>(d, stream);
    if (a.bias)
      return plan.pair ? launch_rows_t<D, 4, true, kFeatBias, FA_BF>(d, stream)
                       : launch_rows_t<D, 4, false, kFeatBias, FA_BF>(d, stream);
  }
  d.alibi = a.alibi;
  if (a.alibi)
    return plan.pair ? launch_rows_t<D, 4, true, kFeatAlibi, FA_BF>(d, stream)
                     : launch_rows_t<D, 4, false, kFeatAlibi, FA_BF>(d, stream);
  if (plan.waves == 8) return launch_rows_t<D, 8, false, 0, FA_BF>(d, stream);
  return plan.pair ? launch_rows_t<D, 4, true, 0, FA_BF>(d, stream)
                   : launch_rows_t<D, 4, false, 0, FA_BF>(d, stream);
}

}  // namespace fa
