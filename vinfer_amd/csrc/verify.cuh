// Speculative-decoding verify: accept each draft token with probability min(1, p / q), where p
// and q are the target's and the draft's final probabilities of that token; at the first
// rejection, draw the replacement from the residual max(0, p - q) (renormalised); when every
// draft is accepted, the target's own draw at the position after the last draft is the bonus
// token. This is the rule of Leviathan, Kalman, Matias 2023 and Chen et al. 2023 ("speculative
// sampling"), which emits tokens distributed exactly as the target's p.
//
// Everything is decided in the sampling kernel's own fixed point, so it is exact integer
// arithmetic: a token's mass is P = rint(p~ * 2^42) (p~ = exp(z - max z) after the filters,
// 0 for dropped tokens) and its probability P / S, S the row's kept mass. Then
//   accept  <=>  m * Q_d * S_t < P_d * S_d * 2^24      (m = floor(u * 2^24))
//   residual weight of token i:  w_i = max(0, (P_i * S_d >> s) - (Q_i * S_t >> s)),
// with s = floor(log2(max(S_t, S_d))), which keeps the sum below 2^63 and each weight within a
// factor two of the target mass it stands for. The drawn token is the first id (ascending)
// whose inclusive prefix of w exceeds floor(m * R / 2^24), R the sum. A point-mass row (greedy,
// degenerate) has mass 2^42 at its token and S = 2^42.
//
// The sampling kernel has already run over the target rows and the draft rows (its RowState output
// gives each row's kept set, max and S), so these kernels read logits only where they decide: the
// drafted tokens' two values per position and, for a rejected position, the target and draft rows,
// once to sum the residual and once more inside the stripe that holds the token. The drafted
// positions' rows are not drawn from (but in the rare row without residual mass). The bonus position's
// row is drawn from where it costs least:
//   * while the target rows fit one round on the CUs, in that launch (BonusDraws), which one more
//     workgroup a sequence makes ~4 us longer; the residuals' launch then works out the acceptance
//     itself (ResidualRow), and a fully accepted sequence is done. V = 151936, us a call in this form
//     against the other one: 8 sequences of 1 draft 30.4/47.2 against 49.1/48.8 (all accepted / drafts
//     from a close draft model), 64 of 2 33.3/52.7 against 53.7/54.5, 128 of 1 34.2/56.1 against
//     52.8/53.6; where every sequence is rejected it is slower by those 4 us;
//   * past one round, where those rows would cost rounds of their own, only after all drafts were
//     accepted (k_verify_accept), in one launch with the residual draws (VerifyRow): 192 sequences
//     of one draft, V = 262144, 137.4 us a call when every target row was sampled first (384 rows, one
//     and a half rounds on 256 CUs) and the residuals took a launch of their own, 89 us now.
// A bf16 row holds at most 65536 distinct values, and its kept ones sit in a short run of keys
// below the row's max: the two terms of w are tabulated per key in LDS for the top kTab keys
// of each row (a kept token below that run is computed directly), so the residual pass costs
// two LDS reads per token instead of two fp64 exponentials and two 128-bit products.
#pragma once

#include <type_traits>

#include "penalty.cuh"
#include "sample.cuh"

namespace vs {

struct VerifyArgs {
  const void* tgt;  // target row (b, j), j <= K, at tgt + (b * (K + 1) + j) * tstride
  int64_t tstride;
  const void* drf;  // draft row (b, j), j < K, at drf + (b * K + j) * dstride
  int64_t dstride;
  int V, K;
  const int32_t* drafts;  // [B * K] drafted tokens
  const float* u_acc;     // [B * K] acceptance uniforms
  const float* u_res;     // [B * K] residual-draw uniforms
  const RowState* ts;     // [B * (K + 1)] (the drafted positions' entries)
  const RowState* ds;     // [B * K]
  int32_t* out_tokens;    // [B * (K + 1)]: the emitted tokens, then -1
  int32_t* out_count;     // [B]
  int32_t* jr;            // [B] the first rejected position (K: none)
  uint32_t* done;         // [B] slices of the row's residual finished
  u64* sums;              // [B * kMaxStripes] per-stripe residual sums
  int32_t* rej;           // [B] the rejected sequences, ascending
  int32_t* acc;           // [B] the others, ascending
  int32_t* nrej;          // [1] how many are rejected
  int B;
  int max_slices;         // most workgroups per rejected row (a power of two)
};

using u128 = unsigned __int128;

constexpr u64 kPointMass = 4398046511104ull;  // 2^42: mass_q(1)

// A row's kept mass in the fixed point of its token masses.
__device__ __forceinline__ u64 kept_mass(const RowState& s) { return s.point >= 0 ? kPointMass : s.S; }

// Token `id` (value x) of a row: its mass under the row's state.
__device__ __forceinline__ u64 token_mass(float x, int id, const RowState& s) {
  if (s.point >= 0) return id == s.point ? kPointMass : 0;
  const bool keep = x >= s.x0 && (!s.partial || x > s.vc || (x == s.vc && id <= s.idr));
  return keep ? mass_q(ptilde(x, s.T, s.mz)) : 0;
}

// floor(u * 2^24) for u in [0, 1) (u * 2^24 is exact in fp32).
__device__ __forceinline__ u64 u24(float u) {
  const float v = u * 16777216.0f;
  return v > 0.0f ? static_cast<u64>(v) : 0ull;
}

// Order-preserving 16-bit key of a bf16 value (its bits), and the value of a key.
__device__ __forceinline__ uint32_t bf16_key(uint32_t bits) { return (bits & 0x8000u) ? (~bits & 0xFFFFu) : (bits | 0x8000u); }
// The key of a token's bf16 value for the residual's table: -0.0 takes +0.0's key (they are one
// value, and the kept set's bound `lo` is +0.0 when it is zero).
__device__ __forceinline__ uint32_t bf16_key_z(uint32_t bits) { return bf16_key(bits == 0x8000u ? 0u : bits); }
__device__ __forceinline__ float bf16_of_key(uint32_t key) {
  const uint32_t bits = (key & 0x8000u) ? (key & 0x7FFFu) : (~key & 0xFFFFu);
  return __uint_as_float(bits << 16);
}

constexpr int kTab = 8192;  // tabulated keys per row (bf16)

// One row's side of the residual: the term (mass * other_S) >> shift of each token. Both forms
// are free of branches (a point row has lo = +inf and its token in pid; other rows pid = -1),
// so that the per-token code stays one straight run.
struct ResidualSide {
  RowState st;
  u64 other_S;
  int shift;
  float lo;                // kept tokens have x >= lo (x0, or the split group's value); point row: +inf
  float vcx;               // the split group's value (partial rows), else NaN
  int pid;                 // a point row's token, else -1
  uint32_t tlo, thi;       // tabulated keys: [tlo, thi] at tab[1 + k - tlo] (tab[0] = 0)
  const u64* tab;
  u64 point_term;  // a point row's token

  __device__ __forceinline__ bool kept(float x, int id) const {
    return (x >= lo) & !((x == vcx) & (id > st.idr));
  }
  // a kept token of value x (not a point row)
  __device__ __forceinline__ u64 kept_term(float x) const {
    return static_cast<u64>((static_cast<u128>(mass_q(ptilde(x, st.T, st.mz))) * other_S) >> shift);
  }
  __device__ __forceinline__ u64 direct(float x, int id) const {
    return kept(x, id) ? kept_term(x) : (id == pid ? point_term : 0ull);
  }
  // bf16 row (not a point row) whose kept keys are all tabulated: the term of key k, value x
  // (every key >= tlo is a value >= lo, every key below maps to entry 0)
  __device__ __forceinline__ u64 term(float x, uint32_t k, int id) const {
    const int i = static_cast<int>(k) - static_cast<int>(tlo) + 1;
    const u64 t = tab[i > 0 ? i : 0];
    return ((x == vcx) & (id > st.idr)) ? 0ull : t;
  }
};

// Whether draft j of sequence b is accepted.
template <class Tin>
__device__ __forceinline__ bool accepts(const VerifyArgs& a, int b, int j) {
  const int K = a.K;
  // (no branch on the token, so that the states' loads do not wait for it; the logits' do)
  const int d = a.drafts[b * K + j];
  const RowState st = a.ts[b * (K + 1) + j];
  const RowState sd = a.ds[b * K + j];
  const int at = d < 0 ? 0 : (d < a.V ? d : a.V - 1);
  const float xt = load_one<Tin>(static_cast<const Tin*>(a.tgt) + static_cast<int64_t>(b * (K + 1) + j) * a.tstride, at);
  const float xd = load_one<Tin>(static_cast<const Tin*>(a.drf) + static_cast<int64_t>(b * K + j) * a.dstride, at);
  const u64 P = token_mass(xt, d, st), Q = token_mass(xd, d, sd);
  const u128 lhs = static_cast<u128>(u24(a.u_acc[b * K + j])) * Q * kept_mass(st);  // < 2^127
  const u128 rhs = (static_cast<u128>(P) * kept_mass(sd)) << 24;
  return (d == at) & (lhs < rhs);  // (a token outside the vocabulary is never accepted)
}

// One workgroup, a thread per sequence: the acceptance chain. Writes the accepted drafts and, when
// all are accepted, the count; leaves the first rejected position in jr, clears the row's slice
// counter and lists the rejected and the accepted sequences (ascending) for the last launch.
template <class Tin>
__global__ __launch_bounds__(kThreads) void k_verify_accept(VerifyArgs a) {
  __shared__ uint32_t red[kWaves];
  exp_table_init();
  __syncthreads();
  const int K = a.K, B = a.B;
  uint32_t listed = 0;
  for (int b0 = 0; b0 < B; b0 += kThreads) {
    const int b = b0 + static_cast<int>(threadIdx.x);
    int j = K;
    if (b < B) {
      for (j = 0; j < K && accepts<Tin>(a, b, j); ++j) {
      }
      int32_t* out = a.out_tokens + static_cast<int64_t>(b) * (K + 1);
      for (int i = 0; i <= K; ++i) out[i] = i < j ? a.drafts[b * K + i] : -1;
      if (j == K) a.out_count[b] = K + 1;  // (the last launch draws the bonus token)
      a.jr[b] = j;
      a.done[b] = 0;
    }
    const uint32_t r = j < K ? 1u : 0u;
    uint32_t tot;
    const uint32_t at = listed + block_excl_scan<uint32_t>(r, red, &tot);
    if (r) a.rej[at] = b;
    else if (b < B) a.acc[b - static_cast<int>(at)] = b;
    listed += tot;
  }
  if (threadIdx.x == 0) *a.nrej = static_cast<int32_t>(listed);
}

// Workgroups per rejected row: the largest power of two with every (row, slice) item on its own
// of the `room` workgroups that the bonus rows leave, at most max_slices.
__device__ __forceinline__ int residual_slices(int nrej, int room, int max_slices) {
  int s = 1;
  while (2 * s <= max_slices && static_cast<int64_t>(2 * s) * nrej <= room) s *= 2;
  return s;
}

// The residual's LDS: the tabulated terms lie over the sampling kernel's histogram, the rest over its
// FastSmem.
struct ResidualSmem {
  u64 cell[kWaves][kMaxStripes];
  u64 red[kWaves];
  u64 sq[4];
  int si[4];
};
static_assert(sizeof(ResidualSmem) <= sizeof(FastSmem), "the residual's scratch lies over FastSmem");
static_assert(2 * kTab * sizeof(u64) <= kChunk * sizeof(uint32_t), "the tables lie over the histogram");

// One (row, slice) item of the residual draw of sequence b, rejected at position jr: the slice sums the residual
// over its share of the row's stripes; the last slice of the row to finish finds the stripe that
// holds floor(m * R / 2^24) and the token inside it. Returns true (in every thread of the last
// slice's workgroup) when the row has no residual mass: the caller draws from the target row.
template <class Tin>
__device__ __forceinline__ bool residual_item(const VerifyArgs& a, int b, int jr, int slice, int slices,
                                              uint32_t* big, ResidualSmem& m) {
  constexpr bool kBf16 = sizeof(Tin) == 2;
  auto& cell = m.cell;
  auto& red = m.red;
  auto& sq = m.sq;
  auto& si = m.si;
  u64* const tab[2] = {reinterpret_cast<u64*>(big), reinterpret_cast<u64*>(big) + kTab};
  const int tid = threadIdx.x;
  const int wv = tid / kWave;
  const int K = a.K;
  const Tin* tgt = static_cast<const Tin*>(a.tgt);
  const Tin* drf = static_cast<const Tin*>(a.drf);
  int32_t* out = a.out_tokens + static_cast<int64_t>(b) * (K + 1);
  // The rejected position's residual, over the target and draft rows at position jr.
  Row<Tin> rt, rd;
  rt.p = tgt + static_cast<int64_t>(b * (K + 1) + jr) * a.tstride;
  rd.p = drf + static_cast<int64_t>(b * K + jr) * a.dstride;
  rt.V = rd.V = a.V;
  rt.nblk = rd.nblk = (a.V + kBlk - 1) / kBlk;
  rt.nstripes = rd.nstripes = (rt.nblk + kThreads - 1) / kThreads;
  rt.bm = rd.bm = nullptr;
  rt.eid = rd.eid = nullptr;
  rt.eval = rd.eval = nullptr;
  rt.nexc = rd.nexc = 0;
  // this workgroup's stripes
  const int per = (rt.nstripes + slices - 1) / slices;
  const int j_begin = slice * per;
  const int j_end = min(rt.nstripes, j_begin + per);
  ResidualSide side[2];
  bool tabled = kBf16;
  side[0].st = a.ts[b * (K + 1) + jr];
  side[1].st = a.ds[b * K + jr];
  const u64 St = kept_mass(side[0].st), Sd = kept_mass(side[1].st);
  const int shift = 63 - __clzll(static_cast<long long>(St > Sd ? St : Sd));
  side[0].other_S = Sd;
  side[1].other_S = St;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    ResidualSide& sd = side[h];
    sd.shift = shift;
    sd.lo = sd.st.point >= 0 ? INFINITY : sd.st.partial && sd.st.vc > sd.st.x0 ? sd.st.vc : sd.st.x0;
    sd.vcx = sd.st.point < 0 && sd.st.partial ? sd.st.vc : NAN;
    sd.pid = sd.st.point >= 0 ? sd.st.point : -1;
    sd.point_term = static_cast<u64>((static_cast<u128>(kPointMass) * sd.other_S) >> shift);
    sd.tab = tab[h];
    sd.tlo = 1;
    sd.thi = 0;  // (empty)
    if constexpr (kBf16) {
      if (sd.st.point < 0) {
        // the largest finite key whose scaled value is <= the row's max (z is monotone in x)
        uint32_t lo = 0x007Fu, hi = 0xFF80u;  // -inf .. +inf
        while (lo < hi) {
          const uint32_t mid = (lo + hi + 1) / 2;
          const float x = bf16_of_key(mid);
          const float z = sd.st.T == 1.0f ? x : x / sd.st.T;
          if (z <= sd.st.mz) lo = mid;
          else hi = mid - 1;
        }
        sd.thi = lo;
        // the smallest key whose value is >= lo (lo need not be a bf16 value)
        uint32_t klo = 0x007Fu;
        if (sd.lo != -INFINITY) {
          klo = bf16_key(__float_as_uint(sd.lo) >> 16);
          if (bf16_of_key(klo) < sd.lo) ++klo;
        }
        sd.tlo = klo;
        if (sd.thi >= sd.tlo && sd.thi - sd.tlo < static_cast<uint32_t>(kTab - 1)) {
          if (tid == 0) tab[h][0] = 0;
          for (uint32_t k = sd.tlo + tid; k <= sd.thi; k += kThreads)
            tab[h][1 + k - sd.tlo] = sd.kept_term(bf16_of_key(k));  // (x >= lo: kept, but for a split group's ids)
        } else {
          tabled = false;  // (uniform) the kept keys do not fit: every term computed directly
        }
      } else {
        tabled = false;  // (uniform) a point row: its one term computed directly
      }
    }
  }
  __syncthreads();
  // The residual is 0 wherever the target drops the token (P = 0).
  const float tlo = side[0].lo;
  const int tpid = side[0].pid;
  auto kept_lanes = [&](const float (&vt)[kBlk], uint32_t valid, int blk) {
    uint32_t kept = 0;
#pragma unroll
    for (int i = 0; i < kBlk; ++i) {
      const bool k = vt[i] >= tlo || blk * kBlk + i == tpid;
      kept |= ((valid >> i) & 1u) && k ? 1u << i : 0u;
    }
    return kept;
  };
  auto weight = [&](float xt, float xd, int id, auto tab_mode) -> u64 {
    u64 pt, qd;
    if constexpr (decltype(tab_mode)::value) {
      pt = side[0].term(xt, bf16_key_z(__float_as_uint(xt) >> 16), id);
      qd = side[1].term(xd, bf16_key_z(__float_as_uint(xd) >> 16), id);
    } else {
      pt = side[0].direct(xt, id);
      qd = side[1].direct(xd, id);
    }
    return pt > qd ? pt - qd : 0;
  };
  auto weights = [&](const float (&vt)[kBlk], const float (&vd)[kBlk], uint32_t kept, int blk, u64 w[kBlk],
                     auto tab_mode) {
#pragma unroll
    for (int i = 0; i < kBlk; ++i) {
      w[i] = 0;
      if (kept & (1u << i)) w[i] = weight(vt[i], vd[i], blk * kBlk + i, tab_mode);
    }
  };
  // Both phases that read the rows, for one mode (tabulated terms or direct ones).
  auto residual = [&](auto tab_mode) -> bool {
    // 1. this slice's per-stripe sums; four stripes' loads of both rows in flight (the draft
    // block is read whether or not a target value in it is kept: a load behind a branch would
    // be waited for alone)
    auto stripe_sum = [&](int j, const float (&vt)[kBlk], const float (&vd)[kBlk], uint32_t valid) {
      const int blk = j * kThreads + tid;
      u64 w[kBlk];
      weights(vt, vd, kept_lanes(vt, valid, blk), blk, w, tab_mode);
      u64 s = 0;
#pragma unroll
      for (int i = 0; i < kBlk; ++i) s += w[i];
      s = wave_sum<u64>(s);
      if (lane_id() == 0) cell[wv][j - j_begin] = s;
    };
    if constexpr (decltype(tab_mode)::value) {
      // Tabulated rows: both values of a word at once. idx2 gives their table entries (the key less
      // the lowest kept one, saturating: 0 for a dropped token, whose term is 0), in a handful of
      // packed instructions; a split group's values past its id take entry 0 too. Two stripes of
      // both rows stay in flight. (As whole blocks of values with a term's own key, range and group
      // tests a token, four stripes loaded and then worked on, the launch of 149 bonus rows
      // and 43 rejected ones of 262144 took 58-60 us, two slices a row; 44 now, the bonus rows' own
      // time. 192 rejected ones, one workgroup each: 143 us a call, now 111.)
      const int nfull = a.V / kBlk;
      const uint16_t* pt = nfull > 0 ? reinterpret_cast<const uint16_t*>(rt.p) : g_unused_block;
      const uint16_t* pd = nfull > 0 ? reinterpret_cast<const uint16_t*>(rd.p) : g_unused_block;
      uint32_t below[2], split[2];  // (key below the lowest kept, the split group's entry) twice
      bool fold[2];                 // a zero may be kept: -0.0 takes +0.0's key
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        below[h] = (side[h].tlo - 1u) * 0x10001u;
        fold[h] = side[h].tlo <= 0x8000u;
        split[h] = side[h].vcx == side[h].vcx
                       ? bf16_key_z(__float_as_uint(side[h].vcx) >> 16) - (side[h].tlo - 1u)
                       : 0u;  // (0: no split group, or one that holds no bf16 value)
        if (split[h] && (__float_as_uint(side[h].vcx) & 0xFFFFu)) split[h] = 0u;
      }
      auto idx2 = [&](uint32_t w, int h) -> ushort2_t {
        if (fold[h]) {  // (uniform) the halves that are 0x8000 become 0
          const ushort2_t nz = __builtin_elementwise_min(__builtin_bit_cast(ushort2_t, w ^ 0x80008000u), ones2());
          w &= ~(__builtin_bit_cast(uint32_t, ones2() - nz) << 15);
        }
        return __builtin_elementwise_sub_sat(__builtin_bit_cast(ushort2_t, ok16x2(w)),
                                             __builtin_bit_cast(ushort2_t, below[h]));
      };
      auto load = [&](int j, uint4& t, uint4& d) {
        const int blk = min(j * kThreads + tid, max(nfull - 1, 0));
        t = ld_block(pt, blk);
        d = ld_block(pd, blk);
      };
      auto one_stripe = [&](int j, uint4 t, uint4 d) {
        const int blk = j * kThreads + tid;
        if (blk >= nfull) {  // the ragged last block; past it nothing (a NaN's bits: entry 0)
          uint32_t wt[4], wd[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            wt[i] = wd[i] = 0xFFFFFFFFu;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              const int id = blk * kBlk + 2 * i + h;
              if (blk == nfull && id < a.V) {
                wt[i] = (wt[i] & ~(0xFFFFu << (16 * h))) | static_cast<uint32_t>(ld_global(reinterpret_cast<const uint16_t*>(rt.p) + id)) << (16 * h);
                wd[i] = (wd[i] & ~(0xFFFFu << (16 * h))) | static_cast<uint32_t>(ld_global(reinterpret_cast<const uint16_t*>(rd.p) + id)) << (16 * h);
              }
            }
          }
          t = make_uint4(wt[0], wt[1], wt[2], wt[3]);
          d = make_uint4(wd[0], wd[1], wd[2], wd[3]);
        }
        const uint32_t wt[4] = {t.x, t.y, t.z, t.w}, wd[4] = {d.x, d.y, d.z, d.w};
        u64 s = 0;
        auto add = [&](uint32_t it, uint32_t id_) {
          const u64 p = tab[0][it], q = tab[1][id_];
          s += p > q ? p - q : 0ull;
        };
        // (uniform over the wave) its ids, and whether a split group ends at or before their last
        const int id0 = (j * kThreads + wv * kWave) * kBlk;
        const bool ends = (split[0] && id0 + kWave * kBlk - 1 > side[0].st.idr) ||
                          (split[1] && id0 + kWave * kBlk - 1 > side[1].st.idr);
        if (ends) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const ushort2_t a2 = idx2(wt[i], 0), b2 = idx2(wd[i], 1);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              const int id = blk * kBlk + 2 * i + h;
              const uint32_t it = h ? a2.y : a2.x, jd = h ? b2.y : b2.x;
              add(split[0] && it == split[0] && id > side[0].st.idr ? 0u : it,
                  split[1] && jd == split[1] && id > side[1].st.idr ? 0u : jd);
            }
          }
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const ushort2_t a2 = idx2(wt[i], 0), b2 = idx2(wd[i], 1);
            add(a2.x, b2.x);
            add(a2.y, b2.y);
          }
        }
        s = wave_sum<u64>(s);
        if (lane_id() == 0) cell[wv][j - j_begin] = s;
      };
      if (j_begin < j_end) {  // (uniform; a slice past the row's stripes has none)
        uint4 t0, d0, t1, d1;
        load(j_begin, t0, d0);
        load(min(j_begin + 1, j_end - 1), t1, d1);
        for (int j = j_begin; j < j_end; j += 2) {
          const uint4 t = t0, d = d0;
          load(min(j + 2, j_end - 1), t0, d0);
          one_stripe(j, t, d);
          if (j + 1 < j_end) {
            const uint4 u = t1, v = d1;
            load(min(j + 3, j_end - 1), t1, d1);
            one_stripe(j + 1, u, v);
          }
        }
      }
    } else
    for (int j0 = j_begin; j0 < j_end; j0 += 4) {
      if (j0 + 4 <= j_end && (j0 + 4) * kThreads * kBlk <= a.V) {
        // (uniform) four stripes wholly inside both rows
        WholeBlock<Tin> qt[4], qd[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          qt[k].load(rt.p, (j0 + k) * kThreads + tid);
          qd[k].load(rd.p, (j0 + k) * kThreads + tid);
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          float vt[kBlk], vd[kBlk];
          qt[k].values(vt);
          qd[k].values(vd);
          stripe_sum(j0 + k, vt, vd, 0xFFu);
        }
      } else {
        for (int j = j0; j < j_end && j < j0 + 4; ++j) {
          const int blk = j * kThreads + tid;
          float vt[kBlk], vd[kBlk];
          const uint32_t valid = blk < rt.nblk ? rt.load(blk, vt) & rd.load(blk, vd) : 0u;
          stripe_sum(j, vt, vd, valid);
        }
      }
    }
    // The stripe sums go to the other slices as relaxed agent-scope atomic stores, which are
    // coherent across the XCDs' L2s by themselves; each writer waits for its stores to complete
    // (vmcnt counts stores too) before the workgroup barrier and the counter's atomic add, and
    // the last slice loads them with agent-scope atomic loads only after that add has returned.
    // Device-scope fences (an L2 write-back and an invalidate per slice, ~15 us of a call)
    // are not needed for these few words; nothing else crosses workgroups here. This rests on
    // gfx950's encoding rather than on the HIP memory model, which orders relaxed atomics only
    // through a release/acquire pair: an agent-scope atomic store or load is a vector store or
    // load with the SC1 bit (device scope), written through the writer's L2 and read from the
    // device's coherence point, and vmcnt(0) returns once the store has reached that point.
    __syncthreads();
    if (tid < j_end - j_begin) {
      u64 t = 0;
      for (int w = 0; w < kWaves; ++w) t += cell[w][tid];
      __hip_atomic_store(&a.sums[b * kMaxStripes + j_begin + tid], t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    __syncthreads();
    if (tid == 0) si[2] = static_cast<int>(atomicAdd(&a.done[b], 1u));
    __syncthreads();
    if (si[2] != slices - 1) return false;  // (uniform) another slice finishes the row
    // 2. (last slice) stripe totals; the stripe where the running sum passes floor(m * R / 2^24)
    if (wv == 0) {
      const int j = lane_id();
      const u64 t = j < rt.nstripes ? __hip_atomic_load(&a.sums[b * kMaxStripes + j], __ATOMIC_RELAXED,
                                                        __HIP_MEMORY_SCOPE_AGENT)
                                    : 0ull;
      const u64 inc = wave_incl_scan<u64>(t);
      const u64 R = dpp::last(inc);
      const u64 m = u24(a.u_res[b * K + jr]);
      u64 tg = m * (R >> 24) + ((m * (R & 0xFFFFFFull)) >> 24);
      if (R > 0 && tg > R - 1) tg = R - 1;
      const bool hit = R > 0 && inc > tg && inc - t <= tg;
      const u64 hm = __ballot(hit);
      if (j == 0) {
        sq[0] = R;
        sq[1] = tg;
        si[1] = hm ? __ffsll(static_cast<long long>(hm)) - 1 : 0;
      }
      if (hit) sq[2] = inc - t;
    }
    __syncthreads();
    if (sq[0] == 0) {  // (uniform) no residual mass: the target's own draw at this position
      if (tid == 0) a.out_count[b] = jr + 1;
      return true;
    }
    const u64 tg = sq[1];
    const int js = si[1];
    const u64 base = sq[2];
    // 3. per-thread sums inside stripe js; the thread whose block holds the target
    u64 w[kBlk] = {};
    const int blk = js * kThreads + tid;
    if ((js + 1) * kThreads * kBlk <= a.V) {  // (uniform) a whole stripe
      WholeBlock<Tin> qt, qd;
      qt.load(rt.p, blk);
      qd.load(rd.p, blk);
      float vt[kBlk], vd[kBlk];
      qt.values(vt);
      qd.values(vd);
      weights(vt, vd, kept_lanes(vt, 0xFFu, blk), blk, w, tab_mode);
    } else if (blk < rt.nblk) {
      float vt[kBlk], vd[kBlk];
      const uint32_t valid = rt.load(blk, vt) & rd.load(blk, vd);
      weights(vt, vd, kept_lanes(vt, valid, blk), blk, w, tab_mode);
    }
    u64 s = 0;
#pragma unroll
    for (int i = 0; i < kBlk; ++i) s += w[i];
    u64 tot;
    const u64 ex = block_excl_scan<u64>(s, red, &tot);
    if (s > 0 && base + ex <= tg && base + ex + s > tg) {
      // 4. this thread walks its eight lanes
      u64 c = base + ex;
      int tok = -1;
#pragma unroll
      for (int i = 0; i < kBlk; ++i) {
        c += w[i];
        if (tok < 0 && w[i] > 0 && c > tg) tok = blk * kBlk + i;
      }
      out[jr] = tok;
      a.out_count[b] = jr + 1;
    }
    return false;
  };
  if (kBf16 && tabled) return residual(std::integral_constant<bool, kBf16>{});
  return residual(std::false_type{});
}

// Target rows past one round on the CUs: the last launch's rows, the bonus rows of the accepted
// sequences (k_sample's row code, one workgroup a row) and the residual draws of the rejected ones,
// (row, slice) items row-major over their list, one item a workgroup: the grid is the larger of B and
// the CUs the items can use (the LDS holds one workgroup a CU), and the slices are chosen to fit it.
// (No loop over the items: with one the compiler kept both kinds' values live across it and spilled,
// 640 bytes a lane, 72-78 us.) The launch's SampleArgs describe the target rows, its out_ids the
// emitted tokens: row (b, j)'s draw is token (b, j).
struct VerifyRow {
  static constexpr bool kOwn = false;
  static constexpr bool kDraws = false;
  VerifyArgs a;
  // The target row this workgroup draws from: a bonus row, or a rejected one without residual mass
  // (after its residual); -1: none.
  template <class Tin>
  __device__ __forceinline__ int row(uint32_t* big, FastSmem& f) const {
    const int nrej = *a.nrej;
    const int nacc = a.B - nrej;
    const int item = blockIdx.x;
    if (item < nacc) return a.acc[item] * (a.K + 1) + a.K;
    const int slices = residual_slices(nrej, static_cast<int>(gridDim.x) - nacc, a.max_slices);
    const int q = item - nacc;
    if (q >= nrej * slices) return -1;
    const int b = a.rej[q / slices];
    const int jr = a.jr[b];
    __syncthreads();  // (publishes the exp table)
    if (!residual_item<Tin>(a, b, jr, q % slices, slices, big, *reinterpret_cast<ResidualSmem*>(&f))) return -1;  // (uniform)
    __syncthreads();  // (the residual's LDS is free)
    return b * (a.K + 1) + jr;
  }
};

// Target rows of one round: all in the first launch, each sequence's last (its bonus row) also drawn
// from, and the slice counters of the last launch cleared by its workgroup.
struct BonusDraws {
  static constexpr bool kOwn = false;
  static constexpr bool kDraws = true;
  int K1;  // K + 1
  uint32_t* done;
  template <class Tin>
  __device__ __forceinline__ int row(uint32_t*, FastSmem&) const {
    const int r = static_cast<int>(blockIdx.x);
    if (draws(r) && threadIdx.x == 0) done[r / K1] = 0;
    return r;
  }
  __device__ __forceinline__ bool draws(int r) const { return r % K1 == K1 - 1; }
};

// Then the launch after the states': the residuals' (row, slice) items, each workgroup working out for
// itself which is its own; an accepted sequence has its tokens already. (The lists of k_verify_accept
// would cost a launch of one workgroup, ~6 us, before this one.)
struct ResidualRow {
  static constexpr bool kOwn = false;
  static constexpr bool kDraws = false;
  VerifyArgs a;
  // Token i of sequence b, first rejected at j: but for token j, which is the bonus token, already
  // there, or the residual's.
  __device__ __forceinline__ void tokens(int b, int j) const {
    const int i = threadIdx.x;
    if (i <= a.K && i != j) a.out_tokens[static_cast<int64_t>(b) * (a.K + 1) + i] = i < j ? a.drafts[b * a.K + i] : -1;
    if (i == 0 && j == a.K) a.out_count[b] = a.K + 1;
  }
  // A target row without residual mass, to draw from (after its residual); -1: none.
  template <class Tin>
  __device__ __forceinline__ int row(uint32_t* big, FastSmem& f) const {
    const int K = a.K, B = a.B;
    const int tid = threadIdx.x;
    const int item = blockIdx.x;
    int b, jr, slice, slices = a.max_slices;  // (uniform)
    if (B * slices <= static_cast<int>(gridDim.x)) {
      // every sequence has all of its slices: only its own acceptance counts (a lane per draft, K <= 64)
      b = item / slices;
      slice = item % slices;
      const int l = static_cast<int>(lane_id());
      __syncthreads();  // (publishes the exp table)
      const u64 no = __ballot(l < K && !accepts<Tin>(a, b, l));
      jr = no ? __ffsll(static_cast<long long>(no)) - 1 : K;
      if (slice == 0) tokens(b, jr);
      if (jr == K) return -1;
    } else {
      // the whole batch's acceptance (a thread per draft, B K < kThreads), and the rejected rows split
      // as far as the grid goes
      int* const first = reinterpret_cast<int*>(big);  // [B] the first rejected position (K: none)
      int* const rej = first + kThreads;               // the rejected sequences, ascending
      if (tid < B) first[tid] = K;
      __syncthreads();  // (publishes the exp table too)
      if (tid < B * K && !accepts<Tin>(a, tid / K, tid % K)) atomicMin(&first[tid / K], tid % K);
      __syncthreads();
      const bool r = tid < B && first[tid] < K;
      uint32_t nrej;
      const uint32_t at = block_excl_scan<uint32_t>(r ? 1u : 0u, f.red32, &nrej);
      if (r) rej[at] = tid;
      if (item < B) tokens(item, first[item]);
      slices = residual_slices(static_cast<int>(nrej), static_cast<int>(gridDim.x), slices);
      if (item >= static_cast<int>(nrej) * slices) return -1;
      __syncthreads();
      b = __builtin_amdgcn_readfirstlane(rej[item / slices]);
      jr = __builtin_amdgcn_readfirstlane(first[b]);
      slice = item % slices;
      __syncthreads();  // (the residual's tables go over the lists)
    }
    if (!residual_item<Tin>(a, b, jr, slice, slices, big, *reinterpret_cast<ResidualSmem*>(&f))) return -1;  // (uniform)
    __syncthreads();  // (the residual's LDS is free)
    return b * (K + 1) + jr;
  }
};

}  // namespace vs
