// The final probabilities of a batch in two launches: k_sample with row states (one workgroup per
// row finds the row's kept set and normaliser, and leaves its penalised ids and values in the
// workspace), then k_probs_write, which spreads the rows' [V] outputs over the whole chip.
//
// Why: a row's outputs are 4 V bytes beside 2-4 V bytes of logits, and one workgroup per row
// keeps all but B CUs idle while it writes them, one fp64 exponential per kept token on one CU's
// SIMDs. 32 bf16 rows of 151936 with top-p 0.95 (29 MB in and out): 104.8 us a call in one launch,
// 32.3 in two, ~23 of it the states' launch (a row's pass and decisions on one CU).
#pragma once

#include "sample.cuh"

namespace vs {

constexpr int kPwThreads = 256;
typedef float f32x4_any_t __attribute__((ext_vector_type(4), aligned(4)));  // (16-byte stores at any fp32 address)
constexpr int kPwTile = kPwThreads * kBlk;  // ids per workgroup

// Grid (ceil(V / kPwTile), B): workgroup (t, r) writes ids kPwTile t .. of row r, a token's
// probability as the one-launch form computes it (the same expressions, so the same bits). Thread
// i takes eight consecutive ids (16-byte loads and stores); in the row's last, partial tile, ids
// i + 256 k (element by element, eight loads in flight). With PEN the tile's penalised
// ids are written again from the row's list, after the workgroup's own bulk stores.
template <class Tin, bool PEN>
__global__ __launch_bounds__(kPwThreads) void k_probs_write(const Tin* logits, int64_t stride, int V, const RowState* state,
                                                            float* out_, int64_t out_stride, Workspace ws_,
                                                            const int32_t* off_, int hstep) {
  exp_table_init();
  const int r = blockIdx.y;
  const int tid = threadIdx.x;
  const Tin* row = as_global(logits) + static_cast<int64_t>(r) * stride;
  float* o = as_global(out_) + static_cast<int64_t>(r) * out_stride;
  const RowState st = as_global(state)[r];
  const int i0 = static_cast<int>(blockIdx.x) * kPwTile;
  const int end = min(V, i0 + kPwTile);
  Kept kept;
  kept.x0 = st.x0;
  kept.vc = st.vc;
  kept.partial = st.partial != 0;
  kept.idr = st.idr;
  const double inv = kMassScale / static_cast<double>(st.S);
  auto prob = [&](float x, int id) -> float {
    if (st.point >= 0) return id == st.point ? 1.0f : 0.0f;
    return kept.keep(x, id) ? static_cast<float>(ptilde(x, st.T, st.mz) * inv) : 0.0f;
  };
  const int b0 = i0 + kBlk * tid;
  float v[kBlk];
  const bool whole = i0 + kPwTile <= V;  // (uniform)
  if (whole) {
    WholeBlock<Tin> q;
    q.load(row, b0 / kBlk);
    q.values(v);
  } else {
#pragma unroll
    for (int e = 0; e < kBlk; ++e) {
      const int i = i0 + tid + e * kPwThreads;
      v[e] = load_one<Tin>(row, min(i, V - 1));
    }
  }
  __syncthreads();  // (the exp table)
  if (whole) {
    f32x4_any_t a, b;
    a.x = prob(v[0], b0);
    a.y = prob(v[1], b0 + 1);
    a.z = prob(v[2], b0 + 2);
    a.w = prob(v[3], b0 + 3);
    b.x = prob(v[4], b0 + 4);
    b.y = prob(v[5], b0 + 5);
    b.z = prob(v[6], b0 + 6);
    b.w = prob(v[7], b0 + 7);
    *reinterpret_cast<f32x4_any_t*>(o + b0) = a;
    *reinterpret_cast<f32x4_any_t*>(o + b0 + 4) = b;
  } else {
#pragma unroll
    for (int e = 0; e < kBlk; ++e) {
      const int i = i0 + tid + e * kPwThreads;
      if (i < end) o[i] = prob(v[e], i);
    }
  }
  if constexpr (PEN) {
    const Workspace ws = globalized(ws_);
    const int h0 = as_global(off_)[r * hstep];
    const int n = static_cast<int>(ws.n_exc[r]);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();  // (every bulk store of the tile is done)
    constexpr int kU = 8;  // (ids in flight per thread; every load is issued, clamped into the list)
    for (int e0 = tid; e0 < n; e0 += kU * kPwThreads) {
      int id[kU];
#pragma unroll
      for (int k = 0; k < kU; ++k) id[k] = ws.exc_id[h0 + min(e0 + k * kPwThreads, n - 1)];
#pragma unroll
      for (int k = 0; k < kU; ++k) {
        const int e = e0 + k * kPwThreads;
        if (e < n && id[k] >= i0 && id[k] < end) o[id[k]] = prob(ws.exc_val[h0 + e], id[k]);
      }
    }
  }
}

}  // namespace vs
