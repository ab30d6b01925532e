// Attention launch planning and launchers; the kernels and their bodies are in attn_body.hpp.
#include "attn_body.hpp"
#include "prefill_form.hpp"

#include <algorithm>

namespace fdllm {

// The chunked kernel's workgroup: query tiles x 2 key parts, 2 query tiles for one sequence and 4 for a
// batched call.  A query's arithmetic does not depend on how many tiles share its workgroup, so the
// results are those of the 4-tile workgroups; with twice the workgroups more compute units take each
// chunk's keys (one sequence, 1.5B, prefix 2048, chunk + merge per layer: 13.0 -> 12.3 us at 32 rows).
// The chunk length is chosen on the 4-tile count for both, so that it, and with it every result, stays
// the same.  (4 key parts of 32 keys measured faster still, 11.9 us, but a key part's online softmax
// then runs over other blocks, which changes the rounding; batched calls on 2 tiles: 128-row partial
// step 2.73 against 2.54 ms.)

// the prefill kernel takes row blocks of at least this many rows without an explicit bias
constexpr int PREFILL_MIN_ROWS = 128;

// one sequence's unmasked call takes attn_seq_kernel below this many rows (us per layer over 8175 keys, the
// loop kernel up to 127 rows and the one-block prefill kernel from there / this one: 48 rows 69 / 19, 83
// rows 168 / 23, 127 rows 221 / 30, 300 rows 185 / 60, 600 rows 193 / 100; over 256 keys 12.5 / 9.9, 16.4 /
// 10.9, 19.6 / 11.3, 20.2 / 17.6, 27.4 / 17.7)
constexpr int SEQ_ONE_MAX_ROWS = 1024;

// attn_seq_kernel: key blocks ahead, waves (key parts) per query tile and query tiles per workgroup.
constexpr int SEQ_DEPTH = 3;
#ifndef FD_SEQ_KH
#define FD_SEQ_KH 2
#endif
#ifndef FD_SEQ_NQW
#define FD_SEQ_NQW 2
#endif
constexpr int SEQ_KH = FD_SEQ_KH, SEQ_NQW = FD_SEQ_NQW;

// One sequence on attn_seq_kernel: S key splits (merged by attn_merge_kernel), and its qg query-tile
// groups dealt to the XCDs in xh runs.  A unit is one run of one (split, kv head): its workgroups share
// the split's K/V through one XCD's L2, so whole units go to an XCD and an XCD with more units than the
// others sets the time (64 rows over 8100 keys: 10 splits in one run each 31.6 us, 8 splits 21.1).  The
// choice is the cheapest of, per xh, no split and as many splits as one workgroup per compute unit
// allows, at the measured 1 us per 64-key block, 3 us per round of workgroups, 4.5 us for the merge launch
// and 4.2 ns per partial tile written and read back.
constexpr int SEQ_ONE_MAX_SPLITS = 40, SEQ_ONE_MAX_RUNS = 8;
static void seq_one_splits(AttnPlan& p, int QT, int nkv, int Lk, int ncu) {
  const int T = (Lk + 63) / 64, per_xcd = std::max(1, ncu / 8);
  float best = 0.f;
  p.S = p.xh = 0;
  for (int xh = 1; xh <= SEQ_ONE_MAX_RUNS; ++xh) {
    const int wgs = (p.qg + xh - 1) / xh;  // of one unit
    for (const int S : {1, std::min({per_xcd / wgs * 8 / (nkv * xh), T / 2, SEQ_ONE_MAX_SPLITS})}) {
      if (S < 1) continue;
      const int rounds = ((S * nkv * xh + 7) / 8 * wgs + per_xcd - 1) / per_xcd;
      const float cost = (float)(rounds * ((T + S - 1) / S + 3)) + (S > 1 ? 4.5f + 0.0042f * (float)(S * QT * nkv) : 0.f);
      if (p.S == 0 || cost < best) {
        best = cost;
        p.S = S;
        p.xh = xh;
      }
    }
  }
}

// Launch plan: short row blocks (the cached decode step) use attn_chunk_kernel with one key chunk of
// CH keys per workgroup; one sequence's longer unmasked calls attn_seq_kernel in key splits (p.seq); the
// others attn_kernel with few, long key ranges per workgroup, or (launch_dt) attn_prefill_kernel.
AttnPlan attn_plan(int rows, int nq, int nkv, int Lk, int target_wgs, int nseq, int mask, int ncu) {
  AttnPlan p{};
  const int QT = ((nq / nkv) * rows + 15) / 16;
  const bool seq = nseq <= 1 && mask == 0 && ncu > 0 && rows < SEQ_ONE_MAX_ROWS;
  // chunked: 128 keys per workgroup unless that leaves fewer workgroups than aimed for; at most 64
  // chunks, so the split merge stays small (longer contexts take the loop kernel), and at most 40 where
  // attn_seq_kernel can take the call: past the splits its merge reads in one round trip the chunk kernel
  // falls behind (rotated queries, 32 rows: 18.1 / 18.5 us at 4096 keys, 29.0 / 20.0 at 6000, 33.0 / 22.8
  // at 8100; 8 rows: 13.6 / 12.9, 19.3 / 13.4, 22.8 / 14.3; the RoPE and append pass of a step adds 4.5 us)
  if (QT <= 12 && (Lk + 127) / 128 <= (seq ? 40 : 64)) {
    p.chunked = 1;
    p.key_groups = 2;
    p.chunk = 128;
    if ((QT + 3) / 4 * nkv * ((Lk + 127) / 128) < target_wgs && (Lk + 63) / 64 <= 64) p.chunk = 64;
    p.q_tiles_per_wg = nseq > 1 ? 4 : 2;
    p.qg = (QT + p.q_tiles_per_wg - 1) / p.q_tiles_per_wg;
    p.S = (Lk + p.chunk - 1) / p.chunk;
    return p;
  }
  p.chunked = 0;
  if (seq) {
    p.seq = 1;
    p.q_tiles_per_wg = SEQ_NQW;
    p.key_groups = SEQ_KH;
    p.qg = (QT + SEQ_NQW - 1) / SEQ_NQW;
    p.chunk = 64;
    seq_one_splits(p, QT, nkv, Lk, ncu);
    return p;
  }
  if (QT >= 32) { p.q_tiles_per_wg = 4; p.key_groups = 1; }
  else { p.q_tiles_per_wg = 4; p.key_groups = 2; }
  p.qg = (QT + p.q_tiles_per_wg - 1) / p.q_tiles_per_wg;
  const int base = p.qg * nkv;
  const int max_splits = std::max(1, (Lk + 32 * p.key_groups - 1) / (32 * p.key_groups));
  int S = std::min(max_splits, std::max(1, (target_wgs + base - 1) / base));
  p.chunk = (((Lk + S - 1) / S) + 31) / 32 * 32;
  p.S = (Lk + p.chunk - 1) / p.chunk;
  return p;
}

size_t attn_partial_floats(const AttnP& a) {
  const int QT = ((a.nq / a.nkv) * a.rows + 15) / 16;
  return (size_t)std::max(a.nseq, 1) * a.nkv * QT * a.S * PSZ;
}

// the merge kernel whose register path covers S splits in one round trip where it can
template <int DT>
static auto merge_kernel_for(int S) {
  return S > 24 ? attn_merge_kernel<DT, 40> : attn_merge_kernel<DT, 24>;
}

template <typename K>
static void raise_lds(K kern, size_t lds) {
  // a runtime that needs no attribute for LDS up to the device limit may reject it: clear that error
  // and let the launch report whether the size fits
  if (lds > 64 * 1024 &&
      hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) !=
          hipSuccess)
    (void)hipGetLastError();
}

template <int DT, int QPW, int KSW>
static hipError_t launch_loop(const AttnP& a, const AttnPlan& p, hipStream_t st) {
  const size_t loop_lds = (size_t)KSW * (KB * KLD + HD * VLD) * 2;
  const size_t merge_lds = (size_t)2 * KSW * QPW * 16 * 4 + (size_t)(KSW - 1) * QPW * (HD / 16) * 64 * 16;
  const size_t lds = std::max(loop_lds, merge_lds);
  if (lds > 160 * 1024) return hipErrorInvalidValue;
  auto kern = attn_kernel<DT, QPW, KSW>;
  raise_lds(kern, lds);
  hipLaunchKernelGGL(kern, dim3(p.qg, a.nkv, a.S), dim3(64 * QPW * KSW), lds, st, a);
  if (a.S > 1) {
    const int QT = ((a.nq / a.nkv) * a.rows + 15) / 16;
    hipLaunchKernelGGL(merge_kernel_for<DT>(a.S), dim3(HD / 16, QT, a.nkv), dim3(64), 0, st, a);
  }
  return hipGetLastError();
}

template <int DT, int CH, int KH, int MASK, int QPW, bool WIN = false>
static hipError_t launch_chunk_kh(const AttnP& a, const AttnPlan& p, hipStream_t st) {
  // K and V^T of the chunk, then (one-sequence calls) the queries the first key part shares
  const size_t loop_lds = (size_t)CH * KLD * 2 + (size_t)HD * (CH + 8) * 2 +
                          (KH > 1 && a.nseq <= 1 ? (size_t)QPW * 4 * 64 * 16 : 0);
  const size_t merge_lds = (size_t)2 * KH * QPW * 16 * 4 + (size_t)(KH - 1) * QPW * (HD / 16) * 64 * 16;
  const size_t lds = std::max(loop_lds, merge_lds);
  if (lds > 160 * 1024) return hipErrorInvalidValue;
  const int nseq = std::max(a.nseq, 1);
  auto kern = attn_chunk_kernel<DT, QPW, KH, CH, MASK, WIN>;
  raise_lds(kern, lds);
  if (nseq == 1)
    hipLaunchKernelGGL(kern, dim3(attn_chunk_grid_1seq(p.qg, a.nkv, a.S)), dim3(64 * QPW * KH), lds, st, a);
  else
    hipLaunchKernelGGL(kern, dim3(p.qg * nseq, a.nkv, a.S), dim3(64 * QPW * KH), lds, st, a);
  if (a.S > 1) {
    const int QT = ((a.nq / a.nkv) * a.rows + 15) / 16;
    hipLaunchKernelGGL(merge_kernel_for<DT>(a.S), dim3(HD / 16, QT, a.nkv * nseq), dim3(64), 0, st, a);
  }
  return hipGetLastError();
}

// attn_plan's workgroup shape: 2 (one sequence) or 4 (batched) query tiles x 2 key parts
template <int DT, int CH, int MASK>
static hipError_t launch_chunk_shape(const AttnP& a, const AttnPlan& p, hipStream_t st) {
  if (p.key_groups != 2) return hipErrorInvalidValue;
  if (a.kwin != nullptr) {
    if constexpr (MASK == 0) {
      if (p.q_tiles_per_wg == 2 && a.rope == nullptr) return launch_chunk_kh<DT, CH, 2, 0, 2, true>(a, p, st);
    }
    return hipErrorInvalidValue;
  }
  if (p.q_tiles_per_wg == 2) return launch_chunk_kh<DT, CH, 2, MASK, 2>(a, p, st);
  if (p.q_tiles_per_wg == 4) return launch_chunk_kh<DT, CH, 2, MASK, 4>(a, p, st);
  return hipErrorInvalidValue;
}
template <int DT, int CH>
static hipError_t launch_chunk_mask(const AttnP& a, const AttnPlan& p, hipStream_t st) {
  switch (a.mask) {
    case 0: return launch_chunk_shape<DT, CH, 0>(a, p, st);
    case 1: return launch_chunk_shape<DT, CH, 1>(a, p, st);
    default: return launch_chunk_shape<DT, CH, 2>(a, p, st);
  }
}

// Long row blocks: the RoPE + KV append pass (unless qkv's epilogue did it), then attn_prefill_kernel in the form of
// prefill_form.hpp (TQ = 3: all of a kv head's twelve tiles per workgroup).
template <int DT, int MASK, int TQ>
static hipError_t launch_prefill_cfg(const AttnP& a, int paired, hipStream_t st) {
  auto kern = attn_prefill_kernel<DT, MASK, TQ>;
  constexpr size_t lds = (size_t)2 * 2 * 128 * HD * 2;  // K and V of two stages of 128 keys
  raise_lds(kern, lds);
  const int nqb = (a.rows + 31) / 32, tiles = 2 * (a.nq / a.nkv);
  hipLaunchKernelGGL(kern, dim3(paired ? (nqb + 1) / 2 : nqb, a.nkv, (tiles + 4 * TQ - 1) / (4 * TQ)), dim3(512), lds, st,
                     a, paired);
  return hipGetLastError();
}

template <int DT, int MASK>
static hipError_t launch_prefill(const AttnP& a, hipStream_t st) {
  if (!a.roped) hipLaunchKernelGGL(rope_kv_kernel<DT>, dim3(a.rows), dim3(128), 0, st, a);
  const PrefillForm f = prefill_form(a.rows, a.nq, a.nkv, a.cus, a.prefill_pair, a.prefill_hpw);
  return f.whole ? launch_prefill_cfg<DT, MASK, 3>(a, f.paired, st) : launch_prefill_cfg<DT, MASK, 1>(a, f.paired, st);
}

// Batched calls without a mask: the RoPE + KV append pass over the call's rows, then attn_seq_kernel.
size_t plan_seq_units(AttnP& a, int ncu) {
  const int QT = ((a.nq / a.nkv) * a.rows + 15) / 16, xg = (QT + SEQ_NQW - 1) / SEQ_NQW;
  int T[MAX_SEQS], s[MAX_SEQS];
  for (int b = 0; b < a.nseq; ++b) {
    T[b] = std::max(1, (a.seq_lk[b] + 63) / 64);
    s[b] = 1;
  }
  int units = a.nseq;
  const bool cnt_ok = a.seq_cnt != nullptr && (size_t)a.nseq * a.nkv * xg * SEQ_NQW <= (size_t)SEQ_CNT_MAX;
  const int cap = cnt_ok && ncu > 0 ? std::min(MAX_SEQ_UNITS, std::max(a.nseq, ncu / (a.nkv * xg))) : a.nseq;
  while (units < cap) {
    int best = 0, bl = 0;
    for (int b = 0; b < a.nseq; ++b) {
      const int l = (T[b] + s[b] - 1) / s[b];
      if (l > bl) { bl = l; best = b; }
    }
    if (bl <= 2 || s[best] >= 16) break;
    ++s[best];
    ++units;
  }
  // sequence-major units (u0 + j indexes the partials), launched longest first: units past what one
  // round of workgroups holds wait for the first to finish, and the shortest wait at least cost
  int ua[MAX_SEQ_UNITS], ut[MAX_SEQ_UNITS], ord[MAX_SEQ_UNITS];
  int u = 0;
  for (int b = 0; b < a.nseq; ++b)
    for (int j = 0; j < s[b]; ++j, ++u) {
      ua[u] = b | (j << 6) | (s[b] << 11) | ((u - j) << 16);
      ut[u] = (T[b] * j / s[b]) | ((T[b] * (j + 1) / s[b]) << 16);
      ord[u] = u;
    }
  auto len = [&](int v) { return (ut[v] >> 16) - (ut[v] & 0xffff); };
  std::stable_sort(ord, ord + u, [&](int x, int y) { return len(x) > len(y); });
  for (int v = 0; v < u; ++v) {
    a.unit_a[v] = ua[ord[v]];
    a.unit_t[v] = ut[ord[v]];
  }
  a.nunits = u;
  return units > a.nseq ? (size_t)u * a.nkv * xg * SEQ_NQW * PSZ : 0;
}

template <int DT>
static hipError_t launch_seq(const AttnP& a, hipStream_t st) {
  const bool one = a.nseq <= 1;
  if (one ? a.S < 1 || a.S > (a.Lk + 63) / 64 : a.nunits < a.nseq || a.nunits > MAX_SEQ_UNITS) return hipErrorInvalidValue;
  if (!a.roped) hipLaunchKernelGGL(rope_kv_kernel<DT>, dim3((one ? 1 : a.nseq) * a.rows), dim3(128), 0, st, a);
  const int QT = ((a.nq / a.nkv) * a.rows + 15) / 16, xg = (QT + SEQ_NQW - 1) / SEQ_NQW;
  const int xh = one ? a.xh : 1, xs = (xg + xh - 1) / xh;
  if (xh < 1) return hipErrorInvalidValue;
  const int units = (one ? a.S : a.nunits) * a.nkv * xh;
  auto kern = attn_seq_kernel<DT, SEQ_DEPTH, SEQ_NQW, SEQ_KH>;
  constexpr size_t lds = (size_t)(SEQ_DEPTH + 1) * 2 * 64 * HD * 2;  // K and V of D + 1 key blocks
  raise_lds(kern, lds);
  hipLaunchKernelGGL(kern, dim3((units + 7) / 8 * 8 * xs), dim3(64 * SEQ_NQW * SEQ_KH), lds, st, a);
  if (one && a.S > 1) hipLaunchKernelGGL(merge_kernel_for<DT>(a.S), dim3(HD / 16, QT, a.nkv), dim3(64), 0, st, a);
  return hipGetLastError();
}

bool attn_takes_roped(const AttnP& a) {
  if (a.nseq > 1 && a.seq_attn && a.mask == 0) return true;
  if (a.nseq <= 1 && a.seq_attn) return true;
  const AttnPlan p = attn_plan(a.rows, a.nq, a.nkv, a.Lk, a.target_wgs, a.nseq, a.mask, a.ncu);
  return !p.chunked && a.nseq <= 1 && a.rows >= PREFILL_MIN_ROWS && a.mask != 2;
}

template <int DT>
static hipError_t launch_dt(const AttnP& a, hipStream_t st) {
  if (a.nseq <= 1 && a.seq_attn) {
    if (a.mask != 0 || (a.ofrag && a.rows > 32)) return hipErrorInvalidValue;
    return launch_seq<DT>(a, st);
  }
  const AttnPlan p = attn_plan(a.rows, a.nq, a.nkv, a.Lk, a.target_wgs, a.nseq, a.mask, a.ncu);
  if (p.seq || (a.roped && !attn_takes_roped(a)) || (a.kwin != nullptr && !p.chunked)) return hipErrorInvalidValue;
  if (p.S != a.S || p.chunk != a.chunk) return hipErrorInvalidValue;
  if (a.ofrag && (a.nseq > 1 || a.rows > 32)) return hipErrorInvalidValue;
  if (a.nseq > MAX_SEQS) return hipErrorInvalidValue;
  if (a.nseq > 1 && a.seq_attn && a.mask == 0) return launch_seq<DT>(a, st);
  if (a.nseq > 1 && !p.chunked) return hipErrorInvalidValue;
  if (!p.chunked && a.nseq <= 1 && a.rows >= PREFILL_MIN_ROWS && a.mask != 2) {
    if (a.mask == 1) return launch_prefill<DT, 1>(a, st);
    return launch_prefill<DT, 0>(a, st);
  }
  if (p.chunked) {
    if (p.chunk == 128) return launch_chunk_mask<DT, 128>(a, p, st);
    return launch_chunk_mask<DT, 64>(a, p, st);
  }
  if (p.key_groups == 1) return launch_loop<DT, 4, 1>(a, p, st);
  return launch_loop<DT, 4, 2>(a, p, st);
}

bool attn_takes_window(const AttnP& a) {
  return a.nseq <= 1 && !a.seq_attn &&
         attn_plan(a.rows, a.nq, a.nkv, a.Lk, a.target_wgs, a.nseq, a.mask, a.ncu).chunked;
}

hipError_t launch_rope_kv(int dt, const AttnP& a, hipStream_t st) {
  if (a.nseq > 1 || a.rope == nullptr) return hipErrorInvalidValue;
  if (dt == DT_BF16) hipLaunchKernelGGL(rope_kv_kernel<DT_BF16>, dim3(a.rows), dim3(128), 0, st, a);
  else hipLaunchKernelGGL(rope_kv_kernel<DT_F16>, dim3(a.rows), dim3(128), 0, st, a);
  return hipGetLastError();
}

hipError_t launch_attention(int dt, const AttnP& a, hipStream_t st) {
  if (dt == DT_BF16) return launch_dt<DT_BF16>(a, st);
  return launch_dt<DT_F16>(a, st);
}

}  // namespace fdllm
