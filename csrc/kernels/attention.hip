// Causal attention over the shard-local KV cache.
//
// K7 of SURVEY.md §2.5 (`[tf5.15] modeling_gpt2.py:201-220`, SDPA causal):
//   softmax(Q K^T / sqrt(hd) + causal) V.  The reference recomputes attention
// over the whole sequence every step and gets causality only implicitly
// (quirk Q3); here the mask is explicit and K/V come from the cache.
//
// Cache layout [slot][kv_head][position][hd] (bf16): one (slot, head) is a
// contiguous run of positions, so every key/value row read is part of one
// linear stream.
//
// attn_decode : one query per sequence (decode).  Memory-bound flash-decoding:
//   block = (sequence, kv head[, key split]); 4 waves stride over the keys; a
//   key row (hd*2 bytes) is read by hd/8 lanes with 16-byte loads, so each
//   wave-instruction streams 1 KiB of contiguous K (then V).  GQA: the G query
//   heads sharing a kv head are served from the same K/V loads.  Online
//   softmax in exp2 domain; waves/splits merged with (m, l) rescaling.
// attn_prefill: packed ragged queries (prefill / chunked prefill).  MFMA
//   16x16x32 bf16 with SWAPPED operands: S^T = K . Q^T puts one query per lane
//   (column) so the row max/sum are lane-local plus a 2-step exchange, and the
//   S^T accumulator registers ARE the P^T B-operand of the PV MFMA (no LDS
//   round trip for P).  V^T fragments come from the row-major V tile via the
//   gfx950 hardware transpose read ds_read_b64_tr_b16.
#include "common.h"

namespace lsd {

constexpr float NEG = -1e30f;

// K/V rows of the decode step are streamed once per layer per step: load them
// non-temporal so they do not evict the weights the other microbatch lane is
// about to re-read from the Infinity Cache (bench A/B, tools/gpu_ab_flags.sh:
// 31.8k -> 32.6k tok/s GPT-2 XL; -DLSD_KV_TEMPORAL restores default policy)
#ifdef LSD_KV_TEMPORAL
#define LSD_KV_LOAD ld8
#else
#define LSD_KV_LOAD ld8_nt
#endif

// One step of a sum over lanes that lie OFF apart, of the first N of V values: the upper lanes go on with the
// upper half of them, the lower ones with the lower half (N = 1: both).  idx: the first value a lane has.
template <int OFF, int N, int V>
__device__ __forceinline__ void fold_step(float (&v)[V], int& idx, int lane) {
  if constexpr (N == 1) {
    v[0] += wave_xor_n(v[0], OFF);
  } else {
    constexpr int h = N / 2;
    const bool up = (lane & OFF) != 0;
#pragma unroll
    for (int i = 0; i < h; ++i) {
      const float send = up ? v[i] : v[i + h], keep = up ? v[i + h] : v[i];
      v[i] = keep + wave_xor_n(send, OFF);
    }
    if (up) idx += h;
  }
}

// NWV waves per block, U keys per lane group in flight.  Full batches: 4 waves, 4 keys, V behind the
// scores (fewer live registers, and the other blocks on the CU hide the latency; V with K costs two lanes of
// 256 sequences 1.5 %).  Small ones (fewer (sequence, head) items than CUs): 8 keys or more than 4 waves, an
// item's K and V requested in one round of loads instead of a chain of dependent ones.
// There a launch is its chain: position, K and V, scores, merges.  The merges are kept short: a wave scales its
// sums once by its own maximum and folds them over its key groups, each lane going on with half of its columns
// (7 exchanges for 8 columns, 24 when every lane merges all of them pair by pair), and a thread for two columns
// merges the waves.  12 heads of 64, one sequence of 204 keys 4.7 -> 4.0 us, on 4 waves of 8 keys for 8 of 4 3.7.
template <int HD, int G, int U, int NWV>
__global__ __launch_bounds__(NWV * 64) void attn_decode_kernel(
    const bf16* __restrict__ q, long ldq, const bf16* __restrict__ kc,
    const bf16* __restrict__ vc, const int* __restrict__ seq_slots,
    const int* __restrict__ qpos, bf16* out, long ldo, float* part_o, float* part_ml, int n_kv,
    int max_seq, int splits, float scale_log2, int n_items) {
  constexpr int LPK = HD / 8;    // lanes per key row
  constexpr int KPI = 64 / LPK;  // keys per wave-instruction
  constexpr bool ROUND = NWV > 4 || U > 4;  // V with K
  __shared__ float sm_o[NWV][G][HD];
  __shared__ float sm_ml[NWV][G][2];
  // work item = (sequence, kv head); a capped grid (lsd_attn_set_max_wg) loops
  // over items so the kernel occupies only part of the chip and a concurrent
  // lane's GEMMs keep the rest
  for (int item = blockIdx.x; item < n_items; item += gridDim.x) {
    const int b = item / n_kv, kvh = item % n_kv, split = blockIdx.y;
    const int lane = lane_id(), w = threadIdx.x >> 6;
    const int ds = lane % LPK, kg = lane / LPK;
    const int ctx = qpos[b] + 1;
    const int per = (ctx + splits - 1) / splits;
    const int k_lo = split * per, k_hi = min(ctx, k_lo + per);
    const long base = ((long)seq_slots[b] * n_kv + kvh) * (long)max_seq * HD + ds * 8;

    float qf[G][8];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      bf16x8 qq = ld8(q + (long)b * ldq + (long)(kvh * G + g) * HD + ds * 8);
#pragma unroll
      for (int j = 0; j < 8; ++j) qf[g][j] = bf2f(qq[j]) * scale_log2;
    }
    float m[G], l[G], o[G][8];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      m[g] = NEG;
      l[g] = 0.f;
#pragma unroll
      for (int j = 0; j < 8; ++j) o[g][j] = 0.f;
    }

    for (int c0 = k_lo + w * KPI; c0 < k_hi; c0 += NWV * KPI * U) {
      bf16x8 kv[U], vv[U];
      int key[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        key[u] = c0 + u * NWV * KPI + kg;
        const int kk = min(key[u], k_hi - 1);
        kv[u] = LSD_KV_LOAD(kc + base + (long)kk * HD);
      }
      if constexpr (ROUND) {
#pragma unroll
        for (int u = 0; u < U; ++u) vv[u] = LSD_KV_LOAD(vc + base + (long)min(key[u], k_hi - 1) * HD);
      }
      float s[G][U];
#pragma unroll
      for (int g = 0; g < G; ++g)
#pragma unroll
        for (int u = 0; u < U; ++u) {
          float acc = 0.f;
#pragma unroll
          for (int j = 0; j < 8; ++j) acc += qf[g][j] * bf2f(kv[u][j]);
#pragma unroll
          for (int msk = 1; msk < LPK; msk <<= 1) acc += wave_xchg_n(acc, msk);
          s[g][u] = key[u] < k_hi ? acc : NEG;
        }
      if constexpr (!ROUND) {
#pragma unroll
        for (int u = 0; u < U; ++u) vv[u] = LSD_KV_LOAD(vc + base + (long)min(key[u], k_hi - 1) * HD);
      }
#pragma unroll
      for (int g = 0; g < G; ++g) {
        float mx = s[g][0];
#pragma unroll
        for (int u = 1; u < U; ++u) mx = fmaxf(mx, s[g][u]);
        const float mn = fmaxf(m[g], mx);
        const float alpha = exp2f(m[g] - mn);
        float p[U], ps = 0.f;
#pragma unroll
        for (int u = 0; u < U; ++u) {
          p[u] = exp2f(s[g][u] - mn);
          ps += p[u];
        }
        l[g] = l[g] * alpha + ps;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          float a = o[g][j] * alpha;
#pragma unroll
          for (int u = 0; u < U; ++u) a += p[u] * bf2f(vv[u][j]);
          o[g][j] = a;
        }
        m[g] = mn;
      }
    }

    // merge the key groups of this wave (lanes with equal ds: exact xor partners)
#pragma unroll
    for (int g = 0; g < G; ++g) {
      float mw = m[g];
#pragma unroll
      for (int msk = LPK; msk < 64; msk <<= 1) mw = fmaxf(mw, wave_xor_n(mw, msk));
      const float f = exp2f(m[g] - mw);
      float lw = l[g] * f;
#pragma unroll
      for (int msk = LPK; msk < 64; msk <<= 1) lw += wave_xor_n(lw, msk);
      float v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = o[g][j] * f;
      int idx = 0;
      fold_step<32, 8>(v, idx, lane);
      fold_step<16, 4>(v, idx, lane);
      if constexpr (LPK == 8) {
        fold_step<8, 2>(v, idx, lane);
        sm_o[w][g][ds * 8 + idx] = v[0];
      } else {
        *reinterpret_cast<f32x2*>(&sm_o[w][g][ds * 8 + idx]) = f32x2{v[0], v[1]};
      }
      if (lane == 0) {
        sm_ml[w][g][0] = mw;
        sm_ml[w][g][1] = lw;
      }
    }
    __syncthreads();
    // merge the waves: two columns of a head a thread
    for (int t = threadIdx.x; t < G * (HD / 2); t += NWV * 64) {
      const int g = t / (HD / 2), d = t % (HD / 2) * 2;
      float mv[NWV], mm = NEG;
#pragma unroll
      for (int ww = 0; ww < NWV; ++ww) mm = fmaxf(mm, mv[ww] = sm_ml[ww][g][0]);
      float ll = 0.f, a = 0.f, c = 0.f;
#pragma unroll
      for (int ww = 0; ww < NWV; ++ww) {
        const float f = exp2f(mv[ww] - mm);
        const f32x2 x = *reinterpret_cast<const f32x2*>(&sm_o[ww][g][d]);
        ll += sm_ml[ww][g][1] * f;
        a += x[0] * f;
        c += x[1] * f;
      }
      const int h = kvh * G + g;
      if (splits == 1) {
        const float inv = ll > 0.f ? 1.f / ll : 0.f;
        *reinterpret_cast<bf16x2*>(out + (long)b * ldo + (long)h * HD + d) = pack2(a * inv, c * inv);
      } else {
        const int nh = n_kv * G;
        const long pi = ((long)b * nh + h) * splits + split;
        *reinterpret_cast<f32x2*>(part_o + pi * HD + d) = f32x2{a, c};
        if (d == 0) {
          part_ml[pi * 2] = mm;
          part_ml[pi * 2 + 1] = ll;
        }
      }
    }
    __syncthreads();  // sm_o is reused by this block's next item
  }
}

// Decode attention FUSED with the attention output projection and its
// residual add, for small batches (single stream: B <= 4 rows).  At batch 1
// a GPT-2 XL layer's attention (5.7 us) and out-projection GEMV (4.8 us, a
// 5 MB weight read at 1.1 TB/s) are both latency-bound launches
// (profiles/r2_single_stream_analysis.log); here one launch does both:
//   block (kv head h, column chunk c): attention of every sequence for the G
//   query heads of kv head h (the decode kernel's loop, K and V requested in
//   one round; recomputed by each of the C chunk blocks of h -- L2-served
//   re-reads of a few tens of KB), kept in fp32 in LDS; then the partial
//   out-projection  part[c][h][b][n] = sum_{k in head h's slice} o[b][k] W[n][k]
//   for the chunk's NC output columns (W's [N][nh*HD] rows: the slice is
//   G*HD contiguous bf16 per column).
// The n_kv partials of a column chunk are summed by the chunk's LAST-arriving
// block in kv-head order (deterministic), plus the bias, into the fp32
// residual x.  Hand-off (guide §6 Guideline 16 / MI355X_MICROARCH hand-off
// table row 1): write-through (sc1, relaxed agent-scope) partial stores ->
// every wave's vmcnt(0) -> barrier -> one lane's agent-scope ticket add; the
// block whose add returns n_kv - 1 reads the partials with sc1 loads.
template <int HD, int G, int NWV, int BMAX>
__global__ __launch_bounds__(NWV * 64) void attn_oproj_kernel(
    const bf16* __restrict__ q, long ldq, const bf16* __restrict__ kc, const bf16* __restrict__ vc,
    const int* __restrict__ seq_slots, const int* __restrict__ qpos, int B, int n_kv, int max_seq,
    float scale_log2, const bf16* __restrict__ W, long ldw, const bf16* __restrict__ bias, float* x,
    int N, int NC, float* part, int* cnt) {
  constexpr int LPK = HD / 8;    // lanes per key row
  constexpr int KPI = 64 / LPK;  // keys per wave-instruction
  constexpr int U = 2;
  constexpr int KS = G * HD;     // this kv head's slice of the out-projection's K
  constexpr int LPC = KS / 8 <= 64 ? KS / 8 : 64;  // lanes per output column
  constexpr int R = KS / (8 * LPC);                 // 16-B pieces of W per lane
  constexpr int CPI = 64 / LPC;                     // columns per wave-instruction
  static_assert(64 % LPC == 0 && R * 8 * LPC == KS, "out-projection slice per lane");
  __shared__ float sm[NWV][G][LPK][10];
  __shared__ float so[BMAX][KS];
  __shared__ int s_flag;
  const int kvh = blockIdx.x, c = blockIdx.y;
  const int lane = lane_id(), w = threadIdx.x >> 6;
  const int ds = lane % LPK, kg = lane / LPK;

  for (int b = 0; b < B; ++b) {
    const int ctx = qpos[b] + 1;
    const long base = ((long)seq_slots[b] * n_kv + kvh) * (long)max_seq * HD + ds * 8;
    float qf[G][8];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const bf16x8 qq = ld8(q + (long)b * ldq + (long)(kvh * G + g) * HD + ds * 8);
#pragma unroll
      for (int j = 0; j < 8; ++j) qf[g][j] = bf2f(qq[j]) * scale_log2;
    }
    float m[G], l[G], o[G][8];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      m[g] = NEG;
      l[g] = 0.f;
#pragma unroll
      for (int j = 0; j < 8; ++j) o[g][j] = 0.f;
    }
    for (int c0 = w * KPI; c0 < ctx; c0 += NWV * KPI * U) {
      bf16x8 kv[U], vv[U];
      int key[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {  // K and V of the round requested together
        key[u] = c0 + u * NWV * KPI + kg;
        const int kk = min(key[u], ctx - 1);
        kv[u] = ld8(kc + base + (long)kk * HD);
        vv[u] = ld8(vc + base + (long)kk * HD);
      }
      float sc[G][U];
#pragma unroll
      for (int g = 0; g < G; ++g)
#pragma unroll
        for (int u = 0; u < U; ++u) {
          float acc = 0.f;
#pragma unroll
          for (int j = 0; j < 8; ++j) acc += qf[g][j] * bf2f(kv[u][j]);
#pragma unroll
          for (int msk = 1; msk < LPK; msk <<= 1) acc += wave_xchg_n(acc, msk);
          sc[g][u] = key[u] < ctx ? acc : NEG;
        }
#pragma unroll
      for (int g = 0; g < G; ++g) {
        float mx = sc[g][0];
#pragma unroll
        for (int u = 1; u < U; ++u) mx = fmaxf(mx, sc[g][u]);
        const float mn = fmaxf(m[g], mx);
        const float alpha = exp2f(m[g] - mn);
        float p[U], ps = 0.f;
#pragma unroll
        for (int u = 0; u < U; ++u) {
          p[u] = exp2f(sc[g][u] - mn);
          ps += p[u];
        }
        l[g] = l[g] * alpha + ps;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          float a = o[g][j] * alpha;
#pragma unroll
          for (int u = 0; u < U; ++u) a += p[u] * bf2f(vv[u][j]);
          o[g][j] = a;
        }
        m[g] = mn;
      }
    }
#pragma unroll
    for (int msk = LPK; msk < 64; msk <<= 1) {
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const float mo = wave_xor_n(m[g], msk), lo = wave_xor_n(l[g], msk);
        const float mn = fmaxf(m[g], mo);
        const float a = exp2f(m[g] - mn), bb = exp2f(mo - mn);
        l[g] = l[g] * a + lo * bb;
#pragma unroll
        for (int j = 0; j < 8; ++j) o[g][j] = o[g][j] * a + wave_xor_n(o[g][j], msk) * bb;
        m[g] = mn;
      }
    }
    if (kg == 0) {
#pragma unroll
      for (int g = 0; g < G; ++g) {
        sm[w][g][ds][0] = m[g];
        sm[w][g][ds][1] = l[g];
#pragma unroll
        for (int j = 0; j < 8; ++j) sm[w][g][ds][2 + j] = o[g][j];
      }
    }
    __syncthreads();
    if (w == 0 && kg == 0) {
#pragma unroll
      for (int g = 0; g < G; ++g) {
        float mm = NEG;
#pragma unroll
        for (int ww = 0; ww < NWV; ++ww) mm = fmaxf(mm, sm[ww][g][ds][0]);
        float ll = 0.f, oo[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ww = 0; ww < NWV; ++ww) {
          const float f = exp2f(sm[ww][g][ds][0] - mm);
          ll += sm[ww][g][ds][1] * f;
#pragma unroll
          for (int j = 0; j < 8; ++j) oo[j] += sm[ww][g][ds][2 + j] * f;
        }
        const float inv = ll > 0.f ? 1.f / ll : 0.f;
#pragma unroll
        for (int j = 0; j < 8; ++j) so[b][g * HD + ds * 8 + j] = oo[j] * inv;
      }
    }
    __syncthreads();  // so[b] complete; sm reused by the next sequence
  }

  // ---- partial out-projection of this kv head's slice, NC columns
  const int n0 = c * NC;
  const int sub = lane % LPC;
  for (int cb = w * CPI; cb < NC; cb += NWV * CPI) {  // wave-uniform trip count (lane reductions)
    const int cc = cb + lane / LPC, n = n0 + cc;
    const bool valid = cc < NC && n < N;
    float wf[R][8];
#pragma unroll
    for (int rr = 0; rr < R; ++rr) {
      const bf16x8 wv = ld8(W + (long)min(n, N - 1) * ldw + (long)kvh * KS + (rr * LPC + sub) * 8);
#pragma unroll
      for (int j = 0; j < 8; ++j) wf[rr][j] = bf2f(wv[j]);
    }
    for (int b = 0; b < B; ++b) {
      float acc = 0.f;
#pragma unroll
      for (int rr = 0; rr < R; ++rr)
#pragma unroll
        for (int j = 0; j < 8; ++j) acc += so[b][(rr * LPC + sub) * 8 + j] * wf[rr][j];
#pragma unroll
      for (int msk = 1; msk < LPC; msk <<= 1) acc += wave_xchg_n(acc, msk);
      if (valid && sub == 0)
        __hip_atomic_store(part + (((long)c * n_kv + kvh) * B + b) * NC + cc, acc, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0) {
    const int t = __hip_atomic_fetch_add(cnt + c, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    s_flag = (t == n_kv - 1);
    if (t == n_kv - 1) __hip_atomic_store(cnt + c, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  if (!s_flag) return;
  // ---- last arriver: x[b][n] += bias[n] + sum_h part[c][h][b][n], kv heads in order
  for (int i = threadIdx.x; i < B * NC; i += NWV * 64) {
    const int b = i / NC, cc = i % NC, n = n0 + cc;
    if (n >= N) continue;
    float s = 0.f;
#pragma unroll 8
    for (int h = 0; h < n_kv; ++h)
      s += __hip_atomic_load(part + (((long)c * n_kv + h) * B + b) * NC + cc, __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
    float* xp = x + (long)b * N + n;
    *xp = *xp + (s + (bias ? bf2f(bias[n]) : 0.f));
  }
}

// Merge split-K decode partials: one wave per (sequence, head).  What it costs is the round
// trips to memory: the partials of AT_ONCE splits are requested together with all maxima and sums,
// not split by split behind them (1 sequence, 16 splits, with the kernel in front: 17.8 -> 7.2 us).
// MAXL: splits / 64, rounded up.  Requests beyond the last split are not free: 16 of them for two
// splits cost more than two loads in turn (4 sequences of 260 keys, 12 heads of 64: 6.9 -> 7.2 us; with
// 4 at once 6.9), so up to 4 splits take the short form.
template <int HD, int AT_ONCE, int MAXL>
__global__ __launch_bounds__(64) void attn_decode_combine_kernel(const float* part_o,
                                                                 const float* part_ml, bf16* out,
                                                                 long ldo, int nh, int splits) {
  constexpr int DPL = HD / 64;  // columns per lane
  __shared__ float ws[64 * MAXL];
  const int b = blockIdx.x / nh, h = blockIdx.x % nh, lane = threadIdx.x;
  const long p0 = ((long)b * nh + h) * splits;
  const float* po = part_o + p0 * HD + lane * DPL;
  float v[AT_ONCE][DPL];
  auto load = [&](int s0) {
#pragma unroll
    for (int i = 0; i < AT_ONCE; ++i)
#pragma unroll
      for (int d = 0; d < DPL; ++d) v[i][d] = po[(long)min(s0 + i, splits - 1) * HD + d];
  };
  float m[MAXL], l[MAXL];
#pragma unroll
  for (int i = 0; i < MAXL; ++i) {
    const int s = min(lane + i * 64, splits - 1);
    m[i] = part_ml[(p0 + s) * 2];
    l[i] = lane + i * 64 < splits ? part_ml[(p0 + s) * 2 + 1] : 0.f;
  }
  load(0);
  float mm = m[0];
#pragma unroll
  for (int i = 1; i < MAXL; ++i) mm = fmaxf(mm, m[i]);
  mm = wave_max(mm);
  float ll = 0.f;
#pragma unroll
  for (int i = 0; i < MAXL; ++i) {
    const float f = exp2f(m[i] - mm);
    ll += l[i] * f;
    ws[lane + i * 64] = lane + i * 64 < splits ? f : 0.f;
  }
  ll = wave_sum(ll);
  __syncthreads();
  float oo[DPL] = {};
  for (int s0 = 0; s0 < splits; s0 += AT_ONCE) {
    if (s0) load(s0);
#pragma unroll
    for (int i = 0; i < AT_ONCE; ++i)
#pragma unroll
      for (int d = 0; d < DPL; ++d) oo[d] += v[i][d] * (s0 + i < splits ? ws[s0 + i] : 0.f);
  }
#pragma unroll
  for (int d = 0; d < DPL; ++d)
    out[(long)b * ldo + (long)h * HD + lane * DPL + d] = f2bf(ll > 0.f ? oo[d] / ll : 0.f);
}

// ---------------------------------------------------------------------------
// Prefill: 64 QT queries of a head per block (4 waves x 16 QT), 64-key tiles in LDS
// ---------------------------------------------------------------------------
// Bound by what a wave does between its products: reading every key and value of a tile
// from LDS and some ten instructions per score.  So
//  * a wave takes two tiles of 16 queries (QT = 2) where that leaves blocks enough: each
//    fragment read feeds both.
//  * K and V go to LDS by DMA, a tile ahead in the other of two buffers, with 32-bit offsets from
//    the tile's first key (64-bit lane addresses: 7937 tokens, 32 heads over 8, 17 us of 590 more); their 16-byte chunks
//    are permuted within a row so that both the row reads of K and the transposing reads
//    of V, 8 rows by 32 bytes at a time, meet every bank once.
//  * sums are rescaled only where a query's maximum moved, and only tiles on the diagonal are
//    masked.  (A maximum that lags by up to 2^6 saves 3 % more, but the largest weight is
//    then not exactly one: the error against 64 bits grows by as much.)
//  * waves behind a sequence's last query only bring their part of the tiles: of short prompts
//    that is most of them (25 heads of 64: 64 x 20 tokens 11.1 -> 8.9 us, 128 x 10 17.2 -> 12.9).
//  * a kv head's blocks run side by side on one XCD, whose L2 then holds its keys, and a
//    sequence's longest first: the last ones to end are short.
// Before (one 16-query tile per wave, K and V through registers) -> now:
//   32 heads over 8 of 128: 7937 tokens 1290 -> 570 us (900 TF/s), 8 x 500 80 -> 42, 500 16 -> 12
//   25 heads of 64: 4 x 1000 tokens 72 -> 41 us, 20 x 200 27 -> 19
typedef short short4v __attribute__((ext_vector_type(4)));

__device__ __forceinline__ bf16x4 ds_read_tr(const bf16* lds_ptr) {
  typedef __attribute__((address_space(3))) bf16x4 lds_bf16x4;
  return __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)(lds_ptr));
}


template <int HD, int QT>
__global__ __launch_bounds__(256, 2) void attn_prefill_kernel(
    const bf16* __restrict__ q, long ldq, const bf16* __restrict__ kc,
    const bf16* __restrict__ vc, const int* __restrict__ tiles, int n_tiles,
    const int* __restrict__ seq_slots, const int* __restrict__ q_start,
    const int* __restrict__ cu_q, bf16* out, long ldo, int nh, int n_kv, int max_seq,
    float scale_log2) {
  constexpr int KT = 64;              // keys per tile
  constexpr int CPR = HD / 8;         // 16-B chunks per row
  constexpr int RPI = 64 / CPR;       // rows an LDS-DMA instruction brings
  constexpr int NI = KT / RPI / 4;    // instructions per wave and tile, of K and of V
  __shared__ __attribute__((aligned(16))) bf16 smem[2][2][KT * HD];
  // row's chunk c stands at c ^ swz(row)
  auto swz = [](int row) {
    return HD == 128 ? ((row & 7) << 1) | ((row >> 3) & 1) : (row & 6) | ((row >> 3) & 1);
  };

  // (kv head, tile from the last one on, head of the group)
  const int G = nh / n_kv, L = xcd_remap(blockIdx.x, gridDim.x);
  const int kvh = L / (G * n_tiles), at = L - kvh * G * n_tiles, behind = G == 1 ? at : at / G;
  const int x = n_tiles - 1 - behind, h = kvh * G + at - behind * G;
  const int bseq = tiles[x * 2], qoff = tiles[x * 2 + 1];
  const int qlen = cu_q[bseq + 1] - cu_q[bseq];
  const int st = q_start[bseq];
  const int lane = lane_id(), w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int q0 = qoff + w * QT * 16;           // the wave's first query (row within the sequence)
  const int kmax = st + min(qoff + 64 * QT, qlen);  // keys [0, kmax) are needed by the tile
  const int last_key = q0 < qlen ? st + q0 + QT * 16 - 1 : -1;  // of the wave; -1: it has no queries
  const int ntile = (kmax + KT - 1) / KT;
  const long base = ((long)seq_slots[bseq] * n_kv + kvh) * (long)max_seq * HD;

  bf16x8 qf[QT][HD / 32];
  f32x4 o[QT][HD / 16];
  float m[QT], lsum[QT];
#pragma unroll
  for (int t = 0; t < QT; ++t) {
    const long qrow = cu_q[bseq] + min(q0 + t * 16 + r, qlen - 1);
#pragma unroll
    for (int kk = 0; kk < HD / 32; ++kk) qf[t][kk] = ld8(q + qrow * ldq + (long)h * HD + kk * 32 + g * 8);
#pragma unroll
    for (int di = 0; di < HD / 16; ++di) o[t][di] = f32x4{0.f, 0.f, 0.f, 0.f};
    m[t] = NEG;
    lsum[t] = 0.f;
  }
  auto load_tile = [&](int kt, int buf) {
    const long at = base + (long)kt * KT * HD;
    const int last = kmax - 1 - kt * KT;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int row = (w * NI + i) * RPI + lane / CPR;
      const unsigned off = (min(row, last) * HD + (((lane % CPR) ^ swz(row)) << 3)) * 2;  // bytes
      lds_dma16(kc + at, smem[buf][0] + (w * NI + i) * 512, off, 0);
      lds_dma16(vc + at, smem[buf][1] + (w * NI + i) * 512, off, 0);
    }
  };
  load_tile(0, 0);
  for (int kt = 0; kt < ntile; ++kt) {
    const bf16 *ks = smem[kt & 1][0], *vs = smem[kt & 1][1];
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this wave's part of the tile has landed
    __builtin_amdgcn_s_barrier();        // ... and every wave's; the other buffer is read
    asm volatile("" ::: "memory");
    if (kt + 1 < ntile) load_tile(kt + 1, (kt + 1) & 1);
    if (kt * KT > last_key) continue;  // behind all of the wave's queries

    // S^T[key][q] for 4 subtiles of 16 keys
    f32x4 s[QT][4];
#pragma unroll
    for (int ni = 0; ni < 4; ++ni) {
#pragma unroll
      for (int t = 0; t < QT; ++t) s[t][ni] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < HD / 32; ++kk) {
        const bf16x8 kf = *reinterpret_cast<const bf16x8*>(ks + (ni * 16 + r) * HD + (((kk * 4 + g) ^ swz(r)) << 3));
#pragma unroll
        for (int t = 0; t < QT; ++t) s[t][ni] = mfma16(kf, qf[t][kk], s[t][ni]);
      }
    }
    const bool whole = (kt + 1) * KT - 1 <= st + q0;  // every query of the wave sees all keys
#pragma unroll
    for (int t = 0; t < QT; ++t) {
      if (!whole) {
        const int last = st + q0 + t * 16 + r - kt * KT;
#pragma unroll
        for (int ni = 0; ni < 4; ++ni)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (ni * 16 + 4 * g + i > last) s[t][ni][i] = NEG;
      }
      // tile max (lane-local over 16 keys, then across g); the scale is positive
      float tmax = s[t][0][0];
#pragma unroll
      for (int ni = 0; ni < 4; ++ni)
#pragma unroll
        for (int i = 0; i < 4; ++i) tmax = fmaxf(tmax, s[t][ni][i]);
      tmax *= scale_log2;
      tmax = fmaxf(tmax, wave_xchg<16>(tmax));
      tmax = fmaxf(tmax, wave_xchg<32>(tmax));
      if (__any(tmax > m[t])) {
        const float mn = fmaxf(m[t], tmax);
        const float alpha = __builtin_amdgcn_exp2f(m[t] - mn);
        m[t] = mn;
        lsum[t] *= alpha;
#pragma unroll
        for (int di = 0; di < HD / 16; ++di) o[t][di] *= alpha;
      }
      float ps[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ni = 0; ni < 4; ++ni)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float e = __builtin_amdgcn_exp2f(fmaf(s[t][ni][i], scale_log2, -m[t]));
          s[t][ni][i] = e;
          ps[i] += e;
        }
      lsum[t] += (ps[0] + ps[1]) + (ps[2] + ps[3]);
    }
    // O^T[d][q] += V^T[d][key] . P^T[key][q]; k-slot j of group g <-> key
    // 32kk + 4g + j (j < 4), 32kk + 16 + 4g + (j - 4) (j >= 4)
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      bf16x8 pf[QT];
#pragma unroll
      for (int t = 0; t < QT; ++t)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          pf[t][j] = f2bf(s[t][2 * kk][j]);
          pf[t][4 + j] = f2bf(s[t][2 * kk + 1][j]);
        }
      const int r0 = 4 * g + (r >> 2);
#pragma unroll
      for (int di = 0; di < HD / 16; ++di) {
        const bf16* v = vs + (kk * 32 + r0) * HD + (((2 * di + ((r >> 1) & 1)) ^ swz(r0)) << 3) + 4 * (r & 1);
        const bf16x4 lo = ds_read_tr(v), hi = ds_read_tr(v + 16 * HD);
        const bf16x8 vf = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
#pragma unroll
        for (int t = 0; t < QT; ++t) o[t][di] = mfma16(vf, pf[t], o[t][di]);
      }
    }
  }
#pragma unroll
  for (int t = 0; t < QT; ++t) {
    const int qi = q0 + t * 16 + r;
    float l = lsum[t];
    l += wave_xchg<16>(l);
    l += wave_xchg<32>(l);
    if (qi >= qlen) continue;
    const float inv = l > 0.f ? 1.f / l : 0.f;
    bf16* op = out + (long)(cu_q[bseq] + qi) * ldo + (long)h * HD;
#pragma unroll
    for (int di = 0; di < HD / 16; ++di) st4(op + di * 16 + 4 * g, pack4(o[t][di] * inv));
  }
}

// ---------------------------------------------------------------------------
// Decode, grouped-query heads on MFMA: one wave per (sequence, kv head)
// ---------------------------------------------------------------------------
// The VALU decode kernel above spends per key G x HD multiply-adds on the
// scores and as many on P.V, plus a 16-lane reduction per score: with
// Llama-3's G = 4 query heads of HD = 128 per kv head it is VALU-bound (about
// 3.6 TB/s of KV at 256 sequences against the 6.3 TB/s HBM floor).  Here the
// G queries of one kv head are the columns of an MFMA tile, the prefill
// kernel's swapped-operand scheme with a key tile instead of a query tile:
//   S^T[key][q] = K[key][d] . Q^T[d][q]      (16 keys x 16 columns, G valid)
//   O^T[d][q]  += V^T[d][key] . P^T[key][q]  (P^T straight from S^T's registers,
//                                             V^T via ds_read_b64_tr_b16)
// 32-key tiles of K and V are streamed with non-temporal 16-byte loads into
// registers (the next tile's loads in flight under the current tile's math),
// then staged through this wave's own LDS region for the fragment reads.
// Waves are independent: no block barrier.  The math is ~2% of the HBM time
// of the KV stream, so the kernel runs at the KV roofline.
//
// NW waves per block.  SPLIT_P: the weights enter the second product as three bf16 terms, which
// hold all 24 bits of them, for the calls whose weights the VALU kernel would hold in fp32.
template <int HD, int G, int NW, bool SPLIT_P>
__global__ __launch_bounds__(NW * 64) void attn_decode_mfma_kernel(
    const bf16* __restrict__ q, long ldq, const bf16* __restrict__ kc, const bf16* __restrict__ vc,
    const int* __restrict__ seq_slots, const int* __restrict__ qpos, bf16* out, long ldo,
    float* part_o, float* part_ml, int n_kv, int max_seq, int splits, float scale_log2,
    int n_items) {
  static_assert(G >= 1 && G <= 16, "G query heads per kv head fit one MFMA column tile");
  constexpr int KT = 32;             // keys per tile
  constexpr int LDR = HD + 8;        // padded LDS row (elements): +16 B
  constexpr int CPR = HD / 8;        // 16-B chunks per key row
  constexpr int CH = KT * CPR / 64;  // chunks per lane per tile (per K and per V)
  __shared__ __attribute__((aligned(16))) bf16 lds[NW][2][KT * LDR];
  const int lane = lane_id(), w = threadIdx.x >> 6;
  const int item = blockIdx.x * NW + w;
  if (item >= n_items) return;  // waves are independent: no barriers below
  bf16* ks = lds[w][0];
  bf16* vs = lds[w][1];
  const int b = item / n_kv, kvh = item % n_kv;
  const int ctx = qpos[b] + 1;
  // split blockIdx.y of the context (more waves than items), of whole tiles where many waves share
  // the memory: 40 sequences of 780 keys in 4 splits of 195 29.8 us, of 224 26.8.  (Few waves wait for
  // their own loads, which that makes larger.)  Behind the context's end a split has no keys.
  constexpr int UNIT = SPLIT_P ? 1 : KT;
  const int per = ((ctx + splits - 1) / splits + UNIT - 1) / UNIT * UNIT;
  const int k_lo = blockIdx.y * per, k_hi = min(ctx, k_lo + per);
  const long base = ((long)seq_slots[b] * n_kv + kvh) * (long)max_seq * HD;
  const int r = lane & 15, g = lane >> 4;

  // Q^T fragments: column r = query head kvh * G + r (zero columns past G)
  bf16x8 qf[HD / 32];
#pragma unroll
  for (int kk = 0; kk < HD / 32; ++kk) {
    bf16x8 z = {};
    qf[kk] = r < G ? ld8(q + (long)b * ldq + (long)(kvh * G + r) * HD + kk * 32 + g * 8) : z;
  }
  f32x4 o[HD / 16];
#pragma unroll
  for (int di = 0; di < HD / 16; ++di) o[di] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = NEG, lsum = 0.f;

  const int ntile = k_hi > k_lo ? (k_hi - k_lo + KT - 1) / KT : 0;
  bf16x8 kreg[CH], vreg[CH];
  auto load_tile = [&](int t) {
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int idx = lane + c * 64;
      const int key = min(k_lo + t * KT + idx / CPR, k_hi - 1);
      const long off = base + (long)key * HD + (idx % CPR) * 8;
      kreg[c] = LSD_KV_LOAD(kc + off);
      vreg[c] = LSD_KV_LOAD(vc + off);
    }
  };
  if (ntile > 0) load_tile(0);
  for (int t = 0; t < ntile; ++t) {
    // the previous tile's fragment reads must be done before the overwrite
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int idx = lane + c * 64;
      st8(ks + (idx / CPR) * LDR + (idx % CPR) * 8, kreg[c]);
      st8(vs + (idx / CPR) * LDR + (idx % CPR) * 8, vreg[c]);
    }
    __builtin_amdgcn_s_waitcnt(0xC07F);  // this wave's LDS writes landed
    __builtin_amdgcn_wave_barrier();
    if (t + 1 < ntile) load_tile(t + 1);  // in flight under this tile's math

    f32x4 sacc[2];
#pragma unroll
    for (int ni = 0; ni < 2; ++ni) {
      sacc[ni] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < HD / 32; ++kk) {
        const bf16x8 kf = *reinterpret_cast<const bf16x8*>(ks + (ni * 16 + r) * LDR + kk * 32 + g * 8);
        sacc[ni] = mfma16(kf, qf[kk], sacc[ni]);
      }
    }
    float tmax = NEG;
#pragma unroll
    for (int ni = 0; ni < 2; ++ni)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int key = k_lo + t * KT + ni * 16 + 4 * g + i;
        const float sv = key < k_hi ? sacc[ni][i] * scale_log2 : NEG;
        sacc[ni][i] = sv;
        tmax = fmaxf(tmax, sv);
      }
    tmax = fmaxf(tmax, wave_xchg<16>(tmax));
    tmax = fmaxf(tmax, wave_xchg<32>(tmax));
    const float mn = fmaxf(m, tmax);
    const float alpha = exp2f(m - mn);
    m = mn;
    float ps = 0.f;
#pragma unroll
    for (int ni = 0; ni < 2; ++ni)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float p = exp2f(sacc[ni][i] - mn);
        sacc[ni][i] = p;
        ps += p;
      }
    lsum = lsum * alpha + ps;
#pragma unroll
    for (int di = 0; di < HD / 16; ++di) o[di] *= alpha;
    // O^T += V^T . P^T over the 32 keys: k-slot j of group g <-> key 4g + j
    // (j < 4), 16 + 4g + (j - 4) (j >= 4)
    bf16x8 pf, pm, pl;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float e = sacc[j >> 2][j & 3];
      pf[j] = f2bf(e);
      const float e2 = e - bf2f(pf[j]);
      pm[j] = f2bf(e2);
      pl[j] = f2bf(e2 - bf2f(pm[j]));
    }
    const int r0 = 4 * g + (r >> 2);
#pragma unroll
    for (int di = 0; di < HD / 16; ++di) {
      const int col = di * 16 + 4 * (r & 3);
      const bf16x4 lo = ds_read_tr(vs + r0 * LDR + col);
      const bf16x4 hi = ds_read_tr(vs + (r0 + 16) * LDR + col);
      const bf16x8 vf = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      if constexpr (SPLIT_P) o[di] = mfma16(vf, pm, mfma16(vf, pl, o[di]));
      o[di] = mfma16(vf, pf, o[di]);
    }
  }
  lsum += wave_xchg<16>(lsum);
  lsum += wave_xchg<32>(lsum);
  if (r < G && splits > 1) {  // unnormalised partial for attn_decode_combine_kernel
    const long pi = ((long)b * n_kv * G + kvh * G + r) * splits + blockIdx.y;
    float* po = part_o + pi * HD;
#pragma unroll
    for (int di = 0; di < HD / 16; ++di) *reinterpret_cast<f32x4*>(po + di * 16 + 4 * g) = o[di];
    if (g == 0) {
      part_ml[pi * 2] = m;
      part_ml[pi * 2 + 1] = lsum;
    }
  } else if (r < G) {
    const float inv = lsum > 0.f ? 1.f / lsum : 0.f;
    bf16* op = out + (long)b * ldo + (long)(kvh * G + r) * HD;
#pragma unroll
    for (int di = 0; di < HD / 16; ++di) {
      bf16x4 rr;
#pragma unroll
      for (int i = 0; i < 4; ++i) rr[i] = f2bf(o[di][i] * inv);
      st4(op + di * 16 + 4 * g, rr);
    }
  }
}

}  // namespace lsd

using namespace lsd;

static int g_attn_max_wg = 0;  // 0: one workgroup per (sequence, kv head)
extern "C" void lsd_attn_set_max_wg(int v) { g_attn_max_wg = v; }
static int g_attn_small_waves = 0;  // waves per block for small decode batches (4, 8, 16; 88; 0: decode_keys)
static int g_attn_small_waves128 = 88;  // ... for 128-dim heads
extern "C" void lsd_attn_set_small_waves(int v) { g_attn_small_waves = v; }
extern "C" void lsd_attn_set_small_waves128(int v) { g_attn_small_waves128 = v; }
// waves per block for full decode batches, by head dim (4 or 8); 8 also
// requests V with K (lsd_attn_set_large_waves: tuning / A/B)
static int g_attn_large_waves64 = 4, g_attn_large_waves128 = 4;
// grouped-query decode on MFMA (attn_decode_mfma_kernel) for HD = 128,
// G in {2, 4, 8}: from this many waves ((sequence, kv head) items x context
// splits) with bf16 weights, below with three terms; 0 = off
// (lsd_attn_set_mfma_min).
static int g_attn_mfma_min = 256;
extern "C" void lsd_attn_set_mfma_min(int v) { g_attn_mfma_min = v; }
extern "C" void lsd_attn_set_large_waves(int hd, int v) {
  v = (v == 8 || v == 42 || v == 2) ? v : 4;
  if (hd == 64) g_attn_large_waves64 = v;
  else g_attn_large_waves128 = v;
}

static hipError_t attn_decode_combine(const float* part_o, const float* part_ml, bf16* out, long ldo,
                                      int B, int nh, int hd, int splits, hipStream_t st) {
  if (splits > 1) {
#define LSD_COMBINE(HDV, AT, ML)                                                                  \
  hipLaunchKernelGGL((attn_decode_combine_kernel<HDV, AT, ML>), dim3(B * nh), dim3(64), 0, st,     \
                     part_o, part_ml, out, ldo, nh, splits)
#define LSD_COMBINE_HD(HDV)                                      \
  if (splits <= 4) LSD_COMBINE(HDV, 4, 1);                       \
  else if (splits <= 8) LSD_COMBINE(HDV, 8, 1);                  \
  else if (splits <= 64) LSD_COMBINE(HDV, 16, 1);                \
  else LSD_COMBINE(HDV, 16, 4);
    if (splits > 256) return hipErrorInvalidValue;
    if (hd == 64) { LSD_COMBINE_HD(64) } else { LSD_COMBINE_HD(128) }
#undef LSD_COMBINE_HD
#undef LSD_COMBINE
  }
  return hipGetLastError();
}

static bool attn_on_mfma(int G, int hd) {
  return g_attn_mfma_min > 0 && hd == 128 && g_attn_max_wg == 0 && (G == 2 || G == 4 || G == 8);
}

// How many parts each of the caller's context splits is taken in (the partials are sized for
// all): few waves take short ranges.  A wave needs about 1.2 us per 32 keys; a merge, where the
// caller's splits have none, 2.4 us and what its (sequence, head) pairs add.  32 heads over
// 8: 1 sequence of 912 keys, 4 splits -> 16: 13.0 -> 6.9 us; 8 of 2000, 4 -> 8: 22.3 -> 17.1 (weights
// in two terms; three add 3 %); from 640 waves on lsd_attn_decode_total sees to it.
// One launch against two parts and their merge: 32 sequences of 20 keys 3.8 against 7.1 us, of
// 130 8.2 against 10.4, of 260 14 against 13.2; four parts: 1 sequence of 60 keys 4.8 against
// 5.8, of 100 7.3 against 6.0.  keys: the longest context, 0 where the caller does not know it.
extern "C" int lsd_attn_decode_split(int B, int n_kv, int G, int hd, int splits, int keys) {
  if (!attn_on_mfma(G, hd)) return 1;
  const long waves = (long)B * n_kv * splits;
  const int most = waves > 160 ? (int)(640 / waves) : 4;
  int best = 1;
  long least = 0;
  for (int f = 1; f == 1 || (f <= most && f * splits <= 256); ++f) {
    const long tiles = ((long)keys + 32 * splits * f - 1) / (32 * splits * f);
    const long cost = 120 * tiles + (splits * f > 1 ? 240 + (long)B * n_kv * G / 5 : 0);  // 1/100 us
    if (f == 1 || cost < least) { best = f; least = cost; }
  }
  return best;
}

// Splits that the kernel takes for a caller's `splits`.  What a launch of mixed contexts waits for
// is the longest one's chain of tiles, so calls of 256 waves and more, which few parts leave
// below six waves a CU, take up to 1536 waves of 128 keys and more; not from 512 items on, where a
// merge of its own costs what shorter chains give (64 sequences of 300 keys 17.8 us in one
// split, 19.4 in two), and no more than 16 (5 of 4000 keys: 20.9 us in 16, 22.2 in 32).  32 heads
// over 8, mixed lengths: 40 sequences of 70 .. 1490 keys, 3 splits 31.4 us, 4 29.3; 16 of
// 200 .. 2000, 4 -> 12 25.3 and 21.7; 48 of 150 .. 350, 1 -> 3 17.3 and 15.2; 32 heads over 16, 30 of
// 16 .. 1000, 2 -> 6 24.9 and 18.0.
extern "C" int lsd_attn_decode_total(int B, int n_kv, int G, int hd, int splits, int keys) {
  const int total = splits * lsd_attn_decode_split(B, n_kv, G, hd, splits, keys);
  const long items = (long)B * n_kv;
  if (!attn_on_mfma(G, hd) || items * splits < g_attn_mfma_min || items < 1 || items >= 512 || keys <= 256) return total;
  return std::max(total, (int)std::min<long>({1536 / items, (keys + 127) / 128, 16}));
}

// Keys in flight a lane group of 64-dim ungrouped heads on 4 waves, whose blocks take 8 times as many keys a
// wave and round: as few as hold the keys of a split in one round, behind 128 keys 8 (rounds of 256).  us for
// 2 / 4 / 8 (before, 8 waves of 4 keys up to 128 blocks, 4 of 4 beyond), contexts from half of the longest on:
//   12 items   40 keys 2.9 3.1 3.5 (4.0)   100 3.3 3.1 3.5 (4.1)   200 4.9 4.3 3.8 (4.6)   450 8.4 6.6 5.7 (5.9)
//   300        40 4.1 4.3 4.6 (4.6)        100 4.6 4.6 5.0 (5.0)   200 6.0 5.6 5.6 (5.9)   700 12.2 11.1 11.0 (11.4)
//   2400       40 8.0 10.4 12.1 (11.8)     100 11.1 12.0 13.2 (13.3)  200 17.2 17.4 16.9 (18.3)  1000 72.2 70.5 69.4 (71.0)
//   5000       16 10.5 15.3 17.7 (17.9)    100 17.9 20.7 23.6 (22.9)  200 31.4 31.0 30.5 (32.1)  450 65.8 64.4 63.3 (64.9)
// From 2048 items on 4 behind 128 keys: V with K costs two lanes of 256 sequences of 25 heads, which share the
// chip, 0.2 % of their tokens and 1.5 % of a step.
static int decode_keys(int keys, long items) {
  if (keys <= (items < 512 ? 64 : 128)) return 2;
  return keys <= 128 || items >= 2048 ? 4 : 8;
}

// total: lsd_attn_decode_total's; part_o and part_ml hold as many.  keys: the longest context, 0 where not known
extern "C" hipError_t lsd_attn_decode(const bf16* q, long ldq, const bf16* kc, const bf16* vc,
                                      const int* seq_slots, const int* qpos, bf16* out, long ldo,
                                      float* part_o, float* part_ml, int B, int nh, int n_kv,
                                      int hd, int max_seq, int splits, int total, int keys, float scale_log2,
                                      hipStream_t st) {
  if (B == 0) return hipSuccess;
  const int G = nh / n_kv;
  const int n_items = B * n_kv;
  const int gx = g_attn_max_wg > 0 ? (n_items < g_attn_max_wg ? n_items : g_attn_max_wg) : n_items;
  // grouped heads: on MFMA at any size (1 sequence of 912 keys with the merge 15.7 -> 7.2 us, 4 of
  // them 16.6 -> 8.8, 1 of 100 11.5 -> 5.8 against the VALU kernel).  Below g_attn_mfma_min waves
  // the weights keep all their bits, in three terms (two of 16 bits together: 7.0, 8.5 and 5.7 us)
  // (16 heads over 8, 24 sequences of 130 keys: 8.2 -> 9.4 us, where the VALU kernel is ahead; of
  // 60 and of 260 5.6 -> 5.3 and 13.8 -> 12.1)
  // One wave a block, so that the waves spread evenly over the CUs: in blocks of four, 1024 to
  // 2047 waves left some with twice the others' (160 sequences of 30 .. 400 keys, 1280 waves 31.6 ->
  // 29.1 us, 130 of 100 .. 900 58.3 -> 53.0, 40 of 1000 .. 8000 in 4 splits 183 -> 138).  From 2048 on, eight a
  // CU either way, blocks of four are up to 2 % ahead (256 of 400 .. 800: 106.4 and 108.7).
  if (attn_on_mfma(G, hd)) {
    const bool few = (long)n_items * splits < g_attn_mfma_min;
    splits = total;
#define LSD_DEC_MFMA(GV, NWV, SP)                                                                \
  if (G == GV && few == SP && (few || n_items * splits < 2048) == (NWV == 1)) {                 \
    hipLaunchKernelGGL((attn_decode_mfma_kernel<128, GV, NWV, SP>), dim3((n_items + NWV - 1) / NWV, splits), \
                       dim3(64 * NWV), 0, st, q, ldq, kc, vc, seq_slots, qpos, out, ldo, part_o, part_ml, \
                       n_kv, max_seq, splits, scale_log2, n_items);                              \
    return attn_decode_combine(part_o, part_ml, out, ldo, B, nh, hd, splits, st);                \
  }
#define LSD_DEC_MFMA_G(GV) \
  LSD_DEC_MFMA(GV, 1, true) LSD_DEC_MFMA(GV, 1, false) LSD_DEC_MFMA(GV, 4, false)
    LSD_DEC_MFMA_G(2)
    LSD_DEC_MFMA_G(4)
    LSD_DEC_MFMA_G(8)
#undef LSD_DEC_MFMA_G
#undef LSD_DEC_MFMA
    return hipErrorInvalidValue;
  }
  // 64-dim ungrouped heads: decode_keys.  Others: fewer blocks than half the CUs: wider blocks
  // (g_attn_small_waves waves), K and V of an item requested in one round of loads.
  // full batches: 4 waves (unroll 4) by default; 8 waves, 4 waves with
  // unroll 2 (42) and 2 waves (2) for A/B (lsd_attn_set_large_waves)
  const int lw = hd == 64 ? g_attn_large_waves64 : g_attn_large_waves128;
  // small grids: g_attn_small_waves (8; 88 = 8 waves with 8 keys per wave in
  // flight, so a 256-key context of a 128-dim head is one round of loads:
  // Llama-3 8B single stream 3.196 -> 3.172-3.181 ms, batch 4 3.757 -> 3.735;
  // profiles/r6_attn_u8.log)
  const int swd = hd == 128 ? g_attn_small_waves128 : g_attn_small_waves;
  int sw = (long)gx * splits <= 128 ? swd : (lw == 8 || lw == 42 || lw == 2 ? lw : 4);
  if (sw == 0 || sw == 4) {
    if (hd == 64 && G == 1 && (sw == 0 || (long)gx * splits > 128)) {
      const int u = decode_keys(((keys > 0 ? std::min(keys, max_seq) : max_seq) + splits - 1) / splits, n_items);
      sw = u == 2 ? 42 : u == 8 ? 48 : 4;
    } else if (sw == 0) {
      sw = 8;
    }
  }
  dim3 grid(gx, splits);
#define LSD_DEC(HDV, GV)                                                                        \
  if (hd == HDV && G == GV) {                                                                   \
    if (sw == 16)                                                                               \
      hipLaunchKernelGGL((attn_decode_kernel<HDV, GV, 2, 16>), grid, dim3(1024), 0, st, q, ldq, \
                         kc, vc, seq_slots, qpos, out, ldo, part_o, part_ml, n_kv, max_seq,     \
                         splits, scale_log2, n_items);                                          \
    else if (sw == 8)                                                                           \
      hipLaunchKernelGGL((attn_decode_kernel<HDV, GV, 4, 8>), grid, dim3(512), 0, st, q, ldq,   \
                         kc, vc, seq_slots, qpos, out, ldo, part_o, part_ml, n_kv, max_seq,     \
                         splits, scale_log2, n_items);                                          \
    else if (sw == 88 && GV <= 4)                                                               \
      hipLaunchKernelGGL((attn_decode_kernel<HDV, (GV <= 4 ? GV : 1), 8, 8>), grid, dim3(512),  \
                         0, st, q, ldq, kc, vc, seq_slots, qpos, out, ldo, part_o, part_ml,     \
                         n_kv, max_seq, splits, scale_log2, n_items);                           \
    else if (sw == 48 && HDV == 64 && GV == 1)                                                  \
      hipLaunchKernelGGL((attn_decode_kernel<HDV, GV, (HDV == 64 && GV == 1 ? 8 : 4), 4>), grid, dim3(256), 0, st, q, ldq, \
                         kc, vc, seq_slots, qpos, out, ldo, part_o, part_ml, n_kv, max_seq,     \
                         splits, scale_log2, n_items);                                          \
    else if (sw == 42)                                                                          \
      hipLaunchKernelGGL((attn_decode_kernel<HDV, GV, 2, 4>), grid, dim3(256), 0, st, q, ldq,   \
                         kc, vc, seq_slots, qpos, out, ldo, part_o, part_ml, n_kv, max_seq,     \
                         splits, scale_log2, n_items);                                          \
    else if (sw == 2)                                                                           \
      hipLaunchKernelGGL((attn_decode_kernel<HDV, GV, 4, 2>), grid, dim3(128), 0, st, q, ldq,   \
                         kc, vc, seq_slots, qpos, out, ldo, part_o, part_ml, n_kv, max_seq,     \
                         splits, scale_log2, n_items);                                          \
    else                                                                                        \
      hipLaunchKernelGGL((attn_decode_kernel<HDV, GV, 4, 4>), grid, dim3(256), 0, st, q, ldq,   \
                         kc, vc, seq_slots, qpos, out, ldo, part_o, part_ml, n_kv, max_seq,     \
                         splits, scale_log2, n_items);                                          \
    goto combine;                                                                               \
  }
  LSD_DEC(64, 1)
  LSD_DEC(64, 2)
  LSD_DEC(64, 4)
  LSD_DEC(128, 1)
  LSD_DEC(128, 2)
  LSD_DEC(128, 4)
  LSD_DEC(128, 8)
#undef LSD_DEC
  return hipErrorInvalidValue;
combine:
  return attn_decode_combine(part_o, part_ml, out, ldo, B, nh, hd, splits, st);
}

// rows: queries of a tile (64 or 128)
extern "C" hipError_t lsd_attn_prefill(const bf16* q, long ldq, const bf16* kc, const bf16* vc,
                                       const int* tiles, int n_tiles, int rows, const int* seq_slots,
                                       const int* q_start, const int* cu_q, bf16* out, long ldo,
                                       int nh, int n_kv, int hd, int max_seq, float scale_log2,
                                       hipStream_t st) {
  if (n_tiles == 0) return hipSuccess;
  const dim3 grid(n_tiles * nh), block(256);
#define LSD_PF(HDV, QTV)                                                                          \
  if (hd == HDV && rows == 64 * QTV) {                                                            \
    hipLaunchKernelGGL((attn_prefill_kernel<HDV, QTV>), grid, block, 0, st, q, ldq, kc, vc, tiles, \
                       n_tiles, seq_slots, q_start, cu_q, out, ldo, nh, n_kv, max_seq, scale_log2); \
    return hipGetLastError();                                                                     \
  }
  LSD_PF(64, 1)
  LSD_PF(64, 2)
  LSD_PF(128, 1)
  LSD_PF(128, 2)
#undef LSD_PF
  return hipErrorInvalidValue;
}

// Fused decode attention + output projection + residual add (B <= 4).
// part: fp32 [C][n_kv][B][NC] workspace, cnt: >= C zeroed ticket counters
// (re-armed by each chunk's last arriver).
extern "C" hipError_t lsd_attn_oproj(const bf16* q, long ldq, const bf16* kc, const bf16* vc,
                                     const int* seq_slots, const int* qpos, int B, int nh, int n_kv,
                                     int hd, int max_seq, float scale_log2, const bf16* W, long ldw,
                                     const bf16* bias, float* x, int N, int NC, float* part, int* cnt,
                                     hipStream_t st) {
  if (B == 0) return hipSuccess;
  if (B > 4 || NC < 1) return hipErrorInvalidValue;
  const int G = nh / n_kv;
  const dim3 grid(n_kv, (N + NC - 1) / NC), block(512);
#define LSD_AOP(HDV, GV)                                                                           \
  if (hd == HDV && G == GV) {                                                                      \
    hipLaunchKernelGGL((attn_oproj_kernel<HDV, GV, 8, 4>), grid, block, 0, st, q, ldq, kc, vc,     \
                       seq_slots, qpos, B, n_kv, max_seq, scale_log2, W, ldw, bias, x, N, NC, part, \
                       cnt);                                                                       \
    return hipGetLastError();                                                                      \
  }
  LSD_AOP(64, 1)
  LSD_AOP(128, 1)
  LSD_AOP(128, 2)
  LSD_AOP(128, 4)
  LSD_AOP(128, 8)
#undef LSD_AOP
  return hipErrorInvalidValue;
}
