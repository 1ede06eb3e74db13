// Prompt GEMM of some hundred to some thousand rows:  C[M,N] = A[M,K] . W[N,K]^T  (+ epilogue)
//
// Tiles of 64 MI x 64 NJ on four waves, for launches that 256 x 256 tiles (gemm_p8 in gemm.hip) share out badly among
// the CUs: 1000 x 6464 is 104 of those and takes as long as 256.  Before -> now, K = 2048 where not said, us:
// 500 x 4800 23.2 -> 13.3, 500 x 6400 with GELU 22.5 -> 14.3 (K = 1600), 512 x 6144 x 4096 48.5 -> 29.8, 1000 x 6464 31.9
// -> 29.5, 2000 x 11264 with SiLU 86.8 -> 78.5, 8000 x 6464 184 -> 172, 2000 x 1600 x 6400 77 -> 43.
//
// A block takes a K-tile (64 deep) in two pairs: the upper half of each wave row's rows of A and each wave column's
// rows of W, then the lower halves.  Four phases of 2 MI NJ products follow (upper, upper) (upper, lower) (lower, lower)
// (lower, upper); each reads the fragments of the next one's new operand, and W's upper half of the next K-tile goes to
// the registers that its lower half leaves, hence tiles unrolled in pairs.  A wave is alone on its SIMD, or one of two
// blocks', so the order of its instructions is written down: a product, then a read or a DMA beside it.
// Pairs lie in a ring of S LDS slots; a pair's slot is loaded again behind the barrier that follows its last read,
// twice a K-tile, and its data are there two barriers before they are read.
// What bounds it: a K-tile's DMA, 16 issue cycles each beside products of 16 (256 x 256 at this order 1.02 us a K-tile,
// without DMA 0.91, without reads 1.01, products alone 0.87), for small tiles what a CU takes in (60 to 65 GB/s beside
// its products), and some 5 to 9 us a block in front of its first product and behind its last.
// 256 x 256 in this order is no faster than gemm_p8, which power holds on long launches.
#include "gemm_epilogue.h"

#include <algorithm>

namespace lsd {

namespace {
typedef __attribute__((address_space(3))) void lds_void;
}

template <int N, class F, int I = 0>
__device__ __forceinline__ void count_up(F f) {
  if constexpr (I < N) {
    f(Int<I>{});
    count_up<N, F, I + 1>(f);
  }
}

// c += a b.  More than 128 sums a lane: named as AGPRs, or the compiler moves them about between the products.
// It does not know these for matrix instructions then and leaves no wait states around them: settle() does.
template <bool AGPR>
__device__ __forceinline__ void mma_at(f32x4& c, bf16x8 a, bf16x8 b) {
  if constexpr (AGPR) {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
  } else {
    c = mfma16(a, b, c);
  }
}

// In front of the first product and behind the last: the sums stand in their AGPRs, and no copy of them passes this
template <bool AGPR, int R, int Q>
__device__ __forceinline__ void settle(f32x4 (&c)[R][Q]) {
  if constexpr (AGPR) {
#pragma unroll
    for (int k = 0; k < 2; ++k) {
#pragma unroll
      for (int i = 0; i < R; ++i)
#pragma unroll
        for (int j = 0; j < Q; ++j) asm volatile("" : "+a"(c[i][j]));
      if (k == 0) asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
    }
  }
}

// Which of n things, spread over `places`, stands at place `at` (-1: none)
constexpr int stood(int at, int n, int places) {
  for (int x = 0; x < n; ++x)
    if (x * places / n == at) return x;
  return -1;
}

// S: ring slots, BPC: blocks a CU
template <int EPI, int MI, int NJ, int S, int BPC>
__global__ __launch_bounds__(256, BPC) void gemm_wave4_kernel(GemmParams p, int tiles_m, int tiles_n, int G) {
#if defined(__HIP_DEVICE_COMPILE__)  // (the host pass takes the launch stub alone; it emits none with this body)
  constexpr int BM = 64 * MI, BN = 64 * NJ, PA = MI * 4096, PAIR = (MI + NJ) * 4096, ND = MI + NJ, NP = 2 * MI * NJ;
  constexpr bool AGPR = MI * NJ > 8;
  static_assert((S - 1) * ND <= 63, "the wait counter holds 63 loads");
  static_assert(S * PAIR >= BM * BN * 2 + BM * 8, "C and the rows' positions are staged in the ring");
  __shared__ __attribute__((aligned(16))) char smem[S * PAIR];
  const int bid = xcd_remap(blockIdx.x, gridDim.x), KT = p.K / 64, per_split = tiles_m * tiles_n;
  int split = 0, tile_id = bid, kb = 0, T = KT;  // K-tiles of this split
  if (p.splits > 1) {
    split = bid / per_split;
    tile_id = bid % per_split;
    kb = (int)((long)KT * split / p.splits);
    T = (int)((long)KT * (split + 1) / p.splits) - kb;
  }
  int tm, tn;
  tile_order(tile_id, tiles_m, tiles_n, G, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;
  const int lane = lane_id(), w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wr = w >> 1, wc = w & 1, r = lane & 15, g = lane >> 4;

  // [half * MI + i][half * NJ + j], W rows x A rows: a lane has 4 columns of C in one row
  f32x4 acc[2 * MI][2 * NJ];
#pragma unroll
  for (int i = 0; i < 2 * MI; ++i)
#pragma unroll
    for (int j = 0; j < 2 * NJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  // This lane's 16 bytes of each DMA of a pair, from the tile's first row (rows behind the last one read that one
  // again): row pr of a part is row pr % 16 MI of half h of wave row pr / 16 MI, chunks XOR-swizzled
  const bf16* base[2] = {p.A + (long)m0 * p.lda + (long)kb * 64, p.W + (long)n0 * p.ldw + (long)kb * 64};
  int off[2][ND];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int x = 0; x < ND; ++x) {
      const bool ofw = x >= MI;
      const int q = ofw ? NJ : MI, pr = (w * q + (ofw ? x - MI : x)) * 8 + (lane >> 3);
      const int row = pr / (16 * q) * 32 * q + h * 16 * q + pr % (16 * q);
      const int ld = (int)(ofw ? p.ldw : p.lda), last = (ofw ? p.N - n0 : p.M - m0) - 1;
      off[h][x] = (min(row, last) * ld + (((lane & 7) ^ ((pr >> 1) & 7)) << 3)) * 2;
    }
  // (behind the last K-tile: loads of nothing, so the waits count alike)
  auto dma = [&](int t, int h, int slot, int x) {
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)base[x >= MI], 0, t < T ? 0x7fffffff : 0, 0x00020000);
    const int dst = x < MI ? (w * MI + x) * 1024 : PA + (w * NJ + x - MI) * 1024;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void*)(smem + slot * PAIR + dst), 16, off[h][x], t < T ? t * 128 : 0, 0, 0);
  };
  bf16x8 fa[2][2][MI], fb[2][2][NJ];  // [half][32-deep part][.]
  const int sw = (g ^ ((r >> 1) & 7)) << 4;
  const int la = (wr * 16 * MI + r) * 128 + sw, lb = PA + (wc * 16 * NJ + r) * 128 + sw;
  // this wave's reads of the slot just left are done, the next pair has landed, and so with every wave
  auto meet = [&] {
    __builtin_amdgcn_s_waitcnt(vmcnt_imm((S - 2) * ND) & ~(0xF << 8));
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };
  auto next = [](int s, int d) { s += d; return s >= S ? s - S : s; };
  // One phase: products of a (half mh) and b (half nh), over the first three quarters of them reads of the next
  // operand from `from`, over both phases of a pair its DMA: half hc of K-tile t into `slot`
  auto phase = [&](auto ph, bf16x8 (&a)[2][MI], bf16x8 (&b)[2][NJ], auto& dst, auto nr, int from, int t, auto h, int slot) {
    constexpr int q = decltype(ph)::v, mh = q >> 1, nh = q == 1 || q == 2, NR = decltype(nr)::v, H = NR / 2, hc = decltype(h)::v;
    const char* s0 = smem + from;
    const char* s1 = smem + (from ^ 64);
    count_up<NP>([&](auto pc) {
      constexpr int P = decltype(pc)::v, kk = P / (MI * NJ), i = P / NJ % MI, j = (i & 1) ? NJ - 1 - P % NJ : P % NJ, D = (q & 1) * NP + P;
      mma_at<AGPR>(acc[mh * MI + i][nh * NJ + j], b[kk][j], a[kk][i]);
      constexpr int x = stood(P, NR, NP * 3 / 4), y = stood(D - 1, ND, 2 * NP);
      if constexpr (x >= 0) dst[x / H][x % H] = *reinterpret_cast<const bf16x8*>((x / H ? s1 : s0) + (x % H) * 2048);
      if constexpr (y >= 0) dma(t, hc, slot, y);
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  // K-tile t, its pairs in slots s0 and s0 + 1; bx holds W's upper half, by is free
  auto tile = [&](int t, int s0, bf16x8 (&bx)[2][NJ], bf16x8 (&by)[2][NJ]) {
    const int s1 = next(s0, 1), s2 = next(s0, 2 % S);
    phase(Int<0>{}, fa[0], bx, by, Int<2 * NJ>{}, s1 * PAIR + lb, t + S / 2, Int<S & 1>{}, s0);
    phase(Int<1>{}, fa[0], by, fa[1], Int<2 * MI>{}, s1 * PAIR + la, t + S / 2, Int<S & 1>{}, s0);
    meet();
    phase(Int<2>{}, fa[1], by, fa[0], Int<2 * MI>{}, s2 * PAIR + la, t + (S + 1) / 2, Int<(S + 1) & 1>{}, s1);
    phase(Int<3>{}, fa[1], bx, by, Int<2 * NJ>{}, s2 * PAIR + lb, t + (S + 1) / 2, Int<(S + 1) & 1>{}, s1);
    meet();
  };
#pragma unroll
  for (int k = 0; k < S; ++k)
#pragma unroll
    for (int x = 0; x < ND; ++x) dma(k >> 1, k & 1, k, x);
  __builtin_amdgcn_s_waitcnt(vmcnt_imm((S - 1) * ND));
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) {
#pragma unroll
    for (int i = 0; i < MI; ++i) fa[0][kk][i] = *reinterpret_cast<const bf16x8*>(smem + (la ^ kk * 64) + i * 2048);
#pragma unroll
    for (int j = 0; j < NJ; ++j) fb[0][kk][j] = *reinterpret_cast<const bf16x8*>(smem + (lb ^ kk * 64) + j * 2048);
  }
  meet();
  settle<AGPR>(acc);
  int t = 0, s0 = 0;
  for (; t + 1 < T; t += 2) {
    tile(t, s0, fb[0], fb[1]);
    s0 = next(s0, 2 % S);
    tile(t + 1, s0, fb[1], fb[0]);
    s0 = next(s0, 2 % S);
  }
  if (t < T) tile(t, s0, fb[0], fb[1]);
  settle<AGPR>(acc);

  // ---- epilogue, on the sums.  This lane's columns of tile j and rows of tile i:
  const int col0 = wc * 32 * NJ + 4 * g, row0 = wr * 32 * MI + r;
  bf16x4 bias[2 * NJ] = {};
  if constexpr (EPI == EPI_BF16 || EPI == EPI_GELU || EPI == EPI_QKV || EPI == EPI_RESID)
    if (p.bias)
#pragma unroll
      for (int j = 0; j < 2 * NJ; ++j) bias[j] = ld4(p.bias + min(n0 + col0 + j * 16, p.N - 4));
  int pos[2 * MI] = {};  // QKV: of this lane's rows
  if (EPI == EPI_QKV && p.rope)
#pragma unroll
    for (int i = 0; i < 2 * MI; ++i) pos[i] = p.tpos[min(m0 + row0 + i * 16, p.M - 1)];
  // x += C in place, 16 bytes a lane; the next rows' x is requested in front of the stores
  if constexpr (EPI == EPI_RESID) {
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        reinterpret_cast<float*>(p.out) + (long)m0 * p.ldo, 0, min(p.M - m0, BM) * (int)p.ldo * 4, 0x00020000);
    auto at = [&](int i, int j) {  // out of range behind the last row or column
      const int n = n0 + col0 + j * 16;
      return n < p.N ? ((row0 + i * 16) * (int)p.ldo + n) * 4 : 0x7fffffff;
    };
    f32x4 x[2][2 * NJ];
    auto load = [&](int i) {
#pragma unroll
      for (int j = 0; j < 2 * NJ; ++j) x[i & 1][j] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, at(i, j), 0, 0));
    };
    load(0);
#pragma unroll
    for (int i = 0; i < 2 * MI; ++i) {
      if (i + 1 < 2 * MI) load(i + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < 2 * NJ; ++j) {
        f32x4 v = acc[i][j];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = x[i & 1][j][e] + (v[e] + bf2f(bias[j][e]));
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), rs, at(i, j), 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (loads of nothing still write zeros to LDS)
    return;
  }
  // every DMA landed before C overwrites the ring
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  __syncthreads();
  if (EPI == EPI_SLAB && !p.slab_bf16) {
    float* out = p.slab + (long)split * p.M * p.N;
#pragma unroll
    for (int i = 0; i < 2 * MI; ++i)
#pragma unroll
      for (int j = 0; j < 2 * NJ; ++j) {
        const int m = m0 + row0 + i * 16, n = n0 + col0 + j * 16;
        if (m < p.M && n < p.N) *reinterpret_cast<f32x4*>(out + (long)m * p.N + n) = acc[i][j];
      }
    return;
  }
  // bf16 results, the tile staged whole: 8-byte writes, 16-byte chunks XOR-swizzled by the row
  constexpr int WC = EPI == EPI_SILU_MUL ? BN / 2 : BN, CH = WC / 8, SWZ = CH % 16 == 0 ? 15 : CH % 8 == 0 ? 7 : 3;
  bf16* ct = reinterpret_cast<bf16*>(smem);
  int* tab = reinterpret_cast<int*>(smem + BM * BN * 2);  // QKV: the rows' positions and slots
  auto put = [&](int i, int col, f32x4 v) {
    const int row = row0 + i * 16;
    st4(ct + row * WC + (((col >> 3) ^ (row & SWZ)) << 3) + (col & 7), pack4(v));
  };
  const int qk = p.q_size + p.kv_size;
  if constexpr (EPI == EPI_QKV)
    if (threadIdx.x < BM) {
      const int m = min(m0 + (int)threadIdx.x, p.M - 1);
      tab[threadIdx.x] = p.tpos[m];
      tab[BM + threadIdx.x] = p.tslot[m];
    }
  // act: the gated activation, chosen outside the loops
  auto fill = [&](auto act) {
#pragma unroll
    for (int i = 0; i < 2 * MI; ++i) {
      if constexpr (EPI == EPI_SILU_MUL) {  // W rows in 16-row blocks [gate | up]
#pragma unroll
        for (int j = 0; j < 2 * NJ; j += 2) {
          f32x4 v;
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = gated<decltype(act)::v>(acc[i][j][e], acc[i][j + 1][e], p.act_scale);
          put(i, wc * 16 * NJ + j * 8 + 4 * g, v);
        }
      } else {
#pragma unroll
        for (int j = 0; j < 2 * NJ; ++j) {
          f32x4 v = acc[i][j];
          if constexpr (EPI != EPI_SLAB)
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] += bf2f(bias[j][e]);
          if constexpr (EPI == EPI_GELU)
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = gelu_new(v[e]);
          put(i, col0 + j * 16, v);
        }
      }
    }
  };
  if (EPI == EPI_QKV && p.rope && n0 < qk) {
    // (cos, sin) of this lane's two adjacent (even, odd) pairs, which turn together: of half of the rows at once
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      f32x4 cs[MI][2 * NJ];
#pragma unroll
      for (int j = 0; j < 2 * NJ; ++j) {
        const int n = n0 + col0 + j * 16;
        int head, d0;
        hd_split(p.hd, min(n, qk - 4) - (n < p.q_size ? 0 : p.q_size), head, d0);
#pragma unroll
        for (int i = 0; i < MI; ++i)
          cs[i][j] = *reinterpret_cast<const f32x4*>(p.rope + ((long)pos[h * MI + i] * (p.hd >> 1) + (d0 >> 1)) * 2);
      }
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < 2 * NJ; ++j) {
          f32x4 v = acc[h * MI + i][j];
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] += bf2f(bias[j][e]);
          float o[4] = {v[0], v[1], v[2], v[3]};
          turn_pair(o[0], o[1], cs[i][j][0], cs[i][j][1]);
          turn_pair(o[2], o[3], cs[i][j][2], cs[i][j][3]);
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = n0 + col0 + j * 16 < qk ? o[e] : v[e];
          put(h * MI + i, col0 + j * 16, v);
        }
    }
  } else if (EPI == EPI_SILU_MUL && p.glu == GLU_CLAMPED) {
    fill(Int<GLU_CLAMPED>{});
  } else if (EPI == EPI_SILU_MUL && p.glu == GLU_GELU) {
    fill(Int<GLU_GELU>{});
  } else {
    fill(Int<GLU_SILU>{});
  }
  __syncthreads();
  bf16* out = EPI == EPI_SLAB ? reinterpret_cast<bf16*>(p.slab) + (long)split * p.M * p.N : reinterpret_cast<bf16*>(p.out);
  const long ldo = EPI == EPI_SLAB ? p.N : p.ldo;
  const int c0 = EPI == EPI_SILU_MUL ? n0 / 2 : n0, cols = EPI == EPI_SILU_MUL ? p.N / 2 : p.N;
#pragma unroll 8
  for (int c = threadIdx.x; c < BM * CH; c += 256) {
    const int row = c / CH, ch = c % CH, m = m0 + row, n = c0 + ch * 8;
    if (m >= p.M || n >= cols) continue;
    bf16* dst = out + (long)m * ldo + n;
    if constexpr (EPI == EPI_QKV)
      if (n >= p.q_size) {
        int head, d;
        hd_split(p.hd, n < qk ? n - p.q_size : n - qk, head, d);
        dst = (n < qk ? p.kc : p.vc) + (((long)tab[BM + row] * p.n_kv + head) * p.max_seq + tab[row]) * p.hd + d;
      }
    st8(dst, ld8(ct + row * WC + ((ch ^ (row & SWZ)) << 3)));
  }
#endif
}

// MI, NJ, S, blocks a CU, and what a launch takes in 1/1000 us: its fixed part, each round of blocks behind the first,
// a round's K-tile with one block a CU, with two.  Fitted to 169 products of 280 to 18000 rows (N 1024 to 14336, K 768
// to 6400) on a card kept at work, 6 % off on average.  The tile so chosen is 0.5 % behind the best of these and of what
// was there before, and 14 % ahead of the latter on average, never more than 3 % behind it.
#define LSD_WAVE4_TILES(X)                                                                                      \
  X(2, 2, 4, 2, 4850, 2580, 496, 835) X(3, 2, 4, 2, 5890, 3770, 544, 1089) X(3, 3, 6, 1, 6640, 7540, 705, 0)      \
  X(4, 2, 3, 2, 6400, 4390, 791, 1358) X(4, 3, 5, 1, 7500, 10750, 849, 0) X(3, 4, 5, 1, 7460, 10050, 867, 0)

static long wave4_cost(int M, int N, int K, int S, int mi, int nj, int bpc, int fixed, int round, int one, int two) {
  const long tiles = (long)((M + 64 * mi - 1) / (64 * mi)) * ((N + 64 * nj - 1) / (64 * nj)) * S, cap = 256 * bpc;
  const long rounds = (tiles + cap - 1) / cap, last = tiles - cap * (rounds - 1), KT = K / 64;
  return fixed + round * (rounds - 1) + KT * ((rounds - 1) * (bpc == 2 ? two : one) + (bpc == 2 && last > 256 ? two : one)) / S;
}

// The tile of a launch: MI * 100 + NJ * 10 + blocks a CU, 0 where other kernels are ahead: 256 x 256 tiles (6.3 us,
// 11.8 a round, 1.072 a K-tile), and 128 x 64 ones up to one a CU (500 x 4096 x 2048 18.1 us, here 21.2; 700 x 4096,
// 384 of them, 25.5 and 19.9; 300 x 4800 x 1600, 225, 14.5 and 16.2; 300 x 6400, 300, 21.1 and 16.3).
static int wave4_tile(int M, int N, int K, int S) {
  if (M <= 256 || K % 64 != 0 || S < 1 || S > K / 64) return 0;
  if ((long)((M + 127) / 128) * ((N + 63) / 64) * S <= 256) return 0;
  int best = 0;
  long least = wave4_cost(M, N, K, S, 4, 4, 1, 6320, 11770, 1072, 0);
#define LSD_WAVE4(MI, NJ, SLOTS, B, F, R, C1, C2)                                    \
  {                                                                                  \
    const long c = wave4_cost(M, N, K, S, MI, NJ, B, F, R, C1, C2);                  \
    if (c < least) { best = MI * 100 + NJ * 10 + B; least = c; }                     \
  }
  LSD_WAVE4_TILES(LSD_WAVE4)
#undef LSD_WAVE4
  return best;
}

// What a launch takes that writes S slabs, and the norm that adds them up (1/1000 us): the tiles' times above, 128 x 64 ones where
// they are up to one a CU, and each slab written and read.  Fitted to 264 residual projections of 260 to 3000 rows (N 768 to 4096, K 768
// to 14336) in 2 to 8 slabs with their norm, weights from HBM: the number so chosen is 0.6 % behind the best on average.
static long slabs_cost(int M, int N, int K, int S) {
  long c = 5500 + 570L * (K / 64) / S;
  if ((long)((M + 127) / 128) * ((N + 63) / 64) * S > 256) {
    c = wave4_cost(M, N, K, S, 4, 4, 1, 6320, 11770, 1072, 0);
#define LSD_WAVE4(MI, NJ, SLOTS, B, F, R, C1, C2) c = std::min(c, wave4_cost(M, N, K, S, MI, NJ, B, F, R, C1, C2));
    LSD_WAVE4_TILES(LSD_WAVE4)
#undef LSD_WAVE4
  }
  return c + S * (150 + (long)M * N * 11 / 10000);
}

template <int EPI>
static hipError_t wave4_launch(const GemmParams& p, int code, hipStream_t st) {
#define LSD_WAVE4(MI, NJ, S, B, F, R, C1, C2)                                                                     \
  if (code == MI * 100 + NJ * 10 + B) {                                                                            \
    const int tm = (p.M + 64 * MI - 1) / (64 * MI), tn = (p.N + 64 * NJ - 1) / (64 * NJ);                          \
    hipLaunchKernelGGL((gemm_wave4_kernel<EPI, MI, NJ, S, B>), dim3(tm * tn * p.splits), dim3(256), 0, st, p, tm, tn, 16 / MI); \
    return hipGetLastError();                                                                                      \
  }
  LSD_WAVE4_TILES(LSD_WAVE4)
#undef LSD_WAVE4
  return hipErrorInvalidValue;
}

}  // namespace lsd

using namespace lsd;

// Slabs of a prompt's residual projection whose rule leaves S > 1: 2 to 8, or S.  Against the rule's, which knows 128 x 64 and
// 256 x 256 tiles, 6 % less on average with their norm: 1000 x 768 x 768 in 6 14.9 us, in 3 11.8; 700 x 768 x 1024 in 8 14.1, in 4 11.6;
// 260 x 1600 x 1600 in 7 13.3, in 5 11.2; 333 x 4096 x 4096 in 3 25.2, in 4 23.0.  Prompts of GPT-2, 360 tokens 676 -> 610 us, GPT-2 medium,
// 720 1676 -> 1608, GPT-2 XL, 750 4874 -> 4788.
extern "C" int lsd_gemm_prompt_slabs(int M, int N, int K, int S) {
  if (S <= 1 || M <= 256 || K % 64 != 0 || K < 256) return S;
  int best = 0;
  long least = 0;
  for (int s = 2; s <= 8 && s <= K / 128; ++s) {
    const long c = slabs_cost(M, N, K, s);
    if (best == 0 || c < least) { best = s; least = c; }
  }
  return S <= 8 || slabs_cost(M, N, K, S) >= least ? best : S;
}

extern "C" int lsd_gemm_wave4_tile(int M, int N, int K, int epi, int S) { return epi == EPI_F32 ? 0 : wave4_tile(M, N, K, S); }

// code: lsd_gemm_wave4_tile's
extern "C" hipError_t lsd_gemm_wave4(const GemmParams* p, int epi, int code, hipStream_t st) {
  switch (epi) {
#define LSD_WAVE4_EPI(E) \
  case E: return wave4_launch<E>(*p, code, st);
    LSD_WAVE4_EPI(EPI_BF16)
    LSD_WAVE4_EPI(EPI_GELU)
    LSD_WAVE4_EPI(EPI_SILU_MUL)
    LSD_WAVE4_EPI(EPI_RESID)
    LSD_WAVE4_EPI(EPI_QKV)
    LSD_WAVE4_EPI(EPI_SLAB)
#undef LSD_WAVE4_EPI
    default: return hipErrorInvalidValue;
  }
}
