// Projections of some tens of rows on gfx950: out[M, N] = x[M, K] . W[N, K]^T for M <= 256, bf16
// in, fp32 MFMA accumulate: decode batches, short prompts, the next message of a session.
//
// The weights are still read once and set the floor, but a block that read all of x for 16
// weight rows of its own (stream.hip) would spend its intake on x.  So x is shared:
//   * a block of WN waves holds x of 16 to 256 rows in LDS, shared by the waves, and 16 weight
//     rows of its own for each; both are filled by LDS-DMA, 8 rows x 128 bytes an instruction
//     (chunks XORed so that fragment reads have no bank conflicts; weights packed as for
//     stream.hip, ops.stream_pack, are one KB in fragment order instead);
//   * every wave reads all of x from LDS, 128 KB a stage of 128 rows and 8 waves, so the rows of a
//     block are few more than the step's: 16 apart up to 96, then 32.  us with heights of 64,
//     128, 192 and 256 -> now: 4096 x 4096 at 20 / 77 / 150 rows 8.2 / 11.8 / 15.8 -> 7.6 / 10.0 /
//     14.9, 6144 x 4096 at 77 15.6 -> 12.5, gated 28672 x 4096 at 20 / 77 / 224 49.6 / 53.7 / 71.8
//     -> 46.0 / 50.0 / 65.1; 112 beside 128 is not worth its code.  Waves of two weight units read
//     x half as often and were no faster (28672 x 4096 at 77 51.6, at 256 92): half as many waves
//     issue the DMA;
//   * WN is 8, or 4 where few columns would leave CUs without a block, unsliced 2 while its blocks
//     are one a CU; S blocks share a column tile's K and write fp32 slabs, which the next kernel sums.  S depends on
//     the weight alone (ops.panel_slices), and so does the order in which a wave walks its slice's K: a
//     row's result does not depend on how many rows the step has;
//   * rows of a weight are a power of two of bytes apart, or nearly, and blocks walk them in step, so
//     at any time all would ask a few memory channels for their 128 bytes of every row.  Where it is
//     faster, blocks therefore take the chunks of a power of two in other orders: by the number of
//     their eight weight units, whatever the waves and rows, so that bits do not depend on them, and
//     with its bits reversed, so that blocks that run together are far apart.  Of 64 chunks each such
//     block has an order of its own, of 32 two next to each other share one, which is the better of both
//     (us at 8 / 32 / 77 / 128 rows, shared / each its own: gated 16384 x 2048 12.2 / 13.8, 13.2 / 14.8, 17.4
//     / 18.3, 22.7 / 23.2; 8192 x 8192 in 4 slices 23.6 / 29.1, 23.1 / 29.9, 25.5 / 32.1, 30.1 / 34.3; 4096 x
//     14336 in 7 alike; but 32768 x 2048 at 8 26.4 / 22.4, above alike).  It is faster with row-major weights
//     of 64 MB and more in walks of 32 chunks (rows, or their slices, of 4 KB), gated also of 64: where the
//     line lies is measured, not derived, since plain walks of 64 lose.  A packed copy of such a weight is
//     walked in order, so its products have other roundings than the weight's own.  us, in
//     order / apart, at 32 / 77 / 128 rows: gated 28672 x 4096 42.8 / 39.0, 47.4 / 44.9, 55.1 / 53.4; gated
//     16384 x 4096 28.9 / 24.6, 33.9 / 31.0, 42.4 / 41.5; gated 16384 x 2048 17.3 / 14.5, 20.5 / 18.6,
//     24.1 / 23.1; 32768 x 2048 30.8 / 23.0, 32.6 / 24.8, 34.9 / 29.0; 131072 x 2048 103 / 88, 117 / 103,
//     144 / 125; 4096 x 14336 in 7 slices 25.9 / 20.9, 28.8 / 25.2, 32.8 / 29.7; 8192 x 8192 in 4 33.0 / 25.0,
//     35.3 / 27.1, 38.1 / 35.4.  Others lose or gain nothing (at 32 rows, plain 12288 x 4096 22.7 / 35.4,
//     28672 x 4096 43.0 / 62.4, 128256 x 4096 181 / 199, gated 8192 x 8192 30.9 / 43.3, 8192 x 4096 in 4
//     slices 13.9 / 15.7, 5120 x 13824 in 6 25.7 / 25.5), smaller ones may (8192 x 2048 gated 9.6 / 9.2,
//     4096 x 4096 7.9 / 8.8), and packed ones, 2 KB a chunk and unit (28672 x 4096 40.3 / 47.1);
//   * a ring of NS stages, of which NS - 1 stay in flight across the one raw barrier of a stage.
//     Past the end the loads go to one line, so that every wait counts the same number of loads.
//     The DMA is written as asm: hipcc, not knowing which stage a fragment read belongs to,
//     otherwise waits for all of it before some of the reads.
//   EPI 0  out = acc            EPI 1  out = act(g + b) * (u + b), W = [Wg; Wu]
//   EPI 2  fp32 slabs [S][M][N]
// and of experts, whose rows are expert-sorted assignments in segments of 64 or 128 (a block
// takes one segment; past the live ones it leaves):
//   EPI 5  silu(g) * u of the assignments' token rows, in sorted order
//   EPI 8  as 5, the routing weight on the input and a clamped GLU     EPI 10  gelu(up)
//   EPI 6  rows in sorted order, out[assignment] = routing weight (if given) * acc
#include "common.h"

using namespace omnia;

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ float4v mfma16(short8 a, short8 b, float4v c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

struct PanelArgs {
  void* out;
  const bf16_t *x, *w;  // [M, ldx]; [N, K], EPI 1 [2N, K]
  int M, N, K, S;
  int64_t ldx, ldo;
  const float* bias;  // EPI 1: [2N] or null
  int gelu;
  const int *sorted, *blk_expert, *n_blocks;  // experts
  const float* route_w;
  int topk, n_assign, e_lo;
  float alpha, limit;
};

constexpr bool grouped(int epi) { return epi >= 5; }
constexpr bool paired(int epi) { return epi == 1 || epi == 5 || epi == 8; }

template <int N>
struct Int {
  static constexpr int value = N;
};

template <int N>
__device__ __forceinline__ void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"i"(N) : "memory");
}

// 16 bytes a lane from its global address to LDS, lane-linear from the wave's byte address ``at``,
// which the load takes from m0.  hipcc reserves m0: it allocates no value to it (and warns that a
// clobber of it is undefined), and sets it for each instruction of its own that reads it; this
// file's have none (in the listing m0 is written by these lines alone).  NT: weights, read once (28672 x 4096
// at 16 rows 47.0 -> 43.1 us row-major, 44.2 -> 39.9 packed)
template <bool NT>
__device__ __forceinline__ void dma16(const void* src, uint32_t at) {
  if constexpr (NT)
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off nt" ::"s"(at),
                 "v"(src)
                 : "memory");
  else
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(at),
                 "v"(src)
                 : "memory");
}

// stages of (16 mf + 16 wn) x 128 bytes: up to 80 KB, two blocks a CU, where that is 3 stages
// or more (28672 x 4096 at 16 rows, 3 / 6 stages: 38.5 / 39.9 us), else up to 144 KB
constexpr int stages(int mf, int wn) {
  const int kb = 2 * (mf + wn), fit = (kb <= 26 ? 80 : 144) / kb;
  return fit > 5 ? 5 : fit;
}

// What the first loads need comes as arguments of their own: 14 words that are in registers when a
// wave starts (a struct is loaded from memory).
template <int MF, int WN, int EPI, bool PK>
__global__ __launch_bounds__(64 * WN, 1) void panel_kernel(const bf16_t* x, const bf16_t* w,
                                                           int64_t ldx, const int* n_blocks,
                                                           const int* blk_expert, int M, int N,
                                                           int K_, int S, PanelArgs p) {
  p.x = x, p.w = w, p.ldx = ldx, p.n_blocks = n_blocks, p.blk_expert = blk_expert;
  p.M = M, p.N = N, p.K = K_, p.S = S;
  constexpr int BM = 16 * MF, NS = stages(MF, WN);
  // DMA instructions of a wave and stage for x: XI, of the last XW waves XI - 1
  constexpr int XI = (2 * MF + WN - 1) / WN, XW = XI * WN - 2 * MF;
  constexpr int L = XI + 2;  // loads of a wave and stage
  static_assert(NS >= 3, "ring");
  constexpr int XS = BM * 64, ST = XS + WN * 1024;  // a stage: x, then the waves' weights
  __shared__ __attribute__((aligned(16))) bf16_t xs[NS][ST];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fr = lane & 15, fq = lane >> 4;
  const int units = paired(EPI) ? p.N >> 3 : p.N >> 4, tiles = (units + WN - 1) / WN;
  const int bid = xcd_remap(blockIdx.x, gridDim.x), seg = blockIdx.y;
  const bf16_t* W = p.w;
  if constexpr (grouped(EPI)) {
    if (seg >= *p.n_blocks) return;
    W += (int64_t)(p.blk_expert[seg] - p.e_lo) * (paired(EPI) ? 2 * p.N : p.N) * p.K;
  }
  const int split = bid / tiles, tile = bid - split * tiles;
  const int unit0 = tile * WN + wv, unit = unit0 < units ? unit0 : units - 1;
  const bool full = XW == 0 || wv < WN - XW;
  const int K = p.K, nch = K >> 6;
  const int c0 = split * nch / p.S, n = (split + 1) * nch / p.S - c0;  // 64-k chunks: stages
  // stage s of this block is chunk s ^ turn of its slice, by its weights' place alone (of 32 chunks the
  // lowest bit of the number falls off: two neighbours share an order)
  int turn = 0;
  if (!PK && !grouped(EPI) && (n == 32 || (paired(EPI) && n == 64)) &&
      (int64_t)p.N * K >= (paired(EPI) ? 1 << 24 : 1 << 25))
    turn = (int)(__builtin_bitreverse32(tile * WN >> 3) >> 26) & ((n & -n) - 1);

  // this wave's weights: row-major, rows 8h.. of the unit and 16-byte chunk lane & 7 of each;
  // packed, lane 16q + r's chunk of step h
  const bf16_t* wp[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    auto at = [&](int rr) -> int64_t {  // weight row of the unit's row rr
      if constexpr (paired(EPI)) return (rr < 8 ? 0 : (int64_t)p.N - 8) + (int64_t)unit * 8 + rr;
      return (int64_t)unit * 16 + rr;
    };
    if constexpr (PK) {
      const int64_t r = at(fr);
      wp[h] = W + (r >> 4) * 16 * K + h * 512 + 128 * fq + 8 * (r & 15);
    } else {
      const int rr = 8 * h + (lane >> 3);
      wp[h] = W + at(rr) * K + (((lane & 7) ^ (rr & 7)) << 3);
    }
  }
  const bf16_t* xp[XI];  // DMA instruction i of this wave: 8 rows
#pragma unroll
  for (int i = 0; i < XI; ++i) {
    const int r = (wv + i * WN) * 8 + (lane >> 3);
    if (!full && i == XI - 1) {
      xp[i] = p.x;
      continue;
    }
    int64_t row = r < p.M ? r : p.M - 1;
    if constexpr (EPI == 6) {
      row = seg * BM + r;
    } else if constexpr (grouped(EPI)) {  // the assignment's token (padding: the first one)
      const int f = p.sorted[seg * BM + r];
      row = f < p.n_assign ? f / p.topk : 0;
    }
    xp[i] = p.x + row * p.ldx + (((lane & 7) ^ (r & 7)) << 3);
  }
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane(
      (uint32_t)(uintptr_t)(__attribute__((address_space(3))) bf16_t*)&xs[0][0]);
  auto issue = [&](int slot, int s) {  // stage s into a slot
    const uint32_t dst = lds0 + slot * ST * 2;
    const bool in = s < n;
    const int64_t c = c0 + (s ^ turn);
#pragma unroll
    for (int i = 0; i < XI; ++i)
      if (full || i < XI - 1)
        dma16<false>(in ? xp[i] + c * 64 : p.x, dst + (wv + i * WN) * 1024);
#pragma unroll
    for (int h = 0; h < 2; ++h)
      dma16<true>(in ? wp[h] + c * (PK ? 1024 : 64) : p.x, dst + XS * 2 + wv * 2048 + h * 1024);
  };
  auto landed = [&](auto left) {  // this wave's loads but those of the newest ``left`` stages
    if (full)
      wait_vm<decltype(left)::value * L>();
    else
      wait_vm<decltype(left)::value * (L - 1)>();
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };
  float4v acc[MF];
#pragma unroll
  for (int i = 0; i < MF; ++i) acc[i] = {0.f, 0.f, 0.f, 0.f};
  auto compute = [&](const bf16_t* src) {
    const bf16_t* wb = src + XS + wv * 1024;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int ch = ((4 * h + fq) ^ (fr & 7)) << 3;  // rows 16i + fr share their XOR
      const short8 w =
          *reinterpret_cast<const short8*>(PK ? wb + h * 512 + lane * 8 : wb + fr * 64 + ch);
#pragma unroll
      for (int i = 0; i < MF; ++i)
        acc[i] = mfma16(*reinterpret_cast<const short8*>(src + (16 * i + fr) * 64 + ch), w, acc[i]);
    }
  };
#pragma unroll
  for (int s = 0; s < NS - 1; ++s) issue(s, s);
  int at = 0;
  for (; at + NS < n; at += NS)
#pragma unroll
    for (int u = 0; u < NS; ++u) {
      landed(Int<NS - 2>());
      issue((u + NS - 1) % NS, at + u + NS - 1);
      compute(xs[u]);
      __builtin_amdgcn_sched_barrier(0);
    }
  // up to NS stages are left, the last of them perhaps not yet asked for; each is waited for by
  // itself, since a slice may be a dozen stages (6144 x 4096 in 5 slices at 150 / 256 rows, with
  // one wait for what is left, 19.9 / 22.3 us, now 16.2 / 20.4)
  const bool more = at + NS == n;
  auto last = [&](auto i) {
    constexpr int u = decltype(i)::value;
    if constexpr (u < NS) {
      if (at + u >= n) return;
      if constexpr (u == 0) {
        landed(Int<NS - 2>());
        if (more) issue(NS - 1, at + NS - 1);
      } else if constexpr (u == NS - 1) {
        landed(Int<0>());
      } else {
        if (more)
          landed(Int<NS - 1 - u>());
        else
          landed(Int<NS - 2 - u>());
      }
      compute(xs[u]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  last(Int<0>());
  last(Int<1>());
  last(Int<2>());
  last(Int<3>());
  last(Int<4>());
  wait_vm<0>();  // loads past the end: none may land in the LDS of a block that follows

  // lane: rows 16i + 4fq + r, column fr
  if (unit0 >= units) return;
#pragma unroll
  for (int i = 0; i < MF; ++i) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = 16 * i + 4 * fq + r;
      float v = acc[i][r], u = 0.f;
      if constexpr (paired(EPI)) u = __shfl_xor(v, 8, 64);  // the up half, to the gate half's lanes
      const int64_t col = paired(EPI) ? (int64_t)unit * 8 + (fr & 7) : (int64_t)unit * 16 + fr;
      if (paired(EPI) && fr >= 8) continue;
      bf16_t* out = reinterpret_cast<bf16_t*>(p.out);
      if constexpr (grouped(EPI)) {
        const int row = seg * BM + m, f = p.sorted[row];
        if (f >= p.n_assign) continue;
        if constexpr (EPI == 6) {
          out[f * p.ldo + col] = f2bf(p.route_w ? p.route_w[f] * v : v);
        } else if constexpr (EPI == 5) {
          out[row * p.ldo + col] = f2bf(siluf_(v) * u);
        } else if constexpr (EPI == 8) {
          const float wt = p.route_w[f];
          out[row * p.ldo + col] = f2bf(clamped_glu(wt * v, wt * u, p.alpha, p.limit));
        } else {
          out[row * p.ldo + col] = f2bf(gelu_erf16_(v));
        }
      } else if (m < p.M) {
        if constexpr (EPI == 1) {
          if (p.bias) {
            v += p.bias[col];
            u += p.bias[p.N + col];
          }
          out[m * p.ldo + col] = f2bf((p.gelu ? gelu_tanh_(v) : siluf_(v)) * u);
        } else if constexpr (EPI == 0) {
          out[m * p.ldo + col] = f2bf(v);
        } else {
          reinterpret_cast<float*>(p.out)[((int64_t)split * p.M + m) * p.N + col] = v;
        }
      }
    }
  }
}

template <int MF, int WN, int EPI>
int launch(const PanelArgs& p, bool packed, hipStream_t s, int segs = 1) {
  const int units = paired(EPI) ? p.N / 8 : p.N / 16;
  const dim3 grid((units + WN - 1) / WN * p.S, segs);
#define OMNIA_PANEL(PK)                                                                       \
  panel_kernel<MF, WN, EPI, PK><<<grid, 64 * WN, 0, s>>>(p.x, p.w, p.ldx, p.n_blocks,         \
                                                         p.blk_expert, p.M, p.N, p.K, p.S, p)
  if (packed)
    OMNIA_PANEL(true);
  else
    OMNIA_PANEL(false);
#undef OMNIA_PANEL
  return (int)hipGetLastError();
}

template <int WN, int EPI>
int by_rows(const PanelArgs& p, bool packed, hipStream_t s) {
  switch ((p.M + 15) / 16) {
    case 1: return launch<1, WN, EPI>(p, packed, s);
    case 2: return launch<2, WN, EPI>(p, packed, s);
    case 3: return launch<3, WN, EPI>(p, packed, s);
    case 4: return launch<4, WN, EPI>(p, packed, s);
    case 5: return launch<5, WN, EPI>(p, packed, s);
    case 6: return launch<6, WN, EPI>(p, packed, s);
    case 7: case 8: return launch<8, WN, EPI>(p, packed, s);
    case 9: case 10: return launch<10, WN, EPI>(p, packed, s);
    case 11: case 12: return launch<12, WN, EPI>(p, packed, s);
    case 13: case 14: return launch<14, WN, EPI>(p, packed, s);
    default: return launch<16, WN, EPI>(p, packed, s);
  }
}

template <int EPI>
int by_waves(const PanelArgs& p, int wn, bool packed, hipStream_t s) {
  if constexpr (EPI != 2)
    if (wn == 2) return by_rows<2, EPI>(p, packed, s);
  return wn == 8 ? by_rows<8, EPI>(p, packed, s) : by_rows<4, EPI>(p, packed, s);
}

template <int EPI>
int by_segment(const PanelArgs& p, int bm, int wn, bool packed, int segs, hipStream_t s) {
  if (bm == 64)
    return wn == 8 ? launch<4, 8, EPI>(p, packed, s, segs) : launch<4, 4, EPI>(p, packed, s, segs);
  return wn == 8 ? launch<8, 8, EPI>(p, packed, s, segs) : launch<8, 4, EPI>(p, packed, s, segs);
}

}  // namespace

extern "C" {

// 0 on success, < 0 for what the kernel does not cover (checked before any launch).  wn: waves
// a block (4, 8; epi 0 and 1: 2).
int omnia_panel(int epi, void* out, const void* x, const void* w, int M, int N, int K, int S,
                int64_t ldx, int64_t ldo, int wn, int packed, const float* bias, int gelu,
                hipStream_t s) {
  if (epi < 0 || epi > 2) return -1;
  if (M < 1 || M > 256) return -2;
  if (K < 64 || K % 64 || ldx < K || ldx % 8) return -3;
  if (S < 1 || S > 16 || S > K / 64 || (epi != 2 && S != 1)) return -4;
  if (N < 16 || N % 16 || N > 1 << 24) return -5;
  if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w)) & 15) return -6;
  if (bias && epi != 1) return -7;
  if (wn != 4 && wn != 8 && (wn != 2 || epi == 2)) return -8;
  const PanelArgs p{out, (const bf16_t*)x, (const bf16_t*)w, M, N, K, S, ldx, ldo, bias, gelu,
                    nullptr, nullptr, nullptr, nullptr, 1, 0, 0, 0.f, 0.f};
  if (epi == 0) return by_waves<0>(p, wn, packed, s);
  if (epi == 1) return by_waves<1>(p, wn, packed, s);
  return by_waves<2>(p, wn, packed, s);
}

// Grouped products over segments of bm (64, 128) rows as omnia_moe_align makes them.  Modes and
// operands as omnia_moe_gemm.
int omnia_panel_moe(int mode, void* out, const void* A, const void* W, const int* sorted,
                    const int* blk_expert, const int* n_blocks, const float* route_w, int K, int N,
                    int topk, int n_assign, int e_lo, int max_blocks, int bm, int wn, int packed,
                    float alpha, float limit, hipStream_t s) {
  if (mode < 0 || mode > 3 || K < 64 || K % 64) return -1;
  if (bm != 64 && bm != 128) return -2;
  if (wn != 4 && wn != 8) return -3;
  const int cols = mode == 0 || mode == 2 ? 8 : 16;
  if (N < 16 || N % cols || (packed && N % 16) || N > 1 << 24) return -4;
  if (mode == 2 && !route_w) return -5;
  if (max_blocks == 0) return 0;
  if (max_blocks > 65535 || topk < 1) return -6;
  if ((reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(W)) & 15) return -7;
  const PanelArgs p{out,    (const bf16_t*)A, (const bf16_t*)W, bm,       N,    K,        1,
                    K,      N,                nullptr,          0,        sorted, blk_expert,
                    n_blocks, route_w,        topk,             n_assign, e_lo, alpha,    limit};
  if (mode == 0) return by_segment<5>(p, bm, wn, packed, max_blocks, s);
  if (mode == 1) return by_segment<6>(p, bm, wn, packed, max_blocks, s);
  if (mode == 2) return by_segment<8>(p, bm, wn, packed, max_blocks, s);
  return by_segment<10>(p, bm, wn, packed, max_blocks, s);
}

}  // extern "C"
