// Prefill GEMM with fused epilogues on gfx950:  out = X[M, K] . W[N, K]^T  for
// prefill chunks (M = hundreds to 16K rows), bf16 operands, fp32 MFMA accumulate.
// QKV (with RoPE and the paged KV write), O, SwiGLU, down (with the residual add).
//
// Main loop: a 256x256 tile by four waves, 2 x 2, one a SIMD, 128 x 128 of the tile each (256
// fp32 accumulators a lane, in AGPRs), in K-tiles of 64:
//   * what bounds a large product is power: MFMAs from registers alone reach 2.45 PF/s on zeros
//     and 2.04 on normal values (16x16x32; 32x32x16 1.80), so the loop moves as little as it
//     can.  A wave of 128 x 128 reads 128 KB of LDS a K-tile and CU, where eight waves of
//     128 x 64 read 224; the products go in a snake, each keeps an operand of the one before;
//   * a K-tile is four 16 KB half-tiles (A0 A1: rows 0-127, 128-255 of X, B0 B1: of W), filled
//     by LDS-DMA (16 bytes a lane; chunk c of row r at c ^ (r & 7), so that fragment reads have
//     no bank conflicts), in a ring of ten: two K-tiles and B of a third, as W often comes from HBM
//     and x from the L2 of the XCD (us with A / B of the third: gated 28672 x 4096 at 512 rows 98 /
//     95.6, at 2001 329 / 324, at 2560 in a model 444 / 425, 16384 x 2048 at 16384 744 / 740, plain
//     4096 x 14336 in 8 slices at 512 49.3 / 47.7, experts' up of 8 x 2048 x 4096 at 16384 tokens
//     882 / 876, down at 2001 / 2400 / 8000 / 16384 85.5 / 84, 86.5 / 84.5, 208 / 211, 424 / 427).  EPI 2
//     and 3, of the dense models' large prompts, A of a third (in a model, us a product, A / B: EPI 2
//     at 2560 rows 180 / 182, 8192 408 / 415, 16384 811 / 824, EPI 3 103 / 104, 307 / 309, 608 / 611).
//     Two barriers a K-tile:
//     one once every wave has read it (its slots are asked for again), one once the next has
//     landed, 40 products later; up to 96 KB are in flight, waits are counted;
//   * fragments of 32 k are read half a K-tile ahead, one read every other product, and the 16
//     DMA instructions of a wave stand apart: an address unit takes one in 16 clocks, so a run
//     of them would hold up the products behind it (zeros, 8192-cubed: 16 in a row 636 us,
//     spread 563).  m0 is set before the product that the DMA follows;
//   * products are asm: hipcc's own allocation of 256 accumulators moves some 200 of them a
//     K-tile.  It puts no wait states around asm: pin() stands between accumulators and others;
//   * XCD-aware block order (bijective remap), GM m-tiles a group, so that the blocks of an XCD
//     share W column tiles and X row tiles in its L2: 4 where W stays in the 256 MB Infinity
//     Cache, else 8 (16384 rows of 4096 x 14336 GM 4 / 8: 1270 / 1301 us; of 28672 x 4096
//     2605 / 2574).
// What is left of a tile is its ends: 3 to 4 thousand clocks until its first K-tiles are there and
// 6 to 8 thousand of its epilogue, of a K-tile's 2.3.  One wave a SIMD issues an instruction in about
// 5 clocks, so the accumulators start with the first products' results (256 writes fewer), rows
// without a scale are not multiplied by one (256), a bias is there when it is needed, and the stores
// of a row stand together.  us before / now, tiles of 4 rounds: 4096 rows of 16384 x 256 54.7 / 50.2, x
// 2048 206 / 201, gated with bias 203 / 200, x 4096 377 / 373; of one round 53.2 / 51.5.  The other
// K-tiles' DMAs between the first one's products: no gain.
// Normal values, us before (eight waves, one K-tile ahead) and now, 16384 rows: 4096 x 4096
// 382 / 361, 4096 x 14336 1344 / 1270, 28672 x 4096 2698 / 2574 (1.50 PF/s), 6144 x 4096 578 /
// 554, 2048 x 2048 110 / 100.
// The narrow tile (NF 4: 128 columns, a wave 128 x 64, K-tiles of three halves in a ring of nine) is
// for steps of some hundred rows, whose wide tiles leave CUs without one: a round of them takes
// 0.57 to 0.6 of a wide round, bound by what a CU takes in (48 KB in 0.67 us, where the wide
// tile's 64 KB in 1.09 are at the rate of its products).  us wide / narrow: gated 16384 x 2048 at 512
// rows 45.5 / 32.8, 4096 x 2048 at 2001 42.6 / 30.6; in 4 slices 2048 x 8192 at 999 45.8 / 33.4.
// Epilogues (W is the product's first operand, so a lane holds four neighbouring columns of a
// row; lanes exchange pairs and store 16 bytes, 64 a row and instruction, past LDS):
//   EPI 0  out = rs[r] * acc                                  (plain / row-scaled)
//   EPI 1  out = silu(rs*g) * (rs*u),  W = [Wg; Wu]            (gate_up + SwiGLU)
//   EPI 2  residual += acc  (in place), ss_out[r][tile] = sum of squares of the
//          new bf16 residual row slice                          (O / down)
//   EPI 3  rs-scaled QKV -> RoPE(q) to q_out, RoPE(k) and v to the paged KV cache
//   EPI 5  MoE grouped gate_up + SwiGLU: the 256-row tile's rows are expert-sorted
//          assignments (moe_align at 256-row segments), A rows gathered by token,
//          W = that segment's expert [Wg; Wu]; act written in sorted order
//   EPI 6  MoE grouped down: A = act (sorted order), W = the segment's expert,
//          each row scaled by its routing weight (if given) and scattered to Y[assignment]
//   EPI 8  EPI 5 with the routing weight on the expert's input and a clamped GLU
//   EPI 7  EPI 1 with a bias: out = silu(g + bias[f]) * (u + bias[N + f])
//   EPI 9  EPI 1 with the tanh form of gelu, unscaled: out = gelu(g) * u
//   EPI 10 EPI 5 ungated: gelu (erf form) of the up projection, W = that segment's expert Wu
//   EPI 4  split-K partial: block (m-tile, n-tile, k-slice ks) writes its K-slice's
//          fp32 sum, saturated to fp16, into slab ks of out[S][M][N]; the splitk.hip
//          consumers reduce the slabs (decode projections at M <= 256: one m-tile,
//          the K split fills the chip that N / 256 column tiles alone cannot)
//   EPI 11 EPI 4 with the sums as they are, slabs in fp32
// where rs[r] = rsqrt(sum_t ss_in[r][t] / d + eps): with the RMSNorm weight folded
// into W (W' = W * diag(w), models/llama.py fold_norms), RMSNorm(h) @ W^T ==
// rs * (h @ W'^T), so the normalisation rides the consumer's epilogue and the
// residual's sum of squares rides the producer's -- no RMSNorm, SwiGLU or RoPE
// launch exists in a prefill layer.
#include <type_traits>

#include "common.h"

using namespace omnia;

namespace {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float float2v __attribute__((ext_vector_type(2)));

constexpr int BK = 64;
constexpr int HALF = 128 * BK;  // bf16 elements of a half-tile (16 KB)
// A block's tile: 256 x 256, narrow 256 x 128, flat 128 x 256 (four waves side by side)
enum Shape { WIDE, NARROW, FLAT };
constexpr int ring(int shape) { return (shape == WIDE ? 10 : 9) * HALF; }

struct PArgs {
  void* out;            // EPI 0/1: bf16 [M, ldo]; EPI 2: residual bf16 [M, ldo]; EPI 3: q [M, ldo]
  const bf16_t* X;      // [M, K]
  const bf16_t* W;      // [N, K] ([2N, K] for EPI 1)
  int M, N, K, ldo;
  const float* ss_in;   // [M, ss_in_n] partial sums of squares (nullptr: no row scale)
  int ss_in_n;
  float inv_d, eps;
  float* ss_out;        // EPI 2: [M, N / 256]
  const int* positions;  // EPI 3
  const float* cos_sin;  // [max_pos, 128] = cos[64] | sin[64]
  bf16_t* k_cache;
  bf16_t* v_cache;       // [NB, hkv, BS, 128]
  const int64_t* slots;  // [M] (< 0: no KV write)
  int hq, hkv, block_size;
  int splits;            // EPI 4: K-slices (slabs)
  // EPI 5 / 6 (MoE grouped): sorted assignment ids [max_blocks * 256] (n_assign =
  // padding), per-256-row-segment expert, live segment count, routing weights
  const int* sorted;
  const int* blk_expert;
  const int* n_blocks;
  const float* route_w;
  int topk, n_assign, e_lo;
  const float* bias;     // EPI 7: fp32 [2N]
  float glu_alpha, glu_limit;  // EPI 8
};

// a gate_up epilogue: 128 features per block tile, gate and up halves in one lane
constexpr bool gated(int epi) {
  return epi == 1 || epi == 5 || epi == 7 || epi == 8 || epi == 9;
}
// slabs of K-slices
constexpr bool sliced(int epi) { return epi == 4 || epi == 11; }
// rows are expert-sorted assignments
constexpr bool grouped(int epi) { return epi == 5 || epi == 6 || epi == 8 || epi == 10; }
// wide tiles may be cut in two narrow ones
constexpr bool cuts(int epi) { return epi != 2 && epi != 3 && !sliced(epi); }
// Of ``wide`` tiles with ``light`` half ones behind them, how many of the last round over 256 CUs to
// cut in two.
__host__ __device__ constexpr int cut_tiles(int wide, int light) {
  const int last = wide & 255;
  return 2 * last + light <= 256 ? last : 0;
}
// A rows are token rows gathered by assignment
constexpr bool gathered(int epi) { return epi == 5 || epi == 8 || epi == 10; }

__device__ __forceinline__ float silu(float g) { return g * __builtin_amdgcn_rcpf(1.f + __expf(-g)); }
// acc += a . b.  Accumulators and operands as they lie in registers: no wait states are needed
// between products, between LDS reads and products (hipcc waits for the reads), nor before reads
// that overwrite an operand (it is read at issue)
__device__ __forceinline__ void mfma16(float4v& acc, short8 a, short8 b) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
}
// acc = a . b
__device__ __forceinline__ void mfma16_first(float4v& acc, short8 a, short8 b) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=a"(acc) : "v"(a), "v"(b));
}
// ... and behind it a DMA of 16 bytes a lane to LDS address ``at`` + OFF (lane-linear); ONCE: of what
// no later block reads
#define OMNIA_PRODUCT_DMA(HINT)                                         \
  asm volatile(                                                         \
      "s_add_u32 m0, %5, %6\n\t"                                        \
      "v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0\n\t"                     \
      "global_load_lds_dwordx4 %3, %4" HINT                             \
      : "+a"(acc)                                                       \
      : "v"(a), "v"(b), "v"(voff), "s"(base), "s"(at), "i"(off)         \
      : "memory", "scc")
template <bool ONCE = false>
__device__ __forceinline__ void mfma16_dma(float4v& acc, short8 a, short8 b, uint32_t voff,
                                           const void* base, uint32_t at, int off) {
  if constexpr (ONCE)
    OMNIA_PRODUCT_DMA(" nt");
  else
    OMNIA_PRODUCT_DMA("");
}
#undef OMNIA_PRODUCT_DMA
__device__ __forceinline__ void mfma16_dma(float4v& acc, short8 a, short8 b, const void* src,
                                           uint32_t at, int off) {
  asm volatile(
      "s_add_u32 m0, %4, %5\n\t"
      "v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0\n\t"
      "global_load_lds_dwordx4 %3, off"
      : "+a"(acc)
      : "v"(a), "v"(b), "v"(src), "s"(at), "i"(off)
      : "memory", "scc");
}
__device__ __forceinline__ void dma16(uint32_t voff, const void* base, uint32_t at, int off) {
  asm volatile("s_add_u32 m0, %2, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff),
               "s"(base), "s"(at), "i"(off)
               : "memory", "scc");
}
__device__ __forceinline__ void dma16(const void* src, uint32_t at, int off) {
  asm volatile("s_add_u32 m0, %1, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src),
               "s"(at), "i"(off)
               : "memory", "scc");
}

// two f32 -> packed bf16x2 (low = a), by the hardware's conversion
__device__ __forceinline__ uint32_t pack_b2(float a, float b) {
  const float2v v = {a, b};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}
__device__ __forceinline__ float4v round_b(float4v v) {
  const uint32_t l = pack_b2(v[0], v[1]), h = pack_b2(v[2], v[3]);
  return float4v{__uint_as_float(l << 16), __uint_as_float(l & 0xffff0000u),
                 __uint_as_float(h << 16), __uint_as_float(h & 0xffff0000u)};
}
// two f32 -> packed fp16x2 (low = a), saturated to the fp16 range: a K-slice's
// partial beyond +-65504 stays finite (its slab sum then errs, never turns NaN)
__device__ __forceinline__ uint32_t pack_h2(float a, float b) {
  a = fminf(fmaxf(a, -65504.f), 65504.f);
  b = fminf(fmaxf(b, -65504.f), 65504.f);
  return (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)a) |
         ((uint32_t)__builtin_bit_cast(uint16_t, (_Float16)b) << 16);
}

template <int EPI>
__device__ __forceinline__ uint32_t pack2(float a, float b) {
  if constexpr (EPI == 4) return pack_h2(a, b);
  return pack_b2(a, b);
}

// columns 4q .. 4q + 3 of two neighbouring 16-column blocks (q = lane / 16) -> eight columns:
// block q & 1, columns 8 (q >> 1) ..
template <int EPI>
__device__ __forceinline__ uint4v chunk(float4v c, float4v d) {
  const auto lo = __builtin_amdgcn_permlane16_swap(pack2<EPI>(c[0], c[1]), pack2<EPI>(d[0], d[1]),
                                                   false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap(pack2<EPI>(c[2], c[3]), pack2<EPI>(d[2], d[3]),
                                                   false, false);
  return uint4v{lo[0], hi[0], lo[1], hi[1]};
}

template <int N>
__device__ __forceinline__ void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"i"(N) : "memory");
}

// scale of row i of a tile from row m0, of which Mt are live
template <int EPI>
__device__ __forceinline__ float row_scale(const PArgs& p, int m0, int Mt, int i) {
  if constexpr (EPI == 6 || EPI == 8) {  // the assignment's routing weight
    const int f = p.sorted[m0 + i];
    return f >= p.n_assign ? 0.f : p.route_w ? p.route_w[f] : 1.f;
  }
  const float* s = p.ss_in + (int64_t)(m0 + (i < Mt ? i : Mt - 1)) * p.ss_in_n;
  float t = 0.f;
  for (int k = 0; k < p.ss_in_n; k += 8) {
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = s[k + j < p.ss_in_n ? k + j : k];
#pragma unroll
    for (int j = 0; j < 8; ++j) t += k + j < p.ss_in_n ? v[j] : 0.f;
  }
  return __builtin_amdgcn_rsqf(t * p.inv_d + p.eps);
}

// Tile (mt, nt) of K-slice ks; step t is K-tile t ^ turn; ONCE: W is not read by later tiles
template <int EPI, int SHAPE, bool ONCE = false>
__device__ __forceinline__ void tile(const PArgs& p, bf16_t* __restrict__ lds, int mt, int nt,
                                     int ks, int turn) {
  constexpr int NF = SHAPE == WIDE ? 8 : 4;  // 16-column fragments of a wave
  constexpr int KT = SHAPE == WIDE ? 4 : 3;  // half-tiles of a K-tile: NA of x, then NB of W
  constexpr int NA = SHAPE == FLAT ? 1 : 2, NB = KT - NA, RING = ring(SHAPE);
  constexpr int TN = gated(EPI) ? 64 * NB : 128 * NB;  // output columns per block tile
  constexpr bool GATHER = gathered(EPI);
  const int S = sliced(EPI) ? p.splits : 1, ntn = p.N / TN;
  // (flat: grouped only, the first rows of a segment of 256)
  const int m0 = mt << 8, Mt = p.M - m0 < 256 ? p.M - m0 : 256;
  const int K = p.K, kt0 = ks * (K / BK) / S, nk = (ks + 1) * (K / BK) / S - kt0;
  const int64_t kbase = (int64_t)kt0 * BK;
  const bf16_t* Wb = p.W + kbase;
  if constexpr (grouped(EPI))
    Wb += (int64_t)(p.blk_expert[mt] - p.e_lo) * (gated(EPI) ? 2 * p.N : p.N) * K;

  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = SHAPE == FLAT ? 0 : w >> 1, wc = SHAPE == FLAT ? w : w & 1;
  const int fr = lane & 15, fq = lane >> 4;

  // ---- a bias, and the rows' places in the output, are asked for before the DMAs, which are counted
  constexpr int NG = NF / 2, GU = 64 * NB;
  constexpr int WCOL = (gated(EPI) ? NG : NF) * 16;
  const int f0 = nt * TN + wc * WCOL;
  float4v bg[NG], bu[NG];
  if constexpr (EPI == 7) {
#pragma unroll
    for (int n = 0; n < NG; ++n)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        bg[n][j] = p.bias[f0 + 16 * n + 4 * fq + j];
        bu[n][j] = p.bias[p.N + f0 + 16 * n + 4 * fq + j];
      }
  }
  int place[8];
  if constexpr (EPI == 6) {
#pragma unroll
    for (int m = 0; m < 8; ++m) place[m] = p.sorted[m0 + wr * 128 + 16 * m + fr];
  }

  // ---- DMA sources: instruction i of wave w fills half-tile rows 32w + 8i + lane/8, LDS chunk
  // lane%8 <- global chunk (lane%8) ^ (row & 7)
  const char* base[4];  // A0 A1 B0 B1
  uint32_t vo[4][4];
  const char* va[2][4];  // gathered rows
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    base[h] = (const char*)(p.X + (int64_t)m0 * K + kbase);
    if constexpr (SHAPE != NARROW)
      base[2 + h] = (const char*)(Wb + ((gated(EPI) ? (int64_t)h * p.N + (int64_t)nt * 128
                                                    : (int64_t)nt * 256 + h * 128)) * K);
    else  // one half-tile: gated, 64 rows of the gate's half and (waves 2, 3) 64 of the up's
      base[2] = (const char*)(Wb + (gated(EPI) ? (int64_t)nt * 64 + (w >> 1) * ((int64_t)p.N - 64)
                                               : (int64_t)nt * 128) * K);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = 32 * w + 8 * i + (lane >> 3);
      const uint32_t ch = ((lane & 7) ^ (r & 7)) << 4;
      vo[2 + h][i] = (uint32_t)r * (uint32_t)K * 2u + ch;
      if (h == 1 && NA == 1) continue;
      int ar = h * 128 + r;
      if constexpr (GATHER) {  // the assignment's token row (padding: row 0)
        const int f = p.sorted[m0 + ar];
        va[h][i] = (const char*)(p.X + (int64_t)(f < p.n_assign ? f / p.topk : 0) * K) + ch;
      } else {
        ar = ar < Mt ? ar : Mt - 1;  // rows past the chunk: clamped copies, never stored
        vo[h][i] = (uint32_t)ar * (uint32_t)K * 2u + ch;
      }
    }
  }

  // ---- the ring: half h of K-tile t lies in slot (4t + h) mod 10 (narrow, flat: (3t + h) mod 9),
  // the halves first of which a third is held
  constexpr bool W_AHEAD = SHAPE == WIDE && EPI != 2 && EPI != 3;
  constexpr int SLOT_A = W_AHEAD ? NB * HALF : 0, SLOT_B = W_AHEAD ? 0 : NA * HALF;
  const uint32_t dst0 =
      (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const bf16_t*)lds + 32 * w * 128;
  auto next = [&](int s) __attribute__((always_inline)) {  // a K-tile on
    return s + KT * HALF >= RING ? s + KT * HALF - RING : s + KT * HALF;
  };
  int da = SLOT_A, db = SLOT_B, ka = 0, kb = 0;  // slots and K-tiles to ask for next
  uint32_t qa = 0, qb = 0;                    // of the DMAs under way: LDS address, sources
  const char *pa[2], *pb[2];
  int64_t koff = 0;
  // past the end the last K-tile is loaded again, into slots that nothing reads
  auto set_a = [&]() __attribute__((always_inline)) {
    qa = dst0 + da * 2;
    koff = (int64_t)(gathered(EPI) ? ka ^ turn : ka) * (BK * 2);
    pa[0] = base[0] + koff;
    if constexpr (NA == 2) pa[1] = base[1] + koff;
    ka = ka + 1 < nk ? ka + 1 : nk - 1;
    da = next(da);
  };
  auto set_b = [&]() __attribute__((always_inline)) {
    qb = dst0 + db * 2;
    const int64_t off = (int64_t)(gathered(EPI) ? kb ^ turn : kb) * (BK * 2);
    pb[0] = base[2] + off;
    if constexpr (NB == 2) pb[1] = base[3] + off;
    kb = kb + 1 < nk ? kb + 1 : nk - 1;
    db = next(db);
  };
  auto dma_a = [&](int d) __attribute__((always_inline)) {
    const int h = d >> 2, i = d & 3, off = h * HALF * 2 + i * 1024;
    if constexpr (GATHER) dma16(va[h][i] + koff, qa, off);
    else dma16(vo[h][i], pa[h], qa, off);
  };
  auto dma_b = [&](int d) __attribute__((always_inline)) {
    dma16(vo[2 + (d >> 2)][d & 3], pb[d >> 2], qb, (d >> 2) * HALF * 2 + (d & 3) * 1024);
  };
  // K-tiles 0 and 1, and A or B of 2 (narrow, flat: all of it)
#pragma unroll
  for (int t = 0; t < 3; ++t) {
    if (t < 2 || !W_AHEAD) {
      set_a();
#pragma unroll
      for (int d = 0; d < 4 * NA; ++d) dma_a(d);
    }
    if (t < 2 || W_AHEAD || SHAPE != WIDE) {
      set_b();
#pragma unroll
      for (int d = 0; d < 4 * NB; ++d) dma_b(d);
    }
  }

  // ---- fragments: A rows wr*128 + 16m + fr; B's columns wc*WCOL + 16n + fr, gated those of the
  // gate's part for n < NG and of the up's, GU columns on, for the rest; k chunk 4s + fq of step s
  const bf16_t *fa[2], *fb[2];
  int ra = SLOT_A + wr * HALF, rb = SLOT_B;
  auto set_r = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int at = fr * BK + (((4 * s + fq) ^ (fr & 7)) << 3);
      fa[s] = lds + ra + at;
      fb[s] = lds + rb + wc * WCOL * BK + at;
    }
    ra = next(ra);
    rb = next(rb);
  };
  set_r();
  short8 fx[2][8], fw[2][NF];
  auto read = [&](int set, int s, int j) __attribute__((always_inline)) {  // x 0, all w, x 1..7
    if (j == 0 || j > NF) {
      const int m = j ? j - NF : 0;
      fx[set][m] = *reinterpret_cast<const short8*>(fa[s] + m * 16 * BK);
    } else {
      const int n = j - 1;
      const int at = gated(EPI) ? n / NG * GU * BK + n % NG * 16 * BK : n * 16 * BK;
      fw[set][n] = *reinterpret_cast<const short8*>(fb[s] + at);
    }
  };

  float4v acc[8][NF];  // [m][n]: rows 16m + fr, columns 16n + 4fq + j
  // accumulators settle: a product may be behind them, a read or write of theirs before them
  auto pin = [&]() __attribute__((always_inline)) {
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
#pragma unroll
    for (int i = 0; i < 8 * NF; ++i) asm volatile("" : "+a"(acc[i / NF][i % NF]));
    asm volatile("s_nop 15" ::: "memory");
  };

  // this thread's row scale, ready before the loop
  constexpr bool ROUTED = EPI == 6 || EPI == 8;
  constexpr bool UNSCALED = EPI == 2 || sliced(EPI) || EPI == 5 || EPI == 7 || EPI == 9 || EPI == 10;
  const bool scaled = ROUTED || (!UNSCALED && p.ss_in != nullptr);
  const float own = scaled ? row_scale<EPI>(p, m0, Mt, tid) : 1.f;

  // d: DMA or -1; first: the accumulator's first product
  auto product = [&](int set, int j, int d, bool first) __attribute__((always_inline)) {
    const int m = j / NF, n = (m & 1) ? NF - 1 - j % NF : j % NF;
    if (first) {
      mfma16_first(acc[m][n], fw[set][n], fx[set][m]);
      if (d >= 8) dma_a(d - 8);
      else if (d >= 0) dma_b(d);
    } else if (d < 0) {
      mfma16(acc[m][n], fw[set][n], fx[set][m]);
    } else if (d < 8) {
      mfma16_dma<ONCE>(acc[m][n], fw[set][n], fx[set][m], vo[2 + (d >> 2)][d & 3], pb[d >> 2], qb,
                       (d >> 2) * HALF * 2 + (d & 3) * 1024);
    } else {
      const int h = (d >> 2) - 2, i = d & 3, off = h * HALF * 2 + i * 1024;
      if constexpr (GATHER)
        mfma16_dma(acc[m][n], fw[set][n], fx[set][m], va[h][i] + koff, qa, off);
      else
        mfma16_dma(acc[m][n], fw[set][n], fx[set][m], vo[h][i], pa[h], qa, off);
    }
  };
  // Step s of K-tile t: 8 NF products of 32 k.  FREE: every wave has read the K-tile (its last
  // fragments are asked for by product 30 of step 0, NF 4: 22); its slots take A of t + 2, then,
  // behind LAND, B of t + 3 (not W_AHEAD: B and A; NF 4: B and A of t + 3).  LAND: the loads younger
  // than K-tile t + 1 may be under way (NF 8: B and A of t + 2; NF 4: all of t + 2, 5 of t + 3),
  // K-tile t + 1 is there, and its first fragments are read.
  constexpr int P = 8 * NF, FREE = NF == 8 ? 36 : 26, LAND = NF == 8 ? 12 : 6;
  constexpr int YOUNGER = NF == 8 ? 16 : 17;
  // the DMA behind product j: B's are 0 to 4 NB - 1, A's from 8 on; -1: none
  auto dma_at = [](int s, int j) constexpr {
    if (NF == 8) {
      if (s == 0 && j >= FREE && (j - FREE) % 3 == 0 && (j - FREE) / 3 < 8)
        return (W_AHEAD ? 8 : 0) + (j - FREE) / 3;
      if (s == 1 && j > LAND && (j - LAND) % 6 == 3 && (j - LAND) / 6 < 8)
        return (W_AHEAD ? 0 : 8) + (j - LAND) / 6;
    } else {
      int q = -1;
      if (s == 0 && j >= FREE && (j - FREE) % 2 == 0) q = (j - FREE) / 2;  // 0 to 2
      if (s == 1 && j % 3 == 1 && j < 27) q = 3 + j / 3;
      return q < 4 * NB ? q : 8 + q - 4 * NB;
    }
    return -1;
  };
  // Every fragment asked for is there, and hipcc knows it and puts no waits of its own before the
  // products.  Of those, 26 a K-tile where the first K-tile stands before the loop, and 16 where the loop
  // began with zeroed sums; a wave issues each in 5 clocks (16384 rows, us with 16 / 26 / 3: residual
  // products 861 / 868 / 858, experts' down with places loaded a row at a time 443 / 456, ahead 441).
  auto wait_lds = [] __attribute__((always_inline)) {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
    asm volatile("" ::: "memory");
  };
  auto step = [&](auto SC, auto FIRST) __attribute__((always_inline)) {
    constexpr int s = decltype(SC)::value;
    if (s == 0) wait_lds();
#pragma unroll
    for (int j = 0; j < P; ++j) {
      if (s == 0 && j == FREE) {
        wait_lds();
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
      }
      if (s == 1 && j == LAND) {
        wait_vm<YOUNGER>();
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
      }
      product(s, j, dma_at(s, j), decltype(FIRST)::value);
      if (s == 0 && !(j & 1) && j < 2 * (8 + NF)) read(1, 1, j >> 1);
      if (s == 1 && !(j & 1) && j >= LAND && j < LAND + 2 * (8 + NF)) read(0, 0, (j - LAND) >> 1);
      // addresses of what comes next, between products that hide them
      if (s == 0 && j == FREE - 3) W_AHEAD ? set_a() : set_b();
      if (s == 0 && j == (NF == 8 ? 48 : 29)) set_r();
      if (s == 1 && j == 2) W_AHEAD ? set_b() : set_a();
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  wait_vm<24>();
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int j = 0; j < 8 + NF; ++j) read(0, 0, j);
  step(std::integral_constant<int, 0>{}, std::true_type{});
  step(std::integral_constant<int, 1>{}, std::false_type{});
  for (int t = 1; t < nk; ++t) {
    step(std::integral_constant<int, 0>{}, std::false_type{});
    step(std::integral_constant<int, 1>{}, std::false_type{});
  }
  pin();
  wait_vm<0>();  // the reloads past the end land before LDS is used again, or left

  // ---------------------------------------------------------------- epilogue
  // lane: rows wr*128 + 16m + fr; a pair of 16-column blocks gives it the 16-byte chunk at
  // column 16 (n + (fq & 1)) + 8 (fq >> 1)
  const int row0 = wr * 128 + fr, ccol = 16 * (fq & 1) + 8 * (fq >> 1);
  float* scratch = reinterpret_cast<float*>(lds);
  float rs[8];
  if (scaled) {
    __syncthreads();
    scratch[tid] = own;
    __syncthreads();
#pragma unroll
    for (int m = 0; m < 8; ++m) rs[m] = scratch[row0 + 16 * m];
  } else if constexpr (EPI == 3) {
#pragma unroll
    for (int m = 0; m < 8; ++m) rs[m] = 1.f;
  }
  // a wave issues an instruction in 5 clocks: 256 fewer where rows have no scale
  auto rows = [&](auto put) __attribute__((always_inline)) {
    if (scaled) {
#pragma unroll
      for (int m = 0; m < 8; ++m) put(std::true_type{}, m);
    } else {
#pragma unroll
      for (int m = 0; m < 8; ++m) put(std::false_type{}, m);
    }
  };
  // (the asm keeps hipcc from reading all accumulators ahead of that branch, for both sides)
  auto sums = [&](auto SCALED, int m, int n) __attribute__((always_inline)) {
    float4v v = acc[m][n];
    if constexpr (decltype(SCALED)::value) {
      asm volatile("; scaled" : "+v"(v));
      v *= rs[m];
    } else {
      asm volatile("; plain" : "+v"(v));
    }
    return v;
  };
  bf16_t* out = reinterpret_cast<bf16_t*>(p.out);
  if constexpr (gated(EPI)) {
    // gate (n < NG) and up (n + NG) of features nt*TN + wc*WCOL + 16n + 4fq + j in one lane
    rows([&](auto SCALED, int m) __attribute__((always_inline)) {
      const int r = row0 + 16 * m;
      float4v v[NG];
#pragma unroll
      for (int n = 0; n < NG; ++n) {
        const float4v g = sums(SCALED, m, n), u = sums(SCALED, m, n + NG);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if constexpr (EPI == 7)
            v[n][j] = silu(g[j] + bg[n][j]) * (u[j] + bu[n][j]);
          else if constexpr (EPI == 9)
            v[n][j] = gelu_tanh_(g[j]) * u[j];
          else if constexpr (EPI == 8)
            v[n][j] = clamped_glu(g[j], u[j], p.glu_alpha, p.glu_limit);
          else
            v[n][j] = silu(g[j]) * u[j];
        }
      }
      uint4v c[NG / 2];
#pragma unroll
      for (int n = 0; n < NG; n += 2) c[n / 2] = chunk<EPI>(v[n], v[n + 1]);
      if (r < Mt) {
        bf16_t* o = out + (int64_t)(m0 + r) * p.ldo + f0 + ccol;
#pragma unroll
        for (int n = 0; n < NG; n += 2) *reinterpret_cast<uint4v*>(o + 16 * n) = c[n / 2];
      }
    });
  } else if constexpr (EPI == 2) {
    // residual += tile; the sums of squares of a row's 16-byte chunks meet in pairs: of the two
    // waves, then of a lane, then of its four lanes
    __syncthreads();  // scratch: every wave has left the ring
    float4v* half = reinterpret_cast<float4v*>(scratch);  // [8][wr][64]
    float4v sums[8];
#pragma unroll
    for (int m = 0; m < 8; ++m) {
      const int r = row0 + 16 * m;
      bf16_t* o = out + (int64_t)(m0 + (r < Mt ? r : Mt - 1)) * p.ldo + nt * 256 + wc * 128 + ccol;
      short8 old[4];
#pragma unroll
      for (int n = 0; n < 4; ++n) old[n] = *reinterpret_cast<const short8*>(o + 32 * n);
#pragma unroll
      for (int n = 0; n < 4; ++n) {
        float ss = 0.f;
        const uint4v g = chunk<EPI>(acc[m][2 * n], acc[m][2 * n + 1]);  // rounded, as stored
        uint4v y;
#pragma unroll
        for (int j = 0; j < 8; j += 2) {
          const uint32_t q = g[j >> 1];
          const uint32_t h =
              pack_b2(bf2f((uint16_t)old[n][j]) + __uint_as_float(q << 16),
                      bf2f((uint16_t)old[n][j + 1]) + __uint_as_float(q & 0xffff0000u));
          const float a = __uint_as_float(h << 16), b = __uint_as_float(h & 0xffff0000u);
          ss += a * a;
          ss += b * b;
          y[j >> 1] = h;
        }
        if (r < Mt) *reinterpret_cast<uint4v*>(o + 32 * n) = y;
        sums[m][n] = ss;
      }
      if (wc) half[(m * 2 + wr) * 64 + lane] = sums[m];
    }
    __syncthreads();
    if (!wc) {
#pragma unroll
      for (int m = 0; m < 8; ++m) {
        const float4v v = sums[m] + half[(m * 2 + wr) * 64 + lane];
        float ss = (v[0] + v[2]) + (v[1] + v[3]);
        ss += __shfl_xor(ss, 16, 64);
        ss += __shfl_xor(ss, 32, 64);
        const int r = row0 + 16 * m;
        if (fq == 0 && r < Mt) p.ss_out[(int64_t)(m0 + r) * ntn + nt] = ss;
      }
    }
  } else if constexpr (EPI == 3) {
    // a wave's columns are one head of [q | k | v]; dims d and d + 64 in one lane
    const int head = nt * 2 + wc;
    const bool isq = head < p.hq, isk = !isq && head < p.hq + p.hkv, turn = isq || isk;
    const int kh = isq ? 0 : isk ? head - p.hq : head - p.hq - p.hkv;
#pragma unroll
    for (int m = 0; m < 8; ++m) {
      const int r = row0 + 16 * m, t = m0 + (r < Mt ? r : Mt - 1);
      float4v a[4], b[4];  // rounded first, as the separate kernel's operands are
#pragma unroll
      for (int n = 0; n < 4; ++n) {
        a[n] = round_b(acc[m][n] * rs[m]);
        b[n] = round_b(acc[m][n + 4] * rs[m]);
      }
      if (turn) {
        const float* cs = p.cos_sin + (int64_t)p.positions[t] * 128 + 4 * fq;
#pragma unroll
        for (int n = 0; n < 4; ++n) {
          const float4v c = *reinterpret_cast<const float4v*>(cs + 16 * n);
          const float4v s = *reinterpret_cast<const float4v*>(cs + 64 + 16 * n);
          const float4v x = a[n], y = b[n];
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            a[n][j] = x[j] * c[j] - y[j] * s[j];
            b[n][j] = y[j] * c[j] + x[j] * s[j];
          }
        }
      }
      bf16_t* d = nullptr;
      if (isq) {
        d = out + (int64_t)t * p.ldo + head * 128;
      } else {
        const int64_t slot = p.slots[t];
        if (slot >= 0) {
          const int64_t blk = slot / p.block_size, off = slot - blk * p.block_size;
          d = (isk ? p.k_cache : p.v_cache) + ((blk * p.hkv + kh) * p.block_size + off) * 128;
        }
      }
      const uint4v v0 = chunk<EPI>(a[0], a[1]), v1 = chunk<EPI>(a[2], a[3]);
      const uint4v v2 = chunk<EPI>(b[0], b[1]), v3 = chunk<EPI>(b[2], b[3]);
      if (r < Mt && d) {
        d += ccol;
        *reinterpret_cast<uint4v*>(d) = v0;
        *reinterpret_cast<uint4v*>(d + 32) = v1;
        *reinterpret_cast<uint4v*>(d + 64) = v2;
        *reinterpret_cast<uint4v*>(d + 96) = v3;
      }
    }
  } else if constexpr (EPI == 11) {
    float* slab = reinterpret_cast<float*>(p.out) + (int64_t)ks * p.M * p.N + nt * TN + wc * WCOL;
#pragma unroll
    for (int m = 0; m < 8; ++m) {
      const int r = row0 + 16 * m;
      if (r < Mt)
#pragma unroll
        for (int n = 0; n < NF; ++n)
          *reinterpret_cast<float4v*>(slab + (int64_t)(m0 + r) * p.N + 16 * n + 4 * fq) = acc[m][n];
    }
  } else {
    if constexpr (EPI == 4) out += (int64_t)ks * p.M * p.N;
    rows([&](auto SCALED, int m) __attribute__((always_inline)) {
      const int r = row0 + 16 * m;
      int64_t orow = m0 + r;
      bool live = r < Mt;
      if constexpr (EPI == 6) {  // to the assignment's row
        orow = place[m];
        live = orow < p.n_assign;
      }
      bf16_t* o = out + orow * p.ldo + (int64_t)nt * TN + wc * WCOL + ccol;
      uint4v v[NF / 2];
#pragma unroll
      for (int n = 0; n < NF; n += 2) {
        float4v c = sums(SCALED, m, n), d = sums(SCALED, m, n + 1);
        if constexpr (EPI == 10) {
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            c[j] = gelu_erf16_(c[j]);
            d[j] = gelu_erf16_(d[j]);
          }
        }
        v[n / 2] = chunk<EPI>(c, d);
      }
      if (live) {
#pragma unroll
        for (int n = 0; n < NF; n += 2) *reinterpret_cast<uint4v*>(o + 16 * n) = v[n / 2];
      }
    });
  }
}

// What the first loads need comes as arguments of their own: 14 words that are in registers when a
// wave starts (a struct is loaded from memory).  ONCE: W does not push x out of L2.
template <int EPI, int SHAPE, bool ONCE>
__global__ __launch_bounds__(256, 1) void pgemm_kernel(const bf16_t* X, const bf16_t* W, int M,
                                                       int N, int K, int splits,
                                                       const int* n_blocks, const int* blk_expert,
                                                       const int* sorted, PArgs p) {
  p.X = X, p.W = W, p.M = M, p.N = N, p.K = K, p.splits = splits;
  p.n_blocks = n_blocks, p.blk_expert = blk_expert, p.sorted = sorted;
  __shared__ __attribute__((aligned(1024))) bf16_t lds[ring(SHAPE)];
  constexpr int TN = (gated(EPI) ? 128 : 256) / (SHAPE == NARROW ? 2 : 1);
  constexpr bool MOE = grouped(EPI), CUT = SHAPE == WIDE && cuts(EPI);
  // sliced: the K-slices are extra "m-tiles" of the L2 grouping below (blocks of
  // one slice share its x slice, blocks of one column tile its W rows)
  const int S = sliced(EPI) ? p.splits : 1;
  // MoE: the grid is sized for the worst-case segment count (graph-safe, no host sync); the
  // live tiles are spread over the XCDs, the other blocks leave
  constexpr int WORDS = 4;
  const int lane = threadIdx.x & 63, most = p.M >> 8, ntn = p.N / TN;
  bool light = false, ordered = MOE && SHAPE == WIDE && most <= 64 * WORDS && most * ntn <= 9 * 256;
  // of segments 64 i + lane, asked for beside their number: assignment 128, and whether the segment
  // before is of the same expert
  int half[WORDS], expert[WORDS], last[WORDS];
  if constexpr (MOE && SHAPE == WIDE)
    if (ordered)
#pragma unroll
      for (int i = 0; i < WORDS; ++i)
        if (64 * i < most) {
          const int s = min(64 * i + lane, most - 1);
          half[i] = p.sorted[(int64_t)s * 256 + 128];
          expert[i] = p.blk_expert[s];
          last[i] = p.blk_expert[s ? s - 1 : 0];
        }
  const int mtn1 = MOE ? *p.n_blocks : (p.M + 255) >> 8;
  int heavy_m = mtn1 * S, light_m = 0;  // m-tiles
  // An expert's last segment may have 128 rows or fewer: light, half a tile.  All others come first,
  // so that the last round is of light ones (us before / now, 8 experts of 2048 x 4096: up at 1600
  // tokens of two 136 / 115, 3000 203 / 189, down at 8192 262 / 234, 16384 458 / 421).  Up to 9 rounds:
  // finding them takes 1 us a tile (up at 16384, 16.5 rounds, 893 / 905).
  // Apart from their expert's others they read its weights once more: not from more than a fifth of
  // all on (us without / with: up of 8 x 4096 x 4096 at 2400 tokens of two, 8 of 24 segments, 304 /
  // 383; 8 x 2048 x 6144 at 1300, 8 of 16, 165 / 189; 64 x 2048 x 1024 at 3000 of six, 59 of 123, 226 /
  // 281; 2 of 10 113 / 106, 200 / 198 and, of 4096 x 14336, 545 / 520), but where all tiles are one
  // round and, cut, are not (down of 16 x 2048 x 2048 at 2400, 16 of 32, 58.5 / 51; of 8 x 2048 x 4096
  // at 1000, 4 of 12, all of them cut 60, light ones half as high 63).  Nor where they are few, rounds
  // are few and a tile is soon done (up at 2001, one of 17, 155 / 158; but K = 4096, up of 8 x 4096 x 4096
  // at 1600, one of 16, 250 / 219, down at 4096, three of 35, 268 / 254).  Over 160 such products the rule
  // takes 0.7 % longer than the better of both.
  uint64_t pick[WORDS];
  if constexpr (MOE && SHAPE == WIDE) {
    if (ordered) {
      int full = 0, apart = 0;  // heavy segments, and light ones whose expert has a heavy one
      uint64_t heavy[WORDS];
#pragma unroll
      for (int i = 0; i < WORDS; ++i) {
        heavy[i] = 64 * i < most
                       ? __builtin_amdgcn_ballot_w64(64 * i + lane < mtn1 && half[i] < p.n_assign)
                       : 0;
        full += __popcll(heavy[i]);
        if (64 * i < most)
          apart += __popcll(__builtin_amdgcn_ballot_w64(
              64 * i + lane > 0 && 64 * i + lane < mtn1 && half[i] >= p.n_assign &&
              expert[i] == last[i]));
      }
      ordered = mtn1 * ntn > 128 &&
                (mtn1 * ntn <= 256 ||
                 (5 * apart <= mtn1 &&
                  (p.K >= 4096 || 10 * (mtn1 - full) >= mtn1 || mtn1 * ntn >= 3 * 256)));
      if (ordered) heavy_m = full, light_m = mtn1 - full;
#pragma unroll
      for (int i = 0; i < WORDS; ++i) pick[i] = heavy[i];
    }
  }
  // Wide tiles of a last round that they fill by half or less, with the light ones behind them, are cut
  // in two: two narrow tiles on two CUs take 0.6 of a wide one's time, to the same bits.  us before / now:
  // gated 28672 x 4096 at 600 / 1300 / 2001 rows 168 / 148, 253 / 235, 351 / 329, 16384 x 2048 at 1300 84.1
  // / 77.6; plain 6144 x 4096 at 2600 139 / 126, 2048 x 2048 at 10000 79 / 69; 8 experts of 2048 x 4096, up
  // at 1000 tokens of two 111 / 98, down at 1600 87.5 / 63.2, at 6000 190 / 163.
  const int heavy_t = heavy_m * ntn, light_t = light_m * ntn;
  const int cut = CUT ? cut_tiles(heavy_t, light_t) : 0;
  int b = blockIdx.x, part = -1, bid, mtn = heavy_m;
  if (b < heavy_t - cut) {
    bid = xcd_remap(b, heavy_t - cut);
  } else if (b < heavy_t + cut) {
    b = xcd_remap(b - (heavy_t - cut), 2 * cut);
    bid = heavy_t - cut + (b >> 1);
    part = b & 1;
  } else {
    if (b >= heavy_t + cut + light_t) return;
    bid = xcd_remap(b - heavy_t - cut, light_t);
    light = true;
    mtn = light_m;
    if constexpr (MOE && SHAPE == WIDE)
#pragma unroll
      for (int i = 0; i < WORDS; ++i)
        pick[i] = __builtin_amdgcn_ballot_w64(64 * i + lane < mtn1) & ~pick[i];
  }
  const int64_t w_rows = gated(EPI) ? 2 * p.N : p.N;
  const int gm = w_rows * p.K > (1 << 26) ? 8 : 4;  // 128 MB of W
  const int per_group = gm * ntn;
  const int grp = bid / per_group, gm0 = grp * gm;
  const int gsz = mtn - gm0 < gm ? mtn - gm0 : gm;
  const int idx = bid - grp * per_group;
  const int vmt = gm0 + idx % gsz, nt = idx / gsz;
  const int ks = vmt / mtn1;
  int mt = vmt - ks * mtn1;
  if constexpr (MOE && SHAPE == WIDE) {
    if (ordered) {  // the mt-th of the picked segments
      int before = 0, seg = 0;
#pragma unroll
      for (int i = 0; i < WORDS; ++i) {
        const int rank = before + __popcll(pick[i] & ((1ull << lane) - 1));
        const uint64_t hit = __builtin_amdgcn_ballot_w64((pick[i] >> lane & 1) && rank == mt);
        if (hit) seg = 64 * i + __builtin_ctzll(hit);
        before += __popcll(pick[i]);
      }
      mt = seg;
    }
  }
  // Experts' rows of 4 KB of W, of which all blocks would ask for the same 128 bytes at a time, and so
  // for a few memory channels: eight column tiles, whose blocks share x in an XCD, walk K in an order of
  // their own, with the bits of their number reversed, so that neighbours are far apart.  The order follows
  // the weights' place alone, the expert's own number and the column tile's, so that a row's bits depend
  // neither on the rows beside it nor on the experts that a rank has.  us, up products in order / apart: 8
  // experts of 2048 x 4096 at 600 / 1000 / 2001 tokens of two 83 / 68, 107 / 92, 168 / 143; 16 of 2048 x 2048
  // at 2400 140 / 121; 64 of 2048 x 1024 at 3000 of six 229 / 230; of more than three rounds of tiles, which
  // are apart by themselves, 8 of 2048 x 4096 at 4000 / 8000 / 16384 250 / 252, 460 / 452, 909 / 912.
  // Rows of 2 and 8 KB gain nothing (8 experts of 1024 x 2048 at 2001 48.5 / 49.5, of 1024 x 4096 83.4 / 85.1,
  // of 4096 x 1024 81.1 / 80.4, of 4096 x 2048 145 / 146, 32 of 1024 x 1024 at 2001 of four 57.8 / 63.2; 8 of
  // 4096 x 14336 at 1001 506 / 514), nor do those of the down product (2048 x 4096 at 2001 79 / 78).
  int turn = 0;
  if constexpr (gathered(EPI)) {
    constexpr int PART = SHAPE == NARROW ? 2 : 1;  // of a wide column tile
    const int octets = (ntn / PART + 7) >> 3;
    if (p.K == 32 * BK)
      turn = (int)(__builtin_bitreverse32(nt / PART / 8 + octets * p.blk_expert[mt]) >> 27);
  }
  if constexpr (MOE && SHAPE == WIDE)
    if (light) {
      tile<EPI, FLAT>(p, lds, mt, nt, 0, turn);
      return;
    }
  if constexpr (CUT)
    if (part >= 0) {
      tile<EPI, NARROW>(p, lds, mt, 2 * nt + part, ks, turn);
      return;
    }
  tile<EPI, SHAPE, ONCE>(p, lds, mt, nt, ks, turn);
}

template <int EPI, int SHAPE, bool ONCE = false>
void launch(const PArgs& a, dim3 grid, hipStream_t s) {
  pgemm_kernel<EPI, SHAPE, ONCE><<<grid, 256, 0, s>>>(a.X, a.W, a.M, a.N, a.K, a.splits, a.n_blocks,
                                                      a.blk_expert, a.sorted, a);
}
// Narrow tiles of one m-tile, and of two whose second is more than half full, so that both read W
// together, ask for it past the caches' order of use: us in order / past it, gated 28672 x 4096 at 224 / 256
// rows 67.4 / 61.3, 64.6 / 61.8, 22016 x 4096 at 256 58.7 / 56.5, 16384 x 4096 at 256 / 512 55.4 / 53.8, 61.0
// / 60.4, 16384 x 2048 at 256 / 512 29.8 / 30.0, 32.7 / 32.2, 14336 x 2048 28.9 / 29.4, 30.5 / 30.8, 16384 x
// 1024 at 512 19.6 / 19.1; over 17 sizes at 400 and 512 rows 0.98 to 1.04, 1.2 % faster.  A second m-tile of few
// rows is ahead, and W is read twice (at 257 15360 x 2560 36.5 / 44.4, 16384 x 5120 73.4 / 86.0, 4096 x 14336
// 135 / 179); so do more rows (plain 4096 x 2048 at 1999 31.7 / 33.6) and more rounds (the wide tile, gated
// 28672 x 4096 at 8192 1248 / 1288).  Not beside fp32 slabs (2560 x 10240 in 5 at 257 / 512 30.6 / 35.3, 36.1 /
// 39.1, 4096 x 14336 in 4 53.8 / 59.9, 60.3 / 61.3, 4096 x 8192 34.3 / 33.5, 37.0 / 37.9; 2048 x 8192 in 8
// would gain, 24.3 / 22.0, 23.3 / 23.1); fp16 ones are of one m-tile (4096 x 14336 in 8 at 224 / 256 36.4 /
// 37.5, 37.9 / 36.7).
template <int EPI>
void launch_narrow(const PArgs& a, dim3 grid, hipStream_t s) {
  if constexpr (EPI != 11)
    if (a.M <= 256 || (a.M > 384 && a.M <= 512)) {
      launch<EPI, NARROW, true>(a, grid, s);
      return;
    }
  launch<EPI, NARROW>(a, grid, s);
}

// out = X . W^T on tiles of 128 x 128, a wave 64 x 64 of them, for steps whose larger tiles are half a
// round or less: us, library / here and narrow tile, 2048 x 2048 at 2001 rows 21.7 / 19.0 and 24.2, 4096
// x 2048 at 999 24.6 / 21.2 and 28.7, 3072 x 1024 at 999 14.3 / 11.6 and 15.2 (ops.small_tile_cols).  A K-tile
// is a half-tile of each operand in a ring of five, 128 KB in flight; its 32 products a wave take half of
// the 0.42 us of its intake (78 GB/s a CU), so one barrier a K-tile does: every wave has read K-tile t,
// and t + 1 has landed.
// NF 2: 128 x 64, a wave 64 x 32, in a ring of six (2048 x 2048 at 999 rows 14.6, NF 4 18.5, library 17.3; 2048
// x 4096 24.6, 31.5, 27.7; 2048 x 1024 9.5, 11.5, 11.8).
template <int NF>
__global__ __launch_bounds__(256, 1) void pgemm_small_kernel(bf16_t* out, const bf16_t* X,
                                                             const bf16_t* W, int M, int N, int K,
                                                             int64_t ldo) {
  constexpr int MF = 4, TN = 32 * NF, L = 4 + NF;  // fragments of a wave; DMAs of one a K-tile
  constexpr int DEPTH = NF == 4 ? 5 : 6, STAGE = HALF + TN * BK, RING = DEPTH * STAGE;
  __shared__ __attribute__((aligned(1024))) bf16_t lds[RING];
  const int ntn = N / TN, mtn = (M + 127) >> 7, nk = K / BK;
  const int bid = xcd_remap(blockIdx.x, mtn * ntn), per_group = 4 * ntn;
  const int grp = bid / per_group, gsz = mtn - 4 * grp < 4 ? mtn - 4 * grp : 4;
  const int idx = bid - grp * per_group, mt = 4 * grp + idx % gsz, nt = idx / gsz;
  const int m0 = mt << 7, Mt = M - m0 < 128 ? M - m0 : 128;
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = w >> 1, wc = w & 1, fr = lane & 15, fq = lane >> 4;

  // ---- DMAs, as in tile(): a wave's of x 32 rows, of W 8 NF
  const char* xb = (const char*)(X + (int64_t)m0 * K);
  const char* wb = (const char*)(W + (int64_t)nt * TN * K);
  uint32_t vx[4], vw[NF];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = 32 * w + 8 * i + (lane >> 3);
    vx[i] = (uint32_t)(r < Mt ? r : Mt - 1) * (uint32_t)K * 2u + (((lane & 7) ^ (r & 7)) << 4);
  }
#pragma unroll
  for (int i = 0; i < NF; ++i) {
    const int r = 8 * (NF * w + i) + (lane >> 3);
    vw[i] = (uint32_t)r * (uint32_t)K * 2u + (((lane & 7) ^ (r & 7)) << 4);
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const bf16_t*)lds;
  const uint32_t dx = lds0 + 32 * w * 128, dw = lds0 + HALF * 2 + 8 * NF * w * 128;
  auto next = [](int s) { return s + STAGE == RING ? 0 : s + STAGE; };
  int ds = 0, kt = 0;
  uint32_t ax = 0, aw = 0;
  const char *px = xb, *pw = wb;
  auto set = [&]() __attribute__((always_inline)) {  // past the end the last K-tile again
    ax = dx + ds * 2;
    aw = dw + ds * 2;
    px = xb + (int64_t)kt * (BK * 2);
    pw = wb + (int64_t)kt * (BK * 2);
    kt = kt + 1 < nk ? kt + 1 : nk - 1;
    ds = next(ds);
  };
  auto dma = [&](int d) __attribute__((always_inline)) {
    if (d < 4) dma16(vx[d], px, ax, d * 1024);
    else dma16(vw[d - 4], pw, aw, (d - 4) * 1024);
  };
#pragma unroll
  for (int t = 0; t < DEPTH; ++t) {
    set();
#pragma unroll
    for (int d = 0; d < L; ++d) dma(d);
  }

  int rs = 0;
  const bf16_t *fa[2], *fb[2];
  auto set_r = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int o = rs + fr * BK + (((4 * s + fq) ^ (fr & 7)) << 3);
      fa[s] = lds + o + wr * 64 * BK;
      fb[s] = lds + o + HALF + wc * 16 * NF * BK;
    }
    rs = next(rs);
  };
  short8 fx[2][MF], fw[2][NF];
  auto read = [&](int s, int j) __attribute__((always_inline)) {
    if (j < MF) fx[s][j] = *reinterpret_cast<const short8*>(fa[s] + j * 16 * BK);
    else fw[s][j - MF] = *reinterpret_cast<const short8*>(fb[s] + (j - MF) * 16 * BK);
  };
  auto wait_lds = [] __attribute__((always_inline)) {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
    asm volatile("" ::: "memory");
  };
  float4v acc[MF][NF];  // [m][n]: rows 16m + fr, columns 16n + 4fq + j
  auto k_tile = [&](auto FIRST) __attribute__((always_inline)) {
    wait_lds();
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      if (s) {
        wait_lds();
        wait_vm<(DEPTH - 2) * L>();
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        set();
        set_r();
      }
#pragma unroll
      for (int j = 0; j < MF * NF; ++j) {
        const int m = j / NF, n = (m & 1) ? NF - 1 - j % NF : j % NF;
        if (decltype(FIRST)::value && !s) mfma16_first(acc[m][n], fw[s][n], fx[s][m]);
        else mfma16(acc[m][n], fw[s][n], fx[s][m]);
        // L reads, and L DMAs behind them
        const int rd = NF == 4 ? (j & 1 ? -1 : j >> 1) : j < L ? j : -1;
        const int dm = NF == 4 ? (j & 1 ? j >> 1 : -1) : j - (MF * NF - L);
        if (rd >= 0) read(1 - s, rd);
        if (s && dm >= 0) dma(dm);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  wait_vm<(DEPTH - 1) * L>();
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  set_r();
#pragma unroll
  for (int j = 0; j < L; ++j) read(0, j);
  k_tile(std::true_type{});
  for (int t = 1; t < nk; ++t) k_tile(std::false_type{});
  asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
#pragma unroll
  for (int i = 0; i < MF * NF; ++i) asm volatile("" : "+a"(acc[i / NF][i % NF]));
  asm volatile("s_nop 15" ::: "memory");
  wait_vm<0>();  // the reloads past the end land before LDS is left

  const int ccol = 16 * (fq & 1) + 8 * (fq >> 1);
#pragma unroll
  for (int m = 0; m < MF; ++m) {
    const int r = wr * 64 + 16 * m + fr;
    uint4v v[NF / 2];
#pragma unroll
    for (int n = 0; n < NF; n += 2) v[n / 2] = chunk<0>(acc[m][n], acc[m][n + 1]);
    if (r < Mt) {
      bf16_t* o = out + (int64_t)(m0 + r) * ldo + nt * TN + wc * 16 * NF + ccol;
#pragma unroll
      for (int n = 0; n < NF; n += 2) *reinterpret_cast<uint4v*>(o + 16 * n) = v[n / 2];
    }
  }
}

// one workgroup (256 threads) per row: ss[r] = sum(x[r]^2) (layer-0 input of the
// folded-norm prefill path: the embedding rows have no producer epilogue)
__global__ __launch_bounds__(256) void row_sumsq_kernel(float* __restrict__ ss,
                                                        const bf16_t* __restrict__ x, int d,
                                                        int64_t stride) {
  __shared__ float red[4];
  const bf16_t* row = x + (int64_t)blockIdx.x * stride;
  float t = 0.f;
  for (int c = threadIdx.x * 8; c < d; c += 256 * 8) {
    const short8 v = *reinterpret_cast<const short8*>(row + c);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float f = bf2f((uint16_t)v[j]);
      t += f * f;
    }
  }
  t = block_sum(t, red);
  if (threadIdx.x == 0) ss[blockIdx.x] = t;
}

}  // namespace

extern "C" {

// Returns 0 on success, < 0 for a shape / argument the kernel does not cover
// (checked BEFORE any launch).
int omnia_pgemm_splitk(void* parts, const void* X, const void* W, int M, int N, int K, int S,
                       int cols, int f32, int uneven, hipStream_t s);
int omnia_pgemm_moe(int mode, void* out, const void* A, const void* W, const int* sorted,
                    const int* blk_expert, const int* n_blocks, const float* route_w, int K,
                    int N, int topk, int n_assign, int e_lo, int max_blocks, float alpha,
                    float limit, int cols, hipStream_t s);

int omnia_pgemm(int epi, void* out, const void* X, const void* W, int M, int N, int K, int ldo,
                const float* ss_in, int ss_in_n, float inv_d, float eps, float* ss_out,
                const int* positions, const float* cos_sin, void* k_cache, void* v_cache,
                const int64_t* slots, int hq, int hkv, int block_size, const float* bias,
                int gelu, int cols, hipStream_t s) {
  if (epi < 0 || epi > 3) return -1;
  if (cols && cols != 128 && cols != 256) return -16;
  const bool narrow = cols == 128;
  if (narrow && epi > 1) return -16;
  if (bias && (epi != 1 || ss_in)) return -14;
  if (gelu && (epi != 1 || ss_in || bias)) return -15;
  if (M < 1) return -2;
  if (K <= 0 || K % (2 * BK)) return -3;
  const int tn = (epi == 1 ? 128 : 256) >> (narrow ? 1 : 0);
  if (N <= 0 || N % tn) return -4;
  if ((reinterpret_cast<uintptr_t>(X) | reinterpret_cast<uintptr_t>(W) |
       reinterpret_cast<uintptr_t>(out)) & 15)
    return -5;
  if (ldo % 8 || ldo < (epi == 3 ? hq * 128 : N)) return -6;
  if (ss_in != nullptr && ss_in_n < 1) return -7;
  if (epi == 2 && ss_out == nullptr) return -8;
  if (epi == 3) {
    if (!positions || !cos_sin || !k_cache || !v_cache || !slots || block_size < 1) return -9;
    // the epilogue works per head (a 256-column tile = heads 2nt, 2nt+1 of
    // [q | k | v]), so a tile may straddle the q / k / v boundaries: a TP shard's
    // single KV head (hkv * 128 = 128, Llama-3-70B at TP = 8) is fine
    if (hq < 1 || hkv < 1 || (hq + 2 * hkv) % 2) return -10;
    if (N != (hq + 2 * hkv) * 128) return -11;
    if ((reinterpret_cast<uintptr_t>(k_cache) | reinterpret_cast<uintptr_t>(v_cache)) & 15)
      return -12;
  }
  const int64_t blocks = (int64_t)((M + 255) / 256) * (N / tn);
  if (blocks > (1 << 30)) return -13;
  PArgs a{out, (const bf16_t*)X, (const bf16_t*)W, M, N, K, ldo, ss_in, ss_in_n, inv_d, eps,
          ss_out, positions, cos_sin, (bf16_t*)k_cache, (bf16_t*)v_cache, slots, hq, hkv,
          block_size, 1, nullptr, nullptr, nullptr, nullptr, 0, 0, 0, bias};
  const dim3 grid((unsigned)(blocks + (narrow || !cuts(epi) ? 0 : cut_tiles((int)blocks, 0))));
#define OMNIA_PGEMM(EPI)                                       \
  do {                                                         \
    if (narrow)                                                \
      launch_narrow<EPI>(a, grid, s);             \
    else                                                       \
      launch<EPI, WIDE>(a, grid, s);            \
    return (int)hipGetLastError();                             \
  } while (0)
  if (bias) OMNIA_PGEMM(7);
  if (gelu) OMNIA_PGEMM(9);
  switch (epi) {
    case 0: OMNIA_PGEMM(0);
    case 1: OMNIA_PGEMM(1);
#undef OMNIA_PGEMM
    case 2: launch<2, WIDE>(a, grid, s); break;
    default: launch<3, WIDE>(a, grid, s); break;
  }
  return (int)hipGetLastError();
}

// split-K GEMM: parts[S][M][N] fp16 or fp32, sum over s of parts[s] = X . W^T (EPI 4, 11).
// cols: of a tile, 128 or 256 (0).  uneven: slices of any whole K-tiles, as alike as they can be
// (ops.midm_slices); else all of the same number, an even one.
int omnia_pgemm_splitk(void* parts, const void* X, const void* W, int M, int N, int K, int S,
                       int cols, int f32, int uneven, hipStream_t s) {
  if (cols && cols != 128 && cols != 256) return -16;
  const int tn = cols == 128 ? 128 : 256;
  if (M < 1 || S < 1 || S > 16) return -1;
  if (K <= 0) return -3;
  if (uneven ? K % BK || K / BK < S : K % S || (K / S) % (2 * BK)) return -3;
  if (N <= 0 || N % tn) return -4;
  if ((reinterpret_cast<uintptr_t>(X) | reinterpret_cast<uintptr_t>(W) |
       reinterpret_cast<uintptr_t>(parts)) & 15)
    return -5;
  const int64_t blocks = (int64_t)((M + 255) / 256) * (N / tn) * S;
  if (blocks > (1 << 30)) return -13;
  PArgs a{parts, (const bf16_t*)X, (const bf16_t*)W, M, N, K, N, nullptr, 0, 0.f, 0.f, nullptr,
          nullptr, nullptr, nullptr, nullptr, nullptr, 0, 0, 0, S, nullptr, nullptr, nullptr,
          nullptr, 0, 0, 0};
  const dim3 grid((unsigned)blocks);
  if (f32 && tn == 128)
    launch_narrow<11>(a, grid, s);
  else if (f32)
    launch<11, WIDE>(a, grid, s);
  else if (tn == 128)
    launch_narrow<4>(a, grid, s);
  else
    launch<4, WIDE>(a, grid, s);
  return (int)hipGetLastError();
}

// MoE grouped GEMMs on the 256x256 tile (segments from omnia_moe_align with
// bm = 256).  mode 0: act [max_blocks*256, I] = SwiGLU(x[token] . W_gu[e]^T),
// x [T, d], W_gu [E_loc, 2I, d];  mode 1: Y[assignment] = w_route * act . W_dn[e]^T,
// act [max_blocks*256, I], W_dn [E_loc, d, I], Y [n_assign, d] (w_route null: 1);  mode 2:
// mode 0 with the clamped GLU (alpha, limit) of the weighted input;  mode 3: mode 0
// ungated, gelu(x . W^T), W [E_loc, I, d].  cols: of a tile, 256 (0) or 128; up products gain nothing
// on the narrow one (1600 tokens of two, 8 experts of 2048 x 4096, 136 / 149 us), which knows no light
// segments: tests compare those of the wide one with it.
int omnia_pgemm_moe(int mode, void* out, const void* A, const void* W, const int* sorted,
                    const int* blk_expert, const int* n_blocks, const float* route_w, int K,
                    int N, int topk, int n_assign, int e_lo, int max_blocks, float alpha,
                    float limit, int cols, hipStream_t s) {
  if (mode < 0 || mode > 3 || max_blocks < 0 || topk < 1) return -1;
  if (cols && cols != 128 && cols != 256) return -16;
  const bool narrow = cols == 128;
  const int tn = (mode == 0 || mode == 2 ? 128 : 256) >> (narrow ? 1 : 0);
  if (K <= 0 || K % (2 * BK)) return -3;
  if (N <= 0 || N % tn) return -4;
  if ((reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(W) |
       reinterpret_cast<uintptr_t>(out)) & 15)
    return -5;
  if (!sorted || !blk_expert || !n_blocks || (mode == 2 && !route_w)) return -9;
  if (max_blocks == 0) return 0;
  const int64_t blocks = (int64_t)max_blocks * (N / tn);
  if (blocks > (1 << 30)) return -13;
  PArgs a{out, (const bf16_t*)A, (const bf16_t*)W, max_blocks * 256, N, K, N, nullptr, 0, 0.f,
          0.f, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, 0, 0, 0, 1, sorted,
          blk_expert, n_blocks, route_w, topk, n_assign, e_lo, nullptr, alpha, limit};
  const dim3 grid((unsigned)(blocks + (narrow ? 0 : 128)));  // (128: the most that are cut)
#define OMNIA_PGEMM(EPI)                            \
  do {                                              \
    if (narrow)                                     \
      launch<EPI, NARROW>(a, grid, s); \
    else                                            \
      launch<EPI, WIDE>(a, grid, s); \
    return (int)hipGetLastError();                  \
  } while (0)
  if (mode == 0) OMNIA_PGEMM(5);
  if (mode == 1) OMNIA_PGEMM(6);
  if (mode == 2) OMNIA_PGEMM(8);
  OMNIA_PGEMM(10);
#undef OMNIA_PGEMM
}

// out[M, N] = X . W^T on tiles of 128 x cols (128 or 64)
int omnia_pgemm_small(void* out, const void* X, const void* W, int M, int N, int K, int cols,
                      hipStream_t s) {
  if (cols != 64 && cols != 128) return -16;
  if (M < 1) return -2;
  if (K <= 0 || K % BK || K > (1 << 23)) return -3;
  if (N <= 0 || N % cols) return -4;
  if ((reinterpret_cast<uintptr_t>(X) | reinterpret_cast<uintptr_t>(W) |
       reinterpret_cast<uintptr_t>(out)) & 15)
    return -5;
  const int64_t blocks = (int64_t)((M + 127) / 128) * (N / cols);
  if (blocks > (1 << 30)) return -13;
  const auto kernel = cols == 128 ? pgemm_small_kernel<4> : pgemm_small_kernel<2>;
  kernel<<<(unsigned)blocks, 256, 0, s>>>((bf16_t*)out, (const bf16_t*)X, (const bf16_t*)W, M, N, K,
                                          N);
  return (int)hipGetLastError();
}

int omnia_row_sumsq(float* ss, const void* x, int rows, int d, int64_t stride, hipStream_t s) {
  if (d % 8 || rows < 0) return -1;
  if (rows == 0) return 0;
  row_sumsq_kernel<<<rows, 256, 0, s>>>(ss, (const bf16_t*)x, d, stride);
  return (int)hipGetLastError();
}

}  // extern "C"
