// Projections of a few rows on gfx950: out[M, N] = x[M, K] . W[N, K]^T for M <= 16, bf16 in,
// fp32 MFMA accumulate, with the work that follows in the epilogue.
//
// At these sizes a projection reads its weights once and does little else, and a model step
// is a chain of them: what counts is how fast a short read gets going, and how many launches
// stand between two of them.
//   * A block of 8 waves owns 16, 32 or 64 weight rows (NW = 1, 2, 4) over the whole of K; the
//     waves take turns at 64-k chunks, so together they read one contiguous KB of every row at a
//     time, and meet once, in LDS, at the end.  No slabs, no second kernel, no atomics, a fixed
//     order of sums.
//   * Weights go from HBM to MFMA operand registers; x comes from L2, as it is shared by all
//     blocks.
//   * Row-major weights reach a CU in 64-byte pieces of 16 rows; PK weights (a copy laid out
//     [row / 16][k / 64][k / 32][k / 8][row % 16][8], ops.stream_pack) as one KB a wave
//     instruction: 28672 x 4096 at one row 40.9 us row-major, 37.9 packed; 4096 x 14336 24.5
//     and 20.9.  Streaming loads (nt) help packed reads (41.7 -> 37.9) and hurt row-major ones.
//   * A ring of D chunks a wave is in flight from the first instruction on: 64 or 128 KB of
//     weights a block (NW = 1, 2) and two blocks a CU, or 192 KB (NW = 4) and one.
//   * NORM: x is the residual, whose rows are RMS-normed (the norm's weight is folded into W)
//     and rounded to bf16 as they become operands, as a norm kernel would: no launch, no pass.
//     The rows' sums of squares come from the kernel that wrote the residual (EPI 2).
// Epilogues:
//   EPI 0   out = acc
//   EPI 1   out = act(g + b) * (u + b), W = [Wg; Wu], act silu or gelu (tanh form), b or none
//   EPI 2   residual += acc, in place; sums of squares of its new rows, one per block
//   EPI 3   QKV: rotated q to out, rotated k and v to the paged cache
// and of experts, whose rows are expert-sorted assignments in segments of 16:
//   EPI 5   silu GLU;  EPI 8  clamped GLU of the weighted input;  EPI 10  ungated gelu (erf)
//   EPI 6   down projection, weighted (if asked) and written to the assignment's row
#include "common.h"

using namespace omnia;

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int WAVES = 8;

__device__ __forceinline__ float4v mfma16(short8 a, short8 b, float4v c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

struct StreamArgs {
  void* out;         // EPI 2: the residual; EPI 3: q
  const bf16_t* x;   // [M, ldx]; EPI 6: activations in sorted order
  const bf16_t* w;   // [N, K], gated [2N, K]; experts: [E, ..., K]
  int M, N, K;
  int64_t ldx, ldo;
  const float* ss_in;  // NORM: [M, n_ss] partial sums of squares of the rows of x
  int n_ss;
  float inv_d, eps;
  float* ss_out;       // EPI 2: [M, blocks]
  const float* bias;  // EPI 0: [N], EPI 1: [2N], or null
  int gelu;
  const int* positions;  // EPI 3
  const float* cos_sin;  // [positions, 128] = cos[64] | sin[64]
  bf16_t *k_cache, *v_cache;  // [pages, hkv, page, 128]
  const int64_t* slots;       // < 0: no write
  int hq, hkv, page;
  const int *sorted, *blk_expert, *n_blocks;  // experts
  const int* ids;  // the assignments' experts instead, up to 64
  int e_hi;
  const float* route_w;
  int topk, n_assign, e_lo;
  float alpha, limit;
};

constexpr bool gated(int epi) { return epi == 1 || epi == 5 || epi == 8; }
constexpr bool paired(int epi) { return gated(epi) || epi == 3; }
constexpr bool grouped(int epi) { return epi >= 5; }

// D: chunks in flight of 1 + NW operand fragments, 8 registers each.  What the first loads need
// comes as arguments of their own, 14 words that are in registers when a wave starts (a struct is
// loaded from memory): i0 .. of experts e_lo, e_hi, n_assign and topk, else M and n_ss.
template <int NW, int EPI, bool NORM, bool PK>
__global__ __launch_bounds__(64 * WAVES, NW <= 2 ? 4 : 2) void stream_kernel(
    const bf16_t* x, const bf16_t* w, int64_t ldx, const void* first, int N, int K_, int i0, int i1,
    int i2, int i3, StreamArgs p) {
  p.x = x, p.w = w, p.ldx = ldx, p.N = N, p.K = K_;
  if constexpr (grouped(EPI)) {
    p.ids = reinterpret_cast<const int*>(first);
    p.e_lo = i0, p.e_hi = i1, p.n_assign = i2, p.topk = i3;
  } else {
    p.ss_in = reinterpret_cast<const float*>(first);
    p.M = i0, p.n_ss = i1;
  }
  constexpr int D = NW <= 2 ? 4 : 3, F = 8 * NW;  // F: features of a paired block
  __shared__ __attribute__((aligned(16))) float red[WAVES * NW * 256];
  __shared__ float rsl[NORM ? 16 : 1];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fr = lane & 15, fq = lane >> 4, unit = blockIdx.x;
  const int K = p.K;

  const bf16_t* wbase = p.w;
  int seg = 0, assigned = 0;  // assignment of the segment's row fr
  __shared__ int rows[grouped(EPI) ? 16 : 1];
  if constexpr (grouped(EPI)) {
    seg = blockIdx.y;  // the grid holds the most segments there can be
    int e = p.e_lo;
    if (p.ids) {  // a wave sorts up to 64 assignments by itself: a lane each
      const int id = lane < p.n_assign ? p.ids[lane] : -1;
      uint64_t in = 0;
      int at = seg;  // segment of expert e
      for (;; ++e) {
        if (e == p.e_hi) return;
        in = __builtin_amdgcn_ballot_w64(id == e);
        const int segs = (__builtin_popcountll(in) + 15) >> 4;
        if (at < segs) break;
        at -= segs;
      }
      const int rank = __builtin_popcountll(in & ((1ull << lane) - 1)) - 16 * at;
      const bool mine = id == e && rank >= 0 && rank < 16;
      // each lane's number + 1 to its row's lane (others to lane 32), 0 where no row is
      const int got = __builtin_amdgcn_ds_permute(4 * (mine ? rank : 32), lane + 1);
      assigned = __shfl(got ? got - 1 : p.n_assign, fr, 64);
    } else {
      if (seg >= *p.n_blocks) return;
      e = p.blk_expert[seg];
      assigned = p.sorted[seg * 16 + fr];
    }
    if (lane < 16) rows[lane] = assigned;  // the same from every wave
    wbase += (int64_t)(e - p.e_lo) * (gated(EPI) ? 2 * p.N : p.N) * K;
  }
  // weight row of the block's row rr: halves of a pair are F rows apart in the block
  auto wrow = [&](int rr) -> int64_t {
    if constexpr (gated(EPI))
      return rr < F ? (int64_t)unit * F + rr : (int64_t)p.N + (int64_t)unit * F + rr - F;
    if constexpr (EPI == 3) {
      const int per = 64 / F, head = unit / per, d0 = (unit - head * per) * F;
      return (int64_t)head * 128 + (rr < F ? d0 + rr : 64 + d0 + rr - F);
    }
    return (int64_t)unit * 16 * NW + rr;
  };
  const bf16_t* wp[NW];
#pragma unroll
  for (int j = 0; j < NW; ++j) {
    const int64_t r = wrow(16 * j + fr);
    wp[j] = wbase + (PK ? (r >> 4) * 16 * K + 128 * fq + 8 * (r & 15) : r * K + 8 * fq);
  }
  int64_t xrow;
  if constexpr (grouped(EPI) && EPI != 6) {
    xrow = assigned < p.n_assign ? assigned / p.topk : 0;  // padding: any row, never written
  } else if constexpr (EPI == 6) {
    xrow = seg * 16 + fr;
  } else {
    xrow = fr < p.M ? fr : p.M - 1;
  }
  const bf16_t* xp = p.x + xrow * p.ldx + 8 * fq;

  // row sums of squares: requested before anything else, needed after the weights are on
  // their way
  constexpr int RW = 16 / WAVES;  // rows of a wave
  float sv[NORM ? RW : 1][4];
  if constexpr (NORM) {
#pragma unroll
    for (int r = 0; r < RW; ++r) {
      const int row = wv + WAVES * r < p.M ? wv + WAVES * r : p.M - 1;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int o = lane + 64 * t;
        const float v = p.ss_in[(int64_t)row * p.n_ss + (o < p.n_ss ? o : 0)];
        sv[r][t] = o < p.n_ss ? v : 0.f;
      }
    }
  }

  const int nch = K >> 6, n = (nch - wv + WAVES - 1) / WAVES;  // this wave's chunks
  short8 wr[D][NW][2], xr[D][2];
  auto load = [&](auto& w, auto& x, int i) {
    const int c = wv + WAVES * i;
    const int64_t o = (int64_t)(c < nch ? c : nch - 1) * 64, ow = PK ? 16 * o : o;
#pragma unroll
    for (int j = 0; j < NW; ++j)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const short8* v = reinterpret_cast<const short8*>(wp[j] + ow + (PK ? 512 : 32) * h);
        w[j][h] = PK ? __builtin_nontemporal_load(v) : *v;
      }
#pragma unroll
    for (int h = 0; h < 2; ++h) x[h] = *reinterpret_cast<const short8*>(xp + o + 32 * h);
  };
  float4v acc[NW];
  float rs = 1.f;
#pragma unroll
  for (int j = 0; j < NW; ++j) acc[j] = {0.f, 0.f, 0.f, 0.f};
  auto compute = [&](auto& w, auto& x) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      short8 a = x[h];
      if constexpr (NORM) {
        bf16x8 y;
#pragma unroll
        for (int e = 0; e < 8; ++e) y[e] = (__bf16)(bf2f((uint16_t)a[e]) * rs);
        a = __builtin_bit_cast(short8, y);
      }
#pragma unroll
      for (int j = 0; j < NW; ++j) acc[j] = mfma16(a, w[j][h], acc[j]);
    }
  };
  // Loads are unconditional (past the end: the last chunk again) and stay where they are
  // written, so that every wait counts the loads behind it instead of draining them.
#pragma unroll
  for (int d = 0; d < D; ++d) load(wr[d], xr[d], d);
  if constexpr (NORM) {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int r = 0; r < RW; ++r) {
      const int row = wv + WAVES * r;
      float v = sv[r][0] + sv[r][1] + sv[r][2] + sv[r][3];
      if (p.n_ss > 256 && row < p.M)
        for (int o = 256 + lane; o < p.n_ss; o += 64) v += p.ss_in[(int64_t)row * p.n_ss + o];
      v = wave_sum(v);
      if (lane == 0) rsl[row] = rsqrtf(v * p.inv_d + p.eps);
    }
    __syncthreads();
    rs = rsl[fr];
  }
  int at = 0;
  for (; at + D < n; at += D)
#pragma unroll
    for (int d = 0; d < D; ++d) {
      compute(wr[d], xr[d]);
      load(wr[d], xr[d], at + D + d);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
  for (int d = 0; d < D; ++d)
    if (at + d < n) compute(wr[d], xr[d]);

  // ---- the waves' sums meet: lane holds rows 4fq + r of column 16j + fr
#pragma unroll
  for (int j = 0; j < NW; ++j)
    *reinterpret_cast<float4v*>(red + (wv * NW + j) * 256 + lane * 4) = acc[j];
  __syncthreads();
  // rows 4q + 0..3 of the block's weight row rr
  auto total = [&](int rr, int q) {
    float4v s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int v = 0; v < WAVES; ++v)
      s += *reinterpret_cast<const float4v*>(red + (v * NW + (rr >> 4)) * 256 +
                                             (q * 16 + (rr & 15)) * 4);
    return s;
  };
  constexpr int COLS = paired(EPI) ? F : 16 * NW;
  bf16_t* out = reinterpret_cast<bf16_t*>(p.out);
  if (tid < 4 * COLS) {
    const int c = tid % COLS, q = tid / COLS;
    float4v a = total(c, q), b = {0.f, 0.f, 0.f, 0.f};
    if constexpr (paired(EPI)) b = total(F + c, q);
    float ba = 0.f, bb = 0.f;
    if constexpr (EPI == 0)
      if (p.bias) ba = p.bias[unit * COLS + c];
    if constexpr (EPI == 1)
      if (p.bias) {
        ba = p.bias[unit * F + c];
        bb = p.bias[p.N + unit * F + c];
      }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = 4 * q + r;
      const int64_t col = (int64_t)unit * COLS + c;
      float va = a[r], vb = b[r];
      if constexpr (!grouped(EPI)) {
        if constexpr (EPI == 2) {  // the projection and the sum in bf16, as separate kernels
          float y = 0.f;
          if (m < p.M) {
            bf16_t* o = out + m * p.ldo + col;
            const bf16_t h = f2bf(bf2f(*o) + bf2f(f2bf(va)));
            y = bf2f(h);
            *o = h;
          }
          y = row_sum16(y * y);
          if constexpr (NW >= 2) y += __shfl_xor(y, 16, 64);
          if constexpr (NW == 4) y += __shfl_xor(y, 32, 64);
          if (c == 0 && m < p.M) p.ss_out[(int64_t)m * gridDim.x + unit] = y;
          continue;
        }
        if (m >= p.M) continue;
        if constexpr (EPI == 0) {
          out[m * p.ldo + col] = f2bf(va + ba);
        } else if constexpr (EPI == 1) {
          const float gt = va + ba;
          out[m * p.ldo + col] = f2bf((p.gelu ? gelu_tanh_(gt) : siluf_(gt)) * (vb + bb));
        } else {
          const int per = 64 / F, head = unit / per, dim = (unit - head * per) * F + c;
          va = bf2f(f2bf(va));  // the projection's bf16, which the rotation reads
          vb = bf2f(f2bf(vb));
          if (head < p.hq + p.hkv) {
            const float* cs = p.cos_sin + (int64_t)p.positions[m] * 128 + dim;
            const float cj = cs[0], sj = cs[64], t = va * cj - vb * sj;
            vb = vb * cj + va * sj;
            va = t;
          }
          bf16_t* o = out + m * p.ldo + head * 128 + dim;
          if (head >= p.hq) {
            const int64_t slot = p.slots[m];
            if (slot < 0) continue;
            const bool isk = head < p.hq + p.hkv;
            const int h = isk ? head - p.hq : head - p.hq - p.hkv;
            const int64_t blk = slot / p.page, off = slot - blk * p.page;
            o = (isk ? p.k_cache : p.v_cache) + ((blk * p.hkv + h) * p.page + off) * 128 + dim;
          }
          o[0] = f2bf(va);
          o[64] = f2bf(vb);
        }
      } else {
        const int row = seg * 16 + m, f = rows[m];
        if (f >= p.n_assign) continue;
        if constexpr (EPI == 6) {
          out[f * p.ldo + col] = f2bf(p.route_w ? p.route_w[f] * va : va);
        } else if constexpr (EPI == 5) {
          out[row * p.ldo + col] = f2bf(siluf_(va) * vb);
        } else if constexpr (EPI == 8) {
          const float wt = p.route_w[f];
          out[row * p.ldo + col] = f2bf(clamped_glu(wt * va, wt * vb, p.alpha, p.limit));
        } else {
          out[row * p.ldo + col] = f2bf(gelu_erf16_(va));
        }
      }
    }
  }
}

template <int NW, int EPI, bool NORM>
int launch(const StreamArgs& p, bool packed, int segs, hipStream_t s) {
  const int cols = paired(EPI) ? 8 * NW : 16 * NW;
  const int width = EPI == 3 ? (p.hq + 2 * p.hkv) * 64 : p.N;
  const dim3 grid(width / cols, segs);
  constexpr bool E = grouped(EPI);
  const void* first = E ? (const void*)p.ids : (const void*)p.ss_in;
#define OMNIA_STREAM(PK)                                                                          \
  stream_kernel<NW, EPI, NORM, PK><<<grid, 64 * WAVES, 0, s>>>(                                   \
      p.x, p.w, p.ldx, first, p.N, p.K, E ? p.e_lo : p.M, E ? p.e_hi : p.n_ss,                    \
      E ? p.n_assign : 0, E ? p.topk : 0, p)
  if (packed)
    OMNIA_STREAM(true);
  else
    OMNIA_STREAM(false);
#undef OMNIA_STREAM
  return (int)hipGetLastError();
}

template <int EPI, bool NORM>
int by_width(const StreamArgs& p, int nw, bool packed, int segs, hipStream_t s) {
  if (nw == 1) return launch<1, EPI, NORM>(p, packed, segs, s);
  if (nw == 2) return launch<2, EPI, NORM>(p, packed, segs, s);
  return launch<4, EPI, NORM>(p, packed, segs, s);
}

}  // namespace

extern "C" {

// 0 on success, < 0 for what the kernel does not cover (checked before any launch).
// nw: 16-row fragments of weights a block (1, 2, 4).  ss_in: the rows of x are normed.
int omnia_stream(int epi, void* out, const void* x, const void* w, int M, int N, int K,
                 int64_t ldx, int64_t ldo, int nw, int packed, const float* ss_in, int n_ss,
                 float inv_d, float eps, float* ss_out, const float* bias, int gelu, const int* positions, const float* cos_sin,
                 void* k_cache, void* v_cache, const int64_t* slots, int hq, int hkv, int page,
                 hipStream_t s) {
  if (epi < 0 || epi > 3) return -1;
  if (M < 1 || M > 16) return -2;
  if (K < 64 || K % 64 || ldx < K || ldx % 8) return -3;
  if (nw != 1 && nw != 2 && nw != 4) return -4;
  const int cols = epi == 1 ? 8 * nw : 16 * nw;
  if (N < cols || N % cols || (packed && N % 16) || N / cols > 1 << 20) return -5;
  if (epi == 3 && (N != (hq + 2 * hkv) * 128 || hq < 1 || hkv < 1 || page < 1)) return -6;
  if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w)) & 15) return -7;
  if (bias && epi > 1) return -8;
  if ((ss_in && n_ss < 1) || (epi == 2) != (ss_out != nullptr) || (epi == 2 && ss_in)) return -9;
  const bool norm = ss_in != nullptr;
  StreamArgs p{};
  p.out = out;
  p.x = (const bf16_t*)x;
  p.w = (const bf16_t*)w;
  p.M = M;
  p.N = N;
  p.K = K;
  p.ldx = ldx;
  p.ldo = ldo;
  p.ss_in = ss_in;
  p.n_ss = n_ss;
  p.ss_out = ss_out;
  p.inv_d = inv_d;
  p.eps = eps;
  p.bias = bias;
  p.gelu = gelu;
  p.positions = positions;
  p.cos_sin = cos_sin;
  p.k_cache = (bf16_t*)k_cache;
  p.v_cache = (bf16_t*)v_cache;
  p.slots = slots;
  p.hq = hq;
  p.hkv = hkv;
  p.page = page;
  if (epi == 0) return norm ? by_width<0, true>(p, nw, packed, 1, s) : by_width<0, false>(p, nw, packed, 1, s);
  if (epi == 1) return norm ? by_width<1, true>(p, nw, packed, 1, s) : by_width<1, false>(p, nw, packed, 1, s);
  if (epi == 2) return by_width<2, false>(p, nw, packed, 1, s);
  return norm ? by_width<3, true>(p, nw, packed, 1, s) : by_width<3, false>(p, nw, packed, 1, s);
}

// Grouped products of a few rows an expert: segments of 16 rows as omnia_moe_align makes them,
// or by ids, the experts of up to 64 assignments (one launch less: 4.5 us).  Modes and operands as
// omnia_moe_gemm.
int omnia_stream_moe(int mode, void* out, const void* A, const void* W, const int* ids, int e_hi,
                     const int* sorted,
                     const int* blk_expert, const int* n_blocks, const float* route_w, int K,
                     int N, int topk, int n_assign, int e_lo, int max_blocks, int nw, int packed,
                     float alpha, float limit, hipStream_t s) {
  if (mode < 0 || mode > 3 || K < 64 || K % 64) return -1;
  if (nw != 1 && nw != 2 && nw != 4) return -3;
  const int cols = mode == 0 || mode == 2 ? 8 * nw : 16 * nw;
  if (N < cols || N % cols || (packed && N % 16)) return -4;
  if (mode == 2 && !route_w) return -5;
  if (max_blocks == 0) return 0;
  if (max_blocks > 65535 || topk < 1 || (ids && n_assign > 64)) return -6;
  if ((reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(W)) & 15) return -7;
  StreamArgs p{};
  p.out = out;
  p.x = (const bf16_t*)A;
  p.w = (const bf16_t*)W;
  p.N = N;
  p.K = K;
  p.ldx = K;
  p.ldo = N;
  p.ids = ids;
  p.e_hi = e_hi;
  p.sorted = sorted;
  p.blk_expert = blk_expert;
  p.n_blocks = n_blocks;
  p.route_w = route_w;
  p.topk = topk;
  p.n_assign = n_assign;
  p.e_lo = e_lo;
  p.alpha = alpha;
  p.limit = limit;
  if (mode == 0) return by_width<5, false>(p, nw, packed, max_blocks, s);
  if (mode == 1) return by_width<6, false>(p, nw, packed, max_blocks, s);
  if (mode == 2) return by_width<8, false>(p, nw, packed, max_blocks, s);
  return by_width<10, false>(p, nw, packed, max_blocks, s);
}

}  // extern "C"
