// Latent attention for gfx950: per token the paged cache holds ONE row
//     [c (C, RMS-normed latent, zero-padded to Cp) | k_rot (R, rotated, padded) | 0]
// of Lp elements, [num_pages][page][Lp], shared by every head; head h's unrotated key
// is W_uk[h] c and its value W_uv[h] c.  A query sees the last `window` positions
// (window 0: all).  One fused input projection feeds it, a row of
//     [c_q (Qp) | latent (Cp) | k_rot (Rp) | gate (H)]
//
//   latent_prep     RMS norms of c_q and the latent, rotation of k_rot, page write
//   latent_rotate   rotation of the rotated part of q, in place
//   latent_heads    per-head projection out[t,h] = W[h] x[t,h] (optional sigmoid gate):
//                   absorbs W_uk into the query, expands W_uv after attention
//   latent_attend   generic attention over absorbed queries (any size, bf16 or fp32)
//   latent_decode   decode on MFMA: absorbed queries, all heads of a row share each
//                   staged page tile, split over the window, + latent_merge
//   latent_expand   decode: latent_merge and the expansion of W_uv in one launch
//   latent_gather   cached rows of each sequence's visible range -> dense [Tk] rows
//   latent_prefill  prefill on MFMA: expanded per-head keys and (transposed) values of
//                   the gathered range, online softmax, window mask, output gate
//
// Prefill expands (dim + rot products per score instead of C + rot); decode absorbs
// (one cached row per token for all heads).  Scores and softmax are fp32.
#include "common.h"

using namespace omnia;

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ float4v mfma16(short8 a, short8 b, float4v c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
__device__ __forceinline__ float16v mfma32(short8 a, short8 b, float16v c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

__device__ __forceinline__ int find_seq(const int* q_start, int nseq, int t) {
  int lo = 0, hi = nseq - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (q_start[mid] <= t) lo = mid; else hi = mid - 1;
  }
  return lo;
}

// ----------------------------------------------------------------- latent_prep
// one workgroup per token, bound by the latency of its loads, so all of a thread's are under way
// before the first sum (64 rows of 768 + 512 + 64 4.3 -> 3.6 us); cos_sin: [positions][R] fp32 = (cos[R/2] | sin[R/2])
template <typename T>
__global__ __launch_bounds__(256) void prep_kernel(
    T* __restrict__ cq, T* __restrict__ cache, const T* __restrict__ x, int64_t ldx,
    const float* __restrict__ wq, const float* __restrict__ wc, const int* __restrict__ positions,
    const int64_t* __restrict__ slots, const float* __restrict__ cos_sin, int Q, int Qp, int C,
    int Cp, int R, int Lp, float eps) {
  __shared__ float scratch[8];
  const int t = blockIdx.x, tid = threadIdx.x;
  const T* xq = x + (int64_t)t * ldx;
  const T* xc = xq + Qp;
  const T* xr = xc + Cp;
  const int64_t slot = slots[t];
  const float* cs = cos_sin + (int64_t)positions[t] * R;
  const int half = R / 2;
  // a thread's first NV of each, all asked for before the first is waited for
  constexpr int NV = 4;
  float vq[NV], vc[NV], gq[NV], gc[NV], sq = 0.f, sc = 0.f;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int i = tid + 256 * j;
    vq[j] = vc[j] = gq[j] = gc[j] = 0.f;
    if (i < Q) vq[j] = ldf(xq + i), gq[j] = wq[i];
    if (i < C) vc[j] = ldf(xc + i), gc[j] = wc[i];
  }
  float u0 = 0.f, v0 = 0.f, c0 = 0.f, s0 = 0.f;
  if (slot >= 0 && tid < half)
    u0 = ldf(xr + tid), v0 = ldf(xr + half + tid), c0 = cs[tid], s0 = cs[half + tid];
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    sq += vq[j] * vq[j];
    sc += vc[j] * vc[j];
  }
  for (int i = tid + 256 * NV; i < Q; i += 256) {
    const float v = ldf(xq + i);
    sq += v * v;
  }
  for (int i = tid + 256 * NV; i < C; i += 256) {
    const float v = ldf(xc + i);
    sc += v * v;
  }
  sq = wave_sum(sq);
  sc = wave_sum(sc);
  if ((tid & 63) == 0) {
    scratch[tid >> 6] = sq;
    scratch[4 + (tid >> 6)] = sc;
  }
  __syncthreads();
  sq = ((scratch[0] + scratch[1]) + scratch[2]) + scratch[3];
  sc = ((scratch[4] + scratch[5]) + scratch[6]) + scratch[7];
  const float iq = 1.f / sqrtf(sq / (float)Q + eps), ic = 1.f / sqrtf(sc / (float)C + eps);
  T* cr = cq + (int64_t)t * Qp;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int i = tid + 256 * j;
    if (i < Qp) stf(cr + i, vq[j] * iq * gq[j]);
  }
  for (int i = tid + 256 * NV; i < Qp; i += 256) stf(cr + i, i < Q ? ldf(xq + i) * iq * wq[i] : 0.f);
  if (slot < 0) return;
  T* row = cache + slot * Lp;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int i = tid + 256 * j;
    if (i < C) stf(row + i, vc[j] * ic * gc[j]);
  }
  for (int i = tid + 256 * NV; i < C; i += 256) stf(row + i, ldf(xc + i) * ic * wc[i]);
  for (int i = tid; i < half; i += 256) {
    const bool own = i < 256;
    const float u = own ? u0 : ldf(xr + i), v = own ? v0 : ldf(xr + half + i);
    const float c = own ? c0 : cs[i], s = own ? s0 : cs[half + i];
    stf(row + Cp + i, u * c - v * s);
    stf(row + Cp + half + i, v * c + u * s);
  }
}

// --------------------------------------------------------------- latent_rotate
template <typename T>
__global__ __launch_bounds__(256) void rotate_kernel(T* __restrict__ q, int64_t ldq, int hstride,
                                                     int off, const int* __restrict__ positions,
                                                     const float* __restrict__ cos_sin, int H,
                                                     int R) {
  const int t = blockIdx.x, half = R / 2;
  const float* cs = cos_sin + (int64_t)positions[t] * R;
  for (int i = threadIdx.x; i < H * half; i += 256) {
    const int h = i / half, j = i % half;
    T* p = q + (int64_t)t * ldq + h * hstride + off;
    const float u = ldf(p + j), v = ldf(p + half + j), c = cs[j], s = cs[half + j];
    stf(p + j, u * c - v * s);
    stf(p + half + j, v * c + u * s);
  }
}

// ---------------------------------------------------------------- latent_heads
// out[t, h*ho + n] = sum_k x[t, h*hx + k] W[h][n][k]  (* sigmoid(gate[t*ldg + h])),
// n < N, k < K;  rot (absorb): out[t, h*ho + N + i] = rotated x[t, h*hx + rotx + i]
struct Rot {
  const int* positions;  // null: no rotated part
  const float* cos_sin;
  int R, Rp, rotx, tail;  // tail: out columns after N + Rp to zero
};

// generic: one workgroup per (row, head)
template <typename T>
__global__ __launch_bounds__(256) void heads_kernel(T* __restrict__ out, int64_t ldo, int ho,
                                                    const T* __restrict__ x, int64_t ldx, int hx,
                                                    const T* __restrict__ W, int N, int K,
                                                    const T* __restrict__ gate, int64_t ldg,
                                                    Rot rot) {
  extern __shared__ float xs[];
  const int t = blockIdx.x, h = blockIdx.y;
  const T* xr = x + (int64_t)t * ldx + h * hx;
  for (int k = threadIdx.x; k < K; k += 256) xs[k] = ldf(xr + k);
  __syncthreads();
  const float g = gate ? sigmoidf_(ldf(gate + (int64_t)t * ldg + h)) : 1.f;
  T* orow = out + (int64_t)t * ldo + h * ho;
  for (int n = threadIdx.x; n < N; n += 256) {
    const T* w = W + ((int64_t)h * N + n) * K;
    float a = 0.f;
    for (int k = 0; k < K; ++k) a += xs[k] * ldf(w + k);
    stf(orow + n, a * g);
  }
  if (rot.positions) {
    const int half = rot.R / 2;
    const float* cs = rot.cos_sin + (int64_t)rot.positions[t] * rot.R;
    for (int i = threadIdx.x; i < half; i += 256) {
      const float u = ldf(xr + rot.rotx + i), v = ldf(xr + rot.rotx + half + i);
      stf(orow + N + i, u * cs[i] - v * cs[half + i]);
      stf(orow + N + half + i, v * cs[i] + u * cs[half + i]);
    }
    for (int i = rot.R + threadIdx.x; i < rot.Rp + rot.tail; i += 256) stf(orow + N + i, 0.f);
  }
}

// MFMA form (bf16): grid (ceil(N/64), and one for the rotated part, H, ceil(T/16)), one wave: 16 rows
// x 64 columns, operands straight from L2 (K is a head dimension or the latent: a few hundred),
// four k-steps of loads in flight.  K % 32 == 0.  The rotated part is a chain of small loads: in the
// block of the first columns, behind their products, absorbing took 2.7 / 5.5 / 10.2 / 19.6 us at 1 / 64 /
// 256 / 600 rows of 16 heads of 128 -> 512, in blocks of its own 2.6 / 4.2 / 7.7 / 16.4.
__global__ __launch_bounds__(64) void heads_mfma_kernel(
    bf16_t* __restrict__ out, int64_t ldo, int ho, const bf16_t* __restrict__ x, int64_t ldx,
    int hx, const bf16_t* __restrict__ W, int T, int N, int K, const bf16_t* __restrict__ gate,
    int64_t ldg, Rot rot) {
  const int lane = threadIdx.x;
  const int h = blockIdx.y, n0 = blockIdx.x * 64, r0 = blockIdx.z * 16;
  if (n0 >= N) {  // the last of a row of blocks: the rotated part
    const int half = rot.R / 2, nr = min(16, T - r0);
#pragma unroll 4
    for (int e = lane; e < nr * half; e += 64) {
      const int row = r0 + e / half, i = e % half;
      const float* cs = rot.cos_sin + (int64_t)rot.positions[row] * rot.R;
      const bf16_t* xr = x + (int64_t)row * ldx + h * hx + rot.rotx;
      bf16_t* orow = out + (int64_t)row * ldo + h * ho + N;
      const float u = ldf(xr + i), v = ldf(xr + half + i), c = cs[i], s = cs[half + i];
      stf(orow + i, u * c - v * s);
      stf(orow + half + i, v * c + u * s);
    }
    const int pad = rot.Rp + rot.tail - rot.R;
    for (int e = lane; e < nr * pad; e += 64)
      stf(out + (int64_t)(r0 + e / pad) * ldo + h * ho + N + rot.R + e % pad, 0.f);
    return;
  }
  const int fr = lane & 15, fq = lane >> 4;
  const int ra = min(r0 + fr, T - 1);
  const bf16_t* xa = x + (int64_t)ra * ldx + h * hx + 8 * fq;
  const bf16_t* wb[4];
#pragma unroll
  for (int j = 0; j < 4; ++j)
    wb[j] = W + ((int64_t)h * N + min(n0 + 16 * j + fr, N - 1)) * K + 8 * fq;
  float4v acc[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) acc[j] = float4v{0.f, 0.f, 0.f, 0.f};
  auto steps = [&](int k, auto NS) {
    constexpr int N_ = decltype(NS)::value;
    short8 a[N_], b[N_][4];
#pragma unroll
    for (int u = 0; u < N_; ++u) {
      a[u] = *reinterpret_cast<const short8*>(xa + k + 32 * u);
#pragma unroll
      for (int j = 0; j < 4; ++j) b[u][j] = *reinterpret_cast<const short8*>(wb[j] + k + 32 * u);
    }
#pragma unroll
    for (int u = 0; u < N_; ++u)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[j] = mfma16(a[u], b[u][j], acc[j]);
  };
  int k = 0;
  for (; k + 128 <= K; k += 128) steps(k, std::integral_constant<int, 4>{});
  for (; k < K; k += 32) steps(k, std::integral_constant<int, 1>{});
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int row = r0 + 4 * fq + r;
    if (row >= T) continue;
    const float g = gate ? sigmoidf_(ldf(gate + (int64_t)row * ldg + h)) : 1.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + 16 * j + fr;
      if (n < N) stf(out + (int64_t)row * ldo + h * ho + n, acc[j][r] * g);
    }
  }
}

// Parts of a row's keys on the device (live length), equal and 64-aligned: keys of a part.
__device__ __forceinline__ int part_len(int n, int splits) {
  return ((n + splits - 1) / splits + 63) / 64 * 64;
}

// latent_decode's merge and the expansion of W_uv in one launch: grid (H, ceil(T / RB)), 8 waves, RB
// rows of a head (4, 8 or 16 of the product's 16: few rows spread over the CUs).  Wave w multiplies the
// columns 16 w ..; its weights, all of K, are under way while the waves merge the rows' parts into LDS,
// 256 latent columns a wave and turn.  Bound by the latency of those loads; each of the launches that it
// stands for had one.  us of decode with merge and expansion, before / now, 16 heads of 512 -> 128, rows x
// keys (parts): 1 x 1024 (8) 20.6 / 18.1, 4 x 4000 (32) 25.3 / 25.0, 64 x 1024 (8) 32.0 / 28.4, 256 x 1024
// (2) 71.4 / 65.3.  Where rows have one part there is nothing to merge, and the two stay (600 x 200 53.7 /
// 56.5, 256 x 100 22.4 / 22.0).
__global__ __launch_bounds__(512) void expand_kernel(
    bf16_t* __restrict__ out, int64_t ldo, int ho, const bf16_t* __restrict__ o,
    const float* __restrict__ part_o, const float* __restrict__ part_ml,
    const bf16_t* __restrict__ W, const bf16_t* __restrict__ gate, int64_t ldg,
    const int* __restrict__ positions, int T, int H, int N, int K, int window, int splits, int RB) {
  constexpr int KS = 16;  // k-steps of 32: K <= 512
  __shared__ __attribute__((aligned(16))) bf16_t xs[16][32 * KS + 8];
  const int h = blockIdx.x, r0 = blockIdx.y * RB, lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), fr = lane & 15, fq = lane >> 4;
  const int n = 16 * w + fr;
  short8 b[KS];
  if (16 * w < N) {
    const bf16_t* wb = W + ((int64_t)h * N + min(n, N - 1)) * K + 8 * fq;
#pragma unroll
    for (int u = 0; u < KS; ++u)
      if (32 * u < K) b[u] = *reinterpret_cast<const short8*>(wb + 32 * u);
  }
  float g[4];
#pragma unroll
  for (int r = 0; r < 4; ++r)
    g[r] = sigmoidf_(ldf(gate + (int64_t)min(r0 + 4 * fq + r, T - 1) * ldg + h));
  const int segs = (K + 255) / 256;
  for (int q = w; q < RB * segs; q += 8) {  // wave-uniform
    const int row = r0 + q / segs, c = q % segs * 256 + 4 * lane;
    if (row >= T) break;
    const int64_t bh = (int64_t)row * H + h;
    const int pos = positions[row], lo = window > 0 ? max(0, pos - window + 1) : 0;
    const int keys = max(pos + 1 - lo, 1), pl = part_len(keys, splits), np = (keys + pl - 1) / pl;
    uint2v k = {0, 0};
    if (np <= 1) {
      if (c < K) k = *reinterpret_cast<const uint2v*>(o + bh * K + c);
    } else {
      const float* ml = part_ml + (bh * splits + min(lane, np - 1)) * 2;
      const float m = lane < np ? ml[0] : -INFINITY, l = lane < np ? ml[1] : 0.f;
      const float* po = part_o + bh * splits * K + min(c, K - 4);
      float4v a = {0.f, 0.f, 0.f, 0.f};
      float wt = 0.f;
      for (int p0 = 0; p0 < np; p0 += 8) {
        float4v v[8];
#pragma unroll
        for (int p = 0; p < 8; ++p)
          v[p] = *reinterpret_cast<const float4v*>(po + (int64_t)min(p0 + p, np - 1) * K);
        if (p0 == 0) {
          wt = exp2f(m - wave_max(m)) * l;
          wt = wt / wave_sum(wt);
        }
#pragma unroll
        for (int p = 0; p < 8; ++p)
          if (p0 + p < np) a += v[p] * __shfl(wt, p0 + p, 64);
      }
      k[0] = pack_bf2(a[0], a[1]);
      k[1] = pack_bf2(a[2], a[3]);
    }
    if (c < K) *reinterpret_cast<uint2v*>(&xs[row - r0][c]) = k;
  }
  __syncthreads();
  if (16 * w >= N) return;
  float4v acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int u = 0; u < KS; ++u)  // rows of xs past RB: of products that are not stored
    if (32 * u < K)
      acc = mfma16(*reinterpret_cast<const short8*>(&xs[fr][32 * u + 8 * fq]), b[u], acc);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int i = 4 * fq + r;
    if (i < RB && r0 + i < T && n < N)
      stf(out + (int64_t)(r0 + i) * ldo + h * ho + n, acc[r] * g[r]);
  }
}

// --------------------------------------------------------------- latent_attend
// grid (T, H), 256 threads; any size.  Tiles of 256 keys: a thread scores one key,
// then owns latent columns for the weighted sum.
template <typename T>
__global__ __launch_bounds__(256) void attend_kernel(
    T* __restrict__ out, const T* __restrict__ q, const T* __restrict__ cache,
    const int* __restrict__ block_tables, int bt_stride, const int* __restrict__ q_start, int nseq,
    const int* __restrict__ positions, int page, int H, int Cp, int Lp, int window, float scale) {
  extern __shared__ float sm[];
  float* qs = sm;         // [Lp]
  float* acc = qs + Lp;   // [Cp]
  float* p = acc + Cp;    // [256]
  float* scratch = p + 256;  // [8]
  const int t = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
  const int s = q_start ? find_seq(q_start, nseq, t) : t;
  const int* bt = block_tables + (int64_t)s * bt_stride;
  const int pos = positions[t];
  const int lo = window > 0 ? max(0, pos - window + 1) : 0;
  const T* qr = q + ((int64_t)t * H + h) * Lp;
  for (int i = tid; i < Lp; i += 256) qs[i] = ldf(qr + i);
  for (int i = tid; i < Cp; i += 256) acc[i] = 0.f;
  float m = -INFINITY, l = 0.f;
  for (int k0 = lo; k0 <= pos; k0 += 256) {
    const int n = min(256, pos + 1 - k0);
    __syncthreads();
    float sc = -INFINITY;
    if (tid < n) {
      const int key = k0 + tid;
      const T* row = cache + ((int64_t)bt[key / page] * page + key % page) * Lp;
      float a = 0.f;
      for (int i = 0; i < Lp; ++i) a += qs[i] * ldf(row + i);
      sc = a * scale;
    }
    const float mn = fmaxf(m, block_max(sc, scratch));
    const float e = tid < n ? expf(sc - mn) : 0.f;
    p[tid] = e;
    const float alpha = expf(m - mn);
    l = l * alpha + block_sum(e, scratch);
    m = mn;
    __syncthreads();
    for (int c = tid; c < Cp; c += 256) {
      float a = acc[c] * alpha;
      for (int j = 0; j < n; ++j) {
        const int key = k0 + j;
        a += p[j] * ldf(cache + ((int64_t)bt[key / page] * page + key % page) * Lp + c);
      }
      acc[c] = a;
    }
  }
  for (int c = tid; c < Cp; c += 256) stf(out + ((int64_t)t * H + h) * Cp + c, acc[c] / l);
}

// --------------------------------------------------------------- latent_decode
// grid (rows, ceil(H / (16 HT)), splits), 4 waves.  Tiles of 32 keys, the next one
// loaded into registers while this one is used.  Per tile:
//   QK   each wave one (16 heads x 16 keys) product, its q fragments held in registers;
//        with one head tile (HT = 1) two waves share a product, half the row width each
//   P V  wave w owns latent column tiles w, w+4, ...; V^T fragments by
//        ds_read_b64_tr_b16 from the row-major tile, the keys of the k-step permuted the
//        same way on the P side
template <int HT, int LW>
__global__ __launch_bounds__(256, 2) void decode_kernel(
    bf16_t* __restrict__ out, float* __restrict__ part_o, float* __restrict__ part_ml,
    const bf16_t* __restrict__ q, const bf16_t* __restrict__ cache,
    const int* __restrict__ block_tables, int bt_stride, const int* __restrict__ positions,
    int page_log2, int H, int Cp, int window, float scale_log2) {
  constexpr int NH = 16 * HT, KT = 32, LS = LW + 8;  // LS: an odd number of 16-B units
  // column tiles per wave; those past the latent (the rotated part, or past the row: the
  // next row's columns) are computed and not stored
  constexpr int NT = (LW / 16 + 3) / 4;
  constexpr int KP = 2 / HT;                         // waves sharing one product
  constexpr int NS = LW / 32, NSW = (NS + KP - 1) / KP;
  constexpr int SS = KT + 4, PS = KT + 8;
  constexpr int LCH = LW / 8, TOT = KT * LCH, PN = (TOT + 255) / 256;
  __shared__ __attribute__((aligned(16))) bf16_t tile[KT * LS + 64];
  __shared__ __attribute__((aligned(16))) float sc[KP * NH * SS];
  __shared__ __attribute__((aligned(16))) bf16_t pb[NH * PS];
  __shared__ float st[3 * NH];  // m, l, alpha
  extern __shared__ int pages[];  // this part's block-table entries

  const int b = blockIdx.x, h0 = blockIdx.y * NH, part = blockIdx.z, splits = gridDim.z;
  const int pos = positions[b];
  const int lo = window > 0 ? max(0, pos - window + 1) : 0;
  const int n = pos + 1 - lo, pl = part_len(n, splits), p0 = part * pl;
  if (p0 >= n) return;
  const int kbeg = lo + p0, kend = min(lo + n, kbeg + pl);
  const int nparts = (n + pl - 1) / pl;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, c16 = lane & 15, g4 = lane >> 4;
  const int pg0 = kbeg >> page_log2, pmask = (1 << page_log2) - 1;
  const int qt = HT == 2 ? w & 1 : 0, kt = HT == 2 ? w >> 1 : w & 1, kp = HT == 2 ? 0 : w >> 1;

  short8 qf[NSW];
  {
    const int hh = h0 + 16 * qt + c16;
    const bf16_t* qr = q + ((int64_t)b * H + min(hh, H - 1)) * LW + 8 * g4;
#pragma unroll
    for (int k = 0; k < NSW; ++k) {
      qf[k] = *reinterpret_cast<const short8*>(qr + 32 * min(kp * NSW + k, NS - 1));
      if (hh >= H) qf[k] = short8{0, 0, 0, 0, 0, 0, 0, 0};
    }
  }
  for (int i = tid; i <= ((kend - 1) >> page_log2) - pg0; i += 256)
    pages[i] = block_tables[(int64_t)b * bt_stride + pg0 + i];
  if (tid < NH) {
    st[tid] = -1e30f;
    st[NH + tid] = 0.f;
  }
  __syncthreads();

  short8 reg[PN];
  auto gload = [&](int k0) {
    int64_t row[PN];
#pragma unroll
    for (int i = 0; i < PN; ++i) {  // all page lookups before the first load
      const int c = min(i * 256 + tid, TOT - 1);
      const int key = min(k0 + c / LCH, kend - 1);
      row[i] = ((int64_t)pages[(key >> page_log2) - pg0] << page_log2) + (key & pmask);
    }
#pragma unroll
    for (int i = 0; i < PN; ++i) {
      const int c = min(i * 256 + tid, TOT - 1);
      reg[i] = *reinterpret_cast<const short8*>(cache + row[i] * LW + (c % LCH) * 8);
    }
  };
  gload(kbeg);
  if (tid < 64) tile[KT * LS + tid] = 0;
  float4v acc[HT][NT];
#pragma unroll
  for (int i = 0; i < HT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = float4v{0.f, 0.f, 0.f, 0.f};
  const int ncol = (Cp / 16 - w + 3) / 4;  // this wave's column tiles

  for (int k0 = kbeg; k0 < kend; k0 += KT) {
    __syncthreads();  // the previous tile is consumed
#pragma unroll
    for (int i = 0; i < PN; ++i) {
      const int c = i * 256 + tid;
      if (TOT % 256 == 0 || c < TOT)
        *reinterpret_cast<short8*>(tile + (c / LCH) * LS + (c % LCH) * 8) = reg[i];
    }
    __syncthreads();
    if (k0 + KT < kend) gload(k0 + KT);
    {
      float4v s0 = {0.f, 0.f, 0.f, 0.f}, s1 = s0;
      const bf16_t* kr = tile + (16 * kt + c16) * LS + 8 * g4 + 32 * kp * NSW;
#pragma unroll
      for (int k = 0; k < NSW; ++k) {
        if (KP > 1 && NS % KP && kp * NSW + k >= NS) continue;  // wave-uniform
        const short8 kf = *reinterpret_cast<const short8*>(kr + 32 * k);
        if (k & 1) s1 = mfma16(qf[k], kf, s1);
        else s0 = mfma16(qf[k], kf, s0);
      }
      s0 += s1;
#pragma unroll
      for (int r = 0; r < 4; ++r)
        sc[(kp * NH + 16 * qt + 4 * g4 + r) * SS + 16 * kt + c16] = s0[r] * scale_log2;
    }
    __syncthreads();
    {  // softmax: 256 / NH threads per head, consecutive lanes
      constexpr int TH = 256 / NH, PER = KT / TH;
      const int hh = tid / TH, j0 = (tid % TH) * PER;
      float v[PER], mx = -INFINITY;
#pragma unroll
      for (int j = 0; j < PER; ++j) {
        float x = sc[hh * SS + j0 + j];
        if (KP > 1) x += sc[(NH + hh) * SS + j0 + j];
        v[j] = k0 + j0 + j < kend ? x : -INFINITY;
        mx = fmaxf(mx, v[j]);
      }
#pragma unroll
      for (int o = 1; o < TH; o <<= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
      const float m_old = st[hh], m_new = fmaxf(m_old, mx);
      float sum = 0.f;
#pragma unroll
      for (int j = 0; j < PER; ++j) {
        const float e = __builtin_amdgcn_exp2f(v[j] - m_new);
        pb[hh * PS + j0 + j] = f2bf(e);
        sum += e;
      }
#pragma unroll
      for (int o = 1; o < TH; o <<= 1) sum += __shfl_xor(sum, o, 64);
      const float alpha = __builtin_amdgcn_exp2f(m_old - m_new);
      if (tid % TH == 0) {
        st[hh] = m_new;
        st[NH + hh] = st[NH + hh] * alpha + sum;
        st[2 * NH + hh] = alpha;
      }
    }
    __syncthreads();
    const int qq = c16 >> 2, pp = c16 & 3;
    typedef short v4s __attribute__((ext_vector_type(4)));
    short8 pa[HT];
    float4v al[HT];
#pragma unroll
    for (int i = 0; i < HT; ++i) {
      const bf16_t* pr = pb + (16 * i + c16) * PS + 4 * g4;
      const v4s lo4 = *reinterpret_cast<const v4s*>(pr), hi4 = *reinterpret_cast<const v4s*>(pr + 16);
      pa[i] = __builtin_shufflevector(lo4, hi4, 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
      for (int r = 0; r < 4; ++r) al[i][r] = st[2 * NH + 16 * i + 4 * g4 + r];
    }
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const bf16_t* vr = tile + (4 * g4 + qq) * LS + 16 * (w + 4 * j) + 4 * pp;
      const v4s lo4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (__attribute__((address_space(3))) v4s*)(vr));
      const v4s hi4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (__attribute__((address_space(3))) v4s*)(vr + 16 * LS));
      const short8 vb = __builtin_shufflevector(lo4, hi4, 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
      for (int i = 0; i < HT; ++i) acc[i][j] = mfma16(pa[i], vb, acc[i][j] * al[i]);
    }
  }
  // acc[i][j][r]: head 16 i + 4 g4 + r, latent column 16 (w + 4 j) + c16
#pragma unroll
  for (int i = 0; i < HT; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int hh = 16 * i + 4 * g4 + r;
      if (h0 + hh >= H) continue;
      const float inv = 1.f / st[NH + hh];
      const int64_t bh = (int64_t)b * H + h0 + hh;
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        if (j >= ncol) continue;
        const int c = 16 * (w + 4 * j) + c16;
        if (nparts == 1) out[bh * Cp + c] = f2bf(acc[i][j][r] * inv);
        else part_o[(bh * splits + part) * Cp + c] = acc[i][j][r] * inv;
      }
      if (nparts > 1 && w == 0 && c16 == 0) {
        part_ml[(bh * splits + part) * 2] = st[hh];
        part_ml[(bh * splits + part) * 2 + 1] = st[NH + hh];
      }
    }
}

// grid (rows * H), 128 threads: merge of the parts a row was cut into (at most 64)
__global__ __launch_bounds__(128) void merge_kernel(bf16_t* __restrict__ out,
                                                    const float* __restrict__ part_o,
                                                    const float* __restrict__ part_ml,
                                                    const int* __restrict__ positions, int H,
                                                    int Cp, int window, int splits) {
  __shared__ float wgt[64];
  const int bh = blockIdx.x, pos = positions[bh / H], lane = threadIdx.x & 63;
  const int lo = window > 0 ? max(0, pos - window + 1) : 0;
  const int n = pos + 1 - lo, pl = part_len(n, splits), np = (n + pl - 1) / pl;
  if (np <= 1) return;
  if (threadIdx.x < 64) {
    const float* ml = part_ml + ((int64_t)bh * splits + lane) * 2;
    const float m = lane < np ? ml[0] : -INFINITY, l = lane < np ? ml[1] : 0.f;
    const float w = exp2f(m - wave_max(m)) * l;
    wgt[lane] = w / wave_sum(w);
  }
  __syncthreads();
  for (int c = threadIdx.x * 4; c < Cp; c += 512) {
    const float* po = part_o + (int64_t)bh * splits * Cp + c;
    float4v a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
    for (int p = 0; p < np; ++p)
      a += *reinterpret_cast<const float4v*>(po + (int64_t)p * Cp) * wgt[p];
    uint2v k;
    k[0] = pack_bf2(a[0], a[1]);
    k[1] = pack_bf2(a[2], a[3]);
    *reinterpret_cast<uint2v*>(out + (int64_t)bh * Cp + c) = k;
  }
}

// --------------------------------------------------------------- latent_gather
// dense row i of sequence s (kv_start[s] <= i < kv_start[s+1]) = cached position
// kv_first[s] + i - kv_start[s]; rows past the sequence's length are zero.
// grid (ceil(Tk / 4)), one wave per row
__global__ __launch_bounds__(256) void gather_kernel(
    bf16_t* __restrict__ c, bf16_t* __restrict__ kr, const bf16_t* __restrict__ cache,
    const int* __restrict__ block_tables, int bt_stride, const int* __restrict__ kv_start,
    const int* __restrict__ kv_first, const int* __restrict__ seq_lens, int nseq, int page, int Tk,
    int Cp, int Rp, int Lp) {
  const int i = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (i >= Tk) return;
  const int s = find_seq(kv_start, nseq, i);
  const int key = kv_first[s] + i - kv_start[s];
  const bool ok = key < seq_lens[s];
  const bf16_t* row = cache;
  if (ok) row += ((int64_t)block_tables[(int64_t)s * bt_stride + key / page] * page + key % page) * Lp;
  for (int e = lane * 8; e < Cp + Rp; e += 512) {
    const short8 v = ok ? *reinterpret_cast<const short8*>(row + e) : short8{0, 0, 0, 0, 0, 0, 0, 0};
    if (e < Cp) *reinterpret_cast<short8*>(c + (int64_t)i * Cp + e) = v;
    else *reinterpret_cast<short8*>(kr + (int64_t)i * Rp + e - Cp) = v;
  }
}

// -------------------------------------------------------------- latent_prefill
// grid (n_tiles * H), 4 waves x 32 query rows of one head (a 128-row tile).
//   S^T = K Q^T      lane (query l & 31, hi = l >> 5) holds 32 of its row's 64 scores
//   O^T += V^T P^T   the lane's own scores are the B operand; V^T rows (keys
//                    contiguous) come straight from the transposed value projection
// Keys: kx [Tk][H*Da] | kr [Tk][Rp] (shared by the heads) | zero; vt [H*Vp][Tk].
template <int QW, int VW>
__global__ __launch_bounds__(256, 2) void prefill_kernel(
    bf16_t* __restrict__ out, const bf16_t* __restrict__ q, const bf16_t* __restrict__ kx,
    const bf16_t* __restrict__ kr, const bf16_t* __restrict__ vt, const int* __restrict__ q_start,
    const int* __restrict__ seq_lens, const int* __restrict__ kv_start,
    const int* __restrict__ kv_first, const int* __restrict__ tile_seq,
    const int* __restrict__ tile_q0, int n_tiles, int H, int Da, int Rp, int Tk, int window,
    float scale_log2, const bf16_t* __restrict__ gate, int64_t ldg) {
  constexpr int KS = QW + 8;  // LDS row strides (elements): odd in 16-B / 8-B units
  constexpr int VS = 68;
  __shared__ __attribute__((aligned(16))) bf16_t Kl[64 * KS];
  __shared__ __attribute__((aligned(16))) bf16_t Vl[VW * VS];
  const int id = xcd_remap(blockIdx.x, gridDim.x);  // a head's tiles share an XCD's L2
  // a sequence's last tiles, which see most keys, first: what is left for the end is short
  // (8 x 2048 rows, 16 heads, 225 -> 215 us)
  const int h = id / n_tiles, tl = n_tiles - 1 - (id - h * n_tiles);
  const int s = tile_seq[tl], q0 = tile_q0[tl];
  const int qs = q_start[s], qlen = q_start[s + 1] - qs;
  const int off = seq_lens[s] - qlen, kf = kv_first[s], kst = kv_start[s];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, ql = lane & 31, hi = lane >> 5;
  const int qr = q0 + w * 32 + ql;
  const bool row_ok = qr < qlen;
  const int qpos = off + min(qr, qlen - 1);
  short8 qf[QW / 16];
  {
    const bf16_t* qrow = q + ((int64_t)(qs + min(qr, qlen - 1)) * H + h) * QW + 8 * hi;
#pragma unroll
    for (int ks = 0; ks < QW / 16; ++ks) qf[ks] = *reinterpret_cast<const short8*>(qrow + 16 * ks);
  }
  // visible keys, relative to kv_first: [klo, khi), klo rounded down to a tile
  const int khi = off + min(q0 + 128, qlen) - kf;
  const int klo = window > 0 ? max(0, off + q0 - window + 1 - kf) / 64 * 64 : 0;
  // this wave's rows only need [wlo, whi]
  const int whi = off + min(q0 + w * 32 + 31, qlen - 1) - kf;
  const int wmin = off + min(q0 + w * 32, qlen - 1) - kf;
  const int wlo = window > 0 ? wmin - window + 1 : -1;
  const int rpos = qpos - kf;
  const int rlo = window > 0 ? rpos - window + 1 : -(1 << 30);

  constexpr int KCH = QW / 8, KN = 64 * KCH / 256, VN = VW * 8 / 256;
  short8 kreg[KN], vreg[VN];
  const short8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
  auto gload = [&](int k0) {
#pragma unroll
    for (int i = 0; i < KN; ++i) {
      const int c = i * 256 + tid, r = c / KCH, e = (c % KCH) * 8;
      const int64_t row = kst + k0 + r;  // inside the sequence's 64-aligned range
      kreg[i] = e < Da ? *reinterpret_cast<const short8*>(kx + (row * H + h) * Da + e)
                : e < Da + Rp ? *reinterpret_cast<const short8*>(kr + row * Rp + e - Da)
                              : zero;
    }
#pragma unroll
    for (int i = 0; i < VN; ++i) {
      const int c = i * 256 + tid, v = c >> 3, e = (c & 7) * 8;
      vreg[i] = *reinterpret_cast<const short8*>(vt + ((int64_t)h * VW + v) * Tk + kst + k0 + e);
    }
  };
  auto lwrite = [&]() {
    typedef short v4s __attribute__((ext_vector_type(4)));
#pragma unroll
    for (int i = 0; i < KN; ++i) {
      const int c = i * 256 + tid, r = c / KCH, e = (c % KCH) * 8;
      *reinterpret_cast<short8*>(Kl + r * KS + e) = kreg[i];
    }
#pragma unroll
    for (int i = 0; i < VN; ++i) {
      const int c = i * 256 + tid, v = c >> 3, e = (c & 7) * 8;
      *reinterpret_cast<v4s*>(Vl + v * VS + e) = __builtin_shufflevector(vreg[i], vreg[i], 0, 1, 2, 3);
      *reinterpret_cast<v4s*>(Vl + v * VS + e + 4) = __builtin_shufflevector(vreg[i], vreg[i], 4, 5, 6, 7);
    }
  };

  float m_run = -1e30f, l_run = 0.f;
  float16v o[VW / 32];
#pragma unroll
  for (int d = 0; d < VW / 32; ++d)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[d][r] = 0.f;

  gload(klo);
  for (int k0 = klo; k0 < khi; k0 += 64) {
    __syncthreads();  // every wave is done with the previous tile
    lwrite();
    __syncthreads();
    if (k0 + 64 < khi) gload(k0 + 64);
    if (k0 > whi || k0 + 63 < wlo) continue;  // wave-uniform: no visible key for its rows
    float16v sa[2];
#pragma unroll
    for (int half = 0; half < 2; ++half) {
#pragma unroll
      for (int r = 0; r < 16; ++r) sa[half][r] = 0.f;
#pragma unroll
      for (int ks = 0; ks < QW / 16; ++ks)
        sa[half] = mfma32(*reinterpret_cast<const short8*>(Kl + (half * 32 + ql) * KS + 16 * ks + 8 * hi),
                          qf[ks], sa[half]);
    }
    float mloc = -INFINITY;
    if (k0 + 63 > wmin || k0 < whi - (window > 0 ? window - 1 : 1 << 30)) {
      const int top = rpos - k0 - 4 * hi, bot = rlo - k0 - 4 * hi;
#pragma unroll
      for (int half = 0; half < 2; ++half)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int kk = half * 32 + (r & 3) + 8 * (r >> 2);
          const float v = (kk > top || kk < bot) ? -INFINITY : sa[half][r];
          sa[half][r] = v;
          mloc = fmaxf(mloc, v);
        }
    } else {
#pragma unroll
      for (int half = 0; half < 2; ++half)
#pragma unroll
        for (int r = 0; r < 16; ++r) mloc = fmaxf(mloc, sa[half][r]);
    }
    mloc = fmaxf(mloc, __shfl_xor(mloc, 32, 64)) * scale_log2;
    const bool grow = mloc > m_run + 8.f;  // lazy rescale (see attention.hip)
    if (__builtin_amdgcn_ballot_w64(grow)) {
      const float m_new = grow ? mloc : m_run;
      const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
      l_run *= alpha;
#pragma unroll
      for (int d = 0; d < VW / 32; ++d) o[d] *= alpha;
      m_run = m_new;
    }
    float lsum = 0.f;
#pragma unroll
    for (int half = 0; half < 2; ++half)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(sa[half][r], scale_log2, -m_run));
        sa[half][r] = p;
        lsum += p;
      }
    l_run += lsum + __shfl_xor(lsum, 32, 64);
#pragma unroll
    for (int st = 0; st < 4; ++st) {
      short8 pb;
#pragma unroll
      for (int j = 0; j < 8; ++j)
        pb[j] = __builtin_bit_cast(short, (__bf16)sa[st >> 1][8 * (st & 1) + j]);
      typedef short v4s __attribute__((ext_vector_type(4)));
#pragma unroll
      for (int d = 0; d < VW / 32; ++d) {
        const bf16_t* vr = Vl + (d * 32 + ql) * VS + (st >> 1) * 32 + 16 * (st & 1) + 4 * hi;
        const v4s lo4 = *reinterpret_cast<const v4s*>(vr), hi4 = *reinterpret_cast<const v4s*>(vr + 8);
        o[d] = mfma32(__builtin_shufflevector(lo4, hi4, 0, 1, 2, 3, 4, 5, 6, 7), pb, o[d]);
      }
    }
  }
  if (row_ok) {
    const float g = sigmoidf_(ldf(gate + (int64_t)(qs + qr) * ldg + h)) / l_run;
    bf16_t* orow = out + ((int64_t)(qs + qr) * H + h) * VW;
#pragma unroll
    for (int d = 0; d < VW / 32; ++d)
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        uint2v pk;
        pk[0] = pack_bf2(o[d][4 * m] * g, o[d][4 * m + 1] * g);
        pk[1] = pack_bf2(o[d][4 * m + 2] * g, o[d][4 * m + 3] * g);
        *reinterpret_cast<uint2v*>(orow + d * 32 + 8 * m + 4 * hi) = pk;
      }
  }
}

}  // namespace

extern "C" {

int omnia_latent_prep(void* cq, void* cache, const void* x, int f32, int64_t ldx, const float* wq,
                      const float* wc, const int* positions, const int64_t* slots,
                      const float* cos_sin, int T, int Q, int Qp, int C, int Cp, int R, int Lp,
                      float eps, hipStream_t s) {
  if (R % 2 || Cp < C || Qp < Q || Lp < Cp + R) return -1;
  if (T == 0) return 0;
  if (f32)
    prep_kernel<float><<<T, 256, 0, s>>>((float*)cq, (float*)cache, (const float*)x, ldx, wq, wc,
                                         positions, slots, cos_sin, Q, Qp, C, Cp, R, Lp, eps);
  else
    prep_kernel<bf16_t><<<T, 256, 0, s>>>((bf16_t*)cq, (bf16_t*)cache, (const bf16_t*)x, ldx, wq,
                                          wc, positions, slots, cos_sin, Q, Qp, C, Cp, R, Lp, eps);
  return (int)hipGetLastError();
}

int omnia_latent_rotate(void* q, int f32, int64_t ldq, int hstride, int off, const int* positions,
                        const float* cos_sin, int T, int H, int R, hipStream_t s) {
  if (R % 2 || off + R > hstride) return -1;
  if (T == 0) return 0;
  if (f32)
    rotate_kernel<float><<<T, 256, 0, s>>>((float*)q, ldq, hstride, off, positions, cos_sin, H, R);
  else
    rotate_kernel<bf16_t><<<T, 256, 0, s>>>((bf16_t*)q, ldq, hstride, off, positions, cos_sin, H, R);
  return (int)hipGetLastError();
}

int omnia_latent_heads(void* out, int f32, int64_t ldo, int ho, const void* x, int64_t ldx, int hx,
                       const void* W, int T, int H, int N, int K, const void* gate, int64_t ldg,
                       const int* positions, const float* cos_sin, int R, int Rp, int rotx,
                       int tail, hipStream_t s) {
  if (H > 65535 || K < 1 || N < 1) return -1;
  if (T == 0) return 0;
  const Rot rot{positions, cos_sin, R, Rp, rotx, tail};
  if (f32) {
    if ((size_t)K * 4 > 64 * 1024) return -2;
    heads_kernel<float><<<dim3(T, H), 256, K * 4, s>>>((float*)out, ldo, ho, (const float*)x, ldx,
                                                       hx, (const float*)W, N, K,
                                                       (const float*)gate, ldg, rot);
    return (int)hipGetLastError();
  }
  if (K % 32 || ldx % 8 || hx % 8 || (((uintptr_t)x | (uintptr_t)W) & 15)) return -3;
  const int mt = (T + 15) / 16;
  if (mt > 65535) return -4;
  heads_mfma_kernel<<<dim3((N + 63) / 64 + (positions ? 1 : 0), H, mt), 64, 0, s>>>(
      (bf16_t*)out, ldo, ho, (const bf16_t*)x, ldx, hx, (const bf16_t*)W, T, N, K,
      (const bf16_t*)gate, ldg, rot);
  return (int)hipGetLastError();
}

int omnia_latent_attend(void* out, int f32, const void* q, const void* cache,
                        const int* block_tables, int bt_stride, const int* q_start, int nseq,
                        const int* positions, int T, int page, int H, int Cp, int Lp, int window,
                        float scale, hipStream_t s) {
  const size_t lds = (size_t)(Lp + Cp + 256 + 8) * 4;
  if (H > 65535 || lds > 64 * 1024) return -1;
  if (T == 0) return 0;
  if (f32)
    attend_kernel<float><<<dim3(T, H), 256, lds, s>>>(
        (float*)out, (const float*)q, (const float*)cache, block_tables, bt_stride, q_start, nseq,
        positions, page, H, Cp, Lp, window, scale);
  else
    attend_kernel<bf16_t><<<dim3(T, H), 256, lds, s>>>(
        (bf16_t*)out, (const bf16_t*)q, (const bf16_t*)cache, block_tables, bt_stride, q_start,
        nseq, positions, page, H, Cp, Lp, window, scale);
  return (int)hipGetLastError();
}

#define OMNIA_LATENT_WIDTHS(X) X(64) X(96) X(128) X(192) X(256) X(320) X(448) X(576) X(640)

// 1 if the decode kernel covers these widths
int omnia_latent_decode_covers(int Cp, int Lp) {
  if (Cp % 16 || Lp < Cp) return 0;
#define OMNIA_LW(W) if (Lp == W) return 1;
  OMNIA_LATENT_WIDTHS(OMNIA_LW)
#undef OMNIA_LW
  return 0;
}

int omnia_latent_decode(void* out, float* part_o, float* part_ml, const void* q, const void* cache,
                        const int* block_tables, int bt_stride, const int* positions, int T,
                        int page, int H, int Cp, int Lp, int window, float scale, int splits,
                        int merge, hipStream_t s) {
  if (!omnia_latent_decode_covers(Cp, Lp) || splits < 1 || splits > 64) return -1;
  if (page < 1 || (page & (page - 1))) return -2;
  if (T == 0) return 0;
  int pl2 = 0;
  while ((1 << pl2) < page) ++pl2;
  // longest part a row can be cut into, in pages (its first key may lie inside a page)
  const int maxk = window > 0 && window < bt_stride * page ? window : bt_stride * page;
  const int part = ((maxk + splits - 1) / splits + 63) / 64 * 64;
  const size_t dyn = ((size_t)part / page + 2) * 4;
  if (dyn > 32 * 1024) return -3;
  const float sl2 = scale * 1.4426950408889634f;
  const int ht = H > 16 ? 2 : 1;
  const dim3 grid(T, (H + 16 * ht - 1) / (16 * ht), splits);
#define OMNIA_LD(HT, LW)                                                                     \
  decode_kernel<HT, LW><<<grid, 256, dyn, s>>>(                                              \
      (bf16_t*)out, part_o, part_ml, (const bf16_t*)q, (const bf16_t*)cache, block_tables,   \
      bt_stride, positions, pl2, H, Cp, window, sl2)
#define OMNIA_LW(W)                                          \
  if (Lp == W) {                                             \
    if (ht == 2) OMNIA_LD(2, W); else OMNIA_LD(1, W);        \
  }
  OMNIA_LATENT_WIDTHS(OMNIA_LW)
#undef OMNIA_LW
#undef OMNIA_LD
  if (splits > 1 && merge)
    merge_kernel<<<T * H, 128, 0, s>>>((bf16_t*)out, part_o, part_ml, positions, H, Cp, window,
                                       splits);
  return (int)hipGetLastError();
}

// the merge of omnia_latent_decode (not yet merged) and omnia_latent_heads with W [H, N, K] of its
// latents o [T, H, K], in one launch
int omnia_latent_expand(void* out, int64_t ldo, int ho, const void* o, const float* part_o,
                        const float* part_ml, const void* W, const void* gate, int64_t ldg,
                        const int* positions, int T, int H, int N, int K, int window, int splits,
                        hipStream_t s) {
  if (K % 32 || K < 32 || K > 512 || N < 1 || N > 128 || ho < N) return -1;
  if (splits < 1 || splits > 64 || (splits > 1 && (!part_o || !part_ml)) || !gate) return -2;
  if (((uintptr_t)o | (uintptr_t)W | (uintptr_t)part_o) & 15) return -3;
  if (T == 0) return 0;
  // rows a block: blocks of about one a CU
  const int64_t heads = (int64_t)T * H;
  const int rb = heads > 8 * 256 ? 16 : heads > 4 * 256 ? 8 : 4;
  const int64_t gy = (T + rb - 1) / rb;
  if (gy > 65535) return -4;
  expand_kernel<<<dim3(H, (unsigned)gy), 512, 0, s>>>(
      (bf16_t*)out, ldo, ho, (const bf16_t*)o, part_o, part_ml, (const bf16_t*)W,
      (const bf16_t*)gate, ldg, positions, T, H, N, K, window, splits, rb);
  return (int)hipGetLastError();
}

int omnia_latent_gather(void* c, void* kr, const void* cache, const int* block_tables,
                        int bt_stride, const int* kv_start, const int* kv_first,
                        const int* seq_lens, int nseq, int page, int Tk, int Cp, int Rp, int Lp,
                        hipStream_t s) {
  if (Cp % 8 || Rp % 8 || Lp % 8 || Lp < Cp + Rp) return -1;
  if (Tk == 0) return 0;
  gather_kernel<<<(Tk + 3) / 4, 256, 0, s>>>((bf16_t*)c, (bf16_t*)kr, (const bf16_t*)cache,
                                            block_tables, bt_stride, kv_start, kv_first, seq_lens,
                                            nseq, page, Tk, Cp, Rp, Lp);
  return (int)hipGetLastError();
}

int omnia_latent_prefill(void* out, const void* q, const void* kx, const void* kr, const void* vt,
                         const int* q_start, const int* seq_lens, const int* kv_start,
                         const int* kv_first, const int* tile_seq, const int* tile_q0, int n_tiles,
                         int H, int QW, int Da, int Rp, int VW, int Tk, int window, float scale,
                         const void* gate, int64_t ldg, hipStream_t s) {
  if (Da % 8 || Rp % 8 || Da + Rp > QW || Tk % 64) return -1;
  if (n_tiles == 0) return 0;
  if ((int64_t)n_tiles * H > 2147483647LL) return -2;
  const float sl2 = scale * 1.4426950408889634f;
#define OMNIA_LP(Q, V)                                                                        \
  if (QW == Q && VW == V) {                                                                   \
    prefill_kernel<Q, V><<<n_tiles * H, 256, 0, s>>>(                                         \
        (bf16_t*)out, (const bf16_t*)q, (const bf16_t*)kx, (const bf16_t*)kr,                 \
        (const bf16_t*)vt, q_start, seq_lens, kv_start, kv_first, tile_seq, tile_q0, n_tiles, \
        H, Da, Rp, Tk, window, sl2, (const bf16_t*)gate, ldg);                                \
    return (int)hipGetLastError();                                                            \
  }
#define OMNIA_LPV(Q) OMNIA_LP(Q, 32) OMNIA_LP(Q, 64) OMNIA_LP(Q, 128)
  OMNIA_LPV(32) OMNIA_LPV(64) OMNIA_LPV(96) OMNIA_LPV(128) OMNIA_LPV(192) OMNIA_LPV(256)
#undef OMNIA_LPV
#undef OMNIA_LP
  return -3;
}

}  // extern "C"
