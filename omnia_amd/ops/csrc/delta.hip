// Gated delta rule for gfx950: a recurrence with a [dim x vdim] fp32 state per
// sequence and value head,
//
//     S <- g S ;  u = beta (v - S^T k) ;  S <- S + k u^T ;  o = S^T q
//
// whose q, k, v are short causal convolutions (silu) of projections, q and k made
// unit vectors per head.  One fused input projection feeds it, a row of
//     [q (KH*D) | k (KH*D) | v (H*V) | z (H*V) | b (H) | a (H)]     (row stride ldx).
//
//   delta_prep   convolutions, unit norms, decay and step size of every token
//   delta_step   decode: one token per sequence -- state update, per-head RMS norm and
//                the silu(z) output gate in one launch, one workgroup per (row, head)
//   delta_scan   prefill: each sequence's new tokens in blocks of 16, the state in MFMA
//                accumulators (delta_blocks first solves every block's 16 x 16 system);
//                key dimensions past 256 take a token-by-token scan instead
//   delta_norm   prefill: RMS norm + output gate of the scanned rows
//
// State of sequence slot s: state[s][h][D][Vp] fp32 and conv_state[s][taps-1][C], the
// last taps-1 projection rows (oldest first, in the storage type).  A sequence whose
// first row of this launch is at position 0 starts from zeros, whatever its slot held:
// slots are never cleared.  A negative slot (padded graph row) reads and writes nothing.
// delta_prep only READS conv_state; the step / scan launch that follows it shifts it.
// Everything that enters the recurrence is fp32; decays are carried as logarithms.
#include "common.h"

using namespace omnia;

namespace {

struct Rows {  // which sequence a row belongs to
  const int* q_start;  // null: decode, row = sequence
  int nseq;
  const int* positions;
  const int* slots;  // [nseq]
};

__device__ __forceinline__ int seq_of(const Rows& r, int t, int& row0) {
  if (!r.q_start) {
    row0 = t;
    return t;
  }
  int lo = 0, hi = r.nseq - 1;  // last s with q_start[s] <= t
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (r.q_start[mid] <= t) lo = mid; else hi = mid - 1;
  }
  row0 = r.q_start[lo];
  return lo;
}

// convolution input of channel c at row t - back (back >= 0), zeros before the start
template <typename T>
__device__ __forceinline__ float conv_in(const T* __restrict__ x, int64_t ldx,
                                         const T* __restrict__ cs, int t, int row0, bool fresh,
                                         int taps, int C, int c, int back) {
  const int r = t - back;
  if (r >= row0) return ldf(x + (int64_t)r * ldx + c);
  if (fresh) return 0.f;
  return ldf(cs + (int64_t)(taps - 1 - (row0 - r)) * C + c);
}

// ------------------------------------------------------------------ delta_prep
// grid (T, ceil(units / 4)): one wave per unit -- a q head, a k head, a v head, or
// (last unit) the gates of all heads
template <typename T>
__global__ __launch_bounds__(256) void prep_kernel(
    float* __restrict__ qn, float* __restrict__ kn, T* __restrict__ vc, float* __restrict__ decay,
    float* __restrict__ beta, const T* __restrict__ x, int64_t ldx, const T* __restrict__ conv_w,
    const T* __restrict__ conv_state, const float* __restrict__ a_log,
    const float* __restrict__ dt_bias, Rows rows, int KH, int H, int D, int Dp, int V, int taps) {
  const int t = blockIdx.x, lane = threadIdx.x & 63;
  const int u = blockIdx.y * 4 + (threadIdx.x >> 6);
  const int units = 2 * KH + H + 1;
  if (u >= units) return;
  int row0;
  const int s = seq_of(rows, t, row0);
  const int slot = rows.slots[s];
  const int C = 2 * KH * D + H * V;
  const bool fresh = slot < 0 || rows.positions[row0] == 0;
  const T* cs = conv_state + (int64_t)(slot < 0 ? 0 : slot) * (taps - 1) * C;
  if (u == units - 1) {
    const T* xr = x + (int64_t)t * ldx + C + H * V;
    for (int h = lane; h < H; h += 64) {
      beta[(int64_t)t * H + h] = sigmoidf_(ldf(xr + h));
      const float z = ldf(xr + H + h) + dt_bias[h];
      const float sp = z > 20.f ? z : log1pf(expf(z));
      decay[(int64_t)t * H + h] = -expf(a_log[h]) * sp;
    }
    return;
  }
  const int n = u < 2 * KH ? D : V;
  const int c0 = u < 2 * KH ? u * D : 2 * KH * D + (u - 2 * KH) * V;
  float ss = 0.f;
  float* qk = u < KH ? qn + ((int64_t)t * KH + u) * Dp : kn + ((int64_t)t * KH + (u - KH)) * Dp;
  T* vr = vc + (int64_t)t * H * V + (c0 - 2 * KH * D);
  for (int i = lane; i < n; i += 64) {
    const int c = c0 + i;
    float y = 0.f;
    for (int j = 0; j < taps; ++j)
      y += conv_in(x, ldx, cs, t, row0, fresh, taps, C, c, taps - 1 - j) *
           ldf(conv_w + (int64_t)c * taps + j);
    y = siluf_(y);
    if (u < 2 * KH) {
      ss += y * y;
      qk[i] = y;
    } else {
      stf(vr + i, y);
    }
  }
  if (u >= 2 * KH) return;
  ss = wave_sum(ss);
  float inv = 1.f / sqrtf(ss + 1e-6f);
  if (u < KH) inv *= 1.f / sqrtf((float)D);
  for (int i = lane; i < n; i += 64) qk[i] *= inv;  // each lane rescales what it wrote
  for (int i = n + lane; i < Dp; i += 64) qk[i] = 0.f;
}

// Fast path (taps <= 4, head sizes up to 64 * VEC * NE, even when VEC = 2): a wave takes
// a run of TR consecutive rows of one unit: 8, which reads 11 rows for 8, or 4 while the chip holds
// the waves of all of them at once (32 a CU), since the time is then the chain of a run (us in runs of
// 16 / 8 / 4, 32 units of 128 channels: 100 rows 13.5 / 8.8 / 6.3, 999 17.8 / 12.8 / 11.9, 1300 19.8 /
// 15.1 / 17.1, 8000 69 / 66 / 80; 64 units: 333 16.0 / 11.2 / 9.4, 600 19.3 / 14.1 / 15.9, 999 21.2 / 20.0 /
// 22.1; 128 units: 200 17.8 / 12.3 / 11.0, 333 20.0 / 15.4 / 17.0; 8 units: 4000 18 / 13 / 12.5).  The
// raw inputs of the run are loaded up front, the convolution slides over them in registers, and a
// sequence that starts inside the run (or the run's own start) reloads the taps - 1 inputs before it.
template <typename T, int VEC>
struct Vec;
template <>
struct Vec<bf16_t, 1> {
  static __device__ __forceinline__ void ld(float* o, const bf16_t* p) { o[0] = bf2f(*p); }
  static __device__ __forceinline__ void st(bf16_t* p, const float* v) { *p = f2bf(v[0]); }
};
template <>
struct Vec<bf16_t, 2> {
  static __device__ __forceinline__ void ld(float* o, const bf16_t* p) {
    const uint32_t u = *reinterpret_cast<const uint32_t*>(p);
    o[0] = __uint_as_float(u << 16);
    o[1] = __uint_as_float(u & 0xffff0000u);
  }
  static __device__ __forceinline__ void st(bf16_t* p, const float* v) {
    *reinterpret_cast<uint32_t*>(p) = pack_bf2(v[0], v[1]);
  }
};
template <>
struct Vec<float, 1> {
  static __device__ __forceinline__ void ld(float* o, const float* p) { o[0] = *p; }
  static __device__ __forceinline__ void st(float* p, const float* v) { *p = v[0]; }
};
template <>
struct Vec<float, 2> {
  static __device__ __forceinline__ void ld(float* o, const float* p) {
    const float2 u = *reinterpret_cast<const float2*>(p);
    o[0] = u.x;
    o[1] = u.y;
  }
  static __device__ __forceinline__ void st(float* p, const float* v) {
    *reinterpret_cast<float2*>(p) = make_float2(v[0], v[1]);
  }
};

template <typename T, int VEC, int NE, int TAPS, int TR>
__global__ __launch_bounds__(256) void prep_run_kernel(
    float* __restrict__ qn, float* __restrict__ kn, T* __restrict__ vc, float* __restrict__ decay,
    float* __restrict__ beta, const T* __restrict__ x, int64_t ldx, const T* __restrict__ conv_w,
    const T* __restrict__ conv_state, const float* __restrict__ a_log,
    const float* __restrict__ dt_bias, Rows rows, int n_rows, int KH, int H, int D, int Dp, int V) {
  const int t0 = blockIdx.x * TR, lane = threadIdx.x & 63;
  const int u = blockIdx.y * 4 + (threadIdx.x >> 6);
  const int units = 2 * KH + H + 1;
  if (u >= units) return;
  const int nt = min(TR, n_rows - t0);
  const int C = 2 * KH * D + H * V;
  if (u == units - 1) {
    for (int i = lane; i < nt * H; i += 64) {
      const int t = t0 + i / H, h = i % H;
      const T* xr = x + (int64_t)t * ldx + C + H * V;
      beta[(int64_t)t * H + h] = sigmoidf_(ldf(xr + h));
      const float z = ldf(xr + H + h) + dt_bias[h];
      const float sp = z > 20.f ? z : log1pf(expf(z));
      decay[(int64_t)t * H + h] = -expf(a_log[h]) * sp;
    }
    return;
  }
  const bool isv = u >= 2 * KH;
  const int n = isv ? V : D;
  const int c0 = isv ? 2 * KH * D + (u - 2 * KH) * V : u * D;
  float w[NE][VEC][TAPS], in[TR][NE][VEC];
#pragma unroll
  for (int e = 0; e < NE; ++e) {
    const int i = (e * 64 + lane) * VEC;
    // VEC channels' taps are one run of VEC * TAPS (even) elements
#pragma unroll
    for (int v = 0; v < VEC * TAPS; v += 2) {
      float t2[2] = {0.f, 0.f};
      if (i < n) Vec<T, 2>::ld(t2, conv_w + (int64_t)(c0 + i) * TAPS + v);
      w[e][v / TAPS][v % TAPS] = t2[0];
      w[e][(v + 1) / TAPS][(v + 1) % TAPS] = t2[1];
    }
#pragma unroll
    for (int r = 0; r < TR; ++r) {
#pragma unroll
      for (int v = 0; v < VEC; ++v) in[r][e][v] = 0.f;
      if (i < n && r < nt) Vec<T, VEC>::ld(in[r][e], x + (int64_t)(t0 + r) * ldx + c0 + i);
    }
  }
  int row0, s = seq_of(rows, t0, row0);
  int next = rows.q_start ? rows.q_start[s + 1] : t0 + 1;
  float hist[TAPS][NE][VEC];  // the TAPS - 1 inputs before the current row, oldest first
  auto reload = [&](int t) {
    const int slot = rows.slots[s];
    const bool fresh = slot < 0 || rows.positions[row0] == 0;
    const T* cs = conv_state + (int64_t)(slot < 0 ? 0 : slot) * (TAPS - 1) * C;
#pragma unroll
    for (int j = 0; j < TAPS - 1; ++j) {
      const int r = t - (TAPS - 1 - j);  // wave-uniform source row
      const T* src = r >= row0 ? x + (int64_t)r * ldx : cs + (int64_t)(TAPS - 1 - (row0 - r)) * C;
      const bool zero = r < row0 && fresh;
#pragma unroll
      for (int e = 0; e < NE; ++e) {
        const int i = (e * 64 + lane) * VEC;
#pragma unroll
        for (int v = 0; v < VEC; ++v) hist[j][e][v] = 0.f;
        if (i < n && !zero) Vec<T, VEC>::ld(hist[j][e], src + c0 + i);
      }
    }
  };
  reload(t0);
#pragma unroll
  for (int r = 0; r < TR; ++r) {
    if (r >= nt) break;
    const int t = t0 + r;
    if (t >= next) {  // wave-uniform: the next sequence starts here
      do {
        ++s;
        row0 = next;
        next = rows.q_start ? rows.q_start[s + 1] : t + 1;
      } while (t >= next);
      reload(t);
    }
    float y[NE][VEC], ss = 0.f;
#pragma unroll
    for (int e = 0; e < NE; ++e)
#pragma unroll
      for (int v = 0; v < VEC; ++v) {
        float a = in[r][e][v] * w[e][v][TAPS - 1];
#pragma unroll
        for (int j = 0; j < TAPS - 1; ++j) a += hist[j][e][v] * w[e][v][j];
        a = siluf_(a);
        y[e][v] = a;
        ss += a * a;
#pragma unroll
        for (int j = 0; j + 1 < TAPS - 1; ++j) hist[j][e][v] = hist[j + 1][e][v];
        if (TAPS > 1) hist[TAPS - 2 < 0 ? 0 : TAPS - 2][e][v] = in[r][e][v];
      }
    if (isv) {
      T* vr = vc + (int64_t)t * H * V + (c0 - 2 * KH * D);
#pragma unroll
      for (int e = 0; e < NE; ++e) {
        const int i = (e * 64 + lane) * VEC;
        if (i < n) Vec<T, VEC>::st(vr + i, y[e]);
      }
    } else {
      ss = row_sum16(ss);
      ss += __shfl_xor(ss, 16, 64);
      ss += __shfl_xor(ss, 32, 64);
      float inv = 1.f / sqrtf(ss + 1e-6f);
      if (u < KH) inv *= 1.f / sqrtf((float)D);
      float* qk = u < KH ? qn + ((int64_t)t * KH + u) * Dp : kn + ((int64_t)t * KH + (u - KH)) * Dp;
#pragma unroll
      for (int e = 0; e < NE; ++e) {
        const int i = (e * 64 + lane) * VEC;
#pragma unroll
        for (int v = 0; v < VEC; ++v) y[e][v] *= inv;
        if (i < n) Vec<float, VEC>::st(qk + i, y[e]);
      }
      for (int i = n + lane; i < Dp; i += 64) qk[i] = 0.f;
    }
  }
}

// the conv state after rows [row0, row0 + n): the last taps-1 inputs.  One thread owns
// a channel, reads before it writes.
template <typename T>
__device__ __forceinline__ void shift_conv(const T* __restrict__ x, int64_t ldx, T* cs, int row0,
                                           int n, bool fresh, int taps, int C, int c) {
  // oldest first; new entry i comes from row0 + n - (taps-1) + i, or from the old state
  auto entry = [&](int i) -> T {
    const int r = n - (taps - 1) + i;  // relative to row0
    if (r >= 0) return x[(int64_t)(row0 + r) * ldx + c];
    if (fresh) return (T)0;
    return cs[(int64_t)(taps - 1 + r) * C + c];  // index >= i + n > i: not yet overwritten
  };
  if (taps <= 4) {  // all loads in flight together
    T v[3];
#pragma unroll
    for (int i = 0; i < 3; ++i)
      if (i < taps - 1) v[i] = entry(i);
#pragma unroll
    for (int i = 0; i < 3; ++i)
      if (i < taps - 1) cs[(int64_t)i * C + c] = v[i];
  } else {
    for (int i = 0; i < taps - 1; ++i) cs[(int64_t)i * C + c] = entry(i);
  }
}

// ------------------------------------------------------------------ delta_step
// grid (rows, H), 256 threads.  Thread (cg, rg): 4 state columns cg*4.., the rows
// rg, rg + RG, ... kept in registers (NR of them).  Bound by reading and writing the state, once
// each and not again before the next token: past the caches (non-temporal), and with all else it
// reads asked for before the first barrier.  us at 4 / 16 / 32 / 64 / 200 rows of 16 heads of 128,
// before -> now: 8.7 / 11.7 / 22 / 39 / 101 -> 8.3 / 9.9 / 16 / 28 / 84 (5.0 TB/s; the loads
// alone non-temporal 9.0 / 12.0 / 17.5 / 30 / 90).
template <typename T, int NR>
__global__ __launch_bounds__(256) void step_kernel(
    T* __restrict__ y, float* __restrict__ state, T* __restrict__ conv_state,
    const float* __restrict__ qn, const float* __restrict__ kn, const T* __restrict__ vc,
    const float* __restrict__ decay, const float* __restrict__ beta, const T* __restrict__ x,
    int64_t ldx, const float* __restrict__ norm_w, Rows rows, int KH, int H, int D, int Dp, int V,
    int Vs, int Vp, int taps, float eps) {
  extern __shared__ __attribute__((aligned(16))) float sm[];
  const int t = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
  const int slot = rows.slots[t];
  T* yr = y + ((int64_t)t * H + h) * Vp;
  if (slot < 0) {
    for (int i = tid; i < Vp; i += 256) stf(yr + i, 0.f);
    return;
  }
  const bool fresh = rows.positions[t] == 0;
  const int C = 2 * KH * D + H * V, CG = Vs / 4, RG = 256 / CG;
  float* ks = sm;             // [Dp]
  float* qs = ks + Dp;        // [Dp]
  float* red = qs + Dp;       // [RG][Vs]
  float* us = red + RG * Vs;  // [Vs]
  float* os = us + Vs;        // [Vs]
  float* scratch = os + Vs;   // [8]
  const int kh = h / (H / KH);
  const float* kr = kn + ((int64_t)t * KH + kh) * Dp;
  const float* qr = qn + ((int64_t)t * KH + kh) * Dp;
  const T* vr = vc + ((int64_t)t * H + h) * V;
  const T* zr = x + (int64_t)t * ldx + C + h * V;
  // a thread's first of each loop below over columns
  const float lg = decay[(int64_t)t * H + h], bt = beta[(int64_t)t * H + h];
  const int d0 = min(tid, Dp - 1), v0 = min(tid, V - 1);
  const float k0 = kr[d0], q0 = qr[d0], vv0 = ldf(vr + v0), z0 = ldf(zr + v0), w0 = norm_w[v0];
  const int cg = tid % CG, rg = tid / CG;
  const bool act = rg < RG;
  float4v* S = reinterpret_cast<float4v*>(state + (((int64_t)slot * H + h) * D) * Vs) + cg;
  float4v reg[NR];
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    const int d = rg + i * RG;
    reg[i] = (act && d < D && !fresh) ? __builtin_nontemporal_load(S + (int64_t)d * CG)
                                      : float4v{0.f, 0.f, 0.f, 0.f};
  }
  // this head's share of the convolution state (delta_prep has read it)
  const int per = (C + H - 1) / H;
  T* cs = conv_state + (int64_t)slot * (taps - 1) * C;
  for (int c = h * per + tid; c < min(C, (h + 1) * per); c += 256)
    shift_conv(x, ldx, cs, t, 1, fresh, taps, C, c);
  for (int i = tid; i < Dp; i += 256) {
    ks[i] = i < 256 ? k0 : kr[i];
    qs[i] = i < 256 ? q0 : qr[i];
  }
  __syncthreads();
  const float g = expf(lg);
  float4v acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    const int d = rg + i * RG;
    reg[i] *= g;
    if (d < D) acc += reg[i] * ks[d];
  }
  if (act) *reinterpret_cast<float4v*>(red + rg * Vs + cg * 4) = acc;
  __syncthreads();
  for (int j = tid; j < Vs; j += 256) {
    float sk = 0.f;
    for (int r = 0; r < RG; ++r) sk += red[r * Vs + j];
    us[j] = j < V ? bt * ((j < 256 ? vv0 : ldf(vr + j)) - sk) : 0.f;
  }
  __syncthreads();
  acc = float4v{0.f, 0.f, 0.f, 0.f};
  if (act) {
    const float4v u4 = *reinterpret_cast<const float4v*>(us + cg * 4);
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const int d = rg + i * RG;
      if (d < D) {
        reg[i] += u4 * ks[d];
        acc += reg[i] * qs[d];
        __builtin_nontemporal_store(reg[i], S + (int64_t)d * CG);
      }
    }
    *reinterpret_cast<float4v*>(red + rg * Vs + cg * 4) = acc;
  }
  __syncthreads();
  float ss = 0.f;
  for (int j = tid; j < Vs; j += 256) {
    float o = 0.f;
    for (int r = 0; r < RG; ++r) o += red[r * Vs + j];
    os[j] = o;
    if (j < V) ss += o * o;
  }
  ss = block_sum(ss, scratch);
  const float inv = 1.f / sqrtf(ss / (float)V + eps);
  for (int j = tid; j < Vp; j += 256) {
    const float z = j < 256 || j >= V ? z0 : ldf(zr + j), nw = j < 256 || j >= V ? w0 : norm_w[j];
    stf(yr + j, j < V ? os[j] * inv * nw * siluf_(z) : 0.f);
  }
}

// ------------------------------------------------------------------ delta_scan
// grid (ceil(Vs / 16), H, nseq), 256 threads: wave w, lane l -> state column
// blockIdx.x*16 + 4w + (l >> 4); lane l & 15 holds the key dimensions
// 64 i + 4 (l & 15) + {0..3}, i < NI.  Tokens go through LDS TC at a time.
constexpr int kTC = 16;

template <typename T, int NI>
__global__ __launch_bounds__(256) void scan_kernel(
    float* __restrict__ o, float* __restrict__ state, T* __restrict__ conv_state,
    const float* __restrict__ qn, const float* __restrict__ kn, const T* __restrict__ vc,
    const float* __restrict__ decay, const float* __restrict__ beta, const T* __restrict__ x,
    int64_t ldx, Rows rows, int KH, int H, int D, int Dp, int V, int Vs, int taps) {
  __shared__ __attribute__((aligned(16))) float kb[kTC][NI * 64];
  __shared__ __attribute__((aligned(16))) float qb[kTC][NI * 64];
  __shared__ float vb[kTC][16], gb[kTC], bb[kTC], ob[kTC][16];
  const int h = blockIdx.y, s = blockIdx.z, tid = threadIdx.x;
  const int lane = tid & 63, w = tid >> 6, lg = lane & 15, cl = 4 * w + (lane >> 4);
  const int col0 = blockIdx.x * 16, col = col0 + cl;
  const int row0 = rows.q_start[s], n = rows.q_start[s + 1] - row0;
  const int slot = rows.slots[s];
  if (n <= 0 || slot < 0) return;
  const bool fresh = rows.positions[row0] == 0;
  const int C = 2 * KH * D + H * V, kh = h / (H / KH);
  float* Sg = state + (((int64_t)slot * H + h) * D) * Vs + col;
  float4v S[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int d = 64 * i + 4 * lg + j;
      S[i][j] = (!fresh && d < D && col < Vs) ? Sg[(int64_t)d * Vs] : 0.f;
    }
  for (int t0 = 0; t0 < n; t0 += kTC) {
    const int m = min(kTC, n - t0);
    __syncthreads();  // the previous tokens' LDS reads are done
    for (int i = tid; i < kTC * NI * 16; i += 256) {
      const int tt = i / (NI * 16), d4 = (i % (NI * 16)) * 4;
      float4v kv = {0.f, 0.f, 0.f, 0.f}, qv = {0.f, 0.f, 0.f, 0.f};
      if (tt < m && d4 < Dp) {
        const int64_t e = ((int64_t)(row0 + t0 + tt) * KH + kh) * Dp + d4;
        kv = *reinterpret_cast<const float4v*>(kn + e);
        qv = *reinterpret_cast<const float4v*>(qn + e);
      }
      *reinterpret_cast<float4v*>(&kb[tt][d4]) = kv;
      *reinterpret_cast<float4v*>(&qb[tt][d4]) = qv;
    }
    {
      const int tt = tid >> 4, c = tid & 15;
      const int64_t row = (int64_t)(row0 + t0 + tt) * H + h;
      vb[tt][c] = (tt < m && col0 + c < V) ? ldf(vc + row * V + col0 + c) : 0.f;
      if (c == 0) {
        gb[tt] = tt < m ? expf(decay[row]) : 1.f;
        bb[tt] = tt < m ? beta[row] : 0.f;
      }
    }
    __syncthreads();
#pragma unroll 4
    for (int tt = 0; tt < kTC; ++tt) {  // rows past m: g = 1, beta = 0 leave S as it is
      const float g = gb[tt];
      float4v kr[NI], qr[NI];
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        kr[i] = *reinterpret_cast<const float4v*>(&kb[tt][64 * i + 4 * lg]);
        qr[i] = *reinterpret_cast<const float4v*>(&qb[tt][64 * i + 4 * lg]);
      }
      float4v a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        S[i] *= g;
        a += S[i] * kr[i];
      }
      const float sk = row_sum16((a[0] + a[1]) + (a[2] + a[3]));
      const float u = bb[tt] * (vb[tt][cl] - sk);
      float4v b = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        S[i] += kr[i] * u;
        b += S[i] * qr[i];
      }
      const float ov = row_sum16((b[0] + b[1]) + (b[2] + b[3]));
      if (lg == 0) ob[tt][cl] = ov;
    }
    __syncthreads();
    {
      const int tt = tid >> 4, c = tid & 15;
      if (tt < m && col0 + c < Vs)
        o[((int64_t)(row0 + t0 + tt) * H + h) * Vs + col0 + c] = ob[tt][c];
    }
  }
  if (col < Vs) {
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int d = 64 * i + 4 * lg + j;
        if (d < D) Sg[(int64_t)d * Vs] = S[i][j];
      }
  }
  // convolution state: channels dealt over the sequence's workgroups
  const int nb = gridDim.x * H, b = blockIdx.x * H + h, per = (C + nb - 1) / nb;
  T* cs = conv_state + (int64_t)slot * (taps - 1) * C;
  for (int c = b * per + tid; c < min(C, (b + 1) * per); c += 256)
    shift_conv(x, ldx, cs, row0, n, fresh, taps, C, c);
}

// ---------------------------------------------------------------- blocked scan
// Within a block of 16 tokens, with c_t the running sum of log g, G_t = exp(c_t) and S0
// the state before it,
//     u_t = beta_t (v_t - G_t S0^T k_t - sum_{i<t} exp(c_t - c_i) (k_t . k_i) u_i)
//     o_t = G_t S0^T q_t + sum_{i<=t} exp(c_t - c_i) (q_t . k_i) u_i
//     S   = G_15 S0 + sum_i exp(c_15 - c_i) k_i u_i^T
// (every exponent is <= 0).  The system for U is unit lower triangular; its inverse and
// the q.k matrix depend on neither S0 nor v, so blocks_kernel makes them for all blocks
// at once and the serial part is only products.  All products are fp32 MFMA
// (16x16x4).  A block's record: T' [16][16] (inverse, columns scaled by beta),
// P [16][16], G [16], E [16] = exp(c_15 - c_i).  Tokens past the end: k = q = 0,
// log g = 0, beta = 0.
constexpr int kRec = 2 * 256 + 32;

__device__ __forceinline__ float4v mfma4(float a, float b, float4v c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// first record of sequence s: leaves room for every earlier sequence's ragged block
__device__ __forceinline__ int rec_base(const int* q_start, int s) { return q_start[s] / 16 + s; }

// grid (records, ceil(H / 4)): one wave per (block, head)
template <int ND>
__global__ __launch_bounds__(256) void blocks_kernel(float* __restrict__ rec,
                                                     const float* __restrict__ qn,
                                                     const float* __restrict__ kn,
                                                     const float* __restrict__ decay,
                                                     const float* __restrict__ beta,
                                                     const int* __restrict__ q_start, int nseq,
                                                     int KH, int H, int Dp) {
  __shared__ __attribute__((aligned(16))) float Ls[4][16][20];
  const int id = blockIdx.x, w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int h = blockIdx.y * 4 + w, c16 = lane & 15, g4 = lane >> 4;
  int lo = 0, hi = nseq - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (rec_base(q_start, mid) <= id) lo = mid; else hi = mid - 1;
  }
  const int row0 = q_start[lo], t0 = (id - rec_base(q_start, lo)) * 16;
  const int m = min(16, q_start[lo + 1] - row0 - t0);
  if (m <= 0 || h >= H) return;  // no barrier below: waves are independent
  const int kh = h / (H / KH);
  const bool in = c16 < m;
  const int64_t row = row0 + t0 + (in ? c16 : 0);
  const float* kr = kn + (row * KH + kh) * Dp + 4 * g4;
  const float* qr = qn + (row * KH + kh) * Dp + 4 * g4;
  float4v kk = {0.f, 0.f, 0.f, 0.f}, qk = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < ND; ++j) {
    float4v a = {0.f, 0.f, 0.f, 0.f}, b = a;
    if (in && 16 * j + 4 * g4 < Dp) {
      a = *reinterpret_cast<const float4v*>(kr + 16 * j);
      b = *reinterpret_cast<const float4v*>(qr + 16 * j);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      kk = mfma4(a[r], a[r], kk);
      qk = mfma4(b[r], a[r], qk);
    }
  }
  const float bt = in ? beta[row * H + h] : 0.f;
  float c = in ? decay[row * H + h] : 0.f;
#pragma unroll
  for (int o = 1; o < 16; o <<= 1) {
    const float up = __shfl_up(c, o, 16);
    if (c16 >= o) c += up;
  }
  float* R = rec + ((int64_t)id * H + h) * kRec;
  // lane: column i = c16, rows t = 4 g4 + r
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int t = 4 * g4 + r;
    const float ct = __shfl(c, t, 16), btt = __shfl(bt, t, 16);
    const float e = c16 <= t ? expf(ct - c) : 0.f;
    Ls[w][t][c16] = c16 < t ? btt * e * kk[r] : 0.f;
    R[256 + t * 16 + c16] = e * qk[r];
  }
  __builtin_amdgcn_wave_barrier();
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // this wave's LDS writes
  float T[16];  // column c16 of the inverse, by forward substitution
#pragma unroll
  for (int t = 0; t < 16; ++t) {
    float a = t == c16 ? 1.f : 0.f;
#pragma unroll
    for (int i = 0; i < t; i += 4) {
      const float4v l = *reinterpret_cast<const float4v*>(&Ls[w][t][i]);
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (i + r < t) a -= l[r] * T[i + r];
    }
    T[t] = a;
  }
  if (g4 == 0) {
#pragma unroll
    for (int t = 0; t < 16; ++t) R[t * 16 + c16] = T[t] * bt;
    R[512 + c16] = expf(c);
    R[528 + c16] = expf(__shfl(c, 15, 16) - c);
  }
}

// grid (ceil(Vs / 64), H, nseq), 4 waves: wave w owns state columns 64 x + 16 w + ..15
// as ND accumulator tiles (key dimensions 16 j + 4 (lane >> 4) + r in register r).  The
// accumulator layout serves as the B operand of the next product as it stands: k-step r
// takes dimension (token) 4 (lane >> 4) + r, and the A side is read in that order.
// Bound by its serial chain: a block is 104 fp32 products of one wave (heads of 128), 1.4 of the
// 3.0 us that it takes in a step, and a SIMD has one wave.  Vector instructions add to that, so
// registers hold 2 waves' worth (with more, hipcc keeps S in the accumulators' file and moves it
// back and forth), offsets are made once, and what is not a product goes between products.  16
// heads of 128 in a model step, whose weights leave no operand in the caches: 2048 rows of 8
// sequences 430 -> 381 us (blocks_kernel 66 beside it, as before), 333 of 3 65 -> 59.  Alone and
// repeated, both kernels 371 -> 330 and 68 -> 61.
template <typename T, int ND>
__global__ __launch_bounds__(256, ND <= 8 ? 2 : 1) void scan_blocks_kernel(
    float* __restrict__ o, float* __restrict__ state, T* __restrict__ conv_state,
    const float* __restrict__ rec, const float* __restrict__ qn, const float* __restrict__ kn,
    const T* __restrict__ vc, const T* __restrict__ x, int64_t ldx, Rows rows, int KH, int H,
    int D, int Dp, int V, int Vs, int taps) {
  constexpr int DW = 16 * ND, KS = DW + 4, TS = 20;
  constexpr int NL = (16 * DW / 4 + 255) / 256;  // float4 per thread of one operand block
  // one block's operands; two of them, so the next block is written while this is read
  struct Buf {
    float k[16 * KS], q[16 * KS], t[16 * TS], p[16 * TS], g[32];
  };
  __shared__ __attribute__((aligned(16))) Buf buf[2];
  const int h = blockIdx.y, s = blockIdx.z, tid = threadIdx.x;
  const int lane = tid & 63, w = tid >> 6, c16 = lane & 15, g4 = lane >> 4;
  const int col = blockIdx.x * 64 + 16 * w + c16;
  const int row0 = rows.q_start[s], n = rows.q_start[s + 1] - row0;
  const int slot = rows.slots[s];
  if (n <= 0 || slot < 0) return;
  const bool fresh = rows.positions[row0] == 0;
  const int C = 2 * KH * D + H * V, kh = h / (H / KH);
  float* Sg = state + (((int64_t)slot * H + h) * D) * Vs + col;
  float4v S[ND];
#pragma unroll
  for (int j = 0; j < ND; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int d = 16 * j + 4 * g4 + r;
      S[j][r] = (!fresh && d < D && col < Vs) ? Sg[(int64_t)d * Vs] : 0.f;
    }
  // this thread's share of a block: element e of [16][DW / 4] float4s
  float4v kreg[NL], qreg[NL];
  T vreg[4];
  float treg[2], greg;
  // Vector instructions do not run beside the fp32 products, so addresses are a uniform base and
  // an offset made once.  Loads are unconditional, so that they all are in flight together: rows
  // past the end re-read the last one (their u is 0 whatever k, q and v hold) and columns past
  // the head re-read its last ones (zeroed when they are used).
  const float* R = rec + ((int64_t)rec_base(rows.q_start, s) * H + h) * kRec;
  const int64_t kofs = ((int64_t)row0 * KH + kh) * Dp;
  const T* vp = vc + ((int64_t)row0 * H + h) * V;
  const int64_t kstep = (int64_t)16 * KH * Dp, vstep = (int64_t)16 * H * V;
  const int kd4 = tid % (DW / 4) * 4, vcol = min(col, V - 1);
  uint32_t koff[NL], voff[4];
  auto offsets = [&](int last) {
#pragma unroll
    for (int i = 0; i < NL; ++i)
      koff[i] = min((i * 256 + tid) / (DW / 4), last) * KH * Dp + min(kd4, Dp - 4);
#pragma unroll
    for (int r = 0; r < 4; ++r) voff[r] = min(4 * g4 + r, last) * H * V + vcol;
  };
  auto gload = [&](int bi) {
    const float* kb = kn + kofs + bi * kstep;
    const float* qb = qn + kofs + bi * kstep;
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      kreg[i] = *reinterpret_cast<const float4v*>(kb + koff[i]);
      qreg[i] = *reinterpret_cast<const float4v*>(qb + koff[i]);
    }
    const T* vb = vp + bi * vstep;
#pragma unroll
    for (int r = 0; r < 4; ++r) vreg[r] = vb[voff[r]];
    const float* rr = R + (int64_t)bi * H * kRec;
    treg[0] = rr[(uint32_t)tid];
    treg[1] = rr[256 + (uint32_t)tid];
    greg = rr[512 + (uint32_t)(tid & 31)];
  };
  auto lwrite_rows = [&](Buf& b) {  // k columns past Dp hold zeros from the start
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int tt = (i * 256 + tid) / (DW / 4);
      if (kd4 < Dp && (16 * DW / 4 % 256 == 0 || tt < 16)) {
        *reinterpret_cast<float4v*>(b.k + tt * KS + kd4) = kreg[i];
        *reinterpret_cast<float4v*>(b.q + tt * KS + kd4) = qreg[i];
      }
    }
  };
  auto lwrite_rest = [&](Buf& b) {
    b.t[(tid >> 4) * TS + (tid & 15)] = treg[0];
    b.p[(tid >> 4) * TS + (tid & 15)] = treg[1];
    b.g[tid & 31] = greg;
  };
  const int nblk = (n + 15) / 16;
  float* op = o + ((int64_t)row0 * H + h) * Vs;
  const uint32_t ooff = 4 * g4 * H * Vs + col;
  const int64_t ostep = (int64_t)16 * H * Vs;
  // Operands in registers ahead of their products (heads up to 128; wider ones read LDS as they
  // go): k of the next block from the middle of this one, the rest from the top of the block.
  constexpr bool PRE = ND <= 8;
  float4v ka[PRE ? ND : 1], qa[PRE ? ND : 1];
  float ku[4][PRE ? ND : 1];
  auto rows_of = [&](const float* x, int j) {
    return *reinterpret_cast<const float4v*>(x + c16 * KS + 16 * j + 4 * g4);
  };
  // LDS only: the loads of later blocks stay in flight
  auto sync = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
  float4v v, vnext;
  auto values = [&] {
    float4v t;
#pragma unroll
    for (int r = 0; r < 4; ++r) t[r] = col < V ? ldf(&vreg[r]) : 0.f;
    return t;
  };
  if (Dp < DW) {
    for (int i = tid; i < 2 * (int)sizeof(Buf) / 4; i += 256)
      reinterpret_cast<float*>(buf)[i] = 0.f;
    __syncthreads();
  }
  offsets(min(16, n) - 1);
  gload(0);
  lwrite_rows(buf[0]);
  lwrite_rest(buf[0]);
  v = values();
  if (nblk == 2) offsets(n - 17);
  gload(min(1, nblk - 1));
  sync();
  if constexpr (PRE) {
#pragma unroll
    for (int j = 0; j < ND; ++j) ka[j] = rows_of(buf[0].k, j);
  }
  for (int bi = 0; bi < nblk; ++bi) {
    const Buf& B = buf[bi & 1];
    Buf& N = buf[(bi + 1) & 1];
    float4v G, E, ta, pa;
    float G15;
    // what the block does beside its products, in eight pieces: the next block's operands go to
    // the buffer that every wave left before the last barrier, the loads of the one after it
    // (past the end: the last block's once more) are issued, this block's other operands read
    auto piece = [&](int i) {
      if (i == 0) lwrite_rows(N);
      if (i == 1) {
        lwrite_rest(N);
        vnext = values();
      }
      if (i == 2) {
        const int b = min(bi + 2, nblk - 1);
        if (b == nblk - 1) offsets(n - 16 * b - 1);
        gload(b);
      }
      if (i == 3) {
        G = *reinterpret_cast<const float4v*>(B.g + 4 * g4);
        E = *reinterpret_cast<const float4v*>(B.g + 16 + 4 * g4);
        G15 = B.g[15];
        ta = *reinterpret_cast<const float4v*>(B.t + c16 * TS + 4 * g4);
        pa = *reinterpret_cast<const float4v*>(B.p + c16 * TS + 4 * g4);
        if constexpr (PRE) {
#pragma unroll
          for (int j = 0; j < ND; ++j) qa[j] = rows_of(B.q, j);
        }
      }
      if constexpr (PRE) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (i == 4 + r) {
#pragma unroll
            for (int j = 0; j < ND; ++j) ku[r][j] = B.k[(4 * g4 + r) * KS + 16 * j + c16];
          }
      }
    };
    float4v ks[2], qs[2];
#pragma unroll
    for (int c = 0; c < 2; ++c) ks[c] = qs[c] = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < ND; ++j) {
      const float4v a = PRE ? ka[PRE ? j : 0] : rows_of(B.k, j);
#pragma unroll
      for (int r = 0; r < 4; ++r) ks[r & 1] = mfma4(a[r], S[j][r], ks[r & 1]);
      if constexpr (!PRE) {
        const float4v b = rows_of(B.q, j);
#pragma unroll
        for (int r = 0; r < 4; ++r) qs[r & 1] = mfma4(b[r], S[j][r], qs[r & 1]);
      }
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (i * ND / 8 == j) {
          if constexpr (PRE) __builtin_amdgcn_sched_barrier(0);
          piece(i);
          if constexpr (PRE) __builtin_amdgcn_sched_barrier(0);
        }
    }
    if constexpr (PRE) {
      sync();
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < ND; ++j) ka[j] = rows_of(N.k, j);
      __builtin_amdgcn_sched_barrier(0);
    }
    const float4v res = v - G * (ks[0] + ks[1]);
    float4v u = {0.f, 0.f, 0.f, 0.f};
    // the chain of u runs between the products with q, which do not need it
#pragma unroll
    for (int j = 0; j < ND; ++j) {
      if constexpr (PRE) {
#pragma unroll
        for (int r = 0; r < 4; ++r) qs[r & 1] = mfma4(qa[j][r], S[j][r], qs[r & 1]);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (r * ND / 4 == j) u = mfma4(ta[r], res[r], u);
      if constexpr (PRE) __builtin_amdgcn_sched_barrier(0);
    }
    float4v ov = G * (qs[0] + qs[1]);
#pragma unroll
    for (int j = 0; j < ND; ++j) S[j] *= G15;
    const float4v ue = u * E;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      ov = mfma4(pa[r], u[r], ov);
#pragma unroll
      for (int j = 0; j < ND; ++j)
        S[j] = mfma4(PRE ? ku[r][PRE ? j : 0] : B.k[(4 * g4 + r) * KS + 16 * j + c16], ue[r], S[j]);
    }
    if constexpr (!PRE) sync();
    if (col < Vs) {
      const int m = n - 16 * bi;
      if (m >= 16) {
#pragma unroll
        for (int r = 0; r < 4; ++r) (op + bi * ostep + r * H * Vs)[ooff] = ov[r];
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (4 * g4 + r < m) (op + bi * ostep + r * H * Vs)[ooff] = ov[r];
      }
    }
    v = vnext;
  }
  if (col < Vs) {
#pragma unroll
    for (int j = 0; j < ND; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int d = 16 * j + 4 * g4 + r;
        if (d < D) Sg[(int64_t)d * Vs] = S[j][r];
      }
  }
  const int nb = gridDim.x * H, b = blockIdx.x * H + h, per = (C + nb - 1) / nb;
  T* cs = conv_state + (int64_t)slot * (taps - 1) * C;
  for (int c = b * per + tid; c < min(C, (b + 1) * per); c += 256)
    shift_conv(x, ldx, cs, row0, n, fresh, taps, C, c);
}

// ------------------------------------------------------------------ delta_norm
// one wave per NB consecutive (row, head) pairs, 64 * VEC * NE >= V
template <typename T, int VEC, int NE, int NB>
__global__ __launch_bounds__(256) void norm_kernel(
    T* __restrict__ y, const float* __restrict__ o, const T* __restrict__ x, int64_t ldx, int zoff,
    const float* __restrict__ norm_w, int64_t n, int H, int V, int Vs, int Vp, float eps) {
  const int64_t i0 = ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * NB;
  const int lane = threadIdx.x & 63;
  float ov[NB][NE][VEC], zv[NB][NE][VEC], w[NE][VEC];
#pragma unroll
  for (int e = 0; e < NE; ++e) {
    const int c = (e * 64 + lane) * VEC;
#pragma unroll
    for (int v = 0; v < VEC; ++v) w[e][v] = c < V ? norm_w[c + v] : 0.f;
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const int64_t i = i0 + b;
#pragma unroll
      for (int v = 0; v < VEC; ++v) ov[b][e][v] = zv[b][e][v] = 0.f;
      if (i < n && c < V) {
        Vec<float, VEC>::ld(ov[b][e], o + i * Vs + c);
        Vec<T, VEC>::ld(zv[b][e], x + (i / H) * ldx + zoff + (int)(i % H) * V + c);
      }
    }
  }
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    const int64_t i = i0 + b;
    if (i >= n) return;
    float ss = 0.f;
#pragma unroll
    for (int e = 0; e < NE; ++e)
#pragma unroll
      for (int v = 0; v < VEC; ++v) ss += ov[b][e][v] * ov[b][e][v];
    const float inv = 1.f / sqrtf(wave_sum(ss) / (float)V + eps);
#pragma unroll
    for (int e = 0; e < NE; ++e) {
      const int c = (e * 64 + lane) * VEC;
      float r[VEC];
#pragma unroll
      for (int v = 0; v < VEC; ++v) r[v] = ov[b][e][v] * inv * w[e][v] * siluf_(zv[b][e][v]);
      if (c < Vp) Vec<T, VEC>::st(y + i * Vp + c, r);  // w = 0 past V: the padding is zero
    }
  }
}

template <typename T>
int prep(float* qn, float* kn, void* vc, float* decay, float* beta, const void* x, int64_t ldx,
         const void* conv_w, const void* conv_state, const float* a_log, const float* dt_bias,
         Rows r, int T_, int KH, int H, int D, int Dp, int V, int taps, hipStream_t s) {
  const int big = D > V ? D : V, vec = (D % 2 || V % 2) ? 1 : 2, ne = (big + 64 * vec - 1) / (64 * vec);
  const unsigned uy = (2 * KH + H + 1 + 3) / 4;
  const bool chain = (int64_t)T_ * (2 * KH + H) <= 4 * 32 * 256;  // runs of 4 at once
#define OMNIA_PREP(VEC, NE, TAPS, TR)                                                           \
  do {                                                                                          \
    prep_run_kernel<T, VEC, NE, TAPS, TR><<<dim3((T_ + (TR) - 1) / (TR), uy), 256, 0, s>>>(         \
        qn, kn, (T*)vc, decay, beta, (const T*)x, ldx, (const T*)conv_w, (const T*)conv_state,  \
        a_log, dt_bias, r, T_, KH, H, D, Dp, V);                                                \
    return (int)hipGetLastError();                                                              \
  } while (0)
#define OMNIA_PREP_R(VEC, NE, TAPS)                           \
  do {                                                        \
    if (r.q_start && !chain) OMNIA_PREP(VEC, NE, TAPS, 8);    \
    else if (r.q_start) OMNIA_PREP(VEC, NE, TAPS, 4);         \
    else OMNIA_PREP(VEC, NE, TAPS, 1);                        \
  } while (0)
#define OMNIA_PREP_T(VEC, NE)                  \
  do {                                         \
    if (taps == 2) OMNIA_PREP_R(VEC, NE, 2);   \
    if (taps == 3) OMNIA_PREP_R(VEC, NE, 3);   \
    if (taps == 4) OMNIA_PREP_R(VEC, NE, 4);   \
  } while (0)
  if (vec == 2 && ne == 1) OMNIA_PREP_T(2, 1);
  else if (vec == 2 && ne == 2) OMNIA_PREP_T(2, 2);
#undef OMNIA_PREP_T
#undef OMNIA_PREP_R
#undef OMNIA_PREP
  prep_kernel<T><<<dim3(T_, (2 * KH + H + 1 + 3) / 4), 256, 0, s>>>(
      qn, kn, (T*)vc, decay, beta, (const T*)x, ldx, (const T*)conv_w, (const T*)conv_state, a_log,
      dt_bias, r, KH, H, D, Dp, V, taps);
  return (int)hipGetLastError();
}

template <typename T>
int step(void* y, float* state, void* conv_state, const float* qn, const float* kn, const void* vc,
         const float* decay, const float* beta, const void* x, int64_t ldx, const float* norm_w,
         Rows r, int T_, int KH, int H, int D, int Dp, int V, int Vs, int Vp, int taps, float eps,
         hipStream_t s) {
  const int CG = Vs / 4, RG = 256 / CG, nr = (D + RG - 1) / RG;
  const size_t lds = (size_t)(2 * Dp + (RG + 2) * Vs + 8) * 4;
  if (lds > 64 * 1024) return -4;
#define OMNIA_STEP(N)                                                                          \
  if (nr <= N) {                                                                               \
    step_kernel<T, N><<<dim3(T_, H), 256, lds, s>>>(                                           \
        (T*)y, state, (T*)conv_state, qn, kn, (const T*)vc, decay, beta, (const T*)x, ldx,     \
        norm_w, r, KH, H, D, Dp, V, Vs, Vp, taps, eps);                                        \
    return (int)hipGetLastError();                                                             \
  }
  OMNIA_STEP(1) OMNIA_STEP(2) OMNIA_STEP(4) OMNIA_STEP(8) OMNIA_STEP(16) OMNIA_STEP(32)
  OMNIA_STEP(64)
#undef OMNIA_STEP
  return -5;
}

template <typename T>
int scan(float* o, float* state, void* conv_state, float* rec, const float* qn, const float* kn,
         const void* vc, const float* decay, const float* beta, const void* x, int64_t ldx, Rows r,
         int n_rows, int KH, int H, int D, int Dp, int V, int Vs, int taps, hipStream_t s) {
  const dim3 bgrid(n_rows / 16 + r.nseq, (H + 3) / 4), sgrid((Vs + 63) / 64, H, r.nseq);
#define OMNIA_SCANB(ND)                                                                         \
  if (D <= 16 * ND) {                                                                           \
    blocks_kernel<ND><<<bgrid, 256, 0, s>>>(rec, qn, kn, decay, beta, r.q_start, r.nseq, KH, H, \
                                            Dp);                                                \
    scan_blocks_kernel<T, ND><<<sgrid, 256, 0, s>>>(o, state, (T*)conv_state, rec, qn, kn,      \
                                                    (const T*)vc, (const T*)x, ldx, r, KH, H,   \
                                                    D, Dp, V, Vs, taps);                        \
    return (int)hipGetLastError();                                                              \
  }
  OMNIA_SCANB(2) OMNIA_SCANB(4) OMNIA_SCANB(8) OMNIA_SCANB(16)
#undef OMNIA_SCANB
  const dim3 grid((Vs + 15) / 16, H, r.nseq);
#define OMNIA_SCAN(N)                                                                           \
  if (D <= 64 * N) {                                                                            \
    scan_kernel<T, N><<<grid, 256, 0, s>>>(o, state, (T*)conv_state, qn, kn, (const T*)vc,      \
                                           decay, beta, (const T*)x, ldx, r, KH, H, D, Dp, V,   \
                                           Vs, taps);                                           \
    return (int)hipGetLastError();                                                              \
  }
  OMNIA_SCAN(6)
#undef OMNIA_SCAN
  return -5;
}

}  // namespace

extern "C" {

int omnia_delta_prep(float* qn, float* kn, void* vc, float* decay, float* beta, const void* x,
                     int f32, int64_t ldx, const void* conv_w, const void* conv_state,
                     const float* a_log, const float* dt_bias, const int* q_start, int nseq,
                     const int* positions, const int* slots, int T, int KH, int H, int D, int Dp,
                     int V, int taps, hipStream_t s) {
  if (taps < 1 || KH < 1 || H % KH || Dp % 4 || Dp < D) return -1;
  if (T == 0) return 0;
  const Rows r{q_start, nseq, positions, slots};
  if (f32)
    return prep<float>(qn, kn, vc, decay, beta, x, ldx, conv_w, conv_state, a_log, dt_bias, r, T,
                       KH, H, D, Dp, V, taps, s);
  return prep<bf16_t>(qn, kn, vc, decay, beta, x, ldx, conv_w, conv_state, a_log, dt_bias, r, T,
                      KH, H, D, Dp, V, taps, s);
}

int omnia_delta_step(void* y, float* state, void* conv_state, const float* qn, const float* kn,
                     const void* vc, const float* decay, const float* beta, const void* x, int f32,
                     int64_t ldx, const float* norm_w, const int* positions, const int* slots,
                     int T, int KH, int H, int D, int Dp, int V, int Vs, int Vp, int taps,
                     float eps, hipStream_t s) {
  if (taps < 1 || KH < 1 || H % KH || Dp % 4 || Dp < D || Vs % 4 || Vs < V || Vp < V) return -1;
  if (Vs / 4 > 256) return -2;
  if (T == 0) return 0;
  const Rows r{nullptr, T, positions, slots};
  if (f32)
    return step<float>(y, state, conv_state, qn, kn, vc, decay, beta, x, ldx, norm_w, r, T, KH, H,
                       D, Dp, V, Vs, Vp, taps, eps, s);
  return step<bf16_t>(y, state, conv_state, qn, kn, vc, decay, beta, x, ldx, norm_w, r, T, KH, H,
                      D, Dp, V, Vs, Vp, taps, eps, s);
}

// floats of the block records of n_rows rows in nseq sequences
int64_t omnia_delta_records(int n_rows, int nseq, int H) {
  return (int64_t)(n_rows / 16 + nseq) * H * kRec;
}

int omnia_delta_scan(float* o, float* state, void* conv_state, float* rec, const float* qn,
                     const float* kn, const void* vc, const float* decay, const float* beta,
                     const void* x, int f32, int64_t ldx, const int* q_start, int nseq,
                     const int* positions, const int* slots, int n_rows, int KH, int H, int D, int Dp, int V, int Vs, int taps,
                     hipStream_t s) {
  if (taps < 1 || KH < 1 || H % KH || Dp % 4 || Dp < D || Vs % 4 || Vs < V || n_rows < 0) return -1;
  if (nseq > 65535 || H > 65535) return -2;
  if (nseq == 0) return 0;
  const Rows r{q_start, nseq, positions, slots};
  if (f32)
    return scan<float>(o, state, conv_state, rec, qn, kn, vc, decay, beta, x, ldx, r, n_rows, KH,
                       H, D, Dp, V, Vs, taps, s);
  return scan<bf16_t>(o, state, conv_state, rec, qn, kn, vc, decay, beta, x, ldx, r, n_rows, KH, H,
                      D, Dp, V, Vs, taps, s);
}

int omnia_delta_norm(void* y, const float* o, const void* x, int f32, int64_t ldx, int zoff,
                     const float* norm_w, int T, int H, int V, int Vs, int Vp, float eps,
                     hipStream_t s) {
  if (Vs < V || Vp < V) return -1;
  if (T == 0) return 0;
  const int64_t n = (int64_t)T * H;
  const int vec = (V % 2 || Vp % 2) ? 1 : 2, ne = ((V > Vp ? V : Vp) + 64 * vec - 1) / (64 * vec);
#define OMNIA_DN(VEC, NE, NB)                                                                  \
  do {                                                                                         \
    const unsigned grid = (unsigned)((n + 4 * NB - 1) / (4 * NB));                             \
    if (f32)                                                                                   \
      norm_kernel<float, VEC, NE, NB><<<grid, 256, 0, s>>>((float*)y, o, (const float*)x, ldx, \
                                                           zoff, norm_w, n, H, V, Vs, Vp, eps); \
    else                                                                                       \
      norm_kernel<bf16_t, VEC, NE, NB><<<grid, 256, 0, s>>>((bf16_t*)y, o, (const bf16_t*)x,   \
                                                            ldx, zoff, norm_w, n, H, V, Vs,    \
                                                            Vp, eps);                          \
  } while (0)
  if (vec == 2 && ne == 1) OMNIA_DN(2, 1, 4);
  else if (vec == 2 && ne == 2) OMNIA_DN(2, 2, 2);
  else if (vec == 2 && ne <= 4) OMNIA_DN(2, 4, 1);
  else if (vec == 1 && ne <= 2) OMNIA_DN(1, 2, 1);
  else if (vec == 1 && ne <= 8) OMNIA_DN(1, 8, 1);
  else return -3;
#undef OMNIA_DN
  return (int)hipGetLastError();
}

}  // extern "C"
