// Gated delta rule for gfx950: a recurrence with a [dim x vdim] fp32 state per
// sequence and value head,
//
//     S <- g S ;  u = beta (v - S^T k) ;  S <- S + k u^T ;  o = S^T q
//
// whose q, k, v are short causal convolutions (silu) of projections, q and k made
// unit vectors per head.  One fused input projection feeds it, a row of
//     [q (KH*D) | k (KH*D) | v (H*V) | z (H*V) | b (H) | a (H)]     (row stride ldx).
//
//   delta_prep   convolutions, unit norms, decay and step size of every token (few rows of
//                sequences: delta_prep_blocks, with the blocks' systems of delta_scan)
//   delta_step_conv  decode, one token per sequence, of one or two heads a key head: convolutions,
//                norms, state update, per-head RMS norm and the silu(z) output gate in one launch,
//                one workgroup per (row, key head)
//   delta_step   decode of other sizes: the same behind delta_prep, one workgroup per (row, head)
//   delta_scan   prefill: each sequence's new tokens in blocks of 16, the state in MFMA
//                accumulators (delta_blocks first solves every block's 16 x 16 system);
//                key dimensions past 256 take a token-by-token scan instead
//   delta_norm   prefill: RMS norm + output gate of the scanned rows
//
// State of sequence slot s: state[s][h][D][Vp] fp32 and conv_state[s][taps-1][C], the
// last taps-1 projection rows (oldest first, in the storage type).  A sequence whose
// first row of this launch is at position 0 starts from zeros, whatever its slot held:
// slots are never cleared.  A negative slot (padded graph row) reads and writes nothing.
// delta_prep only READS conv_state; the step / scan launch that follows it shifts it.  delta_step_conv
// reads and shifts the channels of its own heads.
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

// A tap more of a convolution: oldest input, newest, those between.  Fused by name: of the first two
// products hipcc fuses either, and not the same in every kernel, so that fp32 rows differed by which kernel
// their step took.
__device__ __forceinline__ float conv_add(float a, float in, float w) {
  return __builtin_fmaf(in, w, a);
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
        float a = (TAPS > 1 ? hist[0][e][v] : in[r][e][v]) * w[e][v][0];
        if (TAPS > 1) a = conv_add(a, in[r][e][v], w[e][v][TAPS - 1]);
#pragma unroll
        for (int j = 1; j < TAPS - 1; ++j) a = conv_add(a, hist[j][e][v], w[e][v][j]);
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

// delta_prep and delta_step in one launch: a block of 256 threads a head has all R heads of a key
// head of a row, so that the convolution inputs it reads are its own to shift.  Waves 0 and 1 make q
// and k, 2 .. R + 1 the heads' v, 128 channels each, while the state's loads are under way; the rest
// is step_kernel's.  Saves the launch and the round trip of q, k and v: us of both kernels -> this
// one, 8 key heads of two heads of 128, states out of 1 GB, 1 / 8 / 32 / 64 / 96 / 192 / 256 rows
// 10.9 / 11.3 / 19.0 / 31.4 / 44.6 / 83 / 107 -> 8.7 / 11.0 / 16.2 / 27.2 / 42.9 / 79.7 / 102.
template <typename T, int NR, int R>
__global__ __launch_bounds__(256 * R) void step_conv_kernel(
    T* __restrict__ y, float* __restrict__ state, T* __restrict__ conv_state,
    const T* __restrict__ x, int64_t ldx, const T* __restrict__ conv_w,
    const float* __restrict__ a_log, const float* __restrict__ dt_bias,
    const float* __restrict__ norm_w, Rows rows, int KH, int D, int V, int Vs, int Vp, int taps,
    float eps) {
  extern __shared__ __attribute__((aligned(16))) float sm[];
  const int t = blockIdx.x, kh = blockIdx.y, tid = threadIdx.x & 255, lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), own = wv >> 2;
  const int H = KH * R, h = kh * R + own;  // this thread's head
  const int slot = rows.slots[t];
  T* yr = y + ((int64_t)t * H + h) * Vp;
  if (slot < 0) {
    for (int i = tid; i < Vp; i += 256) stf(yr + i, 0.f);
    return;
  }
  const bool fresh = rows.positions[t] == 0;
  const int C = 2 * KH * D + H * V, CG = Vs / 4, RG = 256 / CG;
  float* qs = sm;                      // [128]
  float* ks = qs + 128;                // [128]
  float* vs = ks + 128 + own * 128;    // [R][128]
  float* scratch = ks + 128 * (R + 1);  // [4 R]
  float* red = scratch + 4 * R + own * (RG + 2) * Vs;  // [RG][Vs] of each head, and
  float* us = red + RG * Vs;                           // [Vs]
  float* os = us + Vs;                                 // [Vs]
  const T* xr = x + (int64_t)t * ldx;

  // ---- convolution inputs and weights of two channels a lane; oldest input first
  const bool conv = wv < R + 2, isv = wv >= 2;
  const int n = isv ? V : D, i0 = 2 * lane;
  const int c0 = (isv ? 2 * KH * D + (kh * R + wv - 2) * V : wv * KH * D + kh * D) + i0;
  T* cs = conv_state + (int64_t)slot * (taps - 1) * C + c0;
  float in[2] = {0.f, 0.f}, hist[3][2], cw[2][4];
  const bool lives = conv && i0 < n;
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    hist[j][0] = hist[j][1] = 0.f;
    if (lives && j < taps - 1 && !fresh) Vec<T, 2>::ld(hist[j], cs + (int64_t)j * C);
  }
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int v = 0; v < 2; ++v)
      cw[v][j] = lives && j < taps ? ldf(conv_w + (int64_t)(c0 + v) * taps + j) : 0.f;
  if (lives) Vec<T, 2>::ld(in, xr + c0);
  const float bx = ldf(xr + C + H * V + h), ax = ldf(xr + C + H * V + H + h);
  const float dt = dt_bias[h], al = a_log[h];
  const T* zr = xr + C + h * V;
  const int v0 = min(tid, V - 1);
  const float z0 = ldf(zr + v0), w0 = norm_w[v0];

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
  if (conv) {
    float a[2], ss = 0.f;
#pragma unroll
    for (int v = 0; v < 2; ++v) {
      a[v] = conv_add(hist[0][v] * cw[v][0], in[v],
                      taps == 4 ? cw[v][3] : taps == 3 ? cw[v][2] : cw[v][1]);
#pragma unroll
      for (int j = 1; j < 3; ++j)
        if (j < taps - 1) a[v] = conv_add(a[v], hist[j][v], cw[v][j]);
      a[v] = siluf_(a[v]);
      ss += a[v] * a[v];
    }
    if (isv) {
      T r[2];  // as delta_prep stores them
      stf(r, a[0]);
      stf(r + 1, a[1]);
      float* o = ks + 128 * (wv - 1) + i0;
      if (i0 < n) o[0] = ldf(r), o[1] = ldf(r + 1);
    } else {
      ss = row_sum16(ss);
      ss += __shfl_xor(ss, 16, 64);
      ss += __shfl_xor(ss, 32, 64);
      float inv = 1.f / sqrtf(ss + 1e-6f);
      if (wv == 0) inv *= 1.f / sqrtf((float)D);
      float* o = qs + 128 * wv + i0;
      if (i0 < n) o[0] = a[0] * inv, o[1] = a[1] * inv;
    }
    if (lives) {
#pragma unroll
      for (int j = 0; j < 3; ++j)
        if (j < taps - 1) Vec<T, 2>::st(cs + (int64_t)j * C, j < taps - 2 ? hist[j < 2 ? j + 1 : 2] : in);
    }
  }
  const float z = ax + dt, sp = z > 20.f ? z : log1pf(expf(z));
  const float g = expf(-expf(al) * sp), bt = sigmoidf_(bx);
  __syncthreads();
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
    us[j] = j < V ? bt * (vs[j] - sk) : 0.f;
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
  ss = wave_sum(ss);
  if (lane == 0) scratch[wv] = ss;
  __syncthreads();
  ss = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) ss += scratch[4 * own + i];
  const float inv = 1.f / sqrtf(ss / (float)V + eps);
  for (int j = tid; j < Vp; j += 256) {
    const float zj = j < 256 || j >= V ? z0 : ldf(zr + j), nw = j < 256 || j >= V ? w0 : norm_w[j];
    stf(yr + j, j < V ? os[j] * inv * nw * siluf_(zj) : 0.f);
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

// A block's record, by one wave, from its products k.k and q.k (lane: column c16, rows 4 g4 ..) and
// token c16's log decay and step size; Ls: LDS of this wave
__device__ __forceinline__ void record(float* __restrict__ R, float4v kk, float4v qk, float c,
                                       float bt, float (*Ls)[20]) {
  const int lane = threadIdx.x & 63, c16 = lane & 15, g4 = lane >> 4;
#pragma unroll
  for (int o = 1; o < 16; o <<= 1) {
    const float up = __shfl_up(c, o, 16);
    if (c16 >= o) c += up;
  }
  // lane: column i = c16, rows t = 4 g4 + r
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int t = 4 * g4 + r;
    const float ct = __shfl(c, t, 16), btt = __shfl(bt, t, 16);
    const float e = c16 <= t ? expf(ct - c) : 0.f;
    Ls[t][c16] = c16 < t ? btt * e * kk[r] : 0.f;
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
      const float4v l = *reinterpret_cast<const float4v*>(&Ls[t][i]);
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
  record(rec + ((int64_t)id * H + h) * kRec, kk, qk, in ? decay[row * H + h] : 0.f,
         in ? beta[row * H + h] : 0.f, Ls[w]);
}

// delta_prep and blocks_kernel in one launch: a block makes the 16 tokens of a record for one key head
// and its R heads.  Four waves a unit (q, k, each head's v), four tokens each, whose inputs are loaded
// up front; normed q and k go to memory for the scan and to LDS, from which wave r makes head r's
// record.  D, V <= 128.  Bound by the chain of its loads and of the record's substitution; what it saves
// is a launch and the way of q and k through memory (figures at its rule).
template <typename T, int TAPS, int R>
__global__ __launch_bounds__(256 * (2 + R)) void prep_blocks_kernel(
    float* __restrict__ rec, float* __restrict__ qn, float* __restrict__ kn, T* __restrict__ vc,
    const T* __restrict__ x, int64_t ldx, const T* __restrict__ conv_w,
    const T* __restrict__ conv_state, const float* __restrict__ a_log,
    const float* __restrict__ dt_bias, Rows rows, int KH, int D, int Dp, int V) {
  constexpr int TR = 4, LS = 132;
  __shared__ __attribute__((aligned(16))) float qk[2][16][LS];
  __shared__ __attribute__((aligned(16))) float Ls[R][16][20];
  __shared__ float gates[2][R][16];
  const int id = blockIdx.x, kh = blockIdx.y, lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), u = w >> 2;
  int lo = 0, hi = rows.nseq - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (rec_base(rows.q_start, mid) <= id) lo = mid; else hi = mid - 1;
  }
  const int row0 = rows.q_start[lo], first = row0 + (id - rec_base(rows.q_start, lo)) * 16;
  const int m = min(16, rows.q_start[lo + 1] - first);
  if (m <= 0) return;  // the whole block
  const int H = KH * R, C = 2 * KH * D + H * V;
  const bool isv = u >= 2;
  const int n = isv ? V : D, i = 2 * lane, r0 = TR * (w & 3), nt = min(TR, m - r0), t0 = first + r0;
  const int c0 = (isv ? 2 * KH * D + (kh * R + u - 2) * V : (u * KH + kh) * D) + i;
  const bool lives = i < n;
  float wt[2][TAPS], in[TR][2], hist[TAPS - 1][2];
#pragma unroll
  for (int r = 0; r < TR; ++r) {
    in[r][0] = in[r][1] = 0.f;
    if (lives && r < nt) Vec<T, 2>::ld(in[r], x + (int64_t)(t0 + r) * ldx + c0);
  }
#pragma unroll
  for (int v = 0; v < 2 * TAPS; v += 2) {
    float t2[2] = {0.f, 0.f};
    if (lives) Vec<T, 2>::ld(t2, conv_w + (int64_t)c0 * TAPS + v);
    wt[v / TAPS][v % TAPS] = t2[0];
    wt[(v + 1) / TAPS][(v + 1) % TAPS] = t2[1];
  }
#pragma unroll
  for (int j = 0; j < TAPS - 1; ++j) hist[j][0] = hist[j][1] = 0.f;
  if (t0 - row0 >= TAPS - 1) {
#pragma unroll
    for (int j = 0; j < TAPS - 1; ++j)
      if (lives && nt > 0) Vec<T, 2>::ld(hist[j], x + (int64_t)(t0 - (TAPS - 1 - j)) * ldx + c0);
  } else {  // inputs before the sequence's new tokens
    const int slot = rows.slots[lo];
    const bool fresh = slot < 0 || rows.positions[row0] == 0;
    const T* cs = conv_state + (int64_t)(slot < 0 ? 0 : slot) * (TAPS - 1) * C;
#pragma unroll
    for (int j = 0; j < TAPS - 1; ++j) {
      const int r = t0 - (TAPS - 1 - j);
      const T* src = r >= row0 ? x + (int64_t)r * ldx : cs + (int64_t)(TAPS - 1 - (row0 - r)) * C;
      if (lives && (r >= row0 || !fresh)) Vec<T, 2>::ld(hist[j], src + c0);
    }
  }
  if (w == 8 && lane < 16 * R) {
    const int tt = lane & 15, h = kh * R + (lane >> 4);
    float dec = 0.f, bt = 0.f;
    if (tt < m) {
      const T* xr = x + (int64_t)(first + tt) * ldx + C + H * V;
      bt = sigmoidf_(ldf(xr + h));
      const float z = ldf(xr + H + h) + dt_bias[h];
      const float sp = z > 20.f ? z : log1pf(expf(z));
      dec = -expf(a_log[h]) * sp;
    }
    gates[0][lane >> 4][tt] = dec;
    gates[1][lane >> 4][tt] = bt;
  }
#pragma unroll
  for (int r = 0; r < TR; ++r) {
    float y[2], ss = 0.f;
#pragma unroll
    for (int v = 0; v < 2; ++v) {
      float a = conv_add(hist[0][v] * wt[v][0], in[r][v], wt[v][TAPS - 1]);
#pragma unroll
      for (int j = 1; j < TAPS - 1; ++j) a = conv_add(a, hist[j][v], wt[v][j]);
      a = siluf_(a);
      y[v] = a;
      ss += a * a;
#pragma unroll
      for (int j = 0; j + 1 < TAPS - 1; ++j) hist[j][v] = hist[j + 1][v];
      hist[TAPS - 2][v] = in[r][v];
    }
    if (isv) {
      if (lives && r < nt)
        Vec<T, 2>::st(vc + (int64_t)(t0 + r) * H * V + (c0 - 2 * KH * D), y);
      continue;
    }
    ss = row_sum16(ss);
    ss += __shfl_xor(ss, 16, 64);
    ss += __shfl_xor(ss, 32, 64);
    float inv = 1.f / sqrtf(ss + 1e-6f);
    if (u == 0) inv *= 1.f / sqrtf((float)D);
    y[0] = r < nt ? y[0] * inv : 0.f;  // columns past D are zeros by their inputs
    y[1] = r < nt ? y[1] * inv : 0.f;
    Vec<float, 2>::st(&qk[u][r0 + r][i], y);
    if (r < nt) {
      float* o = (u == 0 ? qn : kn) + ((int64_t)(t0 + r) * KH + kh) * Dp;
      if (lives) Vec<float, 2>::st(o + i, y);
      for (int j = n + lane; j < Dp; j += 64) o[j] = 0.f;
    }
  }
  __syncthreads();
  if (w >= R) return;
  const int c16 = lane & 15, g4 = lane >> 4;
  float4v kk = {0.f, 0.f, 0.f, 0.f}, pk = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    if (16 * j >= Dp) break;
    const float4v b = *reinterpret_cast<const float4v*>(&qk[0][c16][16 * j + 4 * g4]);
    const float4v a = *reinterpret_cast<const float4v*>(&qk[1][c16][16 * j + 4 * g4]);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      kk = mfma4(a[r], a[r], kk);
      pk = mfma4(b[r], a[r], pk);
    }
  }
  record(rec + ((int64_t)id * H + kh * R + w) * kRec, kk, pk, gates[0][w][c16], gates[1][w][c16],
         Ls[w]);
}

// Rows of a tensor as a buffer: reads past ``bytes`` give 0, writes there do nothing.
typedef __amdgpu_buffer_rsrc_t Rsrc;
typedef uint32_t uint4v __attribute__((ext_vector_type(4)));
constexpr uint32_t kOut = 0x80000000u;  // a lane's offset past every buffer

__device__ __forceinline__ Rsrc buffer(const void* base, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, bytes, 0x00020000);
}
__device__ __forceinline__ float4v load4(Rsrc b, uint32_t off) {
  return __builtin_bit_cast(float4v, (uint4v)__builtin_amdgcn_raw_buffer_load_b128(b, off, 0, 0));
}
__device__ __forceinline__ float load1(Rsrc b, uint32_t off) {
  return __builtin_bit_cast(float, (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(b, off, 0, 0));
}
__device__ __forceinline__ void store1(float v, Rsrc b, uint32_t off) {
  __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), b, off, 0, 0);
}

template <int N>
struct Int {
  static constexpr int value = N;
};

// One block's operands in LDS.
template <int ND, int CW>
struct ScanBuf {
  static constexpr int KS = 16 * ND + 4, TS = 20;
  float k[16 * KS], q[16 * KS], t[16 * TS], p[16 * TS], g[32], v[16 * CW * TS];
};
// Two of them: the compute waves read all of a block's between two barriers, while the next
// block's are written over what they read before.  ks, os: parts of K S and of the output.
template <int ND, int NW, int CW>
struct ScanShared {
  ScanBuf<ND, CW> buf[2];
  float4v ks[2][CW][NW][64], os[2][CW][NW][64];
};

// grid (ceil(Vs / (16 CW)) x H, nseq), CW x NW waves that multiply and 4 that move operands and
// outputs.  The former own 16 state columns each (cw) and share the key dimensions: wave w of NW (1, 2 or 4) has
// NJ = ND / NW accumulator tiles (key dimensions 16 (w NJ + j) + 4 (lane >> 4) + r in register r).
// The accumulator layout serves as the B operand of the next product as it stands: k-step r takes
// dimension (token) 4 (lane >> 4) + r, and the A side is read in that order.  Their parts of K S
// meet in LDS, added by all in one order, so that all hold the same u; parts of the output are
// added by the moving waves, a block later.  A wave that has twice the tiles keeps two sums, so that the
// order of additions, and with it every bit of a sequence's results, is that of four waves (one sum a wave
// of two was 1 % faster where the chip is full: 16 heads of 128, 2048 rows of 8 351 -> 354 us).
// Bound by the serial chain of a block where few blocks run: K S, the exchange, T', K^T U, 20 of a
// wave's 29 fp32 products (13.3 ns each) and the latencies between them.  A wave issues an
// instruction in about 5 clocks and none beside its own products, so whatever is not on the chain
// is another wave's work: with the staging in the multiplying waves the 16 heads of 4000 rows below
// took 262 us, with operands straight from global memory 282.  Where the chip is full, fp32
// products and vector instructions share one unit: of heads of 128, a wave of two has 54 products (16 each
// of K S, Q S and K^T U, 4 of T', 2 of P U) and a SIMD 108, of its two blocks: 1.44 of the 2.4 us that a
// block of 32 columns takes.
// us with blocks_kernel, one wave a 16 columns and all of their key dimensions -> now, heads of 128: 16 heads,
// 77 rows 23 -> 14, 1000 151 -> 56, 4000 550 -> 190, 333 of 3 63 -> 38, 60 of 16 38 -> 36, 512 of 32 336 ->
// 336, 2048 of 8 392 -> 354; 32 heads, 333 of 3 68 -> 61, 8192 1168 -> 437, 2048 of 8 686 -> 689; 8 heads of
// 256 x 128, 333 of 3 116 -> 41, 512 of 32 430 -> 368; heads of 64: at their rule in scan.
template <typename T, int ND, int NW, int CW>
__global__
__launch_bounds__(64 * (NW * CW + 4), ND <= 4 || ND / NW <= 2 ? 4 : 2) void scan_blocks_kernel(
    float* __restrict__ o, float* __restrict__ state, T* __restrict__ conv_state,
    const float* __restrict__ rec, const float* __restrict__ qn, const float* __restrict__ kn,
    const T* __restrict__ vc, const T* __restrict__ x, int64_t ldx, Rows rows, int KH, int H,
    int D, int Dp, int V, int Vs, int taps) {
  // NS sums of a wave, of JS tiles each: four in all (two, of the narrowest heads) whatever NW, added in
  // pairs, so that a sequence's results do not depend on the shape that its step takes
  constexpr int NJ = ND / NW, PR = 4 / NW, CN = NW * CW, NS = ND >= 4 ? PR : 2 / NW, JS = NJ / NS;
  // of the sums of a wave, and of those of the waves
  auto pairs = [](auto const& a, auto n) {
    if constexpr (decltype(n)::value == 1)
      return a[0];
    else if constexpr (decltype(n)::value == 2)
      return a[0] + a[1];
    else
      return (a[0] + a[1]) + (a[2] + a[3]);
  };
  using Buf = ScanBuf<ND, CW>;
  constexpr int KS = Buf::KS, TS = Buf::TS;
  static_assert(NJ * NW == ND && (NW == 1 || NW == 2 || NW == 4), "tiles of a wave");
  extern __shared__ __attribute__((aligned(16))) char lds[];
  ScanShared<ND, NW, CW>& sh = *reinterpret_cast<ScanShared<ND, NW, CW>*>(lds);
  const int lane = threadIdx.x & 63, c16 = lane & 15, g4 = lane >> 4;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // neighbours, which read the same keys and queries, on one XCD
  const int nx = (Vs + 16 * CW - 1) / (16 * CW), bid = xcd_remap(blockIdx.x, gridDim.x);
  const int bx = bid % nx, h = bid / nx, s = blockIdx.y;
  const int row0 = rows.q_start[s], n = rows.q_start[s + 1] - row0;
  const int slot = rows.slots[s];
  if (n <= 0 || slot < 0) return;
  const bool fresh = rows.positions[row0] == 0;
  const int nblk = (n + 15) / 16;
  // LDS only: the loads of later blocks stay in flight
  auto sync = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

  if (wv >= CN) {  // ---- the waves that move operands and outputs
    const int tid = threadIdx.x - 64 * CN, kh = h / (H / KH);
    constexpr int DW = 16 * ND, KT = DW / 4, NL = (16 * KT + 255) / 256;
    const int kbytes = KH * Dp * 4, vbytes = H * V * (int)sizeof(T), obytes = H * Vs * 4;
    // A thread's share of a block, in registers from two blocks before it is written to LDS: rows
    // of k and q, values of v, of T' and P, G or E.  Rows past the end, dimensions past Dp and
    // columns past V read as 0, and so does all of a block past the last.
    struct Stage {
      float4v k[NL], q[NL];
      float t, p, g;
      T v[CW];
    } st[2];
    const bool krow = 16 * KT >= 256 || tid < 16 * KT;
    const int kd4 = tid % KT * 4, tok = tid >> 4;
    const uint32_t koff = kd4 < Dp && krow ? tid / KT * kbytes + kd4 * 4 : kOut;
    uint32_t voff[CW], ooff[CW];
#pragma unroll
    for (int c = 0; c < CW; ++c) {
      const int col = (bx * CW + c) * 16 + c16;
      voff[c] = col < V ? tok * vbytes + col * (int)sizeof(T) : kOut;
      ooff[c] = col < Vs ? tok * obytes + col * 4 : kOut;
    }
    // a block's rows, from a head's first of them: what the block's lanes may touch
    auto rows_of = [&](const void* base, int bi, int stride) {
      const int m = min(16, n - 16 * bi);
      return buffer(reinterpret_cast<const char*>(base) + (int64_t)16 * bi * stride,
                    m > 0 ? m * stride : 0);
    };
    const float* kb = kn + ((int64_t)row0 * KH + kh) * Dp;
    const float* qb = qn + ((int64_t)row0 * KH + kh) * Dp;
    const T* vb = vc + ((int64_t)row0 * H + h) * V;
    const float* rb = rec + ((int64_t)rec_base(rows.q_start, s) * H + h) * kRec;
    float* ob = o + ((int64_t)row0 * H + h) * Vs;
    auto gload = [&](Stage& t, int bi) {
      const Rsrc K = rows_of(kb, bi, kbytes), Q = rows_of(qb, bi, kbytes);
      const Rsrc Vb = rows_of(vb, bi, vbytes);
      const Rsrc R = buffer(rb + (int64_t)bi * H * kRec, bi < nblk ? kRec * 4 : 0);
#pragma unroll
      for (int i = 0; i < NL; ++i) {
        t.k[i] = load4(K, koff + i * (256 / KT) * kbytes);
        t.q[i] = load4(Q, koff + i * (256 / KT) * kbytes);
      }
#pragma unroll
      for (int c = 0; c < CW; ++c) {
        if constexpr (sizeof(T) == 2)
          t.v[c] = __builtin_amdgcn_raw_buffer_load_b16(Vb, voff[c], 0, 0);
        else
          t.v[c] = load1(Vb, voff[c]);
      }
      t.t = load1(R, tid * 4);
      t.p = load1(R, 1024 + tid * 4);
      t.g = load1(R, 2048 + (tid & 31) * 4);
    };
    auto lwrite = [&](const Stage& t, Buf& b) {
      if (krow) {
#pragma unroll
        for (int i = 0; i < NL; ++i) {
          const int at = (i * (256 / KT) + tid / KT) * KS + kd4;
          *reinterpret_cast<float4v*>(b.k + at) = t.k[i];
          *reinterpret_cast<float4v*>(b.q + at) = t.q[i];
        }
      }
#pragma unroll
      for (int c = 0; c < CW; ++c) b.v[(16 * c + c16) * TS + tok] = ldf(&t.v[c]);
      b.t[tok * TS + c16] = t.t;
      b.p[tok * TS + c16] = t.p;
      b.g[tid & 31] = t.g;
    };
    auto store = [&](int bi) {
      const Rsrc O = rows_of(ob, bi, obytes);
#pragma unroll
      for (int c = 0; c < CW; ++c) {
        float y[NW];
#pragma unroll
        for (int i = 0; i < NW; ++i) y[i] = sh.os[bi & 1][c][i][16 * (tok >> 2) + c16][tok & 3];
        store1(pairs(y, Int<NW>()), O, ooff[c]);
      }
    };
    auto phase = [&](Stage& t, int bi) {
      lwrite(t, sh.buf[(bi + 1) & 1]);
      gload(t, bi + 3);
      if (bi > 1) store(bi - 2);
      sync();
    };
    gload(st[0], 0);
    gload(st[1], 1);
    lwrite(st[0], sh.buf[0]);
    gload(st[0], 2);
    sync();
    int bi = 0;
#pragma clang loop unroll(disable)
    for (; bi + 1 < nblk; bi += 2) {
      phase(st[1], bi);
      phase(st[0], bi + 1);
    }
    if (bi < nblk) phase(st[1], bi);
    if (nblk > 1) store(nblk - 2);
    sync();
    store(nblk - 1);
    const int C = 2 * KH * D + H * V, nb = nx * H, b = bx * H + h, per = (C + nb - 1) / nb;
    T* cs = conv_state + (int64_t)slot * (taps - 1) * C;
    for (int c = b * per + tid; c < min(C, (b + 1) * per); c += 256)
      shift_conv(x, ldx, cs, row0, n, fresh, taps, C, c);
    return;
  }

  // ---- the waves that multiply: 16 columns (cw) and ND / NW tiles of key dimensions (w) each
  const int cw = wv / NW, w = wv % NW, d0 = 16 * NJ * w, col = (bx * CW + cw) * 16 + c16;
  // the state of this head: past its columns and rows reads are 0 and writes dropped
  const Rsrc Sb = buffer(state + ((int64_t)slot * H + h) * D * Vs, D * Vs * 4);
  auto soff = [&](int j, int r) {
    return col < Vs ? (uint32_t)(((d0 + 4 * g4 + 16 * j + r) * Vs + col) * 4) : kOut;
  };
  float4v S[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r) S[j][r] = fresh ? 0.f : load1(Sb, soff(j, r));
  // operands of a block: k from behind the barrier before it, the rest before its own (one wave reads each
  // into the registers of the one before, 128 in all, of which a CU holds 2 blocks)
  float4v ka[NJ], qa[NJ], ta, G, E, v;
  float ku[4][NJ], pa[PR];
  auto keys = [&](const Buf& b) {
#pragma unroll
    for (int j = 0; j < NJ; ++j)
      ka[j] = *reinterpret_cast<const float4v*>(b.k + c16 * KS + d0 + 16 * j + 4 * g4);
  };
  auto updates = [&](const Buf& b) {
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int j = 0; j < NJ; ++j) ku[r][j] = b.k[(4 * g4 + r) * KS + d0 + 16 * j + c16];
#pragma unroll
    for (int k = 0; k < PR; ++k) pa[k] = b.p[c16 * TS + 4 * g4 + PR * w + k];
  };
  auto block = [&](auto odd) {
    constexpr int P = decltype(odd)::value;
    const Buf& B = sh.buf[P];
    float4v ks[NS], qs[NS], parts[NW], sum;
#pragma unroll
    for (int a = 0; a < NS; ++a) ks[a] = qs[a] = float4v{0.f, 0.f, 0.f, 0.f};
    // product i is one of sum i % NS
    auto tile = [](int i) { return i % NS * JS + (i / NS >> 2); };
    auto qstep = [&](int i) {
      const int j = tile(i), r = i / NS & 3;
      qs[i % NS] = mfma4(qa[j][r], S[j][r], qs[i % NS]);
    };
#pragma unroll
    for (int i = 0; i < 4 * NJ; ++i) {
      const int tj = tile(i), tr = i / NS & 3;
      ks[i % NS] = mfma4(ka[tj][tr], S[tj][tr], ks[i % NS]);
      if (i == 0) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < NJ; ++j)
          qa[j] = *reinterpret_cast<const float4v*>(B.q + c16 * KS + d0 + 16 * j + 4 * g4);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (i == 1) {
        G = *reinterpret_cast<const float4v*>(B.g + 4 * g4);
        v = *reinterpret_cast<const float4v*>(B.v + (16 * cw + c16) * TS + 4 * g4);
        ta = *reinterpret_cast<const float4v*>(B.t + c16 * TS + 4 * g4);
        E = *reinterpret_cast<const float4v*>(B.g + 16 + 4 * g4);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (NW > 1 && i == 2) {
        updates(B);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    // half of the products with q while the parts of K S go out, the others while they come in
    constexpr int Q0 = 2 * NJ, Q1 = 3 * NJ;
    sum = pairs(ks, Int<NS>());
    if constexpr (NW > 1)
      sh.ks[P][cw][w][lane] = sum;
    else
      updates(B);  // (registers of ka)
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < Q0; ++i) qstep(i);
    __builtin_amdgcn_sched_barrier(0);
    sync();
    if constexpr (NW > 1) {
#pragma unroll
      for (int i = 0; i < NW; ++i) parts[i] = sh.ks[P][cw][i][lane];
      keys(sh.buf[1 - P]);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = Q0; i < Q1; ++i) qstep(i);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (NW > 1) sum = pairs(parts, Int<NW>());
    const float4v res = v - G * sum;
    float4v u = {0.f, 0.f, 0.f, 0.f};
    // the chain of u runs between the products with q, which do not need it
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      u = mfma4(ta[r], res[r], u);
#pragma unroll
      for (int i = Q1; i < 4 * NJ; ++i)
        if ((i - Q1) * 4 / NJ == r) qstep(i);
    }
    if constexpr (NW == 1) {
      __builtin_amdgcn_sched_barrier(0);
      keys(sh.buf[1 - P]);  // (registers of qa)
      __builtin_amdgcn_sched_barrier(0);
    }
    // exp(c_15), the last of the 16 tokens'
    const float G3 = G[3], G15 = __builtin_bit_cast(
        float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, G3), 48));
#pragma unroll
    for (int j = 0; j < NJ; ++j) S[j] *= G15;
    const float4v ue = u * E;
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int j = 0; j < NJ; ++j) S[j] = mfma4(ku[r][j], ue[r], S[j]);
#pragma unroll
    for (int a = 0; a < NS; ++a) qs[a] *= G;
#pragma unroll
    for (int i = 0; i < PR; ++i) {  // token PR w + i of a lane's four
      float t = u[i];
#pragma unroll
      for (int k = 1; k < NW; ++k) t = w == k ? u[PR * k + i] : t;
      qs[i * NS / PR] = mfma4(pa[i], t, qs[i * NS / PR]);
    }
    sh.os[P][cw][w][lane] = pairs(qs, Int<NS>());
    __builtin_amdgcn_sched_barrier(0);
  };
  sync();
  keys(sh.buf[0]);
  int bi = 0;
#pragma clang loop unroll(disable)
  for (; bi + 1 < nblk; bi += 2) {
    block(Int<0>());
    block(Int<1>());
  }
  if (bi < nblk) block(Int<0>());
  sync();
#pragma unroll
  for (int j = 0; j < NJ; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r) store1(S[j][r], Sb, soff(j, r));
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

// -3: not covered (delta_prep, and blocks_kernel at the scan, cover all)
template <typename T>
int prep_blocks(float* rec, float* qn, float* kn, void* vc, const void* x, int64_t ldx,
                const void* conv_w, const void* conv_state, const float* a_log,
                const float* dt_bias, Rows r, int T_, int KH, int H, int D, int Dp, int V, int taps,
                hipStream_t s) {
  if (D > 128 || V > 128 || D % 2 || V % 2 || Dp > 128) return -3;
  const dim3 grid(T_ / 16 + r.nseq, KH);
  // A CU holds two blocks (threads): while all of them, 512, are there at once, most of a block's waves
  // wait for the few that make its records at no one's cost.  A second round still pays for up to 640
  // where nearly all blocks have a record: of many short sequences up to half have none, and delta_prep is
  // fast on their few rows.  us of preparation, records and scan, two launches before the scan / one, 8 key
  // heads of two of 128: 20 rows 16.4 / 13.0, 200 25.7 / 21.8, 56 x 2 (504 blocks) 54.3 / 51.9, 22 x 31 (512)
  // 43.3 / 39.5, 32 x 16 (512) 40.4 / 39.6; 3 x 333 (520) 49.3 / 45.7, 8 x 120 (544) 44.1 / 40.6, 8 x 136
  // (608) 48.3 / 46.2, 1200 (608) 77.6 / 77.5; not taken: 33 x 16 (528) 43.7 / 46.9, 60 x 2 (536) 56.6 / 59.1,
  // 24 x 31 (560) 45.0 / 45.2, 40 x 16 (640) 47.7 / 50.9, 2000 (1008) 111.5 / 111.9, 8 x 1000 192 / 202.  Of
  // one head a key head: 3 x 333 39.3 / 34.4, 32 x 16 29.4 / 27.6, 1200 75.6 / 74.1; not taken: 33 x 16 31.6 /
  // 33.5, 20 x 48 37.1 / 37.8, 2000 109.7 / 109.9.  Of heads of 64: 3 x 333 32.1 / 28.1; 33 x 16 25.3 / 28.2.
  const int64_t blocks = (int64_t)grid.x * KH;
  if (blocks > 640 || (blocks > 512 && 4 * r.nseq > T_ / 16)) return -3;
#define OMNIA_PB(TAPS, R)                                                                         \
  if (taps == TAPS && H == R * KH) {                                                              \
    if (T_ == 0 || r.nseq == 0) return 0;                                                         \
    prep_blocks_kernel<T, TAPS, R><<<grid, 256 * (2 + R), 0, s>>>(                                \
        rec, qn, kn, (T*)vc, (const T*)x, ldx, (const T*)conv_w, (const T*)conv_state, a_log,     \
        dt_bias, r, KH, D, Dp, V);                                                                \
    return (int)hipGetLastError();                                                                \
  }
  OMNIA_PB(2, 1) OMNIA_PB(3, 1) OMNIA_PB(4, 1) OMNIA_PB(2, 2) OMNIA_PB(3, 2) OMNIA_PB(4, 2)
#undef OMNIA_PB
  return -3;
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

// -3: not covered (the two kernels above cover all)
template <typename T>
int step_conv(void* y, float* state, void* conv_state, const void* x, int64_t ldx,
              const void* conv_w, const float* a_log, const float* dt_bias, const float* norm_w,
              Rows r, int T_, int KH, int H, int D, int V, int Vs, int Vp, int taps, float eps,
              hipStream_t s) {
  if (D > 128 || V > 128 || D % 2 || V % 2 || taps < 2 || taps > 4 || Vs / 4 > 256) return -3;
  const int CG = Vs / 4, RG = 256 / CG, nr = (D + RG - 1) / RG, R = H / KH;
  // One or two heads a key head.  Four were blocks of 1024 threads, one a CU, each with the states of
  // four heads: slower than the two kernels until the chip is full and again past it (us, two / one, 4
  // key heads of four heads of 128: 1 row 10.9 / 13.6, 8 11.4 / 14.9, 32 19.0 / 18.5, 64 31.2 / 27.1, 72
  // 35.6 / 39.3, 128 52.5 / 51.5, 136 60.7 / 63.6, 256 105.0 / 102.5).
  if (nr > 16 || R > 2) return -3;
  // Of states of half that size (8 rows a thread) a CU holds 7 blocks of step_kernel, and 3 of 512
  // threads here, 6 heads: two kernels while all heads are on the chip at once there and not here (8 key
  // heads of two heads of 128 x 64, 104 rows 25.0 / 26.9, 112 26.7 / 27.9; 96 24.3 / 23.2, 120 30.6 /
  // 29.2).  Elsewhere a CU holds as many heads of both, and the rounds of the two kernels are not a
  // reason: of 128 x 128, 112 / 120 / 128 / 136 rows 49.4 / 52.4 / 53.1 / 61.1 and 49.5 / 51.7 / 53.8 /
  // 60.0, of one head a key head 51.7 / 54.0 / 54.6 / 63.9 and 52.2 / 55.7 / 55.9 / 61.4.
  const int64_t heads = (int64_t)T_ * H;
  if (R == 2 && nr > 4 && nr <= 8 && heads > 6 * 256 && heads <= 7 * 256) return -3;
  const size_t lds = (size_t)(256 + 132 * R + R * (RG + 2) * Vs) * 4;
#define OMNIA_STEP(N, RR)                                                                      \
  if (R == RR && nr <= N) {                                                                    \
    step_conv_kernel<T, N, RR><<<dim3(T_, KH), 256 * RR, lds, s>>>(                            \
        (T*)y, state, (T*)conv_state, (const T*)x, ldx, (const T*)conv_w, a_log, dt_bias,      \
        norm_w, r, KH, D, V, Vs, Vp, taps, eps);                                               \
    return (int)hipGetLastError();                                                             \
  }
  OMNIA_STEP(4, 1) OMNIA_STEP(8, 1) OMNIA_STEP(16, 1) OMNIA_STEP(4, 2) OMNIA_STEP(8, 2)
  OMNIA_STEP(16, 2)
#undef OMNIA_STEP
  return -3;
}

template <typename T>
int scan(float* o, float* state, void* conv_state, float* rec, const float* qn, const float* kn,
         const void* vc, const float* decay, const float* beta, const void* x, int64_t ldx, Rows r,
         int n_rows, int KH, int H, int D, int Dp, int V, int Vs, int taps, hipStream_t s) {
  const dim3 bgrid(n_rows / 16 + r.nseq, (H + 3) / 4);
  // One column group a block, its key dimensions over 4 waves, while those blocks are one a CU: the
  // chain of a block is what the step waits for.  Beyond, two groups of 2 waves (us, one / two: 256
  // blocks 86 / 118, 384 39 / 38, 768 60 / 60, 1024 105 / 90 and 368 / 327).
  // Heads of up to 64, four groups a block, once those are one a CU and leave no more of their groups empty
  // than blocks of two: a wave a group takes all of the key dimensions, so that a column has fewer products
  // and movers, and two blocks a CU wait for one another (us, two of 2 / four of 1, heads of 64 x 64: 512
  // groups 39.2 / 49.8, 1024 60 / 57 and 217 / 209, 2048 110 / 97, 8192 439 / 390, 64 sequences of 2 tokens
  // 23.2 / 18.2, of 32 heads 38.1 / 31.3; of 64 x 48, 6144 414 / 373; of 32 x 64, 2048 76 / 67, 4096 149 / 133;
  // of 24 x 40, 64 sequences of 2 tokens of 32 heads 27.8 / 24.1, where the kernel before took 22.6).
  const int g = (Vs + 15) / 16;
  const int64_t heads = (int64_t)H * r.nseq;
  const bool few = g * heads <= 256, narrow = (g + 3) / 4 * heads >= 256 && (g % 4 == 0 || g % 4 == 3);
#define OMNIA_SPLIT(ND, NW, CW)                                                                   \
  scan_blocks_kernel<T, ND, NW, CW>                                                               \
      <<<dim3((Vs + 16 * CW - 1) / (16 * CW) * H, r.nseq), 64 * (NW * CW + 4),                    \
         sizeof(ScanShared<ND, NW, CW>), s>>>(o, state, (T*)conv_state, rec, qn, kn,              \
                                              (const T*)vc, (const T*)x, ldx, r, KH, H, D, Dp, V, \
                                              Vs, taps)
#define OMNIA_SCANB(ND)                                                                         \
  if (D <= 16 * ND) {                                                                           \
    if (decay)                                                                                  \
      blocks_kernel<ND><<<bgrid, 256, 0, s>>>(rec, qn, kn, decay, beta, r.q_start, r.nseq, KH,  \
                                              H, Dp);                                           \
    if (few)                                                                                    \
      OMNIA_SPLIT(ND, (ND < 4 ? 2 : 4), 1);                                                     \
    else if (ND <= 4 && narrow)                                                                 \
      OMNIA_SPLIT(ND, (ND <= 4 ? 1 : 2), (ND <= 4 ? 4 : 2));                                    \
    else                                                                                        \
      OMNIA_SPLIT(ND, 2, 2);                                                                    \
    return (int)hipGetLastError();                                                              \
  }
  OMNIA_SCANB(2) OMNIA_SCANB(4) OMNIA_SCANB(8) OMNIA_SCANB(16)
#undef OMNIA_SCANB
#undef OMNIA_SPLIT
  if (!decay) return -5;
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
  if (taps < 1 || KH < 1 || H % KH || Dp % 4 || Dp < D || Vs < 4 || Vs % 4 || Vs < V || Vp < V)
    return -1;
  if (Vs / 4 > 256) return -2;
  if (T == 0) return 0;
  const Rows r{nullptr, T, positions, slots};
  if (f32)
    return step<float>(y, state, conv_state, qn, kn, vc, decay, beta, x, ldx, norm_w, r, T, KH, H,
                       D, Dp, V, Vs, Vp, taps, eps, s);
  return step<bf16_t>(y, state, conv_state, qn, kn, vc, decay, beta, x, ldx, norm_w, r, T, KH, H,
                      D, Dp, V, Vs, Vp, taps, eps, s);
}

// omnia_delta_prep and omnia_delta_step of decode rows in one launch; -3 where it does not cover the
// sizes (checked before any launch)
int omnia_delta_step_conv(void* y, float* state, void* conv_state, const void* x, int f32,
                          int64_t ldx, const void* conv_w, const float* a_log,
                          const float* dt_bias, const float* norm_w, const int* positions,
                          const int* slots, int T, int KH, int H, int D, int V, int Vs, int Vp,
                          int taps, float eps, hipStream_t s) {
  if (KH < 1 || H % KH || Vs < 4 || Vs % 4 || Vs < V || Vp < V) return -1;
  if (T == 0) return 0;
  const Rows r{nullptr, T, positions, slots};
  if (f32)
    return step_conv<float>(y, state, conv_state, x, ldx, conv_w, a_log, dt_bias, norm_w, r, T, KH,
                            H, D, V, Vs, Vp, taps, eps, s);
  return step_conv<bf16_t>(y, state, conv_state, x, ldx, conv_w, a_log, dt_bias, norm_w, r, T, KH,
                           H, D, V, Vs, Vp, taps, eps, s);
}

// omnia_delta_prep of sequences' rows, and the block records of omnia_delta_scan, in one launch; -3
// where it does not cover the sizes (checked before any launch)
int omnia_delta_prep_blocks(float* rec, float* qn, float* kn, void* vc, const void* x, int f32,
                            int64_t ldx, const void* conv_w, const void* conv_state,
                            const float* a_log, const float* dt_bias, const int* q_start, int nseq,
                            const int* positions, const int* slots, int T, int KH, int H, int D,
                            int Dp, int V, int taps, hipStream_t s) {
  if (taps < 1 || KH < 1 || H % KH || Dp % 4 || Dp < D) return -1;
  if (KH > 65535) return -2;
  const Rows r{q_start, nseq, positions, slots};
  if (f32)
    return prep_blocks<float>(rec, qn, kn, vc, x, ldx, conv_w, conv_state, a_log, dt_bias, r, T, KH,
                              H, D, Dp, V, taps, s);
  return prep_blocks<bf16_t>(rec, qn, kn, vc, x, ldx, conv_w, conv_state, a_log, dt_bias, r, T, KH,
                             H, D, Dp, V, taps, s);
}

// floats of the block records of n_rows rows in nseq sequences
int64_t omnia_delta_records(int n_rows, int nseq, int H) {
  return (int64_t)(n_rows / 16 + nseq) * H * kRec;
}

// decay and beta null: rec holds the records (omnia_delta_prep_blocks)
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
