// Paged attention for the in-node engine on gfx950.
//
// KV cache layout (shared with rope_kv in elementwise.hip):
//     k_cache, v_cache : [num_blocks, Hkv, BS, 128] bf16
// i.e. one kv-head's rows of a page are contiguous, so a 16-lane group reads a
// whole 256-B token row and a wave-instruction reads 4 consecutive tokens = 1 KiB.
//
// decode  : split-K ("flash-decoding") over partitions of the context, GQA
//           group of G query heads per workgroup sharing one K/V stream;
//           Q.K^T on the MFMA (16x16x32 bf16, heads padded to 16 columns),
//           P.V on the VALU with P in fp32 (8 dims per lane), partitions merged
//           by a second tiny kernel.
// prefill : flash-attention over (cached prefix + new tokens) with causal
//           offset, 64 query rows x 1 head per workgroup (16 rows per wave),
//           K/V tiles of 64 keys gathered from pages into XOR-swizzled LDS,
//           S^T = K.Q^T so each lane owns one query row (softmax row stats are
//           lane-local + 2 shuffles), P^T reused in-register as the B operand of
//           O^T = V^T.P^T with V^T fragments from ds_read_b64_tr_b16.
#include <stdlib.h>

#include "common.h"

using namespace omnia;

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ float4v mfma16(short8 a, short8 b, float4v c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

constexpr int D = 128;

// ============================================================== decode
// Length-balanced split (split_t > 0): a sequence of `len` keys is cut into
// ns = clamp(ceil(len / split_min), ceil(len / cap), split_t) partitions of equal
// page-aligned length -- decided on the device from the live length, so a graph
// captured once splits every context evenly (a host-chosen fixed partition
// leaves one workgroup per (sequence, kv head) at short contexts when the batch
// has few such pairs, e.g. one Llama-3-70B TP=8 rank).  cap and BS divide each
// other's multiples: pl <= cap always.
__device__ __forceinline__ int decode_part_len(int len, int cap, int split_t, int split_min,
                                               int bs) {
  if (split_t <= 0) return cap;
  int ns = min(split_t, (len + split_min - 1) / split_min);
  ns = max(ns, max((len + cap - 1) / cap, 1));
  const int pl = ((len + ns - 1) / ns + bs - 1) / bs * bs;
  return min(pl, cap);
}

// grid: (B, Hkv, max_parts)   block: 256.  Bound by the reads of K and V.  A wave goes through
// every fourth 16-key group by itself, with its own running max: K and V of the next group are
// loaded while this one's scores, softmax and P.V are computed, so that memory never waits for a
// phase of the block, and the waves meet once at the end.  3 waves a SIMD: groups of 32 keys take
// the registers of 2, and short contexts 50 us where these take 39; 4 spill.  us with scores,
// softmax and P.V as phases of the block -> now (32 heads on 8; sequences x keys): 256 x 576
// 127 -> 119 (5.1 TB/s), 128 x 1000 111 -> 104, 64 x 2000 115 -> 112, 32 x 1000 33.7 -> 29.3,
// 4 x 1000 15.3 -> 12.4, 256 x 150 38.2 -> 37.0.  Of
// sequences that share the pages of a prompt prefix a block finds in the caches what another has
// read; K and V that nobody shares go past them (non-temporal) where many long sequences make
// bandwidth the bound.  us through the caches and past them, out of 1.2 GB and more: 256 x 576 109 /
// 106, 256 x 768 148 / 131, 128 x 1000 96 / 86, 64 x 2000 96 / 85, 32 x 1000 26.2 / 23.9; lengths
// from half up to 600 64 x 27.2 / 28.6, to 800 33.7 / 33.7, to 1000 43.6 / 40.8; in partitions 16 x
// 1500 27.3 / 27.2, 8 x 900 13.2 / 13.6.  By the rule: 512 of 256 x 576 shared by all 55.2 -> 55, by
// sequences 32 apart 54 -> 55.9 (past the caches 76), 896 of 128 x 1000 44.8 -> 44.4 and 45 -> 46.7
// (59, 66).
constexpr int NW = 4;
template <int G>
struct DecodeShared {
  float pb[NW][16][G];  // a group's P, wave-private
  float al[NW][G];
  float red[NW][G][D];
  float ml[NW][G][2];
};

// The whole work of a block, K and V past the caches or through them: two copies in the kernel,
// with the registers of one (140; a choice at each load breaks the pipeline of loads, one around
// the loop alone spills).
template <int G, int BS, bool NT>
__device__ __forceinline__ void decode_block(
    DecodeShared<G>& sh, int len, int pl, bf16_t* __restrict__ out,
    float* __restrict__ part_o, float* __restrict__ part_ml, const bf16_t* __restrict__ q,
    const bf16_t* __restrict__ kc, const bf16_t* __restrict__ vc,
    const int* __restrict__ block_tables, int bt_stride, int hkv, int64_t q_stride, int max_parts,
    float scale_log2) {
  auto &pb = sh.pb;
  auto &al = sh.al;
  auto &red = sh.red;
  auto &ml = sh.ml;
  const int b = blockIdx.x, kvh = blockIdx.y, part = blockIdx.z;
  const int p0 = part * pl;
  const int n = min(pl, len - p0);
  const int nparts = (len + pl - 1) / pl;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h0 = kvh * G, c16 = lane & 15, g4 = lane >> 4;
  const int* bt = block_tables + (int64_t)b * bt_stride + p0 / BS;

  // Q^T as the MFMA B operand: column = head (c16, only < G real), k = dims
  short8 qf[4];
  {
    const bf16_t* qrow = q + (int64_t)b * q_stride + (h0 + (c16 < G ? c16 : 0)) * D;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      short8 v = *reinterpret_cast<const short8*>(qrow + kk * 32 + 8 * g4);
      if (c16 >= G) v = short8{0, 0, 0, 0, 0, 0, 0, 0};
      qf[kk] = v;
    }
  }
  // K rows as the A operand (row = key c16 of the group); V: lane = (token g4 of 4, dims 8 c16
  // ..).  A group lies in one page; rows past the end re-read the last one.
  struct Group {
    short8 k[4], v[4];
  };
  const int ngr = (n + 15) / 16, last = n - 1;
  auto page = [&](int c) { return bt[min(c * 16, last) / BS]; };  // past the end: the last page
  auto get = [](const bf16_t* p) {
    const short8* s = reinterpret_cast<const short8*>(p);
    return NT ? __builtin_nontemporal_load(s) : *s;
  };
  auto load = [&](Group& t, int c, int pg) {
    const int k0 = min(c * 16, last & ~15), top = last - k0;
    const int64_t base = (((int64_t)pg * hkv + kvh) * BS + k0 % BS) * D;
    const bf16_t *kb = kc + base, *vb = vc + base;
    const uint32_t ko = min(c16, top) * D + 8 * g4;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) t.k[kk] = get(kb + ko + kk * 32);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t vo = min(4 * i + g4, top) * D + 8 * c16;
      t.v[i] = get(vb + vo);
    }
  };
  // of head c16; a finite start, so that keys whose scores are all -inf get exponents of -inf
  float m_run = -3.4028234e38f, l_run = 0.f;
  float acc[G][8];
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[g][j] = 0.f;
  auto compute = [&](Group& t, int c) {
    // rows past the end have P = 0, which leaves nothing of a V that is finite
    if (n - c * 16 < 16) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (4 * i + g4 >= n - c * 16) t.v[i] = short8{0, 0, 0, 0, 0, 0, 0, 0};
    }
    float4v sc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) sc = mfma16(t.k[kk], qf[kk], sc);
    // sc[r]: key 4 g4 + r of the group, head c16
    const int top = n - c * 16 - 4 * g4;
    float m = -INFINITY;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      sc[r] = r < top ? sc[r] * scale_log2 : -INFINITY;
      m = fmaxf(m, sc[r]);
    }
    m = fmaxf(m, __shfl_xor(m, 16, 64));
    m = fmaxf(m, __shfl_xor(m, 32, 64));
    // the maximum moves only when a head's grows by more than 2^8: P and its sums are fp32
    const bool grow = m > m_run + 8.f;
    const bool any = __builtin_amdgcn_ballot_w64(grow) != 0;
    if (any) {
      const float m_new = grow ? m : m_run;
      const float a = exp2f(m_run - m_new);
      l_run *= a;
      m_run = m_new;
      if (lane < G) al[w][lane] = a;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float p = exp2f(sc[r] - m_run);
      l_run += p;
      if (c16 < G) pb[w][4 * g4 + r][c16] = p;
    }
    __builtin_amdgcn_wave_barrier();
    if (any) {
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const float a = al[w][g];
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[g][j] *= a;
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float p[G];
#pragma unroll
      for (int g = 0; g < G; ++g) p[g] = pb[w][4 * i + g4][g];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float v = bf2f((uint16_t)t.v[i][j]);
#pragma unroll
        for (int g = 0; g < G; ++g) acc[g][j] += p[g] * v;
      }
    }
    __builtin_amdgcn_wave_barrier();
  };
  if (w < ngr) {
    Group t0, t1;
    load(t0, w, page(w));
    int pg = page(w + NW);
    for (int c = w; c < ngr; c += 2 * NW) {
      load(t1, c + NW, pg);
      pg = page(c + 2 * NW);
      compute(t0, c);
      load(t0, c + 2 * NW, pg);
      pg = page(c + 3 * NW);
      if (c + NW < ngr) compute(t1, c + NW);
    }
  }
  l_run += __shfl_xor(l_run, 16, 64);
  l_run += __shfl_xor(l_run, 32, 64);
  if (lane < G) {
    ml[w][lane][0] = m_run;
    ml[w][lane][1] = l_run;
  }
  // over the 4 tokens of a V instruction: lane group g4 ends with two of the 8 dims, half of
  // what a step leaves going to the other lanes
  const bool hi = lane >= 32, mid = g4 & 1;
#pragma unroll
  for (int g = 0; g < G; ++g) {
    float r[4], t[2];
#pragma unroll
    for (int j = 0; j < 4; ++j)
      r[j] = (hi ? acc[g][4 + j] : acc[g][j]) + __shfl_xor(hi ? acc[g][j] : acc[g][4 + j], 32, 64);
#pragma unroll
    for (int j = 0; j < 2; ++j)
      t[j] = (mid ? r[2 + j] : r[j]) + __shfl_xor(mid ? r[j] : r[2 + j], 16, 64);
    *reinterpret_cast<float2*>(&red[w][g][c16 * 8 + g4 * 2]) = float2{t[0], t[1]};
  }
  __syncthreads();
  for (int i = tid; i < G * D; i += 64 * NW) {
    const int g = i / D, d = i % D;
    float m = ml[0][g][0];
#pragma unroll
    for (int wi = 1; wi < NW; ++wi) m = fmaxf(m, ml[wi][g][0]);
    float v = 0.f, l = 0.f;
#pragma unroll
    for (int wi = 0; wi < NW; ++wi) {
      const float e = exp2f(ml[wi][g][0] - m);
      v += e * red[wi][g][d];
      l += e * ml[wi][g][1];
    }
    // a partition whose scores are all -inf weighs nothing among others
    const float inv = l == 0.f && nparts > 1 ? 0.f : 1.f / l;
    const int h = h0 + g;
    if (nparts == 1) {
      out[((int64_t)b * gridDim.y * G + h) * D + d] = f2bf(v * inv);
    } else {
      const int64_t slot = ((int64_t)b * gridDim.y * G + h) * max_parts + part;
      part_o[slot * D + d] = v * inv;
      if (d == 0) {
        part_ml[slot * 2] = m;
        part_ml[slot * 2 + 1] = l;
      }
    }
  }
}

template <int G, int BS>
__global__ __launch_bounds__(64 * NW, G < 8 ? 3 : 2) void decode_attn_kernel(
    bf16_t* __restrict__ out, float* __restrict__ part_o, float* __restrict__ part_ml,
    const bf16_t* __restrict__ q, const bf16_t* __restrict__ kc, const bf16_t* __restrict__ vc,
    const int* __restrict__ block_tables, int bt_stride, const int* __restrict__ seq_lens,
    int hkv, int64_t q_stride, int part_size, int max_parts, float scale_log2, int split_t,
    int split_min) {
  __shared__ __attribute__((aligned(16))) DecodeShared<G> sh;
  const int b = blockIdx.x, part = blockIdx.z;
  const int len = seq_lens[b];
  if (len <= 0) return;
  const int pl = decode_part_len(len, part_size, split_t, split_min, BS);
  const int p0 = part * pl;
  if (p0 >= len) return;
  // Past the caches, where bandwidth is the bound: blocks enough without partitions, two thirds of
  // the sequences long (few long ones are waited for, and such loads come later), and of a long one
  // what no other has the page of, 64 keys into the partition (a row's entries past its length may
  // be anything: at worst the caches are used).  What shares less is read again for less than is
  // gained.  Sharers may be anywhere in the batch, so the block's threads look at all of it, a row
  // each; up to 64 rows every wave for itself, without a barrier
  constexpr int LONG = 512;
  const int B = gridDim.x;
  if (len >= LONG && min(pl, len - p0) >= 192 && B * gridDim.y >= 256) {
    const bool alone = B <= 64;
    const int me = alone ? threadIdx.x & 63 : threadIdx.x, step = alone ? 64 : 64 * NW;
    const int* t = block_tables + min(p0 + 64, len - 1) / BS;
    const int own = t[(int64_t)b * bt_stride];
    int votes = 0;
    uint64_t same = 0;
#pragma unroll 2
    for (int i0 = 0; i0 < B; i0 += step) {
      const int i = min(i0 + me, B - 1), n = i0 + me < B ? seq_lens[i] : 0;
      same |= __builtin_amdgcn_ballot_w64(t[(int64_t)i * bt_stride] == own && i != b);
      votes += __popcll(__builtin_amdgcn_ballot_w64(n >= LONG)) -
               2 * __popcll(__builtin_amdgcn_ballot_w64(n > 0 && n < LONG));
    }
    if (same) votes = -(1 << 28);
    if (!alone) {
      __shared__ int look[NW];
      if ((threadIdx.x & 63) == 0) look[threadIdx.x >> 6] = votes;
      __syncthreads();
      votes = 0;
#pragma unroll
      for (int i = 0; i < NW; ++i) votes += look[i];
    }
    if (votes >= 0) {
      decode_block<G, BS, true>(sh, len, pl, out, part_o, part_ml, q, kc, vc, block_tables,
                                bt_stride, hkv, q_stride, max_parts, scale_log2);
      return;
    }
  }
  decode_block<G, BS, false>(sh, len, pl, out, part_o, part_ml, q, kc, vc, block_tables,
                             bt_stride, hkv, q_stride, max_parts, scale_log2);
}

// grid: (B * Hq)   block: 256.  Latency bound: a lane takes one partition's (m, l) of each 64 and
// the four waves take every fourth partition's row, with the loads of several in flight (one
// after the other, a 2000-key sequence in 32 partitions took 20.3 us with its attention, with this 12.9).
__global__ __launch_bounds__(256) void decode_reduce_kernel(
    bf16_t* __restrict__ out, const float* __restrict__ part_o, const float* __restrict__ part_ml,
    const int* __restrict__ seq_lens, int hq, int part_size, int max_parts, int split_t,
    int split_min, int bs) {
  __shared__ float2 red[3][64];
  const int bh = blockIdx.x;
  const int b = bh / hq;
  const int len = seq_lens[b];
  if (len <= 0) return;
  const int pl = decode_part_len(len, part_size, split_t, split_min, bs);
  const int nparts = (len + pl - 1) / pl;
  if (nparts <= 1) return;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const float2* ml = reinterpret_cast<const float2*>(part_ml) + (int64_t)bh * max_parts;
  const float2* po =
      reinterpret_cast<const float2*>(part_o) + (int64_t)bh * max_parts * (D / 2) + lane;
  float m = -INFINITY;
  for (int p = lane; p < nparts; p += 64) m = fmaxf(m, ml[p].x);
  m = wave_max(m);
  float tot = 0.f;
  float2 acc = {0.f, 0.f};
  for (int p0 = 0; p0 < nparts; p0 += 64) {
    float wl = 0.f;
    if (p0 + lane < nparts) {
      const float2 v = ml[p0 + lane];
      wl = exp2f(v.x - m) * v.y;
    }
    tot += wl;
    const int n = min(64, nparts - p0);
    for (int i0 = w; i0 < n; i0 += 32) {
      float2 v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = po[(int64_t)(p0 + min(i0 + 4 * u, n - 1)) * (D / 2)];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const float g = __shfl(wl, (i0 + 4 * u) & 63, 64);
        if (i0 + 4 * u < n) {
          acc.x += g * v[u].x;
          acc.y += g * v[u].y;
        }
      }
    }
  }
  tot = wave_sum(tot);
  if (w) red[w - 1][lane] = acc;
  __syncthreads();
  if (w) return;
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    acc.x += red[i][lane].x;
    acc.y += red[i][lane].y;
  }
  const uint32_t pk = pack_bf2(acc.x / tot, acc.y / tot);
  reinterpret_cast<uint32_t*>(out)[(int64_t)bh * (D / 2) + lane] = pk;
}

// ============================================================== prefill
__device__ __forceinline__ int kswz(int row, int ch) { return ch ^ (row & 15); }
__device__ __forceinline__ int vswz(int row, int ch) {
  return ch ^ (((row & 3) << 2) | ((row >> 2) & 3));
}

// grid: (Hq / HP, n_tiles)   block: 64*NW (NW waves x 16 query rows = a 16*NW-row
// query tile; every staged 64-key K/V tile feeds all NW waves)
// GQA head packing: each wave carries HP query heads of the same KV head for its
// 16 rows, so every K / V fragment read from LDS (and every K / V tile staged
// from HBM) feeds HP heads' MFMAs -- HP x fewer LDS bytes per FLOP and HP x
// fewer K/V tile loads than one head per block.
template <int BS, int HP, int NW>
__global__ __launch_bounds__(64 * NW) void prefill_attn_kernel(
    bf16_t* __restrict__ out, const bf16_t* __restrict__ q, const bf16_t* __restrict__ kc,
    const bf16_t* __restrict__ vc, const int* __restrict__ block_tables, int bt_stride,
    const int* __restrict__ q_start_loc, const int* __restrict__ seq_lens,
    const int* __restrict__ tile_seq, const int* __restrict__ tile_q0, int hkv, int64_t q_stride,
    int64_t out_stride, float scale_log2, float* __restrict__ lse_out,
    const int* __restrict__ kv_lens) {
  __shared__ __attribute__((aligned(16))) char lds[2 * 64 * 256];
  char* Kl = lds;
  char* Vl = lds + 64 * 256;

  const int h0 = blockIdx.x * HP, tile = blockIdx.y;
  const int hq = gridDim.x * HP;
  const int G = hq / hkv;
  const int kvh = h0 / G;
  const int s = tile_seq[tile], q0 = tile_q0[tile];
  const int qs = q_start_loc[s], qlen = q_start_loc[s + 1] - qs;
  const int ctx = seq_lens[s];
  const int off = ctx - qlen;  // absolute position of query row 0
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int g4 = lane >> 4, c16 = lane & 15;
  const int* bt = block_tables + (int64_t)s * bt_stride;

  // query row owned by this lane (as the MFMA column)
  const int qr = q0 + w * 16 + c16;
  const bool row_ok = qr < qlen;
  const int qr_c = row_ok ? qr : qlen - 1;
  const int qpos = off + qr_c;
  short8 qf[HP][4];
#pragma unroll
  for (int hh = 0; hh < HP; ++hh) {
    const bf16_t* qrow = q + (int64_t)(qs + qr_c) * q_stride + (h0 + hh) * D;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk)
      qf[hh][kk] = *reinterpret_cast<const short8*>(qrow + kk * 32 + 8 * g4);
  }

  const int last_row = min(q0 + 16 * NW - 1, qlen - 1);
  // kv_lens (ring-attention blocks): keys >= klim are not part of this K/V block
  // even where the causal offset would admit them
  const int klim = kv_lens ? kv_lens[s] : 0x7fffffff;
  const int kv_end = min(off + last_row + 1, klim);  // keys [0, kv_end)
  const int ntiles = (kv_end + 63) / 64;
  const int min_qpos = off + q0;

  float m_run[HP], l_run[HP];
  float4v o[HP][8];
#pragma unroll
  for (int hh = 0; hh < HP; ++hh) {
    m_run[hh] = -INFINITY;
    l_run[hh] = 0.f;
#pragma unroll
    for (int mb = 0; mb < 8; ++mb) o[hh][mb] = float4v{0.f, 0.f, 0.f, 0.f};
  }

  constexpr int NCH = 16 / NW;  // 16-B chunks per thread per 64x128 tile
  short8 kreg[NCH], vreg[NCH];
  auto gload = [&](int t) {
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int c = i * 64 * NW + tid;
      const int row = c >> 4, ch = c & 15;
      const int key = t * 64 + row;
      if (key < kv_end) {
        const int64_t base = (((int64_t)bt[key / BS] * hkv + kvh) * BS + (key % BS)) * D + ch * 8;
        kreg[i] = *reinterpret_cast<const short8*>(kc + base);
        vreg[i] = *reinterpret_cast<const short8*>(vc + base);
      } else {
        kreg[i] = short8{0, 0, 0, 0, 0, 0, 0, 0};
        vreg[i] = short8{0, 0, 0, 0, 0, 0, 0, 0};
      }
    }
  };
  auto lwrite = [&]() {
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int c = i * 64 * NW + tid;
      const int row = c >> 4, ch = c & 15;
      *reinterpret_cast<short8*>(Kl + row * 256 + 16 * kswz(row, ch)) = kreg[i];
      *reinterpret_cast<short8*>(Vl + row * 256 + 16 * vswz(row, ch)) = vreg[i];
    }
  };

  gload(0);
  lwrite();
  __syncthreads();

  for (int t = 0; t < ntiles; ++t) {
    if (t + 1 < ntiles) gload(t + 1);
    const int k0 = t * 64;
    // ---- S^T = K . Q^T  (each K fragment feeds HP heads)
    float4v sacc[HP][4];
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) {
#pragma unroll
      for (int hh = 0; hh < HP; ++hh) sacc[hh][nb] = float4v{0.f, 0.f, 0.f, 0.f};
      const int row = nb * 16 + c16;
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) {
        short8 a = *reinterpret_cast<const short8*>(Kl + row * 256 + 16 * kswz(row, kk * 4 + g4));
#pragma unroll
        for (int hh = 0; hh < HP; ++hh) sacc[hh][nb] = mfma16(a, qf[hh][kk], sacc[hh][nb]);
      }
    }
    const bool need_mask = (k0 + 63 > min_qpos) || (k0 + 63 >= ctx) || (k0 + 63 >= klim);
    short8 pb[HP][2];
#pragma unroll
    for (int hh = 0; hh < HP; ++hh) {
      float mloc = -INFINITY;
#pragma unroll
      for (int nb = 0; nb < 4; ++nb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float v = sacc[hh][nb][r] * scale_log2;
          if (need_mask) {
            const int key = k0 + nb * 16 + g4 * 4 + r;
            if (key > qpos || key >= klim) v = -INFINITY;
          }
          sacc[hh][nb][r] = v;
          mloc = fmaxf(mloc, v);
        }
      mloc = fmaxf(mloc, __shfl_xor(mloc, 16, 64));
      mloc = fmaxf(mloc, __shfl_xor(mloc, 32, 64));
      const float m_new = fmaxf(m_run[hh], mloc);
      const float alpha = exp2f(m_run[hh] - m_new);
      float lsum = 0.f;
#pragma unroll
      for (int nb = 0; nb < 4; ++nb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float p = exp2f(sacc[hh][nb][r] - m_new);
          sacc[hh][nb][r] = p;
          lsum += p;
        }
      lsum += __shfl_xor(lsum, 16, 64);
      lsum += __shfl_xor(lsum, 32, 64);
      l_run[hh] = l_run[hh] * alpha + lsum;
      m_run[hh] = m_new;
#pragma unroll
      for (int mb = 0; mb < 8; ++mb) o[hh][mb] *= alpha;
      // ---- P^T as B operand (k order permuted consistently with the V^T reads)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          pb[hh][ks][j] = (short)f2bf(sacc[hh][2 * ks][j]);
          pb[hh][ks][4 + j] = (short)f2bf(sacc[hh][2 * ks + 1][j]);
        }
      }
    }
    // ---- O^T += V^T . P^T  (each V^T fragment feeds HP heads)
    const int qq = c16 >> 2, pp = c16 & 3;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const int r1 = ks * 32 + g4 * 4 + qq;
      const int r2 = r1 + 16;
#pragma unroll
      for (int mb = 0; mb < 8; ++mb) {
        const int ch = 2 * mb + (pp >> 1);
        typedef short v4s __attribute__((ext_vector_type(4)));
        v4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) v4s*)(Vl + r1 * 256 + 16 * vswz(r1, ch) + 8 * (pp & 1)));
        v4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) v4s*)(Vl + r2 * 256 + 16 * vswz(r2, ch) + 8 * (pp & 1)));
        short8 a = short8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
#pragma unroll
        for (int hh = 0; hh < HP; ++hh) o[hh][mb] = mfma16(a, pb[hh][ks], o[hh][mb]);
      }
    }
    __syncthreads();
    if (t + 1 < ntiles) {
      lwrite();
      __syncthreads();
    }
  }

  if (row_ok) {
#pragma unroll
    for (int hh = 0; hh < HP; ++hh) {
      const float inv = 1.f / l_run[hh];
      bf16_t* orow = out + (int64_t)(qs + qr) * out_stride + (h0 + hh) * D;
#pragma unroll
      for (int mb = 0; mb < 8; ++mb) {
        uint2v pk;
        pk[0] = pack_bf2(o[hh][mb][0] * inv, o[hh][mb][1] * inv);
        pk[1] = pack_bf2(o[hh][mb][2] * inv, o[hh][mb][3] * inv);
        *reinterpret_cast<uint2v*>(orow + mb * 16 + g4 * 4) = pk;
      }
      // natural-log sum of exp of the scaled scores (m_run is in log2 units):
      // the merge statistic of ring attention / split-KV prefill
      if (lse_out && g4 == 0)
        lse_out[(int64_t)(qs + qr) * hq + h0 + hh] = (m_run[hh] + log2f(l_run[hh])) * 0.6931471805599453f;
    }
  }
}


// ----------------------------------------------------------- prefill, 32-row waves
// grid: (Hq / HB, n_tiles of 32 query rows)   block: 64 * HB
// One wave = 32 query rows of one head; the HB waves of a block are HB query
// heads of the same KV head over the SAME rows (GQA), so every 64-key K / V
// tile staged in LDS feeds HB heads and no wave of the block runs a causal
// tile the others skip.  Swapped products on 32x32x16 MFMA:
//   S^T = K . Q^T   lane (q = l&31, hi = l>>5) holds 32 of its row's 64 scores
//                   (keys half*32 + crow(r, hi), crow = (r&3) + 8(r>>2) + 4hi),
//                   so row max / sum are in-lane plus one xor-32 shuffle;
//   O^T += V^T . P^T  the P^T B operand of k-step s is the lane's OWN scores
//                   r = 8(s&1)+j of half s>>1 (no lane exchange): the k slots
//                   are permuted to those keys, and the V^T A operand reads the
//                   same keys -- two runs of 4 -- by ds_read_b64_tr_b16 from a
//                   row-major V image.
// Half the LDS bytes per MFMA of the 16-row kernel above (32 rows share every
// K / V fragment) and no cross-lane softmax beyond one shuffle per statistic.
__device__ __forceinline__ float16v mfma32(short8 a, short8 b, float16v c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// byte offset of 16-B chunk ch of row `row` in a [64][256 B] image: serves the
// ds_read_b128 row reads (K) and the transposed reads (V) conflict-free
__device__ __forceinline__ int img(int row, int ch) {
  return row * 256 + 16 * (ch ^ (((row & 3) << 2) | ((row >> 2) & 3)));
}

// Key partitions of a query tile with ``ntiles`` 64-key tiles, at most S, of at least kPartTiles
// tiles each.
constexpr int kPartTiles = 2;
__device__ __forceinline__ int prefill_parts(int ntiles, int S) {
  return max(1, min(S, ntiles / kPartTiles));
}

// SPLIT: gridDim.z blocks share a query tile's keys, decided from the live length, and write fp32
// partials (O unnormalised [z][T][hq][D], max and sum [z][T][hq][2]) for prefill_merge_kernel; a
// tile of one partition writes its result.  The walk over the keys is a serial chain of 1.35 us a
// 64-key tile, which few query tiles leave most of the chip to wait for (3 tiles of 8 blocks on
// 4000 keys: 89 us, 29 in 8 partitions; ops.prefill_parts).
// KS 2: two groups of HB waves, on every other key tile each, joined through LDS in fp32: two tiles
// in 1.95 us.
template <int BS, int HB, bool SPLIT, int KS>
__global__ __launch_bounds__(64 * HB * KS, HB == 4 ? 2 : 1) void prefill_attn32_kernel(
    bf16_t* __restrict__ out, const bf16_t* __restrict__ q, const bf16_t* __restrict__ kc,
    const bf16_t* __restrict__ vc, const int* __restrict__ block_tables, int bt_stride,
    const int* __restrict__ q_start_loc, const int* __restrict__ seq_lens,
    const int* __restrict__ tile_seq, const int* __restrict__ tile_q0, int hkv, int64_t q_stride,
    int64_t out_stride, float scale_log2, float* __restrict__ lse_out,
    const int* __restrict__ kv_lens, float* __restrict__ part_o, float2* __restrict__ part_ml,
    int64_t part_rows) {
  // two K | V stages (separate objects, so the compiler sees that fragment reads
  // of one stage cannot alias the other stage's in-flight LDS-DMA): the next
  // tile is written while this one is still read, one barrier per tile
  constexpr int STAGE = 2 * 64 * 256;
  __shared__ __attribute__((aligned(16))) char st0[STAGE * KS];
  __shared__ __attribute__((aligned(16))) char st1[STAGE * KS];
  // the sequence's page indices for the first kMaxPages pages, staged once: a K/V
  // prefetch is then ONE global load deep instead of a page-table load followed
  // by the data load it feeds
  constexpr int kMaxPages = 1024;
  __shared__ int pg_lds[kMaxPages];
  __shared__ float joined[KS == 2 ? 2 * HB : 1][64];  // maximum and sum of the second group's lanes

  const int hq = gridDim.x * HB;
  const int G = hq / hkv;
  const int tid = threadIdx.x, lane = tid & 63, w = (tid >> 6) & (HB - 1);
  const int group = KS == 2 ? __builtin_amdgcn_readfirstlane(tid / (64 * HB)) : 0;
  const int h = blockIdx.x * HB + w;
  const int kvh = blockIdx.x * HB / G;
  // a sequence's last tiles, which see most keys, first: what is left for the end is short
  // (4 x 1000 rows, 32 heads on 8, 71.2 -> 61.8 us; 8 x 2048 382 -> 373)
  const int tile = gridDim.y - 1 - blockIdx.y;
  const int s = tile_seq[tile], q0 = tile_q0[tile];
  const int qs = q_start_loc[s], qlen = q_start_loc[s + 1] - qs;
  const int ctx = seq_lens[s];
  const int off = ctx - qlen;
  const int ql = lane & 31, hi = lane >> 5;
  const int* bt = block_tables + (int64_t)s * bt_stride;

  const int qr = q0 + ql;
  const bool row_ok = qr < qlen;
  const int qr_c = row_ok ? qr : qlen - 1;
  const int qpos = off + qr_c;
  short8 qf[8];
  {
    const bf16_t* qrow = q + (int64_t)(qs + qr_c) * q_stride + h * D;
#pragma unroll
    for (int ks = 0; ks < 8; ++ks)
      qf[ks] = *reinterpret_cast<const short8*>(qrow + 16 * ks + 8 * hi);
  }
  const int last_row = min(q0 + 31, qlen - 1);
  const int klim = kv_lens ? kv_lens[s] : 0x7fffffff;
  const int kv_end = min(off + last_row + 1, klim);
  int t0 = 0, ntiles = (kv_end + 63) / 64, parts = 1;
  const int min_qpos = off + q0;
  if constexpr (SPLIT) {
    parts = prefill_parts(ntiles, gridDim.z);
    const int z = blockIdx.z;
    if (z >= parts) return;
    t0 = ntiles * z / parts;
    ntiles = ntiles * (z + 1) / parts;
  }

  const int npg = min((kv_end + BS - 1) / BS, kMaxPages);
  for (int i = tid; i < npg; i += 64 * HB * KS) pg_lds[i] = bt[i];
  __syncthreads();

  // K / V tiles go global -> LDS by LDS-DMA (16 B per lane, 4 rows x 256 B per
  // wave instruction, no staging registers); the image's XOR is applied to the
  // per-lane SOURCE chunk (it is an involution).  Keys past kv_end re-read the
  // last valid key: their scores are masked, so P = 0 meets finite V rows.
  constexpr int NCH = 16 / HB;  // wave instructions per wave per 64-key tensor tile
  typedef __attribute__((address_space(3))) void* lds_ptr_t;
  auto dma = [&](int t, auto BUF) {
    char* Kl = (decltype(BUF)::value ? st1 : st0) + group * STAGE;
    char* Vl = Kl + 64 * 256;
    int page[NCH];  // all page lookups before the first DMA issue
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int key = min(t * 64 + 4 * (w * NCH + i) + (lane >> 4), kv_end - 1);
      const int pi = key / BS;
      const int pl = pg_lds[pi < kMaxPages ? pi : 0];  // an LDS read, not a flat one
      page[i] = pi < kMaxPages ? pl : bt[pi];
    }
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int inst = w * NCH + i;
      const int row = 4 * inst + (lane >> 4), c = lane & 15;
      const int key = min(t * 64 + row, kv_end - 1);
      const int64_t base = (((int64_t)page[i] * hkv + kvh) * BS + (key % BS)) * D +
                           8 * (c ^ (((row & 3) << 2) | ((row >> 2) & 3)));
      __builtin_amdgcn_global_load_lds((const void*)(kc + base), (lds_ptr_t)(Kl + inst * 1024),
                                       16, 0, 0);
      __builtin_amdgcn_global_load_lds((const void*)(vc + base), (lds_ptr_t)(Vl + inst * 1024),
                                       16, 0, 0);
    }
  };

  // a row whose keys all lie before the partition keeps the finite start: its exponents are 0
  float m_run = SPLIT || KS == 2 ? -3.4028234e38f : -INFINITY, l_run = 0.f;
  float16v o[4];
#pragma unroll
  for (int db = 0; db < 4; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[db][r] = 0.f;

  // transposed-read lane roles: 16-lane group g = lane >> 4 covers d columns
  // 16 (g & 1) .. +15 of a 32-column block for k-slot half hi = g >> 1; lane
  // 4 qg + p of the group addresses key row qg, columns 4p .. 4p+3
  const int g = lane >> 4, qg = (lane & 15) >> 2, pp = lane & 3;

  using B0 = std::integral_constant<int, 0>;
  using B1 = std::integral_constant<int, 1>;
  if (KS == 1 || t0 + group < ntiles) dma(t0 + group, B0{});
  __syncthreads();  // vmcnt(0) + barrier: every wave's part of the first tile landed
  // one tile on stage BUF while the next one's DMA fills the other stage; the
  // loop is unrolled by the two stages so every LDS address is a compile-time
  // offset from `lds` -- with a runtime stage index hipcc cannot tell the
  // fragment reads from the in-flight DMA's target and drains it (vmcnt(0))
  // before the first read, which serialises the prefetch
  auto body = [&](int t, auto BUF) {
    constexpr int buf = decltype(BUF)::value;
    // the other stage was last read in tile t-1, before the previous barrier
    if (t + KS < ntiles) dma(t + KS, std::integral_constant<int, 1 - buf>{});
    const char* Kl = (buf ? st1 : st0) + group * STAGE;
    const char* Vl = Kl + 64 * 256;
    const int k0 = t * 64;
    if (KS == 2 && t >= ntiles) {  // the other group has one tile more
      __syncthreads();
      return;
    }
    float16v sacc[2];
#pragma unroll
    for (int half = 0; half < 2; ++half) {
#pragma unroll
      for (int r = 0; r < 16; ++r) sacc[half][r] = 0.f;
#pragma unroll
      for (int ks = 0; ks < 8; ++ks) {
        const short8 a = *reinterpret_cast<const short8*>(Kl + img(half * 32 + ql, 2 * ks + hi));
        sacc[half] = mfma32(a, qf[ks], sacc[half]);
      }
    }
    // causal / block mask only on tiles that reach past this wave's first query
    // (a wave-uniform branch): keys past `lim` (relative to k0) score -inf.
    // Scores stay unscaled here; the scale rides the exponent's FMA.
    float mloc = -INFINITY;
    if (k0 + 63 > min(min_qpos, klim - 1)) {
      const int lim = min(qpos, klim - 1) - k0 - 4 * hi;
#pragma unroll
      for (int half = 0; half < 2; ++half)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float v =
              half * 32 + (r & 3) + 8 * (r >> 2) > lim ? -INFINITY : sacc[half][r];
          sacc[half][r] = v;
          mloc = fmaxf(mloc, v);
        }
    } else {
#pragma unroll
      for (int half = 0; half < 2; ++half)
#pragma unroll
        for (int r = 0; r < 16; ++r) mloc = fmaxf(mloc, sacc[half][r]);
    }
    mloc = fmaxf(mloc, __shfl_xor(mloc, 32, 64)) * scale_log2;
    // lazy rescale: the running max moves only when a row's max grows by more
    // than 2^8 (P <= 256 is exact enough in bf16 / fp32); the O / l rescale is
    // skipped when no row of the wave moved (wave-uniform)
    const bool grow = mloc > m_run + 8.f;
    if (__builtin_amdgcn_ballot_w64(grow)) {
      const float m_new = grow ? mloc : m_run;
      const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);  // 0 on the first tile
      l_run *= alpha;
#pragma unroll
      for (int db = 0; db < 4; ++db) o[db] *= alpha;
      m_run = m_new;
    }
    // v_exp_f32 directly (arguments <= 8: underflow to 0 is the intended result)
    float lsum = 0.f;
#pragma unroll
    for (int half = 0; half < 2; ++half)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(sacc[half][r], scale_log2, -m_run));
        sacc[half][r] = p;
        lsum += p;
      }
    lsum += __shfl_xor(lsum, 32, 64);
    l_run += lsum;
    short8 pb[4];
#pragma unroll
    for (int st = 0; st < 4; ++st)
#pragma unroll
      for (int j = 0; j < 8; ++j)  // native RNE convert (v_cvt_pk_bf16_f32)
        pb[st][j] = __builtin_bit_cast(short, (__bf16)sacc[st >> 1][8 * (st & 1) + j]);
    typedef short v4s __attribute__((ext_vector_type(4)));
#pragma unroll
    for (int st = 0; st < 4; ++st) {
      // keys of k-step st for slot half g >> 1: (st>>1)*32 + 16(st&1) + 4(g>>1) + {0..3, 8..11}
      const int kb = (st >> 1) * 32 + 16 * (st & 1) + 4 * (g >> 1) + qg;
#pragma unroll
      for (int db = 0; db < 4; ++db) {
        const int ch = db * 4 + 2 * (g & 1) + (pp >> 1);
        v4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) v4s*)(Vl + img(kb, ch) + 8 * (pp & 1)));
        v4s hv = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) v4s*)(Vl + img(kb + 8, ch) + 8 * (pp & 1)));
        const short8 a = __builtin_shufflevector(lo, hv, 0, 1, 2, 3, 4, 5, 6, 7);  // concat
        o[db] = mfma32(a, pb[st], o[db]);
      }
    }
    __syncthreads();  // tile t+1's DMA landed (vmcnt(0)) and tile t is read by all
  };
  for (int t = t0; t < ntiles; t += 2 * KS) {
    body(t + group, B0{});
    if (t + KS < ntiles) body(t + KS + group, B1{});
  }
  if constexpr (KS == 2) {
    float4v* sums = reinterpret_cast<float4v*>(st0) + w * 16 * 64 + lane;
    if (group) {
#pragma unroll
      for (int i = 0; i < 16; ++i)
        sums[64 * i] = float4v{o[i >> 2][4 * (i & 3)], o[i >> 2][4 * (i & 3) + 1],
                               o[i >> 2][4 * (i & 3) + 2], o[i >> 2][4 * (i & 3) + 3]};
      joined[w][lane] = m_run;
      joined[HB + w][lane] = l_run;
    }
    __syncthreads();
    if (group) return;
    const float m = joined[w][lane], top = fmaxf(m_run, m);
    const float mine = __builtin_amdgcn_exp2f(m_run - top), other = __builtin_amdgcn_exp2f(m - top);
    m_run = top;
    l_run = l_run * mine + joined[HB + w][lane] * other;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float4v v = sums[64 * i];
#pragma unroll
      for (int r = 0; r < 4; ++r)
        o[i >> 2][4 * (i & 3) + r] = o[i >> 2][4 * (i & 3) + r] * mine + v[r] * other;
    }
  }

  if constexpr (SPLIT) {
    if (parts > 1) {
      if (row_ok) {
        const int64_t row = (blockIdx.z * part_rows + qs + qr) * hq + h;
        float4v* orow = reinterpret_cast<float4v*>(part_o + row * D);
#pragma unroll
        for (int db = 0; db < 4; ++db)
#pragma unroll
          for (int m = 0; m < 4; ++m)
            orow[db * 8 + 2 * m + hi] = float4v{o[db][4 * m], o[db][4 * m + 1],
                                                o[db][4 * m + 2], o[db][4 * m + 3]};
        if (hi == 0) part_ml[row] = float2{m_run, l_run};
      }
      return;
    }
  }
  if (row_ok) {
    const float inv = 1.f / l_run;
    bf16_t* orow = out + (int64_t)(qs + qr) * out_stride + h * D;
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        uint2v pk;
        pk[0] = pack_bf2(o[db][4 * m] * inv, o[db][4 * m + 1] * inv);
        pk[1] = pack_bf2(o[db][4 * m + 2] * inv, o[db][4 * m + 3] * inv);
        *reinterpret_cast<uint2v*>(orow + db * 32 + 8 * m + 4 * hi) = pk;
      }
    if (lse_out && hi == 0)
      lse_out[(int64_t)(qs + qr) * hq + h] = (m_run + log2f(l_run)) * 0.6931471805599453f;
  }
}

// grid: (hq, n_tiles, 4)   block: 256.  A block sums the partitions of 8 rows of one head, 32
// lanes a row; rows with one partition have their result already.
__global__ __launch_bounds__(256) void prefill_merge_kernel(
    bf16_t* __restrict__ out, const float* __restrict__ part_o,
    const float2* __restrict__ part_ml, const int* __restrict__ q_start_loc,
    const int* __restrict__ seq_lens, const int* __restrict__ tile_seq,
    const int* __restrict__ tile_q0, int S, int64_t part_rows, int64_t out_stride) {
  const int hq = gridDim.x, h = blockIdx.x, tile = blockIdx.y;
  const int s = tile_seq[tile], q0 = tile_q0[tile];
  const int qs = q_start_loc[s], qlen = q_start_loc[s + 1] - qs;
  const int kv_end = seq_lens[s] - qlen + min(q0 + 32, qlen);
  const int parts = prefill_parts((kv_end + 63) / 64, S);
  const int qr = q0 + blockIdx.z * 8 + (threadIdx.x >> 5), c = threadIdx.x & 31;
  if (parts <= 1 || qr >= qlen) return;
  const int64_t row = (int64_t)(qs + qr) * hq + h, step = part_rows * hq;
  float m = -INFINITY;
  for (int p = 0; p < parts; ++p) m = fmaxf(m, part_ml[p * step + row].x);
  float l = 0.f;
  float4v acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int p = 0; p < parts; ++p) {
    const float2 v = part_ml[p * step + row];
    const float g = __builtin_amdgcn_exp2f(v.x - m);
    l += g * v.y;
    acc += reinterpret_cast<const float4v*>(part_o + (p * step + row) * D)[c] * g;
  }
  uint2v pk;
  pk[0] = pack_bf2(acc[0] / l, acc[1] / l);
  pk[1] = pack_bf2(acc[2] / l, acc[3] / l);
  *reinterpret_cast<uint2v*>(out + (int64_t)(qs + qr) * out_stride + h * D + 4 * c) = pk;
}

}  // namespace

extern "C" {

// workspace: part_o [B*Hq*max_parts*128] f32, part_ml [B*Hq*max_parts*2] f32
int omnia_decode_attention(void* out, float* part_o, float* part_ml, const void* q,
                           const void* k_cache, const void* v_cache, const int* block_tables,
                           int bt_stride, const int* seq_lens, int B, int hq, int hkv,
                           int head_dim, int block_size, int64_t q_stride, int part_size,
                           int max_parts, float scale, int split_t, int split_min,
                           hipStream_t s) {
  if (head_dim != 128) return -1;
  if (part_size % 64 || part_size % block_size) return -2;
  if (split_t > 0 && (split_min <= 0 || split_t > max_parts)) return -5;
  if (B == 0) return 0;
  const int G = hq / hkv;
  const float scale_log2 = scale * 1.4426950408889634f;
  dim3 grid(B, hkv, max_parts);
#define OMNIA_DEC(GG, BB)                                                                      \
  decode_attn_kernel<GG, BB><<<grid, 64 * NW, 0, s>>>(                                         \
      (bf16_t*)out, part_o, part_ml, (const bf16_t*)q, (const bf16_t*)k_cache,                 \
      (const bf16_t*)v_cache, block_tables, bt_stride, seq_lens, hkv, q_stride, part_size,     \
      max_parts, scale_log2, split_t, split_min)
#define OMNIA_DEC_BS(GG)                                \
  if (block_size == 16) OMNIA_DEC(GG, 16);              \
  else if (block_size == 32) OMNIA_DEC(GG, 32);         \
  else if (block_size == 64) OMNIA_DEC(GG, 64);         \
  else return -3;
  if (G == 1) { OMNIA_DEC_BS(1) }
  else if (G == 2) { OMNIA_DEC_BS(2) }
  else if (G == 4) { OMNIA_DEC_BS(4) }
  else if (G == 8) { OMNIA_DEC_BS(8) }
  else return -4;
#undef OMNIA_DEC_BS
#undef OMNIA_DEC
  if (max_parts > 1)
    decode_reduce_kernel<<<B * hq, 256, 0, s>>>((bf16_t*)out, part_o, part_ml, seq_lens, hq,
                                                part_size, max_parts, split_t, split_min,
                                                block_size);
  return (int)hipGetLastError();
}

int omnia_prefill_attention(void* out, const void* q, const void* k_cache, const void* v_cache,
                            const int* block_tables, int bt_stride, const int* q_start_loc,
                            const int* seq_lens, const int* tile_seq, const int* tile_q0,
                            int n_tiles, int hq, int hkv, int head_dim, int block_size,
                            int64_t q_stride, int64_t out_stride, float scale, int hp_req, int q_tile,
                            float* lse_out, const int* kv_lens, float* part_o, float* part_ml, int parts,
                            int64_t part_rows, int n_seqs, int one_group, hipStream_t s) {
  if (head_dim != 128) return -1;
  if (hq % hkv) return -2;
  if (parts > 1 && (q_tile != 32 || lse_out || kv_lens || !part_o || !part_ml)) return -8;
  if (n_tiles == 0) return 0;
  const float scale_log2 = scale * 1.4426950408889634f;
  // heads per wave (GQA packing) and waves per block (query tile = 16 * nw rows)
  const int G = hq / hkv;
  static const int env_hp = getenv("OMNIA_PREFILL_HP") ? atoi(getenv("OMNIA_PREFILL_HP")) : 0;
  int hp = hp_req > 0 ? hp_req : env_hp > 0 ? env_hp : 1;
  if (hp != 1 && hp != 2 && hp != 4) return -5;
  if (G % hp) hp = 1;
  if (q_tile == 32) {
    // 32-row waves, HB heads of one KV head per block (prefill_attn32_kernel)
    const int hb = G % 4 == 0 ? 4 : G % 2 == 0 ? 2 : 1;
    const dim3 grid32(hq / hb, n_tiles, parts > 1 ? parts : 1);
    // two groups where few blocks wait for the longest walk: one a CU from 6 tiles of keys on, two a
    // CU from 15 where portions are so long (768 rows in the mean) that their walks differ: two groups
    // fill the CU and its blocks come one after the other (us with one / two, 32 heads on 8: 300
    // rows 12.4 / 12.5, 512 16.8 / 15.9, 1001 28.4 / 24.0, behind 3000 keys 93 / 77, 3 x 333 14.9 /
    // 16.9, 4 x 512 27.6 / 29.7, 2 x 1000 41.7 / 32.7, behind 3000 keys 147 / 135, 2001 55.8 / 48.8,
    // 32 x 512 140 / 198; behind 512 to 1500 keys 4 x 512 46.8 / 48.4, 8 x 256 46.8 / 50.3, 16 x 100 64
    // / 70; 32 heads on 16, 8 x 100 behind 1000 41.2 / 46.2).  one_group: never, since two fill a
    // CU's registers and most of its LDS
    const int64_t blocks = (int64_t)(hq / hb) * n_tiles * (parts > 1 ? parts : 1);
    const int64_t keys = (int64_t)bt_stride * block_size / (parts > 1 ? parts : 1);
    const bool twice = !one_group && !kv_lens && !lse_out &&
                       (blocks <= 256 ? keys >= 360
                                      : blocks <= 512 && parts <= 1 && keys >= 900 &&
                                            part_rows >= (int64_t)768 * n_seqs);
#define OMNIA_PRE32(BB, HH)                                                                  \
  do {                                                                                       \
    if (parts > 1 && twice) OMNIA_PRE32_S(BB, HH, true, 2);                                  \
    else if (parts > 1) OMNIA_PRE32_S(BB, HH, true, 1);                                      \
    else if (twice) OMNIA_PRE32_S(BB, HH, false, 2);                                         \
    else OMNIA_PRE32_S(BB, HH, false, 1);                                                    \
  } while (0)
#define OMNIA_PRE32_S(BB, HH, SS, KK)                                                        \
  prefill_attn32_kernel<BB, HH, SS, KK><<<grid32, KK * 64 * HH, 0, s>>>(                     \
      (bf16_t*)out, (const bf16_t*)q, (const bf16_t*)k_cache, (const bf16_t*)v_cache,        \
      block_tables, bt_stride, q_start_loc, seq_lens, tile_seq, tile_q0, hkv, q_stride,      \
      out_stride, scale_log2, lse_out, kv_lens, part_o, (float2*)part_ml, part_rows)
#define OMNIA_PRE32_HB(BB)                 \
  if (hb == 4) OMNIA_PRE32(BB, 4);         \
  else if (hb == 2) OMNIA_PRE32(BB, 2);    \
  else OMNIA_PRE32(BB, 1);
    if (block_size == 16) { OMNIA_PRE32_HB(16) }
    else if (block_size == 32) { OMNIA_PRE32_HB(32) }
    else if (block_size == 64) { OMNIA_PRE32_HB(64) }
    else return -3;
#undef OMNIA_PRE32_HB
#undef OMNIA_PRE32
#undef OMNIA_PRE32_S
    if (parts > 1)
      prefill_merge_kernel<<<dim3(hq, n_tiles, 4), 256, 0, s>>>(
          (bf16_t*)out, part_o, (const float2*)part_ml, q_start_loc, seq_lens, tile_seq, tile_q0,
          parts, part_rows, out_stride);
    return (int)hipGetLastError();
  }
  const int nw = q_tile / 16;
  if (q_tile != 64 && q_tile != 128) return -6;
  if (nw == 8 && hp != 1) return -7;
  dim3 grid(hq / hp, n_tiles), block(64 * nw);
#define OMNIA_PRE(BB, HH, NN)                                                                \
  prefill_attn_kernel<BB, HH, NN><<<grid, block, 0, s>>>(                                    \
      (bf16_t*)out, (const bf16_t*)q, (const bf16_t*)k_cache, (const bf16_t*)v_cache,        \
      block_tables, bt_stride, q_start_loc, seq_lens, tile_seq, tile_q0, hkv, q_stride,      \
      out_stride, scale_log2, lse_out, kv_lens)
#define OMNIA_PRE_HP(BB)                              \
  if (nw == 8) OMNIA_PRE(BB, 1, 8);                   \
  else if (hp == 4) OMNIA_PRE(BB, 4, 4);              \
  else if (hp == 2) OMNIA_PRE(BB, 2, 4);              \
  else OMNIA_PRE(BB, 1, 4);
  if (block_size == 16) { OMNIA_PRE_HP(16) }
  else if (block_size == 32) { OMNIA_PRE_HP(32) }
  else if (block_size == 64) { OMNIA_PRE_HP(64) }
  else return -3;
#undef OMNIA_PRE_HP
#undef OMNIA_PRE
  return (int)hipGetLastError();
}

}  // extern "C"
