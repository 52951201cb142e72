// k_attn.hip — the attention half of one decoder layer for one token (decoder_layer_forward,
// ds_moe_decoder.c:339-431; MHA, single-token decode) on the device:
//   k_attn_qkv     : x_norm = ds_rms_norm(x) in its AVX-512 order (recomputed by every block), then
//                    the rows of [Wq; Wk; Wv] in ds_linear_nobias_bf16_qkv's AVX-512 order with its
//                    split of the rows over the reference's threads (ds_kernels.c:844-915), RoPE
//                    (ds_apply_rope_neox) on the q and k rows; k and v go straight into the cache rows pos;
//   k_attn_scores  : per head x chunk of positions the scores and their maximum (with per-head q/k
//                    norms also the norms and RoPE, recomputed by every block);
//   k_attn_av      : per head x chunk the online softmax's coefficients over the causal or R-SWA
//                    positions (below) and the chunk's sum of V rows;
//   k_attn_oproj   : the chunks' sums put together, then proj = Wo·att in ds_bf16_matvec_threaded's
//                    order;
//   k_attn_post    : h = x + proj and n = ds_rms_norm(h) (ds_residual_rms_norm, AVX-512 order).
// A token moves 13 MB of projections and 10 KB per cached position, a few microseconds of HBM time: what
// bounds it is the number of dependent launches (about 2 us each) and the latency inside each of them.
// Everything except the attention's output sum is bit-exact with the reference. The reference's
// attention is a sequential online softmax with ds_fast_expf (ds_kernels.c:2124-2160,
// :2270-2330). Its branch at each position depends only on the running maximum, so these kernels
// take the same branches with the same exp arguments: a prefix-max scan gives each position's
// running maximum P, its factor f = fast_exp(P - s) on a new maximum (the correction) or
// fast_exp(s - P) (its weight), and a suffix product of the later corrections gives each V row's
// final coefficient c; o = sum c*v and sum_e = sum c are then sums in any order. A chunk of positions
// needs the maximum of the positions before it (the chunk maxima that k_attn_scores leaves) and
// hands on its product of corrections, by which the chunks before it are scaled when the sums are
// put together. The result differs from the reference's sequential recurrence by f32 rounding only.
#include "dsh.h"
#include "dsh_avx.h"
#include "k_core.h"

typedef float f32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ int attn_pos(const int *pos_ptr, int pos_add) { return (pos_ptr ? *pos_ptr : 0) + pos_add; }

// Sum over each aligned group of 16 lanes in _mm512_reduce_add_ps's tree (GCC 11): T3[i] = A[8+i] + A[i],
// T6[j] = T3[4+j] + T3[j], (T6[0]+T6[2]) + (T6[1]+T6[3]), lane i holding A[i]. f32 addition commutes,
// so every lane of the group gets the sum's bits; after a step the values repeat, which lets a
// rotation by 4 stand for the exchange with lane ^ 4.
__device__ __forceinline__ float attn_tree16(float v) {
  v += dsh_dpp<0x128>(v);  // row_ror:8
  v += dsh_dpp<0x124>(v);  // row_ror:4
  v += dsh_dpp<0x4E>(v);   // quad_perm [2,3,0,1]
  return v + dsh_dpp<0xB1>(v);
}

// ds_rms_norm's scale (AVX-512 branch): 16 chains of fused squares over n/16 steps, then the tree;
// r = 1/sqrtf(sum/n + eps). Every 16-lane row of every wave computes it (no barrier, no broadcast
// through LDS). x in LDS, n % 16 == 0. All of a lane's LDS reads are issued ahead of its chain of dependent
// steps (read as needed, three at a time, the chain waited for each).
template <int N>
struct attn_rms {
  float v[N / 16];
  __device__ __forceinline__ void read(const float *x) {
#pragma unroll
    for (int i = 0; i < N / 16; i++) v[i] = x[16 * i + (threadIdx.x & 15)];
  }
  __device__ __forceinline__ float scale(float eps) const {
    float acc = 0.0f;
#pragma unroll
    for (int i = 0; i < N / 16; i++) acc = __builtin_fmaf(v[i], v[i], acc);
    return 1.0f / __builtin_sqrtf(attn_tree16(acc) / (float)N + eps);
  }
};

template <int N>
__device__ __forceinline__ float attn_rms_scale(const float *x, float eps) {
  attn_rms<N> r;
  r.read(x);
  __builtin_amdgcn_sched_barrier(0);
  return r.scale(eps);
}

// Path of global row R of [q; k; v] under ds_linear_nobias_bf16_qkv's split: thread t takes rows
// [t*chunk, min((t+1)*chunk, total)) and runs one ds_bf16_matvec_fused per matrix over its part.
__device__ __forceinline__ int qkv_row_path(int R, int q_dim, int kv_dim, int nthreads) {
  const int total = q_dim + 2 * kv_dim;
  const int m = R < q_dim ? 0 : (R < q_dim + kv_dim ? 1 : 2);
  const int base = m == 0 ? 0 : (m == 1 ? q_dim : q_dim + kv_dim);
  const int mend = m == 0 ? q_dim : (m == 1 ? q_dim + kv_dim : total);
  int s = base, e = mend;
  if (nthreads > 1) {
    const int chunk = (total + nthreads - 1) / nthreads;
    const int t = R / chunk;
    s = max(t * chunk, base);
    e = min(min((t + 1) * chunk, total), mend);
  }
  const int len = e - s, off = R - s;
  if (off < (len & ~3)) return DSH_ROW_GROUP4;
  return off < (len & ~1) ? DSH_ROW_GROUP2 : DSH_ROW_SINGLE;
}

// A bf16 row of length 32*N32 by a 16-lane group, 4 bytes per lane and load: lane c holds columns
// 32i + 2c and 32i + 2c + 1 (c < 8: the reference's accumulator a0, else a1). Sixteen lanes to a row (not
// four with 16-byte loads) give a projection of 1280 x 1280 to 4 waves on each of 80 CUs and leave a lane two
// chains of N32 steps instead of eight.
template <int N32>
__device__ __forceinline__ void attn_row_load(uint32_t *wv, const uint16_t *w, int c) {
#pragma unroll
  for (int i = 0; i < N32; i++) wv[i] = ((const uint32_t *)w)[16 * i + c];
}

// The lane's columns of x (LDS), read ahead of their use.
template <int N32>
__device__ __forceinline__ void attn_row_x(f32x2 *xv, const float *x, int c) {
#pragma unroll
  for (int i = 0; i < N32; i++) xv[i] = ((const f32x2 *)x)[16 * i + c];
}

// The row's value (all 16 lanes) in the path's order against x[k] * rs (rounded; SCALE false: x[k]); xv: the
// lane's columns of x, x in LDS for single rows. The 4- and 2-row groups run 32 chains (a0, a1), then
// a0 + a1 and the tree; a single row 16 chains over 16-column steps. Then "+ bias", 0.0f when absent
// (ds_kernels_avx.c:84-87).
template <int N32, bool SCALE>
__device__ __forceinline__ float attn_row(const uint16_t *w, const uint32_t *wv, const f32x2 *xv, const float *x,
                                          float rs, int c, int path) {
  if (path == DSH_ROW_SINGLE) {
    float a = 0.0f;
    for (int i = 0; i < 2 * N32; i++) {
      const float xs = x[16 * i + c];
      a = __builtin_fmaf(dsh_bf16_to_f32(w[16 * i + c]), SCALE ? xs * rs : xs, a);
    }
    return attn_tree16(a) + 0.0f;
  }
  float a0 = 0.0f, a1 = 0.0f;
#pragma unroll
  for (int i = 0; i < N32; i++) {
    a0 = __builtin_fmaf(dsh_bf16lo(wv[i]), SCALE ? xv[i][0] * rs : xv[i][0], a0);
    a1 = __builtin_fmaf(dsh_bf16hi(wv[i]), SCALE ? xv[i][1] * rs : xv[i][1], a1);
  }
  // lane c: chains 2c and 2c+1; a0 + a1 adds lanes c and c + 8, then the tree over pairs of columns
  f32x2 v = {a0, a1};
  v[0] += dsh_dpp<0x128>(v[0]);
  v[1] += dsh_dpp<0x128>(v[1]);
  v[0] += dsh_dpp<0x124>(v[0]);  // T3: columns 8+i and i are lanes c + 4 and c
  v[1] += dsh_dpp<0x124>(v[1]);
  v[0] += dsh_dpp<0x4E>(v[0]);  // T6: lanes c + 2 and c
  v[1] += dsh_dpp<0x4E>(v[1]);
  v[0] += dsh_dpp<0xB1>(v[0]);  // T6[0]+T6[2] and T6[1]+T6[3]
  v[1] += dsh_dpp<0xB1>(v[1]);
  return (v[0] + v[1]) + 0.0f;
}

// ---------------------------------------------------------------------------- QKV
// The input vector x (H floats, H % 256 == 0), summed over NC (1 or 8) copies [NC][H] in copy order, by a
// block of TH threads: a thread holds the f32x4 pieces threadIdx.x + TH * k (past the end it repeats the
// last one, so that the loads stay unconditional and the waits for them counted). load() issues every load,
// so that a kernel can issue its rows behind them; the adds and stores come with store().
template <int H, int NC, int TH>
struct attn_x {
  static constexpr int NK = (H / 4 + TH - 1) / TH;
  f32x4 v[NC][NK], w[NK];
  static __device__ __forceinline__ int piece(int k) { return min((int)threadIdx.x + TH * k, H / 4 - 1); }
  __device__ __forceinline__ void load(const float *x, const float *wn) {
#pragma unroll
    for (int k = 0; k < NK; k++) {
#pragma unroll
      for (int c = 0; c < NC; c++) v[c][k] = ((const f32x4 *)x)[(size_t)c * (H / 4) + piece(k)];
      if (wn) w[k] = ((const f32x4 *)wn)[piece(k)];
    }
  }
  // x to dst (LDS) and x_out (if given), x times the norm's weights to dst_w (if given)
  __device__ __forceinline__ void store(float *dst, float *dst_w, float *x_out) {
#pragma unroll
    for (int k = 0; k < NK; k++) {
      f32x4 a = v[0][k];
#pragma unroll
      for (int c = 1; c < NC; c++) a += v[c][k];
      if ((int)threadIdx.x + TH * k >= H / 4) continue;
      ((f32x4 *)dst)[piece(k)] = a;
      if (dst_w) ((f32x4 *)dst_w)[piece(k)] = a * w[k];
      if (x_out) ((f32x4 *)x_out)[piece(k)] = a;
    }
  }
};
// Threads of a block that puts n floats together, one f32x4 each.
__host__ __device__ constexpr int attn_threads(int n) { return n / 4 > 256 ? n / 4 : 256; }

// 16 rows of one of q, k, v per 256-thread block (16 lanes per row): 240 blocks at 1280 x 1280, about one
// per CU, each with 40 KB of rows in flight behind its input. The rows of a q or k block are eight
// (d, d + head_dim/2) pairs of one head, a pair in one wave, so the block applies RoPE itself (without the per-head
// norms, which need the whole head first: then q and k go out as they are, for k_attn_scores). 5.3 us at
// 1280 x 1280 (9.8 MB, half of it launch and the input's round trip) against 8.1 with 64 rows per block on 60 CUs.
// H == 32*N32; head_dim % 16 == 0.
template <int N32, int NC>
__global__ void __launch_bounds__(256) k_attn_qkv(dsh_attn_t A, const float *x_in, const int *step, int stride,
                                                  float *x_plain, const int *pos_ptr, int pos_add,
                                                  int nthreads) {
  constexpr int H = 32 * N32;
  __shared__ __attribute__((aligned(16))) float s_x[H], s_xw[H];
  const int hd = A.head_dim, half = hd / 2, qd = A.n_heads * hd, bpm = qd / 16, bph = hd / 16;
  const int m = blockIdx.x / bpm, b = blockIdx.x - m * bpm;
  const int c = threadIdx.x & 15, slot = (threadIdx.x >> 4) & 3, wave = threadIdx.x >> 6;
  const int h = b / bph, t = 8 * (b - h * bph) + 2 * wave + (slot & 1) + (slot >> 1) * half;  // q, k
  const int r = m == 2 ? 16 * b + 4 * wave + slot : h * hd + t;
  const uint16_t *w = (m == 0 ? A.wq : (m == 1 ? A.wk : A.wv)) + (size_t)r * H;
  const int path = qkv_row_path(m * qd + r, qd, qd, nthreads);
  const int pos = attn_pos(pos_ptr, pos_add);
  const float *x = step ? x_in + (size_t)(*step) * stride : x_in;
  attn_x<H, NC, 256> X;
  X.load(x, A.in_norm);
  uint32_t wv[N32];
  float cs = 0.0f, sn = 0.0f;
  attn_row_load<N32>(wv, w, c);
  if (m != 2) {
    cs = A.rope_cos[(size_t)pos * hd + t];
    sn = A.rope_sin[(size_t)pos * hd + t];
  }
  __builtin_amdgcn_sched_barrier(0);  // every load is on its way before the first wait
  X.store(s_x, s_xw, blockIdx.x == 0 ? x_plain : nullptr);  // block 0: x for the residual kernel
  __syncthreads();
  attn_rms<H> rms;
  f32x2 xv[N32];
  rms.read(s_x);
  attn_row_x<N32>(xv, s_xw, c);
  __builtin_amdgcn_sched_barrier(0);
  const float rs = rms.scale(A.eps);
  float v = attn_row<N32, true>(w, wv, xv, s_xw, rs, c, path);
  if (m == 2) {
    if (c == 0) A.vc[(size_t)pos * A.kv_stride + r] = v;
    return;
  }
  if (A.q_norm || A.k_norm) {
    if (c == 0) (m == 0 ? A.q : A.k)[r] = v;
    return;
  }
  const float u = __shfl_xor(v, 32);  // the pair's other row
  v = slot < 2 ? __builtin_fmaf(v, cs, -(u * sn)) : __builtin_fmaf(u, sn, v * cs);
  if (c == 0) {
    if (m == 0)
      A.q[r] = v;
    else
      A.kc[(size_t)pos * A.kv_stride + r] = v;
  }
}

// ---------------------------------------------------------------------------- attention core
// 64-position chunks per k_attn_av block: a head's blocks stay within DSH_ATTN_PARTS.
__device__ __forceinline__ int attn_chunks_per_part(int n) {
  return ((n + 63) / 64 + DSH_ATTN_PARTS - 1) / DSH_ATTN_PARTS;
}

// A DPP move with the value id in lanes that have no source.
template <int CTRL>
__device__ __forceinline__ float attn_dpp_or(float v, float id) {
  return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(id), __float_as_int(v), CTRL, 0xF, 0xF, false));
}

// Scans by DPP within the 16-lane rows (an LDS permute per step of a wave-wide scan costs several times
// the latency). attn_row_max_incl: running maximum up to the lane; attn_row_mul_incl: product from the lane on.
__device__ __forceinline__ float attn_row_max_incl(float v) {
  const float lo = -__builtin_huge_valf();
  v = fmaxf(v, attn_dpp_or<0x111>(v, lo));  // row_shr:1, 2, 4, 8
  v = fmaxf(v, attn_dpp_or<0x112>(v, lo));
  v = fmaxf(v, attn_dpp_or<0x114>(v, lo));
  return fmaxf(v, attn_dpp_or<0x118>(v, lo));
}
__device__ __forceinline__ float attn_row_mul_incl(float v) {
  v *= attn_dpp_or<0x101>(v, 1.0f);  // row_shl:1, 2, 4, 8
  v *= attn_dpp_or<0x102>(v, 1.0f);
  v *= attn_dpp_or<0x104>(v, 1.0f);
  return v * attn_dpp_or<0x108>(v, 1.0f);
}

// The attended positions of the token at cache position pos: p < r1 is position p, then r2 + (p - r1)
// ([0, pos+1), or R-SWA's reference tokens [0, prefill_len) and window [ws, pos+1)).
struct attn_span {
  int r1, r2, n;
  __device__ __forceinline__ int j(int p) const { return p < r1 ? p : r2 + (p - r1); }
};
__device__ __forceinline__ attn_span attn_positions(int pos, int prefill_len, int window) {
  const int kv = pos + 1;
  attn_span sp{kv, kv, kv};
  if (window > 0 && pos >= prefill_len) {
    const int ws = prefill_len > kv - window ? prefill_len : kv - window;
    if (ws > prefill_len) sp = attn_span{prefill_len, ws, prefill_len + (kv - ws)};
  }
  return sp;
}

// The per-head norms (ds_rms_norm_per_head; each optional) and RoPE of one head's q and k (into LDS, one
// dimension per thread). Called by every thread of a block of at least HD threads.
template <int HD>
__device__ void attn_rope_head(const dsh_attn_t &A, int h, int pos, float *s_q, float *s_k) {
  const int t = threadIdx.x, half = HD / 2;
  const float *cs = A.rope_cos + (size_t)pos * HD, *sn = A.rope_sin + (size_t)pos * HD;
  if (t < HD) {
    s_q[t] = A.q[h * HD + t];
    s_k[t] = A.k[h * HD + t];
  }
  __syncthreads();
  const float rq = A.q_norm ? attn_rms_scale<HD>(s_q, A.eps) : 0.0f;
  const float rk = A.k_norm ? attn_rms_scale<HD>(s_k, A.eps) : 0.0f;
  __syncthreads();
  if (t < HD) {
    if (A.q_norm) s_q[t] = (s_q[t] * A.q_norm[t]) * rq;
    if (A.k_norm) s_k[t] = (s_k[t] * A.k_norm[t]) * rk;
  }
  __syncthreads();
  float vq = 0.0f, vk = 0.0f;
  if (t < HD) {
    const int d = t < half ? t : t - half;
    const float q1 = s_q[d], q2 = s_q[d + half], k1 = s_k[d], k2 = s_k[d + half];
    if (t < half) {
      vq = __builtin_fmaf(q1, cs[d], -(q2 * sn[d]));
      vk = __builtin_fmaf(k1, cs[d], -(k2 * sn[d]));
    } else {
      vq = __builtin_fmaf(q1, sn[t], q2 * cs[t]);
      vk = __builtin_fmaf(k1, sn[t], k2 * cs[t]);
    }
  }
  __syncthreads();
  if (t < HD) {
    s_q[t] = vq;
    s_k[t] = vk;
  }
  __syncthreads();
}

// Attended positions per score block, and per maximum that a wave of it leaves in A.cm.
#define ATTN_SCH 64
#define ATTN_MCH 16

// Scores, bit-exact: 64 attended positions per 256-thread block (grid: heads x chunks of the cache), 16
// lanes per position, whole cache lines per load and every K row of a wave (16 positions) in flight at once;
// sc[h][p] = ds_dot_f32(q, k_j) * (1/sqrtf(head_dim)) and cm[h][p/16] the maximum of 16 scores. The order is
// ds_dot_f32's (ds_kernels_avx.c:357-377, head_dim % 64 == 0): four 16-lane accumulators over 64-column
// blocks, added pairwise, then the tree. Lane c holds 4 columns of each block; lane quads 0..3 hold accumulators
// 0, 2, 1, 3, so that lanes c and c ^ 8 hold the first pairs, and after that add the values repeat as the
// rotation by 4 needs.
// NORM: the block norms and ropes q and k itself, and the one that holds the token's own position
// writes its k into the cache row pos. 3.5 us at 702 positions, 8.5 at 7002 (36 MB, 4.2 TB/s); one thread per
// position (a row of 512 bytes per lane) took 5.7 and 13.5.
template <int HD, bool NORM>
__global__ void __launch_bounds__(256) k_attn_scores(dsh_attn_t A, const int *pos_ptr, int pos_add, int prefill_len,
                                                     int window) {
  constexpr int NB = HD / 64, PW = ATTN_MCH / 4;
  __shared__ __attribute__((aligned(16))) float s_q[NORM ? HD : 4], s_k[NORM ? HD : 4];
  const int h = blockIdx.x, c = threadIdx.x & 15;
  const int col4 = 8 * ((c >> 2) & 1) + 4 * (c >> 3) + (c & 3);
  const int pos = attn_pos(pos_ptr, pos_add);
  const attn_span sp = attn_positions(pos, prefill_len, window);
  if ((int)blockIdx.y * ATTN_SCH >= sp.n) return;  // whole block
  const int p0 = blockIdx.y * ATTN_SCH + (threadIdx.x >> 6) * ATTN_MCH + ((threadIdx.x & 63) >> 4);
  f32x4 kv[PW][NB], q[NB];
#pragma unroll
  for (int i = 0; i < PW; i++) {
    const float *kr = A.kc + (size_t)sp.j(min(p0 + 4 * i, sp.n - 1)) * A.kv_stride + h * HD;
#pragma unroll
    for (int b = 0; b < NB; b++) kv[i][b] = ((const f32x4 *)kr)[16 * b + col4];
  }
  if (NORM) {
    attn_rope_head<HD>(A, h, pos, s_q, s_k);
    // this block holds position n-1 == pos
    if (((int)blockIdx.y + 1) * ATTN_SCH >= sp.n && (int)threadIdx.x < HD)
      A.kc[(size_t)pos * A.kv_stride + h * HD + threadIdx.x] = s_k[threadIdx.x];
#pragma unroll
    for (int i = 0; i < PW; i++)
      if (p0 + 4 * i >= sp.n - 1)
#pragma unroll
        for (int b = 0; b < NB; b++) kv[i][b] = ((const f32x4 *)s_k)[16 * b + col4];
  }
#pragma unroll
  for (int b = 0; b < NB; b++) q[b] = ((const f32x4 *)(NORM ? s_q : A.q + h * HD))[16 * b + col4];
  const float scale = 1.0f / __builtin_sqrtf((float)HD);
  float mx = -__builtin_huge_valf();
#pragma unroll
  for (int i = 0; i < PW; i++) {
    float a[4];
#pragma unroll
    for (int e = 0; e < 4; e++) {
      a[e] = 0.0f;
#pragma unroll
      for (int b = 0; b < NB; b++) a[e] = __builtin_fmaf(q[b][e], kv[i][b][e], a[e]);
      a[e] += dsh_dpp<0x128>(a[e]);  // accumulators 0+1 and 2+3
      a[e] += dsh_dpp<0x124>(a[e]);  // their sum
      a[e] += dsh_dpp<0x4E>(a[e]);  // T3: columns 8+i and i are lanes c + 2 and c
      a[e] += dsh_dpp<0xB1>(a[e]);  // T6
    }
    const float s = ((a[0] + a[2]) + (a[1] + a[3])) * scale;
    if (p0 + 4 * i < sp.n) {
      if (c == 0) A.sc[(size_t)h * A.max_seq + p0 + 4 * i] = s;
      mx = fmaxf(mx, s);  // a NaN score is never a new maximum: fmaxf skips it
    }
  }
  mx = fmaxf(mx, __shfl_xor(mx, 16));
  mx = fmaxf(mx, __shfl_xor(mx, 32));
  if ((threadIdx.x & 63) == 0) A.cm[(size_t)h * DSH_ATTN_CM(A.max_seq) + p0 / ATTN_MCH] = mx;
}

// V: up to four 64-position chunks per 256-thread block (grid: heads x DSH_ATTN_PARTS), as many as keep a
// head's blocks within DSH_ATTN_PARTS, so that the next kernel has few sums to put together: one up to 1920
// positions (160 blocks for 10 heads at 1000), four at 7680. Wave w computes the coefficients of chunk w
// (lane = position): with P the maximum of the scores before the position (the reference starts from
// max_s = -1e30), a = its correction on a new maximum (else 1), g = 1 on a new maximum (else the weight),
// c = g * (the product of the later corrections of the chunk). Then every thread adds c * v for 4 dimensions
// of 1024/HD-th of the positions, its loads issued before the coefficients are known, and the block writes
// its sum, its sum of c and its product of corrections. 4.0 us at 702 positions, 8.5 at 7002 (36 MB), against 8.9
// and 25.7 for a kernel with one block per head for the coefficients and one for the sums.
template <int HD>
__global__ void __launch_bounds__(256) k_attn_av(dsh_attn_t A, const int *pos_ptr, int pos_add, int prefill_len,
                                                 int window) {
  constexpr int DL = HD / 4, G = 256 / DL, NP = (64 + G - 1) / G;  // lanes per row, rows at once, rows per thread
  __shared__ float s_c[4][64], s_a[4], s_e[4];
  __shared__ __attribute__((aligned(16))) float s_o[G * HD];
  const int h = blockIdx.x, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const attn_span sp = attn_positions(attn_pos(pos_ptr, pos_add), prefill_len, window);
  const int g = attn_chunks_per_part(sp.n);
  const int p0 = blockIdx.y * g * 64;
  if (p0 >= sp.n) return;  // whole block
  const int nc = min(g, (sp.n - p0 + 63) / 64);
  const int d4 = threadIdx.x % DL, pg = threadIdx.x / DL;  // HD 192: the last 16 threads have pg == G
  const float *vh = A.vc + h * HD;
  f32x4 v[NP];
  auto load = [&](int ch) {
#pragma unroll
    for (int i = 0; i < NP; i++)
      v[i] = ((const f32x4 *)(vh + (size_t)sp.j(min(p0 + 64 * ch + pg + G * i, sp.n - 1)) * A.kv_stride))[d4];
  };
  if (wave < nc) {
    const int q0 = p0 + 64 * wave, p = q0 + lane;
    const float *cm = A.cm + (size_t)h * DSH_ATTN_CM(A.max_seq);
    const int nm = q0 / ATTN_MCH;  // maxima before the chunk
    float t[DSH_ATTN_CM_MAX / 64];
    const float sp0 = A.sc[(size_t)h * A.max_seq + min(p, sp.n - 1)];
#pragma unroll
    for (int k = 0; k < DSH_ATTN_CM_MAX / 64; k++) t[k] = cm[min(lane + 64 * k, max(nm - 1, 0))];
    load(0);
    __builtin_amdgcn_sched_barrier(0);  // every load is on its way before the first wait
    const float s = p < sp.n ? sp0 : -__builtin_huge_valf();
    float before = -1e30f;
#pragma unroll
    for (int k = 0; k < DSH_ATTN_CM_MAX / 64; k++) before = fmaxf(before, lane + 64 * k < nm ? t[k] : -1e30f);
    before = dsh_wave_max(before);
    // maximum of the scores before the lane: the row's, and the rows before it
    const int row = lane >> 4;
    const float m = attn_row_max_incl(s);
    float P = fmaxf(before, attn_dpp_or<0x111>(m, -1e30f));
#pragma unroll
    for (int k = 0; k < 3; k++) P = fmaxf(P, row > k ? dsh_readlane(m, 16 * k + 15) : -1e30f);
    const bool nw = s > P;
    const float f = dsh_fast_expf(nw ? P - s : s - P);
    const bool in = p < sp.n;
    // product of the corrections after the lane: the row's, and the rows after it
    const float mul = attn_row_mul_incl(in && nw ? f : 1.0f);
    const float m1 = dsh_readlane(mul, 16), m2 = dsh_readlane(mul, 32), m3 = dsh_readlane(mul, 48);
    const float rows = row == 0 ? m1 * (m2 * m3) : (row == 1 ? m2 * m3 : (row == 2 ? m3 : 1.0f));
    const float dn = attn_dpp_or<0x101>(mul, 1.0f) * rows;
    const float after = dsh_readlane(mul, 0) * (m1 * (m2 * m3));
    const float cf = in ? (nw ? 1.0f : f) * dn : 0.0f;
    s_c[wave][lane] = cf;
    const float se = dsh_wave_sum(cf);
    if (lane == 0) {
      s_a[wave] = after;
      s_e[wave] = se;
    }
  } else {
    load(0);
  }
  __syncthreads();
  f32x4 o = {0.0f, 0.0f, 0.0f, 0.0f};
  float se = 0.0f, prod = 1.0f;
  for (int ch = 0; ch < nc; ch++) {
    const float fall = s_a[ch];
    o *= fall;  // the chunks before it (nothing yet at the first)
    se = se * fall + s_e[ch];
    prod *= fall;
    f32x4 cur[NP];
#pragma unroll
    for (int i = 0; i < NP; i++) cur[i] = v[i];
    if (ch + 1 < nc) load(ch + 1);
#pragma unroll
    for (int i = 0; i < NP; i++) {
      const int p = pg + G * i;
      const float cf = p < 64 ? s_c[ch][p] : 0.0f;
#pragma unroll
      for (int e = 0; e < 4; e++) o[e] = __builtin_fmaf(cf, cur[i][e], o[e]);
    }
  }
  if (pg < G) ((f32x4 *)s_o)[pg * DL + d4] = o;
  __syncthreads();
  const int part = h * DSH_ATTN_PARTS + blockIdx.y;
  if ((int)threadIdx.x < HD) {
    float sum = 0.0f;
#pragma unroll
    for (int k = 0; k < G; k++) sum += s_o[k * HD + threadIdx.x];
    A.part[(size_t)part * HD + threadIdx.x] = sum;
  }
  if (threadIdx.x == 0) {
    A.pa[part] = prod;
    A.pe[part] = se;
  }
}

// ---------------------------------------------------------------------------- O projection
// 16 output rows per block (threads past 256 only help with att); every block puts att together itself (head h: the
// parts' sums times the product of the later parts' corrections, in part order, times 1/sum_e: ds_vec_scale_inplace,
// sum_e > 0), at most 30 x q_dim floats from L2, which costs less than a launch of its own: 5.6 us in all at 702
// positions and 7.1 at 7002, against 5.8 + 3.7 and 5.0 + 9.9 in two kernels. q_dim == 32*N32.
template <int N32>
__global__ void __launch_bounds__(attn_threads(32 * N32))
    k_attn_oproj(dsh_attn_t A, const int *pos_ptr, int pos_add, int prefill_len, int window, int chunk) {
  constexpr int QD = 32 * N32, PP = 16;  // parts in flight
  __shared__ __attribute__((aligned(16))) float s_a[QD];
  __shared__ float s_f[QD / 64 * DSH_ATTN_PARTS], s_inv[QD / 64];
  const int c = threadIdx.x & 15;
  const int r = blockIdx.x * 16 + ((threadIdx.x >> 4) & 15);
  const uint16_t *w = A.wo + (size_t)r * QD;
  const int path = row_path(r, A.H, chunk, false);
  const int n = attn_positions(attn_pos(pos_ptr, pos_add), prefill_len, window).n;
  const int g64 = attn_chunks_per_part(n) * 64, np = (n + g64 - 1) / g64;
  const int dl = A.head_dim / 4;
  constexpr int NH = (QD / 64 + 7) / 8;  // heads per half wave, at most
  f32x4 t[PP];
  const int i0 = min((int)threadIdx.x, QD / 4 - 1), h0 = i0 / dl;  // the thread's f32x4 piece of att
  const f32x4 *q = (const f32x4 *)A.part + (size_t)h0 * DSH_ATTN_PARTS * dl + (i0 - h0 * dl);
  // the factors' inputs, half a wave per head
  const int hw = (threadIdx.x >> 5) & 7, k = threadIdx.x & 31;
  float pa[NH], pe[NH];
#pragma unroll
  for (int i = 0; i < NH; i++) {
    const int at = min(hw + 8 * i, A.n_heads - 1) * DSH_ATTN_PARTS + min(k, np - 1);
    pa[i] = A.pa[at];
    pe[i] = A.pe[at];
  }
#pragma unroll
  for (int j = 0; j < PP; j++) t[j] = q[(size_t)min(j, np - 1) * dl];
  uint32_t wv[N32];
  if (threadIdx.x < 256) attn_row_load<N32>(wv, w, c);
  __builtin_amdgcn_sched_barrier(0);  // every load is on its way before the first wait
#pragma unroll
  for (int i = 0; i < NH; i++) {
    const int h = hw + 8 * i;
    const float a = k < np ? pa[i] : 1.0f, e = k < np ? pe[i] : 0.0f;
    const float mul = attn_row_mul_incl(a), upper = __shfl(mul, 16, 32);
    const float f = attn_dpp_or<0x101>(mul, 1.0f) * (k < 16 ? upper : 1.0f);
    float tot = dsh_row16_sum(e * f);
    tot += __shfl_xor(tot, 16);
    if (h < A.n_heads) {
      if (k < DSH_ATTN_PARTS) s_f[h * DSH_ATTN_PARTS + k] = f;
      if (k == 0) s_inv[h] = tot > 0.0f ? 1.0f / tot : 1.0f;
    }
  }
  __syncthreads();
  if (threadIdx.x < QD / 4) {
    f32x4 o = {0.0f, 0.0f, 0.0f, 0.0f};
    const float *f = s_f + h0 * DSH_ATTN_PARTS;
#pragma unroll
    for (int j = 0; j < PP; j++)
      if (j < np) o += f[j] * t[j];
    if (np > PP) {  // the rest, again with every load in flight
#pragma unroll
      for (int j = PP; j < DSH_ATTN_PARTS; j++) t[j - PP] = q[(size_t)min(j, np - 1) * dl];
#pragma unroll
      for (int j = PP; j < DSH_ATTN_PARTS; j++)
        if (j < np) o += f[j] * t[j - PP];
    }
    ((f32x4 *)s_a)[threadIdx.x] = o * s_inv[h0];
  }
  __syncthreads();
  if (threadIdx.x >= 256) return;
  f32x2 xv[N32];
  attn_row_x<N32>(xv, s_a, c);
  __builtin_amdgcn_sched_barrier(0);
  const float v = attn_row<N32, false>(w, wv, xv, s_a, 1.0f, c, path);
  if (c == 0) A.proj[r] = v;
}

// ---------------------------------------------------------------------------- residual RMSNorm
// R rows per 256-thread block (H / R blocks): every block forms h = x + proj (rounded) in LDS and
// the RMSNorm scale (ds_residual_rms_norm, AVX-512 order), writes its rows of h and n = (h*w)*r
// and, given the next MoE layer's transposed f32 router WrT ([H][E]), the partial router scores of
// its rows (the format of k_dec_partial_scores: one row of 64 per block, its rows added in order).
template <int N32, int R>
__global__ void __launch_bounds__(256) k_attn_post(dsh_attn_t A, const float *x_in, const int *step, int stride,
                                                   float *h_out, float *n_out,
                                                   const float *__restrict__ WrT, int E, float *__restrict__ partials) {
  constexpr int H = 32 * N32;
  __shared__ __attribute__((aligned(16))) float s_h[H];
  __shared__ float s_n[R];
  const float *x = step ? x_in + (size_t)(*step) * stride : x_in;
  const int r0 = blockIdx.x * R;
  float wr[R];
  if (WrT && (int)threadIdx.x < E) {
#pragma unroll
    for (int j = 0; j < R; j++) wr[j] = WrT[(size_t)(r0 + j) * E + threadIdx.x];
  }
  for (int i = threadIdx.x; i < H / 4; i += 256) {
    const f32x4 xv = ((const f32x4 *)x)[i], pv = ((const f32x4 *)A.proj)[i];
    ((f32x4 *)s_h)[i] = xv + pv;
  }
  __syncthreads();
  const float r = attn_rms_scale<H>(s_h, A.eps);
  if (threadIdx.x < R) {
    const int i = r0 + threadIdx.x;
    const float nv = (s_h[i] * A.post_norm[i]) * r;
    h_out[i] = s_h[i];
    n_out[i] = nv;
    s_n[threadIdx.x] = nv;
  }
  __syncthreads();
  if (WrT && threadIdx.x < 64) {
    float p = 0.0f;
    if ((int)threadIdx.x < E) {
#pragma unroll
      for (int j = 0; j < R; j++) p = __builtin_fmaf(wr[j], s_n[j], p);
    }
    partials[(size_t)blockIdx.x * 64 + threadIdx.x] = (int)threadIdx.x < E ? p : 0.0f;
  }
}

// ds_rms_norm of the last hidden state before the LM head (ds_moe_decoder.c:1000), AVX-512 order;
// trunc: ds_bf16_truncate_array after it (:1016-1018, bf16 simulation of model version 3).
template <int N32, int NC>
__global__ void __launch_bounds__(attn_threads(32 * N32))
    k_final_norm(const float *__restrict__ x, const float *__restrict__ w, float eps, int trunc,
                 float *__restrict__ out, float *__restrict__ x_out) {
  constexpr int H = 32 * N32;
  __shared__ __attribute__((aligned(16))) float s_x[H];
  attn_x<H, NC, attn_threads(H)> X;
  X.load(x, nullptr);
  X.store(s_x, nullptr, x_out);
  __syncthreads();
  const float r = attn_rms_scale<H>(s_x, eps);
  for (int i = threadIdx.x; i < H; i += blockDim.x) {
    const float v = (s_x[i] * w[i]) * r;
    out[i] = trunc ? dsh_bf16_round_half_up(v) : v;
  }
}

extern "C" {

int dsh_attn_supported(int H, int n_heads, int head_dim) {
  const int qd = n_heads * head_dim;
  return H % 256 == 0 && H / 256 >= 1 && H / 256 <= 8 && head_dim % 64 == 0 && head_dim <= DSH_ATTN_MAX_HD &&
         qd % 256 == 0 && qd / 256 >= 1 && qd / 256 <= 8;
}

hipError_t dsh_launch_attn(const dsh_attn_t *A, const float *x_in, const int *step, int stride, int ncopies,
                           float *x_plain, const int *pos_ptr, int pos_add, int prefill_len, int window, int nthreads,
                           float *h_out, float *n_out, const float *WrT_next, int E_next, float *partials_next,
                           hipStream_t s) {
  if (!dsh_attn_supported(A->H, A->n_heads, A->head_dim)) return hipErrorInvalidValue;
  if ((ncopies != 1 && ncopies != 8) || (ncopies > 1 && (step || !x_plain))) return hipErrorInvalidValue;
  const float *x_post = ncopies > 1 ? x_plain : x_in;  // the residual kernel reads one plain vector
  const int qd = A->n_heads * A->head_dim;
#define QKV(N)                                                                                              \
  case N:                                                                                                   \
    if (ncopies > 1)                                                                                        \
      k_attn_qkv<8 * N, 8><<<3 * qd / 16, 256, 0, s>>>(*A, x_in, step, stride, x_plain, pos_ptr, pos_add,    \
                                                       nthreads);                                           \
    else                                                                                                    \
      k_attn_qkv<8 * N, 1><<<3 * qd / 16, 256, 0, s>>>(*A, x_in, step, stride, nullptr, pos_ptr, pos_add,    \
                                                       nthreads);                                           \
    break;
  switch (A->H / 256) {
    QKV(1) QKV(2) QKV(3) QKV(4) QKV(5) QKV(6) QKV(7) QKV(8)
    default:
      return hipErrorInvalidValue;
  }
#undef QKV
  const int nch = (A->max_seq + 63) / 64;
  const dim3 gs(A->n_heads, nch), gv(A->n_heads, nch < DSH_ATTN_PARTS ? nch : DSH_ATTN_PARTS);
#define CORE(HD)                                                                                        \
  case HD:                                                                                              \
    if (A->q_norm || A->k_norm)                                                                         \
      k_attn_scores<HD, true><<<gs, 256, 0, s>>>(*A, pos_ptr, pos_add, prefill_len, window);            \
    else                                                                                                \
      k_attn_scores<HD, false><<<gs, 256, 0, s>>>(*A, pos_ptr, pos_add, prefill_len, window);           \
    k_attn_av<HD><<<gv, 256, 0, s>>>(*A, pos_ptr, pos_add, prefill_len, window);                        \
    break;
  switch (A->head_dim) {
    CORE(64) CORE(128) CORE(192) CORE(256)
    default:
      return hipErrorInvalidValue;
  }
#undef CORE
  const int chunk = dsh_chunk_len(A->H, nthreads);
#define OP(N)                                                                                              \
  case N:                                                                                                  \
    k_attn_oproj<8 * N><<<A->H / 16, attn_threads(qd), 0, s>>>(*A, pos_ptr, pos_add, prefill_len, window,  \
                                                               chunk);                                     \
    break;
  switch (qd / 256) {
    OP(1) OP(2) OP(3) OP(4) OP(5) OP(6) OP(7) OP(8)
    default:
      return hipErrorInvalidValue;
  }
#undef OP
#define PO(N, RR)                                                                                           \
  case N:                                                                                                   \
    k_attn_post<8 * N, RR><<<A->H / RR, 256, 0, s>>>(*A, x_post, ncopies > 1 ? nullptr : step, stride,        \
                                                     h_out, n_out, WrT_next, E_next, partials_next);        \
    break;
  if (WrT_next && (E_next <= 0 || E_next > 64)) return hipErrorInvalidValue;
  if (A->H / dsh_dec_partials(A->H) == 8) {
    switch (A->H / 256) {
      PO(1, 8) PO(2, 8) PO(3, 8) PO(4, 8) PO(5, 8)
      default:
        return hipErrorInvalidValue;
    }
  } else {
    switch (A->H / 256) {
      PO(6, 16) PO(7, 16) PO(8, 16)
      default:
        return hipErrorInvalidValue;
    }
  }
#undef PO
  return hipGetLastError();
}

hipError_t dsh_launch_final_norm(const float *x, int ncopies, const float *w, int H, float eps, int trunc, float *out,
                                 float *x_out, hipStream_t s) {
#define FN(N)                                                                           \
  case N:                                                                               \
    if (ncopies > 1)                                                                    \
      k_final_norm<8 * N, 8><<<1, attn_threads(H), 0, s>>>(x, w, eps, trunc, out, x_out);           \
    else                                                                                \
      k_final_norm<8 * N, 1><<<1, attn_threads(H), 0, s>>>(x, w, eps, trunc, out, x_out);           \
    break;
  if (H % 256 || (ncopies != 1 && ncopies != 8)) return hipErrorInvalidValue;
  switch (H / 256) {
    FN(1) FN(2) FN(3) FN(4) FN(5) FN(6) FN(7) FN(8)
    default:
      return hipErrorInvalidValue;
  }
#undef FN
  return hipGetLastError();
}

}  // extern "C"
