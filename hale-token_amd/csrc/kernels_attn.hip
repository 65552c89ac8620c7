// kernels_attn.hip -- the steps on either side of the MoE block on gfx950:
// RMSNorm (src/ops/norm.rs) and one-token grouped-query attention with
// QK-norm, RoPE and a KV cache (src/model/attention.rs, src/ops/rope.rs,
// src/model/kv_cache.rs).
//
// Every sum keeps the reference's order, so every result is bit-identical:
//   - RMSNorm's squares are summed in order (from -0.0 in the reference,
//     Iterator::sum; the start shows only without values), then
//     1 / sqrt(sum / n + eps), then x * scale * w (rms_norm) or
//     x * (scale * w) (rms_norm_in_place);
//   - a score is the in-order sum q[0]k[0] + q[1]k[1] + ... from -0.0,
//     times 1 / sqrt(hd); softmax is softmax_in_place (max, glibc exp, an
//     in-order sum from 0.0, one division per score);
//   - a context element is 0 + p_0 v_0 + p_1 v_1 + ... in position order.
// The products and the exponentials are computed in parallel.  The sums of
// RMSNorm and, in rows of up to 8192 positions, of softmax are formed by many
// lanes with the chain's bits (ordered_sum.h); scores, the context, QK-norm and
// the softmax of longer rows are chains, one lane each.
#pragma clang fp contract(off)

#include "hale_device.h"
#include "kernels.h"
#include "ordered_sum.h"

namespace hale {

constexpr int NORM_MAX = ORDERED_MAX;  // elements of an RMSNorm row
constexpr int HEAD_MAX = 1024;     // largest head_dim

// One work-group per row: out = rms_norm(x + delta, w) with x updated to
// x + delta first when delta is given (add_in_place, then rms_norm).  The
// row and the weights are read once, all loads in flight together, and stay
// in registers through the in-order sum of the squares.  (out may be x
// itself: every element is read before any is written.)
//
// Bound by latency: one load round trip, the ordered sum, one store.  The
// squares go through LDS to become each lane's K consecutive values
// (ordered_sum.h); K NT is the smallest that covers the row, as every unused K
// costs its predicated loads and chain steps.  Rows above 2048 go to 512
// threads: half as many values per lane, for four more turns of the waves
// (one row of 4096 / 8192: 6.4 / 9.7 us with 256, 5.5 / 7.3 with 512; 1500 of
// 8192: 46 and 35).  One row of 2048: 13.9 us with one chain of squares, 4.6
// so (a launch alone is about 3.5).  The sum starts from +0: the reference's
// -0 start shows only without values.
template <int K, int NT>
__global__ __launch_bounds__(NT) void k_rms_norm(float* x, const float* __restrict__ delta,
                                                  const float* __restrict__ w, int n, float eps,
                                                  float* out) {
  // 4 floats of padding every 32 keep the lanes' 16-byte reads at a stride
  // of K floats off each other's banks
  auto at = [](int i) { return i + (i >> 5) * 4; };
  __shared__ __attribute__((aligned(16))) float sq[NT * K + NT * K / 8];
  __shared__ float part[ordered_lds(NT / 64)];
  float* xr = x + (size_t)blockIdx.x * n;
  const float* dr = delta ? delta + (size_t)blockIdx.x * n : nullptr;
  float* orow = out + (size_t)blockIdx.x * n;
  const int tid = threadIdx.x;
  float xv[K], wv[K];
#pragma unroll
  for (int j = 0; j < K; j++) {
    const int i = tid + NT * j;
    if (i < n) {
      xv[j] = xr[i];
      wv[j] = w[i];
    }
  }
  if (dr) {
    float dv[K];
#pragma unroll
    for (int j = 0; j < K; j++) {
      const int i = tid + NT * j;
      if (i < n) dv[j] = dr[i];
    }
#pragma unroll
    for (int j = 0; j < K; j++) {
      const int i = tid + NT * j;
      if (i < n) {
        xv[j] = xv[j] + dv[j];
        xr[i] = xv[j];
      }
    }
  }
#pragma unroll
  for (int j = 0; j < K; j++) {
    const int i = tid + NT * j;
    sq[at(i)] = i < n ? xv[j] * xv[j] : 0.0f;
  }
  __syncthreads();
  float v[K];
#pragma unroll
  for (int q = 0; q < K / 4; q++) {
    const f32x4 t = *(const f32x4*)&sq[at(tid * K + 4 * q)];
    v[4 * q] = t.x;
    v[4 * q + 1] = t.y;
    v[4 * q + 2] = t.z;
    v[4 * q + 3] = t.w;
  }
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const float s = team_sum_in_order<K>(v, 0.0f, wave, NT / 64, part);
  const float scale = 1.0f / sqrtf(s / (float)n + eps);
#pragma unroll
  for (int j = 0; j < K; j++) {
    const int i = tid + NT * j;
    if (i < n) orow[i] = xv[j] * scale * wv[j];
  }
}

// One token's projections and what becomes of them (AttnArgs without the
// buffers between the kernels).
struct TokenArgs {
  const float *q, *k, *v;         // projection outputs
  const float *q_norm, *k_norm;   // [hd] or null
  const float *cos, *sin;         // [hd / 2]
  float eps;
  float *keys, *values;           // the layer cache
  int hd, kv_dim, group, cap, seq;
};

// The cache: values [position][nkv * hd]; keys head by head in pieces of four
// dimensions, [head][hd / 4][position][4], so that a wave whose lanes take one
// position each reads a piece of 64 positions as one kilobyte.
__device__ __forceinline__ size_t key_piece(const TokenArgs& a, int g, int piece, int t) {
  return (((size_t)g * (a.hd / 4) + piece) * a.cap + t) * 4;
}

// Orders a wave's LDS accesses: what its lanes wrote, any of them now reads.
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// QK-norm and RoPE of R heads by one wave, into LDS rows of hd + 4 floats (the
// padding keeps the rows' 16-byte reads 4 banks apart).  load() takes the
// first 128 values of each head and what they are multiplied with into
// registers, unconditionally, so that the key loads which follow it can stay
// in flight while store() runs: loads return in order.  The norm's sum of hd
// squares is one chain per head, a lane each; a wave none of whose heads is
// normed skips it (without QK-norm, 1100 positions of 32 heads of 128: 27.1 ->
// 25.6 us a token; 190 of 16 heads of 256 23.6 -> 21.7, of 4 heads of 1024 44.8
// -> 37.0).  Beyond 128 values the heads' loads go out side by side (8 heads of
// 1024 with QK-norm, 520 positions by two launches: 75.5 us a head after the
// other, 66.1 so).
template <int R>
struct HeadRows {
  const float* src[R];   // wave-uniform
  const float* norm[R];  // or null
  float x[R][2], w[R][2], cs, sn;
  __device__ __forceinline__ void load(const TokenArgs& a) {
    const int lane = __lane_id(), last = a.hd - 1, half = a.hd / 2;
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
      for (int j = 0; j < 2; j++) {
        x[r][j] = src[r][min(lane + 64 * j, last)];
        w[r][j] = (norm[r] ? norm[r] : src[r])[min(lane + 64 * j, last)];
      }
    cs = a.cos[min(lane, half - 1)];
    sn = a.sin[min(lane, half - 1)];
  }
  __device__ __forceinline__ void store(const TokenArgs& a, float* rows) {
    const int lane = __lane_id(), hd = a.hd, half = hd / 2, pitch = hd + 4;
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
      for (int j = 0; j < 2; j++)
        if (lane + 64 * j < hd) rows[r * pitch + lane + 64 * j] = x[r][j];
#pragma unroll 4
    for (int c = 128 + lane; c < hd; c += 64)
#pragma unroll
      for (int r = 0; r < R; r++) rows[r * pitch + c] = src[r][c];
    wave_lds_sync();
    float scale = 0.0f;  // inverse_rms (src/ops/norm.rs:25-28), in order from -0.0
    bool any = false;    // uniform
#pragma unroll
    for (int r = 0; r < R; r++) any = any || norm[r];
    if (any) {
      if (lane < R) {
        const f32x4* row = (const f32x4*)(rows + lane * pitch);
        float s = -0.0f;
#pragma unroll 8
        for (int i = 0; i < hd / 4; i++) {
          const f32x4 v = row[i];
          s = s + v.x * v.x;
          s = s + v.y * v.y;
          s = s + v.z * v.z;
          s = s + v.w * v.w;
        }
        scale = 1.0f / sqrtf(s / (float)hd + a.eps);
      }
      wave_lds_sync();
    }
    // rms_norm_in_place: x = x * (scale * w)
    float sc[R];
#pragma unroll
    for (int r = 0; r < R; r++) sc[r] = lane_value(scale, r);
    if (hd <= 128) {
#pragma unroll
      for (int r = 0; r < R; r++)
#pragma unroll
        for (int j = 0; j < 2; j++)
          if (norm[r] && lane + 64 * j < hd) rows[r * pitch + lane + 64 * j] = x[r][j] * (sc[r] * w[r][j]);
    } else if (any) {
#pragma unroll 4
      for (int c = lane; c < hd; c += 64)
#pragma unroll
        for (int r = 0; r < R; r++)
          if (norm[r]) rows[r * pitch + c] = rows[r * pitch + c] * (sc[r] * norm[r][c]);
    }
    wave_lds_sync();
#pragma unroll 2
    for (int c = lane; c < half; c += 64) {  // Rope::apply (src/ops/rope.rs:36-44)
      const float cc = c < 64 ? cs : a.cos[c], ss = c < 64 ? sn : a.sin[c];
#pragma unroll
      for (int r = 0; r < R; r++) {
        float* row = rows + r * pitch;
        const float p = row[c], q = row[half + c];
        row[c] = p * cc - q * ss;
        row[half + c] = q * cc + p * ss;
      }
    }
    wave_lds_sync();
  }
};

// LayerCache::push of key/value head g (src/model/kv_cache.rs): the prepared
// key row and the value projection, by one wave.
__device__ __forceinline__ void push_head(const TokenArgs& a, int g, const float* krow) {
  for (int i = __lane_id(); i < a.hd; i += 64) {
    a.keys[key_piece(a, g, i / 4, a.seq - 1) + i % 4] = krow[i];
    a.values[(size_t)(a.seq - 1) * a.kv_dim + (size_t)g * a.hd + i] = a.v[(size_t)g * a.hd + i];
  }
}

// q . k in index order from -0.0 (Iterator::sum) of one query row and one
// key row in LDS.
__device__ __forceinline__ float dot_rows(const float* q, const float* k, int hd) {
  const f32x4 *q4 = (const f32x4*)q, *k4 = (const f32x4*)k;
  float s = -0.0f;
#pragma unroll 8
  for (int i = 0; i < hd / 4; i++) {
    const f32x4 x = q4[i], y = k4[i];
    s = s + x.x * y.x;
    s = s + x.y * y.y;
    s = s + x.z * y.z;
    s = s + x.w * y.w;
  }
  return s;
}

// The same for the cached key rows of the lanes' positions (clamped by the
// caller) against NQ query rows in LDS, pieces of KEY_CHUNK dimensions in
// two register sets: start() sends the first two for before the query rows
// exist, so that a head of 128 has one round trip.
constexpr int KEY_CHUNK = 64;
template <int NQ>
struct KeyDots {
  f32x4 r[2][KEY_CHUNK / 4];
  const float* base;
  size_t step;  // floats from a piece to the next
  int pieces;
  __device__ __forceinline__ void load(f32x4* d, int chunk) {
#pragma unroll
    for (int i = 0; i < KEY_CHUNK / 4; i++)
      d[i] = *(const f32x4*)(base + (size_t)min(chunk * (KEY_CHUNK / 4) + i, pieces - 1) * step);
  }
  __device__ __forceinline__ void start(const TokenArgs& a, int g, int t) {
    base = a.keys + key_piece(a, g, 0, t);
    step = (size_t)a.cap * 4;
    pieces = a.hd / 4;
    load(r[0], 0);
    load(r[1], 1);
  }
  __device__ __forceinline__ void add(const f32x4* d, int chunk, const float* q, int pitch, float* s) {
#pragma unroll
    for (int j = 0; j < KEY_CHUNK / 16; j++) {
      const int p0 = chunk * (KEY_CHUNK / 4) + 4 * j;
      if (p0 < pieces) {  // uniform; hd is a multiple of 16
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const f32x4 y = d[4 * j + i];
#pragma unroll
          for (int h = 0; h < NQ; h++) {
            const f32x4 x = *(const f32x4*)(q + h * pitch + 4 * (p0 + i));
            s[h] = s[h] + x.x * y.x;
            s[h] = s[h] + x.y * y.y;
            s[h] = s[h] + x.z * y.z;
            s[h] = s[h] + x.w * y.w;
          }
        }
      }
    }
  }
  __device__ __forceinline__ void finish(const float* q, int pitch, float* s) {
#pragma unroll
    for (int h = 0; h < NQ; h++) s[h] = -0.0f;
    const int chunks = (pieces + KEY_CHUNK / 4 - 1) / (KEY_CHUNK / 4);
    for (int c = 0; c < chunks; c += 2) {
      add(r[0], c, q, pitch, s);
      if (c + 2 < chunks) load(r[0], c + 2);
      if (c + 1 < chunks) add(r[1], c + 1, q, pitch, s);
      if (c + 3 < chunks) load(r[1], c + 3);
    }
  }
};

// scores[h][t] = (q_h . key_t) / sqrt(hd) for t < seq.  A work-group takes 64
// positions of one key/value head for up to SC_HEADS query heads of its
// group: lanes are positions, each wave carries SC_WAVE_HEADS heads' chains
// side by side and norms and rotates those heads itself, under its key loads:
// 7.6 us (512 - 3000 positions of four key/value heads) where a launch for
// the norm and one for the scores took 3.7 and 5.0.  The last work-group in
// x does so for the new key too, pushes it and the new value, and scores it.
//
// Bound by latency: launch, key round trip, the chains of two rounded
// operations per dimension.  A wave's keys come through L1, which a
// second head per wave halves.  Position blocks are contiguous per XCD
// (work-group x runs on XCD x % 8): each score row is written in long runs
// per XCD.
constexpr int SC_POS = 64;
constexpr int SC_WAVES = 4;
constexpr int SC_WAVE_HEADS = 2;
constexpr int SC_HEADS = SC_WAVES * SC_WAVE_HEADS;
constexpr int SC_ROWS = SC_WAVE_HEADS + 1;  // LDS rows per wave: its heads, the new key

__global__ __launch_bounds__(64 * SC_WAVES) void k_attn_scores(TokenArgs a, int ld, float scale,
                                                               float* __restrict__ scores) {
  extern __shared__ __attribute__((aligned(16))) float s_heads[];  // SC_WAVES * SC_ROWS rows of hd + 4
  const int g = blockIdx.y;  // key/value head
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int pitch = a.hd + 4;
  // the wave's first head and how many it has (none beyond the group)
  const int first = (int)blockIdx.z * SC_HEADS + wave * SC_WAVE_HEADS;
  const int nq = min(SC_WAVE_HEADS, a.group - first);
  if (nq <= 0) return;
  const int h0 = g * a.group + first;
  float* rows = s_heads + (size_t)wave * SC_ROWS * pitch;
  const int nbx = gridDim.x - 1;  // blocks of cached positions
  if ((int)blockIdx.x == nbx) {
    HeadRows<SC_ROWS> heads;
#pragma unroll
    for (int r = 0; r < SC_WAVE_HEADS; r++) {
      heads.src[r] = a.q + (size_t)(h0 + min(r, nq - 1)) * a.hd;
      heads.norm[r] = a.q_norm;
    }
    heads.src[SC_WAVE_HEADS] = a.k + (size_t)g * a.hd;
    heads.norm[SC_WAVE_HEADS] = a.k_norm;
    heads.load(a);
    heads.store(a, rows);
    const float* krow = rows + SC_WAVE_HEADS * pitch;
    if (first == 0) push_head(a, g, krow);
    if (lane < nq) scores[(size_t)(h0 + lane) * ld + a.seq - 1] = dot_rows(rows + lane * pitch, krow, a.hd) * scale;
    return;
  }
  const int bx = nbx % 8 ? (int)blockIdx.x : (int)(blockIdx.x % 8) * (nbx / 8) + (int)blockIdx.x / 8;
  const int t = bx * SC_POS + lane;
  HeadRows<SC_WAVE_HEADS> heads;
#pragma unroll
  for (int r = 0; r < SC_WAVE_HEADS; r++) {
    heads.src[r] = a.q + (size_t)(h0 + min(r, nq - 1)) * a.hd;
    heads.norm[r] = a.q_norm;
  }
  heads.load(a);
  __builtin_amdgcn_sched_barrier(0);
  KeyDots<SC_WAVE_HEADS> dots;
  dots.start(a, g, min(t, a.seq - 2));
  __builtin_amdgcn_sched_barrier(0);
  heads.store(a, rows);
  float s[SC_WAVE_HEADS];
  dots.finish(rows, pitch, s);
#pragma unroll
  for (int h = 0; h < SC_WAVE_HEADS; h++)
    if (h < nq && t < a.seq - 1) scores[(size_t)(h0 + h) * ld + t] = s[h] * scale;
}

// softmax_in_place over each head's scores (one work-group per head): the
// max in any order, the exponentials in parallel, their sum in order by one
// thread, then one division per score.  The probabilities replace the
// scores.  Up to SM_CHUNK scores stay in LDS from the first read to the
// division, and there the in-order sum (about 10 cycles per dependent add)
// runs in lane 0 of wave 0 while waves 1-3 form the exponentials of the
// next SM_PIPE positions.  Longer rows go through global memory in chunks
// of SM_CHUNK.
constexpr int SM_CHUNK = 12288;  // exponentials per LDS chunk (48 KB)
constexpr int SM_PIPE = 512;     // positions per step of the pipelined sum

__global__ __launch_bounds__(256) void k_attn_softmax(float* __restrict__ scores, int seq, int ld) {
  __shared__ __attribute__((aligned(16))) float buf[SM_CHUNK];
  __shared__ float red[4];
  __shared__ float bcast[1];
  float* sc = scores + (size_t)blockIdx.x * ld;
  const int tid = threadIdx.x;
  // max: fold(-inf, f32::max); order-free (a NaN is skipped either way)
  const bool resident = seq <= SM_CHUNK;
  // 16 loads per thread in flight before they are reduced
  float m = -INFINITY;
  for (int t0 = tid; t0 < seq; t0 += 256 * 16) {
    float v[16];
#pragma unroll
    for (int j = 0; j < 16; j++) {
      const int t = t0 + 256 * j;
      v[j] = t < seq ? sc[t] : -INFINITY;
    }
#pragma unroll
    for (int j = 0; j < 16; j++) {
      const int t = t0 + 256 * j;
      m = fmaxf(m, v[j]);
      if (resident && t < seq) buf[t] = v[j];
    }
  }
  m = wave_max_f32(m);
  if ((tid & 63) == 0) red[tid >> 6] = m;
  __syncthreads();
  m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  if (resident) {
    // step k: waves 1-3 exponentiate block k + 1 while lane 0 adds block k
    const int nblk = (seq + SM_PIPE - 1) / SM_PIPE;
    auto expo = [&](int k) {
      const int e = min(seq, (k + 1) * SM_PIPE);
      for (int t = k * SM_PIPE + tid - 64; t < e; t += 192) buf[t] = hale_expf(buf[t] - m);
    };
    float sum = 0.0f;  // sum += exp(v - max), index order
    if (tid >= 64) expo(0);
    __syncthreads();
    for (int k = 0; k < nblk; k++) {
      if (tid == 0) sum = lds_sum_in_order_a16(buf + k * SM_PIPE, min(SM_PIPE, seq - k * SM_PIPE), sum);
      else if (tid >= 64 && k + 1 < nblk) expo(k + 1);
      __syncthreads();
    }
    if (tid == 0) bcast[0] = sum;
    __syncthreads();
    sum = bcast[0];
    for (int t = tid; t < seq; t += 256) sc[t] = buf[t] / sum;
    return;
  }
  float sum = 0.0f;  // sum += v from 0.0, carried by thread 0
  for (int c0 = 0; c0 < seq; c0 += SM_CHUNK) {
    const int n = min(SM_CHUNK, seq - c0);
    for (int t = tid; t < n; t += 256) {
      const float e = hale_expf(sc[c0 + t] - m);
      sc[c0 + t] = e;
      buf[t] = e;
    }
    __syncthreads();
    if (tid == 0) sum = lds_sum_in_order(buf, n, sum);
    __syncthreads();
  }
  if (tid == 0) bcast[0] = sum;
  __syncthreads();
  sum = bcast[0];
  for (int t = tid; t < seq; t += 256) sc[t] = sc[t] / sum;
}

// The context ctx[h][c] = 0 + p_0 v_0[c] + p_1 v_1[c] + ... in position
// order.  A work-group takes one key/value head, 16 of its columns and up
// to CTX_HEADS query heads of its group; thread (query head, column) of the
// first wave carries one chain.  A dependent f32 add costs about 10 cycles
// on one wave, and one wave issues about one instruction per 6 cycles, so
// the chains only read products and add them: one 16-byte LDS read per 4
// positions from their own row of a product tile [head x 16 + column][T].
// Waves 1-3 fill the product tile of tile i + 1 while the chains add tile
// i.  Their items are 4 columns of one position's values (16 bytes, kept in
// registers) and 4 positions of one head's probabilities (16 bytes), which
// go to a small LDS tile one iteration before the products that use them,
// so the probabilities that the softmax kernel has just written arrive in
// few, wide loads.  NST register stages of items are in flight.
constexpr int CTX_COLS = 16;
constexpr int CTX_HEADS = 2;       // query heads per work-group (32 chains)
constexpr int CTX_T = 256;         // positions per tile
constexpr int CTX_RP = CTX_T + 4;  // row pitch: rows 4 banks apart modulo 64
constexpr int CTX_ITEMS = (CTX_T * CTX_COLS / 4 + 191) / 192;  // value items per loading thread
static_assert(CTX_HEADS * CTX_T / 4 <= 192, "one probability item per loading thread");

__global__ __launch_bounds__(256) void k_attn_ctx(const float* __restrict__ probs,
                                                  const float* __restrict__ values, int hd,
                                                  int kv_dim, int group, int seq, int ld,
                                                  float* __restrict__ ctx) {
  constexpr int T = CTX_T, RP = CTX_RP;
  __shared__ __attribute__((aligned(16))) float prod[2][CTX_HEADS * CTX_COLS * RP];
  __shared__ __attribute__((aligned(16))) float pbuf[2][CTX_HEADS * T];
  const int g = blockIdx.x;               // key/value head
  const int c0 = blockIdx.y * CTX_COLS;   // first column
  const int h0 = blockIdx.z * CTX_HEADS;  // first query head within the group
  const int nh = min(CTX_HEADS, group - h0);
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ntiles = (seq + T - 1) / T;
  auto tile_n = [&](int ti) { return min(T, seq - ti * T); };

  if (wave == 0) {
    // the chains: two barriers before the first tile, then one per tile
    float acc = 0.0f;
    __syncthreads();
    __syncthreads();
    for (int ti = 0; ti < ntiles; ti++) {
      if (tid < nh * CTX_COLS) acc = lds_sum_in_order_a16(&prod[ti & 1][tid * RP], tile_n(ti), acc);
      __syncthreads();
    }
    if (tid < nh * CTX_COLS)
      ctx[(size_t)(g * group + h0 + tid / CTX_COLS) * hd + c0 + tid % CTX_COLS] = acc;
    return;
  }

  // waves 1-3: value item i = lt + 192 j of a tile is position i / 4,
  // columns 4q .. 4q + 3 with q = i % 4; probability item lt is head
  // lt / (T / 4), positions 4 (lt % (T / 4)) .. + 3
  constexpr int NLOAD = 192;
  const int lt = tid - 64;
  const float* vbase = values + (size_t)g * hd + c0;
  const float* pbase = probs + ((size_t)g * group + h0) * ld;
  const bool pitem = lt < nh * (T / 4);
  const int ph = lt / (T / 4), pt = 4 * (lt % (T / 4));
  struct Stage {
    f32x4 v[CTX_ITEMS];
    f32x4 p;
  };
  constexpr int NST = 4;
  Stage r[NST];
  auto load = [&](Stage& R, int ti) {
    if (ti >= ntiles) return;
    const int t0 = ti * T, n = tile_n(ti);
    const float* vb = vbase + (size_t)t0 * kv_dim;
#pragma unroll
    for (int j = 0; j < CTX_ITEMS; j++) {
      const int i = lt + NLOAD * j, t = i / 4, q = i % 4;
      if (i < T * 4 && t < n) R.v[j] = *(const f32x4*)(vb + (size_t)t * kv_dim + 4 * q);
    }
    // reads up to 3 past n stay inside the row: ld is a multiple of 4
    if (pitem && pt < n) R.p = *(const f32x4*)(pbase + (size_t)ph * ld + t0 + pt);
  };
  auto store_p = [&](const Stage& R, int b) {
    if (pitem) *(f32x4*)&pbuf[b][ph * T + pt] = R.p;
  };
  // products of the items into product buffer b (positions past the tile's
  // end are not written; the chains never read them)
  auto multiply = [&](const Stage& R, int b, int n) {
#pragma unroll
    for (int j = 0; j < CTX_ITEMS; j++) {
      const int i = lt + NLOAD * j, t = i / 4, q = i % 4;
      if (i < T * 4 && t < n) {
#pragma unroll
        for (int hh = 0; hh < CTX_HEADS; hh++) {
          if (hh < nh) {
            const float p = pbuf[b][hh * T + t];
            float* d = &prod[b][(hh * CTX_COLS + 4 * q) * RP + t];
            d[0] = p * R.v[j].x;
            d[RP] = p * R.v[j].y;
            d[2 * RP] = p * R.v[j].z;
            d[3 * RP] = p * R.v[j].w;
          }
        }
      }
    }
  };
  // Stage s holds the tiles ti with ti % NST == s.  Tile ti's probabilities
  // go to LDS at iteration ti - 2, its products form at iteration ti - 1,
  // and its stage is refilled at iteration ti (each step a barrier after
  // the previous one, so no load waits for a store of the same registers).
#pragma unroll
  for (int j = 0; j < NST; j++) load(r[j], j);
  if (ntiles > 0) store_p(r[0], 0);
  __syncthreads();
  if (ntiles > 0) multiply(r[0], 0, tile_n(0));
  if (ntiles > 1) store_p(r[1], 1);
  __syncthreads();
  for (int ti0 = 0; ti0 < ntiles; ti0 += NST) {
#pragma unroll
    for (int j = 0; j < NST; j++) {
      const int ti = ti0 + j;  // the chains add tile ti
      if (ti < ntiles) {
        if (ti + 1 < ntiles) multiply(r[(j + 1) % NST], (ti + 1) & 1, tile_n(ti + 1));
        if (ti + 2 < ntiles) store_p(r[(j + 2) % NST], ti & 1);
        load(r[j], ti + NST);
        __syncthreads();
      }
    }
  }
}

// softmax_in_place and the context in one kernel, for score rows up to
// SMC_MAX positions: a work-group takes one query head and SMC_COLS of its
// columns.  All waves form the head's exp values in LDS, four of them sum
// those in order (ordered_sum.h: K consecutive values per lane), and all
// divide; then wave 0's lanes carry the context chains, one column each,
// while waves 1-7 form the products p_t v_t[c] two tiles ahead.
//
// Bound by the context chains: one dependent add (2.6 ns) and a quarter of a
// 16-byte LDS read per position.  The order below takes 3.2 ns: batches of
// 32 positions with one wait each, the next batch's reads in pairs of
// additions early in the batch (a read and a wait before every four
// additions: 3.7 ns), running on over tile borders (a tile's products are
// complete one barrier before its first read, so the reads need not start
// anew: 1.2 us per 256 positions otherwise).  The sum was a second such
// chain before them (4.1 ns per position).  32 heads of 128 over four
// key/value heads, mean of the lengths up to 3000: 23.4 us with two chains
// (16 columns of two heads per work-group), 13.7 us so; up to 190: 7.0 and
// 5.7 us.  32 columns of one head: each work-group forms half as many exp
// values, and a value row is one 128-byte line.  A head's work-groups repeat
// its softmax, which no launch boundary then separates from the products.
// The heads of a group read the same value lines, so grid x is the key/value
// head and its columns: a multiple of 8 of them keeps a line on one XCD.
constexpr int SMC_MAX = ORDERED_MAX;
constexpr int SMC_COLS = 32;
constexpr int SMC_THREADS = 512;
constexpr int SMC_T = 128;         // positions per tile, a multiple of 64
constexpr int SMC_RP = SMC_T + 4;  // row pitch of a product tile: rows 4 banks apart
constexpr int SMC_LOADERS = SMC_THREADS - 64;  // product threads: waves 1-7
constexpr int SMC_ITEMS = (SMC_T * SMC_COLS / 4 + SMC_LOADERS - 1) / SMC_LOADERS;  // per product thread
// exp values in LDS: 4 floats of padding every 32, as in k_rms_norm
__device__ __host__ constexpr int exp_at(int t) { return t + (t >> 5) * 4; }

// SHORT: the same work-group prepares its head and the new key and scores the
// head itself, one or two positions per thread, so that a token's attention is
// one launch.  The new position's key and value come from the projections: the
// first work-group of a key/value head pushes them to the cache meanwhile.
// Against it stand the scores, formed once per column block: the longer the
// row and the larger the head, the more keys each work-group reads through L1.
// Its registers admit one work-group per CU, so beyond 256 of them it runs in
// turns.  Hence at most SHORT_GROUPS work-groups, and rows up to 512; to 768
// where a norm, which the score launch would do in front of its keys, lengthens
// the other way, and the head has at most SHORT_HEAD values.  A token's whole
// call, one launch / two, us: 32 heads of 128, QK-norm, four key/value heads,
// 190 / 440 / 520 / 760 / 900 positions 19.4 / 21.8 / 23.1 / 25.4 / 26.5 and
// 23.2 / 24.6 / 25.1 / 26.1 / 26.6; without the norm 19.1 / 21.6 / 22.9 / 25.1 /
// 26.1 and 20.9 / 22.4 / 22.9 / 24.0 / 24.5; 64 heads (256 work-groups) 520
// positions 29.2 / 30.9; 96 heads (384) 190 positions 39.2 / 35.7; 16 heads of
// 256, 440 / 520 positions 27.9 / 30.0 and 28.5 / 29.1; 16 heads of 512, 190 /
// 520 positions 36.9 / 50.5 and 41.8 / 44.3.
constexpr int SHORT_MAX = 768;
constexpr int SHORT_HEAD = 128;
constexpr unsigned SHORT_GROUPS = 256;
template <int K, bool SHORT>  // 256 K >= seq
__global__ __launch_bounds__(SMC_THREADS) void k_attn_softmax_ctx(TokenArgs a, const float* __restrict__ scores,
                                                                  int ld, float scale, float* __restrict__ ctx) {
  constexpr int T = SMC_T, RP = SMC_RP, NBUF = 3;
  __shared__ __attribute__((aligned(16))) float ebuf[exp_at(256 * K)];
  __shared__ __attribute__((aligned(16))) float prod[NBUF][SMC_COLS * RP];
  __shared__ float red[SMC_THREADS / 64];
  __shared__ float part[ordered_lds(4)];
  __shared__ __attribute__((aligned(16))) float s_qk[SHORT ? 2 * (HEAD_MAX + 4) : 4];
  const int hd = a.hd, kv_dim = a.kv_dim, seq = a.seq;
  const int blocks = (hd + SMC_COLS - 1) / SMC_COLS;  // column blocks of a head
  const int g = blockIdx.x / blocks;                  // key/value head
  const int c0 = blockIdx.x % blocks * SMC_COLS;      // first column
  const int ncols = min(SMC_COLS, hd - c0);           // a multiple of 16
  const int h = g * a.group + blockIdx.y;             // query head
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int ntiles = (seq + T - 1) / T;

  // value items of the product threads: item i of a tile is position i / 8, columns
  // 4q .. 4q + 3 with q = i % 8; the first NST tiles go out before the softmax
  // (every load unconditional, clamped to the last position and column: under
  // a branch each one would wait for the load before it)
  constexpr int NLOAD = SMC_LOADERS;
  const int lt = max(tid - 64, 0);  // wave 0 repeats the first item's loads
  const float* vbase = a.values + (size_t)g * hd + c0;
  const float* vnew = a.v + (size_t)g * hd + c0;
  constexpr int NST = 4;
  f32x4 r[NST][SMC_ITEMS];
  auto load = [&](f32x4* R, int ti) {
#pragma unroll
    for (int j = 0; j < SMC_ITEMS; j++) {
      const int i = lt + NLOAD * j, t = min(ti * T + i / 8, seq - 1), c = min(4 * (i % 8), ncols - 4);
      const float* row = SHORT && t == seq - 1 ? vnew : vbase + (size_t)t * kv_dim;
      R[j] = *(const f32x4*)(row + c);
    }
  };
  // the head's scores, then its values: loads return in order
  constexpr int SPT = (256 * K + SMC_THREADS - 1) / SMC_THREADS;
  float sc[SPT];
  if constexpr (SHORT) {
    const int pitch = hd + 4;
    HeadRows<1> head;  // wave 0: the query head, wave 1: the new key
    head.src[0] = wave == 1 ? a.k + (size_t)g * hd : a.q + (size_t)h * hd;
    head.norm[0] = wave == 1 ? a.k_norm : a.q_norm;
    head.load(a);
    __builtin_amdgcn_sched_barrier(0);
    KeyDots<1> dots;
    dots.start(a, g, max(min(tid, seq - 2), 0));
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < NST; j++) load(r[j], j);
    __builtin_amdgcn_sched_barrier(0);
    if (wave < 2) head.store(a, s_qk + wave * pitch);
    __syncthreads();
    if (c0 == 0 && blockIdx.y == 0 && wave == 6) push_head(a, g, s_qk + pitch);
#pragma unroll
    for (int j = 0; j < SPT; j++) {
      sc[j] = 0.0f;
      if (SMC_THREADS * j + wave * 64 < seq - 1) {
        if (j) dots.start(a, g, min(tid + SMC_THREADS * j, seq - 2));
        dots.finish(s_qk, pitch, &sc[j]);
      }
    }
    // the new position, the row's last: by a lane of the last wave, whose
    // own positions few rows reach
    if (tid == SMC_THREADS - 1) red[0] = dot_rows(s_qk, s_qk + pitch, hd);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < SPT; j++) {
      const int t = tid + SMC_THREADS * j;
      if (t == seq - 1) sc[j] = red[0];
      sc[j] = t < seq ? sc[j] * scale : -INFINITY;
    }
    __syncthreads();
  } else {
    const float* srow = scores + (size_t)h * ld;
#pragma unroll
    for (int j = 0; j < SPT; j++) {
      const int t = tid + SMC_THREADS * j;
      sc[j] = t < seq ? srow[t] : -INFINITY;
    }
#pragma unroll
    for (int j = 0; j < NST; j++) load(r[j], j);
  }

  // max: fold(-inf, f32::max); order-free (a NaN is skipped either way)
  float m = -INFINITY;
#pragma unroll
  for (int j = 0; j < SPT; j++) m = fmaxf(m, sc[j]);
  m = wave_max_f32(m);
  if (lane == 0) red[wave] = m;
  ExpTable tab;
  tab.load();
  __syncthreads();
  m = red[0];
#pragma unroll
  for (int i = 1; i < SMC_THREADS / 64; i++) m = fmaxf(m, red[i]);
#pragma unroll
  for (int j = 0; j < SPT; j++) {
    const int t = tid + SMC_THREADS * j;
    sc[j] = wave_expf(sc[j] - m, tab);  // every lane takes part
    if (t >= seq) sc[j] = 0.0f;
    if (t < 256 * K) ebuf[exp_at(t)] = sc[j];
  }
  __syncthreads();
  float v[K];
#pragma unroll
  for (int k = 0; k < K; k++) v[k] = ebuf[exp_at((tid & 255) * K + k)];
  const float sum = team_sum_in_order<K>(v, 0.0f, wave, (seq + 64 * K - 1) / (64 * K), part);
#pragma unroll
  for (int j = 0; j < SPT; j++) {
    const int t = tid + SMC_THREADS * j;
    if (t < seq) ebuf[exp_at(t)] = sc[j] / sum;
  }
  __syncthreads();

  if (wave == 0) {
    // two barriers before the first tile (tiles 0 and 1 are formed), then
    // one per tile.  Positions past the end carry +0 products: acc starts at
    // +0 and so is never the -0 that they would change.
    const f32x4* col = (const f32x4*)&prod[0][(lane & (SMC_COLS - 1)) * RP];  // lanes 32-63 repeat
    constexpr int BUF = SMC_COLS * RP / 4;
    f32x4 A[8], B[8];
    float acc = 0.0f;
    auto batch = [&](const f32x4* X, f32x4* Y, const f32x4* next) {
      asm volatile("" ::"v"(X[7].w));  // the batch's one wait
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int q = 0; q < 8; q++) {
        if (q < 4) Y[2 * q] = next[2 * q];
        __builtin_amdgcn_sched_barrier(0);
        acc = acc + X[q].x;
        acc = acc + X[q].y;
        __builtin_amdgcn_sched_barrier(0);
        if (q < 4) Y[2 * q + 1] = next[2 * q + 1];
        __builtin_amdgcn_sched_barrier(0);
        acc = acc + X[q].z;
        acc = acc + X[q].w;
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 8; q++) A[q] = col[q];
    int buf = 0;
    __syncthreads();
    for (int ti = 0; ti < ntiles; ti++) {
      const f32x4* p = col + buf * BUF;
      buf = buf + 1 == NBUF ? 0 : buf + 1;
      const f32x4* after = col + buf * BUF;  // the next tile's first batch (stale after the last tile)
      const int nb = (min(T, seq - ti * T) + 63) / 64;
      for (int i = 0; i < nb; i++) {
        batch(A, B, p + 8);
        p += 16;
        batch(B, A, i + 1 < nb ? p : after);
      }
      __syncthreads();
    }
    if (lane < ncols) ctx[(size_t)h * hd + c0 + lane] = acc;
    return;
  }
  auto multiply = [&](const f32x4* R, int ti) {
    const int t0 = ti * T, n = min(T, seq - t0), n64 = (n + 63) & ~63;
    float* P = prod[ti % NBUF];
#pragma unroll
    for (int j = 0; j < SMC_ITEMS; j++) {
      const int i = lt + NLOAD * j, t = i / 8, q = i % 8;
      const bool in = t < n;
      const float pr = ebuf[exp_at(min(t0 + t, seq - 1))];
      if (t < n64 && 4 * q < ncols) {
        float* d = P + 4 * q * RP + t;
        d[0] = in ? pr * R[j].x : 0.0f;
        d[RP] = in ? pr * R[j].y : 0.0f;
        d[2 * RP] = in ? pr * R[j].z : 0.0f;
        d[3 * RP] = in ? pr * R[j].w : 0.0f;
      }
    }
  };
  // stage s holds the tiles ti with ti % NST == s
  multiply(r[0], 0);
  load(r[0], NST);
  __syncthreads();
  if (ntiles > 1) multiply(r[1], 1);
  load(r[1], NST + 1);
  __syncthreads();
  for (int ti0 = 0; ti0 < ntiles; ti0 += NST) {
#pragma unroll
    for (int j = 0; j < NST; j++) {
      const int ti = ti0 + j;  // the chains add tile ti
      if (ti < ntiles) {
        if (ti + 2 < ntiles) multiply(r[(j + 2) % NST], ti + 2);
        load(r[(j + 2) % NST], ti + 2 + NST);  // its products are formed
        __syncthreads();
      }
    }
  }
}

hipError_t launch_rms_norm(float* x, const float* delta, const float* w, size_t rows, size_t n,
                           float eps, float* out, hipStream_t st) {
  if (rows == 0) return hipSuccess;
  if (n == 0 || n > (size_t)NORM_MAX || rows > 0x7fffffffu) return hipErrorInvalidValue;
  auto run = [&](auto kernel, unsigned nt) { return launch(kernel, (unsigned)rows, nt, 0, st, x, delta, w, (int)n, eps, out); };
  if (n <= 1024) return run(k_rms_norm<4, 256>, 256);
  if (n <= 2048) return run(k_rms_norm<8, 256>, 256);
  if (n <= 4096) return run(k_rms_norm<8, 512>, 512);
  return run(k_rms_norm<16, 512>, 512);
}

hipError_t launch_attention_core(const AttnArgs& a, hipStream_t st) {
  // head_dim a multiple of 16 (context column blocks, key chunks), GQA group
  // <= 16, score rows 16-byte aligned
  if (a.hd < 16 || a.hd > HEAD_MAX || a.hd % CTX_COLS || a.nh < 1 || a.nkv < 1 || a.nh % a.nkv ||
      a.nh / a.nkv > 16 || a.seq < 1 || a.seq > a.cap || a.cap > a.ld || a.ld % 4)
    return hipErrorInvalidValue;
  const int kv_dim = a.nkv * a.hd, group = a.nh / a.nkv;
  const float scale = 1.0f / sqrtf((float)a.hd);
  const TokenArgs t{a.q, a.k, a.v, a.q_norm, a.k_norm, a.cos, a.sin, a.eps, a.keys, a.values,
                    a.hd, kv_dim, group, a.cap, a.seq};
  const dim3 gsc((unsigned)(a.nkv * ((a.hd + SMC_COLS - 1) / SMC_COLS)), (unsigned)group);
  auto softmax_ctx = [&](auto kernel) {
    return launch(kernel, gsc, SMC_THREADS, 0, st, t, (const float*)a.scores, a.ld, scale, a.ctx);
  };
  const bool normed = a.q_norm || a.k_norm;
  if (gsc.x * gsc.y <= SHORT_GROUPS && a.seq <= (normed && a.hd <= SHORT_HEAD ? SHORT_MAX : 512)) {
    if (a.seq <= 512) return softmax_ctx(k_attn_softmax_ctx<2, true>);
    return softmax_ctx(k_attn_softmax_ctx<4, true>);
  }
  const dim3 gs((unsigned)((a.seq - 1 + SC_POS - 1) / SC_POS + 1), (unsigned)a.nkv,
                (unsigned)((group + SC_HEADS - 1) / SC_HEADS));
  hipError_t e = launch(k_attn_scores, gs, 64 * SC_WAVES, (uint32_t)(SC_WAVES * SC_ROWS * (a.hd + 4) * sizeof(float)), st,
                        t, a.ld, scale, a.scores);
  if (e != hipSuccess) return e;
  if (a.seq <= 2048) return softmax_ctx(k_attn_softmax_ctx<8, false>);
  if (a.seq <= 4096) return softmax_ctx(k_attn_softmax_ctx<16, false>);
  if (a.seq <= SMC_MAX) return softmax_ctx(k_attn_softmax_ctx<32, false>);
  e = launch(k_attn_softmax, (unsigned)a.nh, 256, 0, st, a.scores, a.seq, a.ld);
  if (e != hipSuccess) return e;
  const dim3 gc((unsigned)a.nkv, (unsigned)(a.hd / CTX_COLS), (unsigned)((group + CTX_HEADS - 1) / CTX_HEADS));
  return launch(k_attn_ctx, gc, 256, 0, st, (const float*)a.scores, (const float*)a.values, a.hd, kv_dim, group, a.seq,
                a.ld, a.ctx);
}

}  // namespace hale
