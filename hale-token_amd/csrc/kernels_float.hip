// kernels_float.hip -- matvec over float weights (f32, f16, bf16) on gfx950.
//
// The reference's float dot (src/tensor/quant.rs:146-233) keeps eight lane
// accumulators: acc[l] = acc[l] + w[8i+l] * x[8i+l] for i = 0, 1, ...
// (products rounded, then added; no fused multiply-add), then
//   ((acc0 + acc4) + (acc1 + acc5)) + ((acc2 + acc6) + (acc3 + acc7))
// (reduce, :36-40) plus the sum of the last cols % 8 products.  f32 rows
// add that tail as Iterator::sum (from -0.0, dot_f32 :186-194); f16 and
// bf16 rows go through dot_decoded (:166-184), whose tail starts at +0.0.
// Each of a row's 8 chains is one sequential sum, so one lane per chain
// folds it; the products are computed in parallel.
//
// Work-group: 8 rows, 256 threads.  Per chunk of FK columns every thread
// loads 16-byte pieces of the rows (coalesced along each row) and its x,
// converts f16/bf16 to f32, and parks the products in LDS; wave 0 then folds
// them, lane (row r, chain l) reading products 8i + l of row r in order.
// Two LDS buffers; the loads of up to NS chunks are in flight during a fold.
// HBM-bound for many rows (151,936 x 2048 bf16: 102-103 us with one chunk in
// flight, 97.6 us with four: 6.4 TB/s); few rows wait for the round trip and
// wave 0's fold (5120 x 2048 bf16 8.1 -> 7.4 us).
#pragma clang fp contract(off)

#include "hale_device.h"
#include "kernels.h"

namespace hale {

constexpr int FR = 8;        // rows per work-group (FR * 8 fold threads, whole waves)
constexpr int FK = 512;      // columns per chunk
constexpr int FPAD = 8;      // row pitch FK + FPAD = 8 (mod 64) floats: the fold
                             // threads (row r, chain l) of a wave read banks 8r + l

template <int DT>
struct FloatFmt;
template <> struct FloatFmt<F32> { static constexpr int PER16 = 4; };   // values per 16 B
template <> struct FloatFmt<F16> { static constexpr int PER16 = 8; };
template <> struct FloatFmt<BF16> { static constexpr int PER16 = 8; };

template <int DT>
__device__ __forceinline__ void unpack16(const u32x4& v, float* o) {
  if constexpr (DT == F32) {
    o[0] = __uint_as_float(v.x);
    o[1] = __uint_as_float(v.y);
    o[2] = __uint_as_float(v.z);
    o[3] = __uint_as_float(v.w);
  } else {
    const unsigned u[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; i++) {
      if constexpr (DT == F16) {
        o[2 * i] = h2f((uint16_t)(u[i] & 0xffffu));
        o[2 * i + 1] = h2f((uint16_t)(u[i] >> 16));
      } else {  // bf16 is the upper half of an f32
        o[2 * i] = __uint_as_float(u[i] << 16);
        o[2 * i + 1] = __uint_as_float(u[i] & 0xffff0000u);
      }
    }
  }
}

// The matrices of one launch (all cols long): work-groups first[i] ..
// first[i + 1] - 1 take matrix i.
struct FloatMats {
  const uint8_t* w[MATVEC_MANY];
  float* out[MATVEC_MANY];
  int rows[MATVEC_MANY], first[MATVEC_MANY];
  __device__ __forceinline__ int of(int group) const {
    int i = 0;
#pragma unroll
    for (int j = 1; j < MATVEC_MANY; j++) i = group >= first[j] ? j : i;
    return i;
  }
};

// VEC: every row starts 16-byte aligned, so a piece is one 16-byte load;
// otherwise it is read value by value.  MANY: several matrices; one alone
// skips the choice (2 % of a 151,936 x 2048 projection's time).  NS: chunks
// in flight (float_ring).
template <int DT, bool VEC, bool MANY, int NS>
__global__ __launch_bounds__(256) void k_gemv_float(FloatMats m, const float* __restrict__ x,
                                                    int cols) {
  constexpr int PER = FloatFmt<DT>::PER16;
  constexpr int ESZ = DT == F32 ? 4 : 2;
  constexpr int UPR = FK / PER;          // 16-byte pieces per row of a chunk
  constexpr int LPT = FR * UPR / 256;    // pieces per thread per chunk
  constexpr int RPP = 256 / UPR;         // rows one pass of the 256 threads covers
  static_assert(LPT * 256 == FR * UPR && LPT * RPP == FR, "chunk tiling");
  static_assert(FR % 8 == 0 && FR * 8 <= 256, "fold threads fill whole waves");
  __shared__ __attribute__((aligned(16))) float prod[2][FR][FK + FPAD];

  const int tid = threadIdx.x;
  const int mi = MANY ? m.of((int)blockIdx.x) : 0;
  const uint8_t* __restrict__ w = m.w[mi];
  float* __restrict__ out = m.out[mi];
  const int rows = m.rows[mi];
  const int row0 = ((int)blockIdx.x - m.first[mi]) * FR;
  const int done = cols / 8 * 8;         // columns covered by the lane accumulators
  const int nchunks = (done + FK - 1) / FK;
  const size_t rb = (size_t)cols * ESZ;  // row bytes

  // piece j of this thread: row r_j, columns c .. c + PER - 1 of the chunk
  const int cpiece = (tid % UPR) * PER;
  struct Regs {
    u32x4 w[LPT];
    float x[PER];
  };
  auto load = [&](Regs& R, int ch) {
    // `done` is a multiple of 8 and PER 4 or 8, so a piece below `done` ends
    // at or before it; rows past the matrix's end are clamped (loaded, never
    // written).  With several chunks in flight pieces past the row's end repeat
    // the last one: every load is then unconditional, where under a branch
    // each would wait for the one before.
    const int cp = ch * FK + cpiece;
    if (NS == 1 && cp >= done) return;
    const int c = NS == 1 ? cp : min(cp, done - PER);
#pragma unroll
    for (int j = 0; j < LPT; j++) {
      const int r = min(row0 + j * RPP + tid / UPR, rows - 1);
      const uint8_t* src = w + (size_t)r * rb + (size_t)c * ESZ;
      if constexpr (VEC) {
        R.w[j] = __builtin_nontemporal_load((const u32x4*)src);
      } else if constexpr (DT == F32) {
        const unsigned* s4 = (const unsigned*)src;
        R.w[j] = u32x4{s4[0], s4[1], s4[2], s4[3]};
      } else {
        const uint16_t* s2 = (const uint16_t*)src;
        R.w[j] = u32x4{s2[0] | ((unsigned)s2[1] << 16), s2[2] | ((unsigned)s2[3] << 16),
                       s2[4] | ((unsigned)s2[5] << 16), s2[6] | ((unsigned)s2[7] << 16)};
      }
    }
#pragma unroll
    for (int q = 0; q < PER / 4; q++) {
      const f32x4 v = *(const f32x4*)(x + c + 4 * q);
      R.x[4 * q] = v.x;
      R.x[4 * q + 1] = v.y;
      R.x[4 * q + 2] = v.z;
      R.x[4 * q + 3] = v.w;
    }
  };

  // fold thread (row fr, chain fl): the first FR * 8 threads
  constexpr int NF = FR * 8;
  const int fr = tid >> 3, fl = tid & 7;
  float acc = 0.0f;
  // chunk ch from R, which then takes chunk `next` (none: negative)
  auto step = [&](Regs& R, int ch, int next) {
    const int c0 = ch * FK;
    const int ncols = min(FK, done - c0);
    float(*P)[FK + FPAD] = prod[ch & 1];
    if (cpiece < ncols) {
#pragma unroll
      for (int j = 0; j < LPT; j++) {
        float wf[PER];
        unpack16<DT>(R.w[j], wf);
        float* dst = &P[j * RPP + tid / UPR][cpiece];
#pragma unroll
        for (int q = 0; q < PER; q++) dst[q] = wf[q] * R.x[q];  // the rounded product
      }
    }
    __syncthreads();
    if (next >= 0) load(R, next);
    if (tid < NF) acc = lds_sum_strided<8>(&P[fr][fl], ncols / 8, acc);
  };
  // NS chunks in flight (the launcher's rows have as many): one round trip
  // for a bf16 row of 2048 instead of four
  Regs R[NS];
  int ch = 0;
  if constexpr (NS > 1) {
#pragma unroll
    for (int j = 0; j < NS; j++) {
      load(R[j], j);
      __builtin_amdgcn_sched_barrier(0);
    }
    for (; ch + 2 * NS <= nchunks; ch += NS)
#pragma unroll
      for (int j = 0; j < NS; j++) step(R[j], ch + j, ch + NS + j);
#pragma unroll
    for (int j = 0; j < NS; j++) step(R[j], ch + j, ch + NS + j < nchunks ? ch + NS + j : -1);
    ch += NS;
#pragma unroll
    for (int j = 0; j < NS; j++)
      if (ch + j < nchunks) step(R[j], ch + j, -1);
  } else if (nchunks > 0) {
    load(R[0], 0);
    for (; ch < nchunks; ch++) step(R[0], ch, ch + 1 < nchunks ? ch + 1 : -1);
  }

  if (tid < NF) {
    // reduce (src/tensor/quant.rs:36-40) across the row's 8 chain lanes
    const float a4 = __shfl_down(acc, 4, 8);
    const float s = acc + a4;                    // lanes 0-3: acc_l + acc_{l+4}
    const float s1 = __shfl_down(s, 1, 8);
    const float t = s + s1;                      // lanes 0, 2: pair sums
    const float t2 = __shfl_down(t, 2, 8);
    const float red = t + t2;                    // lane 0: (s0 + s1) + (s2 + s3)
    const int row = row0 + fr;
    if (fl == 0 && row < rows) {
      // the last cols % 8 products, summed in order
      float tail = -0.0f;
      const uint8_t* wr = w + (size_t)row * rb;
      for (int i = done; i < cols; i++) {
        float wi;
        if constexpr (DT == F32) {
          wi = ((const float*)wr)[i];
        } else if constexpr (DT == F16) {
          wi = h2f(((const uint16_t*)wr)[i]);
        } else {
          wi = __uint_as_float((unsigned)((const uint16_t*)wr)[i] << 16);
        }
        tail = tail + wi * x[i];
      }
      if constexpr (DT != F32) tail = 0.0f + tail;  // dot_decoded's `let mut tail = 0.0`
      out[row] = red + tail;
    }
  }
}

// encode_row for the half formats (src/tensor/quant.rs:274-292): half's
// f16::from_f32 / bf16::from_f32, round to nearest even; a NaN keeps its
// sign and top payload bits and becomes quiet.
template <int DT>
__device__ __forceinline__ uint16_t encode_half(float f) {
  const unsigned x = __float_as_uint(f);
  const bool nan = (x & 0x7fffffffu) > 0x7f800000u;
  if constexpr (DT == F16) {
    if (nan) return (uint16_t)(((x >> 16) & 0x8000u) | 0x7e00u | ((x & 0x7fffffu) >> 13));
    return f2h(f);  // v_cvt_f16_f32: round to nearest even, subnormals kept
  } else {
    if (nan) return (uint16_t)((x >> 16) | 0x0040u);
    unsigned q = x >> 16;
    const unsigned rem = x & 0xffffu;
    if (rem > 0x8000u || (rem == 0x8000u && (q & 1u))) q++;  // may carry into inf
    return (uint16_t)q;
  }
}

// One value per thread: any alignment, and the last n % 4.
template <int DT>
__global__ __launch_bounds__(256) void k_encode_half(const float* __restrict__ v, size_t n,
                                                     uint16_t* __restrict__ out) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) out[i] = encode_half<DT>(v[i]);
}

// Four values per thread and step (values 16-byte, out 8-byte aligned),
// HALF_U steps in flight.
constexpr int HALF_U = 4;
template <int DT>
__global__ __launch_bounds__(256) void k_encode_half4(const float* __restrict__ v, size_t pieces,
                                                      uint16_t* __restrict__ out) {
  const size_t p0 = (size_t)blockIdx.x * (256 * HALF_U) + threadIdx.x;
  f32x4 x[HALF_U];
#pragma unroll
  for (int u = 0; u < HALF_U; u++) x[u] = ((const f32x4*)v)[p0 + 256 * u < pieces ? p0 + 256 * u : pieces - 1];
#pragma unroll
  for (int u = 0; u < HALF_U; u++) {
    const size_t p = p0 + 256 * u;
    if (p >= pieces) break;
    uint64_t w = 0;
#pragma unroll
    for (int j = 0; j < 4; j++) w |= (uint64_t)encode_half<DT>(x[u][j]) << 16 * j;
    ((uint64_t*)out)[p] = w;
  }
}

hipError_t launch_encode_half(int dtype, const float* values, size_t n, void* out, hipStream_t st) {
  if (n == 0) return hipSuccess;
  if (dtype != F16 && dtype != BF16) return hipErrorInvalidValue;
  uint16_t* o = (uint16_t*)out;
  if (n >= 4 && (uintptr_t)values % 16 == 0 && (uintptr_t)out % 8 == 0) {
    const size_t pieces = n / 4;
    const unsigned grid = (unsigned)((pieces + 256 * HALF_U - 1) / (256 * HALF_U));
    const hipError_t e = dtype == F16 ? launch(k_encode_half4<F16>, grid, 256, 0, st, values, pieces, o)
                                      : launch(k_encode_half4<BF16>, grid, 256, 0, st, values, pieces, o);
    if (e != hipSuccess || n % 4 == 0) return e;
    values += 4 * pieces;
    o += 4 * pieces;
    n %= 4;
  }
  const unsigned grid = (unsigned)((n + 255) / 256);
  return dtype == F16 ? launch(k_encode_half<F16>, grid, 256, 0, st, values, n, o)
                      : launch(k_encode_half<BF16>, grid, 256, 0, st, values, n, o);
}

// Chunks in flight.  Several where waits for the round trip show: with fewer
// than two work-groups per CU (cold, one chunk / several: bf16 512 x 2048 5.1 /
// 4.8 us, 2048 x 4096 8.7 / 8.1, 3000 x 14336 28.9 / 25.8, f32 2048 x 2048 6.8 /
// 6.1), and for half rows of exactly four chunks, which one pass of straight
// code covers (5120 x 2048 8.1 / 7.4, 151,936 x 2048 102 / 97.6).  With more
// work-groups they cover for each other, and the longer code and its registers
// cost (bf16 4096 x 4096 10.1 / 10.7, f32 40,000 x 1500 40.4 / 42.0).
static int float_ring(int dtype, size_t cols, size_t groups) {
  const size_t nchunks = (cols / 8 * 8 + FK - 1) / FK;
  const int ns = dtype == F32 ? 2 : 4;
  if (nchunks < (size_t)ns) return 1;
  return groups < 512 || (dtype != F32 && nchunks == 4) ? ns : 1;
}

hipError_t launch_gemv_float(int dtype, const void* w, const float* x, size_t rows, size_t cols,
                             float* out, hipStream_t st) {
  return launch_gemv_float_many(dtype, 1, &w, x, &rows, cols, &out, st);
}

hipError_t launch_gemv_float_many(int dtype, int n, const void* const* w, const float* x, const size_t* rows,
                                  size_t cols, float* const* out, hipStream_t st) {
  if (n < 1 || n > MATVEC_MANY || cols > (size_t)INT32_MAX - FK) return hipErrorInvalidValue;
  if ((uintptr_t)x % 16) return hipErrorInvalidValue;  // x is read in 16-byte pieces
  const int esz = dtype == F32 ? 4 : 2;
  bool vec = (cols * esz) % 16 == 0;
  FloatMats m{};
  size_t groups = 0;
  for (int i = 0; i < MATVEC_MANY; i++) {
    m.first[i] = i < n ? (int)groups : INT32_MAX;
    if (i >= n) continue;
    if (rows[i] > (size_t)INT32_MAX - FR) return hipErrorInvalidValue;
    m.w[i] = (const uint8_t*)w[i];
    m.out[i] = out[i];
    m.rows[i] = (int)rows[i];
    vec = vec && (uintptr_t)w[i] % 16 == 0;
    groups += (rows[i] + FR - 1) / FR;
    if (groups > (size_t)INT32_MAX) return hipErrorInvalidValue;
  }
  if (groups == 0) return hipSuccess;
  auto run = [&](auto kernel) { return launch(kernel, (unsigned)groups, 256, 0, st, m, x, (int)cols); };
  const bool ring = float_ring(dtype, cols, groups) > 1;
#define HALE_FLOAT_RING(D, V, M) (ring ? run(k_gemv_float<D, V, M, D == F32 ? 2 : 4>) : run(k_gemv_float<D, V, M, 1>))
#define HALE_FLOAT_CASE(D)                                                                      \
  if (dtype == D)                                                                               \
    return vec ? (n > 1 ? HALE_FLOAT_RING(D, true, true) : HALE_FLOAT_RING(D, true, false))     \
               : (n > 1 ? HALE_FLOAT_RING(D, false, true) : HALE_FLOAT_RING(D, false, false));
  HALE_FLOAT_CASE(F32)
  HALE_FLOAT_CASE(F16)
  HALE_FLOAT_CASE(BF16)
#undef HALE_FLOAT_RING
#undef HALE_FLOAT_CASE
  return hipErrorInvalidValue;
}

}  // namespace hale
