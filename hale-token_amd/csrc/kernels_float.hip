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
// HBM-bound for many rows (151,936 x 2048 bf16, not in the caches: 110 us, 5.7
// TB/s); few rows wait for the round trips and wave 0's fold.
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

// Rows row0 .. row0 + FR - 1 of one matrix, by one work-group.  VEC: every row
// starts 16-byte aligned, so a piece is one 16-byte load; otherwise it is read
// value by value.  NS: chunks in flight (float_ring).
template <int DT, bool VEC, int NS>
__device__ __forceinline__ void gemv_float_rows(const uint8_t* __restrict__ w, const float* __restrict__ x,
                                                int row0, int rows, int cols, float* __restrict__ out) {
  constexpr int PER = FloatFmt<DT>::PER16;
  constexpr int ESZ = DT == F32 ? 4 : 2;
  constexpr int UPR = FK / PER;          // 16-byte pieces per row of a chunk
  constexpr int LPT = FR * UPR / 256;    // pieces per thread per chunk
  constexpr int RPP = 256 / UPR;         // rows one pass of the 256 threads covers
  static_assert(LPT * 256 == FR * UPR && LPT * RPP == FR, "chunk tiling");
  static_assert(FR % 8 == 0 && FR * 8 <= 256, "fold threads fill whole waves");
  __shared__ __attribute__((aligned(16))) float prod[2][FR][FK + FPAD];

  const int tid = threadIdx.x;
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
    const int c = NS == 1 ? cp : min(cp, done - PER);
    const bool in = NS > 1 || c < done;
#pragma unroll
    for (int j = 0; j < LPT; j++) {
      const int r = min(row0 + j * RPP + tid / UPR, rows - 1);
      const uint8_t* src = w + (size_t)r * rb + (size_t)c * ESZ;
      if (in) {
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
    }
    if (in) {
#pragma unroll
      for (int q = 0; q < PER / 4; q++) {
        const f32x4 v = *(const f32x4*)(x + c + 4 * q);
        R.x[4 * q] = v.x;
        R.x[4 * q + 1] = v.y;
        R.x[4 * q + 2] = v.z;
        R.x[4 * q + 3] = v.w;
      }
    }
  };

  // fold thread (row fr, chain fl): the first FR * 8 threads
  constexpr int NF = FR * 8;
  const int fr = tid >> 3, fl = tid & 7;
  float acc = 0.0f;
  // chunk ch from R, which then takes chunk `next` if there is one
  auto step = [&](Regs& R, int ch, int next, bool more) {
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
    if (more) load(R, next);
    if (tid < NF) acc = lds_sum_strided<8>(&P[fr][fl], ncols / 8, acc);
  };
  // NS chunks in flight (the launcher's rows have as many)
  Regs R[NS];
  if constexpr (NS > 1) {
    int ch = 0;
#pragma unroll
    for (int j = 0; j < NS; j++) {
      load(R[j], j);
      __builtin_amdgcn_sched_barrier(0);
    }
    for (; ch + 2 * NS <= nchunks; ch += NS)
#pragma unroll
      for (int j = 0; j < NS; j++) step(R[j], ch + j, ch + NS + j, true);
#pragma unroll
    for (int j = 0; j < NS; j++) step(R[j], ch + j, ch + NS + j, ch + NS + j < nchunks);
    ch += NS;
#pragma unroll
    for (int j = 0; j < NS; j++)
      if (ch + j < nchunks) step(R[j], ch + j, 0, false);
  } else {
    if (nchunks > 0) load(R[0], 0);
    for (int ch = 0; ch < nchunks; ch++) step(R[0], ch, ch + 1, ch + 1 < nchunks);
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

template <int DT, bool VEC, int NS>
__global__ __launch_bounds__(256) void k_gemv_float(const uint8_t* __restrict__ w, const float* __restrict__ x,
                                                    int rows, int cols, float* __restrict__ out) {
  gemv_float_rows<DT, VEC, NS>(w, x, blockIdx.x * FR, rows, cols, out);
}

// The matrices of one launch (all cols long): work-groups first[i] ..
// first[i + 1] - 1 take matrix i.
struct FloatMats {
  const uint8_t* w[MATVEC_MANY];
  float* out[MATVEC_MANY];
  int rows[MATVEC_MANY], first[MATVEC_MANY];
};

template <int DT, bool VEC, int NS>
__global__ __launch_bounds__(256) void k_gemv_float_many(FloatMats m, const float* __restrict__ x, int cols) {
  const int g = blockIdx.x;
  int i = 0;
#pragma unroll
  for (int j = 1; j < MATVEC_MANY; j++) i = g >= m.first[j] ? j : i;
  gemv_float_rows<DT, VEC, NS>(m.w[i], x, (g - m.first[i]) * FR, m.rows[i], cols, m.out[i]);
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

// One value per thread: any alignment.
template <int DT>
__global__ __launch_bounds__(256) void k_encode_half(const float* __restrict__ v, size_t n,
                                                     uint16_t* __restrict__ out) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) out[i] = encode_half<DT>(v[i]);
}

// Four values per thread and step (values 16-byte, out 8-byte aligned), U steps
// in flight; the last n % 4 by the first threads of the launch.
template <int DT, int U>
__global__ __launch_bounds__(256) void k_encode_half4(const float* __restrict__ v, size_t n,
                                                      uint16_t* __restrict__ out) {
  const size_t pieces = n / 4;
  const size_t p0 = (size_t)blockIdx.x * (256 * U) + threadIdx.x;
  const size_t last = pieces * 4 + threadIdx.x;
  if (blockIdx.x == 0 && last < n) out[last] = encode_half<DT>(v[last]);
  f32x4 x[U];
#pragma unroll
  for (int u = 0; u < U; u++) x[u] = ((const f32x4*)v)[p0 + 256 * u < pieces ? p0 + 256 * u : pieces - 1];
#pragma unroll
  for (int u = 0; u < U; u++) {
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
    const bool wide = convert_wide(n / 4);
    const unsigned per = wide ? 1024 : 256, grid = (unsigned)((n / 4 + per - 1) / per);
    auto run = [&](auto kernel) { return launch(kernel, grid, 256, 0, st, values, n, o); };
    if (dtype == F16) return wide ? run(k_encode_half4<F16, 4>) : run(k_encode_half4<F16, 1>);
    return wide ? run(k_encode_half4<BF16, 4>) : run(k_encode_half4<BF16, 1>);
  }
  const unsigned grid = (unsigned)((n + 255) / 256);
  return dtype == F16 ? launch(k_encode_half<F16>, grid, 256, 0, st, values, n, o)
                      : launch(k_encode_half<BF16>, grid, 256, 0, st, values, n, o);
}

// Whether a launch keeps several chunks in flight (two of f32, four of half
// values) instead of one ahead: rows of four chunks and more, and either at most
// a work-group per CU, where nothing else covers the round trips, or half rows so
// many that the launch is a stream through memory.  Between them a CU's
// work-groups cover for each other, one's loads under another's fold, and sending
// every load first only brings their folds together.  One ahead / several, us,
// weights not in the caches: bf16 2048 x 2048 / 4096 / 8192 6.8 / 6.5, 10.1 / 9.4,
// 16.1 / 14.5; f32 2048 x 2048 / 5120 8.1 / 7.3, 15.2 / 11.7; bf16 3000 x 4096
// 10.8 / 11.4, 5120 x 2048 8.0 / 8.9, 8192 x 4096 14.9 / 17.7, 32,768 x 5120 55.2 /
// 55.8, 50,000 x 2048 40.6 / 38.3, 151,936 x 2048 116 / 110; f32 launches of many
// work-groups draw (20,000 x 4096 54.4 / 54.4).  Of a matrix that is already in
// L2 several chunks cost the few work-groups up to 0.3 us (bf16 64 x 3072 5.65 /
// 5.95).  Rows of fewer chunks have nothing to keep in flight (f32 2048 x 1500 6.7 /
// 6.9).  Off the 16 bytes half rows gain alike (bf16 2048 x 4100 11.5 / 10.0), rows
// of f32 do not (2048 x 2050 9.1 / 9.4).
static bool float_ring(int dtype, bool vec, size_t cols, size_t groups) {
  const size_t nchunks = (cols / 8 * 8 + FK - 1) / FK;
  if (nchunks < 4 || (!vec && dtype == F32)) return false;
  return groups <= 256 || (vec && dtype != F32 && groups >= 6144);
}

hipError_t launch_gemv_float(int dtype, const void* w, const float* x, size_t rows, size_t cols,
                             float* out, hipStream_t st) {
  if (rows == 0) return hipSuccess;
  if (rows > (size_t)INT32_MAX - FR || cols > (size_t)INT32_MAX - FK) return hipErrorInvalidValue;
  if ((uintptr_t)x % 16) return hipErrorInvalidValue;  // x is read in 16-byte pieces
  const int esz = dtype == F32 ? 4 : 2;
  const bool vec = (cols * esz) % 16 == 0 && (uintptr_t)w % 16 == 0;
  const unsigned groups = (unsigned)((rows + FR - 1) / FR);
  auto run = [&](auto kernel) {
    return launch(kernel, groups, 256, 0, st, (const uint8_t*)w, x, (int)rows, (int)cols, out);
  };
#define HALE_FLOAT_CASE(D)                                                                       \
  if (dtype == D) {                                                                              \
    constexpr int NS = D == F32 ? 2 : 4;                                                         \
    if (float_ring(D, vec, cols, groups))                                                        \
      return vec ? run(k_gemv_float<D, true, NS>) : run(k_gemv_float<D, D == F32, NS>);          \
    return vec ? run(k_gemv_float<D, true, 1>) : run(k_gemv_float<D, false, 1>);                 \
  }
  HALE_FLOAT_CASE(F32)
  HALE_FLOAT_CASE(F16)
  HALE_FLOAT_CASE(BF16)
#undef HALE_FLOAT_CASE
  return hipErrorInvalidValue;
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
#define HALE_FLOAT_CASE(D)                                                                            \
  if (dtype == D) {                                                                                   \
    constexpr int NS = D == F32 ? 2 : 4;                                                              \
    if (float_ring(D, vec, cols, groups))                                                             \
      return vec ? run(k_gemv_float_many<D, true, NS>) : run(k_gemv_float_many<D, D == F32, NS>);     \
    return vec ? run(k_gemv_float_many<D, true, 1>) : run(k_gemv_float_many<D, false, 1>);            \
  }
  HALE_FLOAT_CASE(F32)
  HALE_FLOAT_CASE(F16)
  HALE_FLOAT_CASE(BF16)
#undef HALE_FLOAT_CASE
  return hipErrorInvalidValue;
}

}  // namespace hale
