// The forward-side half of the activation handoff: the serving step's save of
// the finetuning rows into the activation store the backward reads.
//
// Semantics: deltaserve-plugin/deltaserve/ft_save_op.py:72-93 (the
// graph-capturable save op) and accumulate.py:324-343 (arm_op_step):
//   rows = x.index_select(0, src) (+ r.index_select(0, src)),  in x's dtype
//   buf.index_copy_(0, dst, rows.to(buf.dtype))
// with src/dst persistent int64 index tensors of a fixed length (max_saved):
// the first n entries gather the step's FT rows into buffer rows
// offset .. offset+n-1, the rest point at row 0 and the scratch row
// buf[max_saved]. The scratch row is never read by the backward (every
// consumer slices [:n]); this kernel skips those slots instead of writing
// them, which also removes their memory traffic. The final save point's
// input ids go through the same index pair (accumulate.py:598-622).
//
// Slots whose source row lies outside x (or the id vector) are skipped too:
// the gather never reads out of bounds.
//
// Both kernels take a fixed row count and read the indices from device
// memory, so a captured graph replays them with fresh indices each step.
#include "kernels.h"

namespace dsb {

namespace {
template <int T>
DSB_DEV float load_as_float(const void* p, long i);
template <>
DSB_DEV float load_as_float<DSB_DT_BF16>(const void* p, long i) {
  return (float)reinterpret_cast<const bf16*>(p)[i];
}
template <>
DSB_DEV float load_as_float<DSB_DT_F16>(const void* p, long i) {
  return (float)reinterpret_cast<const _Float16*>(p)[i];
}
template <>
DSB_DEV float load_as_float<DSB_DT_F32>(const void* p, long i) {
  return reinterpret_cast<const float*>(p)[i];
}
// round to the input dtype (the reference adds in x's dtype)
template <int T>
DSB_DEV float round_to(float v);
template <>
DSB_DEV float round_to<DSB_DT_BF16>(float v) { return (float)(bf16)v; }
template <>
DSB_DEV float round_to<DSB_DT_F16>(float v) { return (float)(_Float16)v; }
template <>
DSB_DEV float round_to<DSB_DT_F32>(float v) { return v; }
}  // namespace

// 8 consecutive elements as floats (16-byte aligned: one 16-byte load, two for
// fp32).
template <int T>
DSB_DEV void load8_as_float(const void* p, long i, float v[8]) {
  if constexpr (T == DSB_DT_F32) {
    const f32x4* q = reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(p) + i);
    const f32x4 a = q[0], b = q[1];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[e] = a[e];
      v[4 + e] = b[e];
    }
  } else if constexpr (T == DSB_DT_F16) {
    typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
    const f16x8 a = *reinterpret_cast<const f16x8*>(reinterpret_cast<const _Float16*>(p) + i);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = (float)a[e];
  } else {
    unpack8(ldg128(reinterpret_cast<const bf16*>(p) + i), v);
  }
}

// The grid's x is the index slot, its y a run of kSaveRun columns of the row;
// a thread moves kSaveVec groups of 8 columns, loaded before the first is
// stored. VEC: 16-byte accesses (rows, strides and width allow them), else
// element by element. One block per row with one load in flight per thread,
// and residual rows element by element, took 13.6 µs per launch for the
// 256-row saves of a 5120-wide model (residual and 34816-wide rows, 34 µs of
// them in 17 launches at copy rate); now 7.9 µs.
constexpr int kSaveVec = 2, kSaveRun = 256 * 8 * kSaveVec;
template <int T, bool VEC>
__global__ __launch_bounds__(256) void save_rows_kernel(const void* __restrict__ x, long ldx,
                                                        const void* __restrict__ r, long ldr,
                                                        long x_rows,
                                                        const int64_t* __restrict__ src,
                                                        const int64_t* __restrict__ dst, int width,
                                                        bf16* __restrict__ buf, long ldbuf,
                                                        long buf_rows) {
  const long d = dst[blockIdx.x], s = src[blockIdx.x];
  if (d < 0 || d >= buf_rows - 1) return;  // the scratch row (and out of range): skipped
  if (s < 0 || s >= x_rows) return;  // a source row outside x: skipped
  const long xo = s * ldx, ro = s * ldr, bo = d * ldbuf;
  const int c0 = blockIdx.y * kSaveRun;
  if constexpr (VEC) {
    if (T == DSB_DT_BF16 && !r) {  // a copy: the bits as they are, NaN payloads included
      u32x4 v[kSaveVec];
#pragma unroll
      for (int i = 0; i < kSaveVec; ++i) {
        const int c = c0 + (threadIdx.x + 256 * i) * 8;
        if (c < width) v[i] = ldg128(reinterpret_cast<const bf16*>(x) + xo + c);
      }
#pragma unroll
      for (int i = 0; i < kSaveVec; ++i) {
        const int c = c0 + (threadIdx.x + 256 * i) * 8;
        if (c < width) stg128(buf + bo + c, v[i]);
      }
      return;
    }
    float v[kSaveVec][8], w[kSaveVec][8];
#pragma unroll
    for (int i = 0; i < kSaveVec; ++i) {
      const int c = c0 + (threadIdx.x + 256 * i) * 8;
      if (c < width) {
        load8_as_float<T>(x, xo + c, v[i]);
        if (r) load8_as_float<T>(r, ro + c, w[i]);
      }
    }
#pragma unroll
    for (int i = 0; i < kSaveVec; ++i) {
      const int c = c0 + (threadIdx.x + 256 * i) * 8;
      if (c >= width) continue;
      if (r) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[i][e] = round_to<T>(v[i][e] + w[i][e]);
      }
      stg128(buf + bo + c, pack8(v[i]));
    }
  } else {
    const int end = min(width, c0 + kSaveRun);
    for (int c = c0 + threadIdx.x; c < end; c += 256) {
      float v = load_as_float<T>(x, xo + c);
      if (r) v = round_to<T>(v + load_as_float<T>(r, ro + c));
      buf[bo + c] = (bf16)v;
    }
  }
}

__global__ __launch_bounds__(256) void save_ids_kernel(const int64_t* __restrict__ ids,
                                                       long ids_len,
                                                       const int64_t* __restrict__ src,
                                                       const int64_t* __restrict__ dst, int count,
                                                       int64_t* __restrict__ out, long out_len) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= count) return;
  const long d = dst[i];
  const long s = src[i];
  if (d < 0 || d >= out_len || s < 0 || s >= ids_len) return;
  out[d] = ids[s];
}

hipError_t save_rows(const void* x, long ldx, const void* r, long ldr, long x_rows, int dtype,
                     const int64_t* src, const int64_t* dst, int count, int width, bf16* buf,
                     long ldbuf, long buf_rows, hipStream_t s) {
  if (count <= 0 || width <= 0) return hipSuccess;
  const long es = dtype == DSB_DT_F32 ? 4 : 2;
  const bool vec = width % 8 == 0 && ldx * es % 16 == 0 && (!r || ldr * es % 16 == 0) &&
                   ldbuf % 8 == 0 &&
                   (((unsigned long)x | (unsigned long)r | (unsigned long)buf) & 15) == 0;
  const dim3 grid(count, (width + kSaveRun - 1) / kSaveRun);
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, s, x, ldx, r, ldr, x_rows, src, dst, width, buf,
                       ldbuf, buf_rows);
    return hipGetLastError();
  };
  switch (dtype) {
    case DSB_DT_BF16:
      return vec ? go(save_rows_kernel<DSB_DT_BF16, true>) : go(save_rows_kernel<DSB_DT_BF16, false>);
    case DSB_DT_F16:
      return vec ? go(save_rows_kernel<DSB_DT_F16, true>) : go(save_rows_kernel<DSB_DT_F16, false>);
    case DSB_DT_F32:
      return vec ? go(save_rows_kernel<DSB_DT_F32, true>) : go(save_rows_kernel<DSB_DT_F32, false>);
    default:
      return hipErrorInvalidValue;
  }
}

hipError_t save_ids(const int64_t* ids, long ids_len, const int64_t* src, const int64_t* dst, int count,
                    int64_t* out, long out_len, hipStream_t s) {
  if (count <= 0) return hipSuccess;
  hipLaunchKernelGGL(save_ids_kernel, dim3((count + 255) / 256), dim3(256), 0, s, ids, ids_len, src,
                     dst, count, out, out_len);
  return hipGetLastError();
}

}  // namespace dsb
