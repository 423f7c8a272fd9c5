// Direct (no K staging) GEMM family and the element-op kernels.
//
// Direct GEMM: what the reference pipeline emits for "tile-k=0" options, its
// default (docs/stage7.md:9-20; lib/Transforms/Gpu.cpp:188-197): the launch is
// grid (ceil(N/BN), ceil(M/BM)) x block (BN/TN, BM/TM), each thread owns a
// TM x TN sub-tile of its block tile and runs the K loop from +0.0 with one
// fused multiply-add per k, in sequential k order, then the fused epilogue.
// That arithmetic is bit-identical to the reference's naive kernel
// (docs/numerics.md:53), any shape is accepted and edges are masked.  Where
// every buffer is 16-byte aligned the runtime runs the same chains on the matrix
// cores instead (staged_gemm.hpp, sequential k; the same bits); this kernel
// serves the rest: unaligned buffers, and ragged matrices of 2^31 elements.
//
// Element-op kernels: programs with no matmul (tforge.bias_add / relu / add
// alone, or chains of them) run one IEEE operation per op, so results are
// bit-exact against NumPy float32 (python/tforge_gpu.py:116-126).
//
// Split-K reduction: the second launch of a staged matmul compiled with
// split-k=S (a backend option): C = epi(slice 0 + ... + slice S-1).
#include <algorithm>

#include "epilogue.hpp"

namespace tfk {

template <int TM, int TN>
__global__ void direct_gemm_kernel(GemmParams p) {
  const long m_base = ((long)blockIdx.y * blockDim.y + threadIdx.y) * TM;
  const long n_base = ((long)blockIdx.x * blockDim.x + threadIdx.x) * TN;
  if (m_base >= p.M || n_base >= p.N) return;
  float acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = 0.0f;
  const bool full = m_base + TM <= p.M && n_base + TN <= p.N;
  for (int k = 0; k < p.K; ++k) {
    float a[TM], b[TN];
#pragma unroll
    for (int i = 0; i < TM; ++i) a[i] = (full || m_base + i < p.M) ? p.A[(m_base + i) * p.lda + k] : 0.0f;
#pragma unroll
    for (int j = 0; j < TN; ++j) b[j] = (full || n_base + j < p.N) ? p.B[(long)k * p.ldb + n_base + j] : 0.0f;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_fmaf(a[i], b[j], acc[i][j]);
  }
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const long m = m_base + i, n = n_base + j;
      if (m < p.M && n < p.N) p.C[m * p.ldc + n] = apply_epi1(acc[i][j], p.epi, m, (int)n);
    }
}

// Element ops on buffers that are not 16-byte aligned: the options' own
// geometry, one element at a time.
template <int TM, int TN>
__global__ void elementwise_kernel(EltParams p) {
  const long m_base = ((long)blockIdx.y * blockDim.y + threadIdx.y) * TM;
  const long n_base = ((long)blockIdx.x * blockDim.x + threadIdx.x) * TN;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const long m = m_base + i, n = n_base + j;
      if (m < p.M && n < p.N) p.Y[m * p.ldy + n] = apply_epi1(p.X[m * p.ldx + n], p.epi, m, (int)n);
    }
}

// Element ops on 16-byte aligned buffers, whatever the options' tiles: the
// matrices are contiguous, so they are one stream of M * N elements, one 128-bit
// vector per lane, and odd row lengths cost nothing (the bias column of a vector
// is its element index mod N).  Bound by HBM.  Every byte is touched once, so
// the accesses are non-temporal (cached ones: 1-8% slower on buffers that start
// in HBM).  A workgroup's WAVES waves read as many segments of SEG KiB, 1 KiB each,
// and consecutive workgroups walk the segments: workgroups that read 4 KiB in
// one piece keep fewer HBM banks busy.  Back to back on cold buffers (us), one
// piece / 8 waves x 32 KiB / 4 waves x 4 KiB: relu 2047x4093 12.4 / 11.3 / 11.7,
// add 8192^2 124.0 / 119.1 / 119.2, relu 16384^2 324 / 313 / 307, add 16384^2
// 499 / 481 / 469; so 8 x 32 below kHugeStream elements, 4 x 4 from there.
// Against one element per thread on 16x16 tiles -> this: relu 2047x4093 27.8 ->
// 11.3, add 4096^2 56.6 -> 31.5, add 8192^2 217 -> 119; against 1x4 elements on 4x256
// tiles: relu 2047x4093 25.1 -> 11.3, relu 8192^2 80.2 -> 79.3, bias_add 8192^2
// 81.6 -> 79.3 (6.77 TB/s).
constexpr long kHugeStream = 1L << 27;
constexpr long kMaxFlatGrid = 1L << 22;  // 2^32 elements in 4-wave workgroups

// The bias of stream elements 4 * q .. + 3, the first in column n; columns wrap at
// N (N may be 1).
template <typename Idx>
__device__ __forceinline__ f32x4 flat_bias(const float *bias, Idx n, Idx N) {
  if (n + 4 <= N) return *reinterpret_cast<const f32x4_u *>(bias + n);
  f32x4 v;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    v[e] = bias[n];
    n = n + 1 == N ? 0 : n + 1;
  }
  return v;
}

// Idx: unsigned where M * N < 2^32, else unsigned long.  ONE: the chain has at
// most one bias and one add operand, which then arrive, like the op kinds (8
// bits each in `kinds`), in preloaded arguments (13 SGPRs): a wave moves only
// 2-4 KiB, and waiting for the epilogue's fields from the argument segment made
// relu at 8192^2 78.7 -> 82.0 us, bias_add 80.0 -> 89.5.  `inv` = floor(2^32 / N).
template <typename Idx, bool ONE, unsigned WAVES, unsigned SEG>
__global__ void __launch_bounds__(64 * WAVES)
elementwise_flat_kernel(const float *X, float *Y, long total, const float *bias, const float *R, unsigned N, unsigned inv,
                        unsigned kinds, EltParams p) {
  const unsigned lane = threadIdx.x & 63;
  const unsigned wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const Idx vecs = (Idx)((unsigned long)total / 4);
  auto kind = [&](int i) __attribute__((always_inline)) { return (int)(kinds >> (8 * i)) & 255; };
  auto body = [&](Idx b) __attribute__((always_inline)) {
    const Idx piece = (b / SEG * WAVES + wave) * SEG + b % SEG;
    const Idx q = piece * 64 + lane;
    if (q >= vecs) return;
    f32x4 v = __builtin_nontemporal_load(reinterpret_cast<const f32x4 *>(X) + q);
    // Column of this lane's first element: the wave's first column (scalar; the
    // estimated quotient is the true one or one less), then at most one wrap
    // where a row holds a wave's 256 elements.
    auto column = [&]() __attribute__((always_inline)) {
      const Idx e0 = piece * 256;
      Idx n0;
      if constexpr (sizeof(Idx) == 4) {
        n0 = e0 - __umulhi(e0, inv) * N;
        if (n0 >= N) n0 -= N;
      } else {
        n0 = e0 % N;
      }
      Idx n = n0 + 4 * lane;
      if (N >= 256) return n >= N ? n - N : n;
      return n % N;
    };
    // Every operand is requested before the first is used.
    f32x4 r[ONE ? 2 : kMaxEpi];
    if constexpr (ONE) {
      if (bias) r[0] = flat_bias<Idx>(bias, column(), N);
      if (R) r[1] = __builtin_nontemporal_load(reinterpret_cast<const f32x4 *>(R) + q);
    } else {
#pragma unroll
      for (int i = 0; i < kMaxEpi; ++i) {
        if (kind(i) == EPI_BIAS) r[i] = flat_bias<Idx>(p.epi.ptr[i], column(), N);
        else if (kind(i) == EPI_ADD) r[i] = __builtin_nontemporal_load(reinterpret_cast<const f32x4 *>(p.epi.ptr[i]) + q);
      }
    }
#pragma unroll
    for (int i = 0; i < kMaxEpi; ++i) {
      const int k = kind(i);
      if (k == EPI_NONE) break;
      if (k == EPI_BIAS) {
        v += r[ONE ? 0 : i];
      } else if (k == EPI_ADD) {
        v += r[ONE ? 1 : i];
      } else if (k == EPI_RELU) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = relu_ieee(v[e]);
      } else if (k == EPI_ADD_SELF) {
        v = v + v;
      }
    }
    __builtin_nontemporal_store(v, reinterpret_cast<f32x4 *>(Y) + q);
  };
  if constexpr (sizeof(Idx) == 4) {
    body(blockIdx.x);  // the grid covers every piece
  } else {
    constexpr Idx kSpan = 64 * WAVES * SEG;
    for (Idx b = blockIdx.x; b < (vecs + kSpan - 1) / kSpan * SEG; b += gridDim.x) body(b);
  }
  // The last M * N mod 4 elements, one lane each.
  if (blockIdx.x == 0 && threadIdx.x < (total & 3)) {
    const long at = (total & ~3L) + threadIdx.x;
    const long m = at / N;
    const int n = (int)(at - m * N);
    Y[at] = apply_epi1(X[at], p.epi, m, n);
  }
}

template <int TM, int TN>
hipError_t launch_direct(const GemmParams &p, dim3 grid, dim3 block, hipStream_t stream) {
  hipLaunchKernelGGL((direct_gemm_kernel<TM, TN>), grid, block, 0, stream, p);
  return hipGetLastError();
}

template <int TM, int TN>
hipError_t launch_elementwise(const EltParams &p, dim3 grid, dim3 block, hipStream_t stream) {
  hipLaunchKernelGGL((elementwise_kernel<TM, TN>), grid, block, 0, stream, p);
  return hipGetLastError();
}

using FlatFn = void (*)(const float *, float *, long, const float *, const float *, unsigned, unsigned, unsigned, EltParams);
struct FlatKernel {
  const char *name;
  FlatFn fn;
  unsigned waves, seg;
};

static int count_kind(const EltParams &p, int kind) {
  int n = 0;
  for (int i = 0; i < p.epi.nops; ++i) n += p.epi.kind[i] == kind;
  return n;
}

#define TF_FLAT(IDX, ONE, WAVES, SEG) \
  FlatKernel{"tf_elementwise_flat_" #IDX "_" #ONE "_w" #WAVES "s" #SEG, &elementwise_flat_kernel<IDX, ONE, WAVES, SEG>, WAVES, SEG}
static const FlatKernel &flat_kernel(const EltParams &p) {
  static const FlatKernel kFlat[3][2] = {{TF_FLAT(uint32_t, false, 8, 32), TF_FLAT(uint32_t, true, 8, 32)},
                                         {TF_FLAT(uint32_t, false, 4, 4), TF_FLAT(uint32_t, true, 4, 4)},
                                         {TF_FLAT(uint64_t, false, 4, 4), TF_FLAT(uint64_t, true, 4, 4)}};
  const long total = (long)p.M * p.N;
  const bool one = count_kind(p, EPI_BIAS) <= 1 && count_kind(p, EPI_ADD) <= 1;
  return kFlat[total < kHugeStream ? 0 : total < (1L << 32) ? 1 : 2][one];
}
#undef TF_FLAT

static dim3 flat_grid(const EltParams &p, const FlatKernel &k) {
  const long vecs = (long)p.M * p.N / 4, span = 64 * k.waves * k.seg;
  return dim3((unsigned)std::min(std::max(1L, (vecs + span - 1) / span * k.seg), kMaxFlatGrid));
}

FlatLaunch elementwise_flat_launch(const EltParams &p) {
  const FlatKernel &k = flat_kernel(p);
  return {k.name, reinterpret_cast<const void *>(k.fn), flat_grid(p, k), dim3(64 * k.waves)};
}

hipError_t launch_elementwise_flat(const EltParams &p, hipStream_t stream) {
  unsigned kinds = 0;
  const float *bias = nullptr, *r = nullptr;
  for (int i = 0; i < p.epi.nops; ++i) {
    kinds |= (unsigned)p.epi.kind[i] << (8 * i);
    if (p.epi.kind[i] == EPI_BIAS) bias = p.epi.ptr[i];
    if (p.epi.kind[i] == EPI_ADD) r = p.epi.ptr[i];
  }
  const FlatKernel &k = flat_kernel(p);
  const unsigned n = (unsigned)p.N, inv = n > 1 ? (unsigned)((1UL << 32) / n) : ~0u;
  hipLaunchKernelGGL(k.fn, flat_grid(p, k), dim3(64 * k.waves), 0, stream, p.X, p.Y, (long)p.M * p.N, bias, r, n, inv, kinds,
                     p);
  return hipGetLastError();
}

// Split-K reduction: one thread per 4 consecutive outputs; the partial-sum
// slices are read 4 at a time (independent loads in flight) and added in
// slice order, so the result does not depend on scheduling.
__global__ void __launch_bounds__(256) splitk_reduce_kernel(ReduceParams p) {
  const long q = (long)blockIdx.x * 256 + threadIdx.x;
  const long per_row = (p.N + 3) / 4;
  if (q >= (long)p.M * per_row) return;
  const long m = q / per_row;
  const int n = (int)(q - m * per_row) * 4;
  const float *src = p.ws + m * p.ws_ld + n;
  auto ld = [&](int s) { return *reinterpret_cast<const f32x4 *>(src + s * p.ws_slice); };
  f32x4 v = ld(0);
  int s = 1;
  for (; s + 4 <= p.splits; s += 4) {
    const f32x4 t0 = ld(s), t1 = ld(s + 1), t2 = ld(s + 2), t3 = ld(s + 3);
    v += t0;
    v += t1;
    v += t2;
    v += t3;
  }
  for (; s < p.splits; ++s) v += ld(s);
  if ((p.ldc & 3) == 0 && n + 4 <= p.N) {
    *reinterpret_cast<f32x4 *>(p.C + m * p.ldc + n) = apply_epi4(v, p.epi, m, n);
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (n + e < p.N) p.C[m * p.ldc + n + e] = apply_epi1(v[e], p.epi, m, n + e);
  }
}

hipError_t launch_splitk_reduce(const ReduceParams &p, hipStream_t stream) {
  const long quads = (long)p.M * ((p.N + 3) / 4);
  hipLaunchKernelGGL(splitk_reduce_kernel, dim3((unsigned)((quads + 255) / 256)), dim3(256), 0, stream, p);
  return hipGetLastError();
}

// The registry tables are host data (they hold host launch stubs).
#ifndef __HIP_DEVICE_COMPILE__
#define TF_DIRECT(TM, TN)                                                                       \
  KernelEntry{FAM_DIRECT, 0, 0, TM, TN, 0, 0, 0, 0, "tf_direct_t" #TM "x" #TN,                \
              reinterpret_cast<const void *>(&direct_gemm_kernel<TM, TN>), &launch_direct<TM, TN>, \
              nullptr, 0}
#define TF_ELT(TM, TN)                                                                          \
  KernelEntry{FAM_ELEMENTWISE, 0, 0, TM, TN, 0, 0, 0, 0, "tf_elementwise_t" #TM "x" #TN,      \
              reinterpret_cast<const void *>(&elementwise_kernel<TM, TN>), nullptr,             \
              &launch_elementwise<TM, TN>, 0}
#define TF_BOTH(TM, TN) TF_DIRECT(TM, TN), TF_ELT(TM, TN)

// Thread tiles 1, 2, 4, 8 in each dimension.
extern const KernelEntry kDirectEntries[] = {
    TF_BOTH(1, 1), TF_BOTH(1, 2), TF_BOTH(1, 4), TF_BOTH(1, 8), TF_BOTH(2, 1), TF_BOTH(2, 2),
    TF_BOTH(2, 4), TF_BOTH(2, 8), TF_BOTH(4, 1), TF_BOTH(4, 2), TF_BOTH(4, 4), TF_BOTH(4, 8),
    TF_BOTH(8, 1), TF_BOTH(8, 2), TF_BOTH(8, 4), TF_BOTH(8, 8),
};
extern const int kDirectCount = sizeof(kDirectEntries) / sizeof(kDirectEntries[0]);
#else
// Device pass: instantiate the kernels the host table names.
#define TF_INST(TM, TN)                                                  \
  template __global__ void direct_gemm_kernel<TM, TN>(GemmParams);       \
  template __global__ void elementwise_kernel<TM, TN>(EltParams);
TF_INST(1, 1) TF_INST(1, 2) TF_INST(1, 4) TF_INST(1, 8)
TF_INST(2, 1) TF_INST(2, 2) TF_INST(2, 4) TF_INST(2, 8)
TF_INST(4, 1) TF_INST(4, 2) TF_INST(4, 4) TF_INST(4, 8)
TF_INST(8, 1) TF_INST(8, 2) TF_INST(8, 4) TF_INST(8, 8)
#endif  // __HIP_DEVICE_COMPILE__

}  // namespace tfk
