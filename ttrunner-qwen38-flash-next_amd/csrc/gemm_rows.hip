// Projections of a layer for more token rows than qm_gemv takes, gfx950:
// y[m][n] = sum_k W[n][k] x[m][k] for up to GR_MAX_M rows, on the matrix cores.
//
// At these row counts (a batch of sequences decoding, a few drafted tokens) the
// product is still a stream over the weights: 50 MB for a DeltaNet layer's
// input projections, 0.8 GFLOP at 16 rows. As in gemv.hip the projections that
// read the same input are one launch over their concatenated rows with a
// segment table for the outputs, and the output projection can add its result
// into the residual streams (reference/model.py:79-81), with gemv.hip's
// roundings.
//
// Work split: a workgroup takes TN tiles of 16 weight rows against MT tiles of
// 16 token rows; its waves split k, 64 units (1 KB) of every row each. A wave
// reads whole 1 KB row segments (not the operand's own shape, 16 rows x 64 bytes
// a load: see to_frags), all of them in flight at once, and turns them into
// operands through LDS of its own, without a barrier. The waves' partial results meet in LDS.
//
// Measured with weights from memory, against the library's GEMMs that served
// these row counts (us): DeltaNet input projections (50 MB) 45.3 -> 13.8 at 16
// rows (3.7 TB/s), 44.7 -> 17.5 at 32, 45.5 -> 26.2 at 64 (the weights are read
// once per 32 rows; once per 16, as at other k, it was 20.6 and 33.9); output projection (17 MB) 11.8 -> 6.5 at 16,
// with the reinjection's own launch (4.7 us) gone as well.
#include "rows_mma.h"
#include "qwen4mix_internal.h"

namespace {

constexpr int GR_MAX_M = 64;
constexpr int GR_PRE = 4;          // residual streams whose values load with the weights

template <typename T>
struct GemmRowsArgs {
  const T* w;     // [N, K]
  const T* x;     // [M, K]
  int M, N, K;
  int n_seg;
  int seg_end[QM_GEMV_MAX_SEG];
  T* seg_out[QM_GEMV_MAX_SEG];
  T* hyper;       // reinjection: [M, streams * N], updated in place
  const T* inject;
  int streams;
};

// grid (ceil(N / (16 TN)), ceil(M / (16 MT))), NW waves; K = NW * PASS * 64 units
template <typename T, int NW, int PASS, int TN, int MT, bool RJ>
__global__ __launch_bounds__(64 * NW) void gemm_rows_kernel(GemmRowsArgs<T> A) {
  constexpr int VE = Chunk<T>::VE;
  static_assert(TN * MT <= NW, "a wave finishes a 16x16 result");
  __shared__ uint4 s_rows[NW][16 * ROW_US];
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int g4 = lane >> 4, r16 = lane & 15;
  const int n0 = blockIdx.x * 16 * TN, m0 = blockIdx.y * 16 * MT;
  // the result this wave finishes: weight tile wid / MT, token tile wid % MT
  const int m = m0 + 16 * (wid % MT) + r16;
  RowAcc<T> acc[TN][MT];
  float hv[GR_PRE][4], iv[GR_PRE];
#pragma unroll
  for (int p = 0; p < PASS; ++p) {
    const long k0 = (long)((p * NW + wid) * 64 + lane) * VE;
    u32x4_t xr[MT][16], wr[TN][16];
#pragma unroll
    for (int u = 0; u < MT; ++u)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        xr[u][r] = *reinterpret_cast<const u32x4_t*>(A.x + (long)min(m0 + 16 * u + r, A.M - 1) * A.K + k0);
#pragma unroll
    for (int t = 0; t < TN; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        wr[t][r] = *reinterpret_cast<const u32x4_t*>(A.w + (long)min(n0 + 16 * t + r, A.N - 1) * A.K + k0);
    if constexpr (RJ) {
      // the residual values and inject weights of this lane's outputs, in the
      // weights' round trip
      if (p == 0 && wid < TN * MT) {
        const int n = min(n0 + 16 * (wid / MT) + 4 * g4, A.N - 4), mc = min(m, A.M - 1);
#pragma unroll
        for (int s = 0; s < GR_PRE; ++s) {
          const int sc = min(s, A.streams - 1);
          load_act4(A.hyper + ((long)mc * A.streams + sc) * A.N + n, hv[s]);
          iv[s] = Act<T>::load(A.inject, (long)mc * A.streams + sc);
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    u32x4_t xf[MT][16], wf[16];
#pragma unroll
    for (int u = 0; u < MT; ++u) to_frags(s_rows[wid], xr[u], lane, r16, g4, xf[u]);
#pragma unroll
    for (int t = 0; t < TN; ++t) {
      to_frags(s_rows[wid], wr[t], lane, r16, g4, wf);
#pragma unroll
      for (int i = 0; i < 16; ++i)
#pragma unroll
        for (int u = 0; u < MT; ++u) {
          acc[t][u].step(__builtin_bit_cast(uint4, wf[i]), __builtin_bit_cast(uint4, xf[u][i]));
          if (i % 4 == 3) acc[t][u].block();
        }
    }
  }
  // the waves' sums: lane holds rows n0 + 16 t + 4 g4 + i of token row m0 + 16 u + r16
  f32x4_t* red = reinterpret_cast<f32x4_t*>(s_rows);       // [NW][TN * MT][64]
  __syncthreads();
#pragma unroll
  for (int t = 0; t < TN; ++t)
#pragma unroll
    for (int u = 0; u < MT; ++u) red[(wid * TN * MT + t * MT + u) * 64 + lane] = acc[t][u].sum();
  __syncthreads();
  if (wid >= TN * MT) return;
  f32x4_t v = red[wid * 64 + lane];
#pragma unroll
  for (int w = 1; w < NW; ++w) v += red[(w * TN * MT + wid) * 64 + lane];
  const int n = n0 + 16 * (wid / MT) + 4 * g4;
  if (m >= A.M || n >= A.N) return;
  if constexpr (RJ) {                                       // N is a multiple of 4
    float y[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) y[i] = Act<T>::round(v[i]);
    for (int s = 0; s < A.streams; ++s) {
      T* hp = A.hyper + ((long)m * A.streams + s) * A.N + n;
      float h[4], inj, o[4];
      if (s < GR_PRE) {
#pragma unroll
        for (int u = 0; u < GR_PRE; ++u)
          if (u == s) {
            inj = iv[u];
#pragma unroll
            for (int i = 0; i < 4; ++i) h[i] = hv[u][i];
          }
      } else {
        inj = Act<T>::load(A.inject, (long)m * A.streams + s);
        load_act4(hp, h);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] = add_rn(h[i], Act<T>::round(mul_rn(y[i], inj)));
      store_act4(hp, o);
    }
  } else {
    int s = 0, start = 0;
    while (s + 1 < A.n_seg && n >= A.seg_end[s]) { start = A.seg_end[s]; ++s; }
    const int n_s = A.seg_end[s] - start;
    T* o = A.seg_out[s] + (long)m * n_s + (n - start);
    if (n + 4 <= A.seg_end[s] && (reinterpret_cast<uintptr_t>(o) & (4 * sizeof(T) - 1)) == 0) {
      const float q[4] = {v[0], v[1], v[2], v[3]};
      store_act4(o, q);
    } else {
      for (int i = 0; i < 4 && n + i < A.N; ++i) {
        while (s + 1 < A.n_seg && n + i >= A.seg_end[s]) { start = A.seg_end[s]; ++s; }
        Act<T>::store(A.seg_out[s], (long)m * (A.seg_end[s] - start) + (n + i - start), v[i]);
      }
    }
  }
}

template <typename T, int NW, int PASS, int TN, int MT, bool RJ>
int launch_tile(const GemmRowsArgs<T>& A, hipStream_t stream) {
  hipLaunchKernelGGL((gemm_rows_kernel<T, NW, PASS, TN, MT, RJ>),
                     dim3((A.N + 16 * TN - 1) / (16 * TN), (A.M + 16 * MT - 1) / (16 * MT)), dim3(64 * NW), 0, stream, A);
  QM_CHECK_LAUNCH();
  return QM_OK;
}

template <typename T, bool RJ>
int launch_rows(const GemmRowsArgs<T>& A, hipStream_t stream) {
  const int segs = A.K / (64 * Chunk<T>::VE);               // 1 KB segments of a row
  // four waves hold two weight tiles against one token tile, or one against
  // two (more than 16 rows: the weights are then read once per 32)
  if (segs == 4) return A.M <= 16 ? launch_tile<T, 4, 1, 2, 1, RJ>(A, stream) : launch_tile<T, 4, 1, 1, 2, RJ>(A, stream);
  if (segs == 8) return launch_tile<T, 8, 1, 1, 1, RJ>(A, stream);
  if constexpr (sizeof(T) == 4)
    if (segs == 16) return launch_tile<T, 8, 2, 1, 1, RJ>(A, stream);
  return qm_fail(QM_ERR_UNSUPPORTED, "qm_gemm_rows: unsupported k");
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

bool k_covered(int act_dtype, int k) {
  return act_dtype == QM_ACT_BF16 ? (k == 2048 || k == 4096) : (k == 1024 || k == 2048 || k == 4096);
}

template <typename T>
int run_gemm(int m, int n, int k, const void* w, const void* x, int n_seg, const int* seg_rows, void* const* seg_out,
             hipStream_t stream) {
  GemmRowsArgs<T> A = {};
  A.w = static_cast<const T*>(w); A.x = static_cast<const T*>(x);
  A.M = m; A.N = n; A.K = k; A.n_seg = n_seg;
  int end = 0;
  for (int s = 0; s < n_seg; ++s) {
    end += seg_rows[s];
    A.seg_end[s] = end;
    A.seg_out[s] = static_cast<T*>(seg_out[s]);
  }
  if (end != n) return qm_fail(QM_ERR_ARG, "qm_gemm_rows: segment rows must add up to n");
  return launch_rows<T, false>(A, stream);
}

template <typename T>
int run_reinject(int m, int n, int k, const void* w, const void* x, int streams, const void* inject, void* hyper,
                 hipStream_t stream) {
  GemmRowsArgs<T> A = {};
  A.w = static_cast<const T*>(w); A.x = static_cast<const T*>(x);
  A.M = m; A.N = n; A.K = k; A.n_seg = 1; A.seg_end[0] = n;
  A.hyper = static_cast<T*>(hyper); A.inject = static_cast<const T*>(inject); A.streams = streams;
  return launch_rows<T, true>(A, stream);
}

}  // namespace

extern "C" int qm_gemm_rows(int act_dtype, int m, int n, int k, const void* w, const void* x, int n_seg,
                            const int* seg_rows, void* const* seg_out, hipStream_t stream) {
  if (act_dtype != QM_ACT_BF16 && act_dtype != QM_ACT_F32)
    return qm_fail(QM_ERR_DTYPE, "qm_gemm_rows: act_dtype must be QM_ACT_F32 or QM_ACT_BF16");
  if (m <= 0 || m > GR_MAX_M) return qm_fail(QM_ERR_UNSUPPORTED, "qm_gemm_rows: m must be 1..64");
  if (n <= 0 || !k_covered(act_dtype, k))
    return qm_fail(QM_ERR_UNSUPPORTED, "qm_gemm_rows: k must be 2048 or 4096 (bf16), 1024, 2048 or 4096 (f32)");
  if (!w || !x || !seg_rows || !seg_out) return qm_fail(QM_ERR_ARG, "qm_gemm_rows: null pointer");
  if (!aligned16(w) || !aligned16(x)) return qm_fail(QM_ERR_ARG, "qm_gemm_rows: w and x must be 16-byte aligned");
  if (n_seg <= 0 || n_seg > QM_GEMV_MAX_SEG) return qm_fail(QM_ERR_ARG, "qm_gemm_rows: 1..8 output segments");
  for (int s = 0; s < n_seg; ++s)
    if (seg_rows[s] <= 0 || !seg_out[s]) return qm_fail(QM_ERR_ARG, "qm_gemm_rows: empty segment or null output");
  if (act_dtype == QM_ACT_BF16) return run_gemm<bf16_t>(m, n, k, w, x, n_seg, seg_rows, seg_out, stream);
  return run_gemm<float>(m, n, k, w, x, n_seg, seg_rows, seg_out, stream);
}

extern "C" int qm_gemm_rows_reinject(int act_dtype, int m, int n, int k, const void* w, const void* x, int streams,
                                     const void* inject, void* hyper, hipStream_t stream) {
  if (act_dtype != QM_ACT_BF16 && act_dtype != QM_ACT_F32)
    return qm_fail(QM_ERR_DTYPE, "qm_gemm_rows_reinject: act_dtype must be QM_ACT_F32 or QM_ACT_BF16");
  if (m <= 0 || m > GR_MAX_M) return qm_fail(QM_ERR_UNSUPPORTED, "qm_gemm_rows_reinject: m must be 1..64");
  if (n <= 0 || n % 4 || streams <= 0) return qm_fail(QM_ERR_ARG, "qm_gemm_rows_reinject: bad sizes (n a multiple of 4)");
  if (!k_covered(act_dtype, k))
    return qm_fail(QM_ERR_UNSUPPORTED,
                   "qm_gemm_rows_reinject: k must be 2048 or 4096 (bf16), 1024, 2048 or 4096 (f32)");
  if (!w || !x || !inject || !hyper) return qm_fail(QM_ERR_ARG, "qm_gemm_rows_reinject: null pointer");
  if (!aligned16(w) || !aligned16(x) || !aligned16(hyper))
    return qm_fail(QM_ERR_ARG, "qm_gemm_rows_reinject: w, x and hyper must be 16-byte aligned");
  if (act_dtype == QM_ACT_BF16) return run_reinject<bf16_t>(m, n, k, w, x, streams, inject, hyper, stream);
  return run_reinject<float>(m, n, k, w, x, streams, inject, hyper, stream);
}
