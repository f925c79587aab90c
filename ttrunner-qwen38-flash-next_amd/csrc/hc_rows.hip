// The hyper-connection read gate over many token rows, gfx950: the mix of
// hc.hip (reference/model.py:53-77) with both products on the matrix cores.
//
// hc.hip dots each weight row with up to four token rows per workgroup, which
// streams the 10.6 MB of weights once for a few rows; at many rows that means
// every workgroup normalises its rows again and the vector units do all the
// products. Here the down|inject product is split by residual stream: a
// stream's sum of squares and its K range belong together, so a workgroup
// normalises its operand on the way into the product and nothing of
// [rows, streams * hidden] goes through memory. The streams' partial sums
// (float) meet where the low-rank values are formed; the normalised values are
// formed again from hyper where the gate needs them (one multiply-add more per
// element instead of a write and a read).
//
// Few rows: hc_rows_down (a workgroup per 16 weight rows, stream and 16 token
// rows; each of its four waves takes a quarter of the stream, every load in
// flight at once) and hc_rows_up (a workgroup per 16 hidden positions and 16
// token rows, a wave per stream; it forms the low-rank values of its rows from
// the partial sums itself). Latency bound: two launches of about 5 us.
// Many rows: hc_many_down (32 or 64 token rows of a stream per workgroup),
// hc_many_low (the low-rank values, once), hc_many_up (a wave holds the gates
// of all streams for its positions, so the mean needs no exchange). Bound by
// LDS reads and address rate, not by memory (75 MB) or matrix cores (21 GFLOP).
//
// The whole mix, before (hc.hip at every row count) and now, us, rank 320,
// 4 x 2048, weights in cache: bf16 24.7 -> 10.9 at 14 rows, 66.8 -> 15.1 at 64,
// 122 -> 24 at 128, 272 -> 42 at 300, 1761 -> 63 at 2000 (335 TFLOP/s); float
// 35.6 -> 18.2 at 14, 239 -> 56 at 128, 545 -> 123 at 300, 3580 -> 474 at 2000.
//
// Roundings are where hc.hip makes them; only the order of the float sums
// differs.
#include "rows_mma.h"
#include "qwen4mix_internal.h"

namespace {

constexpr int HR_NT = 256;
constexpr int HR_STREAMS = 4;      // the many-rows kernels' stream count

template <typename T>
struct HrArgs {
  const T* hyper;      // [M, streams * hidden]
  const float* norm_w; // [streams * hidden]
  const T* w_di;       // [n_rows, streams * hidden]
  const T* w_up;       // [streams * hidden, rank]
  float* part;         // [streams, M, np] partial down|inject products
  float* rstd;         // [M, streams]
  T* low;              // [M, rank] (many rows)
  T* mixed;            // [M, hidden]
  T* inject;           // [M, streams] or null
  int M, streams, hidden, rank, n_rows, np;
  float eps;
};

// sigmoid of a gate, a value rounded to T, under a rounding to T: in bf16 by the
// hardware exponential and reciprocal (five instructions where the precise chain
// takes about forty, and there is one per element of [rows, streams * hidden]:
// mix and reinjection of 2000 rows 79.1 us, with the chain 84.5), in float by the
// precise chain. Unrounded, the short form is up to 3.4e-6 (at x = -80) from the sigmoid
// where the chain is 1.2e-7; rounded, the two are the same for each of the 65536
// values that x can have. The denominator's 2^-32 keeps the reciprocal of the
// largest out of the denormals, which the hardware's flushes.
template <typename T> __device__ __forceinline__ float gate_sigmoid(float x);
template <> __device__ __forceinline__ float gate_sigmoid<bf16_t>(float x) {
  const float e = __builtin_amdgcn_exp2f(-1.44269504f * x);
  return __builtin_amdgcn_rcpf(fmaf(e, 0x1p-32f, 0x1p-32f)) * 0x1p-32f;
}
template <> __device__ __forceinline__ float gate_sigmoid<float>(float x) { return sigmoid_f(x); }

// low-rank value (or inject weight) from the summed down|inject product
template <typename T>
__device__ __forceinline__ float low_value(float lin, float streams) {
  return silu_f(Act<T>::round(div_rn(Act<T>::round(lin), streams)));
}
template <typename T>
__device__ __forceinline__ float inject_value(float lin, float streams) {
  return 2.0f * Act<T>::round(sigmoid_f(Act<T>::round(div_rn(Act<T>::round(lin), streams))));
}

// one unit normalised: round_T((x * r) * w)
template <typename T>
__device__ __forceinline__ uint4 norm_unit(const uint4& x, float r, const float* w) {
  constexpr int VE = Chunk<T>::VE;
  float y[VE];
#pragma unroll
  for (int i = 0; i < VE; ++i) y[i] = mul_rn(mul_rn(Chunk<T>::get(x, i), r), w[i]);
  return Chunk<T>::pack(y);
}

template <typename T>
__device__ __forceinline__ float unit_sumsq(const uint4& x, float acc) {
#pragma unroll
  for (int i = 0; i < Chunk<T>::VE; ++i) {
    const float v = Chunk<T>::get(x, i);
    acc = fmaf(v, v, acc);
  }
  return acc;
}

// ---------------------------------------------------------------------------
// few rows: grid (ceil(n_rows / 16), streams, ceil(M / 16)); NS = k-steps of a
// wave's quarter of the stream. One token row per lane column.
template <typename T, int NS>
__global__ __launch_bounds__(HR_NT) void hc_rows_down_kernel(HrArgs<T> A) {
  constexpr int VE = Chunk<T>::VE;
  constexpr bool LINES = NS % 16 == 0;                // 1 KB row segments, turned into operands through LDS
  constexpr int NG = LINES ? NS / 16 : 1;
  __shared__ float s_ss[4][16];
  __shared__ f32x4_t s_acc[3][64];
  __shared__ float4 s_nw[NS * 4 * VE];                // the stream's norm weights
  __shared__ uint4 s_rows[LINES ? 4 : 1][LINES ? 16 * ROW_US : 1];
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int g4 = lane >> 4, r16 = lane & 15;
  const int n0 = blockIdx.x * 16, s = blockIdx.y, m0 = blockIdx.z * 16;
  const long K = (long)A.streams * A.hidden;
  const int k0 = s * A.hidden + wid * NS * 4 * VE;    // the wave's quarter of the stream
  u32x4_t x[NS], w[NS];
  if constexpr (LINES) {
    u32x4_t xr[NG][16], wr[NG][16];
#pragma unroll
    for (int q = 0; q < NG; ++q)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        xr[q][r] = *reinterpret_cast<const u32x4_t*>(A.hyper + (long)min(m0 + r, A.M - 1) * K + k0 + (q * 64 + lane) * VE);
#pragma unroll
    for (int q = 0; q < NG; ++q)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        wr[q][r] = *reinterpret_cast<const u32x4_t*>(A.w_di + (long)min(n0 + r, A.n_rows - 1) * K + k0 + (q * 64 + lane) * VE);
    const float4* nwp = reinterpret_cast<const float4*>(A.norm_w + (long)s * A.hidden);
#pragma unroll
    for (int i = 0; i < NS * 4 * VE / HR_NT; ++i) s_nw[tid + HR_NT * i] = nwp[tid + HR_NT * i];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < NG; ++q) {
      u32x4_t f[16];
      to_frags(s_rows[wid], xr[q], lane, r16, g4, f);
#pragma unroll
      for (int i = 0; i < 16; ++i) x[16 * q + i] = f[i];
    }
#pragma unroll
    for (int q = 0; q < NG; ++q) {
      u32x4_t f[16];
      to_frags(s_rows[wid], wr[q], lane, r16, g4, f);
#pragma unroll
      for (int i = 0; i < 16; ++i) w[16 * q + i] = f[i];
    }
  } else {
    const T* xp = A.hyper + (long)min(m0 + r16, A.M - 1) * K + k0 + g4 * VE;
    const T* wp = A.w_di + (long)min(n0 + r16, A.n_rows - 1) * K + k0 + g4 * VE;
#pragma unroll
    for (int i = 0; i < NS; ++i) x[i] = *reinterpret_cast<const u32x4_t*>(xp + i * 4 * VE);
#pragma unroll
    for (int i = 0; i < NS; ++i) w[i] = *reinterpret_cast<const u32x4_t*>(wp + i * 4 * VE);
    const float4* nwp = reinterpret_cast<const float4*>(A.norm_w + (long)s * A.hidden);
#pragma unroll
    for (int i = 0; i < (NS * 4 * VE + HR_NT - 1) / HR_NT; ++i)
      if (tid + HR_NT * i < NS * 4 * VE) s_nw[tid + HR_NT * i] = nwp[tid + HR_NT * i];
    __builtin_amdgcn_sched_barrier(0);
  }

  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < NS; ++i) ss = unit_sumsq<T>(__builtin_bit_cast(uint4, x[i]), ss);
  ss = xor32_sum(xor16_sum(ss));
  if (lane < 16) s_ss[wid][lane] = ss;
  __syncthreads();
  ss = (s_ss[0][r16] + s_ss[1][r16]) + (s_ss[2][r16] + s_ss[3][r16]);
  const float r = rsqrt_rn(add_rn(div_rn(ss, (float)A.hidden), A.eps));
  if (blockIdx.x == 0 && wid == 0 && lane < 16 && m0 + lane < A.M) A.rstd[(long)(m0 + lane) * A.streams + s] = r;

  RowAcc<T> acc;
#pragma unroll
  for (int i = 0; i < NS; ++i) {
    float nw[VE];
#pragma unroll
    for (int v = 0; v < VE / 4; ++v) {
      const float4 f = s_nw[((wid * NS + i) * 4 + g4) * (VE / 4) + v];
      nw[4 * v] = f.x; nw[4 * v + 1] = f.y; nw[4 * v + 2] = f.z; nw[4 * v + 3] = f.w;
    }
    acc.step(__builtin_bit_cast(uint4, w[i]), norm_unit<T>(__builtin_bit_cast(uint4, x[i]), r, nw));
    if (i % 4 == 3) acc.block();
  }
  // the four quarters of the stream meet in wave 0: lane holds weight rows
  // n0 + 4 g4 .. + 3 of token row m0 + r16
  const f32x4_t a = acc.sum();
  if (wid) s_acc[wid - 1][lane] = a;
  __syncthreads();
  if (wid == 0 && m0 + r16 < A.M) {
    const f32x4_t t = (a + s_acc[0][lane]) + (s_acc[1][lane] + s_acc[2][lane]);
    float* o = A.part + ((long)s * A.M + m0 + r16) * A.np + n0 + 4 * g4;
    *reinterpret_cast<float4*>(o) = make_float4(t[0], t[1], t[2], t[3]);
  }
}

// few rows: grid (hidden / 16, ceil(M / 16)), a wave per stream; NR = k-steps
// of the rank.
template <typename T, int NR>
__global__ __launch_bounds__(HR_NT) void hc_rows_up_kernel(HrArgs<T> A) {
  constexpr int VE = Chunk<T>::VE;
  constexpr int RANK = NR * 4 * VE;
  constexpr int LS = RANK + VE;                      // LDS row stride of the low-rank tile: one unit of padding
  __shared__ __attribute__((aligned(16))) T s_low[16 * LS];
  static_assert(HR_NT == 64 * HR_STREAMS && 16 * (RANK / 4) % HR_NT == 0, "a wave per stream, whole rounds");
  __shared__ float s_g[HR_STREAMS][16][17];
  const int tid = threadIdx.x, lane = tid & 63, s = tid >> 6;
  const int g4 = lane >> 4, r16 = lane & 15;
  const int h0 = blockIdx.x * 16, m0 = blockIdx.y * 16;
  const long K = (long)A.streams * A.hidden;
  constexpr float fs = HR_STREAMS;
  // this wave's up rows (16 rows are one run of memory; operands through LDS),
  // and what its gates multiply
  __shared__ uint4 s_up[HR_STREAMS][16 * (4 * NR + 1)];
  u32x4_t w[NR];
  const T* wp = A.w_up + ((long)s * A.hidden + h0) * RANK;
#pragma unroll
  for (int i = 0; i < NR; ++i) w[i] = *reinterpret_cast<const u32x4_t*>(wp + (i * 64 + lane) * VE);
  const int mc = min(m0 + r16, A.M - 1);
  const int col = s * A.hidden + h0 + 4 * g4;
  float hv[4], nw[4];
  load_act4(A.hyper + (long)mc * K + col, hv);
  load_act4(A.norm_w + col, nw);
  const float r = A.rstd[(long)mc * A.streams + s];

  // low-rank values of the 16 rows: the streams' partial sums in order, every
  // load of a thread requested before the first is used
  constexpr int PER = 16 * (RANK / 4) / HR_NT;
  float4 p[PER][HR_STREAMS];
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int e = tid + HR_NT * u;
    const int m = e / (RANK / 4), j = 4 * (e - m * (RANK / 4));
#pragma unroll
    for (int q = 0; q < HR_STREAMS; ++q)
      p[u][q] = *reinterpret_cast<const float4*>(A.part + ((long)q * A.M + min(m0 + m, A.M - 1)) * A.np + j);
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int e = tid + HR_NT * u;
    const int m = e / (RANK / 4), j = 4 * (e - m * (RANK / 4));
    const float v[4] = {low_value<T>(((p[u][0].x + p[u][1].x) + p[u][2].x) + p[u][3].x, fs),
                        low_value<T>(((p[u][0].y + p[u][1].y) + p[u][2].y) + p[u][3].y, fs),
                        low_value<T>(((p[u][0].z + p[u][1].z) + p[u][2].z) + p[u][3].z, fs),
                        low_value<T>(((p[u][0].w + p[u][1].w) + p[u][2].w) + p[u][3].w, fs)};
    store_act4(s_low + m * LS + j, v);
  }
  if (A.inject && blockIdx.x == 0 && tid < 16 * A.streams) {
    const int m = tid / A.streams, q = tid - m * A.streams;
    if (m0 + m < A.M) {
      const float* p = A.part + (long)(m0 + m) * A.np + A.rank + q;
      float t = p[0];
      for (int u = 1; u < A.streams; ++u) t += p[(long)u * A.M * A.np];
      Act<T>::store(A.inject, (long)(m0 + m) * A.streams + q, inject_value<T>(t, fs));
    }
  }
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    const int e = i * 64 + lane, row = e / (4 * NR);
    *reinterpret_cast<u32x4_t*>(&s_up[s][row * (4 * NR + 1) + e - row * (4 * NR)]) = w[i];
  }
  __syncthreads();
  RowAcc<T> acc;
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    acc.step(s_up[s][r16 * (4 * NR + 1) + i * 4 + g4], *reinterpret_cast<const uint4*>(s_low + r16 * LS + (i * 4 + g4) * VE));
    if (i % 4 == 3) acc.block();
  }
  // lane: hidden positions h0 + 4 g4 + i of token row r16
  const f32x4_t lin = acc.sum();
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float n = Act<T>::round(mul_rn(mul_rn(hv[i], r), nw[i]));
    s_g[s][4 * g4 + i][r16] = Act<T>::round(Act<T>::round(gate_sigmoid<T>(Act<T>::round(lin[i]))) * n);
  }
  __syncthreads();
  const int h = tid & 15, mo = tid >> 4;
  if (m0 + mo < A.M) {
    float sum = 0.f;
#pragma unroll
    for (int q = 0; q < HR_STREAMS; ++q) sum += s_g[q][h][mo];
    Act<T>::store(A.mixed, (long)(m0 + mo) * A.hidden + h0 + h, div_rn(sum, fs));
  }
}

// ---------------------------------------------------------------------------
// many rows: grid (ceil(M / 64), streams, ceil(n_rows / 128)). The stream's 64
// rows pass in slices of 32 units: normalised into LDS, then eight k-steps of
// (4 token tiles) x (2 weight tiles) per wave, the weights straight from L2.
// A slice's loads (96 KB a workgroup) are in flight during the slice before.
template <typename T>
__global__ __launch_bounds__(HR_NT) void hc_many_down_kernel(HrArgs<T> A) {
  constexpr int VE = Chunk<T>::VE;
  constexpr int SU = 32;                              // units of a row per slice
  constexpr int US = SU + 1;                          // LDS row stride: one unit of padding
  __shared__ uint4 s_x[2][64 * US];
  __shared__ float s_r[64];
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int g4 = lane >> 4, r16 = lane & 15;
  const int m0 = blockIdx.x * 64, s = blockIdx.y, n0 = blockIdx.z * 128 + wid * 32;
  const long K = (long)A.streams * A.hidden;
  const int n_slice = A.hidden / (SU * VE), n_run = A.hidden / (16 * VE);
  const T* xs = A.hyper + (long)s * A.hidden;

  // sums of squares: 16 lanes per row, 4 rows per wave at a time
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = 16 * wid + 4 * i + g4;
    const T* p = xs + (long)min(m0 + row, A.M - 1) * K + r16 * VE;
    float ss = 0.f;
    for (int c = 0; c < n_run; c += 4) {              // n_run is a multiple of 4
      uint4 q[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) q[u] = *reinterpret_cast<const uint4*>(p + (long)(c + u) * 16 * VE);
#pragma unroll
      for (int u = 0; u < 4; ++u) ss = unit_sumsq<T>(q[u], ss);
    }
    ss = row16_sum(ss);
    const float r = rsqrt_rn(add_rn(div_rn(ss, (float)A.hidden), A.eps));
    if (r16 == 0) {
      s_r[row] = r;
      if (blockIdx.z == 0 && m0 + row < A.M) A.rstd[(long)(m0 + row) * A.streams + s] = r;
    }
  }
  __syncthreads();

  // a thread's units of a slice: unit tid % 32 of rows tid / 32 + 8 i
  const int xu = tid & 31, xr = tid >> 5;
  const T* xp[8];
  float rr[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    xp[i] = xs + (long)min(m0 + xr + 8 * i, A.M - 1) * K + xu * VE;
    rr[i] = s_r[xr + 8 * i];
  }
  const float* nwp = A.norm_w + (long)s * A.hidden + xu * VE;
  const T* wp[2];
#pragma unroll
  for (int t = 0; t < 2; ++t) wp[t] = A.w_di + (long)min(n0 + 16 * t + r16, A.n_rows - 1) * K + (long)s * A.hidden + g4 * VE;
  uint4 xq[8], wq[2][8];
  float nw[VE];
  auto fetch = [&](int c) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 8; ++i) xq[i] = *reinterpret_cast<const uint4*>(xp[i] + (long)c * SU * VE);
#pragma unroll
    for (int v = 0; v < VE / 4; ++v) {
      const float4 f = *reinterpret_cast<const float4*>(nwp + (long)c * SU * VE + 4 * v);
      nw[4 * v] = f.x; nw[4 * v + 1] = f.y; nw[4 * v + 2] = f.z; nw[4 * v + 3] = f.w;
    }
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int u = 0; u < 8; ++u) wq[t][u] = *reinterpret_cast<const uint4*>(wp[t] + ((long)c * SU + 4 * u) * VE);
  };
  RowAcc<T> acc[4][2];
  fetch(0);
  for (int c = 0; c < n_slice; ++c) {
    uint4* buf = s_x[c & 1];
#pragma unroll
    for (int i = 0; i < 8; ++i) buf[(xr + 8 * i) * US + xu] = norm_unit<T>(xq[i], rr[i], nw);
    uint4 wc[2][8];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int u = 0; u < 8; ++u) wc[t][u] = wq[t][u];
    __syncthreads();
    fetch(min(c + 1, n_slice - 1));
#pragma unroll
    for (int u = 0; u < 8; ++u) {
#pragma unroll
      for (int mt = 0; mt < 4; ++mt) {
        const uint4 a = buf[(16 * mt + r16) * US + 4 * u + g4];
#pragma unroll
        for (int t = 0; t < 2; ++t) acc[mt][t].step(wc[t][u], a);
      }
      if (u % 4 == 3)
#pragma unroll
        for (int mt = 0; mt < 4; ++mt)
#pragma unroll
          for (int t = 0; t < 2; ++t) acc[mt][t].block();
    }
  }
#pragma unroll
  for (int mt = 0; mt < 4; ++mt) {
    const int m = m0 + 16 * mt + r16;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int n = n0 + 16 * t + 4 * g4;
      const f32x4_t v = acc[mt][t].sum();
      if (m < A.M && n < A.np)
        *reinterpret_cast<float4*>(A.part + ((long)s * A.M + m) * A.np + n) = make_float4(v[0], v[1], v[2], v[3]);
    }
  }
}

// bf16, hidden 2048: 32 rows of a stream against every weight row; grid
// (ceil(M / 32), streams), 8 waves. The rows pass in slices of 128 columns,
// normalised into LDS; the weights pass through LDS in slices of 64 columns
// (128 bytes of each row, so that a wave's loads are whole lines: read
// straight into operands, 16 rows of 64 bytes per load, the same product took
// 46 us at 2000 rows), two slices in flight. Wave w < 7 takes weight rows
// 48 w .. + 47.
constexpr int HD_NT = 512, HD_ROWS = 32;
constexpr int HD_WROWS = 336, HD_WU = HD_WROWS * 8;       // weight rows, units of a slice
constexpr int HD_XS = 17;                                 // LDS row stride of the x slice, units
constexpr int HD_PER = (HD_WU + HD_NT - 1) / HD_NT;
constexpr size_t HD_LDS = (size_t)(2 * HD_WU + 2 * HD_ROWS * HD_XS) * 16;

__global__ __launch_bounds__(HD_NT) void hc_many_down_kept_kernel(HrArgs<bf16_t> A) {
  constexpr int VE = 8, NT3 = 3, NX = 16;                 // NX slices of 128 columns
  extern __shared__ uint4 lds[];
  uint4* s_w = lds;                                       // [2][HD_WU], unit u of row n at n * 8 + (u ^ (n & 7))
  uint4* s_x = lds + 2 * HD_WU;                           // [2][32][HD_XS]
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int g4 = lane >> 4, r16 = lane & 15;
  const int m0 = blockIdx.x * HD_ROWS, s = blockIdx.y, n0 = wid * 16 * NT3;
  const long K = (long)A.streams * A.hidden;
  // 16 lanes per row: units r16 + 16 i
  const int row = tid >> 4;
  const bf16_t* xp = A.hyper + (long)min(m0 + row, A.M - 1) * K + (long)s * A.hidden + r16 * VE;
  const float* nwp = A.norm_w + (long)s * A.hidden + r16 * VE;
  // the thread's weight units of a slice: unit tid % 8 of rows tid / 8 + 64 i
  const bf16_t* wp = A.w_di + (long)s * A.hidden + (tid & 7) * VE;
  long wr[HD_PER];
#pragma unroll
  for (int i = 0; i < HD_PER; ++i) wr[i] = (long)min((tid >> 3) + 64 * i, A.n_rows - 1) * K;
  const int wo = (tid >> 3) * 8 + ((tid & 7) ^ ((tid >> 3) & 7));      // + 512 i
  u32x4_t wq0[HD_PER], wq1[HD_PER];
  auto fetch_w = [&](int c, u32x4_t (&q)[HD_PER]) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < HD_PER; ++i) q[i] = *reinterpret_cast<const u32x4_t*>(wp + wr[i] + c * 8 * VE);
  };
  uint4 xq;
  float4 na, nb;
  auto fetch_x = [&](int c) __attribute__((always_inline)) {
    xq = *reinterpret_cast<const uint4*>(xp + c * 16 * VE);
    na = *reinterpret_cast<const float4*>(nwp + c * 16 * VE);
    nb = *reinterpret_cast<const float4*>(nwp + c * 16 * VE + 4);
  };
  fetch_w(0, wq0);
  fetch_w(1, wq1);
  float ss = 0.f;
  {
    uint4 x[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) x[i] = *reinterpret_cast<const uint4*>(xp + i * 16 * VE);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 16; ++i) ss = unit_sumsq<bf16_t>(x[i], ss);
  }
  fetch_x(0);
  ss = row16_sum(ss);
  const float r = rsqrt_rn(add_rn(div_rn(ss, (float)A.hidden), A.eps));
  if (r16 == 0 && m0 + row < A.M) A.rstd[(long)(m0 + row) * A.streams + s] = r;
  f32x4_t acc[2][NT3];
#pragma unroll
  for (int mt = 0; mt < 2; ++mt)
#pragma unroll
    for (int t = 0; t < NT3; ++t) acc[mt][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  // one slice's weights to LDS, the slice two later requested, the products. A
  // buffer is rewritten two slices later, behind the barrier of the one between
  auto slice = [&](int c, int h, const uint4* xs, u32x4_t (&wq)[HD_PER]) __attribute__((always_inline)) {
    uint4* ws = s_w + h * HD_WU;
#pragma unroll
    for (int i = 0; i < HD_PER; ++i)
      if (i + 1 < HD_PER || (tid >> 3) + 64 * i < HD_WROWS) *reinterpret_cast<u32x4_t*>(ws + wo + 512 * i) = wq[i];
    fetch_w(min(c + 2, 2 * NX - 1), wq);
    __syncthreads();
    if (n0 < HD_WROWS) {
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        uint4 a[2];
#pragma unroll
        for (int mt = 0; mt < 2; ++mt) a[mt] = xs[(16 * mt + r16) * HD_XS + h * 8 + 4 * u + g4];
#pragma unroll
        for (int t = 0; t < NT3; ++t) {
          const uint4 w = ws[(n0 + 16 * t + r16) * 8 + ((4 * u + g4) ^ (r16 & 7))];
#pragma unroll
          for (int mt = 0; mt < 2; ++mt)
            acc[mt][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, w),
                                                                 __builtin_bit_cast(bf16x8_t, a[mt]), acc[mt][t], 0, 0, 0);
        }
      }
    }
  };
#pragma unroll 1
  for (int c = 0; c < NX; ++c) {
    uint4* xs = s_x + (c & 1) * HD_ROWS * HD_XS;
    const float nw[8] = {na.x, na.y, na.z, na.w, nb.x, nb.y, nb.z, nb.w};
    xs[row * HD_XS + r16] = norm_unit<bf16_t>(xq, r, nw);
    fetch_x(min(c + 1, NX - 1));
    slice(2 * c, 0, xs, wq0);
    slice(2 * c + 1, 1, xs, wq1);
  }
#pragma unroll
  for (int mt = 0; mt < 2; ++mt) {
    const int m = m0 + 16 * mt + r16;
#pragma unroll
    for (int t = 0; t < NT3; ++t) {
      const int n = n0 + 16 * t + 4 * g4;
      const f32x4_t v = acc[mt][t];
      if (m < A.M && n < A.np)
        *reinterpret_cast<float4*>(A.part + ((long)s * A.M + m) * A.np + n) = make_float4(v[0], v[1], v[2], v[3]);
    }
  }
}

// the low-rank values and inject weights from the streams' partial sums: a
// thread per 4 columns of a row
template <typename T>
__global__ __launch_bounds__(HR_NT) void hc_many_low_kernel(HrArgs<T> A) {
  const int per = A.np / 4;
  const long e = (long)blockIdx.x * HR_NT + threadIdx.x;
  const long m = e / per;
  if (m >= A.M) return;
  const int j = 4 * (int)(e - m * per);
  const float fs = (float)A.streams;
  float4 t = {0.f, 0.f, 0.f, 0.f};
  const float* p = A.part + m * A.np + j;
  float4 q[HR_STREAMS];
#pragma unroll
  for (int s = 0; s < HR_STREAMS; ++s) q[s] = *reinterpret_cast<const float4*>(p + (long)s * A.M * A.np);
  t = q[0];
#pragma unroll
  for (int s = 1; s < HR_STREAMS; ++s) { t.x += q[s].x; t.y += q[s].y; t.z += q[s].z; t.w += q[s].w; }
  const float v[4] = {t.x, t.y, t.z, t.w};
  if (j < A.rank) {
    const float o[4] = {low_value<T>(v[0], fs), low_value<T>(v[1], fs), low_value<T>(v[2], fs), low_value<T>(v[3], fs)};
    store_act4(A.low + m * A.rank + j, o);
  } else if (A.inject) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (j + i < A.rank + A.streams)
        Act<T>::store(A.inject, m * A.streams + (j + i - A.rank), inject_value<T>(v[i], fs));
  }
}

// many rows, float: grid (hidden / 64, ceil(M / 32)); wave w: hidden positions
// h0 + 16 w .. + 15 of every stream for the 32 rows
__global__ __launch_bounds__(HR_NT) void hc_many_up_kernel(HrArgs<float> A) {
  using T = float;
  constexpr int MT = 2;
  constexpr int VE = Chunk<T>::VE;
  constexpr int ST = HR_STREAMS;
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int g4 = lane >> 4, r16 = lane & 15;
  const int h0 = blockIdx.x * 64 + 16 * wid, m0 = blockIdx.y * 16 * MT;
  const long K = (long)ST * A.hidden;
  const T* wp[ST];
  const T* xp[MT];
#pragma unroll
  for (int s = 0; s < ST; ++s) wp[s] = A.w_up + ((long)s * A.hidden + h0 + r16) * A.rank + g4 * VE;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) xp[mt] = A.low + (long)min(m0 + 16 * mt + r16, A.M - 1) * A.rank + g4 * VE;
  RowAcc<T> acc[ST][MT];
  uint4 wn[ST], xn[MT];
  const int n_step = A.rank / (4 * VE);
#pragma unroll
  for (int s = 0; s < ST; ++s) wn[s] = *reinterpret_cast<const uint4*>(wp[s]);
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) xn[mt] = *reinterpret_cast<const uint4*>(xp[mt]);
  for (int i = 0; i < n_step; ++i) {
    uint4 w[ST], x[MT];
#pragma unroll
    for (int s = 0; s < ST; ++s) w[s] = wn[s];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) x[mt] = xn[mt];
    const int nx = min(i + 1, n_step - 1) * 4 * VE;
#pragma unroll
    for (int s = 0; s < ST; ++s) wn[s] = *reinterpret_cast<const uint4*>(wp[s] + nx);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) xn[mt] = *reinterpret_cast<const uint4*>(xp[mt] + nx);
#pragma unroll
    for (int s = 0; s < ST; ++s)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        acc[s][mt].step(w[s], x[mt]);
        if (i % 4 == 3) acc[s][mt].block();
      }
  }
  // lane: positions h0 + 4 g4 + i of token row m0 + 16 mt + r16, every stream
  const int h = h0 + 4 * g4;
  float nw[ST][4];
#pragma unroll
  for (int s = 0; s < ST; ++s) load_act4(A.norm_w + (long)s * A.hidden + h, nw[s]);
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int m = m0 + 16 * mt + r16;
    const int mc = min(m, A.M - 1);
    float hv[ST][4], r[ST];
#pragma unroll
    for (int s = 0; s < ST; ++s) {
      load_act4(A.hyper + (long)mc * K + (long)s * A.hidden + h, hv[s]);
      r[s] = A.rstd[(long)mc * ST + s];
    }
    float sum[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < ST; ++s) {
      const f32x4_t lin = acc[s][mt].sum();
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float n = Act<T>::round(mul_rn(mul_rn(hv[s][i], r[s]), nw[s][i]));
        sum[i] += Act<T>::round(Act<T>::round(gate_sigmoid<T>(Act<T>::round(lin[i]))) * n);
      }
    }
    if (m < A.M) {
      const float o[4] = {div_rn(sum[0], (float)ST), div_rn(sum[1], (float)ST), div_rn(sum[2], (float)ST),
                          div_rn(sum[3], (float)ST)};
      store_act4(A.mixed + (long)m * A.hidden + h, o);
    }
  }
}

// bf16: the up rows of 32 hidden positions (every stream, 80 KB) stay in LDS
// while the row tiles of a group pass; grid (hidden / 32, row groups), 16
// waves, wave w takes tiles w, w + 16, ... of its group for all 32 positions
// (the low-rank rows, loads of 16 rows x 64 bytes, are read once per 32
// positions; once per 16 the kernel took 35 us at 2000 rows, now 18 alone and
// 25 after the down product). Four waves a SIMD, so that one wave's loads
// (hyper comes from HBM) run under the others' products and gates. Row r of up
// tile j is position 8 (r / 4) + 4 j + r % 4, so that a lane ends up with 8
// consecutive positions of a row: 16-byte loads of hyper and stores of mixed.
constexpr int HU_NT = 1024, HU_H = 32;

template <int NR>
__global__ __launch_bounds__(HU_NT) void hc_many_up_kept_kernel(HrArgs<bf16_t> A) {
  constexpr int VE = 8, ST = HR_STREAMS, RANK = NR * 4 * VE;
  constexpr int UR = NR * 4, US = UR + 1;                 // units of an up row, LDS stride
  extern __shared__ uint4 s_w[];                          // [ST][2][16][US], then the norm weights
  float4* s_nw = reinterpret_cast<float4*>(s_w + ST * HU_H * US);   // [ST][HU_H / 4]
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int g4 = lane >> 4, r16 = lane & 15;
  // neighbouring positions on one die (they share lines of hyper)
  const int hb = xcd_remap(blockIdx.x, gridDim.x) * HU_H;
  const int h = hb + 8 * g4;
  const long K = (long)ST * A.hidden;
  const int n_tile = (A.M + 15) / 16;
  for (int e = tid; e < ST * HU_H * UR; e += HU_NT) {
    const int row = e / UR, u = e - row * UR;
    const int s = row / HU_H, p = row - s * HU_H;         // position p is row 4 (p / 8) + p % 4 of tile p / 4 % 2
    s_w[((s * 2 + (p >> 2 & 1)) * 16 + 4 * (p >> 3) + (p & 3)) * US + u] =
        *reinterpret_cast<const uint4*>(A.w_up + ((long)s * A.hidden + hb + p) * RANK + u * VE);
  }
  if (tid < ST * HU_H / 4)
    s_nw[tid] = *reinterpret_cast<const float4*>(A.norm_w + (long)(tid / (HU_H / 4)) * A.hidden + hb + 4 * (tid % (HU_H / 4)));
  __syncthreads();
  for (int t = blockIdx.y * 16 + wid; t < n_tile; t += 16 * gridDim.y) {
    const int m = 16 * t + r16, mc = min(m, A.M - 1);
    uint4 x[NR], hv[ST];
    const bf16_t* p = A.low + (long)mc * RANK + g4 * VE;
#pragma unroll
    for (int i = 0; i < NR; ++i) x[i] = *reinterpret_cast<const uint4*>(p + i * 4 * VE);
#pragma unroll
    for (int s = 0; s < ST; ++s) hv[s] = *reinterpret_cast<const uint4*>(A.hyper + mc * K + (long)s * A.hidden + h);
    const float4 rs = *reinterpret_cast<const float4*>(A.rstd + (long)mc * ST);
    const float r[ST] = {rs.x, rs.y, rs.z, rs.w};
    float sum[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < ST; ++s) {
      f32x4_t acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
      for (int i = 0; i < NR; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const uint4 w = s_w[((s * 2 + j) * 16 + r16) * US + i * 4 + g4];
          acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, w),
                                                           __builtin_bit_cast(bf16x8_t, x[i]), acc[j], 0, 0, 0);
        }
      const uint4 y = norm_unit<bf16_t>(hv[s], r[s], reinterpret_cast<const float*>(s_nw + s * (HU_H / 4) + 2 * g4));
#pragma unroll
      for (int q = 0; q < 8; ++q)
        sum[q] += Act<bf16_t>::round(Act<bf16_t>::round(gate_sigmoid<bf16_t>(Act<bf16_t>::round(acc[q / 4][q % 4]))) *
                                     Chunk<bf16_t>::get(y, q));
      // a stream at a time: all up rows at once would not fit the registers
      __builtin_amdgcn_sched_barrier(0);
    }
    if (m < A.M) {
      float o[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) o[q] = sum[q] * 0.25f;    // / streams, exact
      *reinterpret_cast<uint4*>(A.mixed + (long)m * A.hidden + h) = Chunk<bf16_t>::pack(o);
    }
  }
}

// ---------------------------------------------------------------------------

struct HrLayout {
  size_t part, rstd, low, total;
  int np;
};

HrLayout hr_layout(const qm_hc_geom& g) {
  const size_t es = g.act_dtype == QM_ACT_BF16 ? 2 : 4;
  HrLayout L;
  L.np = (g.rank + g.streams + 15) / 16 * 16;
  L.part = 0;
  L.rstd = qm_align256((size_t)g.streams * g.rows * L.np * sizeof(float));
  L.low = L.rstd + qm_align256((size_t)g.rows * g.streams * sizeof(float));
  L.total = L.low + qm_align256((size_t)g.rows * g.rank * es);
  return L;
}

// Rows up to which the few-rows kernels are faster (their weights are read once
// per 16 rows, the many-rows kernels start at a fixed cost of about 37 / 150 us):
// us for the mix, few / many: bf16 24 / 39 at 128 rows, 31 / 42 at 192, 47 / 42
// at 256 (the many-rows figures flat up to 300); float 123 / 185 at 300, 195 / 230 at 512
template <typename T> struct HrFew;
template <> struct HrFew<bf16_t> { static constexpr int ROWS = 192; };
template <> struct HrFew<float> { static constexpr int ROWS = 512; };

template <typename T>
int run_rows(const qm_hc_geom& g, int as_rows, const void* hyper, const float* norm_w, const void* w_di, int with_inject,
             const void* w_up, void* mixed, void* inject, void* ws, hipStream_t stream) {
  const HrLayout L = hr_layout(g);
  char* base = static_cast<char*>(ws);
  HrArgs<T> A;
  A.hyper = static_cast<const T*>(hyper); A.norm_w = norm_w;
  A.w_di = static_cast<const T*>(w_di); A.w_up = static_cast<const T*>(w_up);
  A.part = reinterpret_cast<float*>(base + L.part); A.rstd = reinterpret_cast<float*>(base + L.rstd);
  A.low = reinterpret_cast<T*>(base + L.low);
  A.mixed = static_cast<T*>(mixed); A.inject = with_inject ? static_cast<T*>(inject) : nullptr;
  A.M = g.rows; A.streams = g.streams; A.hidden = g.hidden; A.rank = g.rank;
  A.n_rows = g.rank + (with_inject ? g.streams : 0); A.np = L.np; A.eps = g.eps;
  const int n_tiles = (A.n_rows + 15) / 16;
  if (as_rows <= HrFew<T>::ROWS) {
    constexpr int VE = Chunk<T>::VE;
    const dim3 gd(n_tiles, g.streams, (g.rows + 15) / 16), gu(g.hidden / 16, (g.rows + 15) / 16);
    if (g.hidden == 2048)
      hipLaunchKernelGGL((hc_rows_down_kernel<T, 2048 / (16 * VE)>), gd, dim3(HR_NT), 0, stream, A);
    else
      hipLaunchKernelGGL((hc_rows_down_kernel<T, 2560 / (16 * VE)>), gd, dim3(HR_NT), 0, stream, A);
    QM_CHECK_LAUNCH();
    hipLaunchKernelGGL((hc_rows_up_kernel<T, 320 / (4 * VE)>), gu, dim3(HR_NT), 0, stream, A);
    QM_CHECK_LAUNCH();
    return QM_OK;
  }
  bool kept = false;
  if constexpr (sizeof(T) == 2) {
    kept = g.hidden == 2048 && L.np == HD_WROWS;
    if (kept) {
      hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(hc_many_down_kept_kernel),
                                         hipFuncAttributeMaxDynamicSharedMemorySize, (int)HD_LDS);
      if (e != hipSuccess) return qm_fail(QM_ERR_LAUNCH, hipGetErrorString(e));
      hipLaunchKernelGGL(hc_many_down_kept_kernel, dim3((g.rows + HD_ROWS - 1) / HD_ROWS, g.streams), dim3(HD_NT),
                         HD_LDS, stream, A);
    }
  }
  if (!kept)
    hipLaunchKernelGGL(hc_many_down_kernel<T>, dim3((g.rows + 63) / 64, g.streams, (A.n_rows + 127) / 128), dim3(HR_NT), 0,
                     stream, A);
  QM_CHECK_LAUNCH();
  const long items = (long)g.rows * (L.np / 4);
  hipLaunchKernelGGL(hc_many_low_kernel<T>, dim3((unsigned)((items + HR_NT - 1) / HR_NT)), dim3(HR_NT), 0, stream, A);
  QM_CHECK_LAUNCH();
  if constexpr (sizeof(T) == 2) {
    // one workgroup per compute unit: 64 or 80 position groups x 4 or 3 row groups
    constexpr size_t lds = (size_t)HR_STREAMS * HU_H * (41 * 16 + sizeof(float));
    const int sets = (g.rows + 255) / 256, groups = 256 / (g.hidden / HU_H);
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(hc_many_up_kept_kernel<10>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return qm_fail(QM_ERR_LAUNCH, hipGetErrorString(e));
    hipLaunchKernelGGL(hc_many_up_kept_kernel<10>, dim3(g.hidden / HU_H, sets < groups ? sets : groups),
                       dim3(HU_NT), lds, stream, A);
  } else {
    hipLaunchKernelGGL(hc_many_up_kernel, dim3(g.hidden / 64, (g.rows + 31) / 32), dim3(HR_NT), 0, stream, A);
  }
  QM_CHECK_LAUNCH();
  return QM_OK;
}

}  // namespace

bool qm_hc_rows_covers(const qm_hc_geom& g) {
  return g.streams == HR_STREAMS && g.rank == 320 && (g.hidden == 2048 || g.hidden == 2560);
}

size_t qm_hc_rows_workspace(const qm_hc_geom& g) { return hr_layout(g).total; }

int qm_hc_mix_rows(const qm_hc_geom& g, int as_rows, const void* hyper, const float* norm_w, const void* w_di,
                   int with_inject, const void* w_up, void* mixed, void* inject, void* ws, hipStream_t stream) {
  if (g.act_dtype == QM_ACT_BF16)
    return run_rows<bf16_t>(g, as_rows, hyper, norm_w, w_di, with_inject, w_up, mixed, inject, ws, stream);
  return run_rows<float>(g, as_rows, hyper, norm_w, w_di, with_inject, w_up, mixed, inject, ws, stream);
}
