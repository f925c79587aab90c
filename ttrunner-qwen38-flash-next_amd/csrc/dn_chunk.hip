// Gated delta rule over 64-token chunks in the WY/UT form, gfx950.
//
// chunk_gated_delta_rule (reference/layers.py:195-275). The chunk-local algebra
// is independent across chunks and the state recurrence is not, so the rule
// runs as two launches:
//   dn_chunk_prep   one or four workgroups per (sequence, head, chunk): l2-normalises q
//                   and k, takes the cumulative log-decay (in double, as torch's
//                   CPU cumsum accumulates), forms L = (k beta k^T) * decay
//                   below the diagonal and (q k^T) * decay on and below it,
//                   inverts I + L (16x16 diagonal blocks by substitution, the
//                   blocks below by fp32 MFMA, one sub-diagonal at a time) and
//                   writes w = T (k beta e^cum), u = T (v beta), q e^cum and
//                   k e^(cum_last - cum) to the workspace
//   dn_chunk_scan   one workgroup per (sequence, head, 16 columns of d_v): the
//                   state slice stays on chip while the chunks pass:
//                   v_new = u - w S, out = q_dec S + qk v_new,
//                   S = S e^cum_last + k_dec^T v_new
// The products over d_k and over tokens run on v_mfma_f32_16x16x32_bf16 with
// each fp32 operand split into bf16 high and low parts, x = hi + lo to 16
// significant bits: a b = hi hi + hi lo + lo hi, the lo lo term (2^-18 of the
// product) dropped, every sum accumulated in fp32. One such product costs
// three bf16 MFMAs where the same 16x16x32 product takes eight fp32
// 16x16x4 MFMAs of twice the cycles each. Operand lanes: A[row l%16][k 8(l/16)
// + e], B[k 8(l/16) + e][col l%16], e < 8; result rows 4(l/16)+i, col l%16.
// The state and v_new lie in LDS as [column][dk] and [column][token], so that
// they and every record operand are runs of 8 consecutive elements; either can
// be the A or the B operand (the lane layouts are alike), and which it is says
// whether a lane's 4 results lie along the row or the column: w S and k_dec^T
// v_new come out along [column]'s rows, the output along its channels.
#include "common.h"
#include "qwen4mix_internal.h"

#include <type_traits>

namespace {

constexpr int CK_C = 64;          // tokens per chunk
constexpr int CK_D = 128;         // d_k = d_v
constexpr int CK_NT = 256;        // scan: four waves
constexpr int CP_NT = 512;        // prep: eight waves (the rule over 4096 tokens took 292 us with four, 271 with
                                  // eight, one workgroup per compute unit by its LDS; 248 with two: PrepShared)
constexpr int CK_LD = CK_D + 4;   // LDS row stride of [token][dim] tiles, floats
constexpr int CK_LT = CK_C + 4;   // LDS row stride of [.][token] tiles, floats
constexpr int CK_COLS = 16;       // d_v columns per scan workgroup
// Shorter prefill chunks take the token loop, which works in blocks of 16 tokens:
// two of them are the faster, three are not (kernels alone, 32 heads, us, loop /
// chunked: bf16 12.4 / 14.4 at 24 tokens, 14.2 / 14.5 at 32, 18.0 / 14.6 at 40;
// float 13.9 / 14.4 at 32, 18.0 / 14.7 at 40; four sequences in bf16 29.4 / 31.0
// at 32, 37.1 / 31.8 at 40).
constexpr int CK_MIN_SEQ = 33;
constexpr int CK_PARTS = 4;       // prep workgroups per chunk when chunks are few

// One record per (sequence, head, chunk), in floats. A fragment pair is the
// bf16 high parts of one 16x32 MFMA operand (64 lanes x 8, 1 KB) followed by
// its low parts: FRAG2 floats. Fragment (b, s) of a matrix holds rows 16 b ..
// 16 b + 15 and k-step s (k = 32 s .. 32 s + 31) in operand lane order, so a
// wave's operand load reads 1 KB of contiguous memory.
//   W    w[tok][dk] = T (k beta e^cum)          (token block, dk step)  4 x 4
//   QD   q e^cum [tok][dk] (q l2-normalised, scaled by d^-1/2)          4 x 4
//   QK   (q k^T)[i][j] * decay, j <= i          (i block, j step)       4 x 2
//   KD   k e^(cum_last - cum), as [dk][tok]     (dk block, token step)  8 x 2
//   U    u = T (v beta) as [dv][tok], fp32
//   ECL  e^cum_last in element 0
constexpr long FRAG2 = 512;
constexpr long CK_W = 0;
constexpr long CK_QD = CK_W + 16 * FRAG2;
constexpr long CK_QK = CK_QD + 16 * FRAG2;
constexpr long CK_KD = CK_QK + 8 * FRAG2;
constexpr long CK_U = CK_KD + 16 * FRAG2;
constexpr long CK_ECL = CK_U + CK_C * CK_D;
constexpr long CK_REC = CK_ECL + 64;
static_assert((CK_REC * 4) % 256 == 0, "records stay 256-byte aligned");

// a double moved by DPP (both halves); lanes without a source, or in rows
// outside ROW_MASK, read 0.0
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ double dpp_d(double v) {
  const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
  const int lo = __builtin_amdgcn_update_dpp(0, static_cast<int>(b), CTRL, ROW_MASK, 0xF, true);
  const int hi = __builtin_amdgcn_update_dpp(0, static_cast<int>(b >> 32), CTRL, ROW_MASK, 0xF, true);
  return __builtin_bit_cast(double, (static_cast<unsigned long long>(static_cast<unsigned>(hi)) << 32) |
                                        static_cast<unsigned>(lo));
}

// An fp32 MFMA operand as bf16 high and low parts.
struct Frag {
  bf16x8_t hi, lo;
};

__device__ __forceinline__ float bf16_lo_half(unsigned w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float bf16_hi_half(unsigned w) { return __uint_as_float(w & 0xffff0000u); }

// x = hi + lo: hi rounds x to bf16, lo rounds the (exact) remainder
__device__ __forceinline__ void split2(float a, float b, unsigned& h, unsigned& l) {
  h = pack_bf16x2(a, b);
  l = pack_bf16x2(a - bf16_lo_half(h), b - bf16_hi_half(h));
}

__device__ __forceinline__ Frag split8(const float (&x)[8]) {
  u32x4_t h, l;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    unsigned hh, ll;
    split2(x[2 * i], x[2 * i + 1], hh, ll);
    h[i] = hh;
    l[i] = ll;
  }
  return Frag{__builtin_bit_cast(bf16x8_t, h), __builtin_bit_cast(bf16x8_t, l)};
}

// c + a b over one k-step, the small terms first
__device__ __forceinline__ f32x4_t mfma3(const Frag& a, const Frag& b, f32x4_t c) {
  c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.lo, b.hi, c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.hi, b.lo, c, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.hi, b.hi, c, 0, 0, 0);
}

// lane's operand from a record fragment pair
__device__ __forceinline__ Frag ld_frag(const float* pair, int lane) {
  const char* p = reinterpret_cast<const char*>(pair) + lane * 16;
  return Frag{*reinterpret_cast<const bf16x8_t*>(p), *reinterpret_cast<const bf16x8_t*>(p + 1024)};
}

// the lane's 8 elements of a fragment pair, from fp32 values
__device__ __forceinline__ void st_frag8(float* pair, int lane, const float (&x)[8]) {
  const Frag f = split8(x);
  char* p = reinterpret_cast<char*>(pair) + lane * 16;
  *reinterpret_cast<bf16x8_t*>(p) = f.hi;
  *reinterpret_cast<bf16x8_t*>(p + 1024) = f.lo;
}

// 4 of a lane's 8 elements (e0 .. e0 + 3, e0 = 0 or 4) of a fragment pair
__device__ __forceinline__ void st_frag4(float* pair, int lane, int e0, float a, float b, float c, float d) {
  unsigned h0, l0, h1, l1;
  split2(a, b, h0, l0);
  split2(c, d, h1, l1);
  char* p = reinterpret_cast<char*>(pair) + lane * 16 + e0 * 2;
  *reinterpret_cast<u32x2_t*>(p) = u32x2_t{h0, h1};
  *reinterpret_cast<u32x2_t*>(p + 1024) = u32x2_t{l0, l1};
}

// A result tile's lane holds rows 4 g + v (v < 4) of column r16; when the rows
// are the k index of a fragment pair whose k-step starts at row 32 s of the
// result's block b (rows 16 b ..), its 4 values are elements e0 .. e0 + 3 of
// lane r16 + 16 g' of fragment step s = b / 2
__device__ __forceinline__ void frag_slot(int blk, int g4, int& lane_g, int& e0) {
  lane_g = 2 * (blk & 1) + (g4 >> 1);
  e0 = 4 * (g4 & 1);
}

__device__ __forceinline__ f32x4_t mfma4(float a, float b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ f32x4_t mfma4x4(float4 a, float4 b, f32x4_t c) {
  c = mfma4(a.x, b.x, c);
  c = mfma4(a.y, b.y, c);
  c = mfma4(a.z, b.z, c);
  return mfma4(a.w, b.w, c);
}

__device__ __forceinline__ float4 lds4(const float* p) { return *reinterpret_cast<const float4*>(p); }
__device__ __forceinline__ float4 ld4(const float* p) { return *reinterpret_cast<const float4*>(p); }

// eight consecutive activations as float
__device__ __forceinline__ void load8(const float* p, float* o) {
  const float4 a = ld4(p), b = ld4(p + 4);
  o[0] = a.x; o[1] = a.y; o[2] = a.z; o[3] = a.w;
  o[4] = b.x; o[5] = b.y; o[6] = b.z; o[7] = b.w;
}
__device__ __forceinline__ void load8(const bf16_t* p, float* o) {
  const uint4 u = *reinterpret_cast<const uint4*>(p);
  const unsigned w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    o[2 * i] = bf16_to_f32(static_cast<uint16_t>(w[i] & 0xffffu));
    o[2 * i + 1] = bf16_to_f32(static_cast<uint16_t>(w[i] >> 16));
  }
}

// eight consecutive activations loaded raw (get() converts them), so that a
// run of loads can be issued before any conversion waits on one of them
template <typename T> struct Raw8;
template <> struct Raw8<float> {
  float4 a, b;
  __device__ __forceinline__ void load(const float* p) {
    a = *reinterpret_cast<const float4*>(p);
    b = *reinterpret_cast<const float4*>(p + 4);
  }
  __device__ __forceinline__ void get(float* o) const {
    o[0] = a.x; o[1] = a.y; o[2] = a.z; o[3] = a.w; o[4] = b.x; o[5] = b.y; o[6] = b.z; o[7] = b.w;
  }
};
template <> struct Raw8<bf16_t> {
  uint4 u;
  __device__ __forceinline__ void load(const bf16_t* p) { u = *reinterpret_cast<const uint4*>(p); }
  __device__ __forceinline__ void get(float* o) const {
    const unsigned w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      o[2 * i] = bf16_to_f32(static_cast<uint16_t>(w[i] & 0xffffu));
      o[2 * i + 1] = bf16_to_f32(static_cast<uint16_t>(w[i] >> 16));
    }
  }
};

// lower 16x16 tiles (I, J), J <= I, numbered (0,0) (1,0) (1,1) (2,0) ... (3,3)
__device__ __forceinline__ void tile_ij(int t, int& I, int& J) {
  I = t < 1 ? 0 : t < 3 ? 1 : t < 6 ? 2 : 3;
  J = t - I * (I + 1) / 2;
}

// a lane's operand from a [row][k] bf16 hi / lo LDS tile pair (row stride
// CK_HS): row `row`, k = 32 s + 8 g4 .. + 7
constexpr int CK_HS = CK_D + 8;   // bf16 row stride of the [token][dim] tiles
__device__ __forceinline__ Frag tile_frag(const uint16_t* hi, const uint16_t* lo, int row, int s, int g4) {
  const int o = row * CK_HS + 32 * s + 8 * g4;
  return Frag{*reinterpret_cast<const bf16x8_t*>(hi + o), *reinterpret_cast<const bf16x8_t*>(lo + o)};
}

// the same operand from fp32 [row][dim] LDS rows (stride CK_LD), split on the way
__device__ __forceinline__ Frag row_frag(const float* rows, int row, int s, int g4) {
  const float* o = rows + row * CK_LD + 32 * s + 8 * g4;
  const float4 a = lds4(o), b = lds4(o + 4);
  const float x[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
  return split8(x);
}

// 16x16 tile over the 128 dims of the products of two operands' rows
__device__ __forceinline__ f32x4_t gram16(const Frag (&a)[4], const Frag (&b)[4]) {
  f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < 4; ++s) acc = mfma3(a[s], b[s], acc);
  return acc;
}

template <typename T>
struct ChunkPrepArgs {
  const T* q; const T* k; const T* v;   // token rows of q_stride / v_stride elements
  const float* g; const float* beta;    // [B, S, H]
  float* ws;                            // [B, H, n_chunks] records
  int batch, seq, heads, hk;            // head h reads q/k head h % hk
  int c0, n_chunks;                     // this launch's first chunk, and its chunks (and the records') per head
  int parts;                            // workgroups per chunk: 1 or CK_PARTS
  long q_stride, v_stride;
};

// 71 KB, so that two workgroups of a compute unit run under each other's
// barriers and latencies: k is held once, in fp32, and split as it is read;
// L and T take q's place once the products with q and k are done; v, loaded
// again only then, takes k's once w and k_dec are. 1024 chunks of fp32 took
// 70.9 us with 158 KB and one workgroup, now 58.7 (240 KB of rows and record a
// chunk: 4.3 TB/s); 64 chunks in parts 10.7 and 11.2, which is one workgroup
// per compute unit either way.
struct alignas(16) PrepShared {
  union {
    struct {
      uint16_t h[CK_C * CK_HS], l[CK_C * CK_HS];   // normalised q * d^-1/2, split
    } q;
    struct {
      float L[CK_C][CK_LT];    // (k beta k^T) * decay, strictly lower
      float Tm[CK_C][CK_LT];   // (I + L)^-1, lower
    } m;
  } u;
  float kv[CK_C][CK_LD];       // normalised k, then v * beta: [token][dim]
  float cum[CK_C], beta[CK_C], ecum[CK_C], bec[CK_C], kds[CK_C];
};
static_assert(2 * (sizeof(PrepShared) + 256) <= 160 * 1024, "two workgroups per compute unit");

template <typename T>
__global__ __launch_bounds__(CP_NT, 4) void dn_chunk_prep_kernel(ChunkPrepArgs<T> A) {
  __shared__ PrepShared sh;
  QM_PHASE_DECL
  QM_PHASE(0);
  // A.parts workgroups per chunk: each forms L and T, then writes its share
  // (all of it, or a quarter) of the record. The parts of a chunk read the
  // same q, k and v rows: consecutive workgroups in this order run on one die
  // (xcd_remap), so the rows come from memory once per chunk, not per part
  const int wg = xcd_remap(blockIdx.x, gridDim.x);
  const int part = wg % A.parts;
  const int c = (wg / A.parts) % A.n_chunks;
  const int bh = wg / A.parts / A.n_chunks;
  const int span = CK_PARTS / A.parts;       // quarters this workgroup writes
  const int h = bh % A.heads, b = bh / A.heads;
  const int t0 = (A.c0 + c) * CK_C;
  const int n_valid = min(CK_C, A.seq - t0);
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int g4 = lane >> 4, r16 = lane & 15;
  float* rec = A.ws + ((long)bh * A.n_chunks + c) * CK_REC;
  const int span_sh = span == 1 ? 0 : 2;     // span is 1 or 4
  auto mine = [&](int quarter) __attribute__((always_inline)) { return (quarter >> span_sh) == part; };

  // q and k rows (v's below): eight threads per token, 16 dims each as two runs of 8; run
  // j of thread p is unit p % 4 of the 32 dims 32 (2 j + p / 4) ..
  const int t = tid >> 3, p = tid & 7;
  const bool tok_ok = t < n_valid;
  float qn[16];
  {
    // every load at once, the gates first (the cumulative decay is the
    // longest chain); indices are clamped so that no load sits in a branch
    const bool ok = lane < n_valid;
    const long gi = ((long)b * A.seq + t0 + (ok ? lane : 0)) * A.heads + h;
    const float g_raw = A.g[gi], b_raw = A.beta[gi];
    const long tok = (long)b * A.seq + t0 + (tok_ok ? t : 0);
    const long qo = tok * A.q_stride + (long)(h % A.hk) * CK_D;
    Raw8<T> xq[2], xk[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int d = 8 * (p + 8 * j);
      xq[j].load(A.q + qo + d);
      xk[j].load(A.k + qo + d);
    }
    __builtin_amdgcn_sched_barrier(0);
    float kv[16];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      xq[j].get(qn + 8 * j);
      xk[j].get(kv + 8 * j);
    }

    // gates; padding tokens carry g = 0 and beta = 0
    if (wid == 0) {
      const float gv = ok ? g_raw : 0.f;
      const float bl = ok ? b_raw : 0.f;
      // inclusive scan over the 64 lanes in double on DPP (no LDS round
      // trips): row shifts by 1, 2, 4, 8, then lane 15 of each row to the
      // next row (rows 1, 3), then lane 31 to rows 2 and 3
      double s = gv;
      s += dpp_d<0x111, 0xF>(s);
      s += dpp_d<0x112, 0xF>(s);
      s += dpp_d<0x114, 0xF>(s);
      s += dpp_d<0x118, 0xF>(s);
      s += dpp_d<0x142, 0xA>(s);
      s += dpp_d<0x143, 0xC>(s);
      const float cum = static_cast<float>(s);
      const float last = readlane_f(cum, 63);
      const float ec = expf(cum);
      sh.cum[lane] = cum;
      sh.beta[lane] = bl;
      sh.ecum[lane] = ec;
      sh.bec[lane] = bl * ec;
      sh.kds[lane] = expf(last - cum);
      if (lane == 0 && part == 0) rec[CK_ECL] = expf(last);
    }

    float sq = 0.f, sk = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      sq = fmaf(qn[i], qn[i], sq);
      sk = fmaf(kv[i], kv[i], sk);
    }
    sq += dpp_f<0xB1>(sq);    // lane ^ 1
    sk += dpp_f<0xB1>(sk);
    sq += dpp_f<0x4E>(sq);    // lane ^ 2
    sk += dpp_f<0x4E>(sk);
    sq += dpp_f<0x141>(sq);   // the other quad of eight (its lanes agree by now)
    sk += dpp_f<0x141>(sk);
    const float rq = tok_ok ? rsqrt_rn(sq + 1e-6f) : 0.f;
    const float rk = tok_ok ? rsqrt_rn(sk + 1e-6f) : 0.f;
    const float qscale = 0.08838834764831845f;  // 128^-1/2
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      qn[i] = mul_rn(mul_rn(qn[i], rq), qscale);
      kv[i] = mul_rn(kv[i], rk);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int d = 8 * (p + 8 * j);
      float xq[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) xq[e] = qn[8 * j + e];
      const Frag fq = split8(xq);
      *reinterpret_cast<bf16x8_t*>(&sh.u.q.h[t * CK_HS + d]) = fq.hi;
      *reinterpret_cast<bf16x8_t*>(&sh.u.q.l[t * CK_HS + d]) = fq.lo;
      *reinterpret_cast<float4*>(&sh.kv[t][d]) = make_float4(kv[8 * j], kv[8 * j + 1], kv[8 * j + 2], kv[8 * j + 3]);
      *reinterpret_cast<float4*>(&sh.kv[t][d + 4]) =
          make_float4(kv[8 * j + 4], kv[8 * j + 5], kv[8 * j + 6], kv[8 * j + 7]);
    }
  }
  QM_PHASE(1);
  __syncthreads();
  QM_PHASE(2);

  // q e^cum fragments (QD: token block t / 16, dk step = the run's 32 dims)
  // from the thread's own q values: a run of 8 dims is lane t % 16 + 16 (p % 4)
  if (mine(t >> 4)) {
    const float e = sh.ecum[t];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      float x[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = qn[8 * j + i] * e;
      st_frag8(rec + CK_QD + ((t >> 4) * 4 + 2 * j + (p >> 2)) * FRAG2, (t & 15) + 16 * (p & 3), x);
    }
  }
  QM_PHASE(10);
  // qk = (q k^T) * exp(cum_i - cum_j) for j <= i, as QK fragments: tile
  // (I, J) is computed as k_J q_I^T, so that a lane holds 4 consecutive j of
  // one i; tiles 10 and 11 are the zero blocks (0, 1) and (2, 3) above the
  // diagonal that the scan's 32-wide k-steps read. Tile ti belongs to quarter
  // ti % 4; this workgroup's tiles go round-robin to its waves
  {
    // this workgroup's tiles in order: ti = part, part + 4, part + 8 (one
    // quarter) or all 12; the k-th goes to wave k % 8
    for (int k = wid; k < 3 * span; k += CP_NT / 64) {
      const int ti = span == 1 ? part + 4 * k : k;
      int I, J;
      if (ti < 10) tile_ij(ti, I, J);
      else { I = ti == 10 ? 0 : 2; J = I + 1; }
      f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
      if (ti < 10) {
        Frag fk[4], fq[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          fk[s] = row_frag(&sh.kv[0][0], 16 * J + r16, s, g4);
          fq[s] = tile_frag(sh.u.q.h, sh.u.q.l, 16 * I + r16, s, g4);
        }
        acc = gram16(fk, fq);
      }
      // the decays' operands are read before any exponential, outside the
      // masks, so that their LDS latencies overlap
      const int i = 16 * I + r16;
      const float ci = sh.cum[i];
      const float4 cj = lds4(&sh.cum[16 * J + 4 * g4]);
      const float cjv[4] = {cj.x, cj.y, cj.z, cj.w};
      float x[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const float val = acc[v] * expf(ci - cjv[v]);
        x[v] = ti < 10 && i >= 16 * J + 4 * g4 + v ? val : 0.f;
      }
      int lg, e0;
      frag_slot(J, g4, lg, e0);
      st_frag4(rec + CK_QK + (I * 2 + J / 2) * FRAG2, r16 + 16 * lg, e0, x[0], x[1], x[2], x[3]);
    }
  }
  QM_PHASE(3);
  // L = (k k^T) * beta_i * exp(cum_i - cum_j) for j < i: ten tiles, wave w
  // forms tile w, waves 4 and 5 (which had one q k^T tile fewer when a workgroup
  // forms all of them) tiles 8 and 9 as well; q's space takes them when every
  // wave is done with q
  float (&L)[CK_C][CK_LT] = sh.u.m.L;
  float (&Tm)[CK_C][CK_LT] = sh.u.m.Tm;
  const int n_l = wid == 4 || wid == 5 ? 2 : 1;
  f32x4_t lacc[2];
#pragma unroll
  for (int n = 0; n < 2; ++n)
    if (n < n_l) {
      int I, J;
      tile_ij(wid + 4 * n, I, J);
      Frag fi[4], fj[4];
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        fi[s] = row_frag(&sh.kv[0][0], 16 * I + r16, s, g4);
        fj[s] = row_frag(&sh.kv[0][0], 16 * J + r16, s, g4);
      }
      lacc[n] = gram16(fi, fj);
      const int j = 16 * J + r16;
      const float cj = sh.cum[j];
      const float4 ci = lds4(&sh.cum[16 * I + 4 * g4]), bi = lds4(&sh.beta[16 * I + 4 * g4]);
      const float civ[4] = {ci.x, ci.y, ci.z, ci.w}, biv[4] = {bi.x, bi.y, bi.z, bi.w};
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const float val = (lacc[n][v] * biv[v]) * expf(civ[v] - cj);
        lacc[n][v] = 16 * I + 4 * g4 + v > j ? val : 0.f;
      }
    }
  QM_PHASE(9);
  __syncthreads();
#pragma unroll
  for (int n = 0; n < 2; ++n)
    if (n < n_l) {
      int I, J;
      tile_ij(wid + 4 * n, I, J);
#pragma unroll
      for (int v = 0; v < 4; ++v) L[16 * I + 4 * g4 + v][16 * J + r16] = lacc[n][v];
    }
  QM_PHASE(4);
  __syncthreads();

  if (wid == 0) {
    // (I + L_II)^-1 for the four diagonal blocks; lane = (block, column):
    // x_i = [i == col] - sum_{k<i} L_ik x_k
    // the block's lower triangle is read ahead (rows in runs of 4, the zeros
    // above the diagonal included; rows 1..8, then 9..15: registers), so that
    // the substitution's dependent chain waits on two LDS round trips alone
    const int I = g4, col = r16;
    float x[16];
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const int i0 = half ? 9 : 1, i1 = half ? 16 : 9;
      float4 lr[8][4];
#pragma unroll
      for (int i = i0; i < i1; ++i)
#pragma unroll
        for (int k4 = 0; k4 < (i + 3) / 4; ++k4) lr[i - i0][k4] = lds4(&L[16 * I + i][16 * I + 4 * k4]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = half ? i0 : 0; i < i1; ++i) {
        float acc = i == col ? 1.f : 0.f;
#pragma unroll
        for (int kk = 0; kk < i; ++kk) {
          const float4 v = lr[i - i0][kk / 4];
          const float l = kk % 4 == 0 ? v.x : kk % 4 == 1 ? v.y : kk % 4 == 2 ? v.z : v.w;
          acc = fmaf(-l, x[kk], acc);
        }
        x[i] = acc;
      }
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) Tm[16 * I + i][16 * I + col] = x[i];
  } else {
    // the zero blocks (0, 1) and (2, 3) of T, which the 32-wide k-steps of
    // the w and u products read
    for (int idx = tid - 64; idx < 2 * 256; idx += CP_NT - 64) {
      const int blk = idx >> 8, r = (idx >> 4) & 15, cc = idx & 15;
      Tm[32 * blk + r][32 * blk + 16 + cc] = 0.f;
    }
    // k_dec fragments (KD: dk blocks 2 quarter, 2 quarter + 1, token steps
    // 0..1): lane (dk 16 D + r16, tokens 32 s + 8 g4 ..); this workgroup's
    // fragments are f0 .. f0 + 4 span, the i-th to wave 1 + i % 7
    const int f0 = 4 * span * part;
    for (int i = wid - 1; i < 4 * span; i += CP_NT / 64 - 1) {
      const int f = f0 + i;
      const int D = f >> 1, s = f & 1;
      const int c0 = 32 * s + 8 * g4;
      float x[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = sh.kv[c0 + e][16 * D + r16] * sh.kds[c0 + e];
      st_frag8(rec + CK_KD + f * FRAG2, lane, x);
    }
  }
  // the v rows come in under the rest of T and w (their place is k's, below)
  const bool has_w = A.parts == 1 || part < 2, has_u = A.parts == 1 || part >= 2;
  Raw8<T> xv[2];
  {
    const T* vp = A.v + ((long)b * A.seq + t0 + (tok_ok ? t : 0)) * A.v_stride + (long)h * CK_D;
    if (has_u)
#pragma unroll
      for (int j = 0; j < 2; ++j) xv[j].load(vp + 8 * (p + 8 * j));
  }
  QM_PHASE(5);
  __syncthreads();

  QM_PHASE(6);
  // blocks of T below the diagonal, one sub-diagonal at a time:
  // T_IJ = -T_II sum_{K=J}^{I-1} L_IK T_KJ
  for (int dist = 1; dist < 4; ++dist) {
    if (wid < 4 - dist) {
      const int J = wid, I = wid + dist;
      f32x4_t pp = {0.f, 0.f, 0.f, 0.f};
      for (int K = J; K < I; ++K) {
        const float4 a = lds4(&L[16 * I + r16][16 * K + 4 * g4]);
        const float* tb = &Tm[16 * K + 4 * g4][16 * J + r16];
        pp = mfma4x4(a, make_float4(tb[0], tb[CK_LT], tb[2 * CK_LT], tb[3 * CK_LT]), pp);
      }
      const float4 xa = lds4(&Tm[16 * I + r16][16 * I + 4 * g4]);
      f32x4_t x = {0.f, 0.f, 0.f, 0.f};
      x = mfma4x4(xa, make_float4(pp[0], pp[1], pp[2], pp[3]), x);
#pragma unroll
      for (int v = 0; v < 4; ++v) Tm[16 * I + 4 * g4 + v][16 * J + r16] = -x[v];
    }
    __syncthreads();
  }

  QM_PHASE(7);
  // w = T (k beta e^cum), as w^T = (k beta e^cum)^T T^T so that a lane holds 4
  // consecutive dims of one token, and u = T (v beta), a lane 4 consecutive
  // tokens of one dim: quarter r holds column
  // tiles 4 r .. 4 r + 3 of the 16 (w: 0..7, u: 8..15, 16 dims each), at most
  // eight of either kind a workgroup, one per wave; T is lower triangular, so
  // row block I needs k-steps 0 .. I / 2
  auto column_tile = [&](int tile, auto is_u) __attribute__((always_inline)) {
    const int D = tile & 7;
    float x[2][8];
    float4 tr[4][2][2];
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2)
#pragma unroll
      for (int e = 0; e < 8; ++e) x[s2][e] = sh.kv[32 * s2 + 8 * g4 + e][16 * D + r16];
    if constexpr (!is_u.value) {
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2) {
        const float4 y0 = lds4(&sh.bec[32 * s2 + 8 * g4]), y1 = lds4(&sh.bec[32 * s2 + 8 * g4 + 4]);
        const float y[8] = {y0.x, y0.y, y0.z, y0.w, y1.x, y1.y, y1.z, y1.w};
#pragma unroll
        for (int e = 0; e < 8; ++e) x[s2][e] *= y[e];
      }
    }
#pragma unroll
    for (int I = 0; I < 4; ++I)
#pragma unroll
      for (int s2 = 0; s2 <= I / 2; ++s2) {
        const int c = 32 * s2 + 8 * g4;
        tr[I][s2][0] = lds4(&Tm[16 * I + r16][c]);
        tr[I][s2][1] = lds4(&Tm[16 * I + r16][c + 4]);
      }
    const Frag a[2] = {split8(x[0]), split8(x[1])};
#pragma unroll
    for (int I = 0; I < 4; ++I) {
      f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s2 = 0; s2 <= I / 2; ++s2) {
        const float y[8] = {tr[I][s2][0].x, tr[I][s2][0].y, tr[I][s2][0].z, tr[I][s2][0].w,
                            tr[I][s2][1].x, tr[I][s2][1].y, tr[I][s2][1].z, tr[I][s2][1].w};
        acc = is_u.value ? mfma3(split8(y), a[s2], acc) : mfma3(a[s2], split8(y), acc);
      }
      if constexpr (is_u.value) {
        // acc[v]: token 16 I + 4 g4 + v of dim 16 D + r16
        *reinterpret_cast<float4*>(rec + CK_U + (16 * D + r16) * CK_C + 16 * I + 4 * g4) =
            make_float4(acc[0], acc[1], acc[2], acc[3]);
      } else {
        // acc[v]: dim 16 D + 4 g4 + v of token 16 I + r16
        int lg, e0;
        frag_slot(D, g4, lg, e0);
        st_frag4(rec + CK_W + (I * 4 + D / 2) * FRAG2, r16 + 16 * lg, e0, acc[0], acc[1], acc[2], acc[3]);
      }
    }
  };
  const int n_col = span == 1 ? 4 : 8;       // column tiles of each kind
  if (has_w) {
    if (wid < n_col) column_tile(4 * span * part + wid, std::false_type{});
    __syncthreads();                         // every wave is done with k
  }
  if (has_u) {
    // without w tiles, k_dec's reads of k ended before the barriers above
    const float bv = sh.beta[t];             // 0 for padding tokens
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      float vv[8];
      xv[j].get(vv);
      float* dst = &sh.kv[t][8 * (p + 8 * j)];
      *reinterpret_cast<float4*>(dst) = make_float4(vv[0] * bv, vv[1] * bv, vv[2] * bv, vv[3] * bv);
      *reinterpret_cast<float4*>(dst + 4) = make_float4(vv[4] * bv, vv[5] * bv, vv[6] * bv, vv[7] * bv);
    }
    __syncthreads();
    if (wid < n_col) column_tile((span == 1 ? 4 * part : 8) + wid, std::true_type{});
  }
  QM_PHASE(8);
  QM_PHASE_FLUSH();
}

template <typename T>
struct ChunkScanArgs {
  const float* ws;   // [B, H, n_chunks] records
  float* state;      // [B, H, 128, 128]
  T* out;            // [B, S, H, 128]
  int batch, seq, heads;
  int t0, n_chunks;  // this launch's first token, and its chunks (and the records') per head
};

// A wave's record operands of one chunk, none of which depends on the
// state: the W and QD fragments of its token block (dk steps 0..3), the QK
// fragments of its token block (j steps 0..1, the second from block 2 on), the KD fragments of its two dk
// blocks (token steps 0..1), its 4 values of u and e^cum_last.
struct ScanOps {
  Frag w[4], qd[4], qk[2], kd[2][2];
  float4 u;
  float ecl;
};

__device__ __forceinline__ void load_scan_ops(const float* rec, int wid, int lane, int r16, int g4, int col0,
                                              ScanOps& o) {
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    o.w[s] = ld_frag(rec + CK_W + (wid * 4 + s) * FRAG2, lane);
    o.qd[s] = ld_frag(rec + CK_QD + (wid * 4 + s) * FRAG2, lane);
  }
#pragma unroll
  for (int s = 0; s < 2; ++s)
    if (s == 0 || wid >= 2) o.qk[s] = ld_frag(rec + CK_QK + (wid * 2 + s) * FRAG2, lane);
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int s = 0; s < 2; ++s) o.kd[t][s] = ld_frag(rec + CK_KD + ((2 * wid + t) * 2 + s) * FRAG2, lane);
  o.u = *reinterpret_cast<const float4*>(rec + CK_U + (col0 + r16) * CK_C + 16 * wid + 4 * g4);
  o.ecl = rec[CK_ECL];
}

constexpr int SC_SS = CK_D + 8;   // bf16 row stride of the state tile [column][dk]
constexpr int SC_SV = CK_C + 8;   // bf16 row stride of the v_new tile [column][token]

// lane's A operand of row r16 of a bf16 hi / lo LDS tile pair, k = 32 s + 8 g4 ..
__device__ __forceinline__ Frag lds_frag(const uint16_t* hi, const uint16_t* lo, int stride, int r16, int s, int g4) {
  const int o = r16 * stride + 32 * s + 8 * g4;
  return Frag{*reinterpret_cast<const bf16x8_t*>(hi + o), *reinterpret_cast<const bf16x8_t*>(lo + o)};
}

// four consecutive elements (from r) of column c of a [column][.] bf16 hi / lo tile pair
__device__ __forceinline__ void put4(uint16_t* hi, uint16_t* lo, int stride, int c, int r, float a, float b, float d,
                                     float e) {
  unsigned h0, l0, h1, l1;
  split2(a, b, h0, l0);
  split2(d, e, h1, l1);
  *reinterpret_cast<uint2*>(hi + c * stride + r) = make_uint2(h0, h1);
  *reinterpret_cast<uint2*>(lo + c * stride + r) = make_uint2(l0, l1);
}

// The record loads bound a chunk (109 KB for each of the eight column slices of
// a head, from the die's cache at about 24 bytes a clock and compute unit),
// then its dependent chain (state -> w S -> v_new -> state), 1.4 of 2.25 us a
// chunk when timed without the loads, one wave per SIMD: so nothing is loaded
// that no product takes, every operand is read before its first product, v_new
// and the state come out of their products as 4 consecutive elements of a
// tile's row (one 8-byte LDS write each of high and low parts), and the output's
// products follow the ones that the chain needs. The chain alone: 1.42 -> 1.23
// us; the rule over 4096 tokens in fp32 257 -> 240 us, 4000 in bf16 229 -> 224.
template <typename T>
__global__ __launch_bounds__(CK_NT) void dn_chunk_scan_kernel(ChunkScanArgs<T> A) {
  // the state slice S^T [column][dk] and the chunk's v_new^T [column][token],
  // as bf16 high and low parts
  __shared__ __attribute__((aligned(16))) uint16_t sSh[CK_COLS * SC_SS], sSl[CK_COLS * SC_SS];
  __shared__ __attribute__((aligned(16))) uint16_t sVh[CK_COLS * SC_SV], sVl[CK_COLS * SC_SV];
  QM_PHASE_DECL
  QM_PHASE(0);
  constexpr int NSL = CK_D / CK_COLS;
  const int nwg = A.batch * A.heads * NSL;
  const int wg = xcd_remap(blockIdx.x, nwg);
  const int sl = wg % NSL, bh = wg / NSL;
  const int h = bh % A.heads, b = bh / A.heads;
  const int col0 = sl * CK_COLS;
  const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g4 = lane >> 4, r16 = lane & 15;
  const float* recs = A.ws + (long)bh * A.n_chunks * CK_REC;

  // wave wid keeps dk rows 32 wid .. 32 wid + 31 of the slice as two result
  // tiles: st[t][i] = S[dk 32 wid + 16 t + 4 g4 + i][column r16]
  float* S = A.state + (long)bh * CK_D * CK_D + (long)(32 * wid + 4 * g4) * CK_D + col0 + r16;
  f32x4_t st[2];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) st[t][i] = S[(16 * t + i) * CK_D];
  // operands two chunks ahead: three register sets, the loop unrolled by
  // three so that no set is copied while its loads are in flight. The state
  // and the first two chunks' operands are requested together: the state
  // first, so that its wait leaves the operand loads in flight
  ScanOps o0, o1, o2;
  load_scan_ops(recs, wid, lane, r16, g4, col0, o0);
  load_scan_ops(recs + (long)min(1, A.n_chunks - 1) * CK_REC, wid, lane, r16, g4, col0, o1);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int t = 0; t < 2; ++t)
    put4(sSh, sSl, SC_SS, r16, 32 * wid + 16 * t + 4 * g4, st[t][0], st[t][1], st[t][2], st[t][3]);
  QM_PHASE(1);

  auto chunk = [&](int ci, const ScanOps& cur, ScanOps& ahead) {
    // chunk ci + 2's operands fly during this one
    if (ci + 2 < A.n_chunks) load_scan_ops(recs + (long)(ci + 2) * CK_REC, wid, lane, r16, g4, col0, ahead);
    __syncthreads();
    Frag sa[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) sa[s] = lds_frag(sSh, sSl, SC_SS, r16, s, g4);
    __builtin_amdgcn_sched_barrier(0);
    // w S for tokens 16 wid ..: rows = tokens 16 wid + 4 g4 + i, column r16
    f32x4_t aw = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < 4; ++s) aw = mfma3(cur.w[s], sa[s], aw);
    put4(sVh, sVl, SC_SV, r16, 16 * wid + 4 * g4, cur.u.x - aw[0], cur.u.y - aw[1], cur.u.z - aw[2],
         cur.u.w - aw[3]);
    // (q_dec S)^T: rows = columns 4 g4 + i, column = token 16 wid + r16
    f32x4_t ao = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < 4; ++s) ao = mfma3(sa[s], cur.qd[s], ao);
    __syncthreads();

    // S = S e^cum_last + k_dec^T v_new on this wave's dk rows (the tile is
    // only read again after the next chunk's first barrier)
    const Frag va0 = lds_frag(sVh, sVl, SC_SV, r16, 0, g4), va1 = lds_frag(sVh, sVl, SC_SV, r16, 1, g4);
#pragma unroll
    for (int t = 0; t < 2; ++t) st[t] = f32x4_t{st[t][0] * cur.ecl, st[t][1] * cur.ecl, st[t][2] * cur.ecl, st[t][3] * cur.ecl};
#pragma unroll
    for (int t = 0; t < 2; ++t) st[t] = mfma3(cur.kd[t][0], va0, st[t]);
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      st[t] = mfma3(cur.kd[t][1], va1, st[t]);
      put4(sSh, sSl, SC_SS, r16, 32 * wid + 16 * t + 4 * g4, st[t][0], st[t][1], st[t][2], st[t][3]);
    }

    // out^T += v_new^T qk^T over the causal token steps (j <= i: steps 0 ..
    // wid / 2; the record's QK holds zeros above the diagonal)
    ao = mfma3(va0, cur.qk[0], ao);
    if (wid >= 2) ao = mfma3(va1, cur.qk[1], ao);
    const int tok = A.t0 + ci * CK_C + 16 * wid + r16;
    if (tok < A.seq) {
      T* o = A.out + (((long)b * A.seq + tok) * A.heads + h) * CK_D + col0 + 4 * g4;
#pragma unroll
      for (int i = 0; i < 4; ++i) Act<T>::store(o, i, ao[i]);
    }
    if (ci < 12) QM_PHASE(2 + ci);
  };

  // at least one chunk (the host sends no empty sequence here): no zero-trip
  // test for the compiler to sink the first operand loads behind
  int ci = 0;
  do {
    chunk(ci, o0, o2);
    if (ci + 1 < A.n_chunks) chunk(ci + 1, o1, o0);
    if (ci + 2 < A.n_chunks) chunk(ci + 2, o2, o1);
    ci += 3;
  } while (ci < A.n_chunks);

#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) S[(16 * t + i) * CK_D] = st[t][i];
  QM_PHASE(14);
  QM_PHASE_FLUSH_AT(4096u);
}

// Long sequences run in segments of chunks, prep and scan in turn, each
// segment's records over the last one's: the prep's records are written once
// and read once, and while a segment's stay in the 256 MB memory-side cache the
// scan does not wait for memory. 4096 tokens of 32 heads (302 MB of records):
// 343 us in one segment, 296 in two or four, 313 in eight (each scan starts
// again from the state, about 4 us); 4000 tokens in bf16 315 -> 262 us; 2048
// tokens (151 MB) 150 us in one segment, 145 in two, bf16 131 and 136.
constexpr size_t CK_SEG_BYTES = 160ull << 20;

template <typename T>
int launch_chunked(int batch, int seq, int heads, int hk, long q_stride, long v_stride, const void* q, const void* k,
                   const void* v, const float* g, const float* beta, float* state, void* out, float* ws,
                   hipStream_t stream) {
  const int n_total = (seq + CK_C - 1) / CK_C;
  const size_t chunk_bytes = (size_t)batch * heads * CK_REC * sizeof(float);
  // a segment's outputs are stored before the next one's inputs are read: outputs
  // that lie over inputs take one segment, whose prep reads them all first
  const size_t rows = (size_t)batch * seq, gates = rows * heads * sizeof(float);
  const size_t out_bytes = rows * heads * CK_D * sizeof(T);
  const size_t qk_bytes = ((rows - 1) * q_stride + hk * CK_D) * sizeof(T);
  const size_t v_bytes = ((rows - 1) * v_stride + heads * CK_D) * sizeof(T);
  const bool over = qm_overlap(out, out_bytes, q, qk_bytes) || qm_overlap(out, out_bytes, k, qk_bytes) ||
                    qm_overlap(out, out_bytes, v, v_bytes) || qm_overlap(out, out_bytes, g, gates) ||
                    qm_overlap(out, out_bytes, beta, gates);
  const size_t n_seg = over ? 1 : (n_total * chunk_bytes + CK_SEG_BYTES - 1) / CK_SEG_BYTES;
  const int seg = n_seg < (size_t)n_total ? (int)((n_total + n_seg - 1) / n_seg) : 1;
  for (int c0 = 0; c0 < n_total; c0 += seg) {
    const int n_chunks = seg < n_total - c0 ? seg : n_total - c0;
    ChunkPrepArgs<T> P;
    P.q = static_cast<const T*>(q); P.k = static_cast<const T*>(k); P.v = static_cast<const T*>(v);
    P.g = g; P.beta = beta; P.ws = ws;
    P.batch = batch; P.seq = seq; P.heads = heads; P.hk = hk; P.c0 = c0; P.n_chunks = n_chunks;
    P.q_stride = q_stride; P.v_stride = v_stride;
    // few chunks: four workgroups per chunk so that the launch fills the chip;
    // many: one each, since every workgroup repeats the L and T work
    P.parts = (long)batch * heads * n_chunks < 256 ? CK_PARTS : 1;
    hipLaunchKernelGGL(dn_chunk_prep_kernel<T>, dim3(batch * heads * n_chunks * P.parts), dim3(CP_NT), 0, stream, P);
    QM_CHECK_LAUNCH();
    ChunkScanArgs<T> S;
    S.ws = ws; S.state = state; S.out = static_cast<T*>(out);
    S.batch = batch; S.seq = seq; S.heads = heads; S.t0 = c0 * CK_C; S.n_chunks = n_chunks;
    hipLaunchKernelGGL(dn_chunk_scan_kernel<T>, dim3(batch * heads * (CK_D / CK_COLS)), dim3(CK_NT), 0, stream, S);
    QM_CHECK_LAUNCH();
  }
  return QM_OK;
}

int run_chunked(int act_dtype, int batch, int seq, int heads, int hk, long q_stride, long v_stride, const void* q,
                const void* k, const void* v, const float* g, const float* beta, float* state, void* out, void* ws,
                hipStream_t stream) {
  float* w = static_cast<float*>(ws);
  if (act_dtype == QM_ACT_F32)
    return launch_chunked<float>(batch, seq, heads, hk, q_stride, v_stride, q, k, v, g, beta, state, out, w, stream);
  if (act_dtype == QM_ACT_BF16)
    return launch_chunked<bf16_t>(batch, seq, heads, hk, q_stride, v_stride, q, k, v, g, beta, state, out, w,
                                  stream);
  return qm_fail(QM_ERR_DTYPE, "delta rule: act_dtype must be QM_ACT_F32 or QM_ACT_BF16");
}

}  // namespace

QM_PHASE_ENTRY(dnc)

namespace {
size_t chunk_records_bytes(int batch, int seq, int heads) {
  if (batch <= 0 || seq <= 0 || heads <= 0) return 0;
  const size_t n_chunks = (size_t)(seq + CK_C - 1) / CK_C;
  return (size_t)batch * heads * n_chunks * CK_REC * sizeof(float);
}
}  // namespace

size_t qm_dn_rule_chunk_workspace(int batch, int seq, int heads) {
  return seq < CK_MIN_SEQ ? 0 : chunk_records_bytes(batch, seq, heads);
}

int qm_dn_rule_chunk(int act_dtype, int batch, int seq, int heads, int hk, long q_stride, long v_stride,
                     const void* q, const void* k, const void* v, const float* g, const float* beta, float* state,
                     void* out, void* ws, size_t ws_bytes, hipStream_t stream) {
  if (seq < CK_MIN_SEQ)
    return qm_dn_recurrent_strided(act_dtype, batch, seq, heads, hk, q_stride, v_stride, q, k, v, g, beta, state, out,
                                   stream);
  if (!ws || ws_bytes < chunk_records_bytes(batch, seq, heads))
    return qm_fail(QM_ERR_WORKSPACE, "delta rule: workspace too small for the chunked form");
  return run_chunked(act_dtype, batch, seq, heads, hk, q_stride, v_stride, q, k, v, g, beta, state, out, ws, stream);
}

extern "C" size_t qm_dn_chunked_workspace(int batch, int seq, int heads, int head_dim) {
  if (head_dim != CK_D) return 0;
  return chunk_records_bytes(batch, seq, heads);
}

extern "C" int qm_dn_chunked(int act_dtype, int batch, int seq, int heads, int head_dim, const void* q, const void* k,
                             const void* v, const float* g, const float* beta, float* state, void* out,
                             void* workspace, size_t workspace_bytes, hipStream_t stream) {
  if (head_dim != CK_D) return qm_fail(QM_ERR_UNSUPPORTED, "qm_dn_chunked: head_dim must be 128");
  if (batch <= 0 || seq < 0 || heads <= 0) return qm_fail(QM_ERR_ARG, "qm_dn_chunked: bad sizes");
  if (!q || !k || !v || !g || !beta || !state || !out) return qm_fail(QM_ERR_ARG, "qm_dn_chunked: null pointer");
  if (act_dtype != QM_ACT_F32 && act_dtype != QM_ACT_BF16)
    return qm_fail(QM_ERR_DTYPE, "qm_dn_chunked: act_dtype must be QM_ACT_F32 or QM_ACT_BF16");
  if (seq == 0) return QM_OK;
  if (!workspace || workspace_bytes < chunk_records_bytes(batch, seq, heads))
    return qm_fail(QM_ERR_WORKSPACE, "qm_dn_chunked: workspace too small");
  return run_chunked(act_dtype, batch, seq, heads, heads, (long)heads * CK_D, (long)heads * CK_D, q, k, v, g, beta,
                     state, out, workspace, stream);
}
