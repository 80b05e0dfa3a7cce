// detrt's decoder-layer row ops on gfx950, bit-identical to the CPU reference: the fused
// kernels around the exact int8 GEMMs of one layer (runtime/detgpu/stages.py:154-168 calls
// them; CUDA twins runtime/detgpu/kernels.py:117-353, CPU definitions runtime/detrt/core.py and
// runtime/detrt/stage.py:146-233):
//
//   rmsnorm_quant    N1 / N2 (and the final norm before lm_head) fused with the next quant_act
//   qkv_post         QKV dequant -> per-head RMSNorm (Qwen3) -> rope -> per-head int8 quant of
//                    q, k and v, plus V transposed into the attention kernel's key order
//   swiglu_quant     GU dequant -> SiLU(g) * u -> quant_act (SM, QA4)
//   dequant_residual x + dequant(acc) (R1, R2)
//   embed_rows       the embedding gather (EMBED)
//   rmsnorm          det_rmsnorm alone (the final-norm hidden state)
//
// The quantizing row kernels keep a row in the registers of one or four waves; odd widths, wide
// Hadamard blocks and fp32 gate | up rows keep it in LDS (one workgroup of 256 threads per row).
// qkv_post gives four heads to a wave, one per 16-lane row. Every fp32 step is one correctly rounded op in the reference's
// order (uwc_rows.h).
#include "uwc_rows.h"

// ------------------------------------------------------------------ rmsnorm (+ quant_act)
template <bool QUANT>
__global__ void __launch_bounds__(256) rmsnorm_kernel(const float* __restrict__ x, const float* __restrict__ w, int k,
                                                      int bs, float inv_d, float eps, i8* __restrict__ q,
                                                      float* __restrict__ scale, float* __restrict__ y) {
  extern __shared__ float dx_row[];
  __shared__ DxRed red;
  const long r = blockIdx.x;
  const float* xr = x + r * k;
  for (int i = threadIdx.x; i < k; i += 256) dx_row[i] = xr[i];
  __syncthreads();
  dx_rmsnorm_lds(dx_row, k, w, inv_d, eps, red);
  if constexpr (QUANT) {
    if (k % 512 == 0 && bs <= 512 && (bs <= 1 || (bs & (bs - 1)) == 0))
      dx_quant_lds_g(dx_row, k, bs > 1 ? __builtin_ctz(bs) : 0, 64, q + r * k, scale + r, red);
    else
      dx_quant_lds(dx_row, k, bs, 64, q + r * k, scale + r, red);
  } else {
    float* yr = y + r * k;
    for (int i = threadIdx.x; i < k; i += 256) yr[i] = dx_row[i];
  }
}

// A row in the registers of W waves (W = 1: a wave has its row to itself; W > 1: the workgroup's waves
// share one), G 512-element groups per wave: wave w of the row holds groups w, w + W, ..., lane L
// elements 8 L .. 8 L + 7 of each (the layout of fwht512_rows). k % 8 == 0: lanes past the row's end
// hold zeros and neither load nor store (bs divides k, so the transform keeps them zero).
// TAIL: the row has such lanes (without them every test of the row's end is left out: 4% of a
// 4096 x 2048 rmsnorm_quant).
// One wave per row needs no LDS and no barrier, and the work that does not grow with the row runs
// once; more waves per row finish it sooner and hold a part of the registers each. Where the line
// lies for rmsnorm_quant and for swiglu_quant, whose work per element is several times that, stands at
// their dispatch.
struct RowRed {
  float f[2][4];
  long long l[4];
};

// max / int64 sum over the row's waves (slot: a reduction of its own of the workgroup's RowRed)
template <int W>
__device__ __forceinline__ float row_max(float v, RowRed& red, int slot) {
  v = wave_max(v);
  if constexpr (W > 1) {
    if ((threadIdx.x & 63) == 0) red.f[slot][threadIdx.x >> 6] = v;
    __syncthreads();
    v = red.f[slot][0];
#pragma unroll
    for (int i = 1; i < W; i++) v = fmaxf(v, red.f[slot][i]);
  }
  return v;
}
template <int W>
__device__ __forceinline__ long long row_sum64(long long v, RowRed& red) {
  v = wave_sum64(v);
  if constexpr (W > 1) {
    if ((threadIdx.x & 63) == 0) red.l[threadIdx.x >> 6] = v;
    __syncthreads();
    v = red.l[0] + red.l[1] + red.l[2] + red.l[3];
  }
  return v;
}

// quant_act (qmax 64, dx_quant_lds_g's ops) of a row held as above: the transform, the row's max
// |y|, one 8-byte store per group and lane, the scale by the row's first lane.
template <int G, int W, bool TAIL>
__device__ __forceinline__ void quant_row_regs(float (&y)[G][8], int lane, int w, int k, int lbs, i8* __restrict__ qrow,
                                               float* __restrict__ srow, RowRed& red) {
  const bool neg = fwht512_rows<G>(y, G, lane, lbs);
  float m2 = 0.f;
#pragma unroll
  for (int g = 0; g < G; g++)
#pragma unroll
    for (int j = 0; j < 8; j++) m2 = fmaxf(m2, fabsf(y[g][j]));
  m2 = row_max<W>(m2, red, 1);
  const float fq = 64.0f;
  const float sc = __fdiv_rn(fmaxf(m2, 1e-8f), fq);
  const double rs = neg ? -1.0 / (double)sc : 1.0 / (double)sc;  // the lane holds y or -y
#pragma unroll
  for (int g = 0; g < G; g++) {
    const int at = (g * W + w) * 512 + lane * 8;
    u64 packed = 0;
#pragma unroll
    for (int j = 0; j < 8; j++) {
      const float t = fminf(fmaxf(rintf(uwc_div_rd(y[g][j], rs)), -fq), fq);
      packed |= (u64)(u8)(i8)(int)t << (8 * j);
    }
    if (!TAIL || at < k) *reinterpret_cast<u64*>(qrow + at) = packed;
  }
  if (lane == 0 && w == 0) *srow = lbs > 0 ? __fmul_rn(sc, __fdiv_rn(1.0f, uwc_sqrt_rn((float)(1 << lbs)))) : sc;
}

// rmsnorm + quant_act of rows held in registers (k <= 512 G W, bs = 2^lbs <= 512): the max square
// and the exact fixed-point sum are reductions whose order cannot change the value, then the same
// per-element ops as dx_rmsnorm_lds and dx_quant_lds_g. The 256-thread LDS row kernel's five
// workgroup reductions and LDS passes made it latency-bound (54 us per 8192 x 2048 call against 15
// us of traffic; 25 so).
template <int G, int W, bool TAIL>
__global__ void __launch_bounds__(256) rmsnorm_quant_regs_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                                 int rows, int row_k, int lbs, float inv_d, float eps,
                                                                 i8* __restrict__ q, float* __restrict__ scale) {
  const int k = TAIL || W > 1 ? row_k : 512 * G;
  __shared__ RowRed red;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, wv = W > 1 ? wave : 0;
  const long r = W > 1 ? (long)blockIdx.x : (long)blockIdx.x * 4 + wave;
  if (r >= rows) return;  // W = 1: whole waves, and no barriers below; W = 4: never
  const float* xr = x + r * k;
  float y[G][8];
#pragma unroll
  for (int g = 0; g < G; g++) {
    const int at = (g * W + wv) * 512 + lane * 8;
    float4 a{}, b{};
    if (!TAIL || at < k) a = *reinterpret_cast<const float4*>(xr + at), b = *reinterpret_cast<const float4*>(xr + at + 4);
    y[g][0] = a.x; y[g][1] = a.y; y[g][2] = a.z; y[g][3] = a.w;
    y[g][4] = b.x; y[g][5] = b.y; y[g][6] = b.z; y[g][7] = b.w;
  }
  float mx = 0.f;
#pragma unroll
  for (int g = 0; g < G; g++)
#pragma unroll
    for (int j = 0; j < 8; j++) mx = fmaxf(mx, __fmul_rn(y[g][j], y[g][j]));
  mx = row_max<W>(mx, red, 0);
  const int sh = dx_shift(mx, dx_log2ceil(k));
  long long acc = 0;
#pragma unroll
  for (int g = 0; g < G; g++)
#pragma unroll
    for (int j = 0; j < 8; j++) acc += dx_fix(__fmul_rn(y[g][j], y[g][j]), sh);
  acc = row_sum64<W>(acc, red);
  const float ss = dx_unfix(acc, sh);
  const float rr = __fdiv_rn(1.0f, uwc_sqrt_rn(__fadd_rn(__fmul_rn(ss, inv_d), eps)));
#pragma unroll
  for (int g = 0; g < G; g++) {
    const int at = (g * W + wv) * 512 + lane * 8;
    float4 a{}, b{};
    if (!TAIL || at < k) a = *reinterpret_cast<const float4*>(w + at), b = *reinterpret_cast<const float4*>(w + at + 4);
    const float wvv[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
    for (int j = 0; j < 8; j++) y[g][j] = !TAIL || at < k ? __fmul_rn(__fmul_rn(y[g][j], rr), wvv[j]) : 0.0f;
  }
  quant_row_regs<G, W, TAIL>(y, lane, wv, k, lbs, q + r * k, scale + r, red);
}

// ------------------------------------------------------------------ swiglu + quant_act
// swiglu_quant from int32 gate | up rows held in the registers of W waves (I <= 512 W G, bs <= 512):
// element i = fmul(silu(deq(g_i)), deq(u_i)) as in the LDS row kernel below, then quant_row_regs.
// VALU-bound (det_exp and the division: about 60 instructions an element) where the LDS form waited on
// its nine passes and barriers: I = 14336 at 2000 rows 169 -> 70 us. The test of the row's end stays in
// whole rows of several groups per wave too: without it the compiler loads every group before the first
// is worked on, and the registers cost more than the tests (I = 6144 at 8192 rows 107 -> 113 us).
template <int G, int W, bool TAIL>
__global__ void __launch_bounds__(256) swiglu_quant_regs_kernel(const i32* __restrict__ acc, const float* __restrict__ s3,
                                                                const float* __restrict__ sw, int rows, int row_I, int lbs,
                                                                i8* __restrict__ q, float* __restrict__ scale) {
  const int I = TAIL ? row_I : 512 * G * W;
  __shared__ RowRed red;
  const int lane = threadIdx.x & 63, wave = W > 1 ? threadIdx.x >> 6 : 0;
  const long r = W > 1 ? (long)blockIdx.x : (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (r >= rows) return;  // W = 1: whole waves, and no barriers below; W > 1: never
  const i32* ar = acc + r * 2L * I;
  const float sx = s3[r];
  float y[G][8];
#pragma unroll
  for (int g = 0; g < G; g++) {
    const int at = (W * g + wave) * 512 + lane * 8;
    if (!TAIL || at < I) {
      const v4i g0 = *reinterpret_cast<const v4i*>(ar + at), g1 = *reinterpret_cast<const v4i*>(ar + at + 4);
      const v4i u0 = *reinterpret_cast<const v4i*>(ar + I + at), u1 = *reinterpret_cast<const v4i*>(ar + I + at + 4);
      const float4 wg0 = *reinterpret_cast<const float4*>(sw + at), wg1 = *reinterpret_cast<const float4*>(sw + at + 4);
      const float4 wu0 = *reinterpret_cast<const float4*>(sw + I + at), wu1 = *reinterpret_cast<const float4*>(sw + I + at + 4);
      const int gv[8] = {g0[0], g0[1], g0[2], g0[3], g1[0], g1[1], g1[2], g1[3]};
      const int uv[8] = {u0[0], u0[1], u0[2], u0[3], u1[0], u1[1], u1[2], u1[3]};
      const float wgv[8] = {wg0.x, wg0.y, wg0.z, wg0.w, wg1.x, wg1.y, wg1.z, wg1.w};
      const float wuv[8] = {wu0.x, wu0.y, wu0.z, wu0.w, wu1.x, wu1.y, wu1.z, wu1.w};
#pragma unroll
      for (int j = 0; j < 8; j++) y[g][j] = __fmul_rn(dx_silu(dx_deq(gv[j], sx, wgv[j])), dx_deq(uv[j], sx, wuv[j]));
    } else {
#pragma unroll
      for (int j = 0; j < 8; j++) y[g][j] = 0.0f;
    }
  }
  quant_row_regs<G, W, TAIL>(y, lane, wave, I, lbs, q + r * (long)I, scale + r, red);
}

// acc: rows x 2I (gate | up), int32 accumulators dequantized with s3[row], sw[col], or with FP
// already fp32; row value i = fmul(silu(g_i), u_i) (stage.py:220-221).
template <bool FP>
__global__ void __launch_bounds__(256) swiglu_quant_kernel(const void* __restrict__ acc, const float* __restrict__ s3,
                                                           const float* __restrict__ sw, int I, int bs,
                                                           i8* __restrict__ q, float* __restrict__ scale) {
  extern __shared__ float dx_row[];
  __shared__ DxRed red;
  const long r = blockIdx.x;
  for (int i = threadIdx.x; i < I; i += 256) {
    float g, u;
    if constexpr (FP) {
      const float* ar = static_cast<const float*>(acc) + r * 2L * I;
      g = ar[i];
      u = ar[I + i];
    } else {
      const i32* ar = static_cast<const i32*>(acc) + r * 2L * I;
      const float sx = s3[r];
      g = dx_deq(ar[i], sx, sw[i]);
      u = dx_deq(ar[I + i], sx, sw[I + i]);
    }
    dx_row[i] = __fmul_rn(dx_silu(g), u);
  }
  __syncthreads();
  if (I % 512 == 0 && bs <= 512 && (bs <= 1 || (bs & (bs - 1)) == 0))
    dx_quant_lds_g(dx_row, I, bs > 1 ? __builtin_ctz(bs) : 0, 64, q + r * (long)I, scale + r, red);
  else
    dx_quant_lds(dx_row, I, bs, 64, q + r * (long)I, scale + r, red);
}

// ------------------------------------------------------------------ residual
// out = fadd(x, fmul(fmul(f32(acc), s[row]), sw[col])) (stage.py:217, 224); with FP acc is the
// already dequantized fp32 term.
template <bool FP>
__global__ void dequant_residual_kernel(const void* __restrict__ acc, const float* __restrict__ s,
                                        const float* __restrict__ sw, const float* __restrict__ x, int n, u64 total,
                                        float* __restrict__ out) {
  for (u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (u64)gridDim.x * blockDim.x) {
    float y;
    if constexpr (FP) {
      y = static_cast<const float*>(acc)[i];
    } else {
      const u64 r = i / (u64)n;
      const int c = (int)(i - r * n);
      y = dx_deq(static_cast<const i32*>(acc)[i], s[r], sw[c]);
    }
    out[i] = __fadd_rn(x[i], y);
  }
}

// ------------------------------------------------------------------ embedding gather
// out[t] = table[ids[t]]; an id outside [0, V) yields a zero row and bumps *bad (never read out
// of bounds).
__global__ void embed_kernel(const float* __restrict__ table, long V, int D, const int64_t* __restrict__ ids, int N,
                             float* __restrict__ out, int* __restrict__ bad) {
  const int t = blockIdx.x;
  if (t >= N) return;
  const int64_t id = ids[t];
  const bool ok = id >= 0 && id < V;
  if (!ok && threadIdx.x == 0 && bad) atomicAdd(bad, 1);
  const float* src = table + (ok ? id : 0) * (long)D;
  float* dst = out + (long)t * D;
  for (int i = threadIdx.x; i < D; i += blockDim.x) dst[i] = ok ? src[i] : 0.0f;
}

// ------------------------------------------------------------------ qkv_post
// Position of key j inside its 64-key block in the transposed V the attention kernel reads:
// key 16 kb + 4 kg + ki sits at 16 kg + 4 kb + ki (the order in which a 16x16 score block's
// C registers hand keys to the P x V MFMA's k slots).
__host__ __device__ __forceinline__ int vt_pos(int j) {
  return (j & ~63) | (((j >> 2) & 3) << 4) | (((j >> 4) & 3) << 2) | (j & 3);
}

// Four heads per wave: each 16-lane row of a wave holds one head, a lane NV = HD / 16 adjacent
// dims, so the per-head work that does not grow with the head's size (the row maxima and the
// exact sum of squares as 4-step DPP reductions inside the row, the shift, the correctly rounded
// square root and divisions, the float64 reciprocal) runs once per four heads, and every load
// and store of a lane is one contiguous vector. The rope's partner of dim d is d +- HD / 2, the
// same register of lane l ^ 8 in the row (DPP row_ror:8); rot's sign rides on sin (fl(-a b) is
// -fl(a b)). Heads 16 p + 4 w + r for pass p, wave w, row r, so a row's head is one kind (q, k
// or v) and a branch on it splits rows, never a row.
//
// One workgroup takes QP_TOKENS consecutive tokens, each pass of a wave its tokens in turn; the
// column scales of a pass are loaded once for the four. A V head's quantized bytes of the 4
// tokens stay in the row's registers, so when the tokens are positions 4a .. 4a + 3 of one
// sequence (vt_pos keeps those 4 adjacent) each transposed row gets one 4-byte store instead of 4
// byte stores to rows Tp bytes apart.
#define QP_TOKENS 4
template <int HD, bool FP>
__global__ void __launch_bounds__(256) qkv_post_kernel(
    const void* __restrict__ acc, const float* __restrict__ s1, const float* __restrict__ sw,
    const float* __restrict__ qnw, const float* __restrict__ knw, const float* __restrict__ cosb,
    const float* __restrict__ sinb, long N, int T, int H, int Hkv, float inv_hd, float eps, int qknorm,
    i8* __restrict__ qq, float* __restrict__ qs, i8* __restrict__ kq, float* __restrict__ ks, i8* __restrict__ vq,
    float* __restrict__ vs, i8* __restrict__ vt, int Tp) {
  constexpr int NV = HD / 16;  // dims per lane
  constexpr int L = HD == 32 ? 5 : HD == 64 ? 6 : 7;  // log2(HD)
  constexpr int TK = QP_TOKENS;
  static_assert(TK == 4, "a transposed row's 4-byte store holds the bytes of exactly 4 tokens");
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, row = lane >> 4, sl = lane & 15;
  const int d0 = NV * sl;
  const long n0 = (long)blockIdx.x * TK;
  const int nt = (int)min((long)TK, N - n0);  // tokens of this workgroup (>= 1)
  const int NH = H + 2 * Hkv;
  const long W = (long)NH * HD;
  int pos[TK], bs[TK];
  float sx[TK];
#pragma unroll
  for (int t = 0; t < TK; t++) {
    const long n = n0 + min(t, nt - 1);
    pos[t] = (int)(n % T);
    bs[t] = (int)(n / T);
    sx[t] = FP ? 1.0f : s1[n];
  }
  const bool packed = nt == TK && bs[0] == bs[TK - 1] && (pos[0] & 3) == 0 && ((uintptr_t)vt & 3) == 0;
  // NV consecutive floats, 16-byte aligned for NV >= 4 (8-byte for NV = 2): the host checks the
  // bases, and every offset used here is a multiple of NV
  auto ldv = [](const float* p, float (&v)[NV]) {
    if constexpr (NV % 4 == 0) {
#pragma unroll
      for (int j = 0; j < NV; j += 4) {
        const float4 x = *reinterpret_cast<const float4*>(p + j);
        v[j] = x.x, v[j + 1] = x.y, v[j + 2] = x.z, v[j + 3] = x.w;
      }
    } else {
      const float2 x = *reinterpret_cast<const float2*>(p);
      v[0] = x.x, v[1] = x.y;
    }
  };
  float qn[NV], kn[NV];
  if (qknorm) {
    ldv(qnw + d0, qn);
    ldv(knw + d0, kn);
  }
  const bool low = sl < 8;  // the row's lanes holding the first half of the head
  for (int p = 0; p * 16 < NH; p++) {
    const int hh = 16 * p + 4 * wave + row;  // this row's head
    const bool live = hh < NH;
    const int hc = min(hh, NH - 1);
    const bool isq = hc < H, isv = hc >= H + Hkv;
    const int col = hc * HD + d0;
    float swv[NV];
    if constexpr (!FP) ldv(sw + col, swv);
    u32 pk[NV];
#pragma unroll
    for (int j = 0; j < NV; j++) pk[j] = 0;
#pragma unroll
    for (int t = 0; t < TK; t++) {
      if (t >= nt) break;
      const long n = n0 + t;
      float v[NV];
      if constexpr (FP) {
        ldv(static_cast<const float*>(acc) + n * W + col, v);
      } else {
        const i32* a = static_cast<const i32*>(acc) + n * W + col;
        int av[NV];
        if constexpr (NV % 4 == 0) {
#pragma unroll
          for (int j = 0; j < NV; j += 4) {
            const int4 x = *reinterpret_cast<const int4*>(a + j);
            av[j] = x.x, av[j + 1] = x.y, av[j + 2] = x.z, av[j + 3] = x.w;
          }
        } else {
          const int2 x = *reinterpret_cast<const int2*>(a);
          av[0] = x.x, av[1] = x.y;
        }
#pragma unroll
        for (int j = 0; j < NV; j++) v[j] = dx_deq(av[j], sx[t], swv[j]);
      }
      if (!isv) {
        if (qknorm) {  // det_rmsnorm over the head (qwen3.py:214-216)
          float mx = 0.f;
#pragma unroll
          for (int j = 0; j < NV; j++) mx = fmaxf(mx, __fmul_rn(v[j], v[j]));
          const int sh = dx_shift(row16_max(mx), L);
          long long sq = 0;
#pragma unroll
          for (int j = 0; j < NV; j++) sq += dx_fix(__fmul_rn(v[j], v[j]), sh);
          const float ss = dx_unfix(row16_sum64(sq), sh);
          const float r = __fdiv_rn(1.0f, uwc_sqrt_rn(__fadd_rn(__fmul_rn(ss, inv_hd), eps)));
#pragma unroll
          for (int j = 0; j < NV; j++) v[j] = __fmul_rn(__fmul_rn(v[j], r), isq ? qn[j] : kn[j]);
        }
        // rope: fadd(fmul(z, cos), fmul(rot(z), sin)), rot(z) = cat(-z[half:], z[:half])
        float cs[NV], sn[NV];
        ldv(cosb + (long)pos[t] * HD + d0, cs);
        ldv(sinb + (long)pos[t] * HD + d0, sn);
        float part[NV];
#pragma unroll
        for (int j = 0; j < NV; j++) part[j] = qa_dpp<0x128>(v[j]);  // row_ror:8: lane l ^ 8 of the row
#pragma unroll
        for (int j = 0; j < NV; j++) v[j] = __fadd_rn(__fmul_rn(v[j], cs[j]), __fmul_rn(part[j], low ? -sn[j] : sn[j]));
      }
      // quant_sym(qmax = 127) over the head (core.py:160-166)
      float am = 0.f;
#pragma unroll
      for (int j = 0; j < NV; j++) am = fmaxf(am, fabsf(v[j]));
      const float s = __fdiv_rn(fmaxf(row16_max(am), 1e-8f), 127.0f);
      const double rs = 1.0 / (double)s;
      u32 qb[NV / 2];  // the lane's NV quantized bytes, 2 per 16-bit half (NV >= 2)
#pragma unroll
      for (int j = 0; j < NV; j++) {
        const int qv = (int)fminf(fmaxf(rintf(uwc_div_rd(v[j], rs)), -127.f), 127.f);
        const u32 b = (u32)qv & 0xffu;
        if (j % 2 == 0) qb[j / 2] = b;
        else qb[j / 2] |= b << 8;
        if (packed) pk[j] |= b << (8 * t);
      }
      if (live) {
        i8* qo;
        float* so;
        if (isq) {
          qo = qq + (n * H + hh) * HD;
          so = qs + n * H + hh;
        } else if (!isv) {
          qo = kq + (n * Hkv + (hh - H)) * HD;
          so = ks + n * Hkv + (hh - H);
        } else {
          qo = vq + (n * Hkv + (hh - H - Hkv)) * HD;
          so = vs + n * Hkv + (hh - H - Hkv);
        }
        if constexpr (NV == 2) {
          *reinterpret_cast<unsigned short*>(qo + d0) = (unsigned short)qb[0];
        } else {
#pragma unroll
          for (int j = 0; j < NV / 4; j++)
            *reinterpret_cast<u32*>(qo + d0 + 4 * j) = qb[2 * j] | (qb[2 * j + 1] << 16);
        }
        if (sl == 0) *so = s;
        if (vt && isv && !packed) {
          const int hk = hh - H - Hkv;
#pragma unroll
          for (int j = 0; j < NV; j++)
            vt[((long)(bs[t] * Hkv + hk) * HD + d0 + j) * Tp + vt_pos(pos[t])] = (i8)((qb[j / 2] >> (8 * (j % 2))) & 0xff);
        }
      }
    }
    if (live && vt && isv && packed) {
      const int hk = hh - H - Hkv;
#pragma unroll
      for (int j = 0; j < NV; j++)
        *reinterpret_cast<u32*>(vt + ((long)(bs[0] * Hkv + hk) * HD + d0 + j) * Tp + vt_pos(pos[0])) = pk[j];
    }
  }
}

// V (N x Hkv x HD int8) transposed per (sequence, kv head) into the attention kernel's layout.
__global__ void v_transpose_kernel(const i8* __restrict__ vq, int T, int Hkv, int HD, int Tp, i8* __restrict__ vt) {
  const int n = blockIdx.x, bseq = n / T, pos = n % T;
  for (int i = threadIdx.x; i < Hkv * HD; i += blockDim.x) {
    const int hk = i / HD, d = i % HD;
    vt[((long)(bseq * Hkv + hk) * HD + d) * Tp + vt_pos(pos)] = vq[(long)n * Hkv * HD + i];
  }
}

// ------------------------------------------------------------------ per-op conformance
// out[i] = op(x[i], y[i]) for one of detrt's elementwise fp32 ops, as the kernels above compute
// it: the per-op check of native fp32 against detrt's emulation (runtime/tests/test_fp32_native.py).
__global__ void det_elementwise_kernel(int op, const float* __restrict__ x, const float* __restrict__ y,
                                       float* __restrict__ out, u64 n) {
  for (u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (u64)gridDim.x * blockDim.x) {
    const float a = x[i], b = y ? y[i] : 0.0f;
    float r;
    switch (op) {
      case UWC_OP_ADD: r = __fadd_rn(a, b); break;
      case UWC_OP_SUB: r = __fsub_rn(a, b); break;
      case UWC_OP_MUL: r = __fmul_rn(a, b); break;
      case UWC_OP_DIV: r = __fdiv_rn(a, b); break;
      case UWC_OP_SQRT: r = uwc_sqrt_rn(a); break;
      case UWC_OP_EXP: r = dx_exp(a); break;
      default: r = dx_silu(a); break;
    }
    out[i] = r;
  }
}

// ------------------------------------------------------------------ C-ABI
extern "C" int uwc_det_elementwise(int op, const float* x, const float* y, float* out, int64_t n, hipStream_t stream) {
  const char* fn = "uwc_det_elementwise";
  if (op < UWC_OP_ADD || op > UWC_OP_SILU) return uwc_fail("%s: unknown op %d", fn, op);
  if (!x || !out || n < 0 || (op <= UWC_OP_DIV && !y)) return uwc_fail("%s: null or empty arguments", fn);
  if (n == 0) return UWC_OK;
  const u64 blocks = ((u64)n + 255) / 256;
  hipLaunchKernelGGL(det_elementwise_kernel, dim3((unsigned)(blocks < 65536 ? blocks : 65536)), dim3(256), 0, stream,
                     op, x, y, out, (u64)n);
  return uwc_launch_status(fn);
}

static int row_lds(const char* fn, const void* kern, int k, size_t& smem) {
  smem = (size_t)k * 4;
  if (smem > 160 * 1024) return uwc_fail("%s: a row of %d floats exceeds LDS", fn, k);
  if (smem > 64 * 1024) {
    hipError_t e = hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
    if (e != hipSuccess) return uwc_fail("%s: cannot raise LDS to %zu bytes: %s", fn, smem, hipGetErrorString(e));
  }
  return UWC_OK;
}

static int check_bs(const char* fn, int bs, int k) {
  if (bs > 1 && ((bs & (bs - 1)) || k % bs)) return uwc_fail("%s: bs=%d must be a power of two dividing %d", fn, bs, k);
  return UWC_OK;
}

extern "C" int uwc_rmsnorm_quant_f32(const float* x, const float* w, int rows, int k, int bs, float inv_d, float eps,
                                     int8_t* q, float* scale, hipStream_t stream) {
  const char* fn = "uwc_rmsnorm_quant_f32";
  if (!x || !w || !q || !scale || rows < 0 || k <= 0) return uwc_fail("%s: null or empty arguments", fn);
  int st = check_bs(fn, bs, k);
  if (st) return st;
  if (rows == 0) return UWC_OK;
  const int bse = bs > 1 ? bs : 1;
  if (k % 8 == 0 && k <= 16384 && bse <= 512 && ((uintptr_t)x & 15) == 0 && ((uintptr_t)w & 15) == 0 &&
      ((uintptr_t)q & 7) == 0) {
    const int lbs = __builtin_ctz((unsigned)bse);
#define RMSQ(G, W)                                                                                                        \
  case G:                                                                                                                 \
    return uwc_launch_rows(fn, rows, 256, [&](long r0, int n) {                                                           \
      hipLaunchKernelGGL((k % (512 * W) ? rmsnorm_quant_regs_kernel<G, W, true> : rmsnorm_quant_regs_kernel<G, W, false>), \
                         dim3((unsigned)(W > 1 ? n : (n + 3) / 4)), dim3(256), 0, stream, x + r0 * k, w, n, k, lbs, inv_d,  \
                         eps, q + r0 * k, scale + r0);                                                                    \
    });
    // four waves per row up to per_cu rows per CU, one beyond (us, one wave / four: k = 2048 5.5 / 4.0 at
    // 200 rows, 5.7 / 5.4 at 600, 5.7 / 6.1 at 777, 7.2 / 7.4 at 1200, 22 / 28 at 8192; k = 4096 9.1 / 8.1 at
    // 1000). One wave has no tail tests in whole rows and four leave some of theirs without a group at 1536
    // and 2560 (1536: 4.8 / 5.3 at 600 rows), so whole rows turn earlier there and take one wave throughout
    // up to 1024 (4.0 / 6.0 at 1000 rows); 768: 4.2 / 3.9 at 200 rows, 4.3 / 5.0 at 600. Past 4096 one wave
    // cannot hold a row.
    const int per_cu = k > 3584 ? 4 : k <= 1024 ? k > 512 && k % 512 : k % 512 == 0 && k % 2048 && k < 3072 ? 2 : 3;
    if (k > 4096 || rows <= per_cu * uwc_cu_count()) {
      switch ((k + 2047) / 2048) { RMSQ(1, 4) RMSQ(2, 4) RMSQ(3, 4) RMSQ(4, 4) RMSQ(5, 4) RMSQ(6, 4) RMSQ(7, 4) RMSQ(8, 4) }
    } else {
      switch ((k + 511) / 512) { RMSQ(1, 1) RMSQ(2, 1) RMSQ(3, 1) RMSQ(4, 1) RMSQ(5, 1) RMSQ(6, 1) RMSQ(7, 1) RMSQ(8, 1) }
    }
#undef RMSQ
  }
  size_t smem;
  if ((st = row_lds(fn, (const void*)rmsnorm_kernel<true>, k, smem))) return st;
  return uwc_launch_rows(fn, rows, 256, [&](long r0, int n) {
    hipLaunchKernelGGL(rmsnorm_kernel<true>, dim3((unsigned)n), dim3(256), smem, stream, x + r0 * k, w, k, bs, inv_d, eps,
                       q + r0 * k, scale + r0, (float*)nullptr);
  });
}

extern "C" int uwc_rmsnorm_f32(const float* x, const float* w, int rows, int k, float inv_d, float eps, float* y,
                               hipStream_t stream) {
  const char* fn = "uwc_rmsnorm_f32";
  if (!x || !w || !y || rows < 0 || k <= 0) return uwc_fail("%s: null or empty arguments", fn);
  if (rows == 0) return UWC_OK;
  size_t smem;
  int st = row_lds(fn, (const void*)rmsnorm_kernel<false>, k, smem);
  if (st) return st;
  return uwc_launch_rows(fn, rows, 256, [&](long r0, int n) {
    hipLaunchKernelGGL(rmsnorm_kernel<false>, dim3((unsigned)n), dim3(256), smem, stream, x + r0 * k, w, k, 0, inv_d, eps,
                       (i8*)nullptr, (float*)nullptr, y + r0 * k);
  });
}

extern "C" int uwc_swiglu_quant(const void* acc, const float* s3, const float* sw, int rows, int I, int bs,
                                int8_t* q, float* scale, hipStream_t stream) {
  const char* fn = "uwc_swiglu_quant";
  if (!acc || !q || !scale || rows < 0 || I <= 0) return uwc_fail("%s: null or empty arguments", fn);
  if (!s3 != !sw) return uwc_fail("%s: give both scales (int32 acc) or neither (fp32 rows)", fn);
  int st = check_bs(fn, bs, I);
  if (st) return st;
  if (rows == 0) return UWC_OK;
  const int bse = bs > 1 ? bs : 1;
  if (s3 && I % 8 == 0 && I > 256 && I <= 16384 && bse <= 512 && ((uintptr_t)acc & 15) == 0 && ((uintptr_t)sw & 15) == 0 &&
      ((uintptr_t)q & 7) == 0) {
    const int lbs = __builtin_ctz((unsigned)bse);
    const i32* a = static_cast<const i32*>(acc);
#define SWQ(G, W, TAIL)                                                                                            \
  return uwc_launch_rows(fn, rows, 256, [&](long r0, int n) {                                                      \
    hipLaunchKernelGGL((swiglu_quant_regs_kernel<G, W, TAIL>), dim3((unsigned)(W > 1 ? n : (n + 3) / 4)),          \
                       dim3(W > 1 ? 64 * W : 256), 0, stream, a + r0 * 2 * I, s3 + r0, sw, n, I, lbs, q + r0 * I, \
                       scale + r0);                                                                                \
  })
    // a wave per 512-element group up to four (us against four waves whatever the width: I = 512 at 1000 /
    // 8192 / 32768 rows 4.8 -> 3.9 / 18.7 -> 11.0 / 63 -> 32; 1024 at 700 rows 4.9 -> 4.7; 1536 at 1200 rows
    // 6.9 -> 6.5), but one wave with two groups for many rows of 1024 (8192 rows 23.1 -> 18.6). Wider rows: four
    // beat one at every row count (I = 6144: 18.9 -> 7.2 at 200, 36.9 -> 29.2 at 2000, 124 -> 107 at 8192).
    // Rows of at most 256 elements keep the LDS form, a thread per element (256 x 64 3.8 -> 3.5, 8192 x 64 15 -> 10).
    if (I == 512) SWQ(1, 1, false);
    if (I == 1024 && rows > 4 * uwc_cu_count()) SWQ(2, 1, false);
    if (I == 1536) SWQ(1, 3, false);
    switch ((I + 511) / 512) {
      case 1: SWQ(1, 1, true);
      case 2: SWQ(1, 2, true);
      case 3: SWQ(1, 3, true);
    }
    switch ((I + 2047) / 2048) {
      case 1: SWQ(1, 4, true);
      case 2: SWQ(2, 4, true);
      case 3: SWQ(3, 4, true);
      case 4: SWQ(4, 4, true);
      case 5: SWQ(5, 4, true);
      case 6: SWQ(6, 4, true);
      case 7: SWQ(7, 4, true);
      case 8: SWQ(8, 4, true);
    }
#undef SWQ
  }
  size_t smem;
  const auto kern = s3 ? swiglu_quant_kernel<false> : swiglu_quant_kernel<true>;
  if ((st = row_lds(fn, (const void*)kern, I, smem))) return st;
  return uwc_launch_rows(fn, rows, 256, [&](long r0, int n) {
    hipLaunchKernelGGL(kern, dim3((unsigned)n), dim3(256), smem, stream, static_cast<const u32*>(acc) + r0 * 2 * I,
                       s3 ? s3 + r0 : nullptr, sw, I, bs, q + r0 * I, scale + r0);
  });
}

extern "C" int uwc_dequant_residual(const void* acc, const float* s, const float* sw, const float* x, int rows, int n,
                                    float* out, hipStream_t stream) {
  const char* fn = "uwc_dequant_residual";
  if (!acc || !x || !out || rows < 0 || n <= 0) return uwc_fail("%s: null or empty arguments", fn);
  if (!s != !sw) return uwc_fail("%s: give both scales (int32 acc) or neither (fp32 rows)", fn);
  const u64 total = (u64)rows * n;
  if (total == 0) return UWC_OK;
  const u64 blocks = (total + 255) / 256;
  const dim3 grid((unsigned)(blocks < 65536 ? blocks : 65536));
  if (s)
    hipLaunchKernelGGL(dequant_residual_kernel<false>, grid, dim3(256), 0, stream, acc, s, sw, x, n, total, out);
  else
    hipLaunchKernelGGL(dequant_residual_kernel<true>, grid, dim3(256), 0, stream, acc, s, sw, x, n, total, out);
  return uwc_launch_status(fn);
}

extern "C" int uwc_embed_rows(const float* table, int64_t V, int D, const int64_t* ids, int N, float* out, int* bad,
                              hipStream_t stream) {
  const char* fn = "uwc_embed_rows";
  if (!table || !ids || !out || V <= 0 || D <= 0 || N < 0) return uwc_fail("%s: null or empty arguments", fn);
  if (N == 0) return UWC_OK;
  return uwc_launch_rows(fn, N, 256, [&](long r0, int n) {
    hipLaunchKernelGGL(embed_kernel, dim3((unsigned)n), dim3(256), 0, stream, table, (long)V, D, ids + r0, n, out + r0 * D,
                       bad);
  });
}

extern "C" int uwc_vt_tokens(int T) { return T <= 0 ? 0 : ((T + 63) / 64) * 64; }

extern "C" int uwc_qkv_post(const void* acc, const float* s1, const float* sw, const float* qnw, const float* knw,
                            const float* cosb, const float* sinb, int B, int T, int H, int Hkv, int hd, float eps,
                            int qknorm, int8_t* qq, float* qs, int8_t* kq, float* ks, int8_t* vq, float* vs, int8_t* vt,
                            hipStream_t stream) {
  const char* fn = "uwc_qkv_post";
  if (!acc || !cosb || !sinb || !qq || !qs || !kq || !ks || !vq || !vs) return uwc_fail("%s: null arguments", fn);
  if (!s1 != !sw) return uwc_fail("%s: give both scales (int32 acc) or neither (fp32 rows)", fn);
  if (qknorm && (!qnw || !knw)) return uwc_fail("%s: q/k norm weights are needed with qknorm", fn);
  if (B < 0 || T <= 0 || H <= 0 || Hkv <= 0 || H % Hkv) return uwc_fail("%s: bad B=%d T=%d H=%d Hkv=%d", fn, B, T, H, Hkv);
  if (hd != 32 && hd != 64 && hd != 128) return uwc_fail("%s: head_dim %d not in {32, 64, 128}", fn, hd);
  if (((uintptr_t)acc | (uintptr_t)sw | (uintptr_t)qnw | (uintptr_t)knw | (uintptr_t)cosb | (uintptr_t)sinb |
       (uintptr_t)qq | (uintptr_t)kq | (uintptr_t)vq) & 15)
    return uwc_fail("%s: acc, sw, qnw, knw, cos, sin, qq, kq, vq must be 16-byte aligned", fn);
  const long N = (long)B * T;
  if (N == 0) return UWC_OK;
  if (N > 0x7fffffff) return uwc_fail("%s: too many tokens", fn);
  const float inv_hd = (float)(1.0 / (double)hd);
  const int Tp = uwc_vt_tokens(T);
  const dim3 grid((unsigned)((N + QP_TOKENS - 1) / QP_TOKENS));
#define QKV_LAUNCH(HD)                                                                                               \
  do {                                                                                                               \
    if (s1)                                                                                                          \
      hipLaunchKernelGGL((qkv_post_kernel<HD, false>), grid, dim3(256), 0, stream, acc, s1, sw, qnw, knw, cosb,      \
                         sinb, N, T, H, Hkv, inv_hd, eps, qknorm, qq, qs, kq, ks, vq, vs, vt, Tp);                    \
    else                                                                                                             \
      hipLaunchKernelGGL((qkv_post_kernel<HD, true>), grid, dim3(256), 0, stream, acc, s1, sw, qnw, knw, cosb,       \
                         sinb, N, T, H, Hkv, inv_hd, eps, qknorm, qq, qs, kq, ks, vq, vs, vt, Tp);                    \
  } while (0)
  if (hd == 32) QKV_LAUNCH(32);
  else if (hd == 64) QKV_LAUNCH(64);
  else QKV_LAUNCH(128);
#undef QKV_LAUNCH
  return uwc_launch_status(fn);
}

extern "C" int uwc_v_transpose(const int8_t* vq, int B, int T, int Hkv, int hd, int8_t* vt, hipStream_t stream) {
  const char* fn = "uwc_v_transpose";
  if (!vq || !vt || B < 0 || T <= 0 || Hkv <= 0 || hd <= 0) return uwc_fail("%s: null or empty arguments", fn);
  const long N = (long)B * T;
  if (N == 0) return UWC_OK;
  hipLaunchKernelGGL(v_transpose_kernel, dim3((unsigned)N), dim3(256), 0, stream, vq, T, Hkv, hd, uwc_vt_tokens(T), vt);
  return uwc_launch_status(fn);
}

// ------------------------------------------------------------------ the whole layer
// One host call per layer: at 200 tokens the layer's kernels take about 95 us, and queueing them one
// Python call at a time took 125 (an allocation or two, the stream lookup and the argument
// conversion of every op around 3 us of launch).
namespace {
struct LayerArena {  // byte offsets in the scratch
  uint64_t q, s, s4, x, heads, kq, vq, qs, ks, vs, vt, oc, r1, total;
};
uint64_t up256(uint64_t n) { return (n + 255) & ~255ull; }

LayerArena layer_arena(int B, int T, int D, int H, int Hkv, int hd, int I, int stored_exp) {
  const uint64_t N = (uint64_t)B * T, QH = (uint64_t)H * hd, KH = (uint64_t)Hkv * hd;
  uint64_t widest = (uint64_t)D > QH ? (uint64_t)D : QH;
  if ((uint64_t)I > widest) widest = I;
  // the int32 products of qkv and gate_up and the attention's exponentials follow each other: one place
  uint64_t big = N * (QH + 2 * KH) * 4;
  if (N * 2 * I * 4 > big) big = N * 2 * I * 4;
  const uint64_t es = stored_exp ? uwc_attention_scratch_bytes(B, T, H) : 0;
  if (es > big) big = es;
  LayerArena a{};
  uint64_t at = 0;
  auto take = [&](uint64_t bytes) {
    const uint64_t o = at;
    at += up256(bytes);
    return o;
  };
  a.q = take(N * widest);
  a.s = take(N * 4);
  a.s4 = take(N * 4);  // swiglu_quant reads gate_up's row scales and writes down's
  a.x = take(big);
  a.heads = take(N * QH);
  a.kq = take(N * KH);
  a.vq = take(N * KH);
  a.qs = take(N * H * 4);
  a.ks = take(N * Hkv * 4);
  a.vs = take(N * Hkv * 4);
  a.vt = take((uint64_t)B * KH * uwc_vt_tokens(T));
  a.oc = take(N * QH * 4);
  a.r1 = take(N * D * 4);
  a.total = at;
  return a;
}
}  // namespace

extern "C" uint64_t uwc_decoder_layer_scratch_bytes(int B, int T, int D, int H, int Hkv, int hd, int I, int stored_exp) {
  if (B <= 0 || T <= 0 || D <= 0 || H <= 0 || Hkv <= 0 || hd <= 0 || I <= 0) return 0;
  return layer_arena(B, T, D, H, Hkv, hd, I, stored_exp).total;
}

extern "C" int uwc_decoder_layer_f32(const float* x, int B, int T, int D, int H, int Hkv, int hd, int I,
                                     const float* in_norm, const float* post_norm, const float* q_norm,
                                     const float* k_norm, const float* cos_tab, const float* sin_tab, const int8_t* Wqkv,
                                     const float* sqkv, int bs_qkv, const int8_t* Wo, const float* so, int bs_o,
                                     const int8_t* Wgu, const float* sgu, int bs_gu, const int8_t* Wdown,
                                     const float* sdown, int bs_down, float inv_d, float eps, float inv_sqrt_hd,
                                     int qknorm, int stored_exp, void* scratch, uint64_t scratch_bytes, float* out,
                                     hipStream_t stream) {
  const char* fn = "uwc_decoder_layer_f32";
  if (B <= 0 || T <= 0 || D <= 0 || H <= 0 || Hkv <= 0 || hd <= 0 || I <= 0 || (int64_t)B * T > 0x7fffffff)
    return uwc_fail("%s: bad B=%d T=%d D=%d H=%d Hkv=%d hd=%d I=%d", fn, B, T, D, H, Hkv, hd, I);
  if (!x || !out || !scratch || ((uintptr_t)scratch & 255)) return uwc_fail("%s: null x or out, or a scratch not 256-byte aligned", fn);
  const LayerArena a = layer_arena(B, T, D, H, Hkv, hd, I, stored_exp);
  if (scratch_bytes < a.total)
    return uwc_fail("%s: scratch holds %llu bytes, need %llu", fn, (unsigned long long)scratch_bytes, (unsigned long long)a.total);
  const int N = B * T, QH = H * hd, WQ = (H + 2 * Hkv) * hd;
  char* at = static_cast<char*>(scratch);
  int8_t* q = reinterpret_cast<int8_t*>(at + a.q);
  float *s = reinterpret_cast<float*>(at + a.s), *s4 = reinterpret_cast<float*>(at + a.s4);
  int32_t* acc = reinterpret_cast<int32_t*>(at + a.x);
  float* es = reinterpret_cast<float*>(at + a.x);
  int8_t *qq = reinterpret_cast<int8_t*>(at + a.heads), *kq = reinterpret_cast<int8_t*>(at + a.kq),
         *vq = reinterpret_cast<int8_t*>(at + a.vq), *vt = reinterpret_cast<int8_t*>(at + a.vt);
  float *qs = reinterpret_cast<float*>(at + a.qs), *ks = reinterpret_cast<float*>(at + a.ks),
        *vs = reinterpret_cast<float*>(at + a.vs), *oc = reinterpret_cast<float*>(at + a.oc),
        *r1 = reinterpret_cast<float*>(at + a.r1);
  int st;
  if ((st = uwc_rmsnorm_quant_f32(x, in_norm, N, D, bs_qkv, inv_d, eps, q, s, stream))) return st;
  if ((st = uwc_igemm_i32(q, Wqkv, N, WQ, D, acc, stream))) return st;
  // vt's keys past T (T % 64) keep whatever the scratch held: they only meet zero probabilities
  if ((st = uwc_qkv_post(acc, s, sqkv, q_norm, k_norm, cos_tab, sin_tab, B, T, H, Hkv, hd, eps, qknorm, qq, qs, kq, ks, vq,
                         vs, vt, stream)))
    return st;
  if (stored_exp)
    st = uwc_attention_ws(qq, qs, kq, ks, vt, vs, B, T, H, Hkv, hd, inv_sqrt_hd, oc, es,
                          uwc_attention_scratch_bytes(B, T, H), stream);
  else
    st = uwc_attention(qq, qs, kq, ks, vt, vs, B, T, H, Hkv, hd, inv_sqrt_hd, oc, stream);
  if (st) return st;
  if ((st = uwc_quant_act_f32(oc, N, QH, bs_o, 64, q, s, stream))) return st;
  if ((st = uwc_igemm_dequant_residual_f32(q, Wo, N, D, QH, s, so, x, r1, stream))) return st;
  if ((st = uwc_rmsnorm_quant_f32(r1, post_norm, N, D, bs_gu, inv_d, eps, q, s, stream))) return st;
  if ((st = uwc_igemm_i32(q, Wgu, N, 2 * I, D, acc, stream))) return st;
  if ((st = uwc_swiglu_quant(acc, s, sgu, N, I, bs_down, q, s4, stream))) return st;
  return uwc_igemm_dequant_residual_f32(q, Wdown, N, D, I, s4, sdown, r1, out, stream);
}
