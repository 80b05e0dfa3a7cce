// The per-nonce operand side of a mined forward in one launch, for any rank: the noised operand
// A' = A + E[first] - E[second], the projections X = A StB^T and Y = B' StA^T as balanced base-128 limbs
// with max |X|, max |Y|, and the E copy (miner/ampere/uwc_ampere/kernels.cu:303-404, ops.py:331-336).
//
// A projection is an int8 product with r columns. The row kernels (uwc_noise.hip) give 16 rows to a
// workgroup, which at 1024 rows leaves three quarters of the CUs without one and every workgroup with a
// serial walk over k (rank 128, 1024 x 6144 and 2048 x 6144: 33 + 29 us). Here workgroups take roles:
//   * projection tiles of BT x BT: each of four waves multiplies the tile over every fourth 128-wide
//     k step from its own DMA-fed LDS ring, and the partial sums meet in LDS (as the small tiles of
//     uwc_gemm_plain.hip; int32 sums are exact in any order);
//   * noise blocks of 16 rows x 512 columns: the rows of E and the block's pairs in LDS, two byte
//     lookups per element.
// BT = 64 halves the DMA per product and is taken when its tiles alone reach half of the CUs (1024 x
// 4096 x 2048, 160 such tiles: 16.5 us on 32 x 32 tiles, 10.1 on 64 x 64). Measured (us per call, m x n
// x k, rank 128, the row kernels -> this): 1024 x 2048 x 2048 26.8 -> 10.2, 1024 x 12288 x 2048 44.8 ->
// 16.2, 1024 x 2048 x 6144 58.8 -> 18.4, 4096 x 4096 x 4096 48.6 -> 27.8. There the noise blocks bound
// it: few waves beside the tiles' LDS, two dependent byte lookups per element (uwc_side.hip's noise on
// the matrix cores is faster at rank 64: 17.2 against 19.7).
#include "uwc_dma.h"

namespace {

#define ST_WAVES 4
#define ST_THREADS (ST_WAVES * 64)
#define ST_NROWS 16   // rows of a noise block
#define ST_NCOLS 512  // its columns
#define ST_MAXR 128

struct SideTilesParams {
  const i8 *A, *EA;
  const u32* PA;
  i8* ApEA;
  const i8* StB;
  i8* corrA;
  const i8* Bp;
  const i8* StA;
  i8* corrB;
  i32* maxabs;
  int m, n, k, r, lmax, corr_a_off, ecopy_off, corr_b_off;
};

// One BT x BT tile of src (rows x k) * St^T (r x k): limbs at corr[li][row][off + j], max into *mx.
template <int BT, int S>
__device__ __forceinline__ void side_tile(u8* sm, int* wmax, const i8* src, int rows, int k, const i8* St, int r, int tile,
                                          i8* corr, int off, int lmax, i32* mx) {
  typedef Mfma<32> MM;
  constexpr int NB = BT / 32, SEG = BT / 4, STG = 2 * BT * P_BK, PC = BT / 4, NP = MM::PASSES;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int cols = r / BT, bm0 = tile / cols * BT, bn0 = tile % cols * BT;
  const int KT = k / P_BK;
  const u32 base = __builtin_amdgcn_readfirstlane(p_lds_addr(sm) + (u32)(wave * S * STG));
  const i8* a_win = src + (long)bm0 * k;
  const i8* b_win = St + (long)bn0 * k;
  u32 offs[BT / 8];  // the same rows and chunks of both operands
#pragma unroll
  for (int t = 0; t < BT / 8; t++) {
    const int row = 8 * t + (lane >> 3);
    offs[t] = (u32)((long)row * k + (((lane & 7) ^ p_swz(row)) << 4));
  }
  auto issue = [&](int st, long k0) P_AI {
    p_static_for<SEG>([&](auto dc) P_AI {
      constexpr int d = decltype(dc)::value;
      if constexpr (d < BT / 8) p_dma(offs[d], a_win + k0, base + (u32)(st * STG + d * 1024));
      else p_dma(offs[d - BT / 8], b_win + k0, base + (u32)(st * STG + d * 1024));
    });
  };
  u32 fa[NP][2];
#pragma unroll
  for (int kp = 0; kp < NP; kp++)
#pragma unroll
    for (int o = 0; o < 2; o++) {
      const int rr = lane % 32, c = (8 / NP) * kp + lane / 32;
      fa[kp][o] = base + (u32)(rr * P_BK + ((c ^ p_swz(rr + o * 32)) << 4));
    }
  MM::acc_t acc[NB][NB];
#pragma unroll
  for (int i = 0; i < NB; i++)
#pragma unroll
    for (int q = 0; q < NB; q++) acc[i][q] = MM::acc_t{};
  const int steps = wave < KT ? (KT - 1 - wave) / ST_WAVES + 1 : 0;
#pragma unroll
  for (int s = 0; s < S; s++)
    if (s < steps) issue(s, (long)(wave + s * ST_WAVES) * P_BK);
  for (int j0 = 0; j0 < steps; j0 += S) {
    p_static_for<S>([&](auto sc) P_AI {
      constexpr int st = decltype(sc)::value;
      const int j = j0 + st;
      if (j >= steps) return;
      p_wait_vm<SEG, S - 1>(min(steps - 1 - j, S - 1));
      v4i a[NP][NB], b[NP][NB];
#pragma unroll
      for (int kp = 0; kp < NP; kp++)
#pragma unroll
        for (int q = 0; q < NB; q++) {
          b[kp][q] = p_lds(fa[kp][q & 1] + (u32)(st * STG + (BT + q * 32) * P_BK));
          a[kp][q] = p_lds(fa[kp][q & 1] + (u32)(st * STG + q * 32 * P_BK));
        }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      if (j + S < steps) issue(st, (long)(wave + (j + S) * ST_WAVES) * P_BK);
#pragma unroll
      for (int kp = 0; kp < NP; kp++)
#pragma unroll
        for (int i = 0; i < NB; i++)
#pragma unroll
          for (int q = 0; q < NB; q++) acc[i][q] = MM::mul(b[kp][q], a[kp][i], acc[i][q]);
    });
  }
  // partial sums: piece c4 of row rr at slot rr PC + (c4 ^ (rr % PC)) of the wave's ring
  u8* mine = sm + wave * S * STG;
#pragma unroll
  for (int i = 0; i < NB; i++)
#pragma unroll
    for (int q = 0; q < NB; q++)
#pragma unroll
      for (int g = 0; g < MM::G; g++) {
        const int rr = 32 * i + lane % 32, c4 = 8 * q + 2 * g + lane / 32;
        const auto& v = acc[i][q];
        *reinterpret_cast<v4i*>(mine + (rr * PC + (c4 ^ (rr & (PC - 1)))) * 16) =
            v4i{v[4 * g], v[4 * g + 1], v[4 * g + 2], v[4 * g + 3]};
      }
  __syncthreads();
  const long limb_stride = (long)rows * 2 * r;
  int big = 0;
#pragma unroll
  for (int t = 0; t < BT * PC / ST_THREADS; t++) {
    const int e = t * ST_THREADS + tid, rr = e / PC, c4 = e % PC;
    const u8* at = sm + (rr * PC + (c4 ^ (rr & (PC - 1)))) * 16;
    v4i x = *reinterpret_cast<const v4i*>(at);
#pragma unroll
    for (int w = 1; w < ST_WAVES; w++) x += *reinterpret_cast<const v4i*>(at + w * S * STG);
    int v[4] = {x[0], x[1], x[2], x[3]};
#pragma unroll
    for (int i = 0; i < 4; i++) big = max(big, abs(v[i]));
    i8* out = corr + (long)(bm0 + rr) * 2 * r + off + bn0 + 4 * c4;
    for (int li = 0; li < lmax; li++) {  // balanced digits: d = ((v + 64) mod 128) - 64, v <- (v - d) / 128
      u32 packed = 0;
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int d = ((v[i] + 64) & 127) - 64;
        packed |= (u32)(u8)d << (8 * i);
        v[i] = (v[i] - d) >> 7;
      }
      *reinterpret_cast<u32*>(out + li * limb_stride) = packed;
    }
  }
  if (mx) {  // one global atomic per workgroup
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) big = max(big, __shfl_xor(big, s));
    if (lane == 0) wmax[wave] = big;
    __syncthreads();
    if (tid == 0) atomicMax(mx, max(max(wmax[0], wmax[1]), max(wmax[2], wmax[3])));
  }
}

// Rows row0 .. + 15, columns col0 .. + 511 (or to k) of A' = int8(A + E[first] - E[second]).
__device__ __forceinline__ void side_noise(u8* sm, const SideTilesParams& p, int row0, int col0) {
  u32* pairs = reinterpret_cast<u32*>(sm);
  i8* es = reinterpret_cast<i8*>(sm + ST_NCOLS * 4);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r = p.r, pitch = r + 4;
  const int ncols = min(ST_NCOLS, p.k - col0), nsteps = ncols / 64;
  const int rr = lane & 15, kq = (lane >> 4) * 16;
  const i8* src = p.A + (long)(row0 + rr) * p.k + col0 + kq;
  v4i a[ST_NCOLS / 64 / ST_WAVES];
#pragma unroll
  for (int t = 0; t < ST_NCOLS / 64 / ST_WAVES; t++)
    if (wave + t * ST_WAVES < nsteps) a[t] = *reinterpret_cast<const v4i*>(src + (wave + t * ST_WAVES) * 64);
  for (int i = tid; i < ncols; i += ST_THREADS) pairs[i] = p.PA[col0 + i];
  // E rows at a pitch of r + 4 bytes: the 16 rows a wave looks up at once fall in distinct banks
  for (int i = 4 * tid; i < ST_NROWS * r; i += 4 * ST_THREADS)
    *reinterpret_cast<u32*>(es + i / r * pitch + i % r) = *reinterpret_cast<const u32*>(p.EA + (long)row0 * r + i);
  __syncthreads();
  const i8* er = es + rr * pitch;
#pragma unroll
  for (int t = 0; t < ST_NCOLS / 64 / ST_WAVES; t++) {
    const int j = wave + t * ST_WAVES;
    if (j >= nsteps) break;
    v4i o;
#pragma unroll
    for (int d = 0; d < 4; d++) {
      const v4i p4 = *reinterpret_cast<const v4i*>(pairs + j * 64 + kq + 4 * d);
      const u32 x = (u32)a[t][d];
      u32 w = 0;
#pragma unroll
      for (int b = 0; b < 4; b++) {
        const u32 pr = (u32)p4[b];
        const int v = (int)(i8)(u8)(x >> (8 * b)) + (int)er[pr & 0xFFFF] - (int)er[pr >> 16];
        w |= ((u32)(u8)v) << (8 * b);
      }
      o[d] = (int)w;
    }
    *reinterpret_cast<v4i*>(p.ApEA + (long)(row0 + rr) * p.k + col0 + kq + j * 64) = o;
  }
  if (p.ecopy_off >= 0 && col0 == 0) {
    const long limb_stride = (long)p.m * 2 * r;
    for (int i = 4 * tid; i < ST_NROWS * r; i += 4 * ST_THREADS) {
      const u32 e = *reinterpret_cast<const u32*>(es + i / r * pitch + i % r);
      i8* out = p.corrA + (long)(row0 + i / r) * 2 * r + p.ecopy_off + i % r;
      for (int li = 0; li < p.lmax; li++) *reinterpret_cast<u32*>(out + li * limb_stride) = e;
    }
  }
}

template <int BT, int S>
__global__ void __launch_bounds__(ST_THREADS) side_tiles_kernel(SideTilesParams p) {
  extern __shared__ __attribute__((aligned(1024))) u8 sm[];
  __shared__ int wmax[ST_WAVES];
  const int cols = p.r / BT, tx = p.m / BT * cols, ty = p.n / BT * cols;
  int b = blockIdx.x;
  if (b < ty) {
    side_tile<BT, S>(sm, wmax, p.Bp, p.n, p.k, p.StA, p.r, b, p.corrB, p.corr_b_off, p.lmax, p.maxabs ? p.maxabs + 1 : nullptr);
  } else if ((b -= ty) < tx) {
    side_tile<BT, S>(sm, wmax, p.A, p.m, p.k, p.StB, p.r, b, p.corrA, p.corr_a_off, p.lmax, p.maxabs);
  } else {
    b -= tx;
    const int chunks = (p.k + ST_NCOLS - 1) / ST_NCOLS;
    side_noise(sm, p, b / chunks * ST_NROWS, b % chunks * ST_NCOLS);
  }
}

template <int BT, int S>
void side_tiles_go(hipStream_t stream, const SideTilesParams& p) {
  auto kern = side_tiles_kernel<BT, S>;
  constexpr int lds = ST_WAVES * S * 2 * BT * P_BK;
  static_assert(lds >= ST_NCOLS * 4 + ST_NROWS * (ST_MAXR + 4), "a noise block fits beside the pairs");
  static bool attr = false;  // one attribute call per instantiation (the library is process-wide)
  if (!attr) {
    (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    attr = true;
  }
  const int tiles = (p.m / BT + p.n / BT) * (p.r / BT), noise = p.m / ST_NROWS * ((p.k + ST_NCOLS - 1) / ST_NCOLS);
  hipLaunchKernelGGL(kern, dim3(tiles + noise), dim3(ST_THREADS), lds, stream, p);
}

}  // namespace

extern "C" int uwc_side_project_pairs(const int8_t* A, int m, const int8_t* EA, const uint32_t* PA, int8_t* ApEA,
                                      const int8_t* StB, int8_t* corrA, int corr_a_off, int ecopy_off, const int8_t* Bp,
                                      int n, const int8_t* StA, int8_t* corrB, int corr_b_off, int k, int r,
                                      int32_t* maxabs, int lmax, hipStream_t stream) {
  const char* fn = "uwc_side_project_pairs";
  if (!A || !EA || !PA || !ApEA || !StB || !corrA || !Bp || !StA || !corrB) return uwc_fail("%s: null pointer argument", fn);
  if (m <= 0 || n <= 0 || k <= 0 || m % 32 || n % 32 || k % P_BK || k > (1 << 23))
    return uwc_fail("%s: m=%d and n=%d must be positive multiples of 32 and k=%d of %d (at most 2^23)", fn, m, n, k, P_BK);
  if (r != 32 && r != 64 && r != 128) return uwc_fail("%s: r=%d must be 32, 64 or 128", fn, r);
  if (lmax < 1 || lmax > 4) return uwc_fail("%s: lmax=%d must be 1..4", fn, lmax);
  if ((corr_a_off != 0 && corr_a_off != r) || (corr_b_off != 0 && corr_b_off != r) || (ecopy_off != -1 && ecopy_off != 0 && ecopy_off != r))
    return uwc_fail("%s: corr offsets must be 0 or r (ecopy_off may be -1)", fn);
  if (((uintptr_t)A | (uintptr_t)ApEA | (uintptr_t)Bp | (uintptr_t)StA | (uintptr_t)StB | (uintptr_t)EA | (uintptr_t)PA |
       (uintptr_t)corrA | (uintptr_t)corrB) & 15)
    return uwc_fail("%s: A, EA, PA, ApEA, StA, StB, Bp, corrA and corrB must be 16-byte aligned", fn);
  const SideTilesParams p{A, EA, PA, ApEA, StB, corrA, Bp, StA, corrB, maxabs, m, n, k, r, lmax, corr_a_off, ecopy_off, corr_b_off};
  if (m % 64 == 0 && n % 64 == 0 && r % 64 == 0 && (long)(m / 64 + n / 64) * (r / 64) * 2 >= uwc_cu_count())
    side_tiles_go<64, 1>(stream, p);
  else
    side_tiles_go<32, 2>(stream, p);
  return uwc_launch_status(fn);
}
