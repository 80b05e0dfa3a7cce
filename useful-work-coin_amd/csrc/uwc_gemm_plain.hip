// gfx950 plain int8 x int8 -> int32 GEMM (no transcript, no denoise): the detrt linears and every
// other plain product that does not fill the chip with 256 x 256 tiles, from one decoded token to a
// prefill chunk. Same contract and epilogues as the plain path of uwc_noisy_gemm
// (runtime/detrt/qwen3.py:106-126: int32 out, or fp32 / bf16 of f32(acc) * sx[i] * sw[j], or fp32
// with a residual added). Two kernels, any m, n % 4 == 0, k % 128 == 0:
//
// plain_gemm_kernel, for many tiles:
//   * Workgroup tile BM x BN (64 or 128 rows, 128 or 256 columns), k step 128, 4 wave64s in 2 x 2,
//     each a (BM / 2) x (BN / 2) block of v_mfma_i32_32x32x32_i8.
//   * Operands go HBM -> LDS with global_load_lds_dwordx4 into a ring of S k steps; every wave
//     issues its share of each step (1 KiB segments, the window base in SGPRs, a fixed 32-bit
//     lane offset), S - 1 steps ahead of the one being multiplied. One barrier per k step.
//   * Two fragment sets: the reads of pass p + 1 go out before the MFMAs of pass p.
//   * The epilogue turns pairs of blocks around through LDS so that each store instruction writes
//     whole row segments.
// wave_gemm_kernel, for few: small tiles whose k steps the waves of a workgroup share out (below).
//
// Both:
//   * LDS rows are 128 bytes; 16-byte chunk c of tile row r sits at chunk c ^ ((r ^ (r >> 3)) & 7),
//     so the fragment reads are conflict-free; the swizzle is applied on the global side.
//   * Rows past m or n read the last row again and are never stored.
//   * Transposed C (the B fragment is the MFMA's first operand): a lane holds one row of a block and
//     4 consecutive columns per register group.
//   * int32 sums are exact, so any tiling and k order gives the same accumulators as the other
//     GEMM kernels of this library.
//
// Every shape here used to run on the register-staged 128 x 128 kernel unless its tiles were whole
// (m, n % 128 == 0), and on the kernels of uwc_skinny.hip for m <= 64. Measured (graph-replayed,
// fp32 dequant out, us): 777 x 12288 x 2048 69.0 -> 33.6, 777 x 2048 x 6144 63.3 -> 18.2,
// 200 x 4096 x 2048 28.3 -> 7.0, 100 x 2048 x 6144 60.9 -> 7.3, 33 x 4096 x 14336 26.5 -> 15.0,
// 64 x 6144 x 4096 23.9 -> 7.9, 16 x 2688 x 2560 6.4 -> 4.1, 1 x 2048 x 6144 6.3 -> 4.6.
#include "uwc_dma.h"

#define P_THREADS 256
#define P_OUT_NONE 0
#define P_OUT_I32 1
#define P_OUT_BF16 2
#define P_OUT_F32 3
#define P_OUT_F32R 4  // OUT_F32 with a residual: fadd(res, fmul(fmul(f32(acc), sx), sw))
#define P_OUT_BOTH 5  // OUT_I32 to out and OUT_F32 to out2

namespace {

struct PlainParams {
  const i8* A;
  const i8* B;
  int m, n, k;
  const float* a_scale;
  const float* b_scale;
  void* out;
  int ldc;  // output row stride in elements
  const float* res;  // P_OUT_F32R: the residual rows, of the output's stride
  float* out2;       // P_OUT_BOTH: the fp32 rows, of the output's stride
};

__device__ __forceinline__ u32 p_bf16_rne(float f) {
  const u32 u = __float_as_uint(f);
  return (u + 0x7FFFu + ((u >> 16) & 1u)) >> 16;
}

template <int BM, int BN, int S, bool SPREAD, bool RAGGED, int OUT>
__global__ void __launch_bounds__(P_THREADS) plain_gemm_kernel(PlainParams p) {
  constexpr int WM = BM / 2, WN = BN / 2;  // wave block
  constexpr int MB = WM / 32, NB = WN / 32;  // 32 x 32 MFMA blocks per wave
  constexpr int TA = BM * P_BK, TB = BN * P_BK;  // bytes of one stage's A and B tile
  constexpr int SA = BM / 32, SB = BN / 32;  // 1 KiB DMA segments per wave per k step
  constexpr int SEG = SA + SB;
  static_assert(NB % 2 == 0 && (MB % 2 == 0 || MB == 1), "the epilogue takes column blocks in pairs");
  static_assert(S >= 2 && S <= 4, "ring depth");
  extern __shared__ __attribute__((aligned(1024))) u8 sm[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;

  // workgroup -> tile: XCD-contiguous runs of ids (dispatch is round-robin over 8 XCDs), rastered
  // in groups of 4 tile rows so that one XCD's tiles share A and B panels in its L2
  int bm0, bn0;
  {
    const int npm = (p.m + BM - 1) / BM, npn = (p.n + BN - 1) / BN, total = npm * npn;
    const int xcd = blockIdx.x & 7;
    const int pid = xcd * (total >> 3) + min(xcd, total & 7) + (int)(blockIdx.x >> 3);
    constexpr int GROUP_M = 4;
    const int grp = GROUP_M * npn, gid = pid / grp, first = gid * GROUP_M;
    const int gsz = min(npm - first, GROUP_M), in = pid - gid * grp;
    bm0 = (first + in % gsz) * BM;
    bn0 = (in / gsz) * BN;
  }
  const long k = p.k;
  const int KT = p.k / P_BK;
  const u32 base = __builtin_amdgcn_readfirstlane(p_lds_addr(sm));
  auto lds_a = [&](int st) P_AI { return base + (u32)(st * TA); };
  auto lds_b = [&](int st) P_AI { return base + (u32)(S * TA + st * TB); };

  // DMA: this wave fills segments wave SA + t of A and wave SB + t of B; lane i of a segment
  // writes LDS bytes [16 i, 16 i + 16): tile row 8 s + i / 8, physical chunk i % 8, so it
  // fetches logical chunk (i % 8) ^ swz(row). Rows past the operand's last one read that one again
  // (their products are never stored)
  u32 offa[SA], offb[SB];
#pragma unroll
  for (int t = 0; t < SA; t++) {
    const int row = 8 * (wave * SA + t) + (lane >> 3);
    offa[t] = (u32)((long)(RAGGED ? min(row, p.m - 1 - bm0) : row) * k + (((lane & 7) ^ p_swz(row)) << 4));
  }
#pragma unroll
  for (int t = 0; t < SB; t++) {
    const int row = 8 * (wave * SB + t) + (lane >> 3);
    offb[t] = (u32)((long)(RAGGED ? min(row, p.n - 1 - bn0) : row) * k + (((lane & 7) ^ p_swz(row)) << 4));
  }
  const i8* a_win = p.A + (long)bm0 * k;
  const i8* b_win = p.B + (long)bn0 * k;
  // DMA instructions [D0, D1) of a k step (A segments first, then B)
  auto issue_part = [&](auto d0c, auto d1c, int st, long k0) P_AI {
    constexpr int D0 = decltype(d0c)::value, D1 = decltype(d1c)::value;
    p_static_for<SEG>([&](auto dc) P_AI {
      constexpr int d = decltype(dc)::value;
      if constexpr (d >= D0 && d < D1) {
        if constexpr (d < SA) p_dma(offa[d], a_win + k0, lds_a(st) + (u32)((wave * SA + d) * 1024));
        else p_dma(offb[d - SA], b_win + k0, lds_b(st) + (u32)((wave * SB + d - SA) * 1024));
      }
    });
  };
  auto issue = [&](int st, long k0) P_AI {
    issue_part(std::integral_constant<int, 0>{}, std::integral_constant<int, SEG>{}, st, k0);
  };

  // fragment addresses: row (lane & 31) of the wave's first 32-row block, logical chunk 2 kp +
  // (lane >> 5); the wave's odd blocks (row bit 5 flipped) flip swizzle bit 2, i.e. use pass
  // kp ^ 2's offset
  u32 fa[4], fb[4];
#pragma unroll
  for (int kp = 0; kp < 4; kp++) {
    const int ra = wm * WM + (lane & 31), rb = wn * WN + (lane & 31), c = 2 * kp + (lane >> 5);
    fa[kp] = lds_a(0) + (u32)(ra * P_BK + ((c ^ p_swz(ra)) << 4));
    fb[kp] = lds_b(0) + (u32)(rb * P_BK + ((c ^ p_swz(rb)) << 4));
  }
  struct Frag {
    v4i a[MB], b[NB];
  };
  auto read = [&](Frag& f, int st, int kp) P_AI {
#pragma unroll
    for (int j = 0; j < NB; j++) f.b[j] = p_lds(fb[(j & 1) ? kp ^ 2 : kp] + (u32)(st * TB + j * 32 * P_BK));
#pragma unroll
    for (int i = 0; i < MB; i++) f.a[i] = p_lds(fa[(i & 1) ? kp ^ 2 : kp] + (u32)(st * TA + i * 32 * P_BK));
  };

  v16i acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; i++)
#pragma unroll
    for (int j = 0; j < NB; j++) acc[i][j] = v16i{};

  // prologue: every stage of the ring loading, then step 0 resident and its first pass read
#pragma unroll
  for (int s = 0; s < S; s++)
    if (s < KT) issue(s, (long)s * P_BK);
  p_wait_vm<SEG, S - 1>(min(KT - 1, S - 1));
  __builtin_amdgcn_s_barrier();
  Frag f[2];
  read(f[0], 0, 0);

  // k step kt in stage ST = kt % S (a compile-time constant: every LDS address is a base
  // register plus an immediate). Before the last pass the wave waits for step kt + 1 (vmcnt,
  // then the barrier: every wave has also finished reading stage ST) and refills ST with step
  // kt + S; the last pass reads the next step's first fragments (on the final step a read of a
  // resident stage that nothing uses, which keeps the MFMA code free of branches).
  auto step = [&](auto stc, int kt) P_AI {
    constexpr int ST = decltype(stc)::value;
    p_static_for<4>([&](auto kpc) P_AI {
      constexpr int kp = decltype(kpc)::value;
      constexpr int nst = kp == 3 ? (ST + 1) % S : ST, nkp = (kp + 1) & 3;
      // SPREAD: the refill of the previous step's stage, continued: quarter kp + 1 of its DMA
      // before pass kp (kp < 3) of this step (the first quarter went out after that step's
      // barrier), so that no wave's MFMAs queue behind a whole step's DMA burst
      if constexpr (SPREAD && kp < 3) {
        if (kt >= 1 && kt - 1 + S < KT) {
          constexpr int PST = (ST + S - 1) % S;
          issue_part(std::integral_constant<int, SEG * (kp + 1) / 4>{}, std::integral_constant<int, SEG * (kp + 2) / 4>{},
                     PST, (long)(kt - 1 + S) * P_BK);
        }
      }
      if constexpr (kp == 3) {
        if (kt + 1 < KT) {
          asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
          p_wait_vm<SEG, S - 2>(min(KT - 2 - kt, S - 2));
          __builtin_amdgcn_s_barrier();
          if (kt + S < KT) {
            if constexpr (SPREAD)
              issue_part(std::integral_constant<int, 0>{}, std::integral_constant<int, SEG / 4>{}, ST,
                         (long)(kt + S) * P_BK);
            else
              issue(ST, (long)(kt + S) * P_BK);
          }
        }
      }
      Frag& cur = f[kp & 1];
      read(f[(kp + 1) & 1], nst, nkp);
#pragma unroll
      for (int i = 0; i < MB; i++)
#pragma unroll
        for (int j = 0; j < NB; j++)
          acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(cur.b[j], cur.a[i], acc[i][j], 0, 0, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, MB + NB, 0);
#pragma unroll
      for (int q = 0; q < MB * NB; q++) __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    });
  };
  for (int kt0 = 0; kt0 < KT; kt0 += S) {
    p_static_for<S>([&](auto sc) P_AI {
      const int kt = kt0 + decltype(sc)::value;
      if (kt < KT) step(sc, kt);
    });
  }

  // epilogue: the wave's blocks, two at a time, through its own 8 KiB of the idle ring, stored by
  // rows. In the MFMA layout lane hh 32 + rr holds row rr of a block and, in register group j,
  // columns 8 j + 4 hh .. + 3; that piece goes to slot piece (4 b + j) 64 + hh 32 + (rr ^ 2 (2 j +
  // hh)) for block b of the pair. Store instruction jj then has lane l take row 8 jj + l / 8,
  // columns 4 (l % 8) .. + 3 of a block: 8 whole row segments per instruction instead of 32 rows
  // of 16 bytes (the output burst at the end of a launch drains faster). The XOR keeps the 16
  // lanes of each write (16 rows) and of each read (2 rows x 8 pieces) on distinct 16-byte bank
  // groups. The stores carry the non-temporal hint, so that the output stream does not evict the
  // operand panels other workgroups of the XCD still read from L2 (the M = 2048 Qwen3-1.7B
  // linears 4-8% faster).
  if constexpr (OUT != P_OUT_NONE) {
    constexpr int ES = OUT == P_OUT_BF16 ? 2 : 4;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();  // every wave is done reading the ring
    u8* slot = sm + wave * 8192;
    const int hh = lane >> 5, rr = lane & 31;
    const int rj = (lane & 7) >> 1, rh = lane & 1;  // the piece a row read takes
    // A tile that reaches past the last row or column (n % 4 == 0: four columns in or out together)
    // takes the last operands again there, without a branch, and leaves out the store; whole tiles
    // have a copy of the code without the tests, which cost 5% at 2048 x 12288 x 2048 (and products
    // of whole tiles only a kernel without the edge copy, whose code costs 1%).
    auto emit = [&](auto edge_c) P_AI {
      constexpr bool EDGE = decltype(edge_c)::value;
#pragma unroll
      for (int i = 0; i < MB; i++) {
#pragma unroll
        for (int j0 = 0; j0 < NB; j0 += 2) {
#pragma unroll
          for (int b = 0; b < 2; b++)
#pragma unroll
            for (int g = 0; g < 4; g++) {
              const v16i& v = acc[i][j0 + b];
              *reinterpret_cast<v4i*>(slot + ((4 * b + g) * 64 + hh * 32 + (rr ^ (2 * (2 * g + hh)))) * 16) =
                  v4i{v[4 * g], v[4 * g + 1], v[4 * g + 2], v[4 * g + 3]};
            }
#pragma unroll
          for (int b = 0; b < 2; b++) {
            const int row0 = bm0 + wm * WM + i * 32, col = bn0 + wn * WN + (j0 + b) * 32 + 4 * (lane & 7);
            u8* base = reinterpret_cast<u8*>(p.out) + ((long)row0 * p.ldc + col) * ES;
            const int colc = EDGE ? min(col, p.n - 4) : col;
            float4 sw{};
            if constexpr (OUT != P_OUT_I32) sw = *reinterpret_cast<const float4*>(p.b_scale + colc);
            // the four LDS reads (and row scales) first, then the stores: read, wait, store in turn
            // put an LDS round trip (and a scale load) in front of every store
            v4i xs[4];
            float ascs[4];
            float4 rs[4];
#pragma unroll
            for (int jj = 0; jj < 4; jj++) {
              const int r = 8 * jj + (lane >> 3);
              xs[jj] = *reinterpret_cast<const v4i*>(slot + ((4 * b + rj) * 64 + rh * 32 + (r ^ (2 * (2 * rj + rh)))) * 16);
              const int rowc = EDGE ? min(row0 + r, p.m - 1) : row0 + r;
              if constexpr (OUT != P_OUT_I32) ascs[jj] = p.a_scale[rowc];
              if constexpr (OUT == P_OUT_F32R) rs[jj] = uwc_load_nt(p.res + (long)rowc * p.ldc + colc);
            }
#pragma unroll
            for (int jj = 0; jj < 4; jj++) {
              const int r = 8 * jj + (lane >> 3);
              if (EDGE && (row0 + r >= p.m || col >= p.n)) continue;
              const v4i x = xs[jj];
              u8* dst = base + (long)r * p.ldc * ES;
              if constexpr (OUT == P_OUT_I32) {
                uwc_store_nt(dst, x);
              } else {
                const float asc = ascs[jj];
                const float y0 = __fmul_rn(__fmul_rn((float)x[0], asc), sw.x);
                const float y1 = __fmul_rn(__fmul_rn((float)x[1], asc), sw.y);
                const float y2 = __fmul_rn(__fmul_rn((float)x[2], asc), sw.z);
                const float y3 = __fmul_rn(__fmul_rn((float)x[3], asc), sw.w);
                if constexpr (OUT == P_OUT_F32) {
                  uwc_store_nt(dst, float4{y0, y1, y2, y3});
                } else if constexpr (OUT == P_OUT_BOTH) {
                  uwc_store_nt(dst, x);
                  uwc_store_nt(p.out2 + (long)(row0 + r) * p.ldc + col, float4{y0, y1, y2, y3});
                } else if constexpr (OUT == P_OUT_F32R) {
                  const float4 x0 = rs[jj];
                  uwc_store_nt(dst, float4{__fadd_rn(x0.x, y0), __fadd_rn(x0.y, y1), __fadd_rn(x0.z, y2), __fadd_rn(x0.w, y3)});
                } else {
                  uwc_store_nt(dst, uint2{p_bf16_rne(y0) | (p_bf16_rne(y1) << 16), p_bf16_rne(y2) | (p_bf16_rne(y3) << 16)});
                }
              }
            }
          }
        }
      }
    };
    if (!RAGGED || (bm0 + BM <= p.m && bn0 + BN <= p.n)) emit(std::false_type{});
    else emit(std::true_type{});
  }
}

// The form for few tiles (decode, short prompts, narrow outputs): a workgroup of W waves owns one
// BM x BN tile, and wave w multiplies the whole tile over the k steps w, w + W, w + 2 W, ... through
// an LDS ring of its own (S stages), so that the waves never wait for each other until their partial
// sums meet in LDS at the end (int32 sums are exact: the split cannot change a value). A wave reads
// all of a step's fragments into registers, refills the stage, then multiplies.
//   * What bounds these shapes is how many bytes are in flight from the first cycle on and, per CU,
//     the DMA instructions of its tiles (about 26 cycles each): small tiles put every CU to work
//     (a 2048-column product has 64 tiles of 32 columns, 128 of 16), the k split lets a workgroup
//     ask for W S steps at once, and with no barrier in the loop a late line holds up one wave.
//     A tile whose four waves split its rows and columns instead needs every wave's operands for
//     each step: 100 x 2048 x 6144 takes 17.4 us on 64 x 128 tiles that way, 7.3 on 32 x 32.
//   * ONCE (one row of tiles: every byte of B is read once): B carries the non-temporal hint, so
//     that a weight streaming from HBM does not evict A and the scales. Weights rotated over 1.3 GB:
//     1 x 12288 x 2048 7.0 -> 6.0 us, 1 x 4096 x 14336 12.6 -> 10.7.
template <int BM, int BN, int TB, int W, int S, bool ONCE, int OUT>
__global__ void __launch_bounds__(W * 64) wave_gemm_kernel(PlainParams p) {
  typedef Mfma<TB> MM;
  constexpr int MB = BM / TB, NB = BN / TB, NT = W * 64, NP = MM::PASSES;
  constexpr int SA = BM / 8, SB = BN / 8, SEG = SA + SB;  // 1 KiB DMA segments per k step
  static_assert(TB == 32 || (MB == 1 && NB <= 2), "block parity decides the swizzle");
  constexpr int STG = (BM + BN) * P_BK;                   // bytes of one stage
  constexpr int PC = BN / 4;                              // 16-byte pieces of a row of partial sums
  static_assert(BM * BN * 4 <= S * STG, "a wave's partial sums reuse its ring");
  extern __shared__ __attribute__((aligned(1024))) u8 sm[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // workgroup -> tile: contiguous runs of ids per XCD, the tile rows of a column panel of B adjacent
  int bm0, bn0;
  {
    const int npm = (p.m + BM - 1) / BM, npn = (p.n + BN - 1) / BN, total = npm * npn;
    const int xcd = blockIdx.x & 7;
    const int pid = xcd * (total >> 3) + min(xcd, total & 7) + (int)(blockIdx.x >> 3);
    constexpr int GROUP_M = 8;
    const int grp = GROUP_M * npn, gid = pid / grp, first = gid * GROUP_M;
    const int gsz = min(npm - first, GROUP_M), in = pid - gid * grp;
    bm0 = (first + in % gsz) * BM;
    bn0 = (in / gsz) * BN;
  }
  const int KT = p.k / P_BK;
  const u32 base = __builtin_amdgcn_readfirstlane(p_lds_addr(sm) + (u32)(wave * S * STG));
  const i8* a_win = p.A + (long)bm0 * p.k;
  const i8* b_win = p.B + (long)bn0 * p.k;
  u32 offa[SA], offb[SB];
#pragma unroll
  for (int t = 0; t < SA; t++) {
    const int row = 8 * t + (lane >> 3);
    offa[t] = (u32)((long)min(row, p.m - 1 - bm0) * p.k + (((lane & 7) ^ p_swz(row)) << 4));
  }
#pragma unroll
  for (int t = 0; t < SB; t++) {
    const int row = 8 * t + (lane >> 3);
    offb[t] = (u32)((long)min(row, p.n - 1 - bn0) * p.k + (((lane & 7) ^ p_swz(row)) << 4));
  }
  auto issue = [&](int st, long k0) P_AI {
    p_static_for<SEG>([&](auto dc) P_AI {
      constexpr int d = decltype(dc)::value;
      if constexpr (d < SA) p_dma(offa[d], a_win + k0, base + (u32)(st * STG + d * 1024));
      else if constexpr (ONCE) p_dma_nt(offb[d - SA], b_win + k0, base + (u32)(st * STG + d * 1024));
      else p_dma(offb[d - SA], b_win + k0, base + (u32)(st * STG + d * 1024));
    });
  };
  // fragment addresses of the even and the odd blocks (the swizzle differs in the block's parity)
  // of A in pass kp; B's rows follow A's, swizzled alike
  u32 fa[NP][2];
#pragma unroll
  for (int kp = 0; kp < NP; kp++)
#pragma unroll
    for (int o = 0; o < 2; o++) {
      const int r = lane % TB, c = (8 / NP) * kp + lane / TB;
      fa[kp][o] = base + (u32)(r * P_BK + ((c ^ p_swz(r + o * TB)) << 4));
    }
  typename MM::acc_t acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; i++)
#pragma unroll
    for (int j = 0; j < NB; j++) acc[i][j] = typename MM::acc_t{};

  const int steps = wave < KT ? (KT - 1 - wave) / W + 1 : 0;  // this wave's k steps
#pragma unroll
  for (int s = 0; s < S; s++)
    if (s < steps) issue(s, (long)(wave + s * W) * P_BK);
  for (int j0 = 0; j0 < steps; j0 += S) {
    p_static_for<S>([&](auto sc) P_AI {
      constexpr int st = decltype(sc)::value;
      const int j = j0 + st;
      if (j >= steps) return;
      p_wait_vm<SEG, S - 1>(min(steps - 1 - j, S - 1));
      v4i a[NP][MB], b[NP][NB];
#pragma unroll
      for (int kp = 0; kp < NP; kp++) {
#pragma unroll
        for (int q = 0; q < NB; q++) b[kp][q] = p_lds(fa[kp][q & 1] + (u32)(st * STG + (BM + q * TB) * P_BK));
#pragma unroll
        for (int i = 0; i < MB; i++) a[kp][i] = p_lds(fa[kp][i & 1] + (u32)(st * STG + i * TB * P_BK));
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      if (j + S < steps) issue(st, (long)(wave + (j + S) * W) * P_BK);
#pragma unroll
      for (int kp = 0; kp < NP; kp++)
#pragma unroll
        for (int i = 0; i < MB; i++)
#pragma unroll
          for (int q = 0; q < NB; q++) acc[i][q] = MM::mul(b[kp][q], a[kp][i], acc[i][q]);
    });
  }

  // the partial sums: piece c4 (columns 4 c4 .. + 3) of row r at slot r PC + (c4 ^ (r % PC)) of the
  // wave's ring (its DMA has landed and been read), so that the rows of a write and the pieces of a
  // read fall in distinct 16-byte bank groups; then every thread adds the W copies of its pieces
  if constexpr (OUT != P_OUT_NONE) {
    constexpr int ES = OUT == P_OUT_BF16 ? 2 : 4;
    u8* mine = sm + wave * S * STG;
#pragma unroll
    for (int i = 0; i < MB; i++)
#pragma unroll
      for (int q = 0; q < NB; q++)
#pragma unroll
        for (int g = 0; g < MM::G; g++) {
          const int r = TB * i + lane % TB, c4 = TB / 4 * q + 2 * g + lane / TB;
          const auto& v = acc[i][q];
          *reinterpret_cast<v4i*>(mine + (r * PC + (c4 ^ (r & (PC - 1)))) * 16) =
              v4i{v[4 * g], v[4 * g + 1], v[4 * g + 2], v[4 * g + 3]};
        }
    __syncthreads();
    // past the last row or column (n % 4 == 0) the scales are the last ones again, without a branch,
    // and only the store is left out
    constexpr int TN = (BM * PC + NT - 1) / NT;  // pieces per thread
    v4i xs[TN];
    float4 sws[TN], rs[TN];
    float ascs[TN];
#pragma unroll
    for (int t = 0; t < TN; t++) {
      const int e = t * NT + tid, r = e / PC, c4 = e % PC;
      if (TN * NT > BM * PC && e >= BM * PC) break;
      const int row = min(bm0 + r, p.m - 1), col = min(bn0 + 4 * c4, p.n - 4);
      if constexpr (OUT != P_OUT_I32) {
        sws[t] = *reinterpret_cast<const float4*>(p.b_scale + col);
        ascs[t] = p.a_scale[row];
      }
      if constexpr (OUT == P_OUT_F32R) rs[t] = uwc_load_nt(p.res + (long)row * p.ldc + col);
      const u8* src = sm + (r * PC + (c4 ^ (r & (PC - 1)))) * 16;
      xs[t] = *reinterpret_cast<const v4i*>(src);
#pragma unroll
      for (int w = 1; w < W; w++) xs[t] += *reinterpret_cast<const v4i*>(src + w * S * STG);
    }
#pragma unroll
    for (int t = 0; t < TN; t++) {
      const int e = t * NT + tid, r = e / PC, c4 = e % PC;
      const int row = bm0 + r, col = bn0 + 4 * c4;
      if ((TN * NT > BM * PC && e >= BM * PC) || row >= p.m || col >= p.n) continue;
      const v4i x = xs[t];
      u8* dst = reinterpret_cast<u8*>(p.out) + ((long)row * p.ldc + col) * ES;
      if constexpr (OUT == P_OUT_I32) {
        uwc_store_nt(dst, x);
      } else {
        const float4 sw = sws[t];
        const float asc = ascs[t];
        const float y0 = __fmul_rn(__fmul_rn((float)x[0], asc), sw.x);
        const float y1 = __fmul_rn(__fmul_rn((float)x[1], asc), sw.y);
        const float y2 = __fmul_rn(__fmul_rn((float)x[2], asc), sw.z);
        const float y3 = __fmul_rn(__fmul_rn((float)x[3], asc), sw.w);
        if constexpr (OUT == P_OUT_F32) {
          uwc_store_nt(dst, float4{y0, y1, y2, y3});
        } else if constexpr (OUT == P_OUT_BOTH) {
          uwc_store_nt(dst, x);
          uwc_store_nt(p.out2 + (long)row * p.ldc + col, float4{y0, y1, y2, y3});
        } else if constexpr (OUT == P_OUT_F32R) {
          const float4 x0 = rs[t];
          uwc_store_nt(dst, float4{__fadd_rn(x0.x, y0), __fadd_rn(x0.y, y1), __fadd_rn(x0.z, y2), __fadd_rn(x0.w, y3)});
        } else {
          uwc_store_nt(dst, uint2{p_bf16_rne(y0) | (p_bf16_rne(y1) << 16), p_bf16_rne(y2) | (p_bf16_rne(y3) << 16)});
        }
      }
    }
  }
}

template <int BM, int BN, int TB, int W, int S, bool ONCE, int OUT>
void wave_go(hipStream_t s, const PlainParams& p) {
  auto kern = wave_gemm_kernel<BM, BN, TB, W, S, ONCE, OUT>;
  constexpr int lds = W * S * (BM + BN) * P_BK;
  static_assert(lds <= 160 * 1024, "LDS exceeds 160 KiB");
  static bool attr = false;  // one attribute call per instantiation (the library is process-wide)
  if (!attr) {
    (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    attr = true;
  }
  hipLaunchKernelGGL(kern, dim3(((p.m + BM - 1) / BM) * ((p.n + BN - 1) / BN)), dim3(W * 64), lds, s, p);
}

template <int BM, int BN, int TB, int W, int S>
void wave_out(int out_mode, hipStream_t s, const PlainParams& p) {
  const bool once = p.m <= BM;
#define WAVE_GO(OUT) once ? wave_go<BM, BN, TB, W, S, true, OUT>(s, p) : wave_go<BM, BN, TB, W, S, false, OUT>(s, p)
  switch (out_mode) {
    case P_OUT_I32: WAVE_GO(P_OUT_I32); break;
    case P_OUT_BF16: WAVE_GO(P_OUT_BF16); break;
    case P_OUT_F32R: WAVE_GO(P_OUT_F32R); break;
    case P_OUT_BOTH: WAVE_GO(P_OUT_BOTH); break;
    default: WAVE_GO(P_OUT_F32); break;
  }
#undef WAVE_GO
}

template <int BM, int BN, int S, bool SPREAD, bool RAGGED, int OUT>
void plain_go(hipStream_t s, const PlainParams& p) {
  auto kern = plain_gemm_kernel<BM, BN, S, SPREAD, RAGGED, OUT>;
  constexpr int lds = S * (BM + BN) * P_BK;
  static_assert(lds <= 160 * 1024, "LDS exceeds 160 KiB");
  static bool attr = false;  // one attribute call per instantiation (the library is process-wide)
  if (!attr) {
    (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    attr = true;
  }
  hipLaunchKernelGGL(kern, dim3(((p.m + BM - 1) / BM) * ((p.n + BN - 1) / BN)), dim3(P_THREADS), lds, s, p);
}

template <int BM, int BN, int S, bool SPREAD>
void plain_out(int out_mode, hipStream_t s, const PlainParams& p) {
  switch (out_mode) {
    case P_OUT_NONE: plain_go<BM, BN, S, SPREAD, false, P_OUT_NONE>(s, p); break;
    case P_OUT_I32: plain_go<BM, BN, S, SPREAD, false, P_OUT_I32>(s, p); break;
    case P_OUT_BF16: plain_go<BM, BN, S, SPREAD, false, P_OUT_BF16>(s, p); break;
    default: plain_go<BM, BN, S, SPREAD, false, P_OUT_F32>(s, p); break;
  }
}

// any m, n % 4 == 0 (with an output)
template <int BM, int BN, int S>
void plain_any(int out_mode, hipStream_t s, const PlainParams& p) {
  if (p.m % BM == 0 && p.n % BN == 0) {
    if (out_mode == P_OUT_F32R) return plain_go<BM, BN, S, true, false, P_OUT_F32R>(s, p);
    if (out_mode == P_OUT_BOTH) return plain_go<BM, BN, S, true, false, P_OUT_BOTH>(s, p);
    return plain_out<BM, BN, S, true>(out_mode, s, p);
  }
  switch (out_mode) {
    case P_OUT_I32: plain_go<BM, BN, S, true, true, P_OUT_I32>(s, p); break;
    case P_OUT_BF16: plain_go<BM, BN, S, true, true, P_OUT_BF16>(s, p); break;
    case P_OUT_F32R: plain_go<BM, BN, S, true, true, P_OUT_F32R>(s, p); break;
    case P_OUT_BOTH: plain_go<BM, BN, S, true, true, P_OUT_BOTH>(s, p); break;
    default: plain_go<BM, BN, S, true, true, P_OUT_F32>(s, p); break;
  }
}

}  // namespace

// The configurations of the plain DMA kernel: BM x BN, ring depth; c | 4 spreads each step's DMA.
struct PlainCfg {
  int bm, bn, stages;
};
static const PlainCfg kPlainCfgs[] = {{128, 128, 4}, {128, 256, 3}, {128, 128, 2}, {128, 256, 2}};
#define PLAIN_NCFG 8

int uwc_plain_cfg_count() { return PLAIN_NCFG; }

// Whether configuration cfg takes the shape: whole tiles, whole k steps, 16-byte output rows.
bool uwc_plain_fits(int cfg, int m, int n, int k, int ldc, const void* out, int out_mode, const float* b_scale) {
  if (cfg < 0 || cfg >= PLAIN_NCFG) return false;
  const PlainCfg& c = kPlainCfgs[cfg & 3];
  const bool vec_out = out_mode == P_OUT_NONE || ((uintptr_t)out % 16 == 0 && ldc % 4 == 0);
  // the dequant epilogues read 4 column scales at once
  const bool vec_scale = out_mode != P_OUT_F32 && out_mode != P_OUT_BF16 || (uintptr_t)b_scale % 16 == 0;
  return vec_scale && m % c.bm == 0 && n % c.bn == 0 && k % P_BK == 0 && k >= P_BK && k <= (1 << 23) && vec_out;
}

// Called by uwc_noisy_gemm for a plain GEMM after its argument checks and uwc_plain_fits.
int uwc_gemm_plain(int cfg, const int8_t* A, const int8_t* B, int m, int n, int k, const float* a_scale,
                   const float* b_scale, void* out, int out_mode, int ldc, hipStream_t stream) {
  if (!uwc_plain_fits(cfg, m, n, k, ldc, out, out_mode, b_scale))
    return uwc_fail("uwc_gemm_plain: configuration %d does not take m=%d n=%d k=%d", cfg, m, n, k);
  const PlainParams p{A, B, m, n, k, a_scale, b_scale, out, ldc, nullptr, nullptr};
  switch (cfg) {
    case 0: plain_out<128, 128, 4, false>(out_mode, stream, p); break;
    case 1: plain_out<128, 256, 3, false>(out_mode, stream, p); break;
    case 2: plain_out<128, 128, 2, false>(out_mode, stream, p); break;
    case 3: plain_out<128, 256, 2, false>(out_mode, stream, p); break;
    case 4: plain_out<128, 128, 4, true>(out_mode, stream, p); break;
    case 5: plain_out<128, 256, 3, true>(out_mode, stream, p); break;
    case 6: plain_out<128, 128, 2, true>(out_mode, stream, p); break;
    default: plain_out<128, 256, 2, true>(out_mode, stream, p); break;
  }
  return uwc_launch_status("plain_gemm");
}

// The forms the automatic choice takes, with their tile, the workgroups a CU holds at once (by LDS)
// and the constants of their time in us:
//   start + max((k / 128) max(lat rounds, load x) + per_tile (x - 1), stream MB(B)) + store MB(out)
// for x tiles per CU in `rounds` rounds of `occ`. lat is what a k step of one tile takes (its wave's
// or its barrier's chain), load what it costs a CU that has other tiles to work on, per_tile what else a
// tile after the first costs, stream what reading the n x k weight from HBM takes with the bytes this form
// keeps in flight, store what writing the output (and reading a residual) adds. Fitted to 4660 products
// (m 1 .. 8192; the linears and heads of two models, 33 other n x k and 1278 random ones, n 4 .. 151936, k
// 128 .. 14336; fp32 out, with a residual, with both outputs; weights rotated over 1.3 GB, every form timed
// at each): the form with the least predicted time is on average within 0.8% of the fastest one, within
// 2.3% at nine products of ten, 13% at 99 of 100 and 67% at worst (666 x 10828 x 384 with both outputs);
// fitted to three quarters of the n x k, within 0.7 to 1.3% on average on the fourth. Without the stream
// and store terms it was 1.7%, 5.7%, 25% and 64%, and slower than the kernels before it at 17 x 28672 x
// 4096 (23.1 us; 29.1, now 22.7), 384 x 12288 x 2048 (21.9; 26.9, now 21.9) and 4096 x 1152 x 1152 (11.0;
// 14.3, now 11.1); 300 x 151936 x 2048 with both outputs 224 -> 194.
struct PlainForm {
  int bm, bn, occ;
  float start, lat, load, per_tile, stream, store;
};
static const PlainForm kPlainForms[] = {
    {128, 128, 1, 2.926f, 0.4991f, 0.5102f, 0.6004f, 0.2037f, 0.2054f},  // plain, 4-step ring
    {128, 128, 2, 2.024f, 0.871f, 0.1203f, 0.3671f, 0.1948f, 0.197f},    // plain, 2-step ring
    {64, 128, 2, 2.651f, 0.4285f, 0.3284f, 0.0f, 0.2202f, 0.1739f},      // plain, 3-step ring
    {64, 64, 4, 3.114f, 0.4166f, 0.2283f, 0.2235f, 0.1818f, 0.1077f},    // 2 waves
    {64, 64, 2, 3.068f, 0.1199f, 0.238f, 0.00318f, 0.1701f, 0.1348f},    // 4 waves
    {64, 32, 1, 2.671f, 0.0681f, 0.1599f, 1.263f, 0.1958f, 0.3708f},     // 4 waves, 2 stages
    {32, 32, 2, 2.285f, 0.1266f, 0.1197f, 0.01813f, 0.1719f, 0.3065f},   // 4 waves, 2 stages
    {16, 32, 3, 2.193f, 0.03946f, 0.1232f, 0.0f, 0.1494f, 0.3613f},      // 4 waves, 2 stages
    {16, 16, 3, 2.258f, 0.04214f, 0.07793f, 0.0f, 0.1227f, 0.3837f},     // 4 waves, 3 stages
};

// mb_out: what the output moves (its own bytes, a residual's, a second output's). Runs on the host before
// every product: 32-bit divisions only.
static float plain_form_us(const PlainForm& f, u32 tiles, int ksteps, float mb_b, float mb_out, u32 cus) {
  const u32 x = (tiles + cus - 1) / cus, rounds = (x + f.occ - 1) / f.occ;
  const float step = f.lat * rounds > f.load * x ? f.lat * rounds : f.load * x;
  const float work = ksteps * step + f.per_tile * (x - 1), stream = f.stream * mb_b;
  return f.start + (work > stream ? work : stream) + f.store * mb_out;
}

// Whether uwc_gemm_plain_any takes the product: whole k steps, 16-byte output rows (and residual
// rows), four column scales per load, 32-bit operand offsets within a tile; without an output, whole
// 128 x 128 tiles.
bool uwc_plain_any_fits(int m, int n, int k, int ldc, const void* out, int out_mode, const float* b_scale,
                        const float* res, const float* out2) {
  if (k % P_BK || k < P_BK || k > (1 << 23)) return false;
  if (out_mode == P_OUT_NONE) return m % 128 == 0 && n % 128 == 0;
  const bool vec_out = (uintptr_t)out % 16 == 0 && ldc % 4 == 0 && n % 4 == 0 && (uintptr_t)res % 16 == 0 &&
                       (uintptr_t)out2 % 16 == 0;
  const bool vec_scale = (out_mode == P_OUT_I32 && !out2) || (uintptr_t)b_scale % 16 == 0;
  return vec_out && vec_scale;
}

// The form a product takes: the one predicted fastest, or without an output (timing probes) the 4-step
// ring while a CU has at most one tile and the 2-step one beyond.
int uwc_plain_form(int m, int n, int k, int out_mode, int out_bytes, int cus) {
  if (out_mode == P_OUT_NONE) return (long)(m / 128) * (n / 128) <= cus ? 0 : 1;
  const float mb_b = 1e-6f * n * k, mb_out = 1e-6f * m * n * out_bytes;
  int best = 0;
  float best_us = 0.0f;
  for (int i = 0; i < (int)(sizeof(kPlainForms) / sizeof(kPlainForms[0])); i++) {
    const PlainForm& f = kPlainForms[i];
    // a grid of 2^32 threads or more would be cut off without an error (2^28 rows of 16 columns on 16 x 16 tiles)
    const u64 tiles = (((u64)m + f.bm - 1) >> __builtin_ctz(f.bm)) * (((u64)n + f.bn - 1) >> __builtin_ctz(f.bn));
    if (i > 0 && tiles * P_THREADS > 0xFFFFFFFFull) continue;
    const float us = plain_form_us(f, tiles < 0xFFFFFFFFull ? (u32)tiles : 0xFFFFFFFFu, k / P_BK, mb_b, mb_out, (u32)cus);
    if (i == 0 || us < best_us) best = i, best_us = us;
  }
  return best;
}

// A plain GEMM of any m; res (with P_OUT_F32): the residual, out2 (with P_OUT_I32): the dequantized rows
// beside the sums, both of the output's row stride. Called after the argument checks of uwc_noisy_gemm
// and uwc_plain_any_fits.
int uwc_gemm_plain_any(const int8_t* A, const int8_t* B, int m, int n, int k, const float* a_scale,
                       const float* b_scale, const float* res, void* out, float* out2, int out_mode, int ldc,
                       hipStream_t stream) {
  const PlainParams p{A, B, m, n, k, a_scale, b_scale, out, ldc, res, out2};
  const int mode = res ? P_OUT_F32R : out2 ? P_OUT_BOTH : out_mode;
  const int out_bytes = res || out2 ? 8 : mode == P_OUT_BF16 ? 2 : 4;
  switch (uwc_plain_form(m, n, k, out_mode, out_bytes, uwc_cu_count())) {
    case 0: plain_any<128, 128, 4>(mode, stream, p); break;
    case 1: plain_any<128, 128, 2>(mode, stream, p); break;
    case 2: plain_any<64, 128, 3>(mode, stream, p); break;
    case 3: wave_out<64, 64, 32, 2, 1>(mode, stream, p); break;
    case 4: wave_out<64, 64, 32, 4, 1>(mode, stream, p); break;
    case 5: wave_out<64, 32, 32, 4, 2>(mode, stream, p); break;
    case 6: wave_out<32, 32, 32, 4, 2>(mode, stream, p); break;
    case 7: wave_out<16, 32, 16, 4, 2>(mode, stream, p); break;
    default: wave_out<16, 16, 16, 4, 3>(mode, stream, p); break;
  }
  return uwc_launch_status("plain_gemm");
}
