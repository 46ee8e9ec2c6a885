// The MLP's output projection x = r1 x + p1 (h @ W^T) (W stored (N, K) bf16)
// where its tiles fill the CUs (gemm_big_routes has the measurements against
// k_gemm_ring): 256 x 256 (or 256 x 192) output tiles of
// four waves of 128 x 128 (128 x 96), one work-group (one wave per SIMD) per
// CU, v_mfma_f32_16x16x32_bf16 -- the tile that moves the fewest bytes per
// flop.
//
// Main loop (K tiles of 64, two LDS stages, one barrier per K tile):
//   * the 256 accumulators of a wave live in AGPRs: the MFMA is issued as
//     inline assembly whose accumulator operand is an AGPR ("+a").  With the
//     compiler builtin the accumulators move between AGPRs and VGPRs inside the
//     loop (368 v_accvgpr moves per K tile, measured ~10% slower);
//   * the fragments are read with volatile inline ds_read_b128 in a fixed
//     order -- the first k-step's eight W fragments and the first A fragment,
//     then the second k-step's W fragments -- and each A fragment one group of
//     eight MFMAs ahead of its use, with hand-placed s_waitcnt (the compiler's
//     scheduler otherwise reads every A fragment right before its MFMAs and
//     waits for it);
//   * each of the 16 MFMA groups of a K tile first stores one 16-byte chunk per
//     thread of the next K tile into the other LDS stage and refills that
//     register with the tile after it, so the tile traffic hides behind the
//     MFMAs.  All of these are unconditional (past the last K tile they re-read
//     it and fill the stage no later iteration reads): a branch there makes the
//     compiler wait on every load in flight.  The prologue issues the second
//     tile's loads in the loop's order, so the loop's waits stay vmcnt(15).
//   * LDS tiles are unpadded 128-byte rows with chunk c of row r at slot
//     c ^ ((r >> 1) & 7): conflict-free for the chunk stores and the
//     16-row fragment reads.
// The MFMA operands are swapped (C^T = W A^T) so that a lane holds four
// consecutive columns of one row.  Epilogue: the tile is rounded to bf16 (as
// the reference's eager ops do) into LDS (row pitch 264: the 8-byte writes of
// 16 rows spread over the banks), then each thread mixes 16-byte row chunks (x
// read and written as 16-byte words, the first batch loaded before the
// staging).  With one wave per SIMD nothing hides the epilogue's VALU work, so
// every eager rounding is a packed pair conversion (v_cvt_pk_bf16_f32).
// Work-group i runs on XCD i % 8; each XCD takes a contiguous range of tiles,
// N-fastest, so the N tiles of an M block share its A rows in that XCD's L2.
#include <type_traits>
#include "common.h"
#include "launch.h"

namespace ann {

namespace {

constexpr int BG_BM = 256, BG_BN = 256, BG_BK = 64;   // BG_BN: the widest tile
constexpr int BG_EP = 264;   // bf16 row pitch of the staged output tile
constexpr int BG_EB = 8;     // residual epilogue: 16-byte chunks per thread loaded at once
constexpr size_t BG_LDS_MAIN = (size_t)2 * (BG_BM + BG_BN) * BG_BK * 2;
constexpr size_t BG_LDS_EPI = (size_t)BG_BM * BG_EP * 2;
constexpr size_t BG_LDS = BG_LDS_MAIN > BG_LDS_EPI ? BG_LDS_MAIN : BG_LDS_EPI;

typedef __bf16 bg_bf16x8 __attribute__((ext_vector_type(8)));
typedef float bg_floatx4 __attribute__((ext_vector_type(4)));
typedef unsigned bg_u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) char bg_lds_char;

template <int I, int N, typename F>
__device__ __forceinline__ void bg_static_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    bg_static_for<I + 1, N>(f);
  }
}

__device__ __forceinline__ int bg_off(int r, int c) { return r * BG_BK + ((c ^ ((r >> 1) & 7)) << 3); }

__device__ __forceinline__ void bg_mfma(bg_floatx4& acc, const bg_bf16x8& a, const bg_bf16x8& b) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
}

template <int OFF>
__device__ __forceinline__ bg_bf16x8 bg_lds_read(const bg_lds_char* p) {
  bg_bf16x8 v;
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(p), "i"(OFF));
  return v;
}

template <int N>
__device__ __forceinline__ void bg_wait_lgkm() {
  asm volatile("s_waitcnt lgkmcnt(%0)" ::"i"(N) : "memory");
}

}  // namespace


template <int BN>
__global__ __launch_bounds__(256, 1) void k_gemm_big(const bf16_t* A, int lda, const bf16_t* W,
                                                     int M, int N, int K, EpiArgs ea) {
  static_assert(BN == 256 || BN == 192, "tile width");
  constexpr int NJ = BN / 32;    // 16-column blocks of a wave (two waves across the tile)
  constexpr int NWU = BN / 32;   // W chunks per thread and K tile
  constexpr int CPR = BN / 8;    // 16-byte chunks per output row
  extern __shared__ __attribute__((aligned(16))) bf16_t smem[];
  auto As = [&](int s) { return smem + s * BG_BM * BG_BK; };
  auto Ws = [&](int s) { return smem + 2 * BG_BM * BG_BK + s * BN * BG_BK; };
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int wm = wv >> 1, wn = wv & 1;
  const int ntm = (M + BG_BM - 1) / BG_BM, ntn = N / BN, nt = ntm * ntn;
  const int per = (nt + 7) / 8;
  const int t = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if (t >= nt) return;
  const int tm = t / ntn, tn = t % ntn;
  const int m0 = tm * BG_BM, n0 = tn * BN;
  const int KT = K / BG_BK;

  // staged K-tile chunks: chunk g of a thread is operand g & 1 (A, W), row
  // block g >> 1 (rows (tid >> 3) + 32 u), 16-byte column tid & 7
  bg_u32x4 ra[8], rw[8];
  const int crow = tid >> 3, cc = tid & 7;
  auto gload1 = [&](int op, int u, int kt) {
    const int row = crow + 32 * u;
    if (op == 0)
      ra[u] = *(const bg_u32x4*)(A + (size_t)min(m0 + row, M - 1) * lda + kt * BG_BK + cc * 8);
    else if (u < NWU)
      rw[u] = *(const bg_u32x4*)(W + (size_t)(n0 + row) * K + kt * BG_BK + cc * 8);
  };
  auto lstore1 = [&](int op, int u, int s) {
    const int row = crow + 32 * u;
    if (op == 0) *(bg_u32x4*)(As(s) + bg_off(row, cc)) = ra[u];
    else if (u < NWU) *(bg_u32x4*)(Ws(s) + bg_off(row, cc)) = rw[u];
  };

  bg_floatx4 acc[8][NJ];
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = (bg_floatx4){0.f, 0.f, 0.f, 0.f};
  const int r16 = lane & 15, kg = lane >> 4;

  // prologue: tile 0 into stage 0, tile 1 (clamped) in flight in the
  // loop's order, each load pinned in place
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    gload1(0, u, 0);
    gload1(1, u, 0);
  }
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    lstore1(0, u, 0);
    lstore1(1, u, 0);
  }
  bg_static_for<0, 16>([&](auto gc) __attribute__((always_inline)) {
    constexpr int g = decltype(gc)::value;
    gload1(g & 1, g >> 1, min(1, KT - 1));
    asm volatile("" ::: "memory");
  });
  __syncthreads();

  for (int kt = 0; kt < KT; ++kt) {
    const int s = kt & 1;
    const bf16_t* as = As(s) + (wm * 128 + r16) * BG_BK;
    const bf16_t* ws = Ws(s) + (wn * (BN / 2) + r16) * BG_BK;
    const int ch0 = kg ^ ((r16 >> 1) & 7), ch1 = (4 + kg) ^ ((r16 >> 1) & 7);
    const bg_lds_char* pa0 = (const bg_lds_char*)(as + (ch0 << 3));
    const bg_lds_char* pa1 = (const bg_lds_char*)(as + (ch1 << 3));
    const bg_lds_char* pb0 = (const bg_lds_char*)(ws + (ch0 << 3));
    const bg_lds_char* pb1 = (const bg_lds_char*)(ws + (ch1 << 3));
    bg_bf16x8 b0[NJ], b1[NJ];
    bg_static_for<0, NJ>([&](auto jc) __attribute__((always_inline)) {
      constexpr int j = decltype(jc)::value;
      b0[j] = bg_lds_read<j * 16 * BG_BK * 2>(pb0);
    });
    bg_bf16x8 a = bg_lds_read<0>(pa0);
    bg_static_for<0, NJ>([&](auto jc) __attribute__((always_inline)) {
      constexpr int j = decltype(jc)::value;
      b1[j] = bg_lds_read<j * 16 * BG_BK * 2>(pb1);
    });
    // b0 and a; the b1 reads may still fly.  A wave's LDS reads return in
    // issue order, so lgkmcnt(NJ) leaves only the last NJ issued (the b1
    // reads) outstanding; any scalar load the compiler has in flight counts
    // on the same counter and only makes the wait stricter.  The lgkmcnt(0)
    // after each MFMA group covers the next A fragment the same way.
    bg_wait_lgkm<NJ>();
    bg_static_for<0, 16>([&](auto gc) __attribute__((always_inline)) {
      constexpr int g = decltype(gc)::value;
      constexpr int i = g & 7, kh = g >> 3;
      bg_bf16x8 an = a;
      if constexpr (g < 15) {
        constexpr int ni = (g + 1) & 7;
        an = ((g + 1) >> 3) ? bg_lds_read<ni * 16 * BG_BK * 2>(pa1)
                            : bg_lds_read<ni * 16 * BG_BK * 2>(pa0);
      }
      lstore1(g & 1, g >> 1, s ^ 1);
      gload1(g & 1, g >> 1, min(kt + 2, KT - 1));
      asm volatile("" ::: "memory");
#pragma unroll
      for (int j = 0; j < NJ; ++j) bg_mfma(acc[i][j], kh ? b1[j] : b0[j], a);
      if constexpr (g < 15) bg_wait_lgkm<0>();
      a = an;
    });
    // After the loop the accumulators leave their AGPRs through
    // v_accvgpr_read / _mov (the epilogue and the register allocator's
    // copies).  The compiler's hazard recognizer does not see these MFMAs
    // (inline assembly), so the wait states an XDL result needs before a VALU
    // or v_accvgpr instruction reads it are placed here by hand: the CDNA3 /
    // CDNA4 ISA's MAI dependency table asks NumPasses + 3 (+1 on gfx950) for
    // "XDL write VGPR -> VALU read", 12 for the 8-pass
    // v_mfma_f32_16x16x32_bf16; three s_nop 7 give 24.  In the loop body,
    // after the last MFMA group, every copy on the loop's exit path comes
    // after them; they issue while the MFMA pipe drains the group, before
    // the barrier.
    asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7" ::: "memory");
    __syncthreads();
  }

  // residual epilogue: x chunks of the first batch loaded before the staging
  // (chunk q = tid + 256 u is row q / CPR, columns 8 (q % CPR); rows past M
  // read row M - 1 and are never stored)
  static_assert(CPR % BG_EB == 0, "whole batches");
  bg_u32x4 xv[2][BG_EB];
  auto res_load = [&](int b) {
#pragma unroll
    for (int e = 0; e < BG_EB; ++e) {
      const int q = tid + 256 * (b * BG_EB + e);
      const size_t i = (size_t)min(m0 + q / CPR, M - 1) * ea.ldr + n0 + (q % CPR) * 8;
      xv[b & 1][e] = *(const bg_u32x4*)(ea.x + i);
    }
  };
  res_load(0);
  // ---- stage bf16(y): lane holds row m = block row + r16, columns 4 kg ..
  bf16_t* st = smem;
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int ml = wm * 128 + i * 16 + r16, nl = wn * (BN / 2) + j * 16 + 4 * kg;
      const bg_floatx4 v = acc[i][j];
      *(uint2*)(st + ml * BG_EP + nl) = make_uint2(pack2(v[0], v[1]), pack2(v[2], v[3]));
    }
  __syncthreads();
  // 16-byte row chunks; batch b + 1's loads fly while batch b is mixed and stored
  float lam[5];
#pragma unroll
  for (int e = 0; e < 5; ++e) lam[e] = ea.lam[e];
#pragma unroll
  for (int b = 0; b < CPR / BG_EB; ++b) {
    if (b + 1 < CPR / BG_EB) res_load(b + 1);
#pragma unroll
    for (int e = 0; e < BG_EB; ++e) {
      const int q = tid + 256 * (b * BG_EB + e);
      const int ml = q / CPR, c8 = (q % CPR) * 8;
      const bg_u32x4 y = *(const bg_u32x4*)(st + ml * BG_EP + c8);
      const bg_u32x4 x = xv[b & 1][e];
      bg_u32x4 o;
#pragma unroll
      for (int f = 0; f < 4; ++f) o[f] = mix_mlp_pair(lam, x[f], y[f]);
      if (m0 + ml < M) *(bg_u32x4*)(ea.x + (size_t)(m0 + ml) * ea.ldr + n0 + c8) = o;
    }
  }
}

int device_cus() {
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
      cus <= 0)
    return 256;
  return cus;
}

// Tile width for an M x N output: 256 or 192 columns, whichever needs fewer
// CU-rounds times columns (one work-group per CU), a 192-column tile counted
// 15% dearer per column (less reuse of each A tile: 480 x 16 tiles of 192
// against 480 x 12 of 256 measured 818 against 713 us).
static int big_bn(int M, int N) {
  static const int cus = device_cus();
  if (N % 192) return 256;
  if (N % 256) return 192;
  const long long ntm = (M + BG_BM - 1) / BG_BM;
  auto rounds = [&](int bn) { return (ntm * (N / bn) + cus - 1) / cus; };
  return rounds(192) * 192 * 115 < rounds(256) * 256 * 100 ? 192 : 256;
}

// Whether an (M, N) = (rows, d) product over K comes here instead of
// k_gemm_ring.  Here a full round of the CUs takes 1.53 us per K tile and 17 us
// besides at 256 columns, 1.21 and 17 at 192, and a round that is not full hardly
// less; the ring takes 1.2 times its rule's figure behind the fc projection that
// has just written A (those are of a launch repeated by itself).  So a shape that
// fills its rounds comes here, and most of what is past the memory-side cache,
// where the ring's narrower tiles read A more often.  Measured behind the fc, ring
// / here, us: d 512 (K 2048) at 16384 rows 35 / 59, 40960 90 / 122, 65536 167 /
// 127; d 768 at 8192 rows 52 / 65, 16384 77 / 73, 19200 108 / 90, 32768 161 /
// 149, 65536 328 / 298; d 1024 at 16384 124 / 117, 19200 155 / 213, 32768 323 /
// 261; d 1536 at 4096 98 / 121, 10240 193 / 164, 16384 285 / 261, 32768 569 /
// 512; d 2048 at 8192 233 / 213, 10240 322 / 374, 16384 544 / 472.  Over 99 shapes
// of d 256 .. 2048 the choice loses 0.7% on the faster one in the mean and 11% at
// the worst (12288 rows, d 1024: 97 / 108).
bool gemm_big_routes(int M, int N, int K) {
  static const int cus = device_cus();
  const int bn = big_bn(M, N);
  if (N % bn) return false;
  const long long ring = gemm_ring_ns(EPI_RESID_MLP, false, M, N, K);
  if (ring < 0) return true;
  const long long tiles = (long long)((M + BG_BM - 1) / BG_BM) * (N / bn);
  const long long ns = (tiles + cus - 1) / cus *
                       ((long long)(K / BG_BK) * (bn == 256 ? 1530 : 1210) + 17000);
  return ns * 5 < ring * 6;
}

// Whether gemm_big can take (M, N, K): whole 256- or 192-column tiles, 64-deep
// K tiles, 16-byte aligned rows, and enough tiles (at least 96) for the one-
// work-group-per-CU kernel to fill the chip.
bool gemm_big_fits(const bf16_t* A, int lda, int M, int N, int K, const EpiArgs& ea) {
  if (M < 512 || N % 64 || K % BG_BK || K < BG_BK || lda % 8 || ((uintptr_t)A & 15)) return false;
  const int bn = big_bn(M, N);
  if (N % bn) return false;
  if ((long long)((M + BG_BM - 1) / BG_BM) * (N / bn) < 96) return false;
  return ea.x && ea.lam && ea.ldr % 8 == 0 && ((uintptr_t)ea.x & 15) == 0;
}

template <int BN>
static hipError_t launch_big(const bf16_t* A, int lda, const bf16_t* W, int M, int N, int K,
                             const EpiArgs& ea, hipStream_t st) {
  static PerDevice limit;
  const hipError_t attr = lds_limit(limit, (const void*)k_gemm_big<BN>, BG_LDS);
  if (attr != hipSuccess) return attr;
  const int nt = ((M + BG_BM - 1) / BG_BM) * (N / BN);
  const int grid = (nt + 7) / 8 * 8;
  hipLaunchKernelGGL((k_gemm_big<BN>), dim3(grid), dim3(256), BG_LDS, st, A, lda, W, M, N, K, ea);
  return hipGetLastError();
}

hipError_t gemm_big(const bf16_t* A, int lda, const bf16_t* W, int M, int N, int K,
                    const EpiArgs& ea, hipStream_t st) {
  if (!gemm_big_fits(A, lda, M, N, K, ea)) return hipErrorInvalidValue;
  return big_bn(M, N) == 192 ? launch_big<192>(A, lda, W, M, N, K, ea, st)
                             : launch_big<256>(A, lda, W, M, N, K, ea, st);
}

}  // namespace ann
