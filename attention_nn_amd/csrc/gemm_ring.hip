// Projections y = a @ W^T (W stored (N, K) bf16) of more than 128 rows: one
// ordinary prompt, a batch's prompts, the scoring of a text, the training
// forward.  K tiles of 64 are streamed straight into a ring of NS LDS stages
// (global_load_lds_dwordx4, no register staging), one barrier per K tile; the
// output tile is chosen by the shape (ring_pick).
//
// What bounds it.  Time per K tile (slope over K, residual epilogue) at 32 x 64,
// 64 x 64, 128 x 64, 128 x 128 and 128 x 192: 0.17, 0.24, 0.36, 0.60 and 0.73 us
// with one work-group on each CU, 0.30, 0.38, 0.56, 0.86 and 1.20 for two that
// share one -- 16 and 24 KB a work-group of the 64- and 128 x 64 tiles through
// the CU's load path, about 85 GB/s per CU.  So a shape that leaves CUs idle wants
// small tiles on all of them, and a shape that fills them wants large tiles,
// which move fewer bytes per flop: 0.43 and 0.60 us a work-group at 128 x 128 and
// 128 x 192, where the MFMAs alone take 0.31 and 0.46 (1.75 PFLOP/s, the form's
// measured ceiling).  Two work-groups share a CU at every tile: their barriers
// fall apart in time, so one reads LDS and waits while the other multiplies, and
// one's epilogue runs under the other's main loop.  One work-group of eight waves
// with the same tiles (256 x 128, two or three stages) is slower for that reason
// (proj of 32768 rows, d 768: by 9%), as are K tiles of 32 (half cache lines: 16%)
// and v_mfma_f32_32x32x16 (23% at 128 x 128).
#include <type_traits>
#include "common.h"
#include "epilogue.h"
#include "launch.h"

namespace ann {

namespace {

constexpr int RG_BK = 64;
constexpr int RG_RB = RG_BK * 2;   // bytes of an LDS row

typedef __bf16 rg_bf16x8 __attribute__((ext_vector_type(8)));
typedef float rg_floatx4 __attribute__((ext_vector_type(4)));
typedef uint32_t rg_u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 rg_bf16x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) void rg_lds_void;
typedef short rg_v4i16 __attribute__((ext_vector_type(4)));
typedef short rg_v8i16 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) rg_v4i16 rg_lds_v4i16;

// c + the sum of squares of a fragment's eight values (v_dot2_f32_bf16)
__device__ __forceinline__ float rg_sumsq(const rg_bf16x8& a, float c) {
#pragma unroll
  for (int e = 0; e < 8; e += 2) {
    const rg_bf16x2 v = {a[e], a[e + 1]};
    c = __builtin_amdgcn_fdot2_f32_bf16(v, v, c, false);
  }
  return c;
}

template <int I, int N, typename F>
__device__ __forceinline__ void rg_static_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    rg_static_for<I + 1, N>(f);
  }
}

// This wave's loads but the newest N have landed and its LDS reads are done
// (another wave's load may overwrite what they read), then every wave's.
template <int N>
__device__ __forceinline__ void rg_wait_barrier() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"i"(N) : "memory");
}

// Whether a tile forms rms(A) @ W^T from A itself.
constexpr bool ring_takes_rms(int epi, int bm, int bn) {
  return (epi == EPI_STORE || epi == EPI_RELU2 || epi == EPI_QKV) && bm * bn <= 128 * 64;
}

template <int BM, int BN, int NS>
constexpr size_t rg_lds_bytes() {
  const size_t ring = (size_t)NS * (BM + BN) * RG_RB, epi = (size_t)BM * (BN + 8) * 2;
  return ring > epi ? ring : epi;
}

}  // namespace

// acc = the (m0, n0) tile of C^T = W A^T: block (N block j, M block i), so that a
// lane holds four consecutive columns of one row; ss (SQ): this lane's part of
// the sums of squares of the A rows (row r16 of M block i, summed over the
// four lanes of that r16).  W is (N, K); WT: (K, N), rows of ldw values, whose
// fragments come out of LDS through the transposing read.  LDS from rg_smem's
// start; a barrier has to follow before it is written again.
template <int BM, int BN, int NS, int WR, int WC, bool SQ, bool WT = false>
__device__ __forceinline__ void ring_product(const bf16_t* A, int lda, const bf16_t* W, int M,
                                             int N, int K, int m0, int n0, int wv, int lane,
                                             rg_floatx4 (&acc)[BN / WC / 16][BM / WR / 16],
                                             float (&ss)[BM / WR / 16], int ldw = 0) {
  static_assert(!WT || (BN == 128 && WR * WC == 4 && NS == 2), "256-byte rows of a K tile");
  constexpr int NW = WR * WC;
  constexpr int WM = BM / WR, MT = WM / 16;
  constexpr int WN = BN / WC, NT = WN / 16;
  constexpr int LA = BM / 8 / NW, LW = BN / 8 / NW;   // 1 KB loads per wave per K tile
  constexpr int SB = (BM + BN) * RG_RB;               // bytes of a stage
  extern __shared__ __attribute__((aligned(16))) unsigned char rg_smem[];
  // load u of this wave fills rows 8 (NW u + wv) .. + 7 of the operand's tile
  // in LDS: lane l row l >> 3, slot l & 7, which holds logical 16-byte chunk
  // (l & 7) ^ ((row >> 1) & 7) -- conflict-free for the 16-row fragment reads.
  // Rows past M / N repeat the last one (they feed outputs never stored).
  const bf16_t* pa[LA];
  const bf16_t* pw[LW];
  const int KT = K / RG_BK;
#pragma unroll
  for (int u = 0; u < LA; ++u) {
    const int r = 8 * (NW * u + wv) + (lane >> 3);
    pa[u] = A + (size_t)min(m0 + r, M - 1) * lda + (((lane & 7) ^ ((r >> 1) & 7)) << 3);
  }
#pragma unroll
  for (int u = 0; u < LW; ++u) {
    if constexpr (WT) {
      // four K rows of 256 bytes a load: row lane >> 4, slot lane & 15 holding
      // chunk slot ^ 2 s(row), s = row bits 0, 1 and 3: the transposing reads of
      // a half wave (8 rows, two chunks each) meet every bank group once
      const int r = 4 * (NW * u + wv) + (lane >> 4);
      const int c = (lane & 15) ^ (2 * ((r & 3) | ((r >> 1) & 4)));
      pw[u] = W + (size_t)r * ldw + n0 + c * 8;
    } else {
      const int r = 8 * (NW * u + wv) + (lane >> 3);
      pw[u] = W + (size_t)min(n0 + r, N - 1) * K + (((lane & 7) ^ ((r >> 1) & 7)) << 3);
    }
  }
  const size_t wstep = WT ? (size_t)RG_BK * ldw : (size_t)RG_BK;
  // (the builtin's operands have plain types: clang's host pass drops a kernel
  // in which a type-dependent call of its 16-byte form is instantiated)
  auto issue = [&](int kt, int s) {
    unsigned char* st = rg_smem + s * SB;
#pragma unroll
    for (int u = 0; u < LA; ++u) {
      const bf16_t* src = pa[u] + kt * RG_BK;
      __builtin_amdgcn_global_load_lds(src, (rg_lds_void*)(st + (NW * u + wv) * 1024), 16, 0, 0);
    }
    st += BM * RG_RB;
#pragma unroll
    for (int u = 0; u < LW; ++u) {
      const bf16_t* src = pw[u] + kt * wstep;
      __builtin_amdgcn_global_load_lds(src, (rg_lds_void*)(st + (NW * u + wv) * 1024), 16, 0, 0);
    }
  };

#pragma unroll
  for (int i = 0; i < MT; ++i) ss[i] = 0.f;
#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int i = 0; i < MT; ++i) acc[j][i] = (rg_floatx4){0.f, 0.f, 0.f, 0.f};

  // the k steps of 32 run in order, as in every GEMM here: one product has the
  // same bits whatever the tile (of rms(A): those of the tiles that form it)
  const int r16 = lane & 15, kg = lane >> 4, sw = (r16 >> 1) & 7;
  const int wm = wv / WC, wn = wv % WC;
  const int oa = (wm * WM + r16) * RG_RB, ow = BM * RG_RB + (wn * WN + r16) * RG_RB;
  const int c0 = (kg ^ sw) << 4, c1 = ((4 + kg) ^ sw) << 4;
  // WT: within each 16-lane group, lane m receives column m of four K rows, row
  // e of them addressed by lanes 4e .. 4e + 3; k = 8 kg + 0 .. 3 and + 4 .. 7 in
  // two reads give the fragment of the untransposed form
  int tw[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j)
    tw[j] = BM * RG_RB + (8 * kg + (r16 >> 2)) * 256 +
            ((((wn * WN + j * 16) / 8) ^ (2 * ((r16 >> 2) | ((kg & 1) << 2)))) +
             ((r16 & 3) >> 1)) * 16 + (r16 & 1) * 8;
  auto compute = [&](int s, auto&& mid) {
    const unsigned char* st = rg_smem + s * SB;
    rg_bf16x8 a[2][MT], w[2][NT];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        if constexpr (WT) {
          const unsigned char* src = st + tw[j] + h * 32 * 256;
          const rg_v4i16 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((rg_lds_v4i16*)src);
          const rg_v4i16 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((rg_lds_v4i16*)(src + 4 * 256));
          const rg_v8i16 v = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
          w[h][j] = __builtin_bit_cast(rg_bf16x8, v);
        } else {
          w[h][j] = *(const rg_bf16x8*)(st + ow + j * 16 * RG_RB + (h ? c1 : c0));
        }
      }
#pragma unroll
      for (int i = 0; i < MT; ++i)
        a[h][i] = *(const rg_bf16x8*)(st + oa + i * 16 * RG_RB + (h ? c1 : c0));
    }
    mid();
    __builtin_amdgcn_sched_barrier(0);   // all reads in flight, then the MFMAs
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < MT; ++i) {
#pragma unroll
        for (int j = 0; j < NT; ++j)
          acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[h][j], a[h][i], acc[j][i], 0, 0, 0);
        if constexpr (SQ) ss[i] = rg_sumsq(a[h][i], ss[i]);
      }
  };

  // ring: K tile t in stage t % NS, loaded NS - 1 tiles ahead.  The barrier
  // that follows the wait for tile t also says that every wave is done with
  // the stage of tile t - 1, which tile t + NS - 1 then overwrites.  (With
  // fewer K tiles than that the last one is loaded again, and not used.)
#pragma unroll
  for (int t = 0; t < NS - 1; ++t) issue(min(t, KT - 1), t);
  int s = 0;
  for (int t = 0; t < KT - (NS - 1); ++t) {
    rg_wait_barrier<(NS - 2) * (LA + LW)>();
    // WT: the loads go out after the LDS reads, before whose transposing form
    // the compiler waits for every load into LDS in flight
    auto next = [&]() { issue(t + NS - 1, s == 0 ? NS - 1 : s - 1); };
    if constexpr (!WT) next();
    compute(s, [&]() {
      if constexpr (WT) next();
    });
    s = s + 1 == NS ? 0 : s + 1;
  }
  rg_static_for<0, NS - 1>([&](auto tc) __attribute__((always_inline)) {
    rg_wait_barrier<(NS - 2 - decltype(tc)::value) * (LA + LW)>();
    if (decltype(tc)::value < KT) compute(s, []() {});
    s = s + 1 == NS ? 0 : s + 1;
  });
}

// WR x WC waves.  gm: tile rows per group of the tile order.
template <int EPI, int BM, int BN, int NS, int WR, int WC, bool RAG = false>
__global__ __launch_bounds__(64 * WR * WC) __attribute__((amdgpu_waves_per_eu(2))) void k_gemm_ring(
    const bf16_t* __restrict__ A, int lda, const bf16_t* __restrict__ W, int M, int N, int K,
    int gm, EpiArgs ea) {
  constexpr int NW = WR * WC, TH = 64 * NW;
  constexpr int WM = BM / WR, MT = WM / 16;
  constexpr int WN = BN / WC, NT = WN / 16;
  constexpr int CPR = BN / 8, NCH = BM * CPR / TH, CP = BN + 8;
  constexpr bool RES = EPI == EPI_RESID_ATTN || EPI == EPI_RESID_MLP;
  // the residual operands: loaded first where the tile is small (a few
  // registers, and nothing else hides the latency), after the main loop else
  constexpr bool EARLY = RES && BM * BN <= 128 * 64;
  // the qkv and fc projections are of rms(x).  The small tiles take x itself
  // as A and scale y by the row's rsqrt(mean(x^2) + eps) after the product; the
  // sums of squares come from the A fragments on their way to the MFMAs (four
  // dot instructions each), so that no launch normalises a copy first: 155M
  // prompts of 777 / 300 tokens 690 -> 647 and 594 -> 547 us.  The large tiles
  // have no issue slots for that (d 1536, 128 x 1024 tokens and 24 steps: 36.55
  // ms with it, 35.80 without).  The lm_head always takes the
  // rounded rms(x), so that z is the same bits on every route to it.  Which of
  // the two A is comes from the caller (gemm_ring's rms): for a plain A the small
  // tiles of these epilogues are not picked.
  constexpr bool RMS = ring_takes_rms(EPI, BM, BN);
  static_assert(BM % (8 * NW) == 0 && BN % (8 * NW) == 0 && BM * CPR % TH == 0, "whole loads");
  static_assert(EPI != EPI_QKV || (BN == 128 && TH == 256), "whole heads per tile");
  extern __shared__ __attribute__((aligned(16))) unsigned char rg_smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wv / WC, wn = wv % WC;
  // Tile order: each XCD (work-group b runs on XCD b % 8) takes a contiguous
  // range of the tiles, which are ordered in groups of gm tile rows, column
  // by column, so that the tiles at work together on an XCD share A and W
  // rows in its L2 (a bijection of the grid, correct under any dispatch).
  // gm 4 against row by row, 128 x 128 tiles: qkv of 8192 rows, d 1536, 134 ->
  // 120 us, fc 167 -> 142; d 768 up to 10%; gm 8 equal, 16 slower.
  int tm, tn;
  {
    const int nbn = gridDim.x, nbm = gridDim.y, total = nbn * nbm;
    const int bid = blockIdx.y * nbn + blockIdx.x;
    const int x = bid & 7, q = total >> 3, r = total & 7;
    const int t = x * q + min(x, r) + (bid >> 3);
    const int g = t / (gm * nbn), rem = t - g * gm * nbn;
    const int h = min(gm, nbm - g * gm);
    tn = rem / h;
    tm = g * gm + rem - tn * h;
  }
  const int m0 = tm * BM, n0 = tn * BN;

  // chunk q = tid + TH u of the output tile: row q / CPR, columns 8 (q % CPR)
  uint4 xv[RES ? NCH : 1], zv[EPI == EPI_RESID_ATTN ? NCH : 1];
  auto res_load = [&]() {
#pragma unroll
    for (int u = 0; u < NCH; ++u) {
      const int q = tid + TH * u;
      const size_t i = (size_t)min(m0 + q / CPR, M - 1) * ea.ldr + min(n0 + (q % CPR) * 8, N - 8);
      xv[u] = *(const uint4*)(ea.x + i);
      if constexpr (EPI == EPI_RESID_ATTN) zv[u] = *(const uint4*)(ea.x0 + i);
    }
  };
  if constexpr (EARLY) res_load();

  const int r16 = lane & 15, kg = lane >> 4;
  float ss[MT];
  rg_floatx4 acc[NT][MT];
  ring_product<BM, BN, NS, WR, WC, RMS>(A, lda, W, M, N, K, m0, n0, wv, lane, acc, ss);

  if constexpr (RMS) {
    // a lane's column of C^T is row r16 of its M blocks, whose squares the four
    // lanes of that r16 have summed
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      float t = ss[i];
      t += __shfl_xor(t, 16, 64);
      t += __shfl_xor(t, 32, 64);
      const float f = rsqrtf(t / (float)K + ea.eps);
#pragma unroll
      for (int j = 0; j < NT; ++j) acc[j][i] *= f;
    }
  }
  if constexpr (EPI == EPI_CE) {
    // softcap(bf16(z)) in (0, 23): sum exp(zc) needs no max pass.  Row sums:
    // in-lane over the wave's N blocks, then over the four lane groups, then
    // the column parts through LDS, always in the same order.  Hardware exp2
    // and reciprocal: the IEEE expf and division cost ~35 VALU instructions
    // per logit.  RAG: the vocabulary ends inside the last tile, columns past it
    // add nothing (an instance of its own: a uniform branch between the two costs
    // the whole tiles 5%).
    float* red = (float*)rg_smem;
    float rs[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const int m = m0 + wm * WM + i * 16 + r16;
      const int tg = m < M ? ea.tgt[m] : -1;
      float sum = 0.f;
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int n = n0 + wn * WN + j * 16 + kg * 4 + r;
          const float zc = softcap_fast(rbf(acc[j][i][r]));
          const float e = __builtin_amdgcn_exp2f(zc * 1.4426950408889634f);
          sum += !RAG || n < N ? e : 0.f;
          if (n == tg) ea.ce_tz[m] = zc;
        }
      sum += __shfl_xor(sum, 16, 64);
      sum += __shfl_xor(sum, 32, 64);
      rs[i] = sum;
    }
    __syncthreads();   // every wave is done with the last K tile
    if (wn > 0 && kg == 0) {
#pragma unroll
      for (int i = 0; i < MT; ++i) red[(wn - 1) * BM + wm * WM + i * 16 + r16] = rs[i];
    }
    __syncthreads();
    if (wn == 0 && kg == 0) {
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        const int ml = wm * WM + i * 16 + r16;
        float t = rs[i];
#pragma unroll
        for (int p = 0; p < WC - 1; ++p) t += red[p * BM + ml];
        if (m0 + ml < M) ea.ce_part[(size_t)tn * ea.ldz + m0 + ml] = t;
      }
    }
    return;
  }
  // epilogue: bf16(y) staged in LDS, then 16-byte row chunks
  if constexpr (RES && !EARLY) res_load();
  QkvRows<BM> pr;
  if constexpr (EPI == EPI_QKV) qkv_prefetch<BM>(ea, m0, M, tid, pr);
  __syncthreads();   // every wave is done with the last K tile
  bf16_t* tile = (bf16_t*)rg_smem;
#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const rg_floatx4 y = acc[j][i];
      uint2 v;
      if constexpr (EPI == EPI_RELU2) v = make_uint2(relu2_pair(y[0], y[1]), relu2_pair(y[2], y[3]));
      else v = make_uint2(pack2(y[0], y[1]), pack2(y[2], y[3]));
      *(uint2*)(tile + (wm * WM + i * 16 + r16) * CP + wn * WN + j * 16 + 4 * kg) = v;
    }
  __syncthreads();
  if constexpr (EPI == EPI_QKV) {
    qkv_tile_epilogue<BM, CP>(ea, tile, m0, n0, M, tid, pr);
  } else {
    float lam[5];
    if constexpr (RES) {
#pragma unroll
      for (int e = 0; e < 5; ++e) lam[e] = ea.lam[e];
    }
#pragma unroll
    for (int u = 0; u < NCH; ++u) {
      const int q = tid + TH * u, ml = q / CPR, c8 = (q % CPR) * 8;
      const int m = m0 + ml, n = n0 + c8;
      const uint4 y = *(const uint4*)(tile + ml * CP + c8);
      if (m >= M || n >= N) continue;
      if constexpr (RES) {
        uint4 o;
        if constexpr (EPI == EPI_RESID_ATTN) {
          o.x = mix_attn_pair(lam, xv[u].x, zv[u].x, y.x);
          o.y = mix_attn_pair(lam, xv[u].y, zv[u].y, y.y);
          o.z = mix_attn_pair(lam, xv[u].z, zv[u].z, y.z);
          o.w = mix_attn_pair(lam, xv[u].w, zv[u].w, y.w);
        } else {
          o.x = mix_mlp_pair(lam, xv[u].x, y.x);
          o.y = mix_mlp_pair(lam, xv[u].y, y.y);
          o.z = mix_mlp_pair(lam, xv[u].z, y.z);
          o.w = mix_mlp_pair(lam, xv[u].w, y.w);
        }
        *(uint4*)(ea.x + (size_t)m * ea.ldr + n) = o;
      } else if constexpr (EPI == EPI_LOGITS) {
        const size_t i = (size_t)m * ea.ldz + n;
        if (ea.z) *(uint4*)(ea.z + i) = y;
        if (ea.logits) {
          *(float4*)(ea.logits + i) = make_float4(softcap(lo_f(y.x)), softcap(hi_f(y.x)),
                                                  softcap(lo_f(y.y)), softcap(hi_f(y.y)));
          *(float4*)(ea.logits + i + 4) = make_float4(softcap(lo_f(y.z)), softcap(hi_f(y.z)),
                                                      softcap(lo_f(y.w)), softcap(hi_f(y.w)));
        }
      } else if constexpr (EPI == EPI_RELU2 && BN == 192) {
        // The tile of the large fc outputs, which the next projection reads back
        // once: past the caches.  Plain stores against these, whole calls: 16 x
        // 7680 tokens and 32 steps 44.43 / 44.21 ms, d 1536 128 x 1024 tokens and
        // 24 steps 36.19 / 36.08; prompts of 8 x 512 tokens 1413 / 1386 us, but of
        // 2 x 962 992 / 1004, 16 x 512 2261 / 2273, 32 x 512 3627 / 3637.
        __builtin_nontemporal_store(__builtin_bit_cast(rg_u32x4, y),
                                    (rg_u32x4*)(ea.out + (size_t)m * ea.ldo + n));
      } else {
        *(uint4*)(ea.out + (size_t)m * ea.ldo + n) = y;
      }
    }
  }
}

// ---- Polar Express products ---------------------------------------------------
//
// `batch` independent products of whole 128 x 128 tiles (EPI_PE_A, EPI_PE_B,
// EPI_PE_X), the same ring.  sym (PE_A, PE_B): the output is symmetric, only
// the tiles on and above the diagonal are computed and each one above it is
// also stored transposed.  The tiles of one matrix are neighbours in an XCD's
// range, so its operands (1.2 MB at 768 x 768) stay in that L2.  MuonAdam step
// over the 155M dict: 3.79 -> 3.18 ms against register-staged 128 x 128 tiles
// (k_gemm_bat; the 15 products 2.63 -> 2.0 ms), the same bits.
// PE_X (x' = a x + B x) reads x as the (K, N) operand it is: 60 us a 155M bank
// against 71 with a transposed copy written by each epilogue and read by the
// next product.
constexpr int PE_T = 128;

template <int EPI>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_pe_ring(
    const bf16_t* A, int lda, long long sA, const bf16_t* W, long long sW, int M, int N, int K,
    EpiArgs ea, long long sOut, long long sX) {
  constexpr int CPR = PE_T / 8, NCH = PE_T * CPR / 256, CP = PE_T + 8;
  extern __shared__ __attribute__((aligned(16))) unsigned char rg_smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wv >> 1, wn = wv & 1, r16 = lane & 15, kg = lane >> 4;
  const int nbm = M / PE_T, nbn = N / PE_T;
  const int per = ea.sym ? nbm * (nbm + 1) / 2 : nbm * nbn;
  const int total = gridDim.x, q8 = total >> 3, r8 = total & 7, x8 = blockIdx.x & 7;
  const int t = x8 * q8 + min(x8, r8) + (blockIdx.x >> 3);
  const int z = t / per;
  int tm = 0, tn = t - z * per;
  if (ea.sym) {
    while (tn >= nbm - tm) tn -= nbm - tm++;
    tn += tm;
  } else {
    tm = tn / nbn;
    tn -= tm * nbn;
  }
  const int m0 = tm * PE_T, n0 = tn * PE_T;
  bf16_t* out = ea.out + z * sOut;
  const bf16_t* x = ea.x + z * sX;

  float ss[4];
  rg_floatx4 acc[4][4];
  ring_product<PE_T, PE_T, 2, 2, 2, false, EPI == EPI_PE_X>(A + z * sA, lda, W + z * sW, M, N, K,
                                                            m0, n0, wv, lane, acc, ss, N);
  // chunk q = tid + 256 u of the tile: row q / CPR, columns 8 (q % CPR)
  uint4 xv[EPI == EPI_PE_A ? 1 : NCH];
  if constexpr (EPI != EPI_PE_A) {
#pragma unroll
    for (int u = 0; u < NCH; ++u) {
      const int q = tid + 256 * u;
      xv[u] = *(const uint4*)(x + (size_t)(m0 + q / CPR) * ea.ldr + n0 + (q % CPR) * 8);
    }
  }
  __syncthreads();   // every wave is done with the last K tile
  bf16_t* tile = (bf16_t*)rg_smem;
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const rg_floatx4 y = acc[j][i];
      *(uint2*)(tile + (wm * 64 + i * 16 + r16) * CP + wn * 64 + j * 16 + 4 * kg) =
          make_uint2(pack2(y[0], y[1]), pack2(y[2], y[3]));
    }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < NCH; ++u) {
    const int q = tid + 256 * u, ml = q / CPR, c8 = (q % CPR) * 8;
    uint4* sy = (uint4*)(tile + ml * CP + c8);
    uint4 o = *sy;
    if constexpr (EPI != EPI_PE_A) {
      // each eager product and sum rounded to bf16
      const uint32_t xw[4] = {xv[u].x, xv[u].y, xv[u].z, xv[u].w};
      uint32_t w[4] = {o.x, o.y, o.z, o.w};
#pragma unroll
      for (int f = 0; f < 4; ++f) {
        const uint32_t a = pack2(ea.s0 * lo_f(xw[f]), ea.s0 * hi_f(xw[f]));
        if constexpr (EPI == EPI_PE_B) w[f] = pack2(ea.s1 * lo_f(w[f]), ea.s1 * hi_f(w[f]));
        w[f] = pack2(lo_f(a) + lo_f(w[f]), hi_f(a) + hi_f(w[f]));
      }
      o = make_uint4(w[0], w[1], w[2], w[3]);
      *sy = o;   // kept for a transposed copy
    }
    if (EPI != EPI_PE_X || ea.out) *(uint4*)(out + (size_t)(m0 + ml) * ea.ldo + n0 + c8) = o;
  }
  // transposed: x'^T where PE_X is asked for it, or the mirror of a tile above
  // the diagonal
  bf16_t* dst = EPI == EPI_PE_X ? (ea.outT ? ea.outT + z * sOut : nullptr)
                                : (ea.sym && tn != tm ? out : nullptr);
  if (!dst) return;
  const int ld = EPI == EPI_PE_X ? ea.ldoT : ea.ldo;
  if constexpr (EPI != EPI_PE_A) __syncthreads();
  // a thread takes a column pair and 32 rows, 16-byte runs of each column
  const int cp = tid & 63, rb = tid >> 6;
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const int r0 = rb * 32 + 8 * g;
    uint32_t w[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) w[e] = *(const uint32_t*)(tile + (r0 + e) * CP + 2 * cp);
    uint4 c0, c1;
    c0.x = (w[0] & 0xffffu) | (w[1] << 16); c0.y = (w[2] & 0xffffu) | (w[3] << 16);
    c0.z = (w[4] & 0xffffu) | (w[5] << 16); c0.w = (w[6] & 0xffffu) | (w[7] << 16);
    c1.x = (w[0] >> 16) | (w[1] & 0xffff0000u); c1.y = (w[2] >> 16) | (w[3] & 0xffff0000u);
    c1.z = (w[4] >> 16) | (w[5] & 0xffff0000u); c1.w = (w[6] >> 16) | (w[7] & 0xffff0000u);
    bf16_t* d = dst + (size_t)(n0 + 2 * cp) * ld + m0 + r0;
    *(uint4*)d = c0;
    *(uint4*)(d + ld) = c1;
  }
}

// Whole tiles; the strides and bases of the caller (polar_express) are whole
// matrices of such tiles, 16-byte aligned.
bool pe_ring_fits(int S, int L) { return S >= PE_T && S % PE_T == 0 && L % PE_T == 0; }

hipError_t pe_ring(int epi, const bf16_t* A, int lda, long long sA, const bf16_t* W, long long sW,
                   int M, int N, int K, const EpiArgs& ea, long long sOut, long long sX, int batch,
                   hipStream_t st) {
  const int nbm = M / PE_T, nbn = N / PE_T;
  if (M % PE_T || N % PE_T || K % RG_BK || K < RG_BK || (ea.sym && M != N) ||
      (long long)nbm * nbn * batch > (1 << 30))
    return hipErrorInvalidValue;
  const dim3 grid((ea.sym ? nbm * (nbm + 1) / 2 : nbm * nbn) * batch);
  constexpr size_t lds = rg_lds_bytes<PE_T, PE_T, 2>();   // 64 KB
#define PE_CASE(E)                                                                              \
  case E:                                                                                       \
    hipLaunchKernelGGL((k_pe_ring<E>), grid, dim3(256), lds, st, A, lda, sA, W, sW, M, N, K, ea, \
                       sOut, sX);                                                               \
    return hipGetLastError();
  switch (epi) {
    PE_CASE(EPI_PE_A)
    PE_CASE(EPI_PE_B)
    PE_CASE(EPI_PE_X)
  }
#undef PE_CASE
  return hipErrorInvalidValue;
}

namespace {

template <int EPI, int BM, int BN, int NS, int WR, int WC, bool RAG = false>
hipError_t launch_ring(const bf16_t* A, int lda, const bf16_t* W, int M, int N, int K,
                       const EpiArgs& ea, hipStream_t st) {
  if (!RAG && N % BN) return hipErrorInvalidValue;
  const dim3 grid((N + BN - 1) / BN, (M + BM - 1) / BM);
  hipLaunchKernelGGL((k_gemm_ring<EPI, BM, BN, NS, WR, WC, RAG>), grid, dim3(64 * WR * WC),
                     (rg_lds_bytes<BM, BN, NS>()), st, A, lda, W, M, N, K, 4, ea);
  return hipGetLastError();
}

// dynamic LDS beyond 64 KB has to be asked for
template <int EPI, int BM, int BN, int NS, int WR, int WC, bool RAG = false>
bool ring_attr() {
  return hipFuncSetAttribute((const void*)k_gemm_ring<EPI, BM, BN, NS, WR, WC, RAG>,
                             hipFuncAttributeMaxDynamicSharedMemorySize,
                             (int)rg_lds_bytes<BM, BN, NS>()) == hipSuccess;
}
template <int EPI>
bool ring_attrs() {
  return ring_attr<EPI, 32, 64, 6, 1, 4>() && ring_attr<EPI, 64, 64, 4, 2, 2>() &&
         ring_attr<EPI, 128, 64, 3, 2, 2>() && ring_attr<EPI, 128, 128, 2, 2, 2>() &&
         ring_attr<EPI, 128, 192, 2, 2, 2>();
}

// The tiles, with the time per K tile of a work-group alone on its CU and of
// one of two that share it, and what a launch takes besides, in ns: fitted on the
// o / proj / fc shapes of d 512, 768 and 1536 (within 13% of the slopes above,
// whose epilogue is one of several).
struct RingTile {
  int bm, bn;
  int alone, shared, fixed;
};
constexpr RingTile RING_TILES[] = {
    {32, 64, 150, 145, 2800},   {64, 64, 207, 195, 2900},   {128, 64, 340, 290, 3600},
    {128, 128, 590, 470, 4600}, {128, 192, 780, 660, 5000},
    // QKV only (a 128-column tile holds whole heads).  Its epilogue costs 2 to 3 us
    // a work-group at every tile, which leaves the order of the three to the
    // products: the times of the same tiles transposed, measured as a rule with the
    // three tiles at 19 row counts from 200 to 131072 of d 128, 256, 512, 768 and
    // 1536 (2 us added to the tiles whose x a launch normalises): the fastest or
    // within 5% of it at 92 of the 95, 10% off at the worst.  64 x 128 / 128 x 128 /
    // 192 x 128, d 768: 777 rows 10.4 / 11.9 / 15.6 us, 4096 29.7 / 26.2 / 24.4,
    // 16384 101 / 75 / 77, 131072 811 / 603 / 555.
    {64, 128, 340, 290, 3600},  {192, 128, 780, 660, 5000}};
constexpr int RING_N = 5, RING_QKV_N = 7;

}  // namespace

// Whether tile t can run the epilogue on an A taken as it is (plain), or on
// either A: the qkv and fc epilogues of the small tiles exist with the rms only.
static bool ring_has(const RingTile& t, int i, int epi, bool plain) {
  if (epi == EPI_QKV ? t.bn != 128 : i >= RING_N) return false;
  if (epi == EPI_CE && t.bn < 128) return false;   // partial sums of at most V / 128 tiles
  return !(plain && ring_takes_rms(epi, t.bm, t.bn));
}

// The tile that is done first: the CU with the most work-groups takes them in
// pairs (two are resident).  Measured against every tile of o, proj and fc at 130
// .. 32768 rows of d 512, 768 and 1536: within 5% of the best one at most
// shapes, 15% at the worst (QKV: at RING_TILES).  -1 where no tile divides N (of
// any A: N is a multiple of 64, of 128 for QKV; plain qkv and fc: of 128 or 192;
// the loss takes every N).
static int ring_pick(int epi, bool plain, int M, int N, int K, long long* est_ns = nullptr) {
  static const int cus = device_cus();
  int best = -1;
  long long best_ns = 0;
  for (int i = 0; i < RING_QKV_N; ++i) {
    const RingTile& t = RING_TILES[i];
    if (!ring_has(t, i, epi, plain) || (epi != EPI_CE && N % t.bn)) continue;
    const long long wgs = (long long)((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn);
    const long long n = (wgs + cus - 1) / cus;
    const long long ns = K / RG_BK * (n / 2 * 2 * t.shared + n % 2 * t.alone) + t.fixed;
    if (best < 0 || ns < best_ns) {
      best = i;
      best_ns = ns;
    }
  }
  if (est_ns) *est_ns = best_ns;
  return best;
}

long long gemm_ring_ns(int epi, bool rms, int M, int N, int K) {
  long long ns = 0;
  return ring_pick(epi, !rms, M, N, K, &ns) < 0 ? -1 : ns;
}

int gemm_ring_tile(int epi, bool rms, int M, int N, int K) {
  const int i = ring_pick(epi, !rms, M, N, K);
  return i < 0 ? 0 : RING_TILES[i].bm << 16 | RING_TILES[i].bn;
}

// Rows of A and of the epilogue's operands in 16-byte words, whole 64-column
// tiles (the loss: any vocabulary).
bool gemm_ring_fits(int epi, const bf16_t* A, int lda, const bf16_t* W, int M, int N, int K,
                    const EpiArgs& ea) {
  if (M < 1 || N < 1 || (epi != EPI_CE && N % 64) || K < RG_BK || K % RG_BK || lda % 8 ||
      (((uintptr_t)A | (uintptr_t)W) & 15))
    return false;
  switch (epi) {
    case EPI_STORE:
    case EPI_RELU2:
      return ea.out && ea.ldo % 8 == 0 && ((uintptr_t)ea.out & 15) == 0;
    case EPI_RESID_ATTN:
      return ea.x && ea.x0 && ea.lam && ea.ldr % 8 == 0 &&
             (((uintptr_t)ea.x | (uintptr_t)ea.x0) & 15) == 0;
    case EPI_RESID_MLP:
      return ea.x && ea.lam && ea.ldr % 8 == 0 && ((uintptr_t)ea.x & 15) == 0;
    case EPI_QKV:
      return gemm_qkv_fits(M, N, K, ea);
    case EPI_CE:
      return ea.ce_part && ea.ce_tz && ea.tgt && ea.ldz >= M;
    case EPI_LOGITS:
      return !ea.amax && ea.ldz % 8 == 0 && (((uintptr_t)ea.z | (uintptr_t)ea.logits) & 15) == 0;
    default:
      return false;
  }
}

int gemm_ce_cols(int M, int N, int K) { return RING_TILES[ring_pick(EPI_CE, true, M, N, K)].bn; }

bool gemm_ring_rms(int epi, int M, int N, int K) {
  const int i = ring_pick(epi, false, M, N, K);
  return i >= 0 && ring_takes_rms(epi, RING_TILES[i].bm, RING_TILES[i].bn);
}

hipError_t gemm_ring_prepare() {
  static PerDevice limits;
  int dev = 0;
  const hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  return (hipError_t)limits.once(dev, [] {
    const bool ok = ring_attrs<EPI_STORE>() && ring_attrs<EPI_RELU2>() &&
                    ring_attrs<EPI_RESID_ATTN>() && ring_attrs<EPI_RESID_MLP>() &&
                    ring_attrs<EPI_LOGITS>() && ring_attr<EPI_CE, 128, 128, 2, 2, 2>() &&
                    ring_attr<EPI_CE, 128, 192, 2, 2, 2>() &&
                    ring_attr<EPI_CE, 128, 128, 2, 2, 2, true>() &&
                    ring_attr<EPI_CE, 128, 192, 2, 2, 2, true>() &&
                    ring_attr<EPI_QKV, 128, 128, 2, 2, 2>() &&
                    ring_attr<EPI_QKV, 64, 128, 3, 2, 2>() &&
                    ring_attr<EPI_QKV, 192, 128, 2, 2, 2>();
    return (int)(ok ? hipSuccess : hipErrorInvalidValue);
  });
}

hipError_t gemm_ring(int epi, bool rms, const bf16_t* A, int lda, const bf16_t* W, int M, int N,
                     int K, const EpiArgs& ea, hipStream_t st) {
  if (!gemm_ring_fits(epi, A, lda, W, M, N, K, ea) || (rms && !gemm_ring_rms(epi, M, N, K)))
    return hipErrorInvalidValue;
  const hipError_t e = gemm_ring_prepare();
  if (e != hipSuccess) return e;
  const int tile = ring_pick(epi, !rms, M, N, K);   // none (-1) falls through to the error
#define RING_TILE(E, T, BM, BN, NS, WR, WC) \
  case T: return launch_ring<E, BM, BN, NS, WR, WC>(A, lda, W, M, N, K, ea, st);
#define RING(E)                         \
  switch (tile) {                       \
    RING_TILE(E, 0, 32, 64, 6, 1, 4)    \
    RING_TILE(E, 1, 64, 64, 4, 2, 2)    \
    RING_TILE(E, 2, 128, 64, 3, 2, 2)   \
    RING_TILE(E, 3, 128, 128, 2, 2, 2)  \
    RING_TILE(E, 4, 128, 192, 2, 2, 2)  \
  }                                     \
  break;
  switch (epi) {
    case EPI_STORE: RING(EPI_STORE)
    case EPI_RELU2: RING(EPI_RELU2)
    case EPI_RESID_ATTN: RING(EPI_RESID_ATTN)
    case EPI_RESID_MLP: RING(EPI_RESID_MLP)
    case EPI_LOGITS: RING(EPI_LOGITS)
    case EPI_CE:
      if (tile >= 0 && N % RING_TILES[tile].bn) {
        if (tile == 3) return launch_ring<EPI_CE, 128, 128, 2, 2, 2, true>(A, lda, W, M, N, K, ea, st);
        return launch_ring<EPI_CE, 128, 192, 2, 2, 2, true>(A, lda, W, M, N, K, ea, st);
      }
      switch (tile) {
        RING_TILE(EPI_CE, 3, 128, 128, 2, 2, 2)
        RING_TILE(EPI_CE, 4, 128, 192, 2, 2, 2)
      }
      break;
    case EPI_QKV:
      switch (tile) {
        RING_TILE(EPI_QKV, 3, 128, 128, 2, 2, 2)
        RING_TILE(EPI_QKV, 5, 64, 128, 3, 2, 2)
        RING_TILE(EPI_QKV, 6, 192, 128, 2, 2, 2)
      }
  }
#undef RING
#undef RING_TILE
  return hipErrorInvalidValue;
}

}  // namespace ann
