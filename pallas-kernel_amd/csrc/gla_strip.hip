// Strip-specialised chunk sweep for gfx950 (per-channel gates; GLA forward and reverse, and the
// KDA delta rule): the same recurrences as gla_sweep_kernel (gla_sweep.hip), which cites the
// reference functions they replace.
//
// One workgroup of 8 wave64 owns one (sequence, head, 64-wide V tile; the delta rule also
// takes 16- and 32-wide tiles, one or two consumers).  Waves 0-3 (one per
// SIMD) are consumers: wave j holds the fp32 state of 16 V columns, all K rows, in MFMA
// accumulators for the whole walk, and runs every product that touches it.  Waves 4-7 are
// producers: they load the raw q / k / g / Y rows, do the gate cumsum, the exponentials and
// the bf16 hi / lo splits.  The causal D tiles are the consumers' work, except in the forward
// delta rule, where the producers compute them.  With G the in-chunk inclusive gate cumsum
// (log2 units), Gm half its last row, e = 2^Gm, X~ = q 2^(G-Gm), Z~ = k 2^(Gm-G) (reverse: X~
// and Z~ exchanged), D[p][r] = Z~_p . X~_r on the causal side:
//   T = e S,   out^T = T^T X~^T + Y^T D,   S' = e (T + Z~^T Y)
// (2^Gamma = e^2 and 2^(Gamma-Gm) = e, so one factor per channel serves both; scale is applied
// to the output forward and to D and Z~^T Y in reverse).
//
// The state never leaves the registers: the accumulator tile of a state row block holds, per
// lane, four rows of one column, and two tiles whose rows are taken as channels 8 g + 0..3
// and 8 g + 4..7 (g the lane's 16-lane group) are together one MFMA operand of eight
// consecutive channels (A of out^T, B of w S).  The row order is free, as Z~^T is read
// transposed (ds_read_b64_tr_b16) from addresses of the lane's choosing.
// Each chunk is two intervals between barriers:
//   A: consumers T^T X~^T, D(c)                 | producers Y(c), Z~(c + 1)
//      (forward delta: w S, v_new, T^T X~^T     |            D(c), Z~(c + 1))
//   B: consumers Y^T D, state update, next T    | producers X~(c + 1), cumsum of c + 2
// so the VALU staging of one chunk runs beside the matrix products of another on every SIMD.
// X~, Y and D are single planes (written in the interval that does not read them), Z~ two.
// Planes are row-major without padding, their 16-byte pieces swizzled by row (swz in strip.h).
// Delta rule (KDA): forward, Y = v_new = u - w S comes from the state operand and the staged
// planes of w 2^-Gm (against T = 2^Gm S), token-major, which is the operand layout of the
// products that follow; reverse, the state update gains - w^T dv_new, and dv_new is stored
// transposed per chunk for the WY backward.
// Why the D tiles sit with the consumers: those have the X~ fragments in registers already, and
// with the producers they cost 80 KB more of LDS reads per chunk and made interval A
// producer-bound (9,200 -> 8,900 cycles per training chunk, 8,000 -> 6,700 inference); in the
// forward delta rule the consumers carry w S instead.  The
// fp16 checkpoint goes through LDS to the producers, which store whole 128-byte rows:
// stored from the accumulators it was 64 four-byte-per-lane stores per chunk that held the
// consumers up (interval A 4,600 -> 2,700 cycles).  Producers run at raised wave priority
// where they are the longer side (interval A; in training B as well: 8,900 -> 8,100 cycles).
// fp32 checkpoints (more than 128 value columns) take the same route, 16-byte stores of 256-byte
// rows: chunk_gla forward and backward, B8 T1000 H8 K=128 V=256 bf16, 352 -> 340 us.
// Bounds: a chunk moves 64 KB per workgroup in training and 48 KB in inference, 3.4 / 2.5 us
// at the rate a large copy reaches (4.8 TB/s); measured 4.0 / 3.5 us, VALU issue (~500 per
// producer wave, ~400 per consumer wave and chunk) and LDS reads (~450 KB) next.  B8 T4096 H16
// K=V=128 bf16, one workgroup per CU: training sweeps 362 / 356 -> 255 / 255 us forward /
// reverse, inference forward 303 -> 224 us against a sweep whose eight waves each staged,
// multiplied and passed the state through LDS.  Delta rule, B4 T8192 H32 K=V=128 bf16:
// forward with checkpoints 1187 -> 800 us, without 1047 -> 680, reverse 970 -> 710 (2.7 to
// 3.5 GB per launch, 500-720 us at the copy rate); fp32, B1 T5000 H32 (64 workgroups, so
// latency alone): 756 -> 370, 289 on 16-column tiles.  There the producers keep the default
// priority in interval A.
#include <stdlib.h>

#include <atomic>
#include <type_traits>

#include "gla_sweep.h"
#include "strip.h"
#include "tops_common.h"
#include "tops_hip.h"

namespace tops {

// Phase clocks (a library built with -DTOPS_PHASE_CLOCKS only; the regular build compiles
// none of this): per wave, the shader clock (s_memtime) summed over the chunks, slots 0 work
// of interval A (producers: after the D tiles), 1 wait at its barrier, 2 work of interval B
// (consumers: after the output block; producers: after X~), 3 wait at its barrier, 4 D tiles
// (producers) or output block (consumers), 5 X~ staging (producers) or the state update;
// slot 6 the loop's s_memtime span, slot 7 its s_memrealtime (100 MHz) span.
#ifdef TOPS_PHASE_CLOCKS
constexpr bool kPhaseClocks = true;
#else
constexpr bool kPhaseClocks = false;
#endif
template <bool ON>
struct PhaseClock {
  __device__ void start() {}
  __device__ void tick(int) {}
  __device__ void finish(unsigned long long*, int) {}
};
template <>
struct PhaseClock<true> {
  uint64_t ph[6], t, t0, r0;
  __device__ void start() {
#pragma unroll
    for (int j = 0; j < 6; ++j) ph[j] = 0;
    t = t0 = __builtin_amdgcn_s_memtime();
    r0 = __builtin_amdgcn_s_memrealtime();
  }
  __device__ void tick(int j) {
    const uint64_t x = __builtin_amdgcn_s_memtime();
    ph[j] += x - t;
    t = x;
  }
  // slot: workgroup * 8 + wave; lane 0 writes (vector stores)
  __device__ void finish(unsigned long long* out, int slot) {
    const uint64_t t1 = __builtin_amdgcn_s_memtime(), r1 = __builtin_amdgcn_s_memrealtime();
    if (out == nullptr || (threadIdx.x & 63) != 0) return;
    const rsrc_t R = make_rsrc(out + (size_t)slot * 8, 64);
    const uint64_t v[8] = {ph[0], ph[1], ph[2], ph[3], ph[4], ph[5], t1 - t0, r1 - r0};
#pragma unroll
    for (int j = 0; j < 8; ++j) bst64(R, make_uint2((uint32_t)v[j], (uint32_t)(v[j] >> 32)), 8u * j, 0);
  }
};

// VAR: 1 = fp16 checkpoints of every chunk (training), 2 = no checkpoints (inference), 3 = the
// end state and the decay sums only (the state pass of sequence-parallel segments: Z~ and Y,
// no X~, no output), 0 = the rest (fp32 or paired checkpoints, channel slices).
template <typename TIn, int KP, bool REV, bool DELTA, int VAR, int BV = 64>
__global__ __launch_bounds__(64 * (BV / 16 + 4)) void gla_strip_kernel(SweepParams p) {
  constexpr int C = kChunk;
  constexpr int NC = BV / 16, NPW = 4;       // consumer waves, then producer waves
  static_assert(BV == 64 || VAR == 2, "narrow tiles: no checkpoints (their factors cover 64 columns)");
  constexpr int ES = sizeof(TIn);
  constexpr bool SIN = !In<TIn>::kExactBf16;
  constexpr bool FWD_DELTA = DELTA && !REV;
  constexpr bool REV_DELTA = DELTA && REV;
  constexpr bool SY = SIN || FWD_DELTA;      // Y carries a lo half
  constexpr bool CONS_D = !FWD_DELTA && NC == 4;        // the consumers compute the D tiles
  // reverse delta rule: Z~^T Y is taken in interval A, so Z~ and Y are single planes written
  // in B with X~ (two Z~ planes, w and the checkpoint would not fit the 160 KB)
  constexpr bool ZB = REV_DELTA;
  constexpr int KC = KP / 32;                // 32-channel blocks
  constexpr int NT = 2 * KC;                 // state tiles of a consumer
  constexpr int PL = C * KP;                 // elements of one plane
  constexpr int LY = BV + 8;
  constexpr bool CK16 = VAR == 1;
  constexpr bool CK32 = VAR == 0 && !SIN && !DELTA;    // fp32 checkpoints by the producers
  constexpr bool CKP = CK16 || CK32;
  constexpr bool ST = VAR == 3;
  // producer mapping: a wave covers QW column quads x SW row segments
  constexpr int NQ = KP / 4;
  constexpr int QW = NQ < 16 ? NQ : 16, SW = 64 / QW;
  constexpr int NCW = NQ / QW;               // waves across the columns
  constexpr int NRW = NPW / NCW;               // waves down the rows
  constexpr int RPT = C / (NRW * SW);        // rows per thread (8, 4, 2)
  typedef Words<TIn> Wd;

  __shared__ __attribute__((aligned(16))) uint16_t sX[ST ? 8 : 2 * PL];
  __shared__ __attribute__((aligned(16))) uint16_t sZ[(ZB ? 2 : 4) * PL];
  __shared__ __attribute__((aligned(16))) uint16_t sW[DELTA ? 2 * PL : 8];
  __shared__ __attribute__((aligned(16))) uint16_t sY[FWD_DELTA ? 8 : (SIN ? 2 : 1) * C * LY];
  __shared__ __attribute__((aligned(16))) uint4 sDt[ST ? 1 : 10 * 64];
  __shared__ __attribute__((aligned(16))) float sE[2 * KP];      // e of this and the next chunk
  __shared__ __attribute__((aligned(16))) float sTot[NRW * KP];  // gate totals per row wave
  // checkpoints: the state entering the chunk for the producers to store, fp32 [K][BV]; the
  // delta rule, short of LDS by its w planes, hands it over packed, fp16 [BV][K].  (fp32
  // checkpoints of the delta rule and of fp32 / fp16 inputs, whose planes leave no room, are
  // stored by the consumers, 4 bytes per lane.)
  constexpr int LS = BV + 4, LC = KP + 8;
  __shared__ __attribute__((aligned(16))) float sS[CKP && !DELTA ? KP * LS : 4];
  __shared__ __attribute__((aligned(16))) uint16_t sC[CK16 && DELTA ? BV * LC : 8];
  __shared__ uint32_t sMx[4];                // largest |S| of each wave that takes the maxima

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, lg = lane >> 4;
  const int wg = xcd_remap(blockIdx.x, gridDim.x, p.NV);
  const int vt = wg % p.NV;
  const int hh = (wg / p.NV) % p.H;
  int n = wg / (p.NV * p.H);
  auto seq_end = [&](int j) { return p.seg_end ? p.seg_end[j] : p.cu_seqlens[j + 1]; };
  if (p.cu_seqlens && p.N > 1 && p.N <= 256) {
    // varlen: longest sequence first (LPT) over the slots, ties by index
    const int slot = n;
    if (tid < p.N) {
      const int li = seq_end(tid) - p.cu_seqlens[tid];
      int rank = 0;
      for (int j = 0; j < p.N; ++j) {
        const int lj = seq_end(j) - p.cu_seqlens[j];
        rank += (lj > li) || (lj == li && j < tid);
      }
      if (rank == slot) *(int*)sTot = tid;
    }
    __syncthreads();
    n = *(const int*)sTot;
    __syncthreads();
  }
  n = __builtin_amdgcn_readfirstlane(n);
  const int H = p.H, K = p.K, V = p.V;
  const int LDK = (VAR == 0 && p.ldk > 0) ? p.ldk : K;
  const float scale = p.scale;

  int L, row0, cbase;
  if (p.cu_seqlens) {
    row0 = p.cu_seqlens[n];
    L = seq_end(n) - row0;
    cbase = p.chunk_offsets ? p.chunk_offsets[n] : 0;
  } else {
    row0 = n * p.T;
    L = p.T;
    cbase = n * cdiv(p.T, C);
  }
  const int NTs = cdiv(L, C);
  const uint32_t rowK = (uint32_t)(H * LDK), rowV = (uint32_t)(H * V);
  auto cidx = [&](int it) { return REV ? NTs - 1 - it : it; };
  // fp32 checkpoints: of every chunk or of one parity of the chunk index
  auto keeps_ckpt = [&](int c) {
    return VAR == 0 && p.ckpt && (p.ckpt_par == 0 || ((cbase + c) & 1) == p.ckpt_par - 1);
  };
  auto zbuf = [&](int it) { return sZ + (ZB ? 0 : (it & 1) * (2 * PL)); };   // Z~ of a chunk

  // row reads of a swizzled plane: piece 4 kc + lg of row l16 (+ 16 rows per block)
  int xa[KC];
#pragma unroll
  for (int kc = 0; kc < KC; ++kc) xa[kc] = l16 * KP + (((4 * kc + lg) ^ swz<KP>(l16)) << 3);

  // a causal D tile (Rc, Pc) (Rc = R, Pc = P forward; 3 - R, 3 - P reverse) to its LDS slot
  auto put_d = [&](f32x4 a, int Rc, int Pc) {
    if (Pc == Rc) {                           // the diagonal tile: keep the causal side
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const bool keep = REV ? (4 * lg + r >= l16) : (4 * lg + r <= l16);
        a[r] = keep ? a[r] : 0.f;
      }
    }
    if constexpr (REV) {
#pragma unroll
      for (int r = 0; r < 4; ++r) a[r] *= scale;
    }
    uint2 h, l;
    acc_to_bf16x4(a, h, l);
    sDt[(Rc * (Rc + 1) / 2 + Pc) * 64 + lane] = make_uint4(h.x, h.y, l.x, l.y);
  };

  if (wave >= NC) {
    // ------------------------------------------------------------------ producers
    const int pw = wave - NC;
    const int ptid = tid - 64 * NC;
    const int cq = (lane % QW) + QW * (pw % NCW);
    const int rw = pw / NCW;
    const int sl = lane / QW;                 // row segment within the wave
    const int r0 = (rw * SW + sl) * RPT, c0 = 4 * cq;
    const bool colok = c0 < K;
    const uint32_t offQ = colok ? ((uint32_t)r0 * rowK + c0) * ES : kOOB;
    const uint32_t offG = colok ? ((uint32_t)r0 * rowK + c0) * 4u : kOOB;
    int wa[RPT];                              // plane position of (row r0 + i, columns c0..)
#pragma unroll
    for (int i = 0; i < RPT; ++i)
      wa[i] = (r0 + i) * KP + (((cq >> 1) ^ swz<KP>((r0 + i) & 15)) << 3) + 4 * (cq & 1);
    const int yr = ptid / NC, ycol = 16 * (ptid % NC);
    const bool yok = yr < C;                  // (more producer threads than pieces)
    const int yv = vt * BV + ycol;
    constexpr int YP = 16 / (16 / ES);        // 16-byte pieces of a thread's 16 columns

    typename Wd::W4 rq[RPT], rk[RPT];
    uint4 rg[RPT], rwd[DELTA ? RPT : 1], ry[FWD_DELTA ? 1 : YP];
    // raw loads of one chunk (the range of each resource ends at the chunk's last valid token,
    // a chunk past the sequence has an empty range: zeros)
    struct At { size_t e0; int nval; };
    auto at = [&](int it) {
      const bool in = it < NTs;
      const int c = in ? cidx(it) : 0;
      At a;
      a.nval = in ? min(C, L - c * C) : 0;
      a.e0 = (size_t)(row0 + c * C) * H + hh;
      return a;
    };
    auto load_g = [&](int it) {
      const At a = at(it);
      const rsrc_t R = chunk_rsrc(p.g, a.e0, a.nval, (int)rowK, LDK);
#pragma unroll
      for (int i = 0; i < RPT; ++i) rg[i] = bld128(R, offG, i * rowK * 4);
    };
    auto load_rows = [&](const void* t, int it, typename Wd::W4* r) {
      const At a = at(it);
      const rsrc_t R = chunk_rsrc((const TIn*)t, a.e0, a.nval, (int)rowK, LDK);
#pragma unroll
      for (int i = 0; i < RPT; ++i) r[i] = Wd::ld4(R, offQ, i * rowK * ES);
    };
    auto load_w = [&](int it) {
      const At a = at(it);
      const rsrc_t R = chunk_rsrc(p.w, a.e0, a.nval, (int)rowK, LDK);
#pragma unroll
      for (int i = 0; i < (DELTA ? RPT : 1); ++i) rwd[i] = bld128(R, offG, i * rowK * 4);
    };
    auto load_y = [&](int it) {
      const At a = at(it);
      const rsrc_t R = chunk_rsrc((const TIn*)p.y, a.e0, a.nval, (int)rowV, V);
#pragma unroll
      for (int i = 0; i < YP; ++i) {
        const int v = yv + i * (16 / ES);      // (V % 8 == 0: a piece is inside or outside)
        ry[i] = bld128(R, yok && v < V ? ((uint32_t)yr * rowV + v) * ES : kOOB, 0);
      }
    };

    // gate cumsum of the raw chunk: thread rows, the wave's row segments on the VALU, the wave
    // totals to sTot.  In log2 units, as the kernels before and after the sweep sum it: in
    // natural units, scaled where the exponents are formed, the final state of chunk_gla was
    // 4.79e-6 off instead of 4.06e-6 and KDA's dbeta 7.5e-6 instead of 6.7e-6 at gates of -1.6 a
    // token (times unchanged; one long KDA chain, B1 T5000 H32, 536.0 -> 537.5 us)
    float G[RPT][4], pre[4];
    auto cumsum = [&]() {
      float tot[4];
#pragma unroll
      for (int i = 0; i < RPT; ++i) {
        float x[4];
        unpack4(rg[i], x);
#pragma unroll
        for (int j = 0; j < 4; ++j) G[i][j] = x[j] * kLog2e + (i > 0 ? G[i - 1][j] : 0.f);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float t = G[RPT - 1][j];
        float ex = 0.f;
        if constexpr (SW == 8) {
          const float a = dpp_row<0x128>(t);    // row_ror:8: the row's other segment
          ex = (lane & 8) ? a : 0.f;
          t += a;
        }
        const float a = lane_xor16(t, lane);
        ex += (lane & 16) ? a : 0.f;
        t += a;
        const float b = lane_xor32(t, lane);
        ex += (lane & 32) ? b : 0.f;
        pre[j] = ex;
        tot[j] = t + b;
      }
      if (sl == 0) *(float4*)(sTot + rw * KP + c0) = make_float4(tot[0], tot[1], tot[2], tot[3]);
    };
    // pm: x = G + pm is the exponent G - Gm of a row; gm2 = Gm
    float pm[4], gm2[4], dsum[4] = {0.f, 0.f, 0.f, 0.f};
    auto sums = [&](int buf) {
      float gam[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < NRW; ++s) {
        const float4 t = *(const float4*)(sTot + s * KP + c0);
        if (s < rw) { pre[0] += t.x; pre[1] += t.y; pre[2] += t.z; pre[3] += t.w; }
        gam[0] += t.x; gam[1] += t.y; gam[2] += t.z; gam[3] += t.w;
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        gm2[j] = 0.5f * gam[j];
        if constexpr (ST) dsum[j] += 2.f * gm2[j];   // (a chunk past the sequence adds zero)
        pm[j] = pre[j] - gm2[j];
      }
      if (rw == 0 && sl == 0)
        *(float4*)(sE + buf * KP + c0) =
            make_float4(fast_exp2(gm2[0]), fast_exp2(gm2[1]), fast_exp2(gm2[2]), fast_exp2(gm2[3]));
    };
    // one gated plane: rows times 2^x (up) or 2^-x
    auto put = [&](uint16_t* hi, int i, const float* x) {
      uint32_t h0, h1, l0, l1;
      split_bf16x2(x[0], x[1], h0, l0);
      split_bf16x2(x[2], x[3], h1, l1);
      *(uint2*)(hi + wa[i]) = make_uint2(h0, h1);
      *(uint2*)(hi + PL + wa[i]) = make_uint2(l0, l1);
    };
    // (the first plane of a chunk, Z~, turns the cumsum into the exponents the second reads)
    auto stage = [&](const typename Wd::W4* raw, bool up, bool first, uint16_t* hi) {
#pragma unroll
      for (int i = 0; i < RPT; ++i) {
        float v[4], x[4];
        unpack4(raw[i], v);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if (first) G[i][j] += pm[j];
          x[j] = v[j] * fast_exp2(up ? G[i][j] : -G[i][j]);
        }
        put(hi, i, x);
      }
    };
    auto stage_w = [&]() {
      float f[4] = {1.f, 1.f, 1.f, 1.f};
      if constexpr (FWD_DELTA) {
#pragma unroll
        for (int j = 0; j < 4; ++j) f[j] = fast_exp2(-gm2[j]);
      }
#pragma unroll
      for (int i = 0; i < (DELTA ? RPT : 1); ++i) {
        float v[4];
        unpack4(rwd[i], v);
        if constexpr (FWD_DELTA) {
#pragma unroll
          for (int j = 0; j < 4; ++j) v[j] *= f[j];
        }
        put(sW, i, v);
      }
    };
    auto write_y = [&]() {
      if (!yok) return;
      uint16_t* dst = sY + yr * LY + ycol;
      if constexpr (!SIN) {
#pragma unroll
        for (int i = 0; i < YP; ++i) *(uint4*)(dst + 8 * i) = ry[i];
      } else {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          float x[8];
          if constexpr (ES == 2) {
            unpack8_f16(ry[i], x);
          } else {
            unpack4(ry[2 * i], x);
            unpack4(ry[2 * i + 1], x + 4);
          }
          uint32_t h[4], l[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) split_bf16x2(x[2 * e], x[2 * e + 1], h[e], l[e]);
          *(uint4*)(dst + 8 * i) = make_uint4(h[0], h[1], h[2], h[3]);
          *(uint4*)(dst + C * LY + 8 * i) = make_uint4(l[0], l[1], l[2], l[3]);
        }
      }
    };
    // causal D tiles (Rc, P0 .. P0 + NP - 1) (Rc = R, Pc = P forward; 3 - R, 3 - P reverse),
    // the X~ row block read once
    auto dtiles = [&](auto np, int Rc, int P0, const uint16_t* z) {
      constexpr int NP = decltype(np)::value;
      const int Rt = REV ? 3 - Rc : Rc;
      f32x4 a[NP];
#pragma unroll
      for (int u = 0; u < NP; ++u) a[u] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kc = 0; kc < KC; ++kc) {
        const uint16_t* px = sX + xa[kc] + Rt * (16 * KP);
        const bf16x8 xh = lds8(px), xl = lds8(px + PL);
#pragma unroll
        for (int u = 0; u < NP; ++u) {
          const int Pt = REV ? 3 - (P0 + u) : P0 + u;
          const uint16_t* pz = z + xa[kc] + Pt * (16 * KP);
          const bf16x8 zh = lds8(pz), zl = lds8(pz + PL);
          a[u] = mma<true, true>(a[u], zh, zl, xh, xl);
        }
      }
#pragma unroll
      for (int u = 0; u < NP; ++u) put_d(a[u], Rc, P0 + u);
    };

    // checkpoint of the state entering the chunk: read in interval A (the wave maxima to sMx),
    // stored in B, 8 columns of a row per lane
    constexpr int CU = KP / 32;
    f32x4 cs[CKP && !DELTA ? 2 * CU : 1];
    auto ckpt_read = [&]() {
      if constexpr (DELTA) return;
#pragma unroll
      for (int u = 0; u < CU; ++u) {
        const float* q = sS + ((ptid >> 3) + 32 * u) * LS + 8 * (ptid & 7);
        cs[2 * u] = *(const f32x4*)q;
        cs[2 * u + 1] = *(const f32x4*)(q + 4);
      }
      if constexpr (CK16) state_absmax(cs, sMx, pw, lane);
    };
    auto ckpt_store = [&](int c) {
      if constexpr (DELTA) {
        // read transposed: lane holds columns 32 h + 8 lg + 0..7 of channel 16 cb + l16
        const rsrc_t R = make_rsrc((uint16_t*)p.ckpt + ((size_t)(cbase + c) * H + hh) * LDK * V,
                                   (long long)K * V * 2);
#pragma unroll
        for (int u = 0; u < CU; ++u) {
          const int cb = (pw * CU + u) >> 1, h = (pw * CU + u) & 1;
          const uint16_t* q = sC + (32 * h + 8 * lg + (l16 >> 2)) * LC + 16 * cb + 4 * (l16 & 3);
          const int row = 16 * cb + l16, v = vt * BV + 32 * h + 8 * lg;
          bst128(R, __builtin_bit_cast(uint4, tr2(q, q + 4 * LC)),
                 (row < K && v < V) ? ((uint32_t)row * V + v) * 2u : kOOB, 0);
        }
        return;
      }
      const size_t slot = (size_t)(cbase + c) * H + hh;
      if constexpr (CK32) {
        const rsrc_t R = make_rsrc(p.ckpt + slot * LDK * V, (long long)K * V * 4);
#pragma unroll
        for (int u = 0; u < CU; ++u) {
          const int row = (ptid >> 3) + 32 * u;
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            const int v = vt * BV + 8 * (ptid & 7) + 4 * e;
            bst128(R, __builtin_bit_cast(uint4, cs[2 * u + e]),
                   (row < K && v < V) ? ((uint32_t)row * V + v) * 4u : kOOB, 0);
          }
        }
        return;
      }
      const float sinv = ckpt_tile_scale(sMx);
      if (ptid == 0) p.ckpt_scale[slot * p.NV + vt] = 1.f / sinv;   // powers of two
      const rsrc_t R = make_rsrc((uint16_t*)p.ckpt + slot * LDK * V, (long long)K * V * 2);
      const int v = vt * BV + 8 * (ptid & 7);
#pragma unroll
      for (int u = 0; u < CU; ++u) {
        const int row = (ptid >> 3) + 32 * u;
        uint32_t w[4];
#pragma unroll
        for (int e = 0; e < 4; ++e)
          w[e] = pack_f16x2(cs[2 * u + (e >> 1)][2 * (e & 1)] * sinv, cs[2 * u + (e >> 1)][2 * (e & 1) + 1] * sinv);
        bst128(R, make_uint4(w[0], w[1], w[2], w[3]),
               (row < K && v < V) ? ((uint32_t)row * V + v) * 2u : kOOB, 0);
      }
    };

    const void* pX = REV ? p.k : p.q;         // X~ = q 2^x forward, k 2^-x reverse
    const void* pZ = REV ? p.q : p.k;
    // prologue: chunk 0 staged, the cumsum of chunk 1
    load_g(0);
    load_rows(pZ, 0, rk);
    if constexpr (!ST) load_rows(pX, 0, rq);
    if constexpr (DELTA) load_w(0);
    if constexpr (!FWD_DELTA) load_y(0);
    cumsum();
    __syncthreads();
    sums(0);
    stage(rk, REV, true, sZ);
    if constexpr (ZB) write_y();
    if constexpr (!ST) stage(rq, !REV, false, sX);
    if constexpr (FWD_DELTA) stage_w();
    load_g(1);
    if constexpr (ZB) load_y(1);
    load_rows(pZ, 1, rk);
    if constexpr (!ST) load_rows(pX, 1, rq);
    if constexpr (FWD_DELTA) load_w(1);
    __syncthreads();
    cumsum();
    load_g(2);
    __syncthreads();
    PhaseClock<kPhaseClocks> clk;
    clk.start();
    for (int it = 0; it < NTs; ++it) {
      // A: D and Y of this chunk, Z~ of the next
      __builtin_amdgcn_s_setprio(DELTA && NC == 4 ? 0 : 2);
      const uint16_t* z = zbuf(it);
      if constexpr (CONS_D) {
      } else if (pw == 0) dtiles(std::integral_constant<int, 3>{}, 3, 0, z);
      else if (pw == 1) dtiles(std::integral_constant<int, 3>{}, 2, 0, z);
      else if (pw == 3) dtiles(std::integral_constant<int, 2>{}, 1, 0, z);
      else {
        dtiles(std::integral_constant<int, 1>{}, 3, 3, z);
        dtiles(std::integral_constant<int, 1>{}, 0, 0, z);
      }
      clk.tick(4);
      const bool ck = CK16 || (CK32 && keeps_ckpt(cidx(it)));
      if (ck) ckpt_read();
      if constexpr (!FWD_DELTA && !ZB) {
        write_y();
        load_y(it + 1);
      }
      if constexpr (REV_DELTA) {
        stage_w();
        load_w(it + 1);
      }
      sums((it + 1) & 1);
      if constexpr (!ZB) {
        stage(rk, REV, true, zbuf(it + 1));
        load_rows(pZ, it + 2, rk);
      }
      clk.tick(0);
      __syncthreads();
      clk.tick(1);
      // B: X~ (and w) of the next chunk, the cumsum of the one after
      __builtin_amdgcn_s_setprio(CKP ? 2 : 0);
      if (ck) ckpt_store(cidx(it));
      if constexpr (ZB) {
        stage(rk, REV, true, sZ);
        load_rows(pZ, it + 2, rk);
        write_y();
        load_y(it + 2);
      }
      if constexpr (!ST) {
        stage(rq, !REV, false, sX);
        clk.tick(5);
        load_rows(pX, it + 2, rq);
      }
      if constexpr (FWD_DELTA) {
        stage_w();
        load_w(it + 2);
      }
      cumsum();
      load_g(it + 3);
      clk.tick(2);
      __syncthreads();
      clk.tick(3);
    }
    clk.finish(p.clocks, blockIdx.x * (NC + NPW) + wave);
    if constexpr (ST) {
      if (p.dec_fin && vt == 0 && rw == 0 && sl == 0 && colok)
        *(float4*)(p.dec_fin + (size_t)(n * H + hh) * LDK + c0) =
            make_float4(dsum[0], dsum[1], dsum[2], dsum[3]);
    }
    return;
  }

  // -------------------------------------------------------------------- consumers
  const int j = wave;
  const int vcol = vt * BV + 16 * j + l16;     // this lane's state column
  const bool vok = vcol < V;
  // transposed reads of Z~ (and w): rows 4 lg + l16 / 4 of a 16-row block, piece 4 kc + l16 % 4
  const int rr = 4 * lg + (l16 >> 2);
  int za[KC];
#pragma unroll
  for (int kc = 0; kc < KC; ++kc) za[kc] = rr * KP + (((4 * kc + (l16 & 3)) ^ swz<KP>(rr)) << 3);
  const int ya = rr * LY + 16 * j + 4 * (l16 & 3);

  // state tile (kc, b): lane holds channels 32 kc + 8 lg + 4 b + r of its column
  f32x4 S[NT], T[NT];
  const size_t s_base = (size_t)(n * H + hh) * LDK * V;
  auto s_off = [&](int t) {
    const int ch = 32 * (t >> 1) + 8 * lg + 4 * (t & 1);
    return (ch < K && vok) ? ((uint32_t)ch * V + vcol) * 4u : kOOB;
  };
  {
    const rsrc_t Rs0 = make_rsrc(p.s0 ? p.s0 + s_base : nullptr, p.s0 ? (long long)LDK * V * 4 : 0);
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) S[t][r] = __uint_as_float(bld32(Rs0, s_off(t), (uint32_t)(r * V * 4)));
  }
  __builtin_amdgcn_s_waitcnt(0);

  bf16x8 hh8[KC], hl8[KC];                     // T as an operand, hi / lo
  auto next_T = [&](int buf) {                 // T = e S of the chunk in e buffer buf
#pragma unroll
    for (int kc = 0; kc < KC; ++kc) {
      uint32_t h[4], l[4];
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const float4 e = *(const float4*)(sE + buf * KP + 32 * kc + 8 * lg + 4 * b);
        f32x4& t = T[2 * kc + b];
        const f32x4& s = S[2 * kc + b];
        t[0] = e.x * s[0]; t[1] = e.y * s[1]; t[2] = e.z * s[2]; t[3] = e.w * s[3];
        if constexpr (ST) continue;
        split_bf16x2(t[0], t[1], h[2 * b], l[2 * b]);
        split_bf16x2(t[2], t[3], h[2 * b + 1], l[2 * b + 1]);
      }
      if constexpr (ST) continue;
      hh8[kc] = __builtin_bit_cast(bf16x8, make_uint4(h[0], h[1], h[2], h[3]));
      hl8[kc] = __builtin_bit_cast(bf16x8, make_uint4(l[0], l[1], l[2], l[3]));
    }
  };
  auto store_ckpt = [&](int c) {
    if constexpr (CK16 && DELTA) {
      const float sinv = ckpt_tile_scale(sMx);
      if (tid == 0) p.ckpt_scale[((size_t)(cbase + c) * H + hh) * p.NV + vt] = 1.f / sinv;
#pragma unroll
      for (int kc = 0; kc < KC; ++kc) {
        const f32x4 &a = S[2 * kc], &b = S[2 * kc + 1];
        *(uint4*)(sC + (16 * j + l16) * LC + 32 * kc + 8 * lg) =
            make_uint4(pack_f16x2(a[0] * sinv, a[1] * sinv), pack_f16x2(a[2] * sinv, a[3] * sinv),
                       pack_f16x2(b[0] * sinv, b[1] * sinv), pack_f16x2(b[2] * sinv, b[3] * sinv));
      }
    } else if constexpr (VAR == 0 && !CK32) {
      if (!keeps_ckpt(c)) return;
      const rsrc_t R = make_rsrc(p.ckpt + ((size_t)(cbase + c) * H + hh) * LDK * V, (long long)K * V * 4);
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          bst32(R, __float_as_uint(S[t][r]), s_off(t), (uint32_t)(r * V * 4));
    }
  };
  // forward delta rule: u in the result layout of w S, loaded one chunk ahead
  float ur[FWD_DELTA ? 4 : 1][4];
  auto load_u = [&](int it) {
    const bool in = it < NTs;
    const int c = in ? cidx(it) : 0;
    const rsrc_t R = chunk_rsrc(p.u, (size_t)(row0 + c * C) * H + hh, in ? min(C, L - c * C) : 0, (int)rowV, V);
#pragma unroll
    for (int Rb = 0; Rb < (FWD_DELTA ? 4 : 1); ++Rb)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        ur[Rb][r] = __uint_as_float(bld32(
            R, vok ? ((uint32_t)(16 * Rb + 4 * lg + r) * rowV + vcol) * 4u : kOOB, 0));
  };

  auto publish_S = [&]() {                     // for the producers' checkpoint
    if constexpr (CK16 && DELTA) {
      state_absmax(S, sMx, wave, lane);
    } else if constexpr (CKP) {
      if (CK32 && !p.ckpt) return;
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          sS[(32 * (t >> 1) + 8 * lg + 4 * (t & 1) + r) * LS + 16 * j + l16] = S[t][r];
    }
  };
  publish_S();
  if constexpr (FWD_DELTA) load_u(0);
  __syncthreads();
  __syncthreads();
  next_T(0);
  __syncthreads();
  PhaseClock<kPhaseClocks> clk;
  clk.start();
  for (int it = 0; it < NTs; ++it) {
    const int c = cidx(it);
    const int t0 = c * C;
    const int nval = min(C, L - t0);
    const size_t eo = (size_t)(row0 + t0) * H + hh;

    // ---------------- A: products with X~ (and w)
    store_ckpt(c);
    bf16x8 yh[2], yl[2];                       // Y of token halves: tokens 32 q + 4 lg + 0..3, + 16
    if constexpr (FWD_DELTA) {
      // v_new = u - w S: lane holds (token 16 R + 4 lg + r, its column)
      f32x4 a[4];
#pragma unroll
      for (int Rb = 0; Rb < 4; ++Rb) a[Rb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kc = 0; kc < KC; ++kc) {
        bf16x8 wh[4], wl[4];
#pragma unroll
        for (int Rb = 0; Rb < 4; ++Rb) {
          wh[Rb] = lds8(sW + xa[kc] + Rb * (16 * KP));
          wl[Rb] = lds8(sW + PL + xa[kc] + Rb * (16 * KP));
        }
#pragma unroll
        for (int Rb = 0; Rb < 4; ++Rb) a[Rb] = mfma(wl[Rb], hh8[kc], a[Rb]);
#pragma unroll
        for (int Rb = 0; Rb < 4; ++Rb) a[Rb] = mfma(wh[Rb], hl8[kc], a[Rb]);
#pragma unroll
        for (int Rb = 0; Rb < 4; ++Rb) a[Rb] = mfma(wh[Rb], hh8[kc], a[Rb]);
      }
      const rsrc_t Rvn = chunk_rsrc(p.y32, eo, nval, (int)rowV, V);
      uint2 h[4], l[4];
#pragma unroll
      for (int Rb = 0; Rb < 4; ++Rb) {
#pragma unroll
        for (int r = 0; r < 4; ++r) a[Rb][r] = ur[Rb][r] - a[Rb][r];
        if (VAR != 2 || p.y32) {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            bst32(Rvn, __float_as_uint(a[Rb][r]),
                  vok ? ((uint32_t)(16 * Rb + 4 * lg + r) * rowV + vcol) * 4u : kOOB, 0);
        }
        acc_to_bf16x4(a[Rb], h[Rb], l[Rb]);
      }
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        yh[q] = cat44(h[2 * q], h[2 * q + 1]);
        yl[q] = cat44(l[2 * q], l[2 * q + 1]);
      }
      load_u(it + 1);
    }
    // out^T tiles: lane holds columns 4 lg + r of the strip, token 16 R + l16 (reverse delta
    // rule: dv_new, lane holds tokens 16 R + 4 lg + r of its column)
    f32x4 o[4];
#pragma unroll
    for (int Rb = 0; Rb < 4; ++Rb) o[Rb] = f32x4{0.f, 0.f, 0.f, 0.f};
    // and the wave's share of the D tiles, on the X~ fragments in registers: row block j of Z~
    // with up to three of its tiles; wave 3 also takes tile (R 3, P 0)
    const uint16_t* zc = zbuf(it);
    auto interval_a = [&](auto jc) {
      constexpr int J = decltype(jc)::value;   // Pc of the wave's row block (-1: no D tiles)
      constexpr int ND = J < 0 ? 0 : (J == 3 ? 2 : (J == 2 ? 2 : 3));
      f32x4 a[ND > 0 ? ND : 1];
#pragma unroll
      for (int u = 0; u < ND; ++u) a[u] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kc = 0; kc < KC; ++kc) {
        bf16x8 xh[4], xl[4], zh[2], zl[2];
#pragma unroll
        for (int Rb = 0; Rb < 4; ++Rb) {
          xh[Rb] = lds8(sX + xa[kc] + Rb * (16 * KP));
          xl[Rb] = lds8(sX + PL + xa[kc] + Rb * (16 * KP));
        }
        if constexpr (ND > 0) {
#pragma unroll
          for (int u = 0; u < (J == 3 ? 2 : 1); ++u) {
            const int Pc = u == 0 ? J : 0;
            const uint16_t* pz = zc + xa[kc] + (REV ? 3 - Pc : Pc) * (16 * KP);
            zh[u] = lds8(pz);
            zl[u] = lds8(pz + PL);
          }
        }
#pragma unroll
        for (int Rb = 0; Rb < 4; ++Rb) o[Rb] = REV_DELTA ? mfma(xl[Rb], hh8[kc], o[Rb]) : mfma(hh8[kc], xl[Rb], o[Rb]);
#pragma unroll
        for (int Rb = 0; Rb < 4; ++Rb) o[Rb] = REV_DELTA ? mfma(xh[Rb], hl8[kc], o[Rb]) : mfma(hl8[kc], xh[Rb], o[Rb]);
#pragma unroll
        for (int Rb = 0; Rb < 4; ++Rb) o[Rb] = REV_DELTA ? mfma(xh[Rb], hh8[kc], o[Rb]) : mfma(hh8[kc], xh[Rb], o[Rb]);
#pragma unroll
        for (int u = 0; u < ND; ++u) {
          const int Rc = J == 3 ? 3 : J + u, b = J == 3 ? u : 0;
          const int Rt = REV ? 3 - Rc : Rc;
          a[u] = mma<true, true>(a[u], zh[b], zl[b], xh[Rt], xl[Rt]);
        }
      }
#pragma unroll
      for (int u = 0; u < ND; ++u) put_d(a[u], J == 3 ? 3 : J + u, J == 3 && u == 1 ? 0 : J);
    };
    auto read_y = [&]() {
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const uint16_t* py = sY + ya + 32 * q * LY;
        yh[q] = tr2(py, py + 16 * LY);
        yl[q] = yh[q];
        if constexpr (SY) yl[q] = tr2(py + C * LY, py + C * LY + 16 * LY);
      }
    };
    // Z~^T Y of state tile t, added to a
    auto zty = [&](int t, f32x4 a) {
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const uint16_t* pz = zc + za[t >> 1] + 4 * (t & 1) + 32 * q * KP;
        const bf16x8 zh = tr2(pz, pz + 16 * KP), zl = tr2(pz + PL, pz + PL + 16 * KP);
        a = mma<true, SY>(a, zh, zl, yh[q], yl[q]);
      }
      return a;
    };
    f32x4 dz[ZB ? NT : 1];
    if constexpr (ZB) {
      read_y();
#pragma unroll
      for (int t = 0; t < NT; ++t) dz[t] = zty(t, f32x4{0.f, 0.f, 0.f, 0.f});
    }
    if constexpr (ST) {
    } else if constexpr (!CONS_D) interval_a(std::integral_constant<int, -1>{});
    else if (j == 0) interval_a(std::integral_constant<int, 0>{});
    else if (j == 1) interval_a(std::integral_constant<int, 1>{});
    else if (j == 2) interval_a(std::integral_constant<int, 2>{});
    else interval_a(std::integral_constant<int, 3>{});
    clk.tick(0);
    __syncthreads();
    clk.tick(1);

    // ---------------- B: intra-chunk products, state update
    if constexpr (!FWD_DELTA && !ZB) read_y();
    if constexpr (!ST) {
    uint4 d[10];
#pragma unroll
    for (int t = 0; t < 10; ++t) d[t] = sDt[t * 64 + lane];
#pragma unroll
    for (int Rb = 0; Rb < 4; ++Rb) {
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int P0 = 2 * q, P1 = 2 * q + 1;
        const bool l0 = REV ? (P0 >= Rb) : (P0 <= Rb), l1 = REV ? (P1 >= Rb) : (P1 <= Rb);
        if (!l0 && !l1) continue;
        const int Rc = REV ? 3 - Rb : Rb;
        const uint4 z4 = make_uint4(0u, 0u, 0u, 0u);
        const uint4 a = l0 ? d[Rc * (Rc + 1) / 2 + (REV ? 3 - P0 : P0)] : z4;
        const uint4 b = l1 ? d[Rc * (Rc + 1) / 2 + (REV ? 3 - P1 : P1)] : z4;
        const bf16x8 dh = cat44(make_uint2(a.x, a.y), make_uint2(b.x, b.y));
        const bf16x8 dl = cat44(make_uint2(a.z, a.w), make_uint2(b.z, b.w));
        o[Rb] = REV_DELTA ? mma<true, SY>(o[Rb], dh, dl, yh[q], yl[q])
                          : mma<SY, true>(o[Rb], yh[q], yl[q], dh, dl);
      }
    }
    }
    bf16x8 vh[2], vl[2];                       // reverse delta rule: dv_new as an operand
    if constexpr (REV_DELTA) {
      const rsrc_t Rd = make_rsrc(p.y32 + ((size_t)(cbase + c) * H + hh) * V * C, (long long)V * C * 4);
      uint2 h[4], l[4];
#pragma unroll
      for (int Rb = 0; Rb < 4; ++Rb) {
        bst128(Rd, __builtin_bit_cast(uint4, o[Rb]),
               vok ? ((uint32_t)vcol * C + 16 * Rb + 4 * lg) * 4u : kOOB, 0);
        acc_to_bf16x4(o[Rb], h[Rb], l[Rb]);
      }
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        vh[q] = cat44(h[2 * q], h[2 * q + 1]);
        vl[q] = cat44(l[2 * q], l[2 * q + 1]);
      }
    } else if constexpr (!ST) {
      const rsrc_t Ro = chunk_rsrc((const TIn*)p.out, eo, nval, (int)rowV, V);
      const int v0 = vt * BV + 16 * j + 4 * lg;
#pragma unroll
      for (int Rb = 0; Rb < 4; ++Rb) {
        if constexpr (!REV) {
#pragma unroll
          for (int r = 0; r < 4; ++r) o[Rb][r] *= scale;
        }
        const uint32_t el = (uint32_t)(16 * Rb + l16) * rowV + v0;
        if (VAR != 0 || p.acc_mode == 0) {
          Wd::st4(Ro, o[Rb], v0 < V ? el * ES : kOOB, 0);
        } else {
          // channel slices: the fp32 sum of the slices' outputs
          const rsrc_t Ra = chunk_rsrc(p.acc32, eo, nval, (int)rowV, V);
          acc_slice_t<TIn>(Ro, Ra, o[Rb], v0 < V ? el * 4u : kOOB, v0 < V ? el * ES : kOOB, 0, p.acc_mode);
        }
      }
    }
    clk.tick(4);
    // state update: T += Z~^T Y (forward), S = e T
#pragma unroll
    for (int kc = 0; kc < KC; ++kc) {
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const int t = 2 * kc + b;
        f32x4 a;
        if constexpr (ZB) a = dz[t];
        else a = zty(t, REV ? f32x4{0.f, 0.f, 0.f, 0.f} : T[t]);
        f32x4 w = {0.f, 0.f, 0.f, 0.f};
        if constexpr (REV_DELTA) {
#pragma unroll
          for (int q = 0; q < 2; ++q) {
            const uint16_t* pww = sW + za[kc] + 4 * b + 32 * q * KP;
            const bf16x8 wh = tr2(pww, pww + 16 * KP), wl = tr2(pww + PL, pww + PL + 16 * KP);
            w = mma<true, true>(w, wh, wl, vh[q], vl[q]);
          }
        }
        const float4 e = *(const float4*)(sE + (it & 1) * KP + 32 * kc + 8 * lg + 4 * b);
        const float ev[4] = {e.x, e.y, e.z, e.w};
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float x = REV ? ev[r] * (T[t][r] + scale * a[r]) : ev[r] * a[r];
          if constexpr (REV_DELTA) x -= w[r];
          S[t][r] = x;
        }
      }
    }
    clk.tick(5);
    publish_S();
    next_T((it + 1) & 1);
    clk.tick(2);
    __syncthreads();
    clk.tick(3);
  }
  clk.finish(p.clocks, blockIdx.x * (NC + NPW) + wave);

  if (p.s_fin) {
    const rsrc_t Rsf = make_rsrc(p.s_fin + s_base, (long long)LDK * V * 4);
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) bst32(Rsf, __float_as_uint(S[t][r]), s_off(t), (uint32_t)(r * V * 4));
  }
}

// Whether launch_gla_sweep routes a call to this kernel: per-channel gates without the gate
// shift of the reverse-time recurrence, any input type.  TOPS_SWEEP_SERIAL=1 in the
// environment keeps bf16 calls on gla_sweep_kernel (comparisons), except those that write fp16
// checkpoints, which only this kernel does for per-channel gates; gla_sweep_kernel has no such
// instances of the other types.
bool gla_strip_eligible(const SweepParams& p, bool bf16) {
  if (p.gate_mode != kGateK || p.gshift) return false;
  if (p.ckpt16 || !bf16) return true;
  const char* e = getenv("TOPS_SWEEP_SERIAL");
  return !(e && e[0] == '1');
}

// Compute units of the current device (kept per device; 256 where it cannot be asked).
static int device_cus() {
  static std::atomic<int> known[64];
  int dev = 0, n = 0;
  if (hipGetDevice(&dev) == hipSuccess && dev >= 0 && dev < 64 &&
      (n = known[dev].load(std::memory_order_relaxed)) > 0)
    return n;
  if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) {
    (void)hipGetLastError();
    return 256;
  }
  if (dev >= 0 && dev < 64) known[dev].store(n, std::memory_order_relaxed);
  return n;
}

template <typename TIn, bool REV, bool DELTA>
hipError_t launch_gla_strip(const SweepParams& p, hipStream_t s) {
  const int kp = p.K <= 32 ? 32 : (p.K <= 64 ? 64 : 128);
  const bool plain = !p.acc_mode && !p.ldk;
  if (p.ckpt16 && (!plain || p.ckpt_par || !p.ckpt || !p.ckpt_scale)) return hipErrorInvalidValue;
  const int var = p.ckpt16 ? 1 : ((plain && !p.ckpt) ? 2 : 0);
  dim3 grid(p.NV * p.H * p.N);
  if constexpr (DELTA && !REV) {
    // Few heads and sequences leave CUs idle and the sweep is one long chain: the narrowest
    // value tile whose workgroups are still one round on the device's CUs, the staging repeated
    // but each consumer alone with its LDS reads.  chunk_kda forward without checkpoints, B1
    // T2048 K=V=128 bf16 by heads, tiles of 16 / 32 / 64 columns: H4 137 / 142 / 161 us, H32
    // (256 workgroups of 16) 165 / 170 / 187, H33 294 / 180 / 200, H64 (256 of 32) 324 / 213 /
    // 231, H65 463 / 347 / 245; fp32 and K, V of 64 order the same way on the same lines.  (The
    // per-channel-gate sweeps, whose consumers share the D tiles, gain nothing: 27 us at B1 T512
    // H4 against 30.)
    const long long cus = device_cus();
    const long long wgs = (long long)p.H * p.N;
    const int bv = (var != 2 || wgs * p.NV > cus / 2) ? 64 : (wgs * ((p.V + 15) / 16) <= cus ? 16 : 32);
    if (bv < 64 && wgs * ((p.V + bv - 1) / bv) <= cus) {
      SweepParams q = p;
      q.NV = (p.V + bv - 1) / bv;
      const dim3 gn((unsigned)(q.NV * wgs)), bn(64 * (bv / 16 + 4));
#define TOPS_NARROW(KPV) \
  if (bv == 16) hipLaunchKernelGGL((gla_strip_kernel<TIn, KPV, REV, DELTA, 2, 16>), gn, bn, 0, s, q); \
  else hipLaunchKernelGGL((gla_strip_kernel<TIn, KPV, REV, DELTA, 2, 32>), gn, bn, 0, s, q)
      if (kp == 32) { TOPS_NARROW(32); }
      else if (kp == 64) { TOPS_NARROW(64); }
      else { TOPS_NARROW(128); }
#undef TOPS_NARROW
      return hipGetLastError();
    }
  }
#define TOPS_STRIP(KPV, VARV) \
  hipLaunchKernelGGL((gla_strip_kernel<TIn, KPV, REV, DELTA, VARV>), grid, dim3(512), 0, s, p)
#define TOPS_STRIP_K(KPV) \
  if (var == 1) { \
    if constexpr (std::is_same<TIn, uint16_t>::value) TOPS_STRIP(KPV, 1); \
    else return hipErrorInvalidValue; \
  } else if (var == 2) { \
    /* (the KDA backward always keeps dS) */ \
    if constexpr (!(DELTA && REV)) TOPS_STRIP(KPV, 2); \
    else return hipErrorInvalidValue; \
  } else TOPS_STRIP(KPV, 0)
  if (kp == 32) { TOPS_STRIP_K(32); }
  else if (kp == 64) { TOPS_STRIP_K(64); }
  else { TOPS_STRIP_K(128); }
#undef TOPS_STRIP_K
#undef TOPS_STRIP
  return hipGetLastError();
}

template <typename TIn, bool REV>
hipError_t launch_gla_strip_state(const SweepParams& p, hipStream_t s) {
  const int kp = p.K <= 32 ? 32 : (p.K <= 64 ? 64 : 128);
  dim3 grid(p.NV * p.H * p.N);
  if (kp == 32) hipLaunchKernelGGL((gla_strip_kernel<TIn, 32, REV, false, 3>), grid, dim3(512), 0, s, p);
  else if (kp == 64) hipLaunchKernelGGL((gla_strip_kernel<TIn, 64, REV, false, 3>), grid, dim3(512), 0, s, p);
  else hipLaunchKernelGGL((gla_strip_kernel<TIn, 128, REV, false, 3>), grid, dim3(512), 0, s, p);
  return hipGetLastError();
}

#define TOPS_STRIP_STATE(T) \
  template hipError_t launch_gla_strip_state<T, false>(const SweepParams&, hipStream_t); \
  template hipError_t launch_gla_strip_state<T, true>(const SweepParams&, hipStream_t);
TOPS_STRIP_STATE(uint16_t)
TOPS_STRIP_STATE(float)
TOPS_STRIP_STATE(_Float16)
#undef TOPS_STRIP_STATE

template hipError_t launch_gla_strip<uint16_t, false, true>(const SweepParams&, hipStream_t);
template hipError_t launch_gla_strip<float, false, true>(const SweepParams&, hipStream_t);
template hipError_t launch_gla_strip<uint16_t, true, true>(const SweepParams&, hipStream_t);
template hipError_t launch_gla_strip<float, true, true>(const SweepParams&, hipStream_t);
template hipError_t launch_gla_strip<uint16_t, false, false>(const SweepParams&, hipStream_t);
template hipError_t launch_gla_strip<uint16_t, true, false>(const SweepParams&, hipStream_t);
template hipError_t launch_gla_strip<float, false, false>(const SweepParams&, hipStream_t);
template hipError_t launch_gla_strip<float, true, false>(const SweepParams&, hipStream_t);
template hipError_t launch_gla_strip<_Float16, false, false>(const SweepParams&, hipStream_t);
template hipError_t launch_gla_strip<_Float16, true, false>(const SweepParams&, hipStream_t);

#ifdef TOPS_PHASE_CLOCKS
// Instrumented build only (libtops_pipe_clocks.so, pallas-kernel_amd/phase_clocks.py): one
// strip sweep over B fixed-length sequences of bf16 q, k, y (v forward, dO reverse) and
// fp32 per-channel log gates g [B, T, H, K]; out [B, T, H, V] bf16; fp16 checkpoints when
// ckpt16 / ckpt_scale are given (the training instance), none otherwise (inference); the
// phase clocks of every wave into clocks [B * H * ceil(V / 64), 8, 8].
extern "C" int tops_pipe_phase_clocks(const void* q, const void* k, const float* g, const void* y,
                                      void* out, void* ckpt16, float* ckpt_scale,
                                      unsigned long long* clocks, int B, int T, int H, int K,
                                      int V, int rev, float scale, void* stream) {
  if (!q || !k || !g || !y || !out || !clocks || (!ckpt16) != (!ckpt_scale) || B <= 0 || T <= 0 ||
      H <= 0 || K <= 0 || K > 128 || V <= 0 || K % 4 || V % 8)
    return (int)hipErrorInvalidValue;
  SweepParams p{};
  p.q = q; p.k = k; p.g = g; p.y = y; p.out = out;
  p.ckpt = (float*)ckpt16;
  p.ckpt16 = ckpt16 != nullptr;
  p.ckpt_scale = ckpt_scale;
  p.B = B; p.T = T; p.H = H; p.K = K; p.V = V; p.N = B; p.NV = (V + 63) / 64;
  p.scale = scale;
  p.gate_mode = kGateK;
  p.clocks = clocks;
  const hipError_t e = rev ? launch_gla_strip<uint16_t, true, false>(p, (hipStream_t)stream)
                           : launch_gla_strip<uint16_t, false, false>(p, (hipStream_t)stream);
  return (int)e;
}
#endif

}  // namespace tops
