// Strip-specialised chunk sweep for one log-gate per token (simple GLA: g [B,T,H], or a
// constant g_gamma [H]; bf16 inputs), forward and reverse: the recurrences of gla_sweep_kernel
// (gla_sweep.hip), which cites the reference functions they replace, in the wave roles of
// gla_strip.hip.
//
// Waves 0-3 hold the fp32 state of 16 V columns each in MFMA accumulators and run the
// products; waves 4-7 move q, k and Y into LDS and scan the gate.  With G the in-chunk
// inclusive gate cumsum (log2 units) and Gamma its last entry, (X, Z, Y) = (q, k, v) forward
// and (k, q, dO) reverse:
//   out_r = fx_r X_r S + sum_p D[p][r] Y_p,   S' = 2^Gamma S + sum_p Z_p (fz_p Y_p)^T
//   forward: fx_r = scale 2^G_r,       fz_p = 2^(Gamma - G_p),  D = scale 2^(G_r - G_p) Z_p.X_r, p <= r
//   reverse: fx_r = 2^(Gamma - G_r),   fz_p = scale 2^G_p,      D = scale 2^(G_p - G_r) Z_p.X_r, p >= r
// The gate is one factor per token, so q, k and Y enter their products as read (exact bf16):
// the state, D and fz Y are split into bf16 hi + lo, two products each.  The factors come
// from per-chunk tables one producer wave writes.  Each chunk is two intervals:
//   A: consumers X S, D tiles        | producers Z(c + 1), Y(c)
//   B: consumers Y^T D, state update | producers X(c + 1), gate tables of c + 1, checkpoint
// Bound: HBM (48 KB per workgroup and chunk in training, 2.5 us at the copy rate; 3.3 us
// measured).  Packed T16384 (8 sequences) H32 K=V=128 bf16: training sweeps 405 / 408 ->
// 231 / 220 us forward / reverse, state passes 30 -> 19 us, against the serial sweep with the
// gate moved onto the value side (one workgroup per CU, three barriers, 6.1 us per chunk), on
// the segments of that time; on balanced segments (SegPlan.balance) the sweeps take 196 / 187
// us and the state passes 25.5.  Of the matrix cores' cycles the sweeps use a fifth.
#include <type_traits>

#include "gla_sweep.h"
#include "strip.h"
#include "tops_common.h"
#include "tops_hip.h"

namespace tops {

// VAR as in gla_strip.hip: 1 = fp16 checkpoints of every chunk, 2 = none, 3 = the end state
// and the decay sums only, 0 = fp32 or paired checkpoints, channel slices.
template <int KP, bool REV, int VAR>
__global__ __launch_bounds__(512) void gla_strip_s_kernel(SweepParams p) {
  constexpr int C = kChunk, BV = 64;
  constexpr bool CK16 = VAR == 1, ST = VAR == 3;
  constexpr int KC = KP / 32;                // 32-channel blocks
  constexpr int NT = 2 * KC;                 // state tiles of a consumer
  constexpr int PL = C * KP;                 // elements of one plane
  constexpr int LY = BV + 8, LS = BV + 4;
  constexpr int NP = KP / 32;                // 16-byte pieces of a plane per producer thread
  constexpr int PR = KP / 8;                 // 16-byte pieces of a plane row

  __shared__ __attribute__((aligned(16))) uint16_t sX[ST ? 8 : PL];
  __shared__ __attribute__((aligned(16))) uint16_t sZ[2 * PL];
  __shared__ __attribute__((aligned(16))) uint16_t sY[C * LY];
  __shared__ __attribute__((aligned(16))) uint4 sDt[ST ? 1 : 10 * 64];
  __shared__ __attribute__((aligned(16))) float sG[2][C], sFx[2][C], sFz[2][C];
  __shared__ __attribute__((aligned(16))) float sS[CK16 ? KP * LS : 4];
  __shared__ uint32_t sMx[4];
  __shared__ int sN;

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
      if (rank == slot) sN = tid;
    }
    __syncthreads();
    n = sN;
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

  if (wave >= 4) {
    // ------------------------------------------------------------------ producers
    const int pw = wave - 4;
    const int ptid = tid - 256;
    // a chunk past the sequence has an empty range: zeros
    struct At { size_t e0; int nval; };
    auto at = [&](int it) {
      const bool in = it < NTs;
      const int c = in ? cidx(it) : 0;
      At a;
      a.nval = in ? min(C, L - c * C) : 0;
      a.e0 = (size_t)(row0 + c * C) * H + hh;
      return a;
    };
    // plane pieces of this thread: piece ptid + 256 u, row-major
    uint32_t go[NP];
    int wa[NP];
#pragma unroll
    for (int u = 0; u < NP; ++u) {
      const int row = (ptid + 256 * u) / PR, pc = (ptid + 256 * u) % PR;
      go[u] = 8 * pc < K ? ((uint32_t)row * rowK + 8 * pc) * 2u : kOOB;
      wa[u] = row * KP + ((pc ^ swz<KP>(row & 15)) << 3);
    }
    uint4 rx[NP], rz[NP], ry[2];
    auto load = [&](const void* t, int it, uint4* r) {
      const At a = at(it);
      const rsrc_t R = chunk_rsrc((const uint16_t*)t, a.e0, a.nval, (int)rowK, LDK);
#pragma unroll
      for (int u = 0; u < NP; ++u) r[u] = bld128(R, go[u], 0);
    };
    const int yr = ptid >> 2, ycol = 16 * (ptid & 3), yv = vt * BV + ycol;
    auto load_y = [&](int it) {
      const At a = at(it);
      const rsrc_t R = chunk_rsrc((const uint16_t*)p.y, a.e0, a.nval, (int)rowV, V);
#pragma unroll
      for (int i = 0; i < 2; ++i)              // (V % 8 == 0: a piece is inside or outside)
        ry[i] = bld128(R, yv + 8 * i < V ? ((uint32_t)yr * rowV + yv + 8 * i) * 2u : kOOB, 0);
    };
    auto put = [&](uint16_t* dst, const uint4* r) {
#pragma unroll
      for (int u = 0; u < NP; ++u) *(uint4*)(dst + wa[u]) = r[u];
    };
    auto write_y = [&]() {
#pragma unroll
      for (int i = 0; i < 2; ++i) *(uint4*)(sY + yr * LY + ycol + 8 * i) = ry[i];
    };
    // gate tables of one chunk (first producer wave, lane = token): the inclusive scan over
    // the 64 lanes on the VALU (DPP rows of 16, then the row totals)
    float rgate = 0.f, dsum = 0.f;
    const float gam = p.gate_mode == kGateGamma ? p.g[hh] : 0.f;
    auto load_g = [&](int it) {
      if (pw != 0) return;
      const At a = at(it);
      if (p.gate_mode == kGateS) {
        const rsrc_t R = chunk_rsrc(p.g, a.e0, a.nval, H, 1);
        rgate = __uint_as_float(bld32(R, (uint32_t)lane * H * 4u, 0));
      } else {
        rgate = lane < a.nval ? gam : 0.f;
      }
    };
    auto tables = [&](int buf) {
      if (pw != 0) return;
      float x = rgate * kLog2e;
      x += dpp_row<0x111>(x);                  // row_shr 1, 2, 4, 8: scan of each 16-lane row
      x += dpp_row<0x112>(x);
      x += dpp_row<0x114>(x);
      x += dpp_row<0x118>(x);
      const float t0 = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(x), 15));
      const float t1 = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(x), 31));
      const float t2 = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(x), 47));
      x += lg >= 1 ? t0 : 0.f;
      x += lg >= 2 ? t1 : 0.f;
      x += lg >= 3 ? t2 : 0.f;
      const float tot = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(x), 63));
      const float a = fast_exp2(x), b = fast_exp2(tot - x);
      sG[buf][lane] = x;
      sFx[buf][lane] = REV ? b : scale * a;
      sFz[buf][lane] = REV ? scale * a : b;
      if constexpr (ST) dsum += tot;
    };
    // checkpoint of the state entering the chunk: read in interval A, stored in B
    f32x4 cs[CK16 ? 2 * NP : 1];
    auto ckpt_read = [&]() {
#pragma unroll
      for (int u = 0; u < NP; ++u) {
        const float* q = sS + ((ptid >> 3) + 32 * u) * LS + 8 * (ptid & 7);
        cs[2 * u] = *(const f32x4*)q;
        cs[2 * u + 1] = *(const f32x4*)(q + 4);
      }
      state_absmax(cs, sMx, pw, lane);
    };
    auto ckpt_store = [&](int c) {
      const float sinv = ckpt_tile_scale(sMx);
      const size_t slot = (size_t)(cbase + c) * H + hh;
      if (ptid == 0) p.ckpt_scale[slot * p.NV + vt] = 1.f / sinv;   // powers of two
      const rsrc_t R = make_rsrc((uint16_t*)p.ckpt + slot * LDK * V, (long long)K * V * 2);
      const int v = vt * BV + 8 * (ptid & 7);
#pragma unroll
      for (int u = 0; u < NP; ++u) {
        const int row = (ptid >> 3) + 32 * u;
        uint32_t w[4];
#pragma unroll
        for (int e = 0; e < 4; ++e)
          w[e] = pack_f16x2(cs[2 * u + (e >> 1)][2 * (e & 1)] * sinv, cs[2 * u + (e >> 1)][2 * (e & 1) + 1] * sinv);
        bst128(R, make_uint4(w[0], w[1], w[2], w[3]),
               (row < K && v < V) ? ((uint32_t)row * V + v) * 2u : kOOB, 0);
      }
    };

    const void* pX = REV ? p.k : p.q;
    const void* pZ = REV ? p.q : p.k;
    load_g(0);
    load(pZ, 0, rz);
    if constexpr (!ST) load(pX, 0, rx);
    load_y(0);
    tables(0);
    load_g(1);
    put(sZ, rz);
    load(pZ, 1, rz);
    if constexpr (!ST) {
      put(sX, rx);
      load(pX, 1, rx);
    }
    __syncthreads();
    for (int it = 0; it < NTs; ++it) {
      // A: Y of this chunk, Z of the next
      if constexpr (CK16) ckpt_read();
      write_y();
      load_y(it + 1);
      put(sZ + ((it + 1) & 1) * PL, rz);
      load(pZ, it + 2, rz);
      __syncthreads();
      // B: X and the gate tables of the next chunk
      if constexpr (CK16) ckpt_store(cidx(it));
      if constexpr (!ST) {
        put(sX, rx);
        load(pX, it + 2, rx);
      }
      tables((it + 1) & 1);
      load_g(it + 2);
      __syncthreads();
    }
    if constexpr (ST) {
      // (tables of one chunk past the sequence added a zero)
      if (p.dec_fin && vt == 0 && pw == 0)
        for (int kr = lane; kr < K; kr += 64) p.dec_fin[(size_t)(n * H + hh) * LDK + kr] = dsum;
    }
    return;
  }

  // -------------------------------------------------------------------- consumers
  const int j = wave;
  const int vcol = vt * BV + 16 * j + l16;     // this lane's state column
  const bool vok = vcol < V;
  int xa[KC], za[KC];                          // as gla_strip.hip: row reads, transposed reads
  const int rr = 4 * lg + (l16 >> 2);
#pragma unroll
  for (int kc = 0; kc < KC; ++kc) {
    xa[kc] = l16 * KP + (((4 * kc + lg) ^ swz<KP>(l16)) << 3);
    za[kc] = rr * KP + (((4 * kc + (l16 & 3)) ^ swz<KP>(rr)) << 3);
  }
  const int ya = rr * LY + 16 * j + 4 * (l16 & 3);

  // state tile t = 2 kc + b: lane holds channels 32 kc + 8 lg + 4 b + r of its column
  f32x4 S[NT];
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
  bf16x8 hh8[KC], hl8[KC];                     // S as an operand, hi / lo
  auto split_S = [&]() {
    if constexpr (ST) return;
#pragma unroll
    for (int kc = 0; kc < KC; ++kc) {
      uint2 h0, l0, h1, l1;
      acc_to_bf16x4(S[2 * kc], h0, l0);
      acc_to_bf16x4(S[2 * kc + 1], h1, l1);
      hh8[kc] = cat44(h0, h1);
      hl8[kc] = cat44(l0, l1);
    }
  };
  auto publish_S = [&]() {                     // for the producers' checkpoint
    if constexpr (CK16) {
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          sS[(32 * (t >> 1) + 8 * lg + 4 * (t & 1) + r) * LS + 16 * j + l16] = S[t][r];
    }
  };
  publish_S();
  split_S();
  __syncthreads();
  for (int it = 0; it < NTs; ++it) {
    const int c = cidx(it);
    const int t0 = c * C;
    const int nval = min(C, L - t0);
    const int buf = it & 1;
    const uint16_t* zc = sZ + buf * PL;
    const size_t eo = (size_t)(row0 + t0) * H + hh;

    // ---------------- A: X S (lane: columns 4 lg + r of the strip, token 16 R + l16), D tiles
    if constexpr (VAR == 0) {
      if (p.ckpt && (p.ckpt_par == 0 || ((cbase + c) & 1) == p.ckpt_par - 1)) {
        const rsrc_t R = make_rsrc(p.ckpt + ((size_t)(cbase + c) * H + hh) * LDK * V, (long long)K * V * 4);
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            bst32(R, __float_as_uint(S[t][r]), s_off(t), (uint32_t)(r * V * 4));
      }
    }
    f32x4 o[4];
#pragma unroll
    for (int Rb = 0; Rb < 4; ++Rb) o[Rb] = f32x4{0.f, 0.f, 0.f, 0.f};
    // wave j: row block j of Z with up to three of its causal tiles (Rc, Pc) (Rc = R, Pc = P
    // forward; 3 - R, 3 - P reverse), wave 3 also tile (3, 0), on the X fragments in registers
    auto interval_a = [&](auto jc) {
      constexpr int J = decltype(jc)::value;
      constexpr int ND = J >= 2 ? 2 : 3;
      f32x4 a[ND];
#pragma unroll
      for (int u = 0; u < ND; ++u) a[u] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kc = 0; kc < KC; ++kc) {
        bf16x8 x[4], z[2];
#pragma unroll
        for (int Rb = 0; Rb < 4; ++Rb) x[Rb] = lds8(sX + xa[kc] + Rb * (16 * KP));
#pragma unroll
        for (int u = 0; u < (J == 3 ? 2 : 1); ++u) {
          const int Pc = u == 0 ? J : 0;
          z[u] = lds8(zc + xa[kc] + (REV ? 3 - Pc : Pc) * (16 * KP));
        }
#pragma unroll
        for (int Rb = 0; Rb < 4; ++Rb) o[Rb] = mfma(hl8[kc], x[Rb], o[Rb]);
#pragma unroll
        for (int Rb = 0; Rb < 4; ++Rb) o[Rb] = mfma(hh8[kc], x[Rb], o[Rb]);
#pragma unroll
        for (int u = 0; u < ND; ++u) {
          const int Rc = J == 3 ? 3 : J + u;
          a[u] = mfma(z[J == 3 ? u : 0], x[REV ? 3 - Rc : Rc], a[u]);
        }
      }
#pragma unroll
      for (int u = 0; u < ND; ++u) {
        const int Rc = J == 3 ? 3 : J + u, Pc = J == 3 && u == 1 ? 0 : J;
        const int Rt = REV ? 3 - Rc : Rc, Pt = REV ? 3 - Pc : Pc;
        const float gr = sG[buf][16 * Rt + l16];
        const float4 g4 = *(const float4*)(&sG[buf][16 * Pt + 4 * lg]);
        const float gp[4] = {g4.x, g4.y, g4.z, g4.w};
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          // (a select, not a product: the exponent of a masked entry may overflow)
          const bool keep = Pc < Rc || (REV ? (4 * lg + r >= l16) : (4 * lg + r <= l16));
          const float f = scale * fast_exp2(REV ? gp[r] - gr : gr - gp[r]);
          a[u][r] = keep ? a[u][r] * f : 0.f;
        }
        uint2 h, l;
        acc_to_bf16x4(a[u], h, l);
        sDt[(Rc * (Rc + 1) / 2 + Pc) * 64 + lane] = make_uint4(h.x, h.y, l.x, l.y);
      }
    };
    if constexpr (!ST) {
      if (j == 0) interval_a(std::integral_constant<int, 0>{});
      else if (j == 1) interval_a(std::integral_constant<int, 1>{});
      else if (j == 2) interval_a(std::integral_constant<int, 2>{});
      else interval_a(std::integral_constant<int, 3>{});
    }
    __syncthreads();

    // ---------------- B: intra-chunk products, state update
    bf16x8 y[2], vh[2], vl[2];                 // Y, and fz Y hi / lo: tokens 32 q + 4 lg + 0..3, + 16
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const uint16_t* py = sY + ya + 32 * q * LY;
      y[q] = tr2(py, py + 16 * LY);
      const float4 f0 = *(const float4*)(&sFz[buf][32 * q + 4 * lg]);
      const float4 f1 = *(const float4*)(&sFz[buf][32 * q + 16 + 4 * lg]);
      const uint4 w = __builtin_bit_cast(uint4, y[q]);
      float v[8];
      unpack4(make_uint2(w.x, w.y), v);
      unpack4(make_uint2(w.z, w.w), v + 4);
      f32x4 a = {v[0] * f0.x, v[1] * f0.y, v[2] * f0.z, v[3] * f0.w};
      f32x4 b = {v[4] * f1.x, v[5] * f1.y, v[6] * f1.z, v[7] * f1.w};
      uint2 h0, l0, h1, l1;
      acc_to_bf16x4(a, h0, l0);
      acc_to_bf16x4(b, h1, l1);
      vh[q] = cat44(h0, h1);
      vl[q] = cat44(l0, l1);
    }
    if constexpr (!ST) {
      uint4 d[10];
#pragma unroll
      for (int t = 0; t < 10; ++t) d[t] = sDt[t * 64 + lane];
      const rsrc_t Ro = chunk_rsrc((const uint16_t*)p.out, eo, nval, (int)rowV, V);
      const int v0 = vt * BV + 16 * j + 4 * lg;
#pragma unroll
      for (int Rb = 0; Rb < 4; ++Rb) {
        const float fx = sFx[buf][16 * Rb + l16];
#pragma unroll
        for (int r = 0; r < 4; ++r) o[Rb][r] *= fx;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const int P0 = 2 * q, P1 = 2 * q + 1;
          const bool l0 = REV ? (P0 >= Rb) : (P0 <= Rb), l1 = REV ? (P1 >= Rb) : (P1 <= Rb);
          if (!l0 && !l1) continue;
          const int Rc = REV ? 3 - Rb : Rb;
          const uint4 z4 = make_uint4(0u, 0u, 0u, 0u);
          const uint4 a = l0 ? d[Rc * (Rc + 1) / 2 + (REV ? 3 - P0 : P0)] : z4;
          const uint4 b = l1 ? d[Rc * (Rc + 1) / 2 + (REV ? 3 - P1 : P1)] : z4;
          o[Rb] = mfma(y[q], cat44(make_uint2(a.z, a.w), make_uint2(b.z, b.w)), o[Rb]);
          o[Rb] = mfma(y[q], cat44(make_uint2(a.x, a.y), make_uint2(b.x, b.y)), o[Rb]);
        }
        const uint32_t el = (uint32_t)(16 * Rb + l16) * rowV + v0;
        if (VAR != 0 || p.acc_mode == 0) {
          Words<uint16_t>::st4(Ro, o[Rb], v0 < V ? el * 2u : kOOB, 0);
        } else {
          // channel slices: the fp32 sum of the slices' outputs
          const rsrc_t Ra = chunk_rsrc(p.acc32, eo, nval, (int)rowV, V);
          acc_slice_t<uint16_t>(Ro, Ra, o[Rb], v0 < V ? el * 4u : kOOB, v0 < V ? el * 2u : kOOB, 0,
                                p.acc_mode);
        }
      }
    }
    const float dec = fast_exp2(sG[buf][C - 1]);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      f32x4 a;
#pragma unroll
      for (int r = 0; r < 4; ++r) a[r] = dec * S[t][r];
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const uint16_t* pz = zc + za[t >> 1] + 4 * (t & 1) + 32 * q * KP;
        const bf16x8 z = tr2(pz, pz + 16 * KP);
        a = mfma(z, vl[q], a);
        a = mfma(z, vh[q], a);
      }
      S[t] = a;
    }
    publish_S();
    split_S();
    __syncthreads();
  }

  if (p.s_fin) {
    const rsrc_t Rsf = make_rsrc(p.s_fin + s_base, (long long)LDK * V * 4);
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) bst32(Rsf, __float_as_uint(S[t][r]), s_off(t), (uint32_t)(r * V * 4));
  }
}

bool gla_strip_s_eligible(const SweepParams& p) {
  return (p.gate_mode == kGateS || p.gate_mode == kGateGamma) && !p.gshift;
}

template <bool REV>
hipError_t launch_gla_strip_s(const SweepParams& p, bool state_only, hipStream_t s) {
  const int kp = p.K <= 32 ? 32 : (p.K <= 64 ? 64 : 128);
  const bool plain = !p.acc_mode && !p.ldk;
  if (p.ckpt16 && (!plain || p.ckpt_par || !p.ckpt || !p.ckpt_scale)) return hipErrorInvalidValue;
  const int var = state_only ? 3 : (p.ckpt16 ? 1 : ((plain && !p.ckpt) ? 2 : 0));
  dim3 grid(p.NV * p.H * p.N);
#define TOPS_STRIP(KPV, VARV) \
  hipLaunchKernelGGL((gla_strip_s_kernel<KPV, REV, VARV>), grid, dim3(512), 0, s, p)
#define TOPS_STRIP_K(KPV) \
  switch (var) { \
    case 0: TOPS_STRIP(KPV, 0); break; \
    case 1: TOPS_STRIP(KPV, 1); break; \
    case 2: TOPS_STRIP(KPV, 2); break; \
    default: TOPS_STRIP(KPV, 3); \
  }
  if (kp == 32) { TOPS_STRIP_K(32) }
  else if (kp == 64) { TOPS_STRIP_K(64) }
  else { TOPS_STRIP_K(128) }
#undef TOPS_STRIP_K
#undef TOPS_STRIP
  return hipGetLastError();
}

template hipError_t launch_gla_strip_s<false>(const SweepParams&, bool, hipStream_t);
template hipError_t launch_gla_strip_s<true>(const SweepParams&, bool, hipStream_t);

}  // namespace tops
