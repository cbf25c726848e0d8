// Projection kernels: the dense contractions around the attention core.
//
//   forward : [Z | V] = X [W_phi | W_V]  with the soft-hypercube epilogue
//             (reference: packages/morphottention/csrc/cuda/sm120/project.cuh:16-47,
//              attention.cu:105-111; here computed once per token instead of once
//              per (query tile, key tile) pair)
//   backward: dZ = dphi * phi (1 - phi) with
//               dphi = gate_q dq + gate_k dk + gate_q gate_k dcb
//             (reference K side: project.cuh:49-101; the Q side, which the
//              reference drops, by symmetry),
//             dX = [dZ | dV] [W_phi | W_V]^T,  [dW_phi | dW_V] = X^T [dZ | dV],
//             gate gradients as deterministic fp32 column sums.
#include "common.h"
#include "gemm.h"
#include "internal.h"

namespace morpho {

// ---------------------------------------------------------------- weights^T
// wt = [W_phi | W_V]^T (rows in the projection's column order) for the
// forward projection and wcat = [W_phi | W_V]
// (one row-major matrix) for dX. 64 x 64 tiles with 16-byte loads and
// stores: each thread reads two 8-column pieces of W rows (and writes them to
// wcat), and writes two 8-row pieces of wt rows gathered from the LDS tile.
// HM and D are multiples of 8, so no piece straddles W_phi / W_V or a matrix
// edge.
__global__ __launch_bounds__(256) void transpose_weights_kernel(const f16* __restrict__ W_phi,
                                                                const f16* __restrict__ W_V, f16* __restrict__ wt,
                                                                f16* __restrict__ wcat, Dims dm) {
  __shared__ __align__(16) f16 tile[64][72];  // [d][n]
  const int D = dm.D, HM = dm.HM;
  const int n0 = blockIdx.x * 64, d0 = blockIdx.y * 64, NC = HM + D;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int v = threadIdx.x + 256 * i;
    const int dd = v >> 3, nn = (v & 7) * 8;
    const int dg = d0 + dd, ng = n0 + nn;
    f16x8 x = {};
    if (dg < D && ng < NC) {
      x = ng < HM ? *reinterpret_cast<const f16x8*>(W_phi + (int64_t)dg * HM + ng)
                  : *reinterpret_cast<const f16x8*>(W_V + (int64_t)dg * D + (ng - HM));
      *reinterpret_cast<f16x8*>(wcat + (int64_t)dg * NC + ng) = x;
    }
    *reinterpret_cast<f16x8*>(&tile[dd][nn]) = x;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int v = threadIdx.x + 256 * i;
    const int nn = v >> 3, dd = (v & 7) * 8;
    const int dg = d0 + dd, ng = n0 + nn;
    if (dg < D && ng < NC) {
      f16x8 y;
#pragma unroll
      for (int e = 0; e < 8; ++e) y[e] = tile[dd + e][nn];
      *reinterpret_cast<f16x8*>(wt + (int64_t)proj_row(dm, ng) * D + dg) = y;
    }
  }
}

hipError_t launch_transpose_weights(const Dims& d, const f16* W_phi, const f16* W_V, f16* wt, f16* wcat,
                                    hipStream_t s) {
  dim3 grid((d.HM + d.D + 63) / 64, (d.D + 63) / 64);
  MORPHO_KLAUNCH(transpose_weights_kernel, grid, dim3(256), 0, s, W_phi, W_V, wt, wcat, d);
  return hipGetLastError();
}

// ---------------------------------------------------------------- projection forward
// [Z | V] = X [W_phi | W_V] on BM x BN tiles: 256 x 320 when 320 divides the
// H*M + D columns (e.g. 1280 at B4 N4096 D1024 H16 m16, which makes the grid
// exactly one round of 256 tiles), 256 x 256 otherwise, and 128 x 128 when
// the large tiles would leave most CUs idle (few tokens: B8 N1024 D512 H8 m16
// has 64 large tiles, 320 small ones); between them 128 x 256, where half the
// tile halves the loss of the last round (choose_proj_tiles). The 128 x 128 and 128 x
// 160 tiles run two to a CU with two stages each; with four stages, one to a
// CU, they gained 1 us or lost up to 9 (B64 N128 D1024 H16 m16 31 -> 40).
//
// Epilogue: the values leave straight from the accumulators (lane swaps
// assemble 16-byte stores), the codes through LDS, and no wave waits for
// another's values. What bounds it is the burst of its stores (B4 N4096 D1024
// H16 m16: 97 MB at the end of one round of tiles) and, for code that runs
// once per tile, instruction fetch: the value part is unrolled over a wave's
// column blocks and loses 6 us there if each block carries its own slow paths.
// proj_fwd in us, with 64-row slabs of the whole tile through LDS in fp32 (two of
// the eight waves writing at a time) and this epilogue: B64 N197 D768 H12 m64 142
// and 80, B3 N1500 D1024 H8 m32 42.7 and 23.8 (both mostly from the padded rows,
// fill_sizes), B64 N128 D1024 H16 m16 40.0 and 31.0, B64 N1024 D768 H12 m64 256
// and 246, B4 N4096 D1024 H16 m16 55.4 and 56.0.
template <int BM, int BN, int STAGES>
using ProjGemm = Gemm<BM, BN, 4, true, true, 64, STAGES>;

// e4m3 byte(s) of V_lo * 2^kVloExp, clamped to the format's range (e4m3 has
// no infinity: an overflowing conversion gives NaN) and rounded toward zero:
// the stored remainder is never larger than V - V_hi, so V_hi + remainder
// rounds back to V_hi in fp16 (a single key's output is then exactly V_hi,
// the value the backward's dP = dO V_hi^T sees).
// The conversion with stochastic rounding adds the given random bits below
// the last kept mantissa bit and truncates; with zero random bits it is the
// truncation of the magnitude, i.e. rounding toward zero, in one instruction
// (bit-identical, over every 7th float bit pattern of both signs, to the
// nearest conversion stepped one code toward zero where that overshot).
__device__ __forceinline__ float vlo_scaled(float r) { return fminf(fmaxf(r * (float)(1 << kVloExp), -448.f), 448.f); }
// the codes of four remainders, byte k of the dword = r[k]
__device__ __forceinline__ unsigned vlo_pack4(const float (&r)[4]) {
  int w = __builtin_amdgcn_cvt_sr_fp8_f32(vlo_scaled(r[0]), 0, 0, 0);
  w = __builtin_amdgcn_cvt_sr_fp8_f32(vlo_scaled(r[1]), 0, w, 1);
  w = __builtin_amdgcn_cvt_sr_fp8_f32(vlo_scaled(r[2]), 0, w, 2);
  return (unsigned)__builtin_amdgcn_cvt_sr_fp8_f32(vlo_scaled(r[3]), 0, w, 3);
}
// v_permlane16_swap: the odd 16-lane rows of a change places with the even
// ones of b (a' = a0 b0 a2 b2, b' = a1 b1 a3 b3).
__device__ __forceinline__ void swap16(unsigned& a, unsigned& b) {
  const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}

// Lanes 8..15 of each 16-lane row of a change places with lanes 0..7 of b.
__device__ __forceinline__ void swap8(unsigned& a, unsigned& b, bool upper) {
  const unsigned send = upper ? a : b;
  const unsigned got = (unsigned)__builtin_amdgcn_mov_dpp((int)send, 0x128 /* row_ror:8 */, 0xf, 0xf, false);
  a = upper ? got : a;
  b = upper ? b : got;
}

// Memory row (token) of a row of the projection's row space: batch rows of NR
// rows, the last NR - N of which repeat the batch row's last token.
struct TokenRows {
  int NR, N;
  __device__ __forceinline__ int operator()(int r) const {
    const int b = r / NR;
    return b * N + min(r - b * NR, N - 1);
  }
};

// GEN: a cube projection other than the sigmoid, or the masked diagonal (the
// variants take the projection from d.proj and the exact row maximum)
template <int M, int DV, int BM, int BN, int STAGES, bool GEN>
__global__ __launch_bounds__(kGemmThreads) void proj_fwd_kernel(const f16* __restrict__ X,
                                                               const f16* __restrict__ gate_q,
                                                               const f16* __restrict__ gate_k, Dims d, ProjBuffers p) {
  using G = ProjGemm<BM, BN, STAGES>;
  static_assert(64 * (BN + 4) * 4 + BN * 4 <= G::kLdsBytes, "a pass of 64 code rows and the gates must fit the LDS");
  static_assert(G::WTM == 16 * G::FI && G::FI % 2 == 0 && G::WTM * 4 == BM, "four wave rows of whole block pairs");
  __shared__ __align__(16) char smem[G::kLdsBytes];
  constexpr int CW = 2 * M + 8;

  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = w / G::WN, wn = w % G::WN;
  const int NC = d.HM + d.D;
  const int TR = (int)d.TR;
  int tm, tn;
  if (!gemm_tile_map(blockIdx.x, (TR + BM - 1) / BM, (NC + BN - 1) / BN, tm, tn)) return;
  const int n0 = tn * BN, m0 = tm * BM;
  f32x4 acc[G::FI][G::FJ];
  G::run(X, d.D, p.wt, d.D, TR, NC, m0, n0, 0, d.D, smem, acc, TokenRows{d.NR, d.N});

  // Code columns of the tile: ncode, contiguous in W_phi from code0. Those of
  // this wave come first in its columns: ncw of them, from place cw of the
  // tile's; its value columns are W_V's from vw on.
  const int gpt = d.PCPT > 0 ? BN / d.PGW : 1, col0w = G::WTN * wn;
  const int ncode = d.PCPT > 0 ? gpt * d.PCPT : max(0, min(BN, d.HM - n0)), code0 = d.PCPT > 0 ? tn * ncode : n0;
  const int ncw = gpt == 2 ? d.PCPT : min(max(ncode - col0w, 0), G::WTN), cw = gpt == 2 ? wn * d.PCPT : col0w;
  const int vw = gpt == 2 ? (2 * tn + wn) * d.PVPT
                          : max(col0w - ncode, 0) + (d.PCPT > 0 ? tn * d.PVPT : max(n0 - d.HM, 0));
  const int nvw = min(G::WTN, NC - n0 - col0w);  // columns of this wave up to NC (the last tile of the natural order)
  static_assert(G::WN == 2, "half-tile groups are the two wave columns");
  const int lrow = lane >> 4, lcol = lane & 15;
  // ---- values, straight from the accumulators: vt[bh][dd][n] = V_hi, and the
  // remainder V - V_hi as e4m3 in vlo's tile-major, key-permuted rows. A lane
  // holds 4 consecutive tokens of one column per 16-row block. Swapping 16-lane
  // rows between two blocks leaves it 8 consecutive tokens of one of them (a
  // 16-byte piece of vt, 8 bytes of vlo); with four blocks, swapping 8-lane
  // halves between the two pairs then puts all 64 tokens of a column into one
  // store instruction (8 columns x 128 bytes of vt).
  if (ncode < BN) {
    constexpr int NP2 = G::FI / 2;  // block pairs
    static_assert(NP2 == 1 || NP2 == 2, "wave rows of two or four blocks");
    const bool upper = NP2 == 2 && (lane & 8) != 0;
    // This lane's 8 tokens start at row tb, position n of batch row b (tb % 8
    // == 0 and NR % 8 == 0, so they share the batch row and land on 8
    // consecutive bytes of a vlo row; those past its last token hold zero). In
    // piece q of a 16-column block they are those of column c0 + 8 q.
    const int tb = m0 + G::WTM * wm + (upper ? 32 : 0) + 16 * (lrow & 1) + 8 * (lrow >> 1);
    const int b = tb / d.NR, n = tb - b * d.NR, live = d.N - n;
    const int c0 = NP2 == 2 ? lcol & 7 : lcol;
    f16* const dst0 = p.vt + ((int64_t)b * d.D + c0) * d.NP + n;
    uint8_t* const low0 = p.vlo + (int64_t)b * d.D * d.NP + ((int64_t)(n / 64) * DV + c0) * 64 + vlo_pos(n % 64);
    unsigned mh[4], ml[2];  // the live tokens' halves and bytes
#pragma unroll
    for (int e = 0; e < 4; ++e) mh[e] = live >= 2 * e + 2 ? ~0u : live == 2 * e + 1 ? 0xffffu : 0u;
#pragma unroll
    for (int e = 0; e < 2; ++e)
      ml[e] = live >= 4 * e + 4 ? ~0u : live <= 4 * e ? 0u : ~0u >> (32 - 8 * (live - 4 * e));
#pragma unroll
    for (int j = 0; j < G::FJ; ++j) {
      if (16 * j < ncw || 16 * j >= nvw) continue;  // uniform, like everything up to the lane's column
      const int vcol = vw + 16 * j - ncw;
      unsigned hi[NP2][4], lo[NP2][2];  // [pair][dword]: 8 tokens after the swap
#pragma unroll
      for (int ip = 0; ip < NP2; ++ip) {
#pragma unroll
        for (int ii = 0; ii < 2; ++ii) {
          float vl[4];
          f16x4 vh;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            float x = acc[2 * ip + ii][j][r];
            asm("" : "+v"(x));  // one evaluation for V_hi and the remainder
            vh[r] = (f16)x;
            vl[r] = x - (float)vh[r];
          }
          const uint2 u = __builtin_bit_cast(uint2, vh);
          hi[ip][2 * ii] = u.x;
          hi[ip][2 * ii + 1] = u.y;
          lo[ip][ii] = vlo_pack4(vl);
        }
        swap16(hi[ip][0], hi[ip][2]);
        swap16(hi[ip][1], hi[ip][3]);
        swap16(lo[ip][0], lo[ip][1]);
      }
      if constexpr (NP2 == 2) {
#pragma unroll
        for (int e = 0; e < 4; ++e) swap8(hi[0][e], hi[1][e], upper);
#pragma unroll
        for (int e = 0; e < 2; ++e) swap8(lo[0][e], lo[1][e], upper);
      }
      f16* const dst = dst0 + (int64_t)vcol * d.NP;
      uint8_t* const low = low0 + (int64_t)(vcol / DV) * DV * d.NP + vcol % DV * 64;
      if (tb < TR) {
#pragma unroll
        for (int q = 0; q < NP2; ++q) {
          *reinterpret_cast<uint4*>(dst + (int64_t)8 * q * d.NP) =
              make_uint4(hi[q][0] & mh[0], hi[q][1] & mh[1], hi[q][2] & mh[2], hi[q][3] & mh[3]);
          *reinterpret_cast<uint2*>(low + 512 * q) = make_uint2(lo[q][0] & ml[0], lo[q][1] & ml[1]);
        }
      }
    }
    // the batch row's last group also clears its columns up to NP
    if (tb < TR && live <= 8 && n + 8 < d.NP) {
#pragma unroll 1
      for (int j = 0; j < G::FJ; ++j) {
        if (16 * j < ncw || 16 * j >= nvw) continue;
        const int vcol = vw + 16 * j - ncw;
#pragma unroll 1
        for (int q = 0; q < NP2; ++q) {
          f16* const dst = dst0 + (int64_t)(vcol + 8 * q) * d.NP;
          uint8_t* const low = low0 + (int64_t)(vcol / DV) * DV * d.NP + (vcol % DV + 8 * q) * 64;
#pragma unroll 1
          for (int z = 8; n + z < d.NP; z += 8) {  // n and n + z share the 64-key tile
            *reinterpret_cast<f16x8*>(dst + z) = f16x8{};
            *reinterpret_cast<uint2*>(low + (vlo_pos((n + z) % 64) - vlo_pos(n % 64))) = make_uint2(0u, 0u);
          }
        }
      }
    }
  }
  if (ncode == 0) return;

  // ---- codes, through LDS: passes of 16 KB rows per wave row, 64 KB rows in
  // all (KB of the waves' 16-row blocks, as many as the main loop's LDS
  // holds), so that all the waves write and read in every pass.
  const int SS = ncode + 4;  // row stride (floats): 16-byte rows, the accumulator stores on 64 distinct banks
  float* gtab = reinterpret_cast<float*>(smem);  // gate products G = gq gk of the code columns
  float* stage = gtab + BN;
  int lk = G::FI >= 4 ? 2 : G::FI >= 2 ? 1 : 0;  // log2 of the blocks per pass
  while (lk > 0 && BN * 4 + (64 << lk) * SS * 4 > G::kLdsBytes) --lk;
  const float c1 = 2.0f * d.scale * kLog2e;
  for (int lc = tid; lc < ncode; lc += kGemmThreads) {
    gtab[lc] = (float)gate_q[code0 + lc] * (float)gate_k[code0 + lc];  // code0 + lc = h M + c
  }
  for (int pass = 0; pass < G::FI >> lk; ++pass) {
    if (pass > 0) __syncthreads();  // the previous pass has been consumed
#pragma unroll
    for (int i = 0; i < G::FI; ++i) {
      if (i >> lk != pass) continue;  // uniform
      float* dst = stage + (64 * (i - (pass << lk)) + 16 * wm + 4 * lrow) * SS + cw + lcol;
#pragma unroll
      for (int j = 0; j < G::FJ; ++j)
        if (16 * j < ncw) {  // uniform
#pragma unroll
          for (int r = 0; r < 4; ++r) dst[r * SS + 16 * j] = acc[i][j][r];
        }
    }
    __syncthreads();
    // one (token, head, 8-code chunk) per thread; the M / 8 chunks of a
    // (token, head) sit on consecutive lanes, which meet in xor shuffles for
    // the row sums (a head's M columns are contiguous in both column orders).
    // One thread per (token, head) had left 3/4 of the workgroup idle at m = 64.
    constexpr int kChunks = M / 8;
    static_assert(kGemmThreads % kChunks == 0, "a (token, head) never straddles two passes");
    const int lrows = 6 + lk;  // log2 of the pass's rows
    for (int idx = tid; idx < (ncode / 8) << lrows; idx += kGemmThreads) {  // rows x heads x (M / 8 chunks)
      const int j = idx % kChunks, item = idx / kChunks;
      const int hh = item >> lrows, r = item & ((1 << lrows) - 1);
      const int t = m0 + G::WTM * ((r & 63) >> 4) + 16 * ((pass << lk) + (r >> 6)) + (r & 15);
      const int h = code0 / M + hh;
      const int b = t / d.NR, n = t - b * d.NR;
      const bool active = t < TR && n < d.N;  // the same for every chunk of the item
      const int64_t bhn = (int64_t)(b * d.H + h) * d.N + n;
      const int c8 = 8 * j;
      float sumb = 0.f, tii = 0.f, U = 0.f;
      if (active) {
        const float* zp = stage + r * SS + hh * M + c8;
        const float4 za = *reinterpret_cast<const float4*>(zp), zb = *reinterpret_cast<const float4*>(zp + 4);
        const float z[8] = {za.x, za.y, za.z, za.w, zb.x, zb.y, zb.z, zb.w};
        const float4 ga = *reinterpret_cast<const float4*>(gtab + hh * M + c8);
        const float4 gb = *reinterpret_cast<const float4*>(gtab + hh * M + c8 + 4);
        const float g8[8] = {ga.x, ga.y, ga.z, ga.w, gb.x, gb.y, gb.z, gb.w};
        f16x8 phh, phl, kch, kcl;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float phi = GEN ? cube_project(z[e], d.proj) : sigmoidf_(z[e]);
          const float G = g8[e];
          const float wgt = d.scale * G;
          const float cg = c1 * G;
          f16 a, bb;
          if (GEN) {  // HardTanh01's clamped fma could convert to fp16 in one rounding
            split_exact(phi, a, bb);
            phh[e] = a;
            phl[e] = bb;
          } else {  // a quotient: nothing to fuse the conversion with
            phh[e] = (f16)phi;
            phl[e] = (f16)(phi - (float)phh[e]);
          }
          // kc = cg phi: lo is the exact product minus hi, so hi + lo carries
          // kc to ~2^-22 however hi was rounded, provided lo and the stored
          // hi are one value. The conversion (f16)(cg phi) may otherwise be
          // selected twice, as one rounding of the exact product
          // (v_fma_mixlo_f16) for the fma and as a rounding of the fp32
          // product (v_cvt_pk_f16_f32) for the store, and at an fp16 rounding
          // tie the two differ by an ulp (about 1 code in 16k); the opaque
          // copy makes hi a single value.
          f16 hi = (f16)(cg * phi);
          asm("" : "+v"(hi));
          kch[e] = hi;
          kcl[e] = (f16)__builtin_fmaf(cg, phi, -(float)hi);
          sumb += wgt * phi;
          tii += wgt * phi * (2.f * phi - 1.f);
          U += fmaxf(0.f, wgt * (2.f * phi - 1.f));
        }
        // rows: [phi_hi | aug | phi_lo] and [kc_hi | aug | kc_lo]
        f16* qrow = p.qa + bhn * CW;
        f16* krow = p.ka + bhn * CW;
        *reinterpret_cast<f16x8*>(qrow + c8) = phh;
        *reinterpret_cast<f16x8*>(qrow + M + 8 + c8) = phl;
        *reinterpret_cast<f16x8*>(krow + c8) = kch;
        *reinterpret_cast<f16x8*>(krow + M + 8 + c8) = kcl;
      }
#pragma unroll
      for (int sh = 1; sh < kChunks; sh <<= 1) {  // the item's lanes are all active or all idle
        sumb += __shfl_xor(sumb, sh);
        tii += __shfl_xor(tii, sh);
        U += __shfl_xor(U, sh);
      }
      if (!active || j != 0) continue;
      // base-2 quantities: token bias b = -log2e * sum_c w_c phi_c; self score
      // t_ii and the upper bound U of any score in this query's row (without
      // the row constant, which cancels in the softmax). U bounds the row only
      // for phi in [0, 1], and R >= U - 15 keeps the row's largest weight
      // representable only while the diagonal term is in the row: the
      // identity projection and the masked diagonal take the exact two-pass
      // maximum (an infinite gap).
      const float bias = -kLog2e * sumb;
      const float t_ii = kLog2e * tii;
      const float Ub = kLog2e * U;
      const float R = fmaxf(t_ii, Ub - 15.f);
      const float gap = (GEN && (d.proj == kProjIdentity || d.mask_diag)) ? kFltMax : Ub - t_ii;
      f16 rh, rl, bh_, bl_;
      split_hi_lo(-R, rh, rl);
      split_hi_lo(bias, bh_, bl_);
      const f16 one = (f16)1.f, zero = (f16)0.f;
      *reinterpret_cast<f16x8*>(p.qa + bhn * CW + M) = f16x8{one, one, rh, rl, zero, zero, zero, zero};
      *reinterpret_cast<f16x8*>(p.ka + bhn * CW + M) = f16x8{bh_, bl_, one, one, zero, zero, zero, zero};
      p.tstat[bhn] = make_float4(bias, R, gap, t_ii);
    }
  }
}

template <int M, int DV>
static hipError_t launch_proj_fwd_t(const Dims& d, const f16* X, const f16* gq, const f16* gk, const ProjBuffers& p,
                                    hipStream_t s) {
  const int NC = d.HM + d.D;
  const bool gen = d.proj != kProjSigmoid || d.mask_diag;
#define MORPHO_PROJ_LAUNCH(BM_, BN_, ST_)                                                                      \
  do {                                                                                                         \
    const dim3 g(gemm_tile_grid((int)((d.TR + BM_ - 1) / BM_), (NC + BN_ - 1) / BN_));                         \
    if (gen)                                                                                                   \
      MORPHO_KLAUNCH((proj_fwd_kernel<M, DV, BM_, BN_, ST_, true>), g, dim3(kGemmThreads), 0, s, X, gq, gk, d, p);  \
    else                                                                                                       \
      MORPHO_KLAUNCH((proj_fwd_kernel<M, DV, BM_, BN_, ST_, false>), g, dim3(kGemmThreads), 0, s, X, gq, gk, d, p); \
  } while (0)
  if (d.PBM == 256 && d.PBN == 320)
    MORPHO_PROJ_LAUNCH(256, 320, 2);
  else if (d.PBM == 256)
    MORPHO_PROJ_LAUNCH(256, 256, 2);
  else if (d.PBN == 256)  // one workgroup per CU: room for a third stage
    MORPHO_PROJ_LAUNCH(128, 256, 3);
  else if (d.PBN == 160)
    MORPHO_PROJ_LAUNCH(128, 160, 2);
  else
    MORPHO_PROJ_LAUNCH(128, 128, 2);
#undef MORPHO_PROJ_LAUNCH
  return hipGetLastError();
}

hipError_t launch_proj_fwd(const Dims& d, const f16* X, const f16* gq, const f16* gk, const ProjBuffers& p,
                           hipStream_t s) {
#define MORPHO_PROJ_CASE(MM, VV) \
  if (d.M == MM && d.DV == VV) return launch_proj_fwd_t<MM, VV>(d, X, gq, gk, p, s);
  MORPHO_PROJ_CASE(16, 32) MORPHO_PROJ_CASE(16, 64) MORPHO_PROJ_CASE(16, 128)
  MORPHO_PROJ_CASE(32, 32) MORPHO_PROJ_CASE(32, 64) MORPHO_PROJ_CASE(32, 128)
  MORPHO_PROJ_CASE(64, 32) MORPHO_PROJ_CASE(64, 64) MORPHO_PROJ_CASE(64, 128)
#undef MORPHO_PROJ_CASE
  return hipErrorInvalidValue;
}

// ---------------------------------------------------------------- backward elementwise
// The output depends on the gates only through G = gate_q * gate_k, and with
// dq = sum_j dS_ij phi_j, dk = sum_i dS_ij phi_i, dcb = sum_i dS_ij, r =
// sum_j dS_ij (natural-log score gradients, ungated codes):
//   dL/dphi_tc = scale G_c (2 (dq_tc + dk_tc) - dcb_t - r_t)
//   dL/dG_c    = scale sum_t phi_tc (2 dk_tc - dcb_t)
// (the gate sum uses sum_j dS_ij = 0). dL/dG is taken from the key-side sums
// only, whose terms share the same rounded dS, so its cancellation stays
// exact; then d gate_q = dL/dG gate_k and d gate_k = dL/dG gate_q.
//
// Diagonal correction (softmax attention, diagonal key present). The row sum
// r_t of the rounded dS is 0 in exact arithmetic; what the kernels measure is
// the error of the row's delta: an offset nu in delta makes dS_tj wrong by
// -nu P_tj, so r_t = -nu sum_j P_tj. Where the row is concentrated on its
// diagonal (saturated codes: the other weights are tiny and so is the true
// gradient) that offset, however small (fp32 rounding of dO . O suffices),
// dominates the code gradients. Replacing dS_tt by dS_tt - r_t P_tt cancels
// it: dq, dk and dcb of token t lose c = r_t P_tt times the diagonal's
// operands (phi_hi of t, the codes both products used, and 1), and the row
// sum becomes r_t - c. P_tt = 2^(s_tt - lse_t) (s_tt = t_tt + b_t from the
// projection's statistics) comes from bwd_prep, next to r_t.
// A block of kElemThreads threads covers kGateTokensPerBlock tokens and 256
// projection columns. Each thread owns 8 consecutive columns (one head) and
// every kElemSubs-th token of the block, so all loads and stores are 16-byte
// vectors: a wave covers 32 column groups of 2 tokens, i.e. whole 512-byte dZ
// rows and, per head, 2 consecutive rows of dq / dk. The per-thread gate sums
// meet in LDS in a fixed order. (1024 threads: with a few thousand blocks in
// all, 256-thread blocks left one wave per SIMD to cover the memory latency.)
constexpr int kElemThreads = 1024, kElemSubs = kElemThreads / 32;
static_assert(kGateTokensPerBlock % kElemSubs == 0, "whole tokens per thread");
__global__ __launch_bounds__(kElemThreads) void proj_bwd_elem_kernel(const f16* __restrict__ gate_q,
                                                                     const f16* __restrict__ gate_k, Dims d,
                                                                     ProjBuffers p, BwdBuffers g, int row_corr) {
  __shared__ float red[kElemSubs][257];
  const int c8 = threadIdx.x & 31, sub = threadIdx.x >> 5;
  const int col = blockIdx.y * 256 + 8 * c8;  // first of this thread's 8 columns
  const bool active = col < d.HM;
  const int h = col / d.M, c = col - h * d.M;
  const int NC = d.HM + d.D;
  float sg[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (active) {
    float sG[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) sG[e] = d.scale * (float)gate_q[col + e] * (float)gate_k[col + e];
    const int64_t t0 = (int64_t)blockIdx.x * kGateTokensPerBlock;
#pragma unroll
    for (int k = 0; k < kGateTokensPerBlock / kElemSubs; ++k) {
      const int64_t t = t0 + sub + kElemSubs * k;
      if (t >= d.T) break;
      const int b = (int)(t / d.N), n = (int)(t - (int64_t)b * d.N);
      const int64_t bhn = (int64_t)(b * d.H + h) * d.N + n;
      const f16* qrow = p.qa + bhn * d.CW;
      const f16x8 ph = *reinterpret_cast<const f16x8*>(qrow + c);
      const f16x8 pl = *reinterpret_cast<const f16x8*>(qrow + d.M + 8 + c);
      const float4* dqp = reinterpret_cast<const float4*>(g.dq + bhn * d.M + c);
      const float4* dkp = reinterpret_cast<const float4*>(g.dk + bhn * d.M + c);
      const float4 q0 = dqp[0], q1 = dqp[1], k0 = dkp[0], k1 = dkp[1];
      const float dq[8] = {q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, q1.z, q1.w};
      const float dk[8] = {k0.x, k0.y, k0.z, k0.w, k1.x, k1.y, k1.z, k1.w};
      float dcb = g.dcb[bhn], rs = 0.f, cr = 0.f;
      if (row_corr) {  // uniform
        const float2 rp = reinterpret_cast<const float2*>(g.dr)[bhn];  // {r, P_tt}
        cr = rp.x * rp.y;
        rs = rp.x - cr;
        dcb -= cr;
      }
      f16x8 dz;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float phi = (float)ph[e] + (float)pl[e];
        const float cp = cr * (float)ph[e];
        const float dqe = dq[e] - cp, dke = dk[e] - cp;
        const float dphi = sG[e] * (2.f * (dqe + dke) - dcb - rs);
        dz[e] = (f16)(dphi * cube_project_grad(phi, d.proj));
        sg[e] += phi * (2.f * dke - dcb);
      }
      *reinterpret_cast<f16x8*>(g.dzv + t * NC + col) = dz;
    }
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) red[sub][8 * c8 + e] = sg[e];
  __syncthreads();
  const int cc = blockIdx.y * 256 + threadIdx.x;
  if (threadIdx.x < 256 && cc < d.HM) {
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < kElemSubs; ++i) s += red[i][threadIdx.x];
    g.gpart[(int64_t)blockIdx.x * d.HM + cc] = s;
  }
}

hipError_t launch_proj_bwd_elem(const Dims& d, const f16* gq, const f16* gk, const ProjBuffers& p,
                                const BwdBuffers& g, bool row_corr, hipStream_t s) {
  dim3 grid((unsigned)((d.T + kGateTokensPerBlock - 1) / kGateTokensPerBlock), (d.HM + 255) / 256);
  MORPHO_KLAUNCH(proj_bwd_elem_kernel, grid, dim3(kElemThreads), 0, s, gq, gk, d, p, g, row_corr ? 1 : 0);
  return hipGetLastError();
}

// ---------------------------------------------------------------- backward GEMMs
// One launch computes
//   dX = [dZ | dV] [W_phi | W_V]^T                    (dX tiles)
//   [dW_phi | dW_V] = X^T [dZ | dV]                   (dW tiles, split over tokens)
// in one round of workgroups (BwdGemmPlan): ids [0, n_a) compute g whole dX
// tiles each, ids n_a + p t + j piece j of dW tile t (a near-equal 1/p of the
// tokens) and store its fp32 partial, which dw_reduce adds in piece order.
// g and p give both kinds about the same number of k-steps. (Before, every
// dW split of T / 8 tokens and every dX tile was a workgroup of its own; at
// B4 N4096 D1024 H16 m16 a CU then ran a 32-k-step dW split or 20-k-step dX
// tiles, and the launch took about 52 k-steps per CU for 40 of work: dX alone
// 40.6 us, dW alone 53.4 us, both in one launch 90.1 us.)
// Square BT x BT tiles for both products: 256, or 128 when the plan with
// 128 tiles finishes sooner (few tokens). Either way the waves own 64-row wave
// tiles, which the dX epilogue's slabs rely on.
template <int BT>
struct BwdTiles {
  static constexpr int WM = BT == 256 ? 4 : 2;
  using Dx = Gemm<BT, BT, WM, true, true, 64, 2>;    // A = dZ|dV [T][NC], B = wcat = [W_phi | W_V] [D][NC]
  using Dw = Gemm<BT, BT, WM, false, false, 64, 2>;  // A = X (k-major) [T][D], B = dZ|dV (k-major) [T][NC]
  static constexpr int kLds = Dx::kLdsBytes > Dw::kLdsBytes ? Dx::kLdsBytes : Dw::kLdsBytes;
  static constexpr int kStageStride = BT + 8;  // halves: one 64-row slab of fp16 dX for 16-byte stores
  static_assert(64 * kStageStride * 2 <= kLds, "dX slab must fit the main loop's LDS");
  static_assert(Dx::WN == Dw::WN && Dx::WTM == 64 && Dw::WTM == 64, "shared wave grid, 64-row wave tiles");
  static_assert(Dx::kBK == 64 && Dw::kBK == 64, "the plan counts k-steps of 64");
};

struct BwdGemmArgs {
  const f16* X;
  const f16* wcat;
  f16* dX;
  BwdGemmPlan plan;
};

template <int BT>
__global__ __launch_bounds__(kGemmThreads) void bwd_gemm_kernel(Dims d, BwdBuffers g, BwdGemmArgs a) {
  using DxGemm = typename BwdTiles<BT>::Dx;
  using DwGemm = typename BwdTiles<BT>::Dw;
  constexpr int kDxStageStride = BwdTiles<BT>::kStageStride;
  __shared__ __align__(16) char smem[BwdTiles<BT>::kLds];
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = w / DxGemm::WN, wn = w % DxGemm::WN;  // same wave grid for dX and dW
  const BwdGemmPlan& P = a.plan;
  const int NC = d.HM + d.D;
  const int T = (int)d.T;
  const int id = blockIdx.x;

  if (id < P.n_a) {
    // ---- g dX tiles: tiles s g .. s g + g - 1 of XCD xcd's run of the row
    // panels' column tiles
    const int xcd = id & 7, slot = id >> 3, run = (P.n_dx + 7) / 8;
    for (int q = 0; q < P.g; ++q) {
      const int o = slot * P.g + q, L = xcd * run + o;
      const int tm = L / P.ntn_x, tn = L % P.ntn_x;
      if (o >= run || L >= P.n_dx) break;  // uniform
      if (q > 0) __syncthreads();  // the previous tile's slab reads are done before the stages refill
      const int m0 = tm * BT, n0 = tn * BT;
      f32x4 acc[DxGemm::FI][DxGemm::FJ];
      DxGemm::run(g.dzv, NC, a.wcat, NC, T, d.D, m0, n0, 0, NC, smem, acc);
      // fp16 through LDS in 64-row slabs (slab = wave row), then 16-byte row stores
      f16* st = reinterpret_cast<f16*>(smem);
      for (int slab = 0; slab < BT / 64; ++slab) {
        if (slab > 0) __syncthreads();
        if (wm == slab) {
#pragma unroll
          for (int i = 0; i < DxGemm::FI; ++i)
#pragma unroll
            for (int j = 0; j < DxGemm::FJ; ++j)
#pragma unroll
              for (int r = 0; r < 4; ++r)
                st[(16 * i + 4 * (lane >> 4) + r) * kDxStageStride + DxGemm::WTN * wn + 16 * j + (lane & 15)] =
                    (f16)acc[i][j][r];
        }
        __syncthreads();
        for (int qq = tid; qq < 64 * (BT / 8); qq += kGemmThreads) {
          const int r = qq / (BT / 8), c = 8 * (qq % (BT / 8));
          const int row = m0 + 64 * slab + r, col = n0 + c;
          if (row < T && col < d.D)
            *reinterpret_cast<f16x8*>(a.dX + (int64_t)row * d.D + col) =
                *reinterpret_cast<const f16x8*>(st + r * kDxStageStride + c);
        }
      }
    }
    return;
  }

  // ---- dW: piece j of tile tl. The pieces, taken piece by piece (q = j
  // tiles_w + tl), are dealt to the XCDs in contiguous runs (XCD x = id % 8
  // takes q = x per_x + slot), so an XCD's workgroups share one or two token
  // ranges of X and dZ|dV in its L2.
  const int b = id - P.n_a, per_x = (P.tiles_w * P.p + 7) / 8;
  const int q = (b & 7) * per_x + (b >> 3);
  if ((b >> 3) >= per_x || q >= P.tiles_w * P.p) return;
  const int j = q / P.tiles_w, tl = q - j * P.tiles_w;
  const int ks = dw_piece_k0(P.kw, P.p, j), ke = dw_piece_k0(P.kw, P.p, j + 1);
  const int m0 = (tl / P.ntn_w) * BT, n0 = (tl % P.ntn_w) * BT;
  f32x4 acc[DwGemm::FI][DwGemm::FJ];
  DwGemm::run(a.X, d.D, g.dzv, NC, d.D, NC, m0, n0, 64 * ks, min(64 * ke, T), smem, acc);
  // the piece's partial, tile-local row-major [BT][BT], at tl p + j
  float* part = g.wpart + (int64_t)(tl * P.p + j) * BT * BT;
#pragma unroll
  for (int i = 0; i < DwGemm::FI; ++i)
#pragma unroll
    for (int jj = 0; jj < DwGemm::FJ; ++jj) {
      const int col = DwGemm::WTN * wn + 16 * jj + (lane & 15);
#pragma unroll
      for (int r = 0; r < 4; ++r) part[(DwGemm::WTM * wm + 16 * i + 4 * (lane >> 4) + r) * BT + col] = acc[i][jj][r];
    }
}

hipError_t launch_bwd_gemm(const Dims& d, const ProjBuffers& p, const BwdBuffers& g, const f16* X, f16* dX,
                           hipStream_t s) {
  BwdGemmArgs a;
  a.X = X; a.wcat = p.wcat; a.dX = dX;
  a.plan = bwd_gemm_plan(d);
  const dim3 grid((unsigned)(a.plan.n_a + 8 * ((a.plan.tiles_w * a.plan.p + 7) / 8)));
  if (a.plan.bt == 128)
    MORPHO_KLAUNCH(bwd_gemm_kernel<128>, grid, dim3(kGemmThreads), 0, s, d, g, a);
  else
    MORPHO_KLAUNCH(bwd_gemm_kernel<256>, grid, dim3(kGemmThreads), 0, s, d, g, a);
  return hipGetLastError();
}

// Finalisation of the weight and gate gradients, one launch. Blocks
// [0, nw) sum the dW pieces' partials of [dW_phi | dW_V] (4 consecutive
// outputs per thread; the pieces of the output's tile in order); blocks
// [nw, nw + ceil(HM / 16)) sum the per-block gate partials: 16 columns x 16
// row groups per block, group g summing rows g, g + 16, ... with two
// accumulators, the groups then combined in a fixed order. Both orders are
// fixed, so results are deterministic.
__global__ __launch_bounds__(256) void dw_reduce_kernel(const float* __restrict__ wpart, int bt, int ntn_w, int pieces,
                                                        int D, int HM, f16* __restrict__ dW_phi,
                                                        f16* __restrict__ dW_V, int nw,
                                                        const float* __restrict__ gpart, int nblk, float scale,
                                                        const f16* __restrict__ gate_q, const f16* __restrict__ gate_k,
                                                        f16* __restrict__ d_gate_q, f16* __restrict__ d_gate_k) {
  __shared__ float part[16][17];
  if ((int)blockIdx.x >= nw) {
    const int cl = threadIdx.x & 15, grp = threadIdx.x >> 4;
    const int col = ((int)blockIdx.x - nw) * 16 + cl;
    float s0 = 0.f, s1 = 0.f;
    if (col < HM) {
      int i = grp;
#pragma unroll 4
      for (; i + 16 < nblk; i += 32) {  // unrolled: several loads in flight, same order
        s0 += gpart[(int64_t)i * HM + col];
        s1 += gpart[(int64_t)(i + 16) * HM + col];
      }
      if (i < nblk) s0 += gpart[(int64_t)i * HM + col];
    }
    part[grp][cl] = s0 + s1;
    __syncthreads();
    if (grp == 0 && col < HM) {
      float t = 0.f;
#pragma unroll
      for (int g2 = 0; g2 < 16; ++g2) t += part[g2][cl];
      const float dG = scale * t;
      d_gate_q[col] = (f16)(dG * (float)gate_k[col]);
      d_gate_k[col] = (f16)(dG * (float)gate_q[col]);
    }
    return;
  }
  const int NC = HM + D;
  const int64_t idx = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (idx >= (int64_t)D * NC) return;
  const int row = (int)(idx / NC), col = (int)(idx - (int64_t)row * NC);
  const int tl = (row / bt) * ntn_w + col / bt;
  // 4 columns never straddle a tile; piece z of the tile at partial tl pieces + z
  const int64_t tsz = (int64_t)bt * bt;
  const float* src = wpart + (int64_t)tl * pieces * tsz + (int64_t)(row % bt) * bt + col % bt;
  // pieces summed in order; the loads of 8 are issued before their adds
  float4 s = *reinterpret_cast<const float4*>(src);
  int z = 1;
  for (; z + 8 <= pieces; z += 8) {
    float4 v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = *reinterpret_cast<const float4*>(src + (z + i) * tsz);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      s.x += v[i].x; s.y += v[i].y; s.z += v[i].z; s.w += v[i].w;
    }
  }
  for (; z < pieces; ++z) {
    const float4 v = *reinterpret_cast<const float4*>(src + z * tsz);
    s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w;
  }
  // 4 consecutive columns never straddle HM (HM and NC are multiples of 16)
  f16* dst = col < HM ? dW_phi + (int64_t)row * HM + col : dW_V + (int64_t)row * D + (col - HM);
  *reinterpret_cast<f16x4*>(dst) = f16x4{(f16)s.x, (f16)s.y, (f16)s.z, (f16)s.w};
}

hipError_t launch_dw_reduce(const Dims& d, const BwdBuffers& g, const f16* gq, const f16* gk, f16* dW_phi, f16* dW_V,
                            f16* dgq, f16* dgk, hipStream_t s) {
  const int64_t total = (int64_t)d.D * (d.HM + d.D);
  const int nw = (int)((total / 4 + 255) / 256);
  const int ngate = (d.HM + 15) / 16;
  const int nblk = (int)((d.T + kGateTokensPerBlock - 1) / kGateTokensPerBlock);
  const BwdGemmPlan P = bwd_gemm_plan(d);
  MORPHO_KLAUNCH(dw_reduce_kernel, dim3((unsigned)(nw + ngate)), dim3(256), 0, s, g.wpart, P.bt, P.ntn_w, P.p, d.D,
                 d.HM, dW_phi, dW_V, nw, g.gpart, nblk, d.scale, gq, gk, dgq, dgk);
  return hipGetLastError();
}

}  // namespace morpho
