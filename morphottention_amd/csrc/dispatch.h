// Sizes and launch rules: which tile, split or launch shape a problem takes.
// Host code without HIP, so that a test can evaluate the rules without a GPU.
#pragma once

#include <climits>
#include <cstdint>
#include <initializer_list>

namespace morpho {

// Cube projections phi(z) (cube.cuh:9-17 of the reference): sigmoid (the
// default), clamp((z + 1) / 2, 0, 1), and z itself.
constexpr int kProjSigmoid = 0, kProjHardTanh01 = 1, kProjIdentity = 2;

// Most tokens B N of a call (make_dims refuses more).
constexpr int64_t kMaxTokens = (int64_t)1 << 28;

struct Dims {
  int B, N, D, H, M, DV;  // batch, tokens, model dim, heads, cube_m, head_dim_v
  int NP;                 // N rounded up to a multiple of 64: row length of the V^T layout
  int64_t T;              // B * N tokens
  int NR;                 // rows per batch row in the forward projection's row space: N rounded up to a
                          // multiple of 8 (fill_sizes)
  int64_t TR;             // B * NR rows of that space
  int HM;                 // H * M projection columns
  int CW;                 // 2 * M + 8: code row width (hi/lo split codes + affine augmentation)
  float scale;
  int causal;
  int mask_diag;          // drop key j == query i
  int proj;               // cube projection: kProjSigmoid, kProjHardTanh01 or kProjIdentity
  int det;                // deterministic backward: dq and row sums from per-key-block partials
  // Column order of the forward projection's B operand (wt rows): tiles of
  // PBN columns in groups of PGW (whole or half tiles); when PCPT > 0 group g
  // holds code columns [g PCPT, (g+1) PCPT) then value columns [g PVPT, (g+1)
  // PVPT), so every tile (and, with half tiles, every wave) does the same
  // epilogue work; PCPT == 0 keeps the natural order [W_phi | W_V].
  int PBM, PBN, PGW, PCPT, PVPT;  // PBM: tile rows
};

inline void fill_sizes(Dims& d, int64_t B, int64_t N, int64_t D, int64_t H, int64_t M) {
  d.B = (int)B;
  d.N = (int)N;
  d.NP = (int)((N + 63) / 64 * 64);
  // The projection's rows of one batch row are padded to whole groups of 8
  // tokens, so that its epilogue writes V^T and the remainders of 8 tokens of
  // one column at a time, whatever N is: the padding rows repeat a token and
  // their values are stored as the zeros that the V^T layout wants there. (With
  // unpadded rows every value of a length that 8 does not divide was a 2-byte
  // store: proj_fwd at B64 N197 D768 H12 m64 142 us, padded 79 us with the same
  // epilogue; B2 N9 H8 m32 dv64 167 and 12.4, B1 N1 H1 m16 dv64 178 and 11.6.)
  // A batch row's values take 3 NP D bytes of workspace, so TR stays far below
  // 2^31 on any card.
  d.NR = (int)((N + 7) / 8 * 8);
  d.TR = B * (int64_t)d.NR;
  d.D = (int)D;
  d.H = (int)H;
  d.M = (int)M;
  d.DV = (int)(D / H);
  d.T = B * N;
  d.HM = (int)(H * M);
  d.CW = 2 * (int)M + 8;
}

// Projection tiles: 256 x 320 when 320 divides H*M + D, else 256 x 256.
// When those would fill less than one round of the 256 CUs, 128-row tiles
// of 160 or 128 columns (whichever divides H*M + D and needs fewer rounds
// times tile area; 160 on a tie): e.g. H*M + D = 640, T = 8192 gives 256
// workgroups of 128 x 160 (one round) instead of 320 of 128 x 128. The
// interleaved column order needs whole heads and 16-column blocks per tile,
// and a tile whose width is no multiple of m (160 at m = 64) needs that order,
// or heads would straddle tiles.
inline void choose_proj_tiles(Dims& d) {
  const int NC = d.HM + d.D;
  // tiles of bn columns (bn divides NC) can share the code and value columns
  // evenly: whole heads and whole 16-column blocks each
  auto whole_heads = [&](int bn) {
    const int ntn = NC / bn;
    return d.HM % ntn == 0 && d.D % ntn == 0 && (d.HM / ntn) % d.M == 0 && (d.D / ntn) % 16 == 0;
  };
  d.PBM = 256;
  d.PBN = NC % 320 == 0 ? 320 : 256;
  const int64_t rows = (d.TR + 127) / 128, big = (d.TR + 255) / 256 * ((NC + d.PBN - 1) / d.PBN);
  if (big >= 256) {
    // 128 x 256 tiles (one per CU, three stages) where their rounds, 0.58 of a
    // 256 x 256 round each, are the shorter: a last round of few tiles costs
    // half. proj_fwd in us, 256 -> 128 rows: B64 N197 D768 H12 m64 (300 tiles)
    // 81 -> 69, B64 N256 78 -> 73, B1 N16384 D1024 H16 m32 92 -> 86, B4 N4096
    // D1024 H8 m16 dv128 74 -> 68; the 320-wide tile has no such half.
    const int64_t half = rows * ((NC + 255) / 256);
    if (d.PBN == 256 && 100 * ((big + 255) / 256) > 58 * ((half + 255) / 256)) d.PBM = 128;
  } else {
    int64_t best = -1;
    for (const int bn : {160, 128}) {
      if (NC % bn || (bn % d.M && !whole_heads(bn))) continue;
      const int64_t cost = (rows * (NC / bn) + 255) / 256 * bn;
      if (best < 0 || cost < best) {
        best = cost;
        d.PBM = 128;
        d.PBN = bn;
      }
    }
  }
  d.PGW = d.PBN;
  d.PCPT = d.PVPT = 0;
  if (NC % d.PBN == 0 && whole_heads(d.PBN)) {
    const int ntn = NC / d.PBN;
    // half-tile groups where both halves are whole 16-column blocks
    const int half = (d.HM / ntn) % 32 == 0 && (d.D / ntn) % 32 == 0 ? 2 : 1;
    d.PGW = d.PBN / half;
    d.PCPT = d.HM / ntn / half;
    d.PVPT = d.D / ntn / half;
  }
}

// Whether the longest chain of 128-token blocks of one 128-token workgroup
// (n128 of them) is at least the mean work of one of the 256 CUs: BH n128^2 / 256
// blocks, or BH n128 (n128 + 1) / 512 under the causal mask (`causal_limit` for
// BH (n128 + 1), about 512). The attention kernels then split each chain
// between two groups of waves, one workgroup per CU. Under the causal mask
// there can be more than 256 workgroups; without the long chains that the
// second round's short ones fill up behind, that second round costs more than
// the split gains: attn_fwd in us, not split -> split, causal, 352 workgroups of
// N256 m32 dv64 9.8 -> 15.5, 384 of N512 13.7 -> 16.7, of N640 15.8 -> 18.6, of N768
// 17.4 -> 18.4 (up to 256 workgroups N512 0.92 to 0.97 of the time, beyond N1000
// 0.90 with either).
inline bool few_long_chains(const Dims& d, int causal_limit, bool two_short_rounds = false) {
  const int64_t bh = (int64_t)d.B * d.H, n128 = (d.N + 127) / 128;
  if (!d.causal) return bh * n128 <= 256;
  return bh * (n128 + 1) <= causal_limit && (bh * n128 <= 256 || n128 > 6 || two_short_rounds);
}

// Launch shapes of the attention forward.
constexpr int kFwdRegular = 0, kFwdSmall = 1, kFwdSplit = 2;
// Two 32-query blocks per wave in the regular shape (four waves), else one.
constexpr bool fwd_two_blocks(int M, int DV) { return M <= 32 && DV <= 64 && M * DV <= 1024; }
// Whether the small shape differs from the regular one, which then has 256
// queries per workgroup.
constexpr bool fwd_has_small(int M, int DV) { return fwd_two_blocks(M, DV) || (DV == 128 && M <= 32); }
constexpr bool fwd_has_split(int M, int DV) { return !(M == 64 && DV == 128); }  // two groups' stages fit the LDS
// Launch shape. The split shape where the longest chain of tiles of one
// workgroup is at least the mean work of a CU (few_long_chains): attn_fwd in us,
// small or regular -> split, B1 H8 m16 dv64 N1024 15.9 -> 13.3, N2048 causal
// 28.2 -> 22.7, B1 H16 N2048 31.3 -> 26.4, causal N3001 42.3 -> 33.6, N4096 59.6
// -> 49.4; m64 B1 H8 N2048 causal 39.2 -> 32.8. Beyond: B8 H8 N1024 causal 18.9 ->
// 20.6, unmasked B1 H16 N4096 90.1 -> 92.5. From four key tiles on, six where the
// other shape has 128 queries per workgroup anyway (mean time against not
// split, at N64 1.04 and 1.11, N128 1.03 and 1.10, N256 0.99 and 1.04, N385 0.95 and
// 0.99). Small below two regular workgroups per CU; at dv = 128, where the
// eight waves of a regular workgroup fill a CU, not for one unmasked round of
// them over more than 512 keys (regular -> small, m16: 192 workgroups N1500 41.5
// -> 45.0, N3000 74 -> 82, 256 of N4096 115 -> 123; but 256 of N257 15.5 -> 13.7, 288
// of N3000 153 -> 131, causal 256 of N2048 51.7 -> 44.2).
inline int attn_fwd_shape(const Dims& d) {
  const int most_unsplit = fwd_has_small(d.M, d.DV) ? 192 : 320;
  if (fwd_has_split(d.M, d.DV) && d.N > most_unsplit && few_long_chains(d, 528)) return kFwdSplit;
  const int64_t wgs = (int64_t)((d.N + 255) / 256) * d.B * d.H;
  const bool one_round = d.DV == 128 && !d.causal && wgs <= 256 && d.N > 512;
  return fwd_has_small(d.M, d.DV) && wgs < 2 * 256 && !one_round ? kFwdSmall : kFwdRegular;
}

// Whether the split backward exists: at dv = 128 m = 16 takes 64-query steps,
// whose stages do not fit the LDS twice, and m = 64 would spill 73 values.
constexpr bool bwd_has_split(int M, int DV) { return DV <= 64 || M == 32; }
// The split shape where the longest chain of steps of one workgroup is at
// least the mean work of a CU (few_long_chains). attn_bwd in us, regular ->
// split: B1 H8 m32 dv64 N1024 43.7 -> 26.8, N2048 causal 81.3 -> 47.9, B1 H16
// causal N3001 m16 70.6 -> 52.3, m32 117 -> 87, B1 H16 N2048 m16 51.7 -> 41.9,
// m64 N2048 causal H8 116 -> 78, B2 H8 N1001 m32 dv128 54.8 -> 42.6. Beyond,
// the regular shape: unmasked B1 H16 N4096 m32 177 -> 217, causal B8 H8 N1024
// 55.3 -> 56.4 (dv 128); at m >= 32 it has eight waves on 256 keys and half
// the dq atomics (B1 H16 N4096 causal m64 225 -> 229, m32 157 -> 115), and
// two key blocks are too few steps (B8 H12 N197 m64 28.0 -> 30.4). Two short
// rounds still gain where the regular shape has eight waves (384 workgroups of
// causal N384: m32 dv64 -10 % or more, m16 dv64 +13 %, m32 dv128 +15 %).
inline bool attn_bwd_split(const Dims& d) {
  return bwd_has_split(d.M, d.DV) && !d.det && d.N > 256 &&
         few_long_chains(d, d.M == 64 ? 420 : 528, d.M >= 32 && d.DV <= 64);
}

// The split shape as in the softmax forward. soft_fwd_fast in us, one group
// -> two: B2 N1001 H8 m32 29.0 -> 23.6, B1 N2048 H16 m16 50 -> 42, B1 H16
// causal N3000 m64 91 -> 71, N4096 m32 108 -> 91, B1 N300 H2 m16 11.3 -> 10.5;
// with one key tile +5 %, with two 0 to -10 %.
inline bool soft_fwd_split(const Dims& d) { return d.DV <= 64 && d.N > 64 && few_long_chains(d, 528); }
// As the softmax backward: the split shape where one workgroup's chain of
// steps is at least the mean work of a CU. soft_bwd_fast in us, regular ->
// split: B2 N1001 H8 m16 dv64 74 -> 55, m32 83 -> 60, m64 116 -> 77, B1 H16
// causal N3000 m16 170 -> 121, m64 272 -> 179, N4096 m32 274 -> 223; B1 N300 H2
// m16 32 -> 28. Two groups at dv = 128 would need more registers than two
// waves per SIMD have.
inline bool soft_bwd_split(const Dims& d) { return d.DV <= 64 && d.N > 256 && few_long_chains(d, 528); }

// Lanes per value column of soft_fvals, 8 keys each: as many as the column has
// groups of 8, up to a wave; a workgroup of four waves for few long columns,
// which would leave most of the chip idle. soft_fvals in us, one wave -> four:
// 64 columns N4096 8.4 -> 4.2, 1024 columns N2048 6.0 -> 5.2, N4096 9.8 -> 7.8;
// 2048 columns N2048 7.5 -> 7.5, N4096 13.9 -> 14.3; 8192 columns N4096 53 -> 61,
// N513 10.2 -> 13.9; 32768 columns N513 31 -> 45. Short columns, one wave -> 8
// lanes: 131072 columns N16 69 -> 11.4.
inline int soft_fvals_lanes(const Dims& d) {
  if (d.NP <= 64) return 8;
  if (d.NP <= 128) return 16;
  if (d.NP <= 256) return 32;
  return d.NP > 1024 && (int64_t)d.B * d.D < 2048 ? 256 : 64;
}
// Its workgroups of 256 lanes, which take further columns in turn beyond 2^20:
// one lane group for every column would pass 2^32 work-items within the
// accepted sizes (B D = 2^24 columns of 256 lanes).
inline unsigned soft_fvals_grid(const Dims& d) {
  const int64_t per = 256 / soft_fvals_lanes(d), wgs = ((int64_t)d.B * d.D + per - 1) / per;
  return (unsigned)(wgs < (1 << 20) ? wgs : 1 << 20);
}

// Work decomposition of the backward GEMM launch: one round of kGemmSlots
// workgroups (the CUs of an MI355X; twice as many with 128 x 128 tiles, two
// per CU). Workgroups [0, n_a), n_a / 8 per XCD (workgroup id % 8), compute g
// whole dX tiles each; the next 8 ceil(tiles_w p / 8) each compute one piece
// j < p of a dW tile t (the tile's kw token k-steps split into p near-equal
// ranges; an XCD's workgroups take a contiguous run of the pieces in (j, t)
// order, so they share token ranges). g and p are chosen so that both kinds
// take about the same number of k-steps. Piece j stores an fp32 tile partial that dw_reduce
// adds in piece order, so the result does not depend on timing.
constexpr int kGemmSlots = 256;
struct BwdGemmPlan {
  int bt;                   // tile edge: 256, or 128 when that finishes sooner (few tiles)
  int n_dx, ntn_x, kx;      // dX tiles, dX column tiles, k-steps per dX tile
  int tiles_w, ntn_w, kw;   // dW tiles, dW column tiles, k-steps per dW tile (all tokens)
  int g, n_a;               // dX tiles per type-A workgroup, type-A workgroups
  int p;                    // pieces per dW tile (tiles_w p type-B workgroups and partials)
};
// Plan for tile edge bt and `slots` workgroups (the dW pieces take
// 8 ceil(tiles_w p / 8) of them): for each g (dX tiles per type-A
// workgroup), the most pieces p per dW tile that still fit the round,
// scored by the longer of the two kinds: g kx against ceil(kw / p) k-steps
// (plus one step of epilogue per dX tile or piece). When the dW tiles alone
// fill the round, every workgroup takes one tile over several rounds. The dX
// tiles, row panel by row panel, are dealt to the XCDs in 8 equal runs, so all
// but the panels at a cut are read into one L2 (whole panels per XCD left
// workgroups without a tile: 18 of 168 at B64 N197 D768 H12 m64, where the dW
// pieces then took 50 k-steps instead of 40).
inline BwdGemmPlan plan_for(const Dims& d, int bt, int slots, int64_t& cost) {
  BwdGemmPlan P;
  const int NC = d.HM + d.D, T = (int)d.T;
  P.bt = bt;
  const int ntm_x = (T + bt - 1) / bt;
  P.ntn_x = (d.D + bt - 1) / bt;
  P.n_dx = ntm_x * P.ntn_x;
  P.kx = (NC + 63) / 64;
  P.ntn_w = (NC + bt - 1) / bt;
  P.tiles_w = ((d.D + bt - 1) / bt) * P.ntn_w;
  P.kw = (T + 63) / 64;
  const int per_xcd = (P.n_dx + 7) / 8;  // dX tiles of one XCD
  cost = INT64_MAX;
  P.g = per_xcd;
  P.n_a = 8;
  P.p = 1;
  for (int g = 1; g <= per_xcd; ++g) {
    const int n_a = 8 * ((per_xcd + g - 1) / g);
    int p = (slots - n_a) / P.tiles_w;
    while (p > 0 && n_a + 8 * ((P.tiles_w * p + 7) / 8) > slots) --p;  // whole runs of 8
    if (p < 1) continue;
    p = p < P.kw ? p : P.kw;
    const int64_t ca = (int64_t)g * (P.kx + 1), cb = (P.kw + p - 1) / p + 1;
    const int64_t cst = ca > cb ? ca : cb;
    if (cst < cost) {
      cost = cst;
      P.g = g;
      P.n_a = n_a;
      P.p = p;
    }
    if (ca > cost) break;  // g kx only grows from here
  }
  // no more pieces than the cost needs: each is a partial to write and add (B3
  // N1500 D1024 H8 m32 dv128: 9 -> 4 pieces)
  while (cost != INT64_MAX && P.p > 1 && (P.kw + P.p - 2) / (P.p - 1) + 1 <= cost) --P.p;
  if (cost == INT64_MAX) {
    // dW tiles alone fill the round: one dX tile or one whole dW tile per
    // workgroup over several rounds (the dispatcher balances them)
    P.g = 1;
    P.n_a = 8 * per_xcd;
    P.p = 1;
    cost = ((int64_t)P.n_dx * (P.kx + 1) + (int64_t)P.tiles_w * (P.kw + 1) + slots - 1) / slots;
  }
  return P;
}

inline BwdGemmPlan bwd_gemm_plan(const Dims& d) {
  int64_t c256, c128;
  const BwdGemmPlan p256 = plan_for(d, 256, kGemmSlots, c256);
  if (d.D % 128 != 0 || (d.HM + d.D) % 128 != 0) return p256;
  // 128 x 128 tiles: two workgroups per CU (64 KiB of LDS each), so twice the
  // slots; a k-step does a quarter of the work of a 256 x 256 one at about 2/3
  // of its rate (more LDS and L2 traffic per MFMA), and shares its CU
  const BwdGemmPlan p128 = plan_for(d, 128, 2 * kGemmSlots, c128);
  return 3 * c128 < 4 * c256 ? p128 : p256;
}

}  // namespace morpho
