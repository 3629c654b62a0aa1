// Diagonal-block Cholesky + inverse for the factor (device code, gfx950).
#pragma once
#include "common.hpp"

namespace g2ptq {
namespace {

// Cholesky + inverse of a diagonal block of the factor (nbk×nbk, nbk <= 64),
// shared by factor.hip's potrf kernel and its panel step (the workgroup that
// updates the next diagonal block factors it as soon as it is written).
//
// Blocked right-looking Cholesky in four 16-column panels on a 256-thread
// workgroup (rows at or past nbk are identity rows), and the inverse
// X = L⁻¹ by forward substitution, block row by block row:
//   panel p (wave 0, lane i = row i): the 16 pivots of columns
//     [16p, 16p + 16) in turn, each d = A[j][j], l_ij = A[i][j]·rsqrt(d), and
//     the rank-1 update of the panel's own later columns.  Every 16-lane DPP
//     row also carries the panel's 16×16 diagonal block (lane i: its row
//     i % 16), so that pivots and multipliers reach all lanes by DPP row
//     broadcasts inside the row: no LDS round trip and no v_readlane on the
//     pivot chain, for 16 more fused multiply-adds per lane and pivot at most;
//   trailing update (waves 0 to 2): A[i][c] −= Σ_t l_it·l_ct over the panel's
//     16 columns for 16p + 16 <= c <= i, by 16×16 tiles on
//     v_mfma_f32_16x16x4_f32, which is the ascending chain of four fused
//     multiply-adds per entry bit for bit (measured on MI355X);
//   inverse rows [16p, 16p + 16) (one of waves 1 to 3, lane i = column i,
//     beside the later panels): acc_r = δ_ri − Σ_{j<r} X[j][i]·l_rj,
//     X[r][i] = acc_r·rsqrt(d_r).
// Every entry receives its updates one fused multiply-add at a time in
// increasing column order, as in the unblocked right-looking algorithm (and
// the column-at-a-time forward substitution), so the block factor is that
// algorithm's to the bit; the blocking only moves the bulk of each step's
// work off the 64-step pivot chain.  1/sqrt comes from the hardware
// reciprocal square root (about 1 ulp): the factor is held to fp32
// tolerance, not to correctly rounded bits.  A non-positive (or NaN) pivot is
// recorded (its index + 1) and the steps run on.
constexpr int POT_NB = 64;          // block edge
constexpr int XP = POT_NB + 1;      // LDS row pitch of the block / X buffer
constexpr int LP = POT_NB + 4;      // LDS row pitch of L (16-byte rows)
constexpr int PB = 16;              // panel width
typedef float f32x4 __attribute__((ext_vector_type(4)));

// Lane O of each 16-lane row to the whole row (DPP row_newbcast:O).
template <int O>
__device__ __forceinline__ float row_lane(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x150 + O, 0xf, 0xf, true));
}

// A DPP operand needs two wait states after the VALU write of its register, the
// result of a reciprocal root one before another VALU instruction reads it, and
// the compiler sees neither inside inline assembly, nor is it known which copies
// and reloads it puts before one.  So what belongs together is one statement,
// which nothing can be put into, and which waits for its operands itself.  (The
// broadcasts are operands of the multiply-adds: the compiler keeps a separate
// v_mov_b32_dpp for each.  One statement per multiply-add, the operands' waits
// left to chance, was no faster: the factor of 2048 columns takes 0.71 ms either way.)
#define G2_COLS(c)                                                                              \
  "+&v"(c[0]), "+&v"(c[1]), "+&v"(c[2]), "+&v"(c[3]), "+&v"(c[4]), "+&v"(c[5]), "+&v"(c[6]),    \
      "+&v"(c[7]), "+&v"(c[8]), "+&v"(c[9]), "+&v"(c[10]), "+&v"(c[11]), "+&v"(c[12]),          \
      "+&v"(c[13]), "+&v"(c[14]), "+&v"(c[15])
#define G2_FMA(reg, k, q, b, m)                                                                \
  ".if " #k " >= %" #q "\n\tv_fmac_f32_dpp %" #reg ", %" #b ", -%" #m " row_newbcast:" #k        \
  " row_mask:0xf bank_mask:0xf\n\t.endif\n\t"

// c[k] −= bcast(b, lane k of each row)·m for k = Q, …, 15.
template <int Q>
__device__ __forceinline__ void row_fma(float (&c)[PB], float b, float m) {
  static_assert(PB == 16, "one entry per lane of a row");
#define G2_K(k) G2_FMA(k, k, 18, 16, 17)
  if constexpr (Q < PB)
    asm("s_nop 1\n\t"
        G2_K(0) G2_K(1) G2_K(2) G2_K(3) G2_K(4) G2_K(5) G2_K(6) G2_K(7) G2_K(8) G2_K(9) G2_K(10)
        G2_K(11) G2_K(12) G2_K(13) G2_K(14) G2_K(15)
        : G2_COLS(c)
        : "v"(b), "v"(m), "n"(Q));
#undef G2_K
}

// Pivot J of a panel, whose reciprocal root is rd: the multipliers mp of the
// lane's row of the diagonal block and m of its own row, and the update of the
// columns J + 1, …, the block's (p) before the row's (a); between the two the
// next pivot dn and its reciprocal root rdn, which takes its time beside a's
// updates.  (A wait of two states: m's product and one more, the block's updates
// after p[J + 1]'s, a's updates.)
template <int J>
__device__ __forceinline__ void pot_update(float (&p)[PB], float (&a)[PB], float rd, float& m,
                                           float& dn, float& rdn) {
  float mp;
#define G2_M(k, reg)                                                                           \
  ".if " #k " == %38\n\tv_mul_f32 %34, %" #k ", %36\n\tv_mul_f32 %35, %" #reg ", %36\n\t.endif\n\t"
#define G2_P(k) G2_FMA(k, k, 37, 34, 34)
#define G2_D(k)                                                                                \
  ".if " #k " == %37\n\tv_mov_b32_dpp %32, %" #k " row_newbcast:" #k                            \
  " row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t.endif\n\t"
#define G2_A(k, reg) G2_FMA(reg, k, 37, 34, 35)
  asm(".if %38 == 0\n\ts_nop 0\n\t.endif\n\t"  // the first root is the compiler's instruction
      G2_M(0, 16) G2_M(1, 17) G2_M(2, 18) G2_M(3, 19) G2_M(4, 20) G2_M(5, 21) G2_M(6, 22)
      G2_M(7, 23) G2_M(8, 24) G2_M(9, 25) G2_M(10, 26) G2_M(11, 27) G2_M(12, 28) G2_M(13, 29)
      G2_M(14, 30)
      "s_nop 0\n\t"
      G2_P(1) G2_P(2) G2_P(3) G2_P(4) G2_P(5) G2_P(6) G2_P(7) G2_P(8) G2_P(9) G2_P(10) G2_P(11)
      G2_P(12) G2_P(13) G2_P(14) G2_P(15)
      ".if %37 > 13\n\ts_nop 1\n\t.endif\n\t"
      G2_D(1) G2_D(2) G2_D(3) G2_D(4) G2_D(5) G2_D(6) G2_D(7) G2_D(8) G2_D(9) G2_D(10) G2_D(11)
      G2_D(12) G2_D(13) G2_D(14) G2_D(15)
      "v_rsq_f32 %33, %32\n\t"
      G2_A(1, 17) G2_A(2, 18) G2_A(3, 19) G2_A(4, 20) G2_A(5, 21) G2_A(6, 22) G2_A(7, 23)
      G2_A(8, 24) G2_A(9, 25) G2_A(10, 26) G2_A(11, 27) G2_A(12, 28) G2_A(13, 29) G2_A(14, 30)
      G2_A(15, 31)
      : G2_COLS(p), G2_COLS(a), "=&v"(dn), "=&v"(rdn), "=&v"(mp), "=&v"(m)
      : "v"(rd), "n"(J + 1), "n"(J));
#undef G2_M
#undef G2_P
#undef G2_D
#undef G2_A
}
#undef G2_FMA
#undef G2_COLS

// A panel's pivot J (d, its reciprocal root rd) and the ones after it: lane i
// holds row i's panel columns in a, and row k0 + i % 16's (of the panel's
// diagonal block) in p.
template <int J>
__device__ __forceinline__ void pot_pivots(float (&a)[PB], float (&p)[PB], float (&l)[PB],
                                           float& rdl, float& dl, int i, float d, float rd) {
  if constexpr (J < PB) {
    rdl = (i == J) ? rd : rdl;
    dl = (i == J) ? d : dl;
    float dn = 0.f, rdn = 0.f;
    if constexpr (J + 1 < PB)
      pot_update<J>(p, a, rd, l[J], dn, rdn);
    else
      l[J] = a[J] * rd;
    pot_pivots<J + 1>(a, p, l, rdl, dl, i, dn, rdn);
  }
}

// The 16 pivot steps of the panel at column k0 on wave 0: rows from As, L
// columns to Lm, 1/sqrt of the pivots to rdv.  (Rows above a pivot carry values that nothing reads:
// Lm is read below the diagonal only.)
__device__ __forceinline__ void pot_panel(const float* As, float* Lm, float* rdv, int k0, int i,
                                          int& fail) {
  float a[PB], p[PB], l[PB];
  float rdl = 0.f, dl = 1.f;  // lane j: 1/sqrt of pivot k0 + j, and the pivot
#pragma unroll
  for (int c = 0; c < PB; ++c) p[c] = As[(k0 + (i & 15)) * XP + k0 + c];
#pragma unroll
  for (int c = 0; c < PB; ++c) a[c] = As[i * XP + k0 + c];
  const float d = row_lane<0>(p[0]);
  pot_pivots<0>(a, p, l, rdl, dl, i, d, __builtin_amdgcn_rsqf(d));
#pragma unroll
  for (int c4 = 0; c4 < PB; c4 += 4)
    *reinterpret_cast<float4*>(&Lm[i * LP + k0 + c4]) = make_float4(l[c4], l[c4 + 1], l[c4 + 2], l[c4 + 3]);
  if (i < PB) rdv[k0 + i] = rdl;
  const uint64_t bad = __builtin_amdgcn_ballot_w64(!(dl > 0.f));  // also catches NaN
  if (fail == 0 && bad) fail = k0 + __builtin_ctzll(bad) + 1;
}

// Trailing update by the panel at column k0 of the lower entries at or past
// column k0 + 16: the 16×16 tiles on or below the diagonal, dealt to waves 0
// to 2 (6, 3 and 1 tiles).  Four K = 4 MFMAs per tile in increasing column
// order; a lane holds rows 4·(lane / 16) + v and column lane % 16 of a tile.
__device__ __forceinline__ void pot_trail(float* As, const float* Lm, int k0, int i, int w) {
  const int t0 = k0 + PB, nt = (POT_NB - t0) / 16;
  const int r16 = i & 15, g = i >> 4;
#pragma unroll 1
  for (int q = w; q < nt * (nt + 1) / 2; q += 3) {
    const int ti = q >= 3 ? 2 : q >= 1 ? 1 : 0, tj = q - ti * (ti + 1) / 2;
    const int r0 = t0 + 16 * ti, c0 = t0 + 16 * tj;
    float av[4], bv[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      av[s] = -Lm[(r0 + r16) * LP + k0 + 4 * s + g];
      bv[s] = Lm[(c0 + r16) * LP + k0 + 4 * s + g];
    }
    f32x4 acc;
#pragma unroll
    for (int v = 0; v < 4; ++v) acc[v] = As[(r0 + 4 * g + v) * XP + c0 + r16];
#pragma unroll
    for (int s = 0; s < 4; ++s)
      acc = __builtin_amdgcn_mfma_f32_16x16x4f32(av[s], bv[s], acc, 0, 0, 0);
#pragma unroll
    for (int v = 0; v < 4; ++v)
      As[(r0 + 4 * g + v) * XP + c0 + r16] = acc[v];  // above the diagonal: not read
  }
}

// Rows [r0, r0 + 16) of X = L⁻¹, lane i = column i (one wave), in three parts
// so that the bulk of the later block rows runs beside the panels:
//   acc_q = δ(r0 + q, i) to begin with;
//   pot_inv_bulk: acc_q −= Σ_{j0 <= j < j0 + 16} X[j][i]·l_{r0+q, j}, j in
//     increasing order (X rows below j0 + 16 final in Xs);
//   pot_inv_fin:  the block's own triangle and the rows into Xs.
// Each entry receives the same fused multiply-adds in the same order however
// the j range is split, so the split is invisible in the results.  Lane i
// holds L's row r0 + i % 16, so that l_{r0+q, j} reaches the lanes as a row
// broadcast: 16 LDS words per lane and 16 columns instead of one broadcast
// read per multiplier.
// Sixteen columns from j0 of L's row r0 + i % 16.
__device__ __forceinline__ void pot_load_l(float (&l)[PB], const float* Lm, int r0, int j0, int i) {
#pragma unroll
  for (int u = 0; u < PB; u += 4) {
    const float4 v = *reinterpret_cast<const float4*>(&Lm[(r0 + (i & 15)) * LP + j0 + u]);
    l[u] = v.x; l[u + 1] = v.y; l[u + 2] = v.z; l[u + 3] = v.w;
  }
}

__device__ __forceinline__ void pot_inv_bulk(float (&acc)[PB], const float* Xs, const float* Lm,
                                             int r0, int j0, int i) {
  float l[PB], x[PB];
  pot_load_l(l, Lm, r0, j0, i);
#pragma unroll
  for (int j = 0; j < PB; ++j) x[j] = Xs[(j0 + j) * XP + i];
#pragma unroll
  for (int j = 0; j < PB; ++j) row_fma<0>(acc, l[j], x[j]);  // l_q on lane q of each row
}

template <int Q>
__device__ __forceinline__ void pot_inv_rows(float (&acc)[PB], float (&l)[PB], float rd, float* X,
                                             int i) {
  if constexpr (Q < PB) {
    const float x = acc[Q] * row_lane<Q>(rd);
    X[Q * XP + i] = x;
    row_fma<Q + 1>(acc, l[Q], x);
    pot_inv_rows<Q + 1>(acc, l, rd, X, i);
  }
}

__device__ __forceinline__ void pot_inv_fin(float (&acc)[PB], float* Xs, const float* Lm,
                                            const float* rdv, int r0, int i) {
  float l[PB];
  pot_load_l(l, Lm, r0, r0, i);
  pot_inv_rows<0>(acc, l, rdv[r0 + (i & 15)], Xs + r0 * XP, i);
}

// The factor of the block staged in Xs (lower triangle, identity padded),
// by a 256-thread workgroup.  Lm (64·LP floats) and rdv (64) are scratch.
// Leaves X = L⁻¹ in Xs (rows, lower triangle; what lies above is not
// defined) and returns the failing pivot index + 1, or 0.
// Schedule (waves w0..w3, `|` a barrier; the trailing updates' tiles on w0 to
// w2, block rows of the inverse on w3, w3, w1 and w2):
//   panel0 | trail0, inv0 triangle (w3) |
//   panel1, inv2[j < 16] (w1), inv3[j < 16] (w2), inv1[j < 16] (w3) |
//   trail1, inv1 triangle (w3) |
//   panel2, inv2[16 <= j < 32] (w1), inv3[16 <= j < 32] (w2) |
//   trail2, inv2 triangle (w1) | panel3, inv3[32 <= j < 48] (w2) | inv3 triangle (w2)
// so only the last block row's triangle follows the last panel.  The four
// rounds are a loop: a workgroup runs this code once, so a straight-line
// schedule (62 KB in potrf_diag_kernel) waits for its instructions.
// MI355X, one workgroup alone: 15.9 thousand cycles (21.2 with v_readlane
// and LDS multipliers, VALU trailing updates and the straight-line schedule),
// of which the pivots 2,400 per panel: a fused multiply-add with a DPP operand
// issues in eight cycles, so a panel's 240 are 1,920 of them.
__device__ __forceinline__ int potrf_core(float* Xs, float* Lm, float* rdv, int* fail_s) {
  const int i = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  int fail = 0;
  int own = w == 1 ? 2 : w == 2 ? 3 : 0;  // the wave's block row of the inverse
  float acc[PB];
#pragma unroll
  for (int q = 0; q < PB; ++q) acc[q] = (own * PB + q == i) ? 1.f : 0.f;
#pragma unroll 1
  for (int p = 0; p < 4; ++p) {
    if (w == 0) {
      pot_panel(Xs, Lm, rdv, p * PB, i, fail);
    } else if (p > 0 && p <= own) {
      pot_inv_bulk(acc, Xs, Lm, own * PB, (p - 1) * PB, i);
    }
    __syncthreads();
    if (w < 3) pot_trail(Xs, Lm, p * PB, i, w);
    if (w != 0 && own == p) {
      pot_inv_fin(acc, Xs, Lm, rdv, p * PB, i);
      if (p == 0) {  // w3 goes on with block row 1
        own = 1;
#pragma unroll
        for (int q = 0; q < PB; ++q) acc[q] = (PB + q == i) ? 1.f : 0.f;
      }
    }
    if (p == 3 && threadIdx.x == 0) *fail_s = fail;
    __syncthreads();
  }
  return *fail_s;
}

}  // namespace
}  // namespace g2ptq
