// Minimal Tersoff scalar pieces shared by the kernel families.
//
// Formulas: src/minimal_tersoff.cu:62-119 (fR, fA, fc, g), :147-185 (bond
// order).
#pragma once

#include "device.h"
#include "fastmath.h"
#include "params.h"
#include "population.h"

namespace gpuga {

// Per-parameter-set constants in the form the kernels use: exponent
// prefactors scaled by log2(e) for the exp2 instruction, 1/(R2-R1) and
// 0.5 pi/(R2-R1) for the taper.
struct TLane {
  float cR[2], kR[2], kR2[2], cA[2], kA[2], kA2[2], r0[2];
  float en, mhon, en1, mhon1, beta, beta2, h, r1, r2, inv_span, pif_half;
  float r1min; // population kernels: the smallest R1 of the wave's lanes
};

__host__ __device__ inline TLane tersoff_lane(const TersoffParams& p)
{
  TLane q;
  for (int k = 0; k < 2; ++k) {
    q.cR[k] = p.cR[k];
    q.kR[k] = p.kR[k];
    q.kR2[k] = p.kR[k] * LOG2E;
    q.cA[k] = p.cA[k];
    q.kA[k] = p.kA[k];
    q.kA2[k] = p.kA[k] * LOG2E;
    q.r0[k] = p.r0[k];
  }
  q.en = p.en;
  q.mhon = p.minus_half_over_n;
  q.en1 = p.en - 1.0f;
  q.mhon1 = p.minus_half_over_n - 1.0f;
  q.beta = p.beta;
  q.beta2 = 2.0f * p.beta;
  q.h = p.h;
  q.r1 = p.r1;
  q.r2 = p.r2;
  q.inv_span = 1.0f / (p.r2 - p.r1);
  q.pif_half = 0.5f * p.pi_factor;
  q.r1min = p.r1;
  return q;
}

// fc and dfc/dr (src/minimal_tersoff.cu:77-90)
__device__ __forceinline__ void tersoff_fc(const TLane& q, float d, float& fc, float& fcp)
{
  // 1 below r1, 0 from r2 on (a select), the taper between them under one
  // branch that the wave skips when no lane needs it
  const bool below = d < q.r1;
  fc = below ? 1.0f : 0.0f;
  fcp = 0.0f;
  if (!below && d < q.r2) {
    float sn, cs;
    sincospi01((d - q.r1) * q.inv_span, sn, cs);
    fc = 0.5f * cs + 0.5f;
    fcp = -q.pif_half * sn;
  }
}

// b = (1 + zeta^n)^(-1/2n) and db/dzeta = -1/2 (1 + zeta^n)^(-1/2n - 1)
// zeta^(n - 1), the latter as one exp2 of the summed logarithms (no
// reciprocal); b = 1, b' = 0 below zeta = 1e-16 (src/minimal_tersoff.cu:174-185)
__device__ __forceinline__ void tersoff_bond_order(const TLane& q, float zeta, float& b, float& bp)
{
  const float lz = flog2(zeta);
  const float bzn = fexp2(q.en * lz);
  const float l1 = flog2(1.0f + bzn);
  // the cut-off as selects of the exponents (exp2(0) = 1, exp2(-inf) = 0),
  // so that no branch forms around the exp2 instructions
  const bool tiny = zeta < 1.0e-16f;
  b = fexp2(tiny ? 0.0f : q.mhon * l1);
  bp = -fexp2(tiny ? -__builtin_inff() : fmaf(q.mhon1, l1, fmaf(q.en1, lz, -1.0f)));
}

// fR, fR', fA, fA' (src/minimal_tersoff.cu:62-75) of parameter set k
__device__ __forceinline__ void tersoff_pair(const TLane& q, int k, float d, float& fr, float& frp,
                                             float& fa, float& fap)
{
  const float x = d - q.r0[k];
  fr = q.cR[k] * fexp2(q.kR2[k] * x);
  frp = q.kR[k] * fr;
  fa = q.cA[k] * fexp2(q.kA2[k] * x);
  fap = q.kA[k] * fa;
}

// Both sets' constants as plain values, for a choice between them by selects:
// a select between members of a TLane in memory becomes a load from a selected
// address, and the sets stay in scratch memory (the empty asm keeps the
// compiler from seeing where the values come from).
struct TSets {
  float v[2][7]; // cR, kR, kR2, cA, kA, kA2, r0
};
__device__ __forceinline__ TSets tersoff_sets(const TLane& q)
{
  TSets t;
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const float v[7] = {q.cR[k], q.kR[k], q.kR2[k], q.cA[k], q.kA[k], q.kA2[k], q.r0[k]};
#pragma unroll
    for (int m = 0; m < 7; ++m) {
      t.v[k][m] = v[m];
      asm volatile("" : "+v"(t.v[k][m]));
    }
  }
  return t;
}

// tersoff_pair of set 1 where `second` (wave-uniform), else of set 0
__device__ __forceinline__ void tersoff_pair_sel(const TSets& t, bool second, float d, float& fr,
                                                 float& frp, float& fa, float& fap)
{
  float c[7];
#pragma unroll
  for (int m = 0; m < 7; ++m) c[m] = second ? t.v[1][m] : t.v[0][m];
  const float x = d - c[6];
  fr = c[0] * fexp2(c[2] * x);
  frp = c[1] * fr;
  fa = c[3] * fexp2(c[5] * x);
  fap = c[4] * fa;
}

// Individual p's constants from its genes (every lane of a wave calls it).
template <bool TWO>
__device__ inline TLane tersoff_make(const PopCtl& ctl, int p)
{
  constexpr int V = TWO ? 13 : 9;
  float x[V];
#pragma unroll
  for (int v = 0; v < V; ++v)
    x[v] = denormalise(ldu(ctl.pmin, v), ldu(ctl.pmax, v), ctl.genes[(size_t)p * V + v]);
  TLane q = tersoff_lane(tersoff_params(TWO ? 2 : 1, x));
  // the wave's smallest R1: an atom whose bonds are all shorter has fc = 1,
  // fc' = 0 on every lane
  float m = q.r1;
  const int lane = lane_here();
#pragma unroll
  for (int o = WAVE / 2; o >= 1; o >>= 1) m = fminf(m, wave_xor(m, o, lane));
  q.r1min = m;
  return q;
}

} // namespace gpuga
