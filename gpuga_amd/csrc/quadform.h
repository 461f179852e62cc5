// The fitness of a pair potential over a training set as three quadratic
// forms of the individual's potential curve.
//
// A pair potential's energies, virials and forces are linear in the values of
// U and U' at the pair distances, and U and U' are known everywhere from
// their values at a few Chebyshev nodes per element of the distance range
// (interpolation far below FP32 rounding).  So with v an individual's values
// (nodal values, parameters that enter linearly, and the constant 1), every
// row of residuals (energy - label, virial - label, force - label) is a row
// r . v with r from the training set alone, and the sums of squares are
// v^T Q v with Q = sum r r^T, built once per training set in FP64.
#pragma once

#include "common.h"
#include "device.h"
#include "kernels.h"

namespace gpuga {

constexpr int QP = 16;       // individuals per workgroup of the evaluation
constexpr int QB = 32;       // nodes per element = columns per block
constexpr int kQuadOne = 12; // column of the linear block that holds the constant 1

// Value blocks of QB columns: U at the nodes of element e of pair code c at
// c E + e, U' at CE + c E + e, then one block of linear columns: 4 t + 0..3 =
// the rigid-ion parameters qq_t, C_t, k1_t, k0_t, and the constant 1.
//
// With NN2B's species codes the forms' columns are code 0's values, to which
// the pairs of every code contribute, and the differences of the codes 1 and
// 2 from them: where the species weights are zero the differences are exact
// zeros, and the sums are those of the network without species bit for bit.
struct QuadBasis {
  int codes, E; // pair codes (rigid-ion types, species codes); elements per code
  double d0, len; // element e covers [d0 + e len, d0 + (e + 1) len]
  int rigid;      // rigid ion (linear columns), else NN2B (taper)
  __host__ __device__ bool species() const { return !rigid && codes > 1; }
  __host__ __device__ int CE() const { return codes * E; }
  __host__ __device__ int blocks() const { return 2 * CE() + 1; }
};

// Node m of element e (Chebyshev points of the first kind), as the FP32
// tabulation takes it.
__device__ inline float node_at(const QuadBasis& b, int e, int m)
{
  const float x = __builtin_cosf(PI_F / QB * (m + 0.5f));
  return (float)(b.d0 + b.len * (e + 0.5 + 0.5 * (double)x));
}

// One form: nb column blocks (the first the linear one, then code 0's or, for
// rigid ion, all types', then the differences) and Q as tiles
// (I, J <= I), the ones with J < I doubled, [column of J][row of I] each.
struct QuadForm {
  int nb;
  const int* vblk; // [nb] value block of each column block
  const double* q;
};
constexpr long quad_tiles(long nb) { return nb * (nb + 1) / 2; }

// Do the nodes resolve an individual's curve?  Its last QTAIL Chebyshev
// coefficients in each element show it: where they are small the series has
// converged and the interpolation error is about theirs, else the individual's
// fitness by the forms is not to be used.  Compared are the mean squares, over
// the pairs of the set, of the coefficients and of the terms' magnitude (the
// sum of |w2 tanh| for U, of |w2 sech^2 dz/dr| for U'), which is what the
// nodes' rounding is relative to: of U and U' over the energy configurations'
// pairs, of U' over the force configurations'.
//
// Limits: the coefficients of smooth networks, rounding alone, reach 3.4e-7 of
// the magnitude with the FP32 layer and 7e-6 with the split BF16 one (6000
// networks of 6 to 32 neurons with weights up to 3, and weights up to 6); at the
// limits the interpolation errs by up to 1.8e-6 and 2e-5 of U' (root mean
// square), the BF16 layer's rounding of the nodes by 2e-5 to 1e-4.  The pair
// loop's interpolation errs by up to 6e-6 for networks with weights uniform in
// [-3, 3] and 32 neurons on 1024 points, more for sharper ones.
constexpr int QTAIL = 4;
constexpr int kTailSums = 6; // (coefficients, magnitude) of energy, virial, force
constexpr float kTailFp32 = 1e-6f, kTailBf16 = 1e-5f;
struct SharpSet {
  const float* sums; // [parts][kTailSums][ld]; null: no check (rigid ion)
  int parts;
  float limit2;      // square of the limit
  unsigned* count;   // individuals found by this launch, and, cleared by it,
  unsigned* next;    // the counter of the next one
  int* list;         // [P] the individuals, in any order
  unsigned* any;     // set to 1 when there are some (pinned host memory)
};

// Evaluation of all forms for a population: values [blocks][QB][ld].
struct QuadEval {
  QuadForm form[3]; // energy, virial, force
  const int2* unit; // [units] (form, row block), the longest rows first
  int units;
  const double* values;
  int ld;           // individuals, padded to a multiple of QP
  double* part;     // [units][ld] row-block sums
  unsigned* done;   // [ld / QP]
  SharpSet sharp;   // individuals that the nodes do not resolve
};

// Where the tabulation kernels put U and U' of the nodes.
struct NodeTable {
  QuadBasis b;
  const int2* act; // [n_act] rigid ion: (code E + e, 1) that some row uses;
                   // NN2B: element, mask of the codes that use it (code 0's
                   // always, with the differences of the others)
  int n_act;
  double* values;
  int ld;
  // NN2B: pairs of energy and force configurations in each element of each
  // code, and the rows k = QB - QTAIL, ... of the transform to Chebyshev
  // coefficients, (2 / QB) cos(k theta_m); where the check's sums go
  const float2* pairs; // [CE]
  const float* tail;   // [QTAIL][QB]
  float* sums;
};

// A training set's rows, for the set-up.  col[0][form][block]: column block
// of U's element in the form, col[1]: of U''s, -1 where no row uses it.
struct QuadRows {
  QuadBasis b;
  const int* col;
  int nb[3];
  int D(int form) const { return nb[form] * QB; }
};

// smallest and largest bond length as float bits in range[0], range[1]
// (initialised by the caller)
void launch_bond_range(int B, const float4* bond, unsigned* range, hipStream_t st);
// per-bond rigid-ion factors (r^-6, erfc(a r)/r, -(d/dr) erfc(a r)/r, 1/r)
void launch_ri_table(int B, const float4* bond, float4* tab, hipStream_t st);
// used[force][taper][CE]: elements the pairs of energy / force configurations
// fall into (taper: those of pairs inside the NN2B taper); then [force][CE]: how
// many pairs (at most QCE elements of all codes)
constexpr int QCE = 64;
void launch_quad_used(const DevSet& s, const QuadBasis& b, int* used, hipStream_t st);
// raises the row kernels' LDS limits; false: the rows do not fit
bool quad_prepare(const QuadRows& q);
// rows of the configurations [c0, c1) (energy [c1 - c0][D0], virial
// 6 rows each [..][D1]) and of the force atoms [i0, i1) (3 rows each)
void launch_quad_energy_rows(const DevSet& s, const QuadRows& q, int c0, int c1, double* re,
                             double* rw, hipStream_t st);
void launch_quad_force_rows(const DevSet& s, const QuadRows& q, int i0, int i1, double* rf,
                            hipStream_t st);
// q[tiles][QB * QB] (+)= R^T R of R [rows][nb * QB]; rows a multiple of 4.
// The rows are split over waves whose partial tiles, of kQuadGroup tiles at a
// time, meet in part (quad_part_size).
constexpr int kQuadSplits = 16, kQuadGroup = 512;
constexpr size_t quad_part_size(long nb)
{
  const long t = quad_tiles(nb);
  return (size_t)(t < kQuadGroup ? t : kQuadGroup) * kQuadSplits * QB * QB;
}
void launch_quad_gram(const double* R, int rows, int nb, bool first, double* part, double* q,
                      hipStream_t st);
// Q's tiles, in place, from Chebyshev coefficients to nodal values
void launch_quad_finish(int nb, double* q, hipStream_t st);
// configurations and force atoms whose rows are taken at a time
constexpr int kQuadConfigs = 512, kQuadAtoms = 2048;
constexpr int quad_step(int most, int n) // (rows come in fours)
{
  const int n4 = n < 1 ? 4 : (n + 3) / 4 * 4;
  return n4 < most ? n4 : most;
}

void launch_ri_values(const PopCtl& ctl, const NodeTable& t, hipStream_t st);
// workgroups an individual (parts of its check's sums)
constexpr int nn2b_node_parts(int P) { return P >= 128 ? 1 : 2; }
// the individuals [first, first + count)
void launch_nn2b_nodes(const PopCtl& ctl, const NN2BGrid& g, const NodeTable& t, int first,
                       int count, hipStream_t st);
void launch_quad_eval(const PopCtl& ctl, const QuadEval& q, hipStream_t st);

} // namespace gpuga
