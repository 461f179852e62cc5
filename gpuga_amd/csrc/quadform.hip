// Quadratic forms of the pair potentials' fitness (quadform.h): set-up of the
// matrices Q from a training set, and their evaluation for a population.
//
// Set-up.  Rows are built in the Chebyshev basis T_k of each element (one
// cosine per pair and column), Q = R^T R is taken on the FP64 matrix
// instruction over row chunks, in a fixed order, and each tile is then
// transformed to nodal values (Chebyshev points of the first kind), so that
// an individual's values enter without a transform of their own.
//
// Against the pair loop, whose work is pairs x individuals: a generation of
// 200 individuals on 48 000 oxide atoms (2.7 M pairs) 347 -> 16 us of kernel
// time, of 256 on 57 600 wurtzite atoms (1.5 M pairs, network of 32 neurons)
// 407 -> 37 us.  Its own work does not depend on the training set's size, and
// it was no slower on sets of two cells (two oxide cells, 200 individuals: 74
// -> 52 us a call; 4 wurtzite cells: 90 -> 68 us).
#include "quadform.h"

namespace gpuga {

namespace {

typedef double f64x4 __attribute__((ext_vector_type(4)));
constexpr double PI_D = 3.14159265358979323846;

// cos(k theta) with theta = acos(x): T_k(x)
__device__ __forceinline__ double cheb(int k, double theta) { return cos(k * theta); }

__global__ void __launch_bounds__(256) bond_range(int B, const float4* __restrict__ bond,
                                                  unsigned* range)
{
  // positive floats order as their bits
  unsigned lo = 0xffffffffu, hi = 0u;
  for (int b = blockIdx.x * blockDim.x + threadIdx.x; b < B; b += gridDim.x * blockDim.x) {
    const unsigned d = __float_as_uint(bond[b].w);
    lo = min(lo, d);
    hi = max(hi, d);
  }
#pragma unroll
  for (int o = 1; o < WAVE; o <<= 1) {
    lo = min(lo, (unsigned)__shfl_xor((int)lo, o));
    hi = max(hi, (unsigned)__shfl_xor((int)hi, o));
  }
  if (__lane_id() == 0) {
    atomicMin(&range[0], lo);
    atomicMax(&range[1], hi);
  }
}

// erfc(a d) / d and -(d/dr) of it (a = 0.2, src/ri.cu:80-101)
__device__ __forceinline__ void coulomb(double d, double dinv, double& f, double& h)
{
  f = erfc(0.2 * d) * dinv;
  h = f * dinv + 0.225675833419103 * exp(-0.04 * d * d) * dinv;
}

__global__ void __launch_bounds__(256) ri_table(int B, const float4* __restrict__ bond,
                                                float4* __restrict__ tab)
{
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= B) return;
  const double d = bond[b].w, dinv = 1.0 / d, d2 = dinv * dinv;
  double f, h;
  coulomb(d, dinv, f, h);
  tab[b] = make_float4((float)(d2 * d2 * d2), (float)f, (float)h, (float)dinv);
}

// The element of a pair (code E + e) and acos of its place in it.
__device__ __forceinline__ int locate(const QuadBasis& b, double d, int code, double* theta)
{
  const double u = (d - b.d0) / b.len;
  const int e = min(max((int)u, 0), b.E - 1);
  if (theta) *theta = acos(min(max(2.0 * (u - e) - 1.0, -1.0), 1.0));
  return code * b.E + e;
}

// NN2B's fixed taper (src/nn2b.cu:80-92)
__device__ __forceinline__ void nn2b_taper(double d, double& fc, double& fcp)
{
  fc = fcp = 0.0;
  if (d < NN2B_R1) {
    fc = 1.0;
  } else if (d < NN2B_R2) {
    const double a = (double)NN2B_PI_FACTOR * (d - NN2B_R1);
    fc = 0.5 * cos(a) + 0.5;
    fcp = -0.5 * (double)NN2B_PI_FACTOR * sin(a);
  }
}

__global__ void __launch_bounds__(256) quad_used(DevSet s, QuadBasis b, int* used)
{
  __shared__ int pairs[2 * QCE];
  const int i = blockIdx.x * blockDim.x + threadIdx.x, CE = b.CE();
  for (int x = threadIdx.x; x < 2 * CE; x += blockDim.x) pairs[x] = 0;
  __syncthreads();
  const int force = i < s.N_force ? 1 : 0;
  const int k0 = i < s.N ? s.bond0[i] : 0, k1 = i < s.N ? k0 + s.nn[i] : 0;
  for (int k = k0; k < k1; ++k) {
    if (!force && s.nl[k] < i) continue;
    const float d = s.bond[k].w;
    const int ce = locate(b, d, b.codes > 1 ? s.ptype[k] : 0, nullptr);
    // (every writer stores the same 1)
    const bool taper = !b.rigid && d >= NN2B_R1 && d < NN2B_R2;
    int* u = used + 2 * force * CE;
    u[ce] = 1;
    atomicAdd(&pairs[force * CE + ce], 1);
    if (b.species()) u[ce % b.E] = 1;
    if (taper) {
      u[CE + ce] = 1;
      if (b.species()) u[CE + ce % b.E] = 1;
    }
  }
  __syncthreads();
  for (int x = threadIdx.x; x < 2 * CE; x += blockDim.x)
    if (pairs[x]) atomicAdd(&used[4 * CE + x], pairs[x]);
}

// A pair as the row kernels read it from LDS.
struct PairRec {
  double theta;  // acos of its place in the element
  double fc, ft; // factor of U' (and of U in the energy), of U (taper only)
  double v[6];   // virial coefficients u_a u_b d, or the unit vector in v[0..2]
  double lin[4]; // rigid ion: erfc(a d)/d, -d^-6, -d, -1 (energy)
  double lw[3];  //            h, -6 d^-7, 1 (virial; force with the sign turned)
  int ce, code;
};

__device__ inline PairRec pair_rec(const QuadBasis& b, const float4& r, int code, bool force)
{
  PairRec p;
  const double d = r.w, dinv = 1.0 / d;
  p.code = code;
  p.ce = locate(b, d, b.codes > 1 ? code : 0, &p.theta);
  const double x = r.x, y = r.y, z = r.z;
  if (force) {
    p.v[0] = x * dinv;
    p.v[1] = y * dinv;
    p.v[2] = z * dinv;
  } else {
    p.v[0] = x * x * dinv;
    p.v[1] = y * y * dinv;
    p.v[2] = z * z * dinv;
    p.v[3] = x * y * dinv;
    p.v[4] = y * z * dinv;
    p.v[5] = z * x * dinv;
  }
  p.fc = 1.0;
  p.ft = 0.0;
  if (b.rigid) {
    const double d2 = dinv * dinv, d6 = d2 * d2 * d2;
    double f, h;
    coulomb(d, dinv, f, h);
    p.lin[0] = f;
    p.lin[1] = -d6;
    p.lin[2] = -d;
    p.lin[3] = -1.0;
    p.lw[0] = h;
    p.lw[1] = -6.0 * d6 * dinv;
    p.lw[2] = 1.0;
  } else {
    double fcp;
    nn2b_taper(d, p.fc, fcp);
    p.ft = p.fc * fcp; // f2 = (U' fc + (U fc) fc') / r, src/nn2b.cu:147-148
  }
  return p;
}

// One pair added to a row, lane k on column k of the pair's element: U with
// factor cu (column map mu), U' with cd (md), with species codes also on code
// 0's columns; rigid ion: lanes below nl on the linear columns (the first).
__device__ __forceinline__ void add_pair(double* row, const int* mu, const int* md,
                                         const QuadBasis& b, const PairRec& p, int k, double cu,
                                         double cd, const double* l, int nl, double cl)
{
  const double t = cheb(k, p.theta);
  if (cu != 0.0) row[mu[p.ce] * QB + k] += cu * t;
  if (cd != 0.0) row[md[p.ce] * QB + k] += cd * t;
  if (b.species() && p.ce >= b.E) {
    const int e = p.ce % b.E;
    if (cu != 0.0) row[mu[e] * QB + k] += cu * t;
    if (cd != 0.0) row[md[e] * QB + k] += cd * t;
  }
  if (b.rigid && k < nl) row[p.code * 4 + k] += cl * l[k];
}

constexpr int ENERGY_THREADS = 256, FORCE_THREADS = 96;
constexpr size_t kRowLds = 156 * 1024; // their dynamic LDS at most

// Rows of one energy configuration per workgroup: half-wave 0 its energy,
// half-waves 1-6 its virial components, each over the unordered pairs in bond
// order (so the sums do not depend on scheduling).
__global__ void __launch_bounds__(ENERGY_THREADS) quad_energy_rows(DevSet s, QuadRows q, int c0,
                                                                   double* __restrict__ re,
                                                                   double* __restrict__ rw)
{
  extern __shared__ double lds[];
  PairRec* rec = reinterpret_cast<PairRec*>(lds); // [ENERGY_THREADS]
  double* acc = lds + ENERGY_THREADS * sizeof(PairRec) / sizeof(double);
  __shared__ int cnt[ENERGY_THREADS / WAVE];
  const int t = threadIdx.x, c = c0 + blockIdx.x, CE = q.b.CE();
  const int DE = q.nb[0] * QB, DW = q.nb[1] * QB;
  for (int k = t; k < DE + 6 * DW; k += ENERGY_THREADS) acc[k] = 0.0;
  const int a = t / 32, k = t & 31;
  double* row = a == 0 ? acc : acc + DE + (long)(a - 1) * DW;
  const int form = a == 0 ? 0 : 1;
  const int* mu = q.col + form * CE;
  const int* md = q.col + (3 + form) * CE;
  const int i0 = s.Na_sum[c], i1 = i0 + s.Na[c] - 1;
  const int b0 = s.bond0[i0], b1 = s.bond0[i1] + s.nn[i1];
  for (int bt = b0; bt < b1; bt += ENERGY_THREADS) {
    const int b = bt + t;
    // (the owner of bond b is the neighbour of its reverse)
    const bool on = b < b1 && s.nl[b] > s.nl[s.rev[b]];
    const unsigned long long m = __ballot(on);
    __syncthreads(); // the last batch has been read
    if (__lane_id() == 0) cnt[t / WAVE] = __popcll(m);
    __syncthreads();
    int at = __popcll(m & ((1ull << __lane_id()) - 1ull)), n = 0;
    for (int w = 0; w < ENERGY_THREADS / WAVE; ++w) {
      if (w < t / WAVE) at += cnt[w];
      n += cnt[w];
    }
    if (on) rec[at] = pair_rec(q.b, s.bond[b], s.ptype[b], false);
    __syncthreads();
    if (a < 7)
      for (int j = 0; j < n; ++j) {
        const PairRec& p = rec[j];
        if (a == 0) {
          add_pair(row, mu, md, q.b, p, k, p.fc, 0.0, p.lin, 4, 1.0);
        } else {
          const double v = p.v[a - 1];
          add_pair(row, mu, md, q.b, p, k, -v * p.ft, -v * p.fc, p.lw, 3, v);
        }
      }
  }
  __syncthreads();
  if (a < 7 && k == 0)
    row[kQuadOne] = a == 0 ? -(double)s.pe_ref[c]
                                 : -(double)s.virial_ref[c + (long)s.Nc * (a - 1)];
  __syncthreads();
  double* oe = re + (long)blockIdx.x * DE;
  double* ow = rw + (long)blockIdx.x * 6 * DW;
  for (int x = t; x < DE; x += ENERGY_THREADS) oe[x] = acc[x];
  for (int x = t; x < 6 * DW; x += ENERGY_THREADS) ow[x] = acc[DE + x];
}

// Rows of one force atom per workgroup: a half-wave per component.
__global__ void __launch_bounds__(FORCE_THREADS) quad_force_rows(DevSet s, QuadRows q, int i0,
                                                                 double* __restrict__ rf)
{
  extern __shared__ double lds[];
  PairRec* rec = reinterpret_cast<PairRec*>(lds); // [FORCE_THREADS]
  double* acc = lds + FORCE_THREADS * sizeof(PairRec) / sizeof(double);
  const int t = threadIdx.x, i = i0 + blockIdx.x, CE = q.b.CE();
  const int D = q.nb[2] * QB;
  for (int x = t; x < 3 * D; x += FORCE_THREADS) acc[x] = 0.0;
  const int a = t / 32, k = t & 31;
  double* row = acc + (long)a * D;
  const int* mu = q.col + 2 * CE;
  const int* md = q.col + 5 * CE;
  const int b0 = s.bond0[i], b1 = b0 + s.nn[i];
  for (int bt = b0; bt < b1; bt += FORCE_THREADS) {
    const int n = min(FORCE_THREADS, b1 - bt);
    __syncthreads();
    if (t < n) rec[t] = pair_rec(q.b, s.bond[bt + t], s.ptype[bt + t], true);
    __syncthreads();
    for (int j = 0; j < n; ++j) {
      const PairRec& p = rec[j];
      const double u = p.v[a];
      add_pair(row, mu, md, q.b, p, k, u * p.ft, u * p.fc, p.lw, 3, -u);
    }
  }
  __syncthreads();
  if (k == 0) row[kQuadOne] = -(double)s.force_ref[i + (long)s.N * a];
  __syncthreads();
  double* o = rf + (long)blockIdx.x * 3 * D;
  for (int x = t; x < 3 * D; x += FORCE_THREADS) o[x] = acc[x];
}

// The (I, J) index of a tile.
__device__ __forceinline__ void tile_of(int tile, int& I, int& J)
{
  I = (int)((sqrtf(8.0f * tile + 1.0f) - 1.0f) * 0.5f);
  while ((I + 1) * (I + 2) / 2 <= tile) ++I;
  while (I * (I + 1) / 2 > tile) --I;
  J = tile - I * (I + 1) / 2;
}

// One 32 x 32 tile of R^T R per wave over its split of the rows, four 16 x 16
// products of v_mfma_f64_16x16x4_f64: lane l holds column l % 16 of row
// r + l / 16 of either operand (R is row-major: coalesced), and the results'
// rows 4 x + l / 16, column l % 16.
__global__ void __launch_bounds__(256) quad_gram(const double* __restrict__ R, int rows, int nb,
                                                 int tile0, double* __restrict__ part)
{
  constexpr int splits = kQuadSplits;
  const int lane = __lane_id(), split = blockIdx.y * 4 + wave_first((int)(threadIdx.x / WAVE));
  if (split >= splits) return;
  int I, J;
  tile_of(tile0 + blockIdx.x, I, J);
  const long D = (long)nb * QB;
  const int quads = rows / 4;
  const int q0 = (int)((long)quads * split / splits), q1 = (int)((long)quads * (split + 1) / splits);
  double* out = part + ((long)split * gridDim.x + blockIdx.x) * QB * QB;
  f64x4 c[2][2] = {};
  const double* p = R + (4L * q0 + lane / 16) * D + lane % 16;
#pragma unroll 4
  for (int r = q0; r < q1; ++r, p += 4 * D) {
    const double a0 = p[I * QB], a1 = p[I * QB + 16], b0 = p[J * QB], b1 = p[J * QB + 16];
    c[0][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b0, c[0][0], 0, 0, 0);
    c[0][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b1, c[0][1], 0, 0, 0);
    c[1][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b0, c[1][0], 0, 0, 0);
    c[1][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b1, c[1][1], 0, 0, 0);
  }
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int v = 0; v < 2; ++v)
#pragma unroll
      for (int x = 0; x < 4; ++x)
        out[(16 * u + 4 * x + lane / 16) * QB + 16 * v + lane % 16] = c[u][v][x];
}

// The splits' partial tiles, in order, into (first) or onto the sums.
__global__ void __launch_bounds__(256) quad_fold(const double* __restrict__ part, int first,
                                                 double* __restrict__ q)
{
  for (int x = threadIdx.x; x < QB * QB; x += 256) {
    double* o = q + (long)blockIdx.x * QB * QB + x;
    double sum = first ? 0.0 : *o;
    for (int sp = 0; sp < kQuadSplits; ++sp)
      sum += part[((long)sp * gridDim.x + blockIdx.x) * QB * QB + x];
    *o = sum;
  }
}

// The tiles transformed to nodal values: coefficient k of an element is
// sum_m C[k][m] f(x_m) with C[k][m] = (2 / QB) cos(k theta_m) (half of it for
// k = 0), so Q <- C^T Q C, block by block; the linear block stays.  A tile off
// the diagonal counts twice.
__global__ void __launch_bounds__(256) quad_finish(double* __restrict__ q)
{
  __shared__ double T[QB][QB + 1], C[QB][QB + 1];
  int I, J;
  tile_of(blockIdx.x, I, J);
  const int t = threadIdx.x;
  for (int x = t; x < QB * QB; x += 256) {
    const int k = x / QB, m = x % QB;
    C[k][m] = (k == 0 ? 1.0 : 2.0) / QB * cos(k * (PI_D * (m + 0.5) / QB));
    T[k][m] = q[(long)blockIdx.x * QB * QB + x];
  }
  __syncthreads();
  double o[4];
  if (I > 0) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int m = (t + 256 * u) / QB, j = (t + 256 * u) % QB;
      o[u] = 0.0;
      for (int k = 0; k < QB; ++k) o[u] += C[k][m] * T[k][j];
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 4; ++u) T[(t + 256 * u) / QB][(t + 256 * u) % QB] = o[u];
    __syncthreads();
  }
  if (J > 0) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int m = (t + 256 * u) / QB, j = (t + 256 * u) % QB;
      o[u] = 0.0;
      for (int k = 0; k < QB; ++k) o[u] += T[m][k] * C[k][j];
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 4; ++u) T[(t + 256 * u) / QB][(t + 256 * u) % QB] = o[u];
    __syncthreads();
  }
  const double twice = J < I ? 2.0 : 1.0;
  for (int x = t; x < QB * QB; x += 256)
    q[(long)blockIdx.x * QB * QB + x] = twice * T[x % QB][x / QB];
}

// The rigid-ion curve's values of 64 individuals (one per lane) at the nodes
// of one element (workgroups x < n_act; wave w the nodes w, w + 4, ...), or
// the parameters that enter linearly (x = n_act): src/ri.cu:26-110 in FP64
// from the FP32 parameters.
__global__ void __launch_bounds__(256) ri_values(PopCtl ctl, NodeTable tab)
{
  const int lane = __lane_id(), w = wave_first((int)(threadIdx.x / WAVE));
  const int p = blockIdx.y * WAVE + lane;
  if (p >= tab.ld) return;
  const float* g = ctl.genes + (long)min(p, ctl.P - 1) * ctl.V;
  auto X = [&](int v) { return (double)denormalise(ldu(ctl.pmin, v), ldu(ctl.pmax, v), g[v]); };
  double* out = tab.values + p;
  if ((int)blockIdx.x == tab.n_act) {
    out += (long)2 * tab.b.CE() * QB * tab.ld;
    const double q0 = X(0), rc = X(10), e = erfc(0.2 * rc);
    const double v_rc = e / rc;
    const double dv_rc = -e / (rc * rc) - 0.225675833419103 * exp(-0.04 * rc * rc) / rc;
    for (int t = w; t < 3; t += 4) {
      const double qq = q0 * q0 * (double)RI_K_C * (t == 0 ? 1.0 : t == 1 ? -0.5 : 0.25);
      const double v[4] = {qq, X(3 + 3 * t), qq * dv_rc, qq * (v_rc - dv_rc * rc)};
      for (int u = 0; u < 4; ++u) out[(long)(4 * t + u) * tab.ld] = v[u];
    }
    return;
  }
  const int ce = ldu(tab.act, blockIdx.x).x, t = ce / tab.b.E, el = ce % tab.b.E;
  const double a = X(1 + 3 * t), rate = -1.0 / X(2 + 3 * t);
  double mR = 0.0, kR = 0.0, mA = 0.0, kA = 0.0, r0 = 0.0;
  if (t == 1) {
    const double d0 = X(11), alpha = X(12), S = X(14);
    r0 = X(13);
    if (d0 != 0.0) {
      mR = d0 / (S - 1.0);
      kR = -sqrt(2.0 * S) * alpha;
      mA = S * d0 / (S - 1.0);
      kA = -sqrt(2.0 / S) * alpha;
    }
  }
  double* oU = out + (long)ce * QB * tab.ld;
  double* oD = oU + (long)tab.b.CE() * QB * tab.ld;
  for (int m = w; m < QB; m += 4) {
    const double d = tab.b.d0 + tab.b.len * (el + 0.5 + 0.5 * cos(PI_D * (m + 0.5) / QB));
    double f = 0.0, fp = 0.0;
    if (a != 0.0) {
      f = a * exp(rate * d);
      fp = rate * f;
    }
    if (mA != 0.0 || mR != 0.0) {
      const double R = mR * exp(kR * (d - r0)), A = mA * exp(kA * (d - r0));
      f += R - A;
      fp += kR * R - kA * A;
    }
    oU[(long)m * tab.ld] = f;
    oD[(long)m * tab.ld] = fp;
  }
}

// One row block I of one form for QP individuals per workgroup, the column
// blocks J <= I spread over its four waves: y = sum_J Q_IJ v_J on
// v_mfma_f64_16x16x4_f64 (two products of 16 rows share the values'
// operand), then v_I . y, which is linear in the waves' parts of y.  The last
// workgroup of the QP individuals to finish sums the row blocks in a fixed
// order and writes fitness and terms.
//
// Bound by latency: launching (about 3 us), a wave's operand loads (about 5 us
// here) and the hand-over to the last workgroup (two memory round trips, then
// one for the sums, whose loads are spread over the workgroup; 6 us).  256
// individuals on forms of 17 blocks: 18.3 us with one wave for all column
// blocks of 16 rows, 16.2 us so; with eight waves, whose registers leave one
// workgroup a CU, 21.8 us.  100 individuals on forms of about 46 blocks: 36.2
// us with a unit's workgroups on all XCDs, each fetching the form, 21.8 us so.
constexpr int EVAL_WAVES = 4;

// CHECK: with the individuals that the nodes do not resolve listed (NN2B; rigid
// ion's calls are 0.4 us of 27 shorter without).
template <bool CHECK>
__global__ void __launch_bounds__(EVAL_WAVES * WAVE, 4) quad_eval(PopCtl ctl, QuadEval q)
{
  constexpr int SLICES = EVAL_WAVES * WAVE / QP;
  __shared__ double sh[EVAL_WAVES][QP], fold[3][SLICES][QP], sums[3][QP];
  __shared__ int last;
  const int lane = __lane_id(), w = wave_first((int)(threadIdx.x / WAVE));
  // workgroup -> unit (form and row block) and individuals: the workgroups of
  // a unit run on one XCD (workgroup b on XCD b % 8), one after another, so a
  // tile of Q comes from memory to one L2 once
  const int groups = q.ld / QP;
  const int unit = (int)blockIdx.x / kXcds / groups * kXcds + (int)blockIdx.x % kXcds;
  const int pb = (int)blockIdx.x / kXcds % groups;
  if (CHECK && blockIdx.x == 0 && threadIdx.x == 0) *q.sharp.next = 0u;
  if (unit >= q.units) return;
  const int2 fi = ldu(q.unit, unit);
  const int f = fi.x, I = fi.y;
  const QuadForm F = f == 0 ? q.form[0] : f == 1 ? q.form[1] : q.form[2];
  const long ld = q.ld;
  const int p0 = pb * QP;
  const double* A0 = F.q + quad_tiles(I) * QB * QB + (lane / 16) * QB + lane % 16;
  const double* V = q.values + p0 + lane % 16 + (lane / 16) * ld;
  struct Operands {
    double a[2][8], b[8];
  };
  auto load = [&](int J) {
    Operands o;
    const double* A = A0 + (long)J * QB * QB;
    const double* B = V + (long)ldu(F.vblk, J) * QB * ld;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      o.a[0][k] = A[4 * k * QB];
      o.a[1][k] = A[4 * k * QB + 16];
      o.b[k] = B[4 * k * ld];
    }
    return o;
  };
  f64x4 y[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
  if (w <= I) {
    Operands o = load(w);
    for (int J = w; J <= I; J += EVAL_WAVES) {
      const Operands n = load(min(J + EVAL_WAVES, I));
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        y[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(o.a[0][k], o.b[k], y[0], 0, 0, 0);
        y[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(o.a[1][k], o.b[k], y[1], 0, 0, 0);
      }
      o = n;
    }
  }
  // rows 16 h + 4 x + lane / 16, individual lane % 16
  const double* B = V + (long)ldu(F.vblk, I) * QB * ld;
  double sum = 0.0;
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int x = 0; x < 4; ++x) sum = fma(B[(16 * h + 4 * x) * ld], y[h][x], sum);
  sum += __shfl_xor(sum, 16);
  sum += __shfl_xor(sum, 32);
  if (lane < QP) sh[w][lane] = sum;
  __syncthreads();
  const int t = threadIdx.x;
  const int r0 = f == 0 ? 0 : f == 1 ? q.form[0].nb : q.form[0].nb + q.form[1].nb;
  double* part = q.part + p0;
  if (w == 0) {
    if (lane < QP) {
      double x = 0.0;
#pragma unroll
      for (int u = 0; u < EVAL_WAVES; ++u) x += sh[u][lane];
      cstore(part + (r0 + I) * ld + lane, x);
    }
    publish();
    const unsigned done = wave_atomic_add(&q.done[pb], 1u);
    if (lane == 0) last = done == (unsigned)q.units - 1u;
  }
  __syncthreads();
  if (!last) return;
  observe();
  // row block r of a form in slice r % SLICES, then the slices in order
  const int l = t % QP, sl = t / QP;
  int first = 0;
  float tail[2][kTailSums] = {};
  if (CHECK && t < QP)
#pragma unroll
    for (int k = 0; k < kTailSums; ++k) {
      tail[0][k] = q.sharp.sums[(long)k * ld + p0 + t];
      if (q.sharp.parts > 1) tail[1][k] = q.sharp.sums[(long)(kTailSums + k) * ld + p0 + t];
    }
#pragma unroll
  for (int s = 0; s < 3; ++s) {
    double x = 0.0;
    for (int r = sl; r < q.form[s].nb; r += SLICES) x += cload(part + (first + r) * ld + l);
    fold[s][sl][l] = x;
    first += q.form[s].nb;
  }
  bool resolved = true;
  if (CHECK && t < QP && p0 + t < ctl.P) {
#pragma unroll
    for (int k = 0; k < kTailSums; k += 2) { // (a NaN or an infinite sum: not)
      const float c = tail[0][k] + tail[1][k], size = tail[0][k + 1] + tail[1][k + 1];
      resolved = resolved && c <= q.sharp.limit2 * size && size < __builtin_inff();
    }
  }
  const unsigned long long m = CHECK ? __ballot(!resolved) : 0ull;
  if (w == 0 && m) {
    const int at = (int)wave_atomic_add(q.sharp.count, (unsigned)__popcll(m));
    if (!resolved) q.sharp.list[at + __popcll(m & ((1ull << lane) - 1ull))] = p0 + t;
    if (lane == 0)
      __hip_atomic_store(q.sharp.any, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
  if (t == 0) q.done[pb] = 0u;
  __syncthreads();
  if (t < 3 * QP) {
    double x = 0.0;
    for (int u = 0; u < SLICES; ++u) x += fold[t / QP][u][l];
    // (a sum of squares; rounding may leave it just below zero)
    sums[t / QP][l] = x < 0.0 ? 0.0 : x;
  }
  __syncthreads();
  if (t < QP) {
    const double s[3] = {sums[0][t], sums[1][t], sums[2][t]};
    write_fitness(ctl, p0 + t, s);
  }
}

} // namespace

void launch_bond_range(int B, const float4* bond, unsigned* range, hipStream_t st)
{
  bond_range<<<std::min(1024, (B + 255) / 256), 256, 0, st>>>(B, bond, range);
  GPUGA_HIP(hipGetLastError());
}

void launch_ri_table(int B, const float4* bond, float4* tab, hipStream_t st)
{
  ri_table<<<(B + 255) / 256, 256, 0, st>>>(B, bond, tab);
  GPUGA_HIP(hipGetLastError());
}

void launch_quad_used(const DevSet& s, const QuadBasis& b, int* used, hipStream_t st)
{
  quad_used<<<(s.N + 255) / 256, 256, 0, st>>>(s, b, used);
  GPUGA_HIP(hipGetLastError());
}

static size_t force_lds(const QuadRows& q)
{
  return FORCE_THREADS * sizeof(PairRec) + sizeof(double) * 3 * q.D(2);
}

static size_t quad_energy_lds(const QuadRows& q)
{
  return ENERGY_THREADS * sizeof(PairRec) + sizeof(double) * (q.D(0) + 6 * q.D(1));
}

bool quad_prepare(const QuadRows& q)
{
  const size_t lds[2] = {quad_energy_lds(q), force_lds(q)};
  if (std::max(lds[0], lds[1]) > kRowLds) return false;
  // (a kernel's limit is the process's: the same for every set, of which several
  // may be set up at once on different threads)
  const void* k[2] = {reinterpret_cast<const void*>(&quad_energy_rows),
                      reinterpret_cast<const void*>(&quad_force_rows)};
  for (int i = 0; i < 2; ++i)
    if (lds[i] > 64u * 1024u)
      GPUGA_HIP(hipFuncSetAttribute(k[i], hipFuncAttributeMaxDynamicSharedMemorySize, (int)kRowLds));
  return true;
}

void launch_quad_energy_rows(const DevSet& s, const QuadRows& q, int c0, int c1, double* re,
                             double* rw, hipStream_t st)
{
  quad_energy_rows<<<c1 - c0, ENERGY_THREADS, quad_energy_lds(q), st>>>(s, q, c0, re, rw);
  GPUGA_HIP(hipGetLastError());
}

void launch_quad_force_rows(const DevSet& s, const QuadRows& q, int i0, int i1, double* rf,
                            hipStream_t st)
{
  quad_force_rows<<<i1 - i0, FORCE_THREADS, force_lds(q), st>>>(s, q, i0, rf);
  GPUGA_HIP(hipGetLastError());
}

void launch_quad_gram(const double* R, int rows, int nb, bool first, double* part, double* q,
                      hipStream_t st)
{
  if (rows % 4 != 0) fail("internal: rows of a Gram matrix in fours");
  const long tiles = quad_tiles(nb);
  for (long t = 0; t < tiles; t += kQuadGroup) {
    const unsigned n = (unsigned)std::min<long>(kQuadGroup, tiles - t);
    quad_gram<<<dim3(n, (kQuadSplits + 3) / 4), 256, 0, st>>>(R, rows, nb, (int)t, part);
    GPUGA_HIP(hipGetLastError());
    quad_fold<<<n, 256, 0, st>>>(part, first ? 1 : 0, q + t * QB * QB);
    GPUGA_HIP(hipGetLastError());
  }
}

void launch_quad_finish(int nb, double* q, hipStream_t st)
{
  quad_finish<<<(unsigned)quad_tiles(nb), 256, 0, st>>>(q);
  GPUGA_HIP(hipGetLastError());
}

void launch_ri_values(const PopCtl& ctl, const NodeTable& t, hipStream_t st)
{
  ri_values<<<dim3(t.n_act + 1, (t.ld + WAVE - 1) / WAVE), 256, 0, st>>>(ctl, t);
  GPUGA_HIP(hipGetLastError());
}

void launch_quad_eval(const PopCtl& ctl, const QuadEval& q, hipStream_t st)
{
  const int blocks = (q.units + kXcds - 1) / kXcds * kXcds * (q.ld / QP);
  if (q.sharp.sums) quad_eval<true><<<blocks, EVAL_WAVES * WAVE, 0, st>>>(ctl, q);
  else quad_eval<false><<<blocks, EVAL_WAVES * WAVE, 0, st>>>(ctl, q);
  GPUGA_HIP(hipGetLastError());
}

} // namespace gpuga
