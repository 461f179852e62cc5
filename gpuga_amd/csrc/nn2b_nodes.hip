// NN2B's U and U' at the nodes of the quadratic forms (quadform.h), for every
// individual: the network 1 -> n -> n -> 1 and its derivative
// (src/nn2b.cu:49-78) with the n x n layer on matrix instructions.
//
// A workgroup takes one individual: its genes come in once, by contiguous
// loads (they may be in pinned host memory), and are denormalised into LDS;
// its waves then take the elements, 32 nodes each, all species codes of an
// element in turn.  Weights W1 (output neuron x input neuron) are the A
// operand and the first layer (input neuron x node) is B, so a lane ends with
// half of the output neurons of one node, and the output layer is an in-lane
// sum and one exchange with lane l ^ 32: no pass through LDS, no barrier.
//
// BF16: v_mfma_f32_32x32x16_bf16 with every operand split into two BF16 parts,
// x = hi + lo with hi = bf16(x) and lo = bf16(x - hi) (16 significant bits
// together), a product accumulated as lo lo + lo hi + hi lo + hi hi (n <= 32).
// Otherwise v_mfma_f32_32x32x2_f32.
//
// Each element's last coefficients are taken for the check of SharpSet (quadform.h).
//
// Bound by the 2 n tanh of a node (two transcendental instructions each) and,
// with genes in host memory, by their transfer.  Without the check 256
// individuals, n = 32, 512 nodes took 12.5 us from device memory in BF16 (20.9 us
// with a wave per four elements that gathered its weights and summed the
// output layer through LDS; 14.7 us with the layers' vectors in registers, two
// waves a SIMD), two halves from host memory 19.9 us each, of which the transfer
// alone takes 10; 100 individuals, n = 20, three species codes, FP32: 21.9 us
// (28.9 us with a thread per node on the VALU).  The check adds 1.5 and 0.6 us
// (the magnitudes two instructions a neuron, the coefficients a chain of
// exchanges; through LDS instead of DPP 0.5 us more).  BF16 costs what FP32
// does here: its splits take the VALU as long as FP32 products the matrix unit.
// (Its tanh's derivative not as 1 - t t, which loses it for saturated neurons:
// the check then takes the rounding of 1 in 100 networks of 6 neurons for
// sharpness.)
#include "quadform.h"

namespace gpuga {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

// (x, y) = hi + lo, both round-to-nearest-even BF16, into elements j, j + 1 of
// two operands
__device__ inline void split_bf16(float x, float y, bf16x8& hi, bf16x8& lo, int j)
{
  const bf16x2 h = __builtin_convertvector((f32x2){x, y}, bf16x2);
  const bf16x2 l = __builtin_convertvector((f32x2){x - (float)h[0], y - (float)h[1]}, bf16x2);
  hi[j] = h[0];
  hi[j + 1] = h[1];
  lo[j] = l[0];
  lo[j + 1] = l[1];
}

// C += A B with split operands (smallest terms first; the matrix unit has room
// for lo lo as well)
__device__ inline f32x16 mfma4(const bf16x8& ah, const bf16x8& al, const bf16x8& bh,
                               const bf16x8& bl, f32x16 c)
{
  c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al, bl, c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al, bh, c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, bl, c, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, bh, c, 0, 0, 0);
}

// Four values of each lane summed over its 32 lanes: lane c returns the sum of
// value 2 (c % 2) + c / 2 % 2.
template <int CTRL>
__device__ inline float dpp(float x)
{
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), CTRL, 0xf, 0xf, true));
}
__device__ inline float sums_of_four(const float (&v)[4], int c)
{
  constexpr int XOR1 = 0xb1, XOR2 = 0x4e, ROR4 = 0x124, ROR8 = 0x128; // in rows of 16
  const bool a = c & 1, b = c & 2;
  const float x = (a ? v[2] : v[0]) + dpp<XOR1>(a ? v[0] : v[2]);
  const float y = (a ? v[3] : v[1]) + dpp<XOR1>(a ? v[1] : v[3]);
  float s = (b ? y : x) + dpp<XOR2>(b ? x : y);
  s += dpp<ROR4>(s);
  s += dpp<ROR8>(s);
  return s + __shfl_xor(s, 16);
}

// KS: input neurons per half-wave (n <= 2 KS); NB: blocks of 32 output
// neurons.  Half-wave h holds the input neurons m(s) = 2 s + h (FP32: one pair
// per instruction) or 16 (s / 8) + 8 h + s % 8 (BF16: eight per operand), and
// the output neurons 32 b + 8 (r / 4) + 4 h + r % 4.  W1's operands are in
// registers; the layers' vectors are read from LDS at each use (broadcasts),
// so that four waves fit a SIMD.
template <bool BF16, int KS, int NB, int WAVES>
__global__ void __launch_bounds__(WAVES * WAVE) nn2b_nodes(PopCtl ctl, int n, int species,
                                                           NodeTable tab, int first)
{
  __shared__ float4 l1[2 * KS];      // w0, b0, ws of an input neuron
  __shared__ float2 l2[NB * 32];     // b1, w2 of an output neuron
  __shared__ float bias2;
  extern __shared__ float w1[];      // [n][n + 1] (rows off a power of two: banks)
  const int p = first + blockIdx.y;
  const int V = ctl.V, t = threadIdx.x;
  const float* genes = ctl.genes + (size_t)min(p, ctl.P - 1) * V;
  const int lane = __lane_id(), col = lane & 31, half = lane >> 5;
  // the check that the nodes resolve the curve (SharpSet): this lane's factors,
  // and its sums over the energy, then the force configurations' pairs
  static_assert(QTAIL == 4, "sums_of_four");
  float tf[QTAIL], sums[4] = {};
#pragma unroll
  for (int k = 0; k < QTAIL; ++k) tf[k] = tab.tail[k * QB + col];
  constexpr int T = WAVES * WAVE, LOADS = 4;
  for (int k = t; k < 2 * KS; k += T) l1[k] = make_float4(0, 0, 0, 0);
  for (int k = t; k < NB * 32; k += T) l2[k] = make_float2(0, 0);
  __syncthreads();
  // Four loads in flight per thread: from host memory a round trip takes
  // microseconds.
  for (int v0 = t; v0 < V; v0 += LOADS * T) {
    float g[LOADS], lo[LOADS], hi[LOADS];
#pragma unroll
    for (int k = 0; k < LOADS; ++k) {
      const int v = min(v0 + k * T, V - 1);
      g[k] = genes[v];
      lo[k] = ctl.pmin[v];
      hi[k] = ctl.pmax[v];
    }
#pragma unroll
    for (int k = 0; k < LOADS; ++k) {
      const int v = v0 + k * T;
      if (v >= V) break;
      const float x = denormalise(lo[k], hi[k], g[k]);
      const int block = v / n, m = v - block * n;
      if (block < 1) l1[m].x = x;
      else if (block < 2) l1[m].y = x;
      else if (block < n + 2) w1[(block - 2) * (n + 1) + m] = x;
      else if (block < n + 3) l2[m].x = x;
      else if (block < n + 4) l2[m].y = x;
      else if (v == n * (n + 4)) bias2 = x;
      else l1[v - n * (n + 4) - 1].z = x;
    }
  }
  __syncthreads();
  auto m_of = [&](int s) { return BF16 ? 16 * (s / 8) + 8 * half + s % 8 : 2 * s + half; };
  auto A = [&](int row, int s) {
    const int m = m_of(s);
    return m < n && row < n ? w1[row * (n + 1) + m] : 0.0f;
  };
  float a[BF16 ? 1 : NB][BF16 ? 1 : KS];
  bf16x8 ah[BF16 ? KS / 8 : 1], al[BF16 ? KS / 8 : 1];
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    if constexpr (BF16) {
      if (s % 2 == 0) split_bf16(A(col, s), A(col, s + 1), ah[s / 8], al[s / 8], s % 8);
    } else {
#pragma unroll
      for (int b = 0; b < NB; ++b) a[b][s] = A(32 * b + col, s);
    }
  }

  const int E = tab.b.E, CE = tab.b.CE();
  for (int i = blockIdx.x * WAVES + wave_first(t / WAVE); i < tab.n_act;
       i += gridDim.x * WAVES) {
    const int2 el = ldu(tab.act, i); // element, mask of its codes
    const float d = node_at(tab.b, el.x, col);
    float base = 0.0f; // code 0's U (half 0) or U' (half 1) at the node
    for (int code = 0; code < tab.b.codes; ++code) {
      if (!((el.y >> code) & 1)) continue;
      const float2 pairs = ldu(tab.pairs, code * E + el.x);
      f32x16 z[NB] = {}, zd[NB] = {};
      auto tanh_s = [](float x, float& t, float& s) {
        if constexpr (BF16) ftanh_sech2(x, t, s); // (the operands' 16 bits set the error)
        else tanh_sech2(x, t, s);
      };
      auto layer1 = [&](int s, float& x, float& y) {
        const float4 l = l1[m_of(s)];
        // the species-pair input as a shift of the bias
        const float bias = species ? l.y - l.z * (float)code : l.y;
        float sg;
        tanh_s(l.x * d - bias, x, sg);
        y = sg * l.x;
      };
      if constexpr (BF16) {
#pragma unroll
        for (int k = 0; k < KS / 8; ++k) {
          bf16x8 xh, xl, yh, yl;
#pragma unroll
          for (int j = 0; j < 8; j += 2) {
            float x[2], y[2];
            layer1(8 * k + j, x[0], y[0]);
            layer1(8 * k + j + 1, x[1], y[1]);
            split_bf16(x[0], x[1], xh, xl, j);
            split_bf16(y[0], y[1], yh, yl, j);
          }
          z[0] = mfma4(ah[k], al[k], xh, xl, z[0]);
          zd[0] = mfma4(ah[k], al[k], yh, yl, zd[0]);
        }
      } else {
#pragma unroll
        for (int s = 0; s < KS; ++s) {
          float x, y;
          layer1(s, x, y);
#pragma unroll
          for (int b = 0; b < NB; ++b) {
            z[b] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[b][s], x, z[b], 0, 0, 0);
            zd[b] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[b][s], y, zd[b], 0, 0, 0);
          }
        }
      }
      float u = 0.0f, g = 0.0f, um = 0.0f, gm = 0.0f;
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float2 l = l2[32 * b + 8 * (r >> 2) + 4 * half + (r & 3)];
          float x, sg;
          tanh_s(z[b][r] - l.x, x, sg);
          u = fmaf(l.y, x, u);
          g = fmaf(l.y * sg, zd[b][r], g);
          um = fmaf(__builtin_fabsf(l.y), __builtin_fabsf(x), um);
          gm = fmaf(__builtin_fabsf(l.y * sg), __builtin_fabsf(zd[b][r]), gm);
        }
      // half 0 takes U, half 1 takes U'
      float mine = (half ? g : u) + __shfl_xor(half ? u : g, 32);
      float mag = (half ? gm : um) + __shfl_xor(half ? um : gm, 32);
      if (!half) {
        mine -= bias2;
        mag += __builtin_fabsf(bias2);
      } else { // (tanh_s: two quarters)
        mine *= 16.0f;
        mag *= 16.0f;
      }
      // one of the last coefficients in each lane
      const float c =
        sums_of_four({tf[0] * mine, tf[1] * mine, tf[2] * mine, tf[3] * mine}, col);
      sums[0] = fmaf(pairs.x * c, c, sums[0]);
      sums[1] = fmaf(pairs.x * mag, mag, sums[1]);
      sums[2] = fmaf(pairs.y * c, c, sums[2]);
      sums[3] = fmaf(pairs.y * mag, mag, sums[3]);
      if (code == 0) base = mine;
      // (the codes above 0 as differences from code 0, quadform.h)
      tab.values[((long)(half * CE + code * E + el.x) * QB + col) * tab.ld + p] =
        code == 0 ? (double)mine : (double)mine - (double)base;
    }
  }
  __shared__ float all[WAVES][kTailSums];
  const float sum = sums_of_four(sums, col);
  const int k = 2 * (col & 1) + (col >> 1); // energy: U; virial and force: U'
  if (col < 4 && k + 2 * half < kTailSums && (half || k < 2)) all[t / WAVE][k + 2 * half] = sum;
  __syncthreads();
  if (t < kTailSums) {
    float x = 0.0f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) x += all[w][t];
    tab.sums[((long)blockIdx.x * kTailSums + t) * tab.ld + p] = x;
  }
}

// Populations from 128 on: one workgroup an individual, so that the genes are read
// once; fewer leave CUs idle, and their elements go over two workgroups.
template <bool BF16, int KS, int NB, int WAVES>
void launch(const PopCtl& ctl, const NN2BGrid& g, const NodeTable& t, int first, int count,
            hipStream_t st)
{
  const size_t lds = sizeof(float) * g.n * (g.n + 1);
  const int species = g.codes > 1 ? 1 : 0;
  if (nn2b_node_parts(ctl.P) == 1)
    nn2b_nodes<BF16, KS, NB, WAVES>
      <<<dim3(1, count), WAVES * WAVE, lds, st>>>(ctl, g.n, species, t, first);
  else
    nn2b_nodes<BF16, KS, NB, WAVES / 2>
      <<<dim3(2, count), WAVES / 2 * WAVE, lds, st>>>(ctl, g.n, species, t, first);
}

} // namespace

void launch_nn2b_nodes(const PopCtl& ctl, const NN2BGrid& g, const NodeTable& t, int first,
                       int count, hipStream_t st)
{
  if (g.n > 64) fail("NN2B supports at most 64 neurons");
  if (g.bf16 && g.n <= 16) launch<true, 8, 1, 16>(ctl, g, t, first, count, st);
  else if (g.bf16 && g.n <= 32) launch<true, 16, 1, 16>(ctl, g, t, first, count, st);
  else if (g.n <= 16) launch<false, 8, 1, 16>(ctl, g, t, first, count, st);
  else if (g.n <= 24) launch<false, 12, 1, 16>(ctl, g, t, first, count, st);
  else if (g.n <= 32) launch<false, 16, 1, 16>(ctl, g, t, first, count, st);
  else launch<false, 32, 2, 8>(ctl, g, t, first, count, st);
  GPUGA_HIP(hipGetLastError());
}

} // namespace gpuga
