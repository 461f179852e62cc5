// Minimal Tersoff population kernel for sets with five to twenty neighbours
// within R2 (outer radii past the second shell, dense structures).
//
// The bond loops run over unordered pairs of an atom's bonds.  With c the
// cosine of a pair's angle, x = c - h, S = fc_u fc_v (A_u + A_v) x and
// d c / d r_u = (e_v - c e_u) / d_u (e: unit vectors),
//   zeta_u = beta sum_v fc_v x^2
//   f_u    = coef_u r_u - beta / d_u (sum_v S e_v - e_u sum_v S c)
// (src/minimal_tersoff.cu:147-185, 250-307), so a pair's cosine is all its
// geometry: x and S are computed once for both bonds, and an atom's record
// holds one cosine per pair instead of two (cosine, gradient) rows.
#include <type_traits>

#include "kernels.h"
#include "population.h"
#include "tersoff_math.h"

namespace gpuga {

// Record of M bond slots, in float4: header {neighbours, unlike-type mask,
// first bond}, M bonds (r, d), M unit vectors (e, 1/d), M reverse-bond
// indices, then the cosines of the pairs (u, v), u < v, row v after row
// v - 1, each row padded to whole float4.
__host__ __device__ constexpr int shell_cos(int v) // float offset of row v
{
  int o = 0;
  for (int w = 1; w < v; ++w) o += (w + 3) / 4 * 4;
  return o;
}
__host__ __device__ constexpr int shell_first_cos(int M) { return 1 + 2 * M + M / 4; }
__host__ __device__ constexpr int shell_stride(int M)
{
  return shell_first_cos(M) + shell_cos(M) / 4;
}

// f(0), ..., f(N - 1) with the index as a constant.
template <int N, int I = 0, class F>
__device__ __forceinline__ void upto(F&& f)
{
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    upto<N, I + 1>(f);
  }
}

// The per-bond values of an atom in registers, every loop unrolled, left by a
// scalar branch after the atom's last bond: an atom with fewer neighbours
// than M does no padded work.  The record comes through LDS (the next atom's
// loads in flight during this one): its broadcast reads return in order and
// are waited for one by one, and the unit vectors do not fill the scalar
// registers.  What the pair loops do not touch (fc' / d, the pair part) waits
// in LDS rows, and a scheduling barrier every four pairs keeps their reads from
// moving ahead of one another, so that two waves fit a SIMD.
//
// Bound by the VALU (20 instructions a pair, about 60 a bond) at two waves a
// SIMD.  The looped kernel, which takes any number of neighbours with its
// per-bond values in LDS and every load waited for in turn, took 332 us on
// 6 400 atoms with up to 18 neighbours (15.6 on average), two lane blocks;
// this form 112 us (129 us with the record in scalar registers; twice as many
// registers, one wave a SIMD, without the barriers: 180 us).  On sets of 12, 14
// and 16 neighbours it is 4 to 11 times as fast as bodies of ordered pairs
// with guards, which spilled to scratch (5 400 atoms of 8.3 neighbours, 200
// individuals: a call of 454 -> 113 us).
template <int M, bool TWO>
struct TersoffShell {
  static constexpr int kWaves = 2, kWavesPacked = 2;
  static constexpr bool kSubset = false;
  static constexpr bool kForcePass = true;
  static constexpr int kFoldValues = 24;
  static constexpr bool kPacked = false;
  static constexpr bool kHeaderAhead = false;
  using Lane = TLane;
  using Extra = const float4*;
  static constexpr int RS = shell_stride(M);

  __device__ static Lane make(const PopCtl& ctl, int p) { return tersoff_make<TWO>(ctl, p); }

  // R: the atom's record in LDS; FCP, PF: LDS rows of the wave's lanes for the
  // values that the pair loops do not touch (fc' / d, the pair part of f_ij)
  template <bool FORCE>
  __device__ static void atom(const DevSet& s, const float4* R, float* FCP, float* PF,
                              const TLane& q, int i, int nn, int unl, float* fblk, int lane,
                              Acc& acc)
  {
    const float* C = reinterpret_cast<const float*>(R + shell_first_cos(M));
    // (an empty asm between the passes: the compiler would keep the first
    // pass's reads of the record for the second one)
    constexpr int STEP = 4; // pairs between scheduling barriers
    auto pass = [] { asm volatile("" ::: "memory"); };
    TSets sets;
    if constexpr (TWO) sets = tersoff_sets(q);
    float fc[M], z[M];
    upto<M>([&](auto U) {
      constexpr int u = U;
      if (u < nn) {
        float fcp;
        tersoff_fc(q, R[1 + u].w, fc[u], fcp);
        FCP[u * WAVE + lane] = fcp * R[1 + M + u].w;
        z[u] = 0.0f;
      }
    });
    upto<M>([&](auto V) {
      constexpr int v = V;
      if (v > 0 && v < nn)
        upto<v>([&](auto U) {
          constexpr int u = U;
          const float x = C[shell_cos(v) + u] - q.h;
          const float x2 = x * x;
          z[u] = fmaf(fc[v], x2, z[u]);
          z[v] = fmaf(fc[u], x2, z[v]);
        });
    });
    pass();
    float e = 0.0f, B[M], cx[M], cy[M], cz[M], m[M], ds[M];
    upto<M>([&](auto U) {
      constexpr int u = U;
      if (u < nn) {
        float b, bp, fr, frp, fa, fap;
        tersoff_bond_order(q, q.beta * z[u], b, bp);
        const float d = R[1 + u].w;
        if constexpr (TWO) tersoff_pair_sel(sets, (unl >> u) & 1, d, fr, frp, fa, fap);
        else tersoff_pair(q, 0, d, fr, frp, fa, fap);
        const float rep = fr - b * fa;
        e = fmaf(fc[u], rep, e);
        PF[u * WAVE + lane] = fmaf(FCP[u * WAVE + lane], rep, fc[u] * (frp - b * fap) * R[1 + M + u].w);
        B[u] = bp * fa * fc[u];
        cx[u] = cy[u] = cz[u] = m[u] = ds[u] = 0.0f;
      }
    });
    pass();
    upto<M>([&](auto V) {
      constexpr int v = V;
      if (v > 0 && v < nn) {
        const float4 ev = R[1 + M + v];
        upto<v>([&](auto U) {
          constexpr int u = U;
          const float c = C[shell_cos(v) + u], x = c - q.h, x2 = x * x;
          const float4 eu = R[1 + M + u];
          const float S = fmaf(fc[v], B[u], fc[u] * B[v]) * x;
          const float Sc = S * c;
          cx[u] = fmaf(S, ev.x, cx[u]);
          cy[u] = fmaf(S, ev.y, cy[u]);
          cz[u] = fmaf(S, ev.z, cz[u]);
          cx[v] = fmaf(S, eu.x, cx[v]);
          cy[v] = fmaf(S, eu.y, cy[v]);
          cz[v] = fmaf(S, eu.z, cz[v]);
          m[u] += Sc;
          m[v] += Sc;
          ds[u] = fmaf(B[v], x2, ds[u]);
          ds[v] = fmaf(B[u], x2, ds[v]);
          if constexpr (u % STEP == STEP - 1) __builtin_amdgcn_sched_barrier(0);
        });
      }
    });
    pass();
    float wxx = 0, wyy = 0, wzz = 0, wxy = 0, wyz = 0, wzx = 0;
    upto<M>([&](auto U) {
      constexpr int u = U;
      if (u < nn) {
        const float4 r = R[1 + u], eu = R[1 + M + u];
        const float coef = 0.5f * (PF[u * WAVE + lane] - FCP[u * WAVE + lane] * (q.beta * ds[u]));
        const float hc = q.beta * eu.w;
        const float fx = fmaf(coef, r.x, -hc * fmaf(-m[u], eu.x, cx[u]));
        const float fy = fmaf(coef, r.y, -hc * fmaf(-m[u], eu.y, cy[u]));
        const float fz = fmaf(coef, r.z, -hc * fmaf(-m[u], eu.z, cz[u]));
        if (FORCE) {
          const int rb = wave_first(reinterpret_cast<const record_word*>(R + 1 + 2 * M)[u]);
          float* o = fblk + (size_t)rb * 3 * WAVE + lane;
          cstore(o, fx);
          cstore(o + WAVE, fy);
          cstore(o + 2 * WAVE, fz);
          wxx += fx;
          wyy += fy;
          wzz += fz;
        } else {
          wxx -= r.x * fx;
          wyy -= r.y * fy;
          wzz -= r.z * fz;
          wxy -= r.x * fy;
          wyz -= r.y * fz;
          wzx -= r.z * fx;
        }
      }
    });
    if (FORCE) {
      float* o = fblk + ((size_t)s.bond_force + i) * 3 * WAVE + lane;
      cstore(o, wxx);
      cstore(o + WAVE, wyy);
      cstore(o + 2 * WAVE, wzz);
    } else {
      acc.v[0] += (double)(0.5f * e);
      acc.v[1] += (double)wxx;
      acc.v[2] += (double)wyy;
      acc.v[3] += (double)wzz;
      acc.v[4] += (double)wxy;
      acc.v[5] += (double)wyz;
      acc.v[6] += (double)wzx;
    }
  }

  // A record spread over the wave, word 64 k + l in register k of lane l.
  static constexpr int RW = RS * 4, NW = (RW + WAVE - 1) / WAVE;
  struct Spread {
    int w[NW];
  };
  __device__ static Spread spread_load(const float4* rec, int i)
  {
    const int* w = reinterpret_cast<const int*>(rec + (long)i * RS);
    Spread v;
#pragma unroll
    for (int k = 0; k < NW; ++k) v.w[k] = w[min(WAVE * k + (int)__lane_id(), RW - 1)];
    return v;
  }
  __device__ static void spread_store(float4* buf, const Spread& v)
  {
    record_word* w = reinterpret_cast<record_word*>(buf);
#pragma unroll
    for (int k = 0; k < NW; ++k)
      if (WAVE * k + (int)__lane_id() < RW) w[WAVE * k + __lane_id()] = v.w[k];
  }

  __device__ static void chunk(const DevSet& s, const TLane& q, const WorkItem& it,
                               const PopCtl& ctl, const float4* rec, Acc& acc)
  {
    __shared__ float4 buf[256 / WAVE][RS];
    __shared__ float side[256 / WAVE][2][M * WAVE];
    const int lane = __lane_id(), w = wave_first((int)(threadIdx.x / WAVE));
    float4* R = buf[w];
    Spread v = spread_load(rec, it.a0);
    auto run = [&](auto force) {
      constexpr bool F = decltype(force)::value;
      float* fblk = F ? ctl.bondf + (size_t)it.k * ctl.B_force * 3 * WAVE : nullptr;
      for (int i = it.a0; i < it.a1; ++i) {
        const int nn = __builtin_amdgcn_readlane(v.w[0], 0);
        const int unl = TWO ? __builtin_amdgcn_readlane(v.w[0], 1) : 0;
        spread_store(R, v); // (LDS operations of a wave stay in order)
        v = spread_load(rec, min(i + 1, it.a1 - 1));
        atom<F>(s, R, side[w][0], side[w][1], q, i, nn, unl, fblk, lane, acc);
      }
    };
    if (it.c < s.Nc_force) run(std::true_type{});
    else run(std::false_type{});
  }

  // F_i = sum_j (f_ij - f_ji), then sum_i |F_i - F_ref,i|^2
  // (src/minimal_tersoff.cu:355-383), an atom's loads all in flight together
  __device__ static double force_pass(const DevSet& s, const PopCtl& ctl, const float4* rec,
                                      int a0, int a1, int k, int lane)
  {
    const float* fblk = ctl.bondf + (size_t)k * ctl.B_force * 3 * WAVE + lane;
    const long N = s.N;
    double err = 0.0;
    for (int i = a0; i < a1; ++i) {
      const int* H = reinterpret_cast<const int*>(rec + (long)i * RS);
      const int nn = ldu(H, 0), b0 = ldu(H, 2);
      const float* own = fblk + ((size_t)s.bond_force + i) * 3 * WAVE;
      float fx = cload(own), fy = cload(own + WAVE), fz = cload(own + 2 * WAVE);
#pragma unroll
      for (int u = 0; u < M; ++u) {
        const bool on = u < nn;
        const float* r = on ? fblk + (size_t)(b0 + u) * 3 * WAVE : own;
        const float rx = cload(r), ry = cload(r + WAVE), rz = cload(r + 2 * WAVE);
        fx -= on ? rx : 0.0f;
        fy -= on ? ry : 0.0f;
        fz -= on ? rz : 0.0f;
      }
      const float dx = fx - ldu(s.force_ref, i), dy = fy - ldu(s.force_ref, i + N),
                  dz = fz - ldu(s.force_ref, i + 2 * N);
      err += (double)dx * dx + (double)dy * dy + (double)dz * dz;
    }
    return err;
  }
};

// One thread per atom fills its record from the list's bond and triplet
// tables (unit vectors in FP64, rounded once).
__global__ void __launch_bounds__(64) shell_records(int N, int M, LoopTab t, float4* rec)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= N) return;
  float4* R = rec + (long)i * shell_stride(M);
  const int nn = t.nn[i], b0 = t.b0[i];
  const float4* T = t.tri + t.tri0[i];
  int unl = 0;
  int* rev = reinterpret_cast<int*>(R + 1 + 2 * M);
  float* C = reinterpret_cast<float*>(R + shell_first_cos(M));
  for (int u = 0; u < M; ++u) {
    float4 r = make_float4(0, 0, 0, 1), e = r;
    if (u < nn) {
      r = t.bond[b0 + u];
      const double di = 1.0 / (double)r.w;
      e = make_float4((float)(r.x * di), (float)(r.y * di), (float)(r.z * di), (float)di);
      if (t.ptype[b0 + u] & 1) unl |= 1 << u;
    }
    R[1 + u] = r;
    R[1 + M + u] = e;
    rev[u] = u < nn ? t.rev[b0 + u] : 0;
    for (int w = 0; w < (u + 3) / 4 * 4; ++w)
      C[shell_cos(u) + w] = u < nn && w < u ? T[w * nn + u].x : 0.0f;
  }
  R[0] = make_float4(__int_as_float(nn), __int_as_float(unl), __int_as_float(b0), 0.0f);
}

// bond slots of the kernel that takes max_nn neighbours; 0: none
int tersoff_shell_slots(int max_nn)
{
  for (int M : {8, 16, 20})
    if (max_nn <= M) return M;
  return 0;
}

size_t tersoff_shell_floats4(int N, int M) { return (size_t)N * shell_stride(M); }

void build_shell_records(int N, int M, const LoopTab& t, float4* rec, hipStream_t st)
{
  shell_records<<<(N + 63) / 64, 64, 0, st>>>(N, M, t, rec);
  GPUGA_HIP(hipGetLastError());
}

template <class F>
static void shell_kernel(int M, bool two, F&& f)
{
  switch (M * 2 + (two ? 1 : 0)) {
  case 16: f(population_kernel<TersoffShell<8, false>>); break;
  case 17: f(population_kernel<TersoffShell<8, true>>); break;
  case 32: f(population_kernel<TersoffShell<16, false>>); break;
  case 33: f(population_kernel<TersoffShell<16, true>>); break;
  case 40: f(population_kernel<TersoffShell<20, false>>); break;
  case 41: f(population_kernel<TersoffShell<20, true>>); break;
  default: fail("internal: no Tersoff kernel for this neighbour bound");
  }
}

void launch_tersoff_shell_population(const PopCtl& ctl, const DevSet& s, int M, const float4* rec,
                                     int grid, int block, hipStream_t st)
{
  shell_kernel(M, ctl.V == 13, [&](auto* k) { k<<<grid, block, 0, st>>>(ctl, s, rec); });
  GPUGA_HIP(hipGetLastError());
}

int tersoff_shell_occupancy(int M, bool two, int block)
{
  int n = 0;
  shell_kernel(M, two, [&](auto* k) {
    GPUGA_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k, block, 0));
  });
  return n;
}

} // namespace gpuga
