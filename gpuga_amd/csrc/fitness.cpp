// Fitness evaluator host code: set-up, plug-ins, population plans, predict.
#include "fitness.h"
#include "noalloc.h"

#include <sys/mman.h>
#include <unistd.h>

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstring>
#include <numeric>

namespace gpuga {

int tersoff_population_occupancy(bool two, bool pack, int block);

// Neighbours within R2 the looped Tersoff population kernel takes (its LDS
// rows: 4 x 64 lanes x 4 B per neighbour and wave, 64 KiB at this bound).
constexpr int kLoopMaxNeighbors = 64;
int ri_population_occupancy(int block);
int nn2b_population_occupancy(int block);

// ------------------------------------------------------------ plug-ins

namespace {

// Host denormalisation with float arithmetic and no fused multiply-add,
// exactly as src/fitness.cu:319-324 (this file is compiled with
// -ffp-contract=off).
void denormalise_host(const PotentialSpec& s, const float* genes, float* out)
{
  for (int m = 0; m < s.V; ++m) {
    const float a = s.pmin[m];
    const float b = s.pmax[m] - a;
    const float bx = b * genes[m];
    out[m] = a + bx;
  }
}

class TersoffPotential : public Potential {
public:
  explicit TersoffPotential(int num_types) : num_types_(num_types) {}
  void initialize(int, int) override {}
  void init_bonds(int B)
  {
    b_.resize(std::max(B, 1));
    bp_.resize(std::max(B, 1));
    f12_.resize(3 * (size_t)std::max(B, 1));
  }
  void update_potential(const std::vector<float>& p) override
  {
    q_ = tersoff_params(num_types_, p.data());
  }
  void find_force(const DevSet& s, float* f, float* virial, float* pe, hipStream_t st,
                  float* ws) override
  {
    // workspace: b and b' per bond, then f_ij (3 per bond)
    const size_t B = b_.size();
    if (ws) launch_tersoff_plain(s, q_, ws, ws + B, ws + 2 * B, f, virial, pe, st);
    else launch_tersoff_plain(s, q_, b_.get(), bp_.get(), f12_.get(), f, virial, pe, st);
  }
  size_t workspace_floats() const override { return 5 * b_.size(); }

private:
  int num_types_;
  TersoffParams q_{};
  DeviceBuffer<float> b_, bp_, f12_;
};

class RIPotential : public Potential {
public:
  explicit RIPotential(const float4* tab) : tab_(tab) {}
  void initialize(int, int) override {}
  void update_potential(const std::vector<float>& p) override { q_ = ri_params(p.data()); }
  void find_force(const DevSet& s, float* f, float* virial, float* pe, hipStream_t st,
                  float*) override
  {
    launch_ri_plain(s, q_, tab_, f, virial, pe, st);
  }

private:
  const float4* tab_;
  RIParams q_{};
};

class NN2BPotential : public Potential {
public:
  // species: the first layer also takes the pair's species code
  NN2BPotential(int n, bool species) : n_(n), species_(species) {}
  void initialize(int, int) override { w_.resize(n_ * (n_ + 4) + 1 + (species_ ? n_ : 0)); }
  void update_potential(const std::vector<float>& p) override
  {
    host_ = p;
    dirty_ = true;
  }
  void find_force(const DevSet& s, float* f, float* virial, float* pe, hipStream_t st,
                  float*) override
  {
    if (dirty_) {
      w_.upload(host_, st);
      dirty_ = false;
    }
    launch_nn2b_plain(s, n_, species_, w_.get(), f, virial, pe, st);
  }

private:
  int n_;
  bool species_;
  std::vector<float> host_;
  bool dirty_ = false;
  DeviceBuffer<float> w_;
};

} // namespace

std::unique_ptr<Potential> make_potential(const PotentialSpec& spec, const DeviceSet& ds)
{
  switch (spec.type) {
  case POT_TERSOFF1:
  case POT_TERSOFF2: {
    auto p = std::make_unique<TersoffPotential>(spec.type == POT_TERSOFF2 ? 2 : 1);
    p->init_bonds((int)ds.bond.size());
    return p;
  }
  case POT_RI: return std::make_unique<RIPotential>(ds.ri_tab.get());
  case POT_NN2B:
  case POT_NN2B_SPECIES: {
    auto p = std::make_unique<NN2BPotential>(spec.num_neurons, spec.type == POT_NN2B_SPECIES);
    p->initialize(0, 0);
    return p;
  }
  }
  fail("unsupported potential type.");
}

size_t DeviceSet::bytes() const
{
  return Na.bytes() + Na_sum.bytes() + type.bytes() + nn.bytes() + bond0.bytes() + nl.bytes() +
         rev.bytes() + ptype.bytes() + tri0.bytes() + bond.bytes() + tri.bytes() +
         ri_tab.bytes() + rec.bytes() + mom.bytes() + shell_rec.bytes() + pair_hdr.bytes() +
         pair_tab.bytes() + pe_ref.bytes() + virial_ref.bytes() + force_ref.bytes() + p_nn.bytes() + p_b0.bytes() + p_nl.bytes() +
         p_rev.bytes() + p_ptype.bytes() + p_tri0.bytes() + p_bond.bytes() + p_tri.bytes() +
         ri_cconst.bytes() + ri_fconst.bytes();
}

// ------------------------------------------------------------ set-up

Fitness::Fitness(const std::string& dir, const FitnessOptions& opt) : opt_(opt)
{
  spec_ = read_potential(dir);
  ts_ = read_train(dir);
  setup();
}

Fitness::Fitness(const PotentialSpec& spec, TrainSet ts, const FitnessOptions& opt)
  : opt_(opt), spec_(spec), ts_(std::move(ts))
{
  setup();
}

Fitness::~Fitness()
{
  plans_.clear();
  if (ev0_) (void)hipEventDestroy(ev0_);
  if (ev1_) (void)hipEventDestroy(ev1_);
  for (auto e : ev_half_)
    if (e) (void)hipEventDestroy(e);
  if (stream_) (void)hipStreamDestroy(stream_);
}

void Fitness::device_geometry(std::vector<float4>& bond, std::vector<float4>& tri,
                              std::vector<float4>& rec)
{
  hipStream_t st = stream_;
  // with 5 to 16 neighbours the population kernel has records of its own, and
  // these are built to be looked at
  const bool tersoff = spec_.type == POT_TERSOFF1 || spec_.type == POT_TERSOFF2;
  const int M = tersoff ? record_slots(population_neighbors().max_nn) : 0;
  DeviceBuffer<float4> built;
  if (shell_M_ > 0 && M > 0) {
    built.resize((size_t)ts_.N * record_floats4(M));
    const DeviceNeighbors pd = build_population_tables();
    build_records_device(ts_.N, M, pd, loop_.ptype, loop_.bond, loop_.tri, built.get(), st);
    GPUGA_HIP(hipStreamSynchronize(st));
    drop_population_tables();
  }
  const DeviceBuffer<float4>& r = built.size() > 0 ? built : ds_.rec;
  bond.resize(ds_.bond.size());
  tri.resize(ds_.tri.size());
  rec.resize(r.size());
  ds_.bond.download(bond.data(), bond.size(), st);
  ds_.tri.download(tri.data(), tri.size(), st);
  r.download(rec.data(), rec.size(), st);
  GPUGA_HIP(hipStreamSynchronize(st));
}

DeviceNeighbors Fitness::device_neighbors() const
{
  DeviceNeighbors dn;
  dn.NN = ds_.nn.get();
  dn.start = ds_.bond0.get();
  dn.NL = ds_.nl.get();
  dn.rev = ds_.rev.get();
  dn.tri0 = ds_.tri0.get();
  dn.total = nl_.total;
  return dn;
}

// Tables of the list the Tersoff population kernel reads, in loop_: the full
// ones, or the pruned list's (geometry bit-identical to the full tables' entries
// for the same bonds).
DeviceNeighbors Fitness::build_population_tables()
{
  hipStream_t st = stream_;
  const NeighborList& pn = population_neighbors();
  DeviceNeighbors pd = device_neighbors();
  loop_.ptype = ds_.ptype.get();
  loop_.bond = ds_.bond.get();
  loop_.tri = ds_.tri.get();
  if (pruned_) {
    long long tri_total = 0;
    const std::vector<int> t0 = triplet_offsets(pn, &tri_total);
    ds_.p_nn.upload(pn.NN, st);
    ds_.p_b0.upload(pn.start, st);
    ds_.p_nl.upload(pn.NL.empty() ? std::vector<int>{0} : pn.NL, st);
    ds_.p_rev.upload(pn.rev.empty() ? std::vector<int>{0} : pn.rev, st);
    const std::vector<int> pt = bond_types(ts_, pn, true);
    ds_.p_ptype.upload(pt.empty() ? std::vector<int>{0} : pt, st);
    ds_.p_tri0.upload(t0, st);
    ds_.p_bond.resize(std::max(pn.total, 1));
    ds_.p_tri.resize((size_t)std::max<long long>(tri_total, 1));
    pd.NN = ds_.p_nn.get();
    pd.start = ds_.p_b0.get();
    pd.NL = ds_.p_nl.get();
    pd.rev = ds_.p_rev.get();
    pd.tri0 = ds_.p_tri0.get();
    pd.total = pn.total;
    build_geometry_device(ts_, pd, ds_.p_bond.get(), ds_.p_tri.get(), st);
    loop_.ptype = ds_.p_ptype.get();
    loop_.bond = ds_.p_bond.get();
    loop_.tri = ds_.p_tri.get();
    // (the host vectors above are read before this scope ends)
    GPUGA_HIP(hipStreamSynchronize(st));
  }
  loop_.nn = pd.NN;
  loop_.b0 = pd.start;
  loop_.tri0 = pd.tri0;
  loop_.rev = pd.rev;
  loop_.max_nn = pn.max_nn;
  return pd;
}

void Fitness::drop_population_tables()
{
  for (auto* b : {&ds_.p_nn, &ds_.p_b0, &ds_.p_nl, &ds_.p_rev, &ds_.p_ptype, &ds_.p_tri0})
    b->resize(0);
  ds_.p_bond.resize(0);
  ds_.p_tri.resize(0);
  loop_ = LoopTab{};
}

void Fitness::setup()
{
  int ndev = 0;
  GPUGA_HIP(hipGetDeviceCount(&ndev));
  if (ndev < 1) fail("no HIP device available");
  GPUGA_HIP(hipGetDevice(&device_));
  hipDeviceProp_t prop;
  GPUGA_HIP(hipGetDeviceProperties(&prop, device_));
  num_cu_ = prop.multiProcessorCount;
  GPUGA_HIP(hipStreamCreateWithFlags(&stream_, hipStreamNonBlocking));
  GPUGA_HIP(hipEventCreate(&ev0_));
  GPUGA_HIP(hipEventCreate(&ev1_));
  for (auto& e : ev_half_) GPUGA_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));

  const bool tersoff = spec_.type == POT_TERSOFF1 || spec_.type == POT_TERSOFF2;
  if (spec_.type == POT_RI || spec_.type == POT_NN2B_SPECIES)
    for (int t : ts_.type)
      if (t != 0 && t != 1)
        fail(spec_.type == POT_RI ? "RI potential needs atom types 0 and 1"
                                  : "NN2B with the species input needs atom types 0 and 1");
  nl_ = build_neighbors_device(ts_, spec_.cutoff, stream_);
  for (int i = 0; i < ts_.N; ++i)
    for (int s = 0; s < nl_.NN[i]; ++s)
      if (nl_.NL[nl_.rev[nl_.start[i] + s]] != i)
        fail("neighbour list is not symmetric (reverse bond missing)");
  // pair types on the host (the list is there); the geometry tables and the
  // atom records on the device, from the device copy of the list
  ptype_ = bond_types(ts_, nl_, tersoff);
  const std::vector<int>& ptype = ptype_;

  hipStream_t st = stream_;
  ds_.Na.upload(ts_.Na, st);
  ds_.Na_sum.upload(ts_.Na_sum, st);
  ds_.type.upload(ts_.type, st);
  ds_.nn.upload(nl_.NN, st);
  ds_.bond0.upload(nl_.start, st);
  ds_.nl.upload(nl_.NL.empty() ? std::vector<int>{0} : nl_.NL, st);
  ds_.rev.upload(nl_.rev.empty() ? std::vector<int>{0} : nl_.rev, st);
  ds_.ptype.upload(ptype.empty() ? std::vector<int>{0} : ptype, st);
  DeviceNeighbors dn = device_neighbors();
  if (nl_.total == 0) ds_.bond.upload(std::vector<float4>{make_float4(0, 0, 0, 1)}, st);
  else ds_.bond.resize(nl_.total);
  std::vector<int> tri0;
  if (tersoff) {
    long long tri_total = 0;
    tri0 = triplet_offsets(nl_, &tri_total);
    ds_.tri0.upload(tri0, st);
    if (tri_total == 0) ds_.tri.upload(std::vector<float4>(1), st);
    else ds_.tri.resize((size_t)tri_total);
    dn.tri0 = ds_.tri0.get();
    build_geometry_device(ts_, dn, ds_.bond.get(), ds_.tri.get(), st);
    // The population kernel's records leave out the bonds that no
    // individual's taper reaches (exact zeros in every sum).
    const float reach = tersoff_reach(spec_);
    pruned_ = false;
    if (reach < spec_.cutoff && nl_.total > 0) {
      std::vector<float4> b(nl_.total);
      ds_.bond.download(b.data(), b.size(), st);
      GPUGA_HIP(hipStreamSynchronize(st));
      std::vector<float> d(nl_.total);
      for (int k = 0; k < nl_.total; ++k) d[k] = b[k].w;
      pnl_ = prune_neighbors(nl_, d, reach);
      pruned_ = pnl_.total < nl_.total;
      if (!pruned_) pnl_ = NeighborList();
    }
    const NeighborList& pn = population_neighbors();
    const int M = record_slots(pn.max_nn);
    shell_M_ = pn.max_nn > 4 ? tersoff_shell_slots(pn.max_nn) : 0;
    loop_path_ = pn.max_nn > 4 && shell_M_ == 0;
    if (loop_path_ && pn.max_nn > kLoopMaxNeighbors)
      fail(strfmt("the population kernel supports at most %d neighbours per atom within the "
                  "largest R2 (found %d); use the per-individual backend",
                  kLoopMaxNeighbors, pn.max_nn));
    const DeviceNeighbors pd = build_population_tables();
    if (shell_M_ > 0) {
      ds_.shell_rec.resize(tersoff_shell_floats4(ts_.N, shell_M_));
      build_shell_records(ts_.N, shell_M_, loop_, ds_.shell_rec.get(), st);
    }
    if (pn.max_nn <= 4) {
      ds_.rec.resize((size_t)ts_.N * record_floats4(M));
      build_records_device(ts_.N, M, pd, loop_.ptype, loop_.bond, loop_.tri, ds_.rec.get(), st);
      // An atom's moment record serves a wave when its bonds are shorter than
      // every lane's R1, whose smallest is near the parameter's lower bound.
      // Kept where nine atoms in ten pass at that bound: with half of them,
      // 120 200 atoms and 200 individuals, a call took 335 us with the records
      // and 318 us without (all: 280 and 297 us).
      const int n = ts_.N - ts_.N_force;
      const float r1 = std::min(spec_.pmin[spec_.V - 2], spec_.pmax[spec_.V - 2]);
      ds_.mom.resize((size_t)std::max(n, 1) * kMomWords);
      const int inside =
        build_moments_device(ts_.N_force, ts_.N, pd, loop_.ptype, loop_.bond, r1, ds_.mom.get(), st);
      if (10LL * inside < 9LL * n || n == 0) ds_.mom.resize(0);
    }
    if (!loop_path_) {
      GPUGA_HIP(hipStreamSynchronize(st));
      // the records hold everything the kernel reads of the pruned list
      drop_population_tables();
    }
    ds_.view.bond_force =
      ts_.N_force > 0 ? pn.start[ts_.N_force - 1] + pn.NN[ts_.N_force - 1] : 0;
    dmin_ = dmax_ = 1.0f; // (the NN2B tabulation range; unused here)
  } else {
    ds_.tri0.upload(std::vector<int>(ts_.N, 0), st);
    ds_.tri.upload(std::vector<float4>(1), st);
    build_geometry_device(ts_, dn, ds_.bond.get(), nullptr, st);
    dmin_ = dmax_ = 1.0f;
    if (nl_.total > 0) {
      DeviceBuffer<unsigned> range;
      const unsigned none[2] = {0xffffffffu, 0u};
      unsigned got[2];
      range.upload(none, 2, st);
      launch_bond_range(nl_.total, ds_.bond.get(), range.get(), st);
      range.download(got, 2, st);
      GPUGA_HIP(hipStreamSynchronize(st));
      std::memcpy(&dmin_, &got[0], sizeof dmin_);
      std::memcpy(&dmax_, &got[1], sizeof dmax_);
    }
    if (spec_.type == POT_RI) {
      ds_.ri_tab.resize(std::max(nl_.total, 1));
      launch_ri_table((int)ds_.bond.size(), ds_.bond.get(), ds_.ri_tab.get(), st);
    }
  }
  // the uploads above read host vectors of this scope
  GPUGA_HIP(hipStreamSynchronize(st));
  ds_.pe_ref.upload(ts_.pe_ref, st);
  ds_.virial_ref.upload(ts_.virial_ref, st);
  ds_.force_ref.upload(ts_.force_ref, st);
  GPUGA_HIP(hipStreamSynchronize(st));

  DevSet& v = ds_.view;
  v.Nc = ts_.Nc;
  v.Nc_force = ts_.Nc_force;
  v.N = ts_.N;
  v.N_force = ts_.N_force;
  v.max_nn = nl_.max_nn;
  v.Na = ds_.Na.get();
  v.Na_sum = ds_.Na_sum.get();
  v.type = ds_.type.get();
  v.nn = ds_.nn.get();
  v.bond0 = ds_.bond0.get();
  v.nl = ds_.nl.get();
  v.rev = ds_.rev.get();
  v.ptype = ds_.ptype.get();
  v.bond = ds_.bond.get();
  v.tri0 = ds_.tri0.get();
  v.tri = ds_.tri.get();
  v.rec = ds_.rec.get();
  v.mom = ds_.mom.get();
  v.pe_ref = ds_.pe_ref.get();
  v.virial_ref = ds_.virial_ref.get();
  v.force_ref = ds_.force_ref.get();

  if (!tersoff) {
    setup_quad();
    if (!quad_.on) build_pair_tables();
  }

  potential_ = make_potential(spec_, ds_);
  potential_->initialize(ts_.N, ts_.max_Na);
  // this device's fixed workspace of the allocation-free path, looked up
  // here (set-up) so that the path's calls only use the kept address
  ws_static_ = static_workspace();
  d_pmin_.upload(spec_.pmin, st);
  d_pmax_.upload(spec_.pmax, st);
  GPUGA_HIP(hipStreamSynchronize(st));
  d_f_.resize(3 * (size_t)ts_.N);
  d_virial_.resize(6 * (size_t)ts_.N);
  d_pe_.resize(ts_.N);
  if (10 * (size_t)ts_.N > 3 * kHalf) h_atoms_.resize(2 * kHalf);
  d_cerr_.resize(3 * (size_t)ts_.Nc);
  d_fit1_.resize(1);
  d_terms1_.resize(3);
}

// The tables of the population kernel's pair loops, built on the host from
// the bond geometry.
void Fitness::build_pair_tables()
{
  if (pair_tables_) return;
  hipStream_t st = stream_;
  const std::vector<int>& ptype = ptype_;
  std::vector<Vec4> bond(ds_.bond.size());
  static_assert(sizeof(Vec4) == sizeof(float4), "layout");
  ds_.bond.download(reinterpret_cast<float4*>(bond.data()), bond.size(), st);
  GPUGA_HIP(hipStreamSynchronize(st));
  // the pairs a pair potential evaluates for atom i: all its bonds in force
  // configurations (forces need both directions), j > i elsewhere (energy
  // and virial need each pair once); pair_offsets()[i] = the first of atom
  // i's pairs, [N] = their number
  auto evaluates = [&](int i, int b) { return i < ts_.N_force || nl_.NL[b] > i; };
  auto pair_offsets = [&] {
    std::vector<int> off(ts_.N + 1, 0);
    parallel_for(ts_.N, [&](int i) {
      int c = 0;
      for (int b = nl_.start[i]; b < nl_.start[i] + nl_.NN[i]; ++b) c += evaluates(i, b);
      off[i + 1] = c;
    });
    for (int i = 0; i < ts_.N; ++i) off[i + 1] += off[i];
    return off;
  };
  if (spec_.type == POT_RI) {
    // population form: per atom the pairs it evaluates (all bonds for force
    // configurations, those with j > i for the others), grouped by pair type
    // t_i + t_j.  A force configuration's pair: unit vector and d (one
    // float4); an energy configuration's pair: d and the virial coefficients
    // u_a u_b d (xx, yy, zz, then xy, yz, zx; two float4: the virial then
    // takes one FMA per component).  The header's first word is the atom's
    // first float4.  Of a pair's terms (src/ri.cu:77-110) only the
    // Buckingham exponential and the Morse term are non-linear in the
    // parameters; the others are a parameter times a function of d, so their
    // sums over a configuration (energy, virial) or over an atom's bonds
    // (force) are taken here once, in FP64, and the kernel adds the
    // parameters' combination of them once per configuration or atom.
    const std::vector<int> p0 = pair_offsets();
    auto rows_before = [&](int i) { // float4 rows of the atoms before i
      const long nf = std::min(i, ts_.N_force);
      return (long)p0[nf] + 2 * ((long)p0[i] - p0[nf]);
    };
    const long rows = rows_before(ts_.N);
    if (rows > INT_MAX) fail("rigid-ion pair table too large");
    std::vector<float4> pt((size_t)std::max<long>(rows, 1));
    std::vector<int4> hdr(std::max(ts_.N, 1));
    parallel_for(ts_.N, [&](int i) {
      const int nn = nl_.NN[i], b0 = nl_.start[i];
      const bool force = i < ts_.N_force;
      int cnt[3] = {0, 0, 0};
      const long first = rows_before(i);
      float4* out = &pt[(size_t)first];
      for (int t = 0; t < 3; ++t)
        for (int u = 0; u < nn; ++u) {
          const int b = b0 + u;
          if (ptype[b] != t || !evaluates(i, b)) continue;
          const Vec4 r = bond[b];
          const double dinv = 1.0 / r.w;
          if (force) {
            *out++ = make_float4((float)(r.x * dinv), (float)(r.y * dinv), (float)(r.z * dinv), r.w);
          } else {
            // u_a u_b d = r_a r_b / d
            *out++ = make_float4(r.w, (float)(r.x * r.x * dinv), (float)(r.y * r.y * dinv),
                                 (float)(r.z * r.z * dinv));
            *out++ = make_float4((float)(r.x * r.y * dinv), (float)(r.y * r.z * dinv),
                                 (float)(r.z * r.x * dinv), 0.0f);
          }
          ++cnt[t];
        }
      hdr[i] = make_int4((int)first, cnt[0], cnt[1], cnt[2]);
    });
    ds_.pair_tab.upload(pt, st);
    ds_.pair_hdr.upload(hdr, st);
    // f_6 = 6 d^-7, f_c = erfc(a d)/d, h = -(d/dr) f_c (a = 0.2, as above)
    auto factors = [](double d, double& d6, double& f6, double& fc, double& h) {
      const double dinv = 1.0 / d;
      d6 = std::pow(dinv, 6);
      f6 = 6.0 * d6 * dinv;
      fc = std::erfc(0.2 * d) * dinv;
      h = fc * dinv + 0.225675833419103 * std::exp(-0.04 * d * d) * dinv;
    };
    std::vector<double> cc((size_t)std::max(ts_.Nc, 1) * 3 * kRiTypeConst, 0.0);
    parallel_for(ts_.Nc, [&](int c) {
      if (c < ts_.Nc_force) return;
      double* out = &cc[(size_t)c * 3 * kRiTypeConst];
      for (int i = ts_.Na_sum[c]; i < ts_.Na_sum[c] + ts_.Na[c]; ++i)
        for (int b = nl_.start[i]; b < nl_.start[i] + nl_.NN[i]; ++b) {
          if (!evaluates(i, b)) continue;
          const Vec4 r = bond[b];
          const double d = r.w;
          double d6, f6, fc, h;
          factors(d, d6, f6, fc, h);
          const double v[6] = {r.x * r.x / d, r.y * r.y / d, r.z * r.z / d,
                               r.x * r.y / d, r.y * r.z / d, r.z * r.x / d};
          double* o = out + (size_t)ptype[b] * kRiTypeConst;
          o[0] += 1.0;
          o[1] += d;
          o[2] += fc;
          o[3] += d6;
          for (int a = 0; a < 6; ++a) {
            o[4 + a] += v[a];
            o[10 + a] += v[a] * f6;
            o[16 + a] += v[a] * h;
          }
        }
    });
    ds_.ri_cconst.upload(cc, st);
    std::vector<float> fcon((size_t)std::max(ts_.N_force, 1) * kRiAtomConst, 0.0f);
    parallel_for(ts_.N_force, [&](int i) {
      double o[kRiAtomConst] = {};
      for (int b = nl_.start[i]; b < nl_.start[i] + nl_.NN[i]; ++b) {
        const Vec4 r = bond[b];
        const double d = r.w;
        double d6, f6, fc, h;
        factors(d, d6, f6, fc, h);
        const double u[3] = {r.x / d, r.y / d, r.z / d};
        for (int x = 0; x < 3; ++x) {
          double* w = o + ptype[b] * 9 + x * 3;
          w[0] += u[x] * f6;
          w[1] += u[x];
          w[2] += u[x] * h;
        }
      }
      for (int k = 0; k < kRiAtomConst; ++k) fcon[(size_t)i * kRiAtomConst + k] = (float)o[k];
    });
    ds_.ri_fconst.upload(fcon, st);
    GPUGA_HIP(hipStreamSynchronize(st));
  }
  if (spec_.nn2b()) {
    // population form: per atom the pairs it evaluates (all bonds for force
    // configurations, j > i for the others) in order of distance, so that
    // consecutive pairs read neighbouring rows of the tabulated network; per
    // pair (unit vector, d), the cubic Hermite weights on the tabulation
    // grid (h00, h h10, h01, h h11), and (fc, fc', grid cell, species code)
    // with the reference's fixed taper (src/nn2b.cu:80-92)
    const NN2BGrid grid = nn2b_grid_desc();
    const std::vector<int> p0 = pair_offsets();
    // an energy configuration's pair carries its virial coefficients
    // u_a u_b d (xx, yy, zz, xy; yz, zx) in place of (unit vector, d): four
    // float4 instead of three; the header's first word is the atom's first
    // float4
    auto rows_before = [&](int i) {
      const long nf = std::min(i, ts_.N_force);
      return 3 * (long)p0[nf] + 4 * ((long)p0[i] - p0[nf]);
    };
    const long rows = rows_before(ts_.N);
    if (rows > INT_MAX) fail("NN2B pair table too large");
    std::vector<float4> pt((size_t)std::max<long>(rows, 1));
    std::vector<int4> hdr(std::max(ts_.N, 1));
    parallel_for(ts_.N, [&](int i) {
      const int nn = nl_.NN[i], b0 = nl_.start[i];
      const bool force = i < ts_.N_force;
      std::vector<int> order;
      order.reserve(nn);
      for (int u = 0; u < nn; ++u)
        if (evaluates(i, b0 + u)) order.push_back(b0 + u);
      std::stable_sort(order.begin(), order.end(),
                       [&](int a, int b) { return bond[a].w < bond[b].w; });
      const long first = rows_before(i);
      hdr[i] = make_int4((int)first, (int)order.size(), 0, 0);
      float4* out = &pt[(size_t)first];
      for (int b : order) {
        const Vec4 r = bond[b];
        const double d = r.w, dinv = 1.0 / d;
        const double u = (d - (double)grid.d0) / (double)grid.h;
        const int g = std::max(0, std::min((int)u, grid.G - 2));
        const double t = u - g, t2 = t * t, t3 = t2 * t, h = grid.h;
        double fc = 0.0, fcp = 0.0;
        if (d < NN2B_R1) {
          fc = 1.0;
        } else if (d < NN2B_R2) {
          const double a = (double)NN2B_PI_FACTOR * (d - NN2B_R1);
          fc = 0.5 * std::cos(a) + 0.5;
          fcp = -0.5 * (double)NN2B_PI_FACTOR * std::sin(a);
        }
        if (force) {
          *out++ = make_float4((float)(r.x * dinv), (float)(r.y * dinv), (float)(r.z * dinv), r.w);
        } else {
          *out++ = make_float4((float)(r.x * r.x * dinv), (float)(r.y * r.y * dinv),
                               (float)(r.z * r.z * dinv), (float)(r.x * r.y * dinv));
          *out++ = make_float4((float)(r.y * r.z * dinv), (float)(r.z * r.x * dinv), 0.0f, 0.0f);
        }
        *out++ = make_float4((float)(2 * t3 - 3 * t2 + 1), (float)(h * (t3 - 2 * t2 + t)),
                             (float)(-2 * t3 + 3 * t2), (float)(h * (t3 - t2)));
        // (the species code t_i + t_j picks the individual's table for it)
        const int code = spec_.type == POT_NN2B_SPECIES ? ptype[b] : 0;
        float4 c = make_float4((float)fc, (float)fcp, 0.0f, 0.0f);
        std::memcpy(&c.z, &g, sizeof g);
        std::memcpy(&c.w, &code, sizeof code);
        *out++ = c;
      }
    });
    ds_.pair_tab.upload(pt, st);
    ds_.pair_hdr.upload(hdr, st);
    GPUGA_HIP(hipStreamSynchronize(st));
  }
  DevSet& v = ds_.view;
  v.pair_hdr = ds_.pair_hdr.get();
  v.pair_tab = ds_.pair_tab.get();
  v.ri_cconst = ds_.ri_cconst.get();
  v.ri_fconst = ds_.ri_fconst.get();
  pair_tables_ = true;
}

int Fitness::quad_elements() const
{
  if (nl_.total == 0 || !(dmin_ > 0.0f) || !std::isfinite(dmax_)) return 0;
  // (a label that is no number makes the sums so by itself: left to the pair
  // loop, whose terms then are what they were)
  for (const std::vector<float>* v : {&ts_.pe_ref, &ts_.virial_ref, &ts_.force_ref})
    for (float x : *v)
      if (!std::isfinite(x)) return 0;
  if (spec_.nn2b()) {
    // half as many nodes as the grid has points, in elements of 32.  How sharp
    // an individual's curve is, is judged from its nodes at each evaluation
    // (SharpSet): from 256 points on they resolve part of a population drawn
    // from bounds of 3 (n = 20 on 256 points a quarter of it, n = 32 on 1024 all
    // but a few), and the pair loop takes the rest.  The forms grow with the
    // square of the nodes, so a grid finer than 2048 points (all codes together)
    // stays with the pair loop
    const int G = std::max(opt_.nn2b_grid, 16), codes = spec_.pair_codes();
    if (G < 256 || G > 2048) return 0;
    return codes * G > 4096 ? 0 : G / (2 * QB);
  }
  // Rigid ion: exponentials of known largest rate over genes in [0, 1].  An
  // element of half length s / rate interpolates one to 2e-12 of its largest
  // value at s = 16.
  double rate = 0.0;
  auto lo = [&](int v) { return (double)std::min(spec_.pmin[v], spec_.pmax[v]); };
  auto hi = [&](int v) { return (double)std::max(spec_.pmin[v], spec_.pmax[v]); };
  for (int v = 0; v < spec_.V; ++v)
    if (!std::isfinite(lo(v)) || !std::isfinite(hi(v))) return 0;
  for (int t = 0; t < 3; ++t) {
    if (lo(1 + 3 * t) == 0.0 && hi(1 + 3 * t) == 0.0) continue;
    if (!(lo(2 + 3 * t) > 0.0)) return 0;
    rate = std::max(rate, 1.0 / lo(2 + 3 * t));
  }
  if (lo(11) != 0.0 || hi(11) != 0.0) {
    const double alpha = std::max(std::fabs(lo(12)), std::fabs(hi(12)));
    if (!(lo(14) > 0.0)) return 0;
    rate = std::max({rate, std::sqrt(2.0 * hi(14)) * alpha, std::sqrt(2.0 / lo(14)) * alpha});
  }
  const double e = std::ceil(0.5 * (dmax_ - dmin_) * rate / 16.0);
  return e <= 8.0 ? std::max(1, (int)e) : 0;
}

void Fitness::setup_quad()
{
  const int E = quad_elements();
  if (E == 0) return;
  hipStream_t st = stream_;
  QuadBasis b;
  b.rigid = spec_.type == POT_RI ? 1 : 0;
  b.codes = b.rigid ? 3 : spec_.pair_codes();
  b.E = E;
  b.d0 = dmin_;
  b.len = std::max((double)dmax_ - (double)dmin_, 1e-3) / E;
  const int CE = b.CE();
  // the elements that the pairs of energy and of force configurations use
  if (CE > QCE) fail("internal: elements of the quadratic forms");
  DeviceBuffer<int> d_used;
  std::vector<int> used((size_t)6 * CE, 0);
  d_used.upload(used, st);
  launch_quad_used(ds_.view, b, d_used.get(), st);
  d_used.download(used.data(), used.size(), st);
  GPUGA_HIP(hipStreamSynchronize(st));
  // column blocks of each form and their value blocks; U' enters the virials
  // and forces (U only inside NN2B's taper), U the energies
  std::vector<int> col((size_t)6 * CE, -1), vblk[3];
  std::vector<int2> act;
  int nb[3];
  for (int f = 0; f < 3; ++f) {
    const int* u = &used[f == 2 ? (size_t)2 * CE : 0];
    vblk[f].push_back(2 * CE);
    auto add = [&](int map, int first, const int* used, int ce0, int ce1) {
      for (int ce = ce0; ce < ce1; ++ce)
        if (used[ce]) {
          col[(size_t)map * CE + ce] = (int)vblk[f].size();
          vblk[f].push_back(first + ce);
        }
    };
    // code 0's columns before the differences (rigid ion: no differences)
    const int n0 = b.species() ? E : CE;
    for (int part = 0; part < 2; ++part) {
      const int ce0 = part ? n0 : 0, ce1 = part ? CE : n0;
      add(f == 0 ? 0 : 3 + f, f == 0 ? 0 : CE, u, ce0, ce1);
      if (f > 0) add(f, 0, u + CE, ce0, ce1);
    }
    nb[f] = (int)vblk[f].size();
  }
  auto in_use = [&](int ce) { return used[ce] || used[2 * CE + ce]; };
  for (int k = 0; k < (b.rigid ? CE : E); ++k) {
    int mask = 0;
    for (int c = 0; c < (b.rigid ? 1 : b.codes); ++c) mask |= in_use(c * E + k) ? 1 << c : 0;
    if (mask) act.push_back(make_int2(k, mask));
  }
  QuadRows rows;
  DeviceBuffer<int> d_col;
  d_col.upload(col, st);
  rows.b = b;
  rows.col = d_col.get();
  for (int f = 0; f < 3; ++f) rows.nb[f] = nb[f];
  if (!quad_prepare(rows)) return;
  quad_.basis = b;
  quad_.n_act = (int)act.size();
  quad_.act.upload(act, st);
  std::vector<float2> pairs(CE);
  std::vector<float> tail((size_t)QTAIL * QB);
  if (!b.rigid) {
    for (int ce = 0; ce < CE; ++ce)
      pairs[ce] = make_float2((float)used[4 * CE + ce], (float)used[5 * CE + ce]);
    for (int k = 0; k < QTAIL; ++k)
      for (int m = 0; m < QB; ++m)
        tail[(size_t)k * QB + m] =
          (float)(2.0 / QB * std::cos(M_PI / QB * (m + 0.5) * (QB - QTAIL + k)));
    quad_.pairs.upload(pairs, st);
    quad_.tail.upload(tail, st);
  }
  // Rows in chunks of configurations and force atoms, the Gram products
  // accumulated over the chunks.  Chunks and the split of a chunk's rows over
  // waves do not depend on the columns, so a column's sums do not depend on
  // which others the form has.
  DeviceBuffer<double> R, part;
  size_t most = 0;
  for (int f = 0; f < 3; ++f) {
    quad_.nb[f] = nb[f];
    quad_.q[f].resize((size_t)quad_tiles(nb[f]) * QB * QB);
    quad_.vblk[f].upload(vblk[f], st);
    most = std::max(most, quad_part_size(nb[f]));
  }
  part.resize(most);
  auto gram = [&](int f, const double* r, int n, bool first) {
    launch_quad_gram(r, n, nb[f], first, part.get(), quad_.q[f].get(), st);
  };
  { // energy and virial rows
    const int ne = ts_.Nc - ts_.Nc_force, step = quad_step(kQuadConfigs, ne);
    const size_t D0 = rows.D(0), D1 = rows.D(1);
    R.resize(step * (D0 + 6 * D1));
    double *re = R.get(), *rw = re + step * D0;
    for (int c0 = 0; c0 < std::max(ne, 1); c0 += step) {
      const int n = std::min(step, ne - c0), n4 = quad_step(step, n), c = ts_.Nc_force + c0;
      R.zero(st);
      if (n > 0) launch_quad_energy_rows(ds_.view, rows, c, c + n, re, rw, st);
      gram(0, re, n4, c0 == 0);
      gram(1, rw, 6 * n4, c0 == 0);
    }
  }
  GPUGA_HIP(hipStreamSynchronize(st));
  { // force rows
    const int na = ts_.N_force, step = quad_step(kQuadAtoms, na);
    R.resize((size_t)step * 3 * rows.D(2));
    for (int i0 = 0; i0 < std::max(na, 1); i0 += step) {
      const int n = std::min(step, na - i0);
      R.zero(st);
      if (n > 0) launch_quad_force_rows(ds_.view, rows, i0, i0 + n, R.get(), st);
      gram(2, R.get(), 3 * quad_step(step, n), i0 == 0);
    }
  }
  for (int f = 0; f < 3; ++f) launch_quad_finish(nb[f], quad_.q[f].get(), st);
  std::vector<int2> unit;
  for (int I = std::max({nb[0], nb[1], nb[2]}) - 1; I >= 0; --I)
    for (int f = 0; f < 3; ++f)
      if (I < nb[f]) unit.push_back(make_int2(f, I));
  quad_.unit.upload(unit, st);
  GPUGA_HIP(hipStreamSynchronize(st));
  quad_.on = true;
}

bool Fitness::quad_for(int P, const float* genes) const
{
  if (!quad_.on) return false;
  if (spec_.nn2b()) return true; // (each individual's nodes are checked)
  for (size_t k = 0; k < (size_t)P * spec_.V; ++k)
    if (!(genes[k] >= 0.0f && genes[k] <= 1.0f)) return false;
  return true;
}

// What a plan has on every path: genes, and results in one block on either
// side (terms [P][3] in FP64, fitness [P] in FP32, the status word).
void Fitness::build_results(PopPlan& pl, int P)
{
  pl.P = P;
  pl.K = (P + WAVE - 1) / WAVE;
  pl.out.resize(pl.out_doubles());
  pl.out.zero(stream_);
  pl.genes.resize((size_t)P * spec_.V);
  pl.h_genes.resize((size_t)P * spec_.V);
  pl.h_out.resize(pl.out_doubles());
  std::memset(pl.h_out.get(), 0, sizeof(double) * pl.out_doubles());
  PopCtl& c = pl.ctl;
  c.K = pl.K;
  c.P = P;
  c.V = spec_.V;
  c.genes = pl.genes.get();
  c.pmin = d_pmin_.get();
  c.pmax = d_pmax_.get();
  c.terms = pl.out.get();
  c.fitness = reinterpret_cast<float*>(c.terms + 3 * (size_t)P);
  c.status = reinterpret_cast<unsigned*>(c.fitness + P);
  c.norm = norm();
}

void Fitness::build_quad_plan(PopPlan& pl, int P)
{
  hipStream_t st = stream_;
  build_results(pl, P);
  const int ld = (P + QP - 1) / QP * QP;
  // (the linear block: zeros and the constant 1, the parameters written by
  // each launch)
  const size_t block = (size_t)QB * ld, lin = (size_t)2 * quad_.basis.CE() * block;
  std::vector<double> ones(ld, 1.0);
  pl.qvalues.resize(lin + block);
  pl.qvalues.zero(st);
  GPUGA_HIP(hipMemcpyAsync(pl.qvalues.get() + lin + (size_t)kQuadOne * ld, ones.data(),
                           sizeof(double) * ld, hipMemcpyHostToDevice, st));
  pl.qpart.resize((size_t)quad_.units() * ld);
  pl.qdone.resize(ld / QP);
  pl.qdone.zero(st);
  QuadEval& q = pl.qeval;
  for (int f = 0; f < 3; ++f)
    q.form[f] = QuadForm{quad_.nb[f], quad_.vblk[f].get(), quad_.q[f].get()};
  q.unit = quad_.unit.get();
  q.units = quad_.units();
  q.values = pl.qvalues.get();
  q.ld = ld;
  q.part = pl.qpart.get();
  q.done = pl.qdone.get();
  pl.qnodes = NodeTable{quad_.basis, quad_.act.get(), quad_.n_act, pl.qvalues.get(), ld};
  if (spec_.nn2b()) {
    const int parts = nn2b_node_parts(P);
    pl.qsums.resize((size_t)parts * kTailSums * ld);
    pl.qcount.resize(2);
    pl.qcount.zero(st);
    pl.qlist.resize(P);
    pl.qnodes.pairs = quad_.pairs.get();
    pl.qnodes.tail = quad_.tail.get();
    pl.qnodes.sums = pl.qsums.get();
    const float limit = opt_.nn2b_bf16 && spec_.num_neurons <= 32 ? kTailBf16 : kTailFp32;
    q.sharp.sums = pl.qsums.get();
    q.sharp.parts = parts;
    q.sharp.limit2 = limit * limit;
    q.sharp.list = pl.qlist.get();
    q.sharp.any = pl.h_sharp();
  }
  GPUGA_HIP(hipStreamSynchronize(st));
}

void Fitness::ensure_items(PopPlan& pl)
{
  if (pl.items_built) return;
  build_pair_tables();
  build_plan(pl, pl.P, launch_shape(pl.P));
}

void Fitness::launch_quad(PopPlan& pl, const PopCtl& ctl, hipStream_t st)
{
  launch_quad_values(pl, ctl, 0, pl.P, st);
  launch_quad_eval(pl, ctl, st);
}

void Fitness::launch_quad_eval(PopPlan& pl, const PopCtl& ctl, hipStream_t st)
{
  if (pl.qeval.sharp.sums) {
    pl.qeval.sharp.count = pl.qcount.get() + pl.qturn;
    pl.qturn ^= 1;
    pl.qeval.sharp.next = pl.qcount.get() + pl.qturn;
  }
  gpuga::launch_quad_eval(ctl, pl.qeval, st);
}

PopCtl Fitness::sharp_ctl(const PopPlan& pl, PopCtl ctl) const
{
  ctl.live = pl.qeval.sharp.count;
  ctl.index = pl.qlist.get();
  return ctl;
}

void Fitness::launch_quad_values(PopPlan& pl, const PopCtl& ctl, int first, int count,
                                 hipStream_t st)
{
  if (quad_.basis.rigid) launch_ri_values(ctl, pl.qnodes, st);
  // (with the last individuals, the padding of the values)
  else
    launch_nn2b_nodes(ctl, nn2b_grid_desc(), pl.qnodes, first,
                      first + count == pl.P ? pl.qnodes.ld - first : count, st);
}

NN2BGrid Fitness::nn2b_grid_desc() const
{
  NN2BGrid g;
  g.G = std::max(opt_.nn2b_grid, 16);
  g.n = spec_.num_neurons;
  g.bf16 = opt_.nn2b_bf16;
  g.codes = spec_.pair_codes();
  // one spare cell on each side of the training set's pair-distance range
  const float span = std::max(dmax_ - dmin_, 1e-3f);
  g.h = span / (float)(g.G - 3);
  g.d0 = dmin_ - g.h;
  return g;
}

FitnessNorm Fitness::norm() const
{
  FitnessNorm n;
  n.inv_pss = 1.0 / ts_.potential_square_sum;
  n.inv_vss = 1.0 / ts_.virial_square_sum;
  n.inv_fss = 1.0 / ts_.force_square_sum;
  n.w_energy = spec_.w_energy;
  n.w_stress = spec_.w_stress;
  n.w_force = spec_.w_force;
  return n;
}

size_t Fitness::device_bytes() const
{
  size_t b = ds_.bytes() + quad_.bytes() + d_f_.bytes() + d_virial_.bytes() + d_pe_.bytes() + d_cerr_.bytes();
  for (auto& kv : plans_) {
    const PopPlan& p = *kv.second;
    b += p.qvalues.bytes() + p.qpart.bytes() + p.qsums.bytes() + p.qlist.bytes();
    b += p.items.bytes() + p.part.bytes() + p.err.bytes() + p.bondf.bytes() + p.genes.bytes() +
         p.out.bytes() + p.gpart.bytes() + p.counters.bytes() + p.nn2b_table.bytes();
  }
  return b;
}

// ------------------------------------------------------- population plans

namespace {

long long atom_cost(int type, int nn, bool force_cfg)
{
  if (type == POT_TERSOFF1 || type == POT_TERSOFF2) return (long long)nn * nn + 4LL * nn + 8;
  return (force_cfg ? nn : nn / 2 + 1) + 4;
}

} // namespace

size_t Fitness::plan_bytes(int P) const
{
  const size_t K = (P + WAVE - 1) / WAVE;
  const NeighborList& pn = population_neighbors();
  const size_t B_force = ts_.N_force > 0 ? (size_t)pn.start[ts_.N_force - 1] +
                                             pn.NN[ts_.N_force - 1]
                                         : 0;
  const bool tersoff = spec_.type == POT_TERSOFF1 || spec_.type == POT_TERSOFF2;
  size_t b = K * 3 * ts_.Nc * WAVE * sizeof(double);              // err
  b += (size_t)2 * ts_.Nc * K * 8 * WAVE * sizeof(double);         // part (typical)
  if (tersoff) b += K * (B_force + ts_.N_force) * 3 * WAVE * sizeof(float);       // bondf
  if (spec_.nn2b())
    b += (size_t)3 * spec_.pair_codes() * opt_.nn2b_grid * K * WAVE * sizeof(float);
  return b;
}

LaunchShape Fitness::option_shape() const
{
  LaunchShape sh;
  sh.chunk_cost = opt_.chunk_cost;
  sh.queues = opt_.queues;
  sh.blocks_per_cu = opt_.blocks_per_cu;
  sh.pack = opt_.pack_lanes;
  return sh;
}

void Fitness::build_plan(PopPlan& pl, int P, const LaunchShape& sh)
{
  const int chunk_cost = std::max(sh.chunk_cost, 1);
  const int Nc = ts_.Nc;
  const bool tersoff = spec_.type == POT_TERSOFF1 || spec_.type == POT_TERSOFF2;
  // neighbour counts of the list the kernel reads (Tersoff: the pruned one)
  const NeighborList& pn = tersoff ? population_neighbors() : nl_;
  // (a plan of the forms has results already, perhaps of a launch whose caller
  // has not taken them yet)
  if (pl.P == 0) build_results(pl, P);
  // the looped Tersoff kernel: one wave per workgroup (its LDS rows)
  pl.block = tersoff && loop_path_ ? WAVE : 256;
  pl.chunk_cost = chunk_cost;
  const int tail_split = opt_.tail_split > 0 ? opt_.tail_split : 1;
  const int K = pl.K;

  struct Chunk {
    int c, chunk, a0, a1;
    long long cost;
  };
  std::vector<Chunk> chunks;
  std::vector<int> nch(Nc), slot0(Nc);
  std::vector<long long> cfg_total(Nc, 0);
  for (int c = 0; c < Nc; ++c)
    for (int i = ts_.Na_sum[c]; i < ts_.Na_sum[c] + ts_.Na[c]; ++i)
      cfg_total[c] += atom_cost(spec_.type, pn.NN[i], c < ts_.Nc_force);
  // chunks of configuration c for an item cost of `cost`
  auto chunks_of = [&](int c, long long cost) {
    const long long total = cfg_total[c];
    cost = std::max<long long>(cost, 1);
    int n = (int)std::max<long long>(1, (total + cost - 1) / cost);
    // A configuration smaller than one item comes at the end of its queue
    // (largest first), where the launch drains: it is cut into pieces of
    // 1/tail_split of an item, so that the last items are short.  (Not the
    // three-body force configurations: they come first.)
    if (total < cost && !(tersoff && c < ts_.Nc_force)) {
      const long long piece = std::max<long long>(1, cost / std::max(tail_split, 1));
      n = (int)std::max<long long>(1, (total + piece - 1) / piece);
    }
    return std::min(n, ts_.Na[c]);
  };
  // A three-body force configuration runs two dependent steps (its chunks,
  // then their force assembly), an energy configuration one.  When every item
  // has a SIMD of its own (a launch too small to fill the device, so its time
  // is the longest chain rather than the total work), the force
  // configurations' chunks are cut at half the item cost, so that both
  // chains end together.  (Cut at a third, the waves of a launch of this
  // kind went from 768 to 984 and every atom took longer: 1.03 against 0.87
  // us per energy atom.)
  long long force_cost = chunk_cost;
  if (tersoff && ts_.Nc_force > 0) {
    // (a force configuration of several chunks has an assembly item per
    // chunk; 4 SIMDs per CU)
    long long n_items = 0;
    for (int c = 0; c < Nc; ++c) {
      const bool fc = c < ts_.Nc_force;
      const int n = chunks_of(c, fc ? chunk_cost / 2 : chunk_cost);
      n_items += (long long)n * (fc && n > 1 ? 2 : 1);
    }
    if (n_items * K <= 4LL * num_cu_) force_cost = std::max(chunk_cost / 2, 1);
  }
  int slots = 0;
  for (int c = 0; c < Nc; ++c) {
    const int a0 = ts_.Na_sum[c], a1 = a0 + ts_.Na[c];
    const bool fc = c < ts_.Nc_force;
    const long long total = cfg_total[c];
    const int n = chunks_of(c, fc ? force_cost : chunk_cost);
    nch[c] = n;
    slot0[c] = slots;
    slots += n;
    long long acc = 0;
    int start = a0, k = 0;
    long long cacc = 0;
    for (int i = a0; i < a1; ++i) {
      const long long ci = atom_cost(spec_.type, pn.NN[i], fc);
      acc += ci;
      cacc += ci;
      // cut at the k-th cost quantile, or when the atoms left are exactly
      // the chunks still to make
      const int left_atoms = a1 - (i + 1), left_chunks = n - 1 - k;
      const bool must = left_chunks > 0 && left_atoms == left_chunks;
      const bool want = left_chunks > 0 && left_atoms >= left_chunks && acc * n >= total * (k + 1);
      if (must || want || i == a1 - 1) {
        chunks.push_back(Chunk{c, k, start, i + 1, cacc});
        start = i + 1;
        ++k;
        cacc = 0;
      }
    }
    if (k != n) fail("internal: chunk split mismatch");
  }
  std::stable_sort(chunks.begin(), chunks.end(),
                   [](const Chunk& a, const Chunk& b) { return a.cost > b.cost; });
  // Three-body force configurations first: their force-assembly items then
  // run while the energy configurations' chunks are still being served, and
  // the end of the launch is the smallest energy chunks, which wait for
  // nothing (largest first within each part).  Ordered by size alone, small
  // force configurations came last and their assembly items formed a tail:
  // 20% of the launch with fewer and fewer waves busy.
  if (tersoff)
    std::stable_partition(chunks.begin(), chunks.end(),
                          [&](const Chunk& a) { return a.c < ts_.Nc_force; });
  // A last lane block of at most 16 individuals runs packed: G >= 4 groups
  // of W lanes, each group on every G-th atom of the chunk.  (A packed atom
  // step costs several uniform ones, since its geometry is per lane: with
  // G = 2, P = 216, the launch took 0.607 ms packed against 0.521 ms
  // unpacked; with G = 4, P = 208, 0.458 against 0.523 ms.)
  int G_last = 1;
  if (tersoff && sh.pack && !loop_path_ && shell_M_ == 0) {
    const int Pr = P - (K - 1) * WAVE;
    int W = 1;
    while (W < Pr) W <<= 1;
    if (W <= 16) G_last = WAVE / W;
  }
  pl.groups_last = G_last;
  struct Costed {
    WorkItem w;
    long long cost;
  };
  std::vector<Costed> eval;
  eval.reserve(chunks.size() * K);
  for (const Chunk& ch : chunks)
    for (int k = 0; k < K; ++k) {
      const int G = k == K - 1 ? G_last : 1;
      const int n = ch.a1 - ch.a0, steps = (n + G - 1) / G;
      // (with the assembly of a one-chunk three-body force configuration)
      const long long asm_cost = tersoff && ch.c < ts_.Nc_force && nch[ch.c] == 1 ? 8LL * steps : 0;
      eval.push_back(Costed{WorkItem{ch.c, k, ch.chunk, ch.a0, ch.a1, 0, G, 0},
                            ch.cost * steps / n + asm_cost});
    }
  // three-body force configurations of several chunks: one force-assembly
  // item per chunk and lane block (a configuration of one chunk is
  // assembled by its phase-0 item)
  std::vector<Costed> assemble;
  if (tersoff)
    for (const Chunk& ch : chunks)
      if (ch.c < ts_.Nc_force && nch[ch.c] > 1)
        for (int k = 0; k < K; ++k) {
          const int G = k == K - 1 ? G_last : 1;
          const int n = ch.a1 - ch.a0, steps = (n + G - 1) / G;
          assemble.push_back(
            Costed{WorkItem{ch.c, k, ch.chunk, ch.a0, ch.a1, 1, G, 0}, 8LL * steps});
        }
  pl.n_items = (int)(eval.size() + assemble.size());
  const int waves_per_block = pl.block / WAVE;
  {
    int occ = sh.blocks_per_cu;
    if (occ <= 0) {
      switch (spec_.type) {
      case POT_RI: occ = ri_population_occupancy(pl.block); break;
      case POT_NN2B:
      case POT_NN2B_SPECIES: occ = nn2b_population_occupancy(pl.block); break;
      default:
        occ = shell_M_ > 0 ? tersoff_shell_occupancy(shell_M_, spec_.type == POT_TERSOFF2, pl.block)
              : loop_path_ ? tersoff_loop_occupancy(spec_.type == POT_TERSOFF2, pn.max_nn, pl.block)
                           : tersoff_population_occupancy(spec_.type == POT_TERSOFF2, G_last > 1, pl.block);
        break;
      }
      occ = std::max(occ, 1);
    }
    const int need = (pl.n_items + waves_per_block - 1) / waves_per_block;
    pl.grid = std::max(1, std::min(need, num_cu_ * occ));
    pl.occ = occ;
  }

  // Queues, nq / 8 per XCD (queue q is served first by XCD q / (nq / 8);
  // four per XCD unless the shape says otherwise): whole configurations,
  // balanced by cost (largest configuration to the least loaded queue).
  // Within a queue, phase-0 items largest chunk first, the lane blocks of a
  // chunk together; a force-assembly item follows the last phase-0 item of
  // its configuration by about one item per resident wave of the queue.
  // (at most 64: the kernel keeps one bit per queue in its closed mask)
  const int nq = std::max(1, std::min({sh.queues > 0 ? sh.queues : kQueues,
                                       pl.grid * waves_per_block, 64}));
  std::vector<long long> cfg_cost(Nc, 0);
  for (const Costed& e : eval) cfg_cost[e.w.c] += e.cost;
  for (const Costed& e : assemble) cfg_cost[e.w.c] += e.cost;
  std::vector<int> by_cost(Nc), cfg_q(Nc, 0);
  std::iota(by_cost.begin(), by_cost.end(), 0);
  std::stable_sort(by_cost.begin(), by_cost.end(),
                   [&](int a, int b) { return cfg_cost[a] > cfg_cost[b]; });
  std::vector<long long> load(nq, 0);
  for (int c : by_cost) {
    const int q = (int)(std::min_element(load.begin(), load.end()) - load.begin());
    cfg_q[c] = q;
    load[q] += cfg_cost[c];
  }
  // eval is in chunk order (largest chunk first, its lane blocks together):
  // a packed item stays beside its siblings, so the packed block's
  // force-assembly items do not all wait at the end of the launch
  const long long slack = std::max(1, pl.grid * waves_per_block / nq);
  std::vector<WorkItem> items;
  items.reserve(pl.n_items);
  std::vector<int> qstart(nq + 1, 0);
  for (int q = 0; q < nq; ++q) {
    qstart[q] = (int)items.size();
    // (position key, tie, item): phase-0 items at their rank in the queue,
    // assembly items at rank of their configuration's last phase-0 item +
    // slack (after it in any case)
    struct Keyed {
      long long key;
      int tie;
      WorkItem w;
    };
    std::vector<Keyed> qi;
    std::vector<long long> last(Nc, -1);
    long long pos = 0;
    for (const Costed& e : eval)
      if (cfg_q[e.w.c] == q) {
        qi.push_back(Keyed{pos, 0, e.w});
        last[e.w.c] = pos++;
      }
    int tie = 1;
    for (const Costed& e : assemble)
      if (cfg_q[e.w.c] == q) qi.push_back(Keyed{last[e.w.c] + slack, tie++, e.w});
    std::stable_sort(qi.begin(), qi.end(), [](const Keyed& a, const Keyed& b) {
      return a.key != b.key ? a.key < b.key : a.tie < b.tie;
    });
    for (const Keyed& x : qi) items.push_back(x.w);
  }
  qstart[nq] = (int)items.size();
  pl.nq = nq;

  hipStream_t st = stream_;
  pl.items.upload(items, st);
  pl.qstart.upload(qstart, st);
  // When the grid has a wave for every item, the first wave_slots are spread
  // over the queues in proportion to their lengths (wave w starts at the
  // queue that holds item w), so that each wave's first fetch finds an item.
  // Queues are balanced by cost, not count: with home queues by XCD alone, a
  // queue longer than its share of waves left its last items to waves that
  // had gone through the empty queues first (about 2.6 us per queue tried),
  // and the phase-0 items of small force configurations started up to 7 us
  // late.
  // (kept until the stream synchronisation below: the copy reads it)
  std::vector<int> home;
  int n_home = 0;
  if ((long long)pl.n_items <= (long long)pl.grid * waves_per_block) {
    home.resize(pl.n_items);
    for (int q = 0; q < nq; ++q)
      for (int i = qstart[q]; i < qstart[q + 1]; ++i) home[i] = q;
    pl.home.upload(home, st);
    n_home = pl.n_items;
  }
  pl.cfg_nchunks.upload(nch, st);
  pl.cfg_slot0.upload(slot0, st);
  pl.part.resize((size_t)std::max(slots, 1) * K * 8 * WAVE);
  pl.err.resize((size_t)K * 3 * Nc * WAVE);
  const int B_force =
    ts_.N_force > 0 ? pn.start[ts_.N_force - 1] + pn.NN[ts_.N_force - 1] : 0;
  pl.bondf.resize(tersoff ? std::max<size_t>((size_t)K * (B_force + ts_.N_force) * 3 * WAVE, 1) : 1);
  if (spec_.nn2b())
    pl.nn2b_table.resize((size_t)spec_.pair_codes() * K * nn2b_grid_desc().G * 3 * WAVE);
  const int cfg_group = config_group(Nc);
  const int groups = (Nc + cfg_group - 1) / cfg_group;
  pl.gpart.resize((size_t)K * groups * 3 * WAVE);
  // counters: cnt [Nc*K] | cnt2 [Nc*K] | grp_done [K*groups] | blk_done [K] |
  // (pad to 4 KiB) fetch [nq, kFetchStride apart] | done
  const size_t fetch0 = ((size_t)2 * Nc * K + (size_t)K * groups + K + 1023) / 1024 * 1024;
  // ... then done (one word) and, 8-byte aligned in the next 256 bytes, the
  // closed-queue mask
  const size_t closed0 = fetch0 + (size_t)nq * kFetchStride + 64;
  pl.counters.resize(closed0 + 2);
  pl.counters.zero(st);

  PopCtl& c = pl.ctl;
  c.items = pl.items.get();
  c.n_items = pl.n_items;
  c.nq = nq;
  c.qstart = pl.qstart.get();
  c.home = n_home > 0 ? pl.home.get() : nullptr;
  c.n_home = n_home;
  c.cfg_nchunks = pl.cfg_nchunks.get();
  c.cfg_slot0 = pl.cfg_slot0.get();
  c.part = pl.part.get();
  c.bondf = pl.bondf.get();
  c.B_force = B_force + ts_.N_force; // slots per lane block: bonds, then atoms
  c.err = pl.err.get();
  unsigned* ctr = pl.counters.get();
  c.cnt = ctr;
  c.cnt2 = ctr + (size_t)Nc * K;
  c.grp_done = ctr + (size_t)2 * Nc * K;
  c.blk_done = c.grp_done + (size_t)K * groups;
  c.fetch = ctr + fetch0;
  c.done = c.fetch + (size_t)nq * kFetchStride;
  c.closed = reinterpret_cast<unsigned long long*>(ctr + closed0);
  c.gpart = pl.gpart.get();
  c.cfg_group = cfg_group;
  c.spin_limit = spin_limit_;
  GPUGA_HIP(hipStreamSynchronize(st));
  pl.items_built = true;
}

} // namespace gpuga

namespace gpuga {

PopPlan& Fitness::plan(int P)
{
  auto it = plans_.find(P);
  if (it != plans_.end()) return *it->second;
  auto pl = std::make_unique<PopPlan>();
  if (quad_.on) build_quad_plan(*pl, P);
  else build_plan(*pl, P, launch_shape(P));
  PopPlan& ref = *pl;
  plans_[P] = std::move(pl);
  return ref;
}

void Fitness::launch_population(PopPlan& pl, const PopCtl& ctl, hipStream_t st, int grid)
{
  // (a persistent grid of any size drains the same queues; the results do
  // not depend on it)
  const int G = grid > 0 ? grid : pl.grid;
  switch (spec_.type) {
  case POT_RI: launch_ri_population(ctl, ds_.view, ds_.ri_tab.get(), G, pl.block, st); break;
  case POT_NN2B:
  case POT_NN2B_SPECIES: {
    NN2BGrid g = nn2b_grid_desc();
    launch_nn2b_tabulate(ctl, g, pl.nn2b_table.get(), st);
    launch_nn2b_population(ctl, ds_.view, g, pl.nn2b_table.get(), G, pl.block, st);
    break;
  }
  default: {
    if (shell_M_ > 0) {
      launch_tersoff_shell_population(ctl, ds_.view, shell_M_, ds_.shell_rec.get(), G, pl.block, st);
      break;
    }
    if (loop_path_) {
      launch_tersoff_loop_population(ctl, ds_.view, loop_, G, pl.block, st);
      break;
    }
    // the instantiation with the packed path only when the plan has packed
    // items; the one for lone waves when there is at most a workgroup per CU
    launch_tersoff_population(ctl, ds_.view, G, pl.block, pl.groups_last > 1, G <= num_cu_, st);
    break;
  }
  }
}

void Fitness::check_genes(int P, const float* genes) const
{
  // the pruned records leave out bonds beyond R2 at its upper bound, which
  // bounds R2 for genes in [0, 1] only
  if (!pruned_) return;
  for (int p = 0; p < P; ++p)
    if (!(genes[(size_t)p * spec_.V + spec_.V - 1] <= 1.0f))
      fail("genes must lie in [0, 1] (the outer cut-off radius gene exceeds 1)");
}

void Fitness::compute_async(int P, const float* genes, int share)
{
  if (P < 1) fail("population size must be positive");
  check_genes(P, genes);
  PopPlan& pl = plan(P);
  hipStream_t st = stream_;
  // (a set with quadratic forms, genes outside their range: the pair loop)
  const bool quad = quad_for(P, genes);
  if (!quad) ensure_items(pl);
  // Where the call before this one listed individuals that the forms do not
  // resolve, their launch follows the forms' at once, not after the host has
  // seen this call's list (which decides, so the results are the same): 70
  // individuals of 32 neurons, half of them listed, a call of 151 -> 121 us.
  const bool again = quad && pl.sharp_before && pl.items_built;
  pl.sharp_open = quad && !again;
  // The generation is launched directly (a graph of one or two kernels takes
  // 14 us longer to launch and wait for), and its last kernel writes the
  // results to the pinned block: a copy back would be one more operation on
  // the stream.
  PopCtl ctl = pl.ctl;
  ctl.terms = pl.h_out.get();
  ctl.fitness = reinterpret_cast<float*>(ctl.terms + 3 * (size_t)P);
  ctl.status = pl.h_status();
  *ctl.status = 0u;
  *pl.h_sharp() = 0u;
  float* h = pl.h_genes.get();
  if (quad && !again) {
    // The genes are read in place, each once or a few times.  From 64 Ki genes
    // on in two halves, the second one's copied while the first one's values
    // are computed (256 x 1153: a call of 77 us, 89 in one piece, 83 in three).
    ctl.genes = h;
    if (timing_) GPUGA_HIP(hipEventRecord(ev0_, st));
    const int parts = quad_.basis.rigid || (long)P * spec_.V < 65536 ? 1 : 2;
    for (int k = 0; k < parts; ++k) {
      const int p0 = (int)((long)P * k / parts), p1 = (int)((long)P * (k + 1) / parts);
      const size_t at = (size_t)p0 * spec_.V;
      std::memcpy(h + at, genes + at, sizeof(float) * (size_t)(p1 - p0) * spec_.V);
      launch_quad_values(pl, ctl, p0, p1 - p0, st);
    }
    launch_quad_eval(pl, ctl, st);
  } else {
    const size_t bytes = sizeof(float) * (size_t)P * spec_.V;
    std::memcpy(h, genes, bytes);
    // up to 64 KiB by a kernel: its launch costs less than a copy's
    if (bytes <= 64u * 1024u) launch_copy_in(h, pl.genes.get(), P * spec_.V, st);
    else GPUGA_HIP(hipMemcpyAsync(pl.genes.get(), h, bytes, hipMemcpyHostToDevice, st));
    if (timing_) GPUGA_HIP(hipEventRecord(ev0_, st));
    if (again) {
      launch_quad(pl, ctl, st);
      ctl = sharp_ctl(pl, ctl);
    }
    // share 1, 2, 4 or 8 (rounded up, at most 8): 1/share of the grid (the
    // quadratic forms' launches are short and fill a part of the GPU by
    // themselves)
    int j = 0;
    while (j < 3 && (1 << j) < share) ++j;
    launch_population(pl, ctl, st, std::max(1, (pl.grid + (1 << j) - 1) >> j));
  }
  if (timing_) GPUGA_HIP(hipEventRecord(ev1_, st));
  pending_P_ = P;
}

void Fitness::prepare(int P)
{
  if (opt_.backend != 1) plan(P);
}

void Fitness::run_ga(GA& ga, int first_generation, int generations, float* best, float* elite)
{
  // GA::compute (src/ga.cu:73-92) for `generations` generations with the
  // population on the device: each generation is the population launch on
  // one population buffer followed by the device GA step into the other;
  // the GA's random decisions are drawn on the host a batch ahead (they do
  // not depend on the fitness) and nothing returns to the host until the end
  const int P = ga.params().population_size, V = spec_.V;
  if (ga.V() != V) fail("the GA's parameter count differs from the potential's");
  if (first_generation < 0) fail("generation numbers start at 0");
  if (generations < 1) return;
  check_genes(P, ga.population().data());
  PopPlan& pl = plan(P);
  hipStream_t st = stream_;
  // (crossover and mutation keep genes in [0, 1]: one look at the start)
  const bool quad = quad_for(P, ga.population().data());
  if (!quad) ensure_items(pl);
  // the GA as it was before this call: staging draws advances its random
  // stream, so a failed run restores it
  const GA before = ga;
  if (!pl.dga || !pl.dga->matches(ga))
    pl.dga = std::make_unique<DeviceGA>(ga, pl.genes.get(), 1024, st, opt_.ga_batch);
  // Individuals that the forms do not resolve are evaluated again in their
  // generation from the start where the plan's last run or call had some, else
  // from the first generation that has, in which case the run starts again (its
  // generations up to there are the same bit for bit): a generation that needs none
  // is spared two launches.
  bool again = quad && pl.sharp_before && pl.items_built;
  if (!run_generations(pl, ga, before, first_generation, generations, quad, again, best, elite)) {
    ga = before;
    ensure_items(pl);
    again = true;
    run_generations(pl, ga, before, first_generation, generations, quad, again, best, elite);
  }
  if (quad) pl.sharp_before = *pl.h_sharp() != 0u;
}

bool Fitness::run_generations(PopPlan& pl, GA& ga, const GA& before, int first_generation,
                              int generations, bool quad, bool again, float* best, float* elite)
{
  const int V = spec_.V;
  hipStream_t st = stream_;
  DeviceGA& dga = *pl.dga;
  dga.upload(ga, first_generation, st);
  // batches double from one generation up to the staging capacity, so the
  // device starts after one generation's draws and the host then draws each
  // batch while the device runs the one before
  const int B = dga.batch();
  // (launched directly: replayed from a graph, ten generations of 50
  // individuals took 391 us against 357, four hundred the same per generation
  // on sets of 3 840 and 120 200 atoms, 31.5 and 280 us, and the capture cost a
  // process's first long run up to 4 ms)
  const int H = dga.history_cap();
  std::vector<float> h((size_t)H * (1 + V));
  const bool check = quad && pl.qeval.sharp.sums && !again;
  *pl.h_sharp() = 0u;
  const volatile unsigned* sharp = pl.h_sharp();
  int g = 0; // generations queued
  while (g < generations) {
    const int n = std::min(H, generations - g);
    if (g > 0) dga.restart_history(first_generation + g, st);
    if (timing_) GPUGA_HIP(hipEventRecord(ev0_, st));
    for (int b = 0, ramp = 1, nb = 0; b < n; b += nb, ramp = std::min(2 * ramp, B)) {
      nb = std::min({ramp, B, n - b});
      dga.stage(ga, first_generation + g + b, nb, st);
      const int k0 = (g + b) & 1;
      for (int i = 0; i < nb; ++i) {
        const int k = k0 ^ (i & 1);
        PopCtl ctl = pl.ctl;
        ctl.genes = dga.genes(k);
        if (quad) launch_quad(pl, ctl, st);
        else launch_population(pl, ctl, st);
        if (again) launch_population(pl, sharp_ctl(pl, ctl), st);
        dga.step(k, pl.ctl.fitness, st);
      }
      if (check && *sharp) {
        GPUGA_HIP(hipStreamSynchronize(st));
        return false;
      }
    }
    if (timing_) GPUGA_HIP(hipEventRecord(ev1_, st));
    const unsigned status = dga.collect((g + n) & 1, n, pl.ctl.status, st);
    if (check && *sharp) return false;
    if (timing_) {
      float ms = 0.0f;
      GPUGA_HIP(hipEventElapsedTime(&ms, ev0_, ev1_));
      kernel_ms_ += ms;
      kernel_launches_ += n;
    }
    if (status != 0u) {
      // the device population has advanced on invalid fitness values: drop
      // the device GA, and the GA handle returns to its state before this call
      ga = before;
      pl.dga.reset();
      discard_launch(pl);
    }
    dga.history(h.data(), n, st);
    for (int i = 0; i < n; ++i) {
      if (best) best[g + i] = h[(size_t)i * (1 + V)];
      if (elite)
        std::memcpy(elite + (size_t)(g + i) * V, &h[(size_t)i * (1 + V) + 1], sizeof(float) * V);
    }
    g += n;
  }
  dga.download(ga, generations & 1, st);
  return true;
}

void Fitness::discard_launch(PopPlan& pl)
{
  // A dependency wait of the population kernel ran out: this launch's results
  // are not valid.  A late phase-0 item may also have counted its chunk after
  // the assembly items returned the counter to zero, so every counter and the
  // result block (status word included) start from zero again before the
  // plan is used next (the launch has ended: the stream is synchronised).
  hipStream_t st = stream_;
  GPUGA_HIP(hipStreamSynchronize(st));
  pl.counters.zero(st);
  pl.out.zero(st);
  GPUGA_HIP(hipStreamSynchronize(st));
  fail("population kernel: force-assembly wait timed out; results discarded");
}

void Fitness::set_spin_limit(int spins)
{
  spin_limit_ = spins;
  for (auto& kv : plans_) kv.second->ctl.spin_limit = spins;
}

void Fitness::compute_wait(float* fitness, double* terms)
{
  const int P = pending_P_;
  if (P < 1) fail("no generation in flight");
  GPUGA_HIP(hipStreamSynchronize(stream_));
  PopPlan& pl = *plans_.at(P);
  if (timing_) {
    float ms = 0.0f;
    GPUGA_HIP(hipEventElapsedTime(&ms, ev0_, ev1_));
    kernel_ms_ += ms;
    ++kernel_launches_;
  }
  pending_P_ = 0;
  const double* h_terms = pl.h_out.get();
  const float* h_fitness = reinterpret_cast<const float*>(h_terms + 3 * (size_t)P);
  pl.sharp_before = *pl.h_sharp() != 0u;
  if (pl.sharp_open && pl.sharp_before) {
    // the individuals that the forms do not resolve, by the pair loop
    ensure_items(pl);
    hipStream_t st = stream_;
    GPUGA_HIP(hipMemcpyAsync(pl.genes.get(), pl.h_genes.get(),
                             sizeof(float) * (size_t)P * spec_.V, hipMemcpyHostToDevice, st));
    PopCtl ctl = sharp_ctl(pl, pl.ctl);
    ctl.terms = pl.h_out.get();
    ctl.fitness = reinterpret_cast<float*>(ctl.terms + 3 * (size_t)P);
    ctl.status = pl.h_status();
    if (timing_) GPUGA_HIP(hipEventRecord(ev0_, st));
    launch_population(pl, ctl, st);
    if (timing_) GPUGA_HIP(hipEventRecord(ev1_, st));
    GPUGA_HIP(hipStreamSynchronize(st));
    if (timing_) {
      float ms = 0.0f;
      GPUGA_HIP(hipEventElapsedTime(&ms, ev0_, ev1_));
      kernel_ms_ += ms;
    }
  }
  if (*pl.h_status() != 0u) discard_launch(pl);
  if (fitness) std::memcpy(fitness, h_fitness, sizeof(float) * P);
  if (terms) std::memcpy(terms, h_terms, sizeof(double) * 3 * P);
}

void Fitness::compute(int P, const float* genes, float* fitness, double* terms)
{
  if (opt_.backend == 1) {
    compute_plain(P, genes, fitness, terms);
    return;
  }
  compute_async(P, genes);
  compute_wait(fitness, terms);
}

void Fitness::compute_plain(int P, const float* genes, float* fitness, double* terms)
{
  plain_loop(P, genes, fitness, terms,
             PlainBuffers{nullptr, d_f_.get(), d_virial_.get(), d_pe_.get(), d_fit1_.get(),
                          d_cerr_.get(), d_terms1_.get()});
}

size_t Fitness::carve_plain(char* base, PlainBuffers* b) const
{
  size_t off = 0;
  auto take = [&](size_t bytes) {
    off = (off + 255) / 256 * 256;
    char* p = base ? base + off : nullptr;
    off += bytes;
    return p;
  };
  const size_t N = ts_.N, Nc = ts_.Nc;
  PlainBuffers x;
  const size_t ws = potential_->workspace_floats();
  x.ws = ws ? reinterpret_cast<float*>(take(ws * sizeof(float))) : nullptr;
  x.f = reinterpret_cast<float*>(take(3 * N * sizeof(float)));
  x.virial = reinterpret_cast<float*>(take(6 * N * sizeof(float)));
  x.pe = reinterpret_cast<float*>(take(N * sizeof(float)));
  x.fit1 = reinterpret_cast<float*>(take(sizeof(float)));
  x.cerr = reinterpret_cast<double*>(take(3 * Nc * sizeof(double)));
  x.terms1 = reinterpret_cast<double*>(take(3 * sizeof(double)));
  if (b) *b = x;
  return off;
}

size_t Fitness::noalloc_bytes() const { return carve_plain(nullptr, nullptr); }

void Fitness::compute_plain_noalloc(int P, const float* genes, float* fitness, double* terms)
{
  const size_t need = noalloc_bytes();
  if (need > kStaticWorkspaceBytes)
    fail(strfmt("the allocation-free path needs %zu bytes of device workspace for this "
                "training set; the fixed workspace holds %zu",
                need, kStaticWorkspaceBytes));
  if (!ws_static_) fail("the fixed device workspace was not set up on this device");
  int dev = 0;
  GPUGA_HIP(hipGetDevice(&dev));
  if (dev != device_) fail("the handle's device is not the current device");
  PlainBuffers b;
  carve_plain(static_cast<char*>(ws_static_), &b);
  plain_loop(P, genes, fitness, terms, b);
}

void Fitness::plain_loop(int P, const float* genes, float* fitness, double* terms,
                         const PlainBuffers& b)
{
  // src/fitness.cu:316-333: one parameter set at a time
  std::vector<float> params(spec_.V);
  const FitnessNorm nrm = norm();
  hipStream_t st = stream_;
  for (int n = 0; n < P; ++n) {
    denormalise_host(spec_, genes + (size_t)n * spec_.V, params.data());
    potential_->update_potential(params);
    if (timing_) GPUGA_HIP(hipEventRecord(ev0_, st));
    potential_->find_force(ds_.view, b.f, b.virial, b.pe, st, b.ws);
    launch_fitness_terms(ds_.view, nrm, b.f, b.virial, b.pe, b.cerr, b.fit1, b.terms1, st);
    if (timing_) GPUGA_HIP(hipEventRecord(ev1_, st));
    float fit = 0.0f;
    double t[3];
    GPUGA_HIP(hipMemcpyAsync(&fit, b.fit1, sizeof(float), hipMemcpyDeviceToHost, st));
    GPUGA_HIP(hipMemcpyAsync(t, b.terms1, sizeof(t), hipMemcpyDeviceToHost, st));
    GPUGA_HIP(hipStreamSynchronize(st));
    if (timing_) {
      float ms = 0.0f;
      GPUGA_HIP(hipEventElapsedTime(&ms, ev0_, ev1_));
      kernel_ms_ += ms;
      ++kernel_launches_;
    }
    fitness[n] = fit;
    if (terms) std::memcpy(terms + 3 * (size_t)n, t, sizeof(t));
  }
}

namespace {

// Maps the whole pages of [p, p + n) for writing, where the system can.
void populate(void* p, size_t n)
{
#ifdef MADV_POPULATE_WRITE
  constexpr int advice = MADV_POPULATE_WRITE;
#else
  constexpr int advice = 23; // its value on Linux (since 5.14)
#endif
  const size_t page = (size_t)sysconf(_SC_PAGESIZE);
  const size_t a = ((size_t)p + page - 1) / page * page, b = ((size_t)p + n) / page * page;
  if (b > a) (void)madvise(reinterpret_cast<void*>(a), b - a, advice);
}

} // namespace

void Fitness::find_force(const float* physical, float* f, float* virial, float* pe)
{
  std::vector<float> params(physical, physical + spec_.V);
  potential_->update_potential(params);
  hipStream_t st = stream_;
  potential_->find_force(ds_.view, d_f_.get(), d_virial_.get(), d_pe_.get(), st);
  GPUGA_HIP(hipGetLastError());
  const size_t N = ts_.N;
  // Results of more than 1.5 MiB through the pinned halves of h_atoms_, one
  // filled while the other is copied to the caller: a copy into pageable
  // memory runs at a third of the pinned rate (4 MB: a call of 357 -> 267 us;
  // 1 MB takes 113 us either way).
  const struct {
    const float* from;
    float* to;
    size_t n;
  } part[3] = {{d_pe_.get(), pe, N}, {d_f_.get(), f, 3 * N}, {d_virial_.get(), virial, 6 * N}};
  if (h_atoms_.size() == 0) {
    for (const auto& p : part)
      if (p.to)
        GPUGA_HIP(hipMemcpyAsync(p.to, p.from, sizeof(float) * p.n, hipMemcpyDeviceToHost, st));
    GPUGA_HIP(hipStreamSynchronize(st));
    return;
  }
  struct Piece {
    float* to = nullptr;
    size_t n = 0;
  } piece[2];
  // the caller's pages, while the GPU works: a copy into memory that has not
  // been touched yet would fault on each of them (4.8 MB: 300 us)
  for (const auto& p : part)
    if (p.to) populate(p.to, sizeof(float) * p.n);
  int k = 0;
  auto take = [&](int h) { // wait for half h and hand it to the caller
    if (!piece[h].to) return;
    GPUGA_HIP(hipEventSynchronize(ev_half_[h]));
    std::memcpy(piece[h].to, h_atoms_.get() + h * kHalf, sizeof(float) * piece[h].n);
    piece[h].to = nullptr;
  };
  for (const auto& p : part)
    for (size_t at = 0; p.to && at < p.n; at += kHalf, k ^= 1) {
      take(k);
      const size_t n = std::min(kHalf, p.n - at);
      GPUGA_HIP(hipMemcpyAsync(h_atoms_.get() + k * kHalf, p.from + at, sizeof(float) * n,
                               hipMemcpyDeviceToHost, st));
      GPUGA_HIP(hipEventRecord(ev_half_[k], st));
      piece[k] = Piece{p.to + at, n};
    }
  take(k);
  take(k ^ 1);
}

void Fitness::predict(const std::string& dir, const float* elite)
{
  // src/fitness.cu:335-390
  std::vector<float> params(spec_.V);
  denormalise_host(spec_, elite, params.data());
  const size_t N = ts_.N;
  std::vector<float> f(3 * N), w(6 * N), e(N);
  find_force(params.data(), f.data(), w.data(), e.data());
  auto open = [&](const char* name) {
    std::string path = dir + "/" + name;
    FILE* fid = std::fopen(path.c_str(), "w");
    if (!fid) fail(strfmt("Failed to open %s!", path.c_str()));
    return fid;
  };
  FILE* ff = open("force.out");
  for (int n = 0; n < ts_.N_force; ++n)
    std::fprintf(ff, "%g %g %g %g %g %g\n", f[n], f[n + N], f[n + N * 2], ts_.force_ref[n],
                 ts_.force_ref[n + N], ts_.force_ref[n + N * 2]);
  std::fclose(ff);
  // per-configuration sums in FP32, atom by atom, as the reference writes
  // them (src/fitness.cu:335-345): equal per-atom values give the same text
  auto per_config = [&](FILE* fid, const float* data, const float* ref) {
    for (int c = ts_.Nc_force; c < ts_.Nc; ++c) {
      float sum = 0.0f;
      for (int m = 0; m < ts_.Na[c]; ++m) sum += data[ts_.Na_sum[c] + m];
      std::fprintf(fid, "%g %g\n", sum, ref[c]);
    }
  };
  FILE* fe = open("energy.out");
  per_config(fe, e.data(), ts_.pe_ref.data());
  std::fclose(fe);
  FILE* fv = open("virial.out");
  for (int k = 0; k < 6; ++k) per_config(fv, w.data() + N * k, ts_.virial_ref.data() + ts_.Nc * k);
  std::fclose(fv);
}

int Fitness::heuristic_chunk_cost(int P) const
{
  const bool tersoff = spec_.type == POT_TERSOFF1 || spec_.type == POT_TERSOFF2;
  const std::vector<int>& pnn = tersoff ? population_neighbors().NN : nl_.NN;
  long long total = 0, maxcfg = 0;
  for (int c = 0; c < ts_.Nc; ++c) {
    long long t = 0;
    for (int i = ts_.Na_sum[c]; i < ts_.Na_sum[c] + ts_.Na[c]; ++i)
      t += atom_cost(spec_.type, pnn[i], c < ts_.Nc_force);
    total += t;
    maxcfg = std::max(maxcfg, t);
  }
  const long long K = (P + WAVE - 1) / WAVE;
  long long c = total * K / std::max<long long>(1, 16LL * num_cu_);
  c = std::max<long long>(c, 64);
  c = std::min<long long>(c, std::max<long long>(maxcfg, 64));
  return (int)c;
}

size_t Fitness::estimate_bytes(const PotentialSpec& s, const TrainSet& ts, int P,
                               const FitnessOptions& opt)
{
  // neighbour counts on the device (counting passes of the list build): of the
  // list, and of the bonds that the Tersoff population kernel reads
  const bool tersoff = s.type == POT_TERSOFF1 || s.type == POT_TERSOFF2;
  const float reach = std::max(0.0f, std::min(s.cutoff, tersoff_reach(s)));
  hipStream_t st = nullptr;
  GPUGA_HIP(hipStreamCreateWithFlags(&st, hipStreamNonBlocking));
  std::vector<int> nn, pnn;
  try {
    nn = count_neighbors_device(ts, s.cutoff, st);
    if (tersoff && reach < s.cutoff) pnn = count_neighbors_device(ts, reach, st);
  } catch (...) {
    (void)hipStreamDestroy(st);
    throw;
  }
  GPUGA_HIP(hipStreamDestroy(st));
  struct Lists {
    size_t bonds = 0, tri = 0, force_bonds = 0, cost = 0;
    int most = 0;
  };
  auto lists = [&](const std::vector<int>& c) {
    Lists l;
    for (int i = 0; i < (int)c.size(); ++i) {
      l.bonds += c[i];
      l.tri += (size_t)c[i] * c[i];
      if (i < ts.N_force) l.force_bonds += c[i];
      l.cost += atom_cost(s.type, c[i], i < ts.N_force);
      l.most = std::max(l.most, c[i]);
    }
    l.bonds = std::max<size_t>(l.bonds, 1);
    return l;
  };
  const Lists full = lists(nn), used = pnn.empty() ? full : lists(pnn);
  const size_t N = ts.N, Nc = ts.Nc, B = full.bonds;
  size_t b = N * sizeof(int) * 5 + Nc * sizeof(int) * 2 + B * (3 * sizeof(int) + 16);
  if (tersoff) {
    b += full.tri * 16 + B * 4 * 5; // triplets, per-individual scratch
    // the pruned list's tables (dropped after set-up where records are built)
    if (!pnn.empty()) b += N * 4 * 3 + used.bonds * (3 * sizeof(int) + 16) + used.tri * 16;
    if (used.most <= 4)
      b += N * record_floats4(4) * 16 + (N - ts.N_force) * kMomWords * sizeof(float);
    else if (const int M = tersoff_shell_slots(used.most))
      b += tersoff_shell_floats4(ts.N, M) * 16;
  } else {
    b += B * 48 + N * 16; // the pair loop's tables
    if (s.type == POT_RI) b += B * 16;
  }
  b += Nc * 7 * sizeof(float) + N * 3 * sizeof(float);  // references
  b += N * 10 * sizeof(float) + Nc * 3 * sizeof(double); // per-atom outputs
  const size_t K = (P + WAVE - 1) / WAVE;
  // error terms, and partials of the work items: at most 16 a CU beside one per
  // configuration and lane block, where the options set no other size
  const size_t items = opt.chunk_cost > 0
                         ? K * used.cost / opt.chunk_cost
                         : std::min<size_t>(K * used.cost / 64, 16 * 256);
  b += K * 3 * Nc * WAVE * sizeof(double) + (Nc * K + items) * 8 * WAVE * sizeof(double);
  if (tersoff) b += K * (used.force_bonds + ts.N_force) * 3 * WAVE * sizeof(float);
  if (s.nn2b()) b += (size_t)3 * s.pair_codes() * opt.nn2b_grid * K * WAVE * sizeof(float);
  const int points = s.pair_codes() * opt.nn2b_grid;
  if (s.type == POT_RI || (s.nn2b() && opt.nn2b_grid >= 256 && opt.nn2b_grid <= 2048 && points <= 4096)) {
    // Quadratic forms, with every element in use (rigid ion: at most 8 a type;
    // U's columns enter its virials and forces nowhere): value blocks of the
    // population, the three forms, and while they are built the rows and the
    // partial tiles.
    const size_t ce = s.nn2b() ? points / (2 * QB) : 24;
    const size_t nb[3] = {ce + 1, s.nn2b() ? 2 * ce + 1 : ce + 1, s.nn2b() ? 2 * ce + 1 : ce + 1};
    b += (2 * ce + 1) * QB * sizeof(double) * (size_t)(P + QP);
    for (size_t n : nb) b += quad_tiles((long)n) * QB * QB * sizeof(double);
    const size_t er = (nb[0] + 6 * nb[1]) * quad_step(kQuadConfigs, ts.Nc - ts.Nc_force);
    const size_t fr = 3 * nb[2] * quad_step(kQuadAtoms, ts.N_force);
    b += (std::max(er, fr) * QB + quad_part_size((long)nb[1])) * sizeof(double);
  }
  b += (size_t)P * s.V * sizeof(float) + (size_t)P * 4 * sizeof(double);
  return b;
}

std::vector<double> Fitness::trace(int P, const float* genes)
{
  check_genes(P, genes);
  PopPlan& pl = plan(P);
  ensure_items(pl);
  hipStream_t st = stream_;
  const size_t n = pl.n_items;
  const size_t F = kTraceFields;
  DeviceBuffer<unsigned long long> buf(std::max<size_t>(F * n, 1));
  buf.zero(st);
  std::vector<WorkItem> items(n);
  pl.items.download(items.data(), n, st);
  GPUGA_HIP(hipMemcpyAsync(pl.genes.get(), genes, sizeof(float) * (size_t)P * spec_.V,
                           hipMemcpyHostToDevice, st));
  pl.ctl.trace = buf.get();
  launch_population(pl, pl.ctl, st);
  pl.ctl.trace = nullptr;
  std::vector<unsigned long long> t(F * n);
  buf.download(t.data(), t.size(), st);
  unsigned status = 0;
  GPUGA_HIP(hipMemcpyAsync(&status, pl.ctl.status, sizeof status, hipMemcpyDeviceToHost, st));
  GPUGA_HIP(hipStreamSynchronize(st));
  if (status != 0u) discard_launch(pl);
  int khz = 0;
  GPUGA_HIP(hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, device_));
  const double ns_per_tick = 1e6 / std::max(khz, 1);
  unsigned long long t0 = ~0ull;
  for (size_t i = 0; i < n; ++i) t0 = std::min(t0, t[F * i + 1]);
  auto rel = [&](unsigned long long x) { return ((double)x - (double)t0) * ns_per_tick; };
  std::vector<double> rows;
  rows.reserve(12 * n);
  for (size_t i = 0; i < n; ++i) {
    const WorkItem& w = items[i];
    const unsigned long long* x = &t[F * i];
    rows.insert(rows.end(), {(double)w.c, (double)w.k, (double)w.chunk, (double)w.a0,
                             (double)w.a1, (double)w.phase, (double)x[0], rel(x[1]), rel(x[2]),
                             x[3] ? rel(x[3]) : NAN, x[4] ? rel(x[4]) : NAN,
                             x[5] ? rel(x[5]) : NAN});
  }
  return rows;
}

double Fitness::time_plan(int P, const LaunchShape& sh, int reps, int* occ)
{
  PopPlan pl;
  build_plan(pl, P, sh);
  if (occ) *occ = pl.occ;
  std::vector<float> genes((size_t)P * spec_.V);
  for (size_t i = 0; i < genes.size(); ++i) genes[i] = (float)((i * 2654435761u) % 1000) / 1000.0f;
  hipStream_t st = stream_;
  GPUGA_HIP(hipMemcpyAsync(pl.genes.get(), genes.data(), sizeof(float) * genes.size(),
                           hipMemcpyHostToDevice, st));
  launch_population(pl, pl.ctl, st); // warm-up
  GPUGA_HIP(hipEventRecord(ev0_, st));
  for (int r = 0; r < reps; ++r) launch_population(pl, pl.ctl, st);
  GPUGA_HIP(hipEventRecord(ev1_, st));
  GPUGA_HIP(hipStreamSynchronize(st));
  float ms = 0.0f;
  GPUGA_HIP(hipEventElapsedTime(&ms, ev0_, ev1_));
  return ms / reps;
}

LaunchShape Fitness::launch_shape(int P)
{
  if (opt_.chunk_cost > 0) return option_shape();
  auto t = tuned_.find(P);
  if (t == tuned_.end()) {
    if (quad_.on && spec_.nn2b()) {
      // The loop serves parts of the population, of any size, for which a full
      // launch's timing is no guide; nor is it worth 95 ms of the first call.
      // Items of this cost, against 100 and 700: all of 256 individuals on
      // 57 600 wurtzite atoms 352 (386, 403) us a call, 3 of them 285 (310, 417),
      // 70 individuals 223 (251, 345); 100 on 10 800 atoms with species 197 (200,
      // 248).
      LaunchShape sh = option_shape();
      sh.chunk_cost = 300;
      tuned_[P] = sh;
    } else {
      tune(P);
    }
    t = tuned_.find(P);
  }
  return t->second;
}

void Fitness::plan_shape(int P, int& chunk_cost, int& queues, int& blocks_per_cu,
                         int& groups_last)
{
  if (P < 1) fail("population size must be positive");
  PopPlan& pl = plan(P);
  ensure_items(pl);
  chunk_cost = pl.chunk_cost;
  queues = pl.nq;
  blocks_per_cu = pl.occ;
  groups_last = pl.groups_last;
}

int Fitness::autotune(int P)
{
  if (!quad_.on) return tune(P);
  // Of a set with quadratic forms only the calls that they do not take run the
  // population kernel, and its tables may not be there: the first such call
  // chooses its shape (ensure_items).  With the built-in size, too coarse for
  // rigid ion, calls of 200 individuals on 48 000 oxide atoms with a gene
  // outside [0, 1] took 592 us; 361 us tuned.
  const auto t = tuned_.find(P);
  return t == tuned_.end() ? heuristic_chunk_cost(P) : t->second.chunk_cost;
}

int Fitness::tune(int P)
{
  // Candidate work-item sizes: the whole-configuration cost spread over
  // 1/2 .. 1/32 of the resident waves, and the largest configuration's cost
  // halved step by step (small sets, where latency rather than balance
  // sets the time).  Then, at the best size, the rest of the launch shape
  // that the options leave open: the queue count, one resident workgroup
  // per CU fewer than the occupancy calculator allows, and, when the last
  // lane block qualifies, packing it or not.  Each choice is kept only if
  // its launch is faster.
  const bool tersoff = spec_.type == POT_TERSOFF1 || spec_.type == POT_TERSOFF2;
  const std::vector<int>& pnn = tersoff ? population_neighbors().NN : nl_.NN;
  long long total = 0, maxcfg = 0;
  for (int c = 0; c < ts_.Nc; ++c) {
    long long t = 0;
    for (int i = ts_.Na_sum[c]; i < ts_.Na_sum[c] + ts_.Na[c]; ++i)
      t += atom_cost(spec_.type, pnn[i], c < ts_.Nc_force);
    total += t;
    maxcfg = std::max(maxcfg, t);
  }
  const int K = (P + WAVE - 1) / WAVE;
  const long long waves = (long long)num_cu_ * 4 * 2;
  std::vector<int> cands;
  for (int div : {1, 2, 4, 8, 16}) {
    long long c = total * K / std::max<long long>(1, waves * div / 2);
    c = std::max<long long>(c, 64);
    c = std::min<long long>(c, std::max<long long>(maxcfg, 64));
    cands.push_back((int)c);
  }
  cands.push_back((int)std::max<long long>(maxcfg, 64)); // whole configurations
  for (long long c = maxcfg / 2; c >= 64; c /= 2) cands.push_back((int)c);
  std::sort(cands.begin(), cands.end());
  cands.erase(std::unique(cands.begin(), cands.end()), cands.end());
  LaunchShape best = option_shape();
  best.chunk_cost = cands.back();
  double best_ms = 1e30;
  int best_occ = 0;
  auto consider = [&](const LaunchShape& sh, int reps) {
    int occ = 0;
    const double ms = time_plan(P, sh, reps, &occ);
    if (opt_.verbose)
      std::printf("autotune P=%d chunk_cost=%d queues=%d blocks_per_cu=%d pack=%d: %.4f ms\n", P,
                  sh.chunk_cost, sh.queues, sh.blocks_per_cu, sh.pack, ms);
    if (ms < best_ms) {
      best_ms = ms;
      best = sh;
      best_occ = occ;
    }
  };
  auto with_cost = [&](int c) {
    LaunchShape sh = best;
    sh.chunk_cost = c;
    return sh;
  };
  const LaunchShape base = best;
  for (int c : cands) {
    LaunchShape sh = base;
    sh.chunk_cost = c;
    consider(sh, 3);
  }
  // the neighbourhood of the best (the coarse candidates are a factor of
  // two apart, and launch times differ by about 1% from run to run), the
  // best one timed again alongside
  const int coarse = best.chunk_cost;
  best_ms = 1e30;
  for (double f : {0.6, 0.75, 0.87, 1.0, 1.15, 1.33, 1.6}) {
    const long long c = std::llround(coarse * f);
    if (c >= 64 && c <= std::max<long long>(maxcfg, 64)) consider(with_cost((int)c), 6);
  }
  // queue count (the kernel keeps at most 64)
  if (opt_.queues <= 0) {
    const LaunchShape inc = best;
    for (int nq : {kQueues / 2, kQueues * 2}) {
      LaunchShape sh = inc;
      sh.queues = std::min(nq, 64);
      consider(sh, 6);
    }
  }
  // one resident workgroup per CU fewer (fewer waves sharing a SIMD)
  if (opt_.blocks_per_cu <= 0 && best_occ > 1) {
    LaunchShape sh = best;
    sh.blocks_per_cu = best_occ - 1;
    consider(sh, 6);
  }
  // the packed last lane block against plain lanes
  if (opt_.pack_lanes && tersoff && !loop_path_ && shell_M_ == 0) {
    const int Pr = P - (K - 1) * WAVE;
    if (Pr <= 16) {
      LaunchShape sh = best;
      sh.pack = 0;
      consider(sh, 6);
    }
  }
  tuned_[P] = best;
  return best.chunk_cost;
}

} // namespace gpuga
