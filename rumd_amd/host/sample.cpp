// Sample (include/rumd/Sample.h, src/Sample.cu): CalcF over the potential
// list, FP64 sums, and the captured step blocks of the run loop.
#include <algorithm>
#include <iostream>

#include "rumd_host.h"

namespace {
constexpr unsigned kPbThreshold = 10000;  // src/Sample.cu:36-39
}

Sample::Sample(unsigned pb, unsigned tp) : pb_(pb), tp_(tp) {
  Device::GetDevice().Init();
  hip_check(hipStreamCreate(&stream_), "Sample", "Sample");
  scalars_.resize(16);
}

Sample::~Sample() {
  InvalidateGraphs();
  if (stream_) (void)hipStreamDestroy(stream_);
}

void Sample::SetPB_TP(unsigned pb, unsigned tp) {
  if (pb * std::max(tp, 1u) > 1024)
    throw RUMD_cudaResourceError("Sample", "SetPB_TP", "Too many threads per block (pb*tp>maxthreads)");
  pb_ = pb;
  tp_ = tp;
  if (GetNumberOfParticles()) {
    // reallocate with the new padding, keeping the configuration
    const unsigned n = GetNumberOfParticles();
    std::vector<float> r(4ull * n), v(4ull * n), im(4ull * n), lo;
    std::vector<int32_t> t(n);
    pd_.Get("r", r.data(), stream_);
    if (pd_.MixedPositions()) {
      lo.resize(4ull * n);
      pd_.Get("rlo", lo.data(), stream_);
    }
    pd_.Get("v", v.data(), stream_);
    pd_.Get("im", im.data(), stream_);
    pd_.GetTypes(t.data(), stream_);
    const unsigned nt = pd_.GetNumberOfTypes();
    std::vector<float> masses(nt);
    for (unsigned k = 0; k < nt; ++k) masses[k] = pd_.GetMass(k);
    SetNumberOfParticles(n);
    for (unsigned k = 0; k < nt; ++k) pd_.SetMass(k, masses[k]);
    pd_.SetTypes(t.data(), stream_);
    std::vector<float> x3(3ull * n);
    for (unsigned i = 0; i < n; ++i)
      for (int k = 0; k < 3; ++k) x3[3ull * i + k] = r[4ull * i + k];
    if (!lo.empty() && mixed_) {
      std::vector<double> x64(3ull * n);
      for (unsigned i = 0; i < n; ++i)
        for (int k = 0; k < 3; ++k)
          x64[3ull * i + k] = static_cast<double>(r[4ull * i + k]) + static_cast<double>(lo[4ull * i + k]);
      pd_.SetPositionsFP64(x64.data(), stream_);
    } else {
      pd_.SetPositions(x3.data(), stream_);
    }
    for (unsigned i = 0; i < n; ++i)
      for (int k = 0; k < 3; ++k) x3[3ull * i + k] = v[4ull * i + k];
    pd_.SetVelocities(x3.data(), stream_);
    for (unsigned i = 0; i < n; ++i)
      for (int k = 0; k < 3; ++k) x3[3ull * i + k] = im[4ull * i + k];
    pd_.SetImages(x3.data(), stream_);
  }
}

void Sample::SetMixedPrecisionPositions(bool on) {
  if (on == mixed_) return;
  mixed_ = on;
  if (GetNumberOfParticles()) SetPB_TP(pb_, tp_);
}

void Sample::SetNumberOfParticles(unsigned n) {
  if (n == 0) return;
  if (pb_ == 0) pb_ = n > kPbThreshold ? 64 : 32;
  if (tp_ == 0) tp_ = n > kPbThreshold ? 1 : 4;
  InvalidateGraphs();
  pd_.SetNumberOfParticles(n, pb_, mixed_);
  workspace_.resize(rumdx_workspace_bytes(n));
  if (verbose_) {
    std::cout << "Setting number of particles: N = " << n << ", pb = " << pb_ << ", tp = " << tp_
              << ", virtual particles = " << pd_.GetNumberOfVirtualParticles() << std::endl;
  }
  for (Potential* p : potentials_) p->SetSample(this);
  if (itg_) itg_->SetSample(this);
}

void Sample::SetSimulationBox(SimulationBox* box) {
  box_ = box;
  InvalidateGraphs();
  if (GetNumberOfParticles())
    for (Potential* p : potentials_) p->SetSample(this);
}

void Sample::SetPotential(Potential* p) {
  potentials_.clear();
  AddPotential(p);
}

void Sample::AddPotential(Potential* p) {
  p->SetVerbose(verbose_);
  // non-constraint potentials go to the front (src/Sample.cu:268-274), pair
  // potentials ahead of the others: the first force call of a step then is a
  // pair potential's, whose list build may sort the particles, before any
  // other term (bonds, angles) has been written in the old order
  auto pos = potentials_.begin();
  if (!dynamic_cast<PairPotential*>(p))
    while (pos != potentials_.end() && dynamic_cast<PairPotential*>(*pos)) ++pos;
  potentials_.insert(pos, p);
  if (GetNumberOfParticles()) p->SetSample(this);
  InvalidateGraphs();
}

void Sample::SetIntegrator(Integrator* itg) {
  itg_ = itg;
  if (GetNumberOfParticles()) itg_->SetSample(this);
  InvalidateGraphs();
}

unsigned Sample::GetNumberOfDOFs() const {
  if (user_dofs_) return user_dofs_;
  const unsigned n = GetNumberOfParticles();
  return n ? 3 * n - 3 : 0;  // src/Sample.cu:294-310
}

void Sample::SetMass(unsigned type, float mass) { pd_.SetMass(type, mass); }

float Sample::GetMeanMass() const {
  double m = 0.0;
  for (unsigned t = 0; t < GetNumberOfTypes(); ++t) m += GetNumberThisType(t) * GetMass(t);
  return static_cast<float>(m / GetNumberOfParticles());
}

NeighborList* Sample::FusedCheckList() {
  if (potentials_.empty()) return nullptr;
  auto* pp = dynamic_cast<PairPotential*>(potentials_.front());
  if (!pp || pp->GetNeighborList().GetResolvedMethod() == NeighborList::NONE) return nullptr;
  return &pp->GetNeighborList();
}

void Sample::CalcF(bool calc_stresses) {
  if (!box_) throw RUMD_Error("Sample", "CalcF", "No simulation box has been set");
  if (!GetNumberOfParticles()) throw RUMD_Error("Sample", "CalcF", "Sample has no particles");
  if (potentials_.empty()) std::cerr << "Warning [Sample::CalcF]: No potential has been set" << std::endl;
  BumpSlotEpoch();
  for (size_t k = 0; k < potentials_.size(); ++k) potentials_[k]->CalcF(k == 0, calc_stresses);
}

void Sample::Synchronize() {
  // the lists' flags come back with this synchronisation (a potential that has
  // since been given to another sample launches on that one's stream, which
  // HandleOverflow waits for)
  for (Potential* p : potentials_) {
    auto* pp = dynamic_cast<PairPotential*>(p);
    if (pp != nullptr && pp->GetSample() == this) pp->GetNeighborList().QueueFlagsRead();
  }
  hip_check(hipStreamSynchronize(stream_), "Sample", "Synchronize");
  for (Potential* p : potentials_)
    if (auto* pp = dynamic_cast<PairPotential*>(p))
      if (pp->GetNeighborList().HandleOverflow()) InvalidateGraphs();
}

// FP64 device sums of the per-particle energies / virials (the host loops of
// Sample::GetPotentialEnergy / GetVirial, src/Sample.cu:353-391).
double Sample::GetPotentialEnergy() {
  Synchronize();
  rumdx_check(rumdx_reduce_f4(pd_.d_f.get(), GetNumberOfParticles(), 8u, scalars_.get(), workspace_.get(), stream_),
              "Sample", "GetPotentialEnergy");
  hip_check(hipStreamSynchronize(stream_), "Sample", "GetPotentialEnergy");
  double pe = scalars_.get()[3];
  for (Potential* p : potentials_)
    if (!p->EnergyIncludedInParticleSum()) pe += p->GetPotentialEnergy();
  return pe;
}

double Sample::GetVirial() {
  Synchronize();
  rumdx_check(rumdx_reduce_f4(pd_.d_w.get(), GetNumberOfParticles(), 8u, scalars_.get(), workspace_.get(), stream_),
              "Sample", "GetVirial");
  hip_check(hipStreamSynchronize(stream_), "Sample", "GetVirial");
  double w = scalars_.get()[3] / 6.0;
  for (Potential* p : potentials_)
    if (!p->EnergyIncludedInParticleSum()) w += p->GetVirial();
  return w;
}

// Sample::GetStress (src/Sample.cu:393-444), kinetic part included.
std::vector<double> Sample::GetStress() {
  Synchronize();
  const unsigned n = GetNumberOfParticles();
  double* out = scalars_.get();
  // configurational sums: sts, then w.y and w.z; kinetic sums (all six)
  rumdx_check(rumdx_reduce_f4(pd_.d_sts.get(), n, 15u, out, workspace_.get(), stream_), "Sample", "GetStress");
  rumdx_check(rumdx_reduce_f4(pd_.d_w.get(), n, 6u, out + 4, workspace_.get(), stream_), "Sample", "GetStress");
  rumdx_check(rumdx_kinetic_stress(pd_.Descriptor(), out + 8, workspace_.get(), stream_), "Sample", "GetStress");
  hip_check(hipStreamSynchronize(stream_), "Sample", "GetStress");
  const double conf[6] = {out[0], out[1], out[2], out[3], out[5], out[6]};
  double s[6];
  for (int k = 0; k < 6; ++k) s[k] = conf[k] - out[8 + k];
  const double V = box_->GetVolume();
  std::vector<double> r(6);
  for (int k = 0; k < 6; ++k) r[k] = 0.5 * s[k] / V;
  return r;
}

// Spatial sorting on demand (Sample::SortParticles): the sorted neighbour
// list reorders particles by cell at every rebuild, so a sort is a rebuild.
void Sample::SortParticles() {
  for (Potential* p : potentials_)
    if (auto* pp = dynamic_cast<PairPotential*>(p))
      if (pp->GetNeighborList().IsSorted()) pp->GetNeighborList().ResetNeighborList();
}

void Sample::InvalidateGraphs() {
  for (auto& kv : graphs_) (void)hipGraphExecDestroy(kv.second.exec);
  graphs_.clear();
}

void Sample::SetFusedSteps(bool on) {
  if (on == fused_steps_) return;
  fused_steps_ = on;
  InvalidateGraphs();
}

float Sample::TimeFusedStepKernel(unsigned reps) {
  PrepareRun();
  PairPotential* pp = FusedStepPotential();
  if (pp == nullptr) throw RUMD_Error("Sample", "TimeFusedStepKernel", "the steps of this sample take no fused kernel");
  return pp->TimeFusedStepKernel(reps, itg_->GetTimeStep());
}

PairPotential* Sample::FusedStepPotential() {
  if (!fused_steps_ || potentials_.size() != 1 || dynamic_cast<IntegratorNVT*>(itg_) == nullptr) return nullptr;
  auto* pp = dynamic_cast<PairPotential*>(potentials_.front());
  return (pp != nullptr && pp->CanFuseStep()) ? pp : nullptr;
}

// The potential whose steps run as chains of one kernel each inside captured
// blocks (small samples), or null.
PairPotential* Sample::ChainPotential() {
  if (!fused_steps_ || potentials_.size() != 1 || dynamic_cast<IntegratorNVT*>(itg_) == nullptr) return nullptr;
  auto* pp = dynamic_cast<PairPotential*>(potentials_.front());
  return (pp != nullptr && pp->CanChainSteps()) ? pp : nullptr;
}

void Sample::PrepareRun() {
  if (!box_) throw RUMD_Error("Sample", "Run", "No simulation box has been set");
  if (!itg_) throw RUMD_Error("Sample", "Run", "Integrator has not been set");
  if (potentials_.empty()) throw RUMD_Error("Sample", "Run", "Potential has not been set");
  for (Potential* p : potentials_)
    if (auto* pp = dynamic_cast<PairPotential*>(p)) {
      if (pp->NumTypesInTable() != GetNumberOfTypes()) pp->Initialize();
      NeighborList& nl = pp->GetNeighborList();
      nl.EnsureAllocated();
      // a full sort is due (first build, or positions set by the host): run
      // it now, outside any graph, so that recorded steps hold the tile
      // re-sort of skin-triggered rebuilds (the build settles its capacities)
      if (nl.NeedsFullSort()) nl.UpdateNBlist();
    }
  rumdx_bonded_term terms[RUMDX_MAX_BONDED_TERMS];
  if (FusedStepPotential() != nullptr || ChainPotential() != nullptr || BondedTerms(terms) != 0)
    pd_.EnsureNextPositions();
}

uint32_t Sample::BondedTerms(rumdx_bonded_term* terms) {
  if (!fused_steps_ || potentials_.size() < 2 || potentials_.size() > 1 + RUMDX_MAX_BONDED_TERMS ||
      molecules_ == nullptr || molecules_->SlotIndexArray() == nullptr ||
      dynamic_cast<IntegratorNVT*>(itg_) == nullptr || dynamic_cast<PairPotential*>(potentials_.front()) == nullptr)
    return 0;
  uint32_t n = 0;
  for (size_t k = 1; k < potentials_.size(); ++k)
    if (!potentials_[k]->BondedTerm(&terms[n++])) return 0;
  return n;
}

void Sample::StepOnce(bool zero_momentum, bool store_forces, bool slots_known) {
  if (zero_momentum) itg_->SetMomentumToZero();
  PairPotential* pp = FusedStepPotential();
  if (pp != nullptr && pd_.HasNextPositions()) {
    BumpSlotEpoch();
    static_cast<IntegratorNVT*>(itg_)->IntegrateFused(*pp, store_forces);
    return;
  }
  rumdx_bonded_term terms[RUMDX_MAX_BONDED_TERMS];
  const uint32_t nterms = pd_.HasNextPositions() ? BondedTerms(terms) : 0u;
  if (nterms != 0) {
    if (!box_) throw RUMD_Error("Sample", "CalcF", "No simulation box has been set");
    BumpSlotEpoch();
    const bool known =
        slots_known && static_cast<PairPotential*>(potentials_.front())->GetNeighborList().KeepsSlotIndex();
    potentials_.front()->CalcF(true, false);
    const uint32_t* slot_of = known ? molecules_->SlotIndexArray() : molecules_->SlotIndex();
    static_cast<IntegratorNVT*>(itg_)->IntegrateBonded(terms, nterms, slot_of, store_forces);
    return;
  }
  CalcF(false);
  itg_->Integrate();
}

std::vector<std::pair<unsigned, bool>> Sample::RunSegments(unsigned long first_step, unsigned nsteps,
                                                           unsigned block, unsigned momentum_interval) const {
  if (block == 0) block = 1;
  std::vector<std::pair<unsigned, bool>> seg;
  const unsigned long end = first_step + nsteps;
  for (unsigned long i = first_step; i < end;) {
    unsigned long stop = std::min<unsigned long>(i + block, end);
    if (momentum_interval > 0) {
      // the next reset step after i ends the block before it
      const unsigned long next_reset = (i / momentum_interval + 1) * momentum_interval;
      stop = std::min(stop, next_reset);
    }
    seg.emplace_back(static_cast<unsigned>(stop - i), momentum_interval > 0 && i % momentum_interval == 0);
    i = stop;
  }
  return seg;
}

// Records nsteps steps into a graph (nothing runs); the host-side state that
// recording changes (the fused skin check's pending mark) is restored, so the
// graph can be launched later as if recorded then.
Sample::Block Sample::CaptureBlock(unsigned nsteps, bool reset_first) {
  NeighborList* nl = FusedCheckList();
  float* home = pd_.d_r.get();
  hipGraph_t g = nullptr;
  hip_check(hipStreamBeginCapture(stream_, hipStreamCaptureModeThreadLocal), "Sample", "RunSteps");
  try {
    // the first step re-checks the skin explicitly; later steps use the
    // check fused into the previous integrator step
    if (nl) nl->ResetFusedCheck();
    if (PairPotential* chain = ChainPotential()) {
      if (reset_first) itg_->SetMomentumToZero();
      static_cast<IntegratorNVT*>(itg_)->IntegrateChain(*chain, nsteps);
    } else {
      // the forces of the inner steps are replaced before anything reads them
      auto* itg = nl != nullptr ? dynamic_cast<IntegratorNVT*>(itg_) : nullptr;
      if (itg) itg->Defer(true);
      for (unsigned k = 0; k < nsteps; ++k) StepOnce(k == 0 && reset_first, k + 1 == nsteps, k > 0);
      if (itg) itg->Defer(false);
    }
    // fused steps alternate the two position arrays: the graph ends in the
    // one it starts from (a copy after an odd number of them)
    pd_.MovePositionsTo(home, stream_);
  } catch (...) {
    if (auto* itg = dynamic_cast<IntegratorNVT*>(itg_)) itg->DropDue();
    (void)hipStreamEndCapture(stream_, &g);
    if (g) (void)hipGraphDestroy(g);
    if (pd_.d_r.get() != home) pd_.SwapPositions();  // nothing ran
    throw;
  }
  hip_check(hipStreamEndCapture(stream_, &g), "Sample", "RunSteps");
  hipGraphExec_t exec = nullptr;
  const hipError_t e = hipGraphInstantiate(&exec, g, nullptr, nullptr, 0);
  (void)hipGraphDestroy(g);
  hip_check(e, "Sample", "RunSteps");
  return Block{exec, home};
}

unsigned Sample::PrepareRunSteps(unsigned long first_step, unsigned nsteps, unsigned block,
                                 unsigned momentum_interval) {
  PrepareRun();
  NeighborList* nl = FusedCheckList();
  const bool pending = nl != nullptr && nl->FusedCheckPending();
  unsigned made = 0;
  for (const auto& key : RunSegments(first_step, nsteps, block, momentum_interval)) {
    if (key.first < 2 || graphs_.count(key)) continue;
    graphs_.emplace(key, CaptureBlock(key.first, key.second));
    ++made;
  }
  if (nl) {
    if (pending) nl->NoteFusedCheck(); else nl->ResetFusedCheck();
  }
  return made;
}

void Sample::RunSteps(unsigned long first_step, unsigned nsteps, unsigned block, unsigned momentum_interval) {
  PrepareRun();
  for (const auto& key : RunSegments(first_step, nsteps, block, momentum_interval)) {
    if (key.first < 2) {
      StepOnce(key.second);
      continue;
    }
    auto it = graphs_.find(key);
    if (it == graphs_.end()) it = graphs_.emplace(key, CaptureBlock(key.first, key.second)).first;
    // the graph's first step checks the skin itself (see CaptureBlock)
    if (NeighborList* nl = FusedCheckList()) nl->ResetFusedCheck();
    pd_.MovePositionsTo(it->second.r_home, stream_);
    hip_check(hipGraphLaunch(it->second.exec, stream_), "Sample", "RunSteps");
    for (Potential* p : potentials_)
      if (auto* pp = dynamic_cast<PairPotential*>(p)) pp->GetNeighborList().NoteFlagsChanged();
    if (NeighborList* nl = FusedCheckList()) nl->NoteFusedCheck();
  }
  Synchronize();
}

// Sample::ReadMoleculeData (src/Sample.cu, MoleculeData::ReadTopology).
void Sample::ReadMoleculeData(const std::string& topology_file) {
  CreateMoleculeData()->ReadTopology(topology_file);
  InvalidateGraphs();
}

MoleculeData* Sample::GetMoleculeData() { return molecules_.get(); }

MoleculeData* Sample::CreateMoleculeData() {
  if (!GetNumberOfParticles()) throw RUMD_Error("Sample", "ReadMoleculeData", "Sample has no particles");
  InvalidateGraphs();
  molecules_ = std::make_unique<MoleculeData>(this);
  return molecules_.get();
}
