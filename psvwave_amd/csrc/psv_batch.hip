// psv_batch.hip -- batched forward runs over many models of uneven size.
//
// Each member is a full Model (its own HBM buffers and injection tables).
// The batch keeps, in device memory, the launch arguments of every
// (member, shot, buffer parity) and the list of (member, tile) pairs of all
// members, so one launch per time step advances every model: the grid is
// the union of all members' tiles, large enough to fill the GPU even when
// each model alone is small.  A shot's whole time loop can be captured as
// one HIP graph and replayed.
#include "psv_batch.h"

#include <algorithm>
#include <limits>

namespace psv {

namespace {
void hip_check(hipError_t e, const char *what) {
  if (e == hipSuccess) return;
  (void)hipGetLastError();  // reported here, not by the check of a later launch
  throw RuntimeError(std::string(what) + ": " + hipGetErrorString(e));
}

// n doubles of device memory, zero in the stream's order.
void *zeroed(size_t n, hipStream_t s) {
  void *p = nullptr;
  hip_check(hipMalloc(&p, n * sizeof(double)), "hipMalloc");
  const hipError_t e = launch_fill((double *)p, (long long)n, 0.0, s);
  if (e != hipSuccess) (void)hipFree(p);
  hip_check(e, "zero-fill");
  return p;
}
}  // namespace

Batch::Batch(const std::vector<Config> &cfgs) {
  if (cfgs.empty()) throw ValueError("a batch needs at least one model");
  nt_ = cfgs[0].nt;
  n_shots_ = cfgs[0].n_shots;
  for (const Config &c : cfgs)
    if (c.nt != nt_ || c.n_shots != n_shots_)
      throw ValueError("all models of a batch must share nt and n_shots");
  // the members run their own calls (parameters, adjoint sources, misfits)
  // on the batch's stream: one stream for the whole batch
  create_stream(&stream_);
  try {
    for (const Config &c : cfgs) models_.emplace_back(new Model(c, stream_));
  } catch (...) {
    models_.clear();
    destroy_stream(stream_);
    throw;
  }
  hip_check(hipEventCreate(&ev_[0]), "hipEventCreate");
  hip_check(hipEventCreate(&ev_[1]), "hipEventCreate");
  for (auto &m : models_) points_ += m->grid_points();
  bool lean = true;
  for (auto &m : models_) lean = lean && m->lean_ok();
  if (lean) variant_ = kLeanTz16RingClamp;
  build_tables();
}

Batch::~Batch() {
  if (stream_) (void)hipStreamSynchronize(stream_);
  clear_graphs();
  if (descs_) (void)hipFree(descs_);
  if (ldescs_) (void)hipFree(ldescs_);
  if (tiles_) (void)hipFree(tiles_);
  for (auto p : zero_ptrs_)
    if (p) (void)hipFree(p);
  if (zero_lens_) (void)hipFree(zero_lens_);
  clear_gradient_tables();
  loops_.clear();
  if (loop_cells_) (void)hipFree(loop_cells_);
  if (loop_sync_) (void)hipFree(loop_sync_);
  if (loop_poison_) (void)hipFree(loop_poison_);
  if (loop_status_) (void)hipHostFree(loop_status_);
  for (auto e : ev_)
    if (e) (void)hipEventDestroy(e);
  models_.clear();  // the members run on stream_
  destroy_stream(stream_);
}

Model &Batch::model(int m) {
  if (m < 0 || m >= size()) throw ValueError("model index out of range");
  return *models_[m];
}

const Model &Batch::model(int m) const {
  if (m < 0 || m >= size()) throw ValueError("model index out of range");
  return *models_[m];
}

void Batch::clear_graphs() {
  for (auto g : graphs_)
    if (g) (void)hipGraphExecDestroy(g);
  graphs_.clear();
  if (graph_all_) (void)hipGraphExecDestroy(graph_all_);
  graph_all_ = nullptr;
}

void Batch::set_persistent(bool on) {
  if (on && variant_ != kLeanTz8)
    throw ValueError("the persistent batch loop runs step variant 9 (lean 64 x 8)");
  persistent_ = on;
  clear_graphs();
}

void Batch::set_graph_mode(bool on) {
  if (!on) clear_graphs();
  graph_mode_ = on;
}

void Batch::clear_gradient_tables() {
  if (gfwd_) (void)hipFree(gfwd_);
  if (gadj_) (void)hipFree(gadj_);
  gfwd_ = gadj_ = nullptr;
}

void Batch::set_variant(int variant, int xcd_remap) {
  if (variant != kFusedTz8 && variant != kFusedTz16 && variant != kTwoStepTz8 &&
      variant != kTwoStepTz16 && !step_is_lean(variant))
    throw ValueError("batched runs use step variants 0, 1, 6, 7, 8-13 or 18-28");
  if (step_is_lean(variant))
    for (auto &m : models_)
      if (!m->lean_ok())
        throw ValueError("a member of the batch cannot use the lean step variants");
  variant_ = variant;
  resident_ = false;  // an explicit choice: that kernel, step by step
  xcd_remap_ = xcd_remap ? 1 : 0;
  if (variant != kLeanTz8) persistent_ = false;
  clear_graphs();
  clear_gradient_tables();  // descriptors hold injection-table pointers
  build_tables();
}

void Batch::build_tables() {
  std::vector<int2> tiles;
  std::vector<StepArgs> descs;
  for (size_t m = 0; m < models_.size(); ++m) {
    models_[m]->set_step_variant(variant_, xcd_remap_);
    for (int t = 0; t < models_[m]->tile_count(); ++t)
      tiles.push_back(make_int2((int)m, t));
    for (int s = 0; s < n_shots_; ++s)
      for (int p = 0; p < 2; ++p) descs.push_back(models_[m]->forward_launch_args(s, p));
  }
  if (tiles.size() > (size_t)std::numeric_limits<int>::max())
    throw ValueError("too many tiles in one batch");
  ntiles_ = (int)tiles.size();
  hip_check(hipStreamSynchronize(stream_), "sync");
  if (descs_) hip_check(hipFree(descs_), "hipFree");
  if (ldescs_) hip_check(hipFree(ldescs_), "hipFree");
  if (tiles_) hip_check(hipFree(tiles_), "hipFree");
  descs_ = ldescs_ = nullptr;
  tiles_ = nullptr;
  hip_check(hipMalloc((void **)&descs_, std::max<size_t>(1, descs.size()) * sizeof(StepArgs)),
            "hipMalloc");
  hip_check(hipMalloc((void **)&tiles_, std::max<size_t>(1, tiles.size()) * sizeof(int2)),
            "hipMalloc");
  hip_check(hipMemcpy(descs_, descs.data(), descs.size() * sizeof(StepArgs),
                      hipMemcpyHostToDevice),
            "upload");
  hip_check(hipMemcpy(tiles_, tiles.data(), tiles.size() * sizeof(int2),
                      hipMemcpyHostToDevice),
            "upload");
  ensure_zero_table(0);
}

// The device tables of every member's state set `set` (built before any
// stream capture: the allocation and upload may not be captured).
void Batch::ensure_zero_table(int set) {
  if (!zero_ptrs_[set]) {
    std::vector<double *> ptrs;
    std::vector<long long> lens;
    for (auto &m : models_) {
      m->state_arrays(set, ptrs);
      lens.resize(ptrs.size(), m->padded_points());
      zero_max_ = std::max(zero_max_, m->padded_points());
    }
    for (double *p : ptrs)
      if (!p) throw RuntimeError("a state buffer set is not allocated");
    hip_check(hipMalloc((void **)&zero_ptrs_[set], ptrs.size() * sizeof(double *)),
              "hipMalloc");
    hip_check(hipMemcpy(zero_ptrs_[set], ptrs.data(), ptrs.size() * sizeof(double *),
                        hipMemcpyHostToDevice),
              "upload");
    if (!zero_lens_) {
      hip_check(hipMalloc((void **)&zero_lens_, lens.size() * sizeof(long long)), "hipMalloc");
      hip_check(hipMemcpy(zero_lens_, lens.data(), lens.size() * sizeof(long long),
                          hipMemcpyHostToDevice),
                "upload");
    }
  }
}

void Batch::enqueue_zero_states(int set) {
  if (!zero_ptrs_[set]) throw RuntimeError("state zeroing table missing");
  const int n = 10 * size();
  const int bx = (int)std::min<long long>(64, (zero_max_ + 2047) / 2048);
  hip_check(launch_zero_many(zero_ptrs_[set], zero_lens_, n, std::max(1, bx), stream_),
            "zero states");
}

// Zero every member's state, then advance `nsteps` steps of shot i_shot
// with one launch per step (or per pair of steps), then form the receiver
// running sums when the two-step kernels recorded increments.
void Batch::enqueue_loop(int i_shot, int nsteps) {
  enqueue_zero_states(0);
  if (persistent_) {
    BatchLaunch b{descs_, tiles_, ntiles_, n_shots_, i_shot, 0, 0, 0, xcd_remap_, 0, 1};
    hip_check(launch_batch_persistent(b, 0, nsteps, stream_), "persistent batch loop");
    return;
  }
  const bool two = step_is_two_step(variant_);
  int launch = 0;
  for (int k = 0; k < nsteps;) {
    const bool pair = two && k + 1 < nsteps;
    BatchLaunch b{descs_, tiles_, ntiles_, n_shots_, i_shot, launch & 1,
                  k, k + 1, xcd_remap_, 0, 1};
    hip_check(launch_batch_step(variant_, pair, b, stream_), "batch step");
    k += pair ? 2 : 1;
    ++launch;
  }
  if (two && nsteps == nt_)
    for (auto &m : models_) m->enqueue_receiver_scan(i_shot, stream_);
}

// ---- resident loops ----

// The kernel for launches of `shots` loops of every member: the first that
// holds them all (kLoopFits), or where several launches are needed 28-row tiles,
// two blocks per compute unit: the blocks of a unit mostly belong to different
// loops and hide each other's exchange.  -1: some member fits no kernel.
int Batch::choose_loop_kind(int shots) {
  for (auto &m : models_)
    if (!m->lean_ok() || m->derived().nx < 8 || m->derived().nz < 8) return -1;
  // tiles of all loops and of the largest member
  auto tiles = [&](int kind, long long *most) {
    long long sum = 0;
    *most = 0;
    for (auto &m : models_) {
      const long long t =
          (long long)loop_tiles_x(m->derived().nx) * loop_tiles_z(m->derived().nz, kind);
      sum += t * shots;
      *most = std::max(*most, t);
    }
    return sum;
  };
  auto usable = [&](int kind) {  // the tables of every member
    for (auto &m : models_)
      if (m->loop_tile_columns(kind) == 0) return false;
    return true;
  };
  long long most = 0;
  for (const LoopFit &f : kLoopFits)
    if (tiles(f.kind, &most) <= loop_capacity(f.kind, f.per_unit) && usable(f.kind)) return f.kind;
  for (int k : {kNumLoopKinds - 2, kNumLoopKinds - 1})
    if (tiles(k, &most) > 0 && most <= loop_capacity(k) && usable(k)) return k;
  return -1;
}

bool Batch::resident_available() {
  if (!resident_ || graph_mode_ || persistent_) return false;
  if (loop_skip_ > 0) {
    --loop_skip_;
    return false;
  }
  if (loop_kind_ < 0) loop_kind_ = choose_loop_kind(n_shots_);
  return loop_kind_ >= 0;
}

// The launches of a call, built on first use and kept only once they are
// whole.  Null where the device has no room for them: the call then runs by
// steps, and the next one tries again.
Batch::LoopLaunches *Batch::loop_launches(int which, int i_shot, int steps) {
  const int key = which + 8 * i_shot;
  auto it = loops_.find(key);
  if (it != loops_.end() && which != 4) return &it->second;
  hip_check(hipStreamSynchronize(stream_), "sync");
  try {
    LoopLaunches p = plan_loops(which, i_shot, steps);
    ensure_loop_words((int)p.launches.size());
    return &(loops_[key] = std::move(p));
  } catch (const RuntimeError &) {
    return nullptr;
  }
}

// which: 0 forward_all, 1 forward of i_shot, 2 / 3 forward / adjoint of i_shot
// with the one-shot snapshot stores, 4 the first `steps` steps of forward_all.
Batch::LoopLaunches Batch::plan_loops(int which, int i_shot, int steps) {
  LoopLaunches p;
  // (a launch of one shot may have room for smaller tiles than one of all)
  const int kind = p.kind = which == 0 || which == 4 ? loop_kind_ : choose_loop_kind(1);
  p.forward = which != 3;
  std::vector<LoopRef> refs;
  for (int m = 0; m < size(); ++m)
    for (int s = 0; s < n_shots_; ++s)
      if (which == 0 || which == 4 || s == i_shot)
        refs.push_back({m, s, p.forward, which == 2 || which == 3});
  auto tiles = [&](const LoopRef &r) {
    return models_[r.member]->loop_tile_columns(kind) *
           models_[r.member]->loop_tile_rows_of(kind);
  };
  // first fit, the largest loops first
  std::stable_sort(refs.begin(), refs.end(),
                   [&](const LoopRef &a, const LoopRef &b) { return tiles(a) > tiles(b); });
  std::vector<std::vector<LoopRef>> bins;
  std::vector<int> room;
  for (const LoopRef &r : refs) {
    size_t b = 0;
    while (b < bins.size() && room[b] < tiles(r)) ++b;
    if (b == bins.size()) {
      bins.push_back({});
      room.push_back(loop_capacity(kind));
    }
    bins[b].push_back(r);
    room[b] -= tiles(r);
  }
  const size_t cell_bytes = loop_cells_bytes(kind, 1);
  if (!loop_cells_) {  // for every kernel: the launches of all calls keep pointers into them
    size_t bytes = 0;
    for (int k = 0; k < kNumLoopKinds; ++k)
      bytes = std::max(bytes, loop_cells_bytes(k, loop_capacity(k)));
    loop_cells_ = zeroed(bytes / 8, stream_);
    loop_cells_bytes_ = bytes;
  }
  std::vector<LoopArgs> args;
  std::vector<int4> blocks;
  for (const auto &bin : bins) {
    const int first = (int)p.loops.size(), block0 = (int)blocks.size();
    for (size_t i = 0; i < bin.size(); ++i) {
      const LoopRef &r = bin[i];
      Model &m = *models_[r.member];
      LoopArgs a = m.loop_args(kind, r.shot, r.forward);
      a.cells = (char *)loop_cells_ + cell_bytes * (blocks.size() - block0);
      a.cells_bytes = (unsigned)(cell_bytes * tiles(r));
      if (r.snaps) {
        double *const *store = m.shot_snapshot_store();
        for (int f = 0; f < 5; ++f) a.snap[f] = store[f];
      }
      if (which == 4) a.k1 = steps;
      const int ntx = m.loop_tile_columns(kind);
      for (int t = 0; t < tiles(r); ++t)
        blocks.push_back(make_int4((int)i, t % ntx, t / ntx, 0));
      args.push_back(a);
      p.loops.push_back(r);
    }
    p.launches.emplace_back(first, (int)blocks.size() - block0);
    p.first_block.push_back(block0);
  }
  auto put = [&](auto &dst, const auto &v) {
    void *d = nullptr;
    hip_check(hipMalloc(&d, v.size() * sizeof(v[0])), "hipMalloc");
    dst.reset((typename std::remove_reference_t<decltype(dst)>::pointer)d);
    hip_check(hipMemcpy(d, v.data(), v.size() * sizeof(v[0]), hipMemcpyHostToDevice), "upload");
  };
  put(p.args, args);
  put(p.blocks, blocks);
  return p;
}

// Meeting and status words of as many launches, and the poison word.
void Batch::ensure_loop_words(int launches) {
  if (!loop_poison_) loop_poison_ = (unsigned *)zeroed(1, stream_);
  if (launches <= loop_words_) return;
  // the words there are go last: launches already planned use them
  void *sync = nullptr, *status = nullptr;
  hip_check(hipMalloc(&sync, (size_t)launches * 8), "hipMalloc");
  const hipError_t e = hipHostMalloc(&status, launches * sizeof(unsigned), hipHostMallocDefault);
  if (e != hipSuccess) (void)hipFree(sync);
  hip_check(e, "hipHostMalloc");
  if (loop_sync_) (void)hipFree(loop_sync_);
  if (loop_status_) (void)hipHostFree(loop_status_);
  loop_sync_ = (unsigned *)sync;
  loop_status_ = (unsigned *)status;
  loop_words_ = launches;
}

// The next launches are refused, whatever the step variant.
void Batch::refuse_next_loops() {
  ensure_loop_words(0);
  hip_check(hipStreamSynchronize(stream_), "sync");
  const unsigned one = 1;
  hip_check(hipMemcpy(loop_poison_, &one, sizeof(one), hipMemcpyHostToDevice), "poison");
  resident_ = true;
  loop_skip_ = 0;
}

// Runs the launches of a call (`steps` time steps each) and waits for them:
// whether all took place.  Those that were refused (psv_loop.h) or could not be
// made are, with `redo`, run step by step as whole loops.
bool Batch::run_loops(LoopLaunches &p, int steps, bool redo) {
  const int n = (int)p.launches.size();
  for (int i = 0; i < n; ++i) loop_status_[i] = kLoopNotRun;
  hip_check(launch_fill((double *)loop_sync_, n, 0.0, stream_), "clear loop words");
  for (int i = 0; i < n; ++i) {
    if (loop_tag_ + (unsigned)steps < loop_tag_) {  // the tags start over
      hip_check(launch_fill((double *)loop_cells_,
                            (long long)(loop_cells_bytes_ / 8), 0.0, stream_),
                "clear cells");
      loop_tag_ = 1;
    }
    LoopLaunch l;
    l.loops = p.args.get() + p.launches[i].first;
    l.blocks = p.blocks.get() + p.first_block[i];
    l.nblocks = p.launches[i].second;
    l.tag0 = loop_tag_;
    l.sync = loop_sync_ + 2 * i;
    l.poison = loop_poison_;
    l.status = loop_status_ + i;
    loop_tag_ += (unsigned)steps;  // spent, also where an error follows the launch
    try {
      gated_launch_loop(p.kind, !p.forward, l, stream_);
    } catch (const RuntimeError &) {
      break;
    }
  }
  hip_check(hipStreamSynchronize(stream_), "hipStreamSynchronize");
  bool missing = false;
  for (int i = 0; i < n; ++i) {
    if (loop_status_[i] == kLoopStalled)
      throw RuntimeError("a resident time loop made no progress");
    missing = missing || loop_status_[i] == kLoopNotRun;
  }
  if (!missing) return true;
  loop_skip_ = 64;
  hip_check(launch_fill((double *)loop_poison_, 1, 0.0, stream_), "clear poison");
  for (int i = 0; i < n && redo; ++i) {
    if (loop_status_[i] != kLoopNotRun) continue;
    const int last = i + 1 < n ? p.launches[i + 1].first : (int)p.loops.size();
    for (int k = p.launches[i].first; k < last; ++k)
      models_[p.loops[k].member]->enqueue_store_loop(p.loops[k].shot, p.loops[k].forward,
                                                     p.loops[k].snaps);
  }
  hip_check(hipStreamSynchronize(stream_), "hipStreamSynchronize");
  return false;
}

void Batch::forward(int i_shot) {
  if (i_shot < 0 || i_shot >= n_shots_)
    throw ValueError("i_shot is outside [0, n_shots)");
  if (LoopLaunches *p = resident_available() ? loop_launches(1, i_shot, nt_) : nullptr) {
    hip_check(hipEventRecord(ev_[0], stream_), "hipEventRecord");
    run_loops(*p, nt_);
    end_timing();
    return;
  }
  hip_check(hipEventRecord(ev_[0], stream_), "hipEventRecord");
  if (graph_mode_) {
    if (graphs_.size() != (size_t)n_shots_) graphs_.assign(n_shots_, nullptr);
    if (!graphs_[i_shot]) {
      hip_check(hipStreamSynchronize(stream_), "sync");
      hipGraph_t graph = nullptr;
      hip_check(hipStreamBeginCapture(stream_, hipStreamCaptureModeThreadLocal),
                "hipStreamBeginCapture");
      try {
        enqueue_loop(i_shot, nt_);
      } catch (...) {
        hipGraph_t g2 = nullptr;
        (void)hipStreamEndCapture(stream_, &g2);
        if (g2) (void)hipGraphDestroy(g2);
        throw;
      }
      hip_check(hipStreamEndCapture(stream_, &graph), "hipStreamEndCapture");
      hipGraphExec_t exec = nullptr;
      hipError_t e = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
      (void)hipGraphDestroy(graph);
      hip_check(e, "hipGraphInstantiate");
      graphs_[i_shot] = exec;
      hip_check(hipEventRecord(ev_[0], stream_), "hipEventRecord");
    }
    hip_check(hipGraphLaunch(graphs_[i_shot], stream_), "hipGraphLaunch");
  } else {
    enqueue_loop(i_shot, nt_);
  }
  hip_check(hipEventRecord(ev_[1], stream_), "hipEventRecord");
  hip_check(hipStreamSynchronize(stream_), "hipStreamSynchronize");
  float ms = 0.f;
  hip_check(hipEventElapsedTime(&ms, ev_[0], ev_[1]), "hipEventElapsedTime");
  loop_ms_ += ms;
}

bool Batch::lockstep_available() {
  if (n_shots_ < 2 || n_shots_ > Model::kMaxStateSets || !step_is_lean(variant_) ||
      persistent_ ||
      no_lockstep_room_ || (long long)ntiles_ * n_shots_ > std::numeric_limits<int>::max())
    return false;
  if (ldescs_) return true;
  try {
    for (auto &m : models_) m->ensure_state_sets(n_shots_);
  } catch (const RuntimeError &) {
    // no room: keep what was allocated and run shot by shot; clear the
    // failed allocation's error so that the next launch check does not
    // report it
    (void)hipGetLastError();
    no_lockstep_room_ = true;
    return false;
  }
  for (int set = 1; set < n_shots_; ++set) ensure_zero_table(set);
  std::vector<StepArgs> descs;
  for (auto &m : models_)
    for (int s = 0; s < n_shots_; ++s)
      for (int p = 0; p < 2; ++p) descs.push_back(m->forward_launch_args(s, p, s));
  hip_check(hipMalloc((void **)&ldescs_, descs.size() * sizeof(StepArgs)), "hipMalloc");
  hip_check(hipMemcpy(ldescs_, descs.data(), descs.size() * sizeof(StepArgs),
                      hipMemcpyHostToDevice),
            "upload");
  return true;
}

// Zero the state sets of every member (one per shot), then advance `nsteps`
// steps of every shot with one launch per step (lockstep_available must
// hold).
void Batch::enqueue_lockstep_loop(int nsteps) {
  for (int set = 0; set < n_shots_; ++set) enqueue_zero_states(set);
  for (int k = 0; k < nsteps; ++k) {
    BatchLaunch b{ldescs_, tiles_, ntiles_ * n_shots_, n_shots_, -1, k & 1,
                  k, k + 1, xcd_remap_, 0, 1};
    hip_check(launch_batch_step(variant_, false, b, stream_), "batch step");
  }
}

// The end of a timed region whose work has been enqueued on stream_.
void Batch::end_timing() {
  hip_check(hipEventRecord(ev_[1], stream_), "hipEventRecord");
  hip_check(hipStreamSynchronize(stream_), "hipStreamSynchronize");
  float ms = 0.f;
  hip_check(hipEventElapsedTime(&ms, ev_[0], ev_[1]), "hipEventElapsedTime");
  loop_ms_ += ms;
}

void Batch::forward_all() {
  if (LoopLaunches *p = resident_available() ? loop_launches(0, 0, nt_) : nullptr) {
    hip_check(hipEventRecord(ev_[0], stream_), "hipEventRecord");
    run_loops(*p, nt_);
    end_timing();
    return;
  }
  if (!lockstep_available()) {
    for (int s = 0; s < n_shots_; ++s) forward(s);
    return;
  }
  hip_check(hipEventRecord(ev_[0], stream_), "hipEventRecord");
  if (graph_mode_) {
    // the whole loop (state zeroing and nt launches) captured once and
    // replayed: one host launch per call; the tables it reads were built
    // by lockstep_available, outside the capture
    if (!graph_all_) {
      hip_check(hipStreamSynchronize(stream_), "sync");
      hipGraph_t graph = nullptr;
      hip_check(hipStreamBeginCapture(stream_, hipStreamCaptureModeThreadLocal),
                "hipStreamBeginCapture");
      try {
        enqueue_lockstep_loop(nt_);
      } catch (...) {
        hipGraph_t g2 = nullptr;
        (void)hipStreamEndCapture(stream_, &g2);
        if (g2) (void)hipGraphDestroy(g2);
        throw;
      }
      hip_check(hipStreamEndCapture(stream_, &graph), "hipStreamEndCapture");
      hipGraphExec_t exec = nullptr;
      hipError_t e = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
      (void)hipGraphDestroy(graph);
      hip_check(e, "hipGraphInstantiate");
      graph_all_ = exec;
      hip_check(hipEventRecord(ev_[0], stream_), "hipEventRecord");
    }
    hip_check(hipGraphLaunch(graph_all_, stream_), "hipGraphLaunch");
  } else {
    enqueue_lockstep_loop(nt_);
  }
  hip_check(hipEventRecord(ev_[1], stream_), "hipEventRecord");
  hip_check(hipStreamSynchronize(stream_), "hipStreamSynchronize");
  float ms = 0.f;
  hip_check(hipEventElapsedTime(&ms, ev_[0], ev_[1]), "hipEventElapsedTime");
  loop_ms_ += ms;
}

// Time loop of shot i_shot for every member with the gradient descriptors:
// forward storing each member's snapshots of this shot, or adjoint (time
// steps nt-1 .. 0) correlating with them.
void Batch::enqueue_gradient_loop(int i_shot, bool forward) {
  enqueue_zero_states(0);
  const StepArgs *descs = forward ? gfwd_ : gadj_;
  for (int k = 0; k < nt_; ++k) {
    const int it = forward ? k : nt_ - 1 - k;
    BatchLaunch b{descs, tiles_, ntiles_, n_shots_, i_shot, k & 1, it, it, xcd_remap_,
                  1, si_};
    hip_check(launch_batch_step(variant_, false, b, stream_, nullptr, nullptr,
                                !forward && it % si_ == 0),
              "batch gradient step");
  }
}

void Batch::gradients() {
  if (!batch_gradient_variant_ok(variant_))
    throw ValueError("batched gradients need step variant 0, 1, 8-13 or 18-28");
  si_ = models_[0]->config().snapshot_interval;
  for (auto &m : models_)
    if (m->config().snapshot_interval != si_)
      throw ValueError("batched gradients need one snapshot_interval for all members");
  if (nt_ % si_ != 0)
    throw ValueError("Snapshot interval and size of accumulator don't match! "
                     "(nt must be a multiple of snapshot_interval)");
  // everything is allocated before anything is changed
  bool resident = resident_available();
  for (int s = 0; s < n_shots_ && resident; ++s)
    resident = loop_launches(2, s, nt_) && loop_launches(3, s, nt_);
  if (!resident && !gfwd_) {
    std::vector<StepArgs> f, a;
    for (auto &m : models_) {
      double *const *store = m->shot_snapshot_store();
      for (int s = 0; s < n_shots_; ++s)
        for (int p = 0; p < 2; ++p) {
          f.push_back(m->forward_launch_args(s, p));
          a.push_back(m->adjoint_launch_args(s, p));
          for (int q = 0; q < 5; ++q) f.back().snap[q] = a.back().snap[q] = store[q];
        }
    }
    try {
      hip_check(hipMalloc((void **)&gfwd_, f.size() * sizeof(StepArgs)), "hipMalloc");
      hip_check(hipMalloc((void **)&gadj_, a.size() * sizeof(StepArgs)), "hipMalloc");
      hip_check(hipMemcpy(gfwd_, f.data(), f.size() * sizeof(StepArgs), hipMemcpyHostToDevice),
                "upload");
      hip_check(hipMemcpy(gadj_, a.data(), a.size() * sizeof(StepArgs), hipMemcpyHostToDevice),
                "upload");
    } catch (...) {
      clear_gradient_tables();
      throw;
    }
  }
  for (auto &m : models_) m->reset_kernels();
  hip_check(hipEventRecord(ev_[0], stream_), "hipEventRecord");
  for (int s = 0; s < n_shots_; ++s) {
    // forward s, its adjoint sources (each member's own stream), adjoint s:
    // the kernels accumulate shot by shot, as in the reference's order
    if (resident)
      run_loops(*loop_launches(2, s, nt_), nt_);
    else
      enqueue_gradient_loop(s, true);
    hip_check(hipStreamSynchronize(stream_), "hipStreamSynchronize");
    for (auto &m : models_) m->calculate_l2_adjoint_sources();
    if (resident)
      run_loops(*loop_launches(3, s, nt_), nt_);
    else
      enqueue_gradient_loop(s, false);
  }
  hip_check(hipEventRecord(ev_[1], stream_), "hipEventRecord");
  hip_check(hipStreamSynchronize(stream_), "hipStreamSynchronize");
  float ms = 0.f;
  hip_check(hipEventElapsedTime(&ms, ev_[0], ev_[1]), "hipEventElapsedTime");
  loop_ms_ += ms;
  for (auto &m : models_) {
    m->calculate_l2_misfit();
    m->map_kernels_to_velocity();
  }
}

void Batch::misfits(double *out) {
  for (size_t m = 0; m < models_.size(); ++m)
    out[m] = models_[m]->calculate_l2_misfit();
}

double Batch::autotune(int steps, int *best, double *ms_per_variant) {
  if (steps < 2) throw ValueError("autotune needs at least 2 steps");
  const int candidates[kBatchCandidates] = {
      kFusedTz8, kFusedTz16, kTwoStepTz8, kTwoStepTz16, kLeanTz16,
      kLeanTz8,  kLeanTz12,  kLeanTz20,   kLeanTz24,    kLeanTz32,
      kLeanTz4,  kLeanTz8W6, kLeanTz12W5, kLeanTz8Sep, kLeanTz4Sep, kLeanTz8Ring,
      kLeanTz16Ring, kLeanTz8RingClamp, kLeanTz16RingClamp};
  const int keep_remap = xcd_remap_;
  double best_ms = std::numeric_limits<double>::infinity();
  int best_v = variant_;
  bool lean = true;
  for (auto &m : models_) lean = lean && m->lean_ok();
  for (int k = 0; k < kBatchCandidates; ++k) {
    if (ms_per_variant) ms_per_variant[k] = -1.0;
    if (step_is_lean(candidates[k]) && !lean) continue;
    set_variant(candidates[k], keep_remap);
    // the loop forward_all runs with this variant: the shots in lockstep
    // where it can, else shot 0 alone; timed per step of one shot
    const bool lock = lockstep_available();
    const int n = std::min(steps, nt_);
    auto run = [&]() {
      if (lock)
        enqueue_lockstep_loop(n);
      else
        enqueue_loop(0, n);
    };
    run();  // warm up
    hip_check(hipEventRecord(ev_[0], stream_), "hipEventRecord");
    run();
    hip_check(hipEventRecord(ev_[1], stream_), "hipEventRecord");
    hip_check(hipStreamSynchronize(stream_), "hipStreamSynchronize");
    float ms = 0.f;
    hip_check(hipEventElapsedTime(&ms, ev_[0], ev_[1]), "hipEventElapsedTime");
    double per = ms / (n * (lock ? n_shots_ : 1));
    if (ms_per_variant) ms_per_variant[k] = per;
    if (per < best_ms) {
      best_ms = per;
      best_v = candidates[k];
    }
  }
  set_variant(best_v, keep_remap);
  if (best) *best = best_v;
  // resident loops where they are faster still; not where a launch is refused,
  // since whoever holds the device is likely still there
  resident_ = true;
  const int n = std::min(steps, nt_);
  LoopLaunches *const p = resident_available() ? loop_launches(4, 0, n) : nullptr;
  bool faster = p && run_loops(*p, n, false);  // warm up
  if (faster) {
    hip_check(hipEventRecord(ev_[0], stream_), "hipEventRecord");
    faster = run_loops(*p, n, false);
    hip_check(hipEventRecord(ev_[1], stream_), "hipEventRecord");
    hip_check(hipStreamSynchronize(stream_), "hipStreamSynchronize");
    float ms = 0.f;
    hip_check(hipEventElapsedTime(&ms, ev_[0], ev_[1]), "hipEventElapsedTime");
    faster = faster && ms / (n * n_shots_) < best_ms;
  }
  resident_ = faster;
  return best_ms;
}

}  // namespace psv
