#include "MixedRange.h"

#include <algorithm>
#include <chrono>

namespace {
double now_ms() {
  return std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now().time_since_epoch()).count();
}
// The largest rectangles' index first: the others run beside its long kernels.
constexpr int kQueueOrder[3] = {2, 1, 0};
}  // namespace

MixedRange::~MixedRange() {
  if (graph_) gat_graph_destroy(graph_);
  if (fork_) gat_event_destroy(fork_);
  for (void* e : join_)
    if (e) gat_event_destroy(e);
}

RangeEngine& MixedRange::engine(int i) { return i == 0 ? fsg_.engine() : i == 1 ? grid_.engine() : stig_.engine(); }

const DeviceTree& MixedRange::tree(int i) {
  return i == 0 ? fsg_.deviceTree() : i == 1 ? grid_.deviceTree() : stig_.deviceTree();
}

// One graph, three branches: the coordinating stream records `fork_`, each
// index's stream waits for it, queues its pipeline and records its join
// event, and the coordinating stream waits for all three.
int MixedRange::capture(const int nq[3]) {
  if (graph_) gat_graph_destroy(graph_);
  graph_ = nullptr;
  for (int i = 0; i < 3; ++i)
    if (nq[i] > 0)
      if (int rc = engine(i).reserveResults(nq[i], batch_[i])) return rc;
  void* c = coord_.get();
  GATH_TRY(gat_graph_begin(c), "mixed capture");
  int rc = gat_event_record(fork_, c);
  for (int i : kQueueOrder) {
    if (rc != GAT_OK || nq[i] == 0) continue;
    void* s = engine(i).stream();
    rc = gat_stream_wait_event(s, fork_);
    if (rc == GAT_OK) rc = engine(i).enqueueBatch(tree(i), nq[i], batch_[i]);
    if (rc == GAT_OK) rc = engine(i).enqueueResults(nq[i], batch_[i]);
    if (rc == GAT_OK) rc = gat_event_record(join_[i], s);
    if (rc == GAT_OK) rc = gat_stream_wait_event(c, join_[i]);
  }
  void* g = nullptr;
  const int rc_end = gat_graph_end(c, &g);
  if (rc != GAT_OK) return gath_fail_hip(rc, "mixed capture");
  GATH_TRY(rc_end, "mixed capture");
  graph_ = g;
  std::copy(nq, nq + 3, shape_);
  for (int i = 0; i < 3; ++i) {
    keys_[i] = engine(i).layoutKey(tree(i), nq[i], batch_[i]);
    results_[i][0] = batch_[i].digestDev_.get();
    results_[i][1] = engine(i).resultsHost();
  }
  ++captures;
  return GAT_OK;
}

bool MixedRange::keysMatch(const int nq[3]) {
  for (int i = 0; i < 3; ++i)
    if (nq[i] > 0 && (engine(i).layoutKey(tree(i), nq[i], batch_[i]) != keys_[i] ||
                      batch_[i].digestDev_.get() != results_[i][0] || engine(i).resultsHost() != results_[i][1]))
      return false;
  return true;
}

int MixedRange::run(const MBB* bounds, int n, const MixedConfig& cfg, MixedResult* out) {
  if (!out || n < 0 || (n > 0 && !bounds) || cfg.groupSize < 1) {
    gath_set_error("MixedRange::run: bad arguments");
    return GAT_ERR_ARG;
  }
  for (int i = 0; i < 3; ++i)
    if (tree(i).nnodes == 0) {
      gath_set_error("MixedRange::run: index %d has no device tree (build it with upload)", i);
      return GAT_ERR_STATE;
    }
  const double t0 = now_ms();
  if (int rc = coord_.create()) return rc;
  if (!fork_) GATH_TRY(gat_event_create(&fork_), "mixed events");
  for (void*& e : join_)
    if (!e) GATH_TRY(gat_event_create(&e), "mixed events");
  *out = MixedResult{};
  out->count.assign(size_t(n), 0);
  out->digest.assign(size_t(n), 0);
  out->route.assign(size_t(n), 0);
  std::vector<int> list[3];
  for (int q = 0; q < n; ++q) {
    const double area = std::max(0.0, double(bounds[q].xmax) - bounds[q].xmin) *
                        std::max(0.0, double(bounds[q].ymax) - bounds[q].ymin);
    const int r = area < cfg.fsgMaxArea ? 0 : area < cfg.gridMaxArea ? 1 : 2;
    out->route[q] = int8_t(r);
    list[r].push_back(q);
  }
  // The captured pipelines are the leaf-major form: keep small groups off the
  // direct form while this runs.
  int saved[3];
  for (int i = 0; i < 3; ++i) {
    saved[i] = engine(i).directMaxQueries;
    engine(i).directMaxQueries = 0;
  }
  auto restore = [&] {
    for (int i = 0; i < 3; ++i) engine(i).directMaxQueries = saved[i];
  };
  size_t groups = 0;
  for (auto& l : list) groups = std::max(groups, (l.size() + size_t(cfg.groupSize) - 1) / size_t(cfg.groupSize));
  std::vector<MBB> boxes[3];
  std::vector<uint64_t> dig;
  for (size_t gi = 0; gi < groups; ++gi) {
    int nq[3];
    for (int i = 0; i < 3; ++i) {
      const size_t b = gi * size_t(cfg.groupSize);
      nq[i] = b >= list[i].size() ? 0 : int(std::min(list[i].size() - b, size_t(cfg.groupSize)));
      boxes[i].clear();
      for (int k = 0; k < nq[i]; ++k) boxes[i].push_back(bounds[list[i][b + size_t(k)]]);
    }
    const uint64_t* digests[3] = {nullptr, nullptr, nullptr};
    std::vector<std::pair<uint64_t, uint64_t>> digestSpans;  // device clock
    // Which indexes' answers are in: both quick ways below leave counts and
    // digests in pinned memory.
    bool done[3] = {nq[0] == 0, nq[1] == 0, nq[2] == 0};
    auto waitAll = [&](int rc) -> int {
      for (int i = 0; i < 3; ++i)
        if (nq[i] > 0) {
          const int r = gat_stream_sync(engine(i).stream());
          if (rc == GAT_OK) rc = r;
        }
      return rc;
    };
    // Once the work has been waited for: the answers of the indexes that ran.
    auto collect = [&](bool replay, const bool ran[3]) -> int {
      int rc = GAT_OK;
      for (int i = 0; i < 3 && rc == GAT_OK; ++i) {
        if (nq[i] == 0 || !ran[i]) continue;
        uint64_t clock[2] = {0, 0};
        rc = engine(i).finishResults(nq[i], batch_[i], replay, &done[i], &digests[i], clock);
        if (done[i]) digestSpans.emplace_back(clock[0], clock[1]);
        else ++pipelines.discarded;
      }
      return rc;
    };
    // Step by step: sizes the workspace, which may move its buffers, so the
    // captured graph is dropped first.
    bool stepped = false;
    auto step = [&](int i) -> int {
      if (graph_) gat_graph_destroy(graph_);
      graph_ = nullptr;
      std::fill(shape_, shape_ + 3, -1);
      stepped = true;
      ++pipelines.stepped;
      return i == 0   ? fsg_.rangeQueryBatchedGPU(boxes[i].data(), nq[i], batch_[i], false)
             : i == 1 ? grid_.rangeQueryBatchedGPU(boxes[i].data(), nq[i], batch_[i], false)
                      : stig_.rangeQueryBatchedGPU(boxes[i].data(), nq[i], batch_[i], false);
    };
    bool byStep[3] = {false, false, false};
    const bool captured = cfg.graph && graph_ && std::equal(nq, nq + 3, shape_);
    if (captured) {
      // Replay: stage every index's rectangles, launch the one graph behind
      // them, check capacities.
      int rc = GAT_OK;
      for (int i = 0; i < 3 && rc == GAT_OK; ++i)
        if (nq[i] > 0) {
          rc = engine(i).stageBatch(tree(i), boxes[i].data(), nq[i]);
          if (rc == GAT_OK) rc = gat_event_record(join_[i], engine(i).stream());
          if (rc == GAT_OK) rc = gat_stream_wait_event(coord_.get(), join_[i]);
        }
      // A workspace that moved since the capture: the graph's kernels would
      // read freed memory, so this group runs step by step and is recaptured.
      const bool current = rc == GAT_OK && keysMatch(nq);
      if (current) rc = gat_graph_launch(graph_, coord_.get());
      if (const int r = coord_.sync(); rc == GAT_OK) rc = r;
      const bool all[3] = {true, true, true};
      if (rc == GAT_OK && current) rc = collect(true, all);
      if (rc != GAT_OK) {
        restore();
        return gath_fail_hip(rc, "mixed replay");
      }
      if (current && done[0] && done[1] && done[2]) ++out->replays;
    } else if (graph_ || !cfg.graph || gi + 2 >= groups) {
      // A group of another shape than the captured one, or one not to be captured:
      // the pipelines of the indexes whose workspaces earlier batches have
      // sized are queued on their own streams with one wait (step by step they
      // took a wait per pipeline half and several per index's results, and ran
      // one index after another).  An index whose workspace is too small runs
      // step by step beside them, so nothing queued is thrown away for it.
      int rc = GAT_OK;
      bool queued[3] = {false, false, false};
      for (int i : kQueueOrder) {
        if (rc != GAT_OK || nq[i] == 0) continue;
        rc = engine(i).queueBatch(tree(i), boxes[i].data(), nq[i], batch_[i], &queued[i]);
        if (queued[i]) ++pipelines.queued;
      }
      for (int i = 0; i < 3 && rc == GAT_OK; ++i)
        if (nq[i] > 0 && !queued[i]) {
          if (const int r = step(i)) {  // it has said what failed
            waitAll(r);
            restore();
            return r;
          }
          byStep[i] = true;
        }
      rc = waitAll(rc);
      if (rc == GAT_OK) rc = collect(false, queued);
      if (rc != GAT_OK) {
        restore();
        return gath_fail_hip(rc, "mixed batch");
      }
    }
    // What the quick ways did not take, or what outgrew its workspace there.
    int rc_step = GAT_OK;
    for (int i = 0; i < 3 && rc_step == GAT_OK; ++i)
      if (!done[i] && !byStep[i]) rc_step = step(i);
    // A group that sized its workspaces and is not among the last two is captured.
    if (rc_step == GAT_OK && stepped && cfg.graph && gi + 2 < groups) rc_step = capture(nq);
    if (rc_step != GAT_OK) {
      restore();
      return rc_step;
    }
    const double d0 = now_ms();
    for (int i = 0; i < 3; ++i) {
      if (nq[i] == 0) continue;
      RangeBatch& b = batch_[i];
      int rc = b.syncHost();
      const uint64_t* d = digests[i];
      if (rc == GAT_OK && !done[i]) {
        dig.resize(size_t(nq[i]));
        rc = b.digests(dig.data());
        d = dig.data();
      }
      if (rc != GAT_OK) {
        restore();
        return rc;
      }
      const size_t base = gi * size_t(cfg.groupSize);
      for (int k = 0; k < nq[i]; ++k) {
        const int q = list[i][base + size_t(k)];
        out->count[size_t(q)] = b.count[size_t(k)];
        out->digest[size_t(q)] = d[k];
      }
      out->pairs += b.pairTotal;
      out->candidates += b.candidates;
    }
    out->digestMs += now_ms() - d0;
    if (!digestSpans.empty()) {
      // The time in which the quick ways' digests ran, beside each other or not.
      if (clockKhz_ == 0) {
        const int rc = gat_wall_clock_khz(&clockKhz_);
        if (rc != GAT_OK) {
          restore();
          return gath_fail_hip(rc, "device clock");
        }
      }
      std::sort(digestSpans.begin(), digestSpans.end());
      uint64_t covered = 0, ticks = 0;
      for (const auto& d : digestSpans) {
        const uint64_t from = std::max(d.first, covered);
        if (d.second > from) ticks += d.second - from;
        covered = std::max(covered, d.second);
      }
      out->digestMs += double(ticks) / clockKhz_;
    }
    ++out->groups;
  }
  restore();
  out->ms = now_ms() - t0;
  return GAT_OK;
}
