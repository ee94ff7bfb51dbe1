// The host-side rules that choose a kernel (plan.hpp has no HIP types in it) behind plain C functions,
// for tests/test_plan_rules.py, which compiles this file with g++ and loads it.
#include "../../torch-xpu-ops_amd/csrc/kernels/plan.hpp"
#include "../../torch-xpu-ops_amd/csrc/kernels/team_slots.hpp"

#include <set>
#include <thread>
#include <vector>

using namespace rownorm;

// Streams and an event as the team launches' order sees them: the launches known to be over when a stream's next work
// starts.
struct FakeStreams {
  using Stream = int;
  std::vector<std::set<int>> over;
  std::vector<char> captured;
  std::set<int> event;
  int records = 0, waits = 0, recorded_into_capture = 0;
  bool capturing(Stream s) { return captured[s]; }
  void record(Stream s) { ++records, recorded_into_capture += captured[s], event = over[s]; }
  void wait(Stream s) { ++waits, over[s].insert(event.begin(), event.end()); }
};

extern "C" {

int rule_norm_bwd_reads_elements(int esize, int wsize, int G, int V, int rms, int64_t M, int64_t N) {
  return norm_bwd_reads_elements(esize, wsize, G, V, rms != 0, M, N) ? 1 : 0;
}

// out: workgroups a team, workgroups a channel, packs a lane, whether the next slab is on its way,
// workgroups launched
void rule_gn_bwd_team(int64_t rows, int64_t D, int64_t cp, int esize, int64_t out[5]) {
  const GnBwdTeam t = gn_bwd_team(rows, D, cp, esize, 256);
  out[0] = t.team, out[1] = t.wpc, out[2] = t.v, out[3] = t.ahead, out[4] = t.grid;
}

int rule_gn_team_sums(int64_t rows, int64_t groups, int64_t teams) { return gn_team_sums_columns(rows, groups, teams); }

// out: workgroups a team, packs a lane, lanes along inner, workgroups launched; then whether the tile
// kernel holds D, its lanes along inner and along D, rows a lane and workgroups, chunks
void rule_strided_plan(int backward, int64_t outer, int64_t D, int64_t inner, int esize, int64_t out[10]) {
  StridedPlan p;
  make_strided_plan(backward != 0, outer, D, inner, esize, 256, Override{}, &p);
  out[0] = p.team, out[1] = p.team_v, out[2] = 1 << p.team_tx_log2, out[3] = p.team_grid;
  out[4] = p.resident, out[5] = 1 << p.tx_log2, out[6] = 1 << p.ty_log2, out[7] = p.V, out[8] = p.grid;
  out[9] = p.chunks;
}

// the same call's teams of workgroups that have a compute unit each: workgroups a team, packs a lane, lanes
// along inner, workgroups launched
void rule_strided_large(int backward, int64_t outer, int64_t D, int64_t inner, int esize, int64_t out[4], int widened) {
  StridedPlan p;
  make_strided_plan(backward != 0, outer, D, inner, esize, 256, Override{}, &p, widened != 0);
  out[0] = p.large_team, out[1] = p.large_v, out[2] = 1 << p.large_tx_log2, out[3] = p.large_grid;
}

// the whole-wavefront layout of a norm call: wavefronts a row, packs a lane, rows in registers, threads the
// instance is built for, rows a workgroup works on, workgroups; then the rows of the resident plan's partial sums
void rule_norm_waves(int backward, int64_t M, int64_t N, int esize, int layer_norm, int wide, int want_dx, int64_t out[7]) {
  Plan p;
  make_plan(backward ? OC_NORM_BWD : OC_NORM_FWD, M, N, esize, 256, Override{}, backward != 0, &p, false, layer_norm != 0,
            wide != 0, false, false, false, want_dx != 0);
  const WavesLayout& l = p.waves;
  out[0] = l.waves, out[1] = l.v, out[2] = l.depth, out[3] = l.threads, out[4] = l.slots, out[5] = l.grid;
  out[6] = p.partial_rows;
}

// the team of a long norm forward row on a machine of 256 compute units: workgroups, packs a lane, teams
void rule_norm_team(int64_t M, int64_t N, int esize, int wide, int64_t out[3]) {
  Plan p;
  make_plan(OC_NORM_FWD, M, N, esize, 256, Override{}, false, &p, false, true, wide != 0);
  out[0] = p.team, out[1] = p.team_r ? 0 : p.team_v, out[2] = p.team ? p.team_grid / p.team : 0;
}

// n team launches in turn, number i on stream[i] (per_thread[i]: by a per-thread handle) while the streams of the bits
// captured[i] are under capture.  ran[i]: 0 went without teams, 1 ran behind every team launch before it, 2 did not.
// counts: events recorded, waits, events recorded on a stream under capture.
void rule_team_order(int n, const int* stream, const int* captured, const int* per_thread, int streams, int* ran,
                     int counts[3]) {
  FakeStreams f;
  f.over.resize(streams);
  TeamOrder<FakeStreams> order;
  std::set<int> before;
  for (int i = 0; i < n; ++i) {
    const int s = stream[i];
    f.captured.assign(streams, 0);
    for (int k = 0; k < streams; ++k) f.captured[k] = captured[i] >> k & 1;
    ran[i] = 0;
    if (!order.enter(f, (uintptr_t)s + 1, s, per_thread[i] != 0)) continue;
    ran[i] = f.over[s] == before ? 1 : 2;
    f.over[s].insert(i);
    before.insert(i);
    order.leave(f);
  }
  counts[0] = f.records, counts[1] = f.waits, counts[2] = f.recorded_into_capture;
}

// `threads` threads with a stream each, n launches a thread: the launches that were not behind all others before them
int rule_team_order_threads(int threads, int n) {
  FakeStreams f;
  f.over.resize(threads);
  f.captured.assign(threads, 0);
  TeamOrder<FakeStreams> order;
  std::set<int> before;
  int unordered = 0;
  std::vector<std::thread> ts;
  for (int t = 0; t < threads; ++t)
    ts.emplace_back([&, t] {
      for (int i = 0; i < n; ++i) {
        if (!order.enter(f, (uintptr_t)t + 1, t, false)) continue;
        unordered += f.over[t] != before;  // (between enter and leave: one thread at a time)
        f.over[t].insert(t * n + i);
        before.insert(t * n + i);
        order.leave(f);
      }
    });
  for (auto& t : ts) t.join();
  return unordered + (int)(before.size() != (size_t)threads * n);
}

// What serves a softmax call (widened: float32 output of 16-bit rows): 1 rows in registers, 2 a team, 3 ragged rows held by
// one workgroup, 0 the two passes; out: workgroups of the team, or lanes and packs a lane of the held form
int rule_softmax_route(int backward, int is_log, int64_t M, int64_t N, int esize, int widened, int64_t out[2]) {
  Plan p;
  make_plan(backward ? OC_SOFTMAX_BWD : OC_SOFTMAX_FWD, M, N, esize, 256, Override{}, false, &p);
  out[0] = out[1] = 0;
  if (softmax_team_serves(p, backward != 0, is_log != 0, widened != 0, esize, M, N, 256)) {
    out[0] = p.team;
    return 2;
  }
  if (p.resident) return 1;
  if (!softmax_tail_serves(p, backward != 0, is_log != 0, widened != 0, esize, M, N)) return 0;
  out[0] = p.tail_g, out[1] = p.tail_v;
  return 3;
}

// the backward of long norm rows: wavefronts that share a piece of columns (0: not the two launches without partial
// rows), workgroups of the team that holds four rows at a time (0: none)
void rule_norm_few_rows(int64_t M, int64_t N, int esize, int layer_norm, int wide, int64_t out[2]) {
  Plan p;
  make_plan(OC_NORM_BWD, M, N, esize, 256, Override{}, true, &p, false, layer_norm != 0, wide != 0);
  out[0] = p.few_waves, out[1] = p.team;
}

// one table of slots for streams, as the library keeps one per device
int rule_team_slots() { return kTeamSlots; }
void* rule_slots_new() { return new StreamSlots<kTeamSlots>(); }
void rule_slots_delete(void* t) { delete (StreamSlots<kTeamSlots>*)t; }
int rule_slot_of(void* t, uintptr_t key) { return ((StreamSlots<kTeamSlots>*)t)->of(key); }

// n calls, number at[i] in slot[i]: id[i], clear[i]
void rule_team_ids(int n, const uint64_t* at, const int* slot, unsigned int* id, int* clear) {
  TeamIds<kTeamSlots> ids;
  for (int i = 0; i < n; ++i) {
    bool c = false;
    id[i] = ids.of(at[i], slot[i], &c);
    clear[i] = c;
  }
}
unsigned int rule_team_call_ids() { return kTeamCallIds; }

}  // extern "C"
