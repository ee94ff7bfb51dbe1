// The host-side rules that choose a kernel (plan.hpp has no HIP types in it) behind plain C functions,
// for tests/test_plan_rules.py, which compiles this file with g++ and loads it.
#include "../../torch-xpu-ops_amd/csrc/kernels/plan.hpp"
#include "../../torch-xpu-ops_amd/csrc/kernels/team_slots.hpp"

using namespace rownorm;

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

// one table of slots for streams, as the library keeps one per device
int rule_team_slots() { return kTeamSlots; }
void* rule_slots_new() { return new StreamSlots<kTeamSlots>(); }
void rule_slots_delete(void* t) { delete (StreamSlots<kTeamSlots>*)t; }
int rule_slot_of(void* t, uintptr_t key) { return ((StreamSlots<kTeamSlots>*)t)->of(key); }

}  // extern "C"
