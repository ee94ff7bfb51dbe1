// Host-side choice of the launch layout for one call (no HIP types in here).
//
// Stands in for the reference's work-split heuristics: NormConfig
// (src/ATen/native/xpu/sycl/Norm.h:225-370), layer_norm_wg_size_select
// (LayerNormKernels.cpp:588-616) and get_wgroup_size (SoftMaxKernels.cpp:
// 139-182).  Those are written around Intel EU counts and SIMD32 sub-groups;
// here the split is a small table over the row size for 256 compute units of
// 64-wide wavefronts.
//
// The rule.  A row of N elements is ceil(N / E) 16-byte packs (E = 4 for fp32,
// 8 for 16-bit types).  G lanes share a row and each holds V packs:
//   G = smallest power of two in [8, 1024] with G * V_pref >= packs,
//   V = smallest power of two with G * V >= packs.
// If V exceeds the per-op register budget V_max the multi-pass streaming
// kernel is used instead.  Rows whose length is a whole number of packs take
// the branch-free "fast" kernels; ragged rows (N % E != 0) take the general
// ones, which exist for V = V_pref only (and three packs for 16-bit softmax and
// the 16-bit norms).  Measured exceptions for rows that
// leave many of those lanes idle (hidden sizes that are not powers of two) or
// that would take 1024 lanes: norm_layout() and the softmax / GroupNorm rules
// in make_plan() pick three or five packs a lane, or fewer lanes.  Workgroup
// size and grid size per op class are set by block_threads() and default_bpc()
// below.
#pragma once
#include <stdint.h>

namespace rownorm {

enum OpClass {
  OC_NORM_FWD = 0,
  OC_NORM_BWD = 1,
  OC_SOFTMAX_FWD = 2,
  OC_SOFTMAX_BWD = 3,
  OC_GROUP_FWD = 4,  // GroupNorm: rows are (sample, group) slabs, no per-column registers
  OC_GROUP_BWD = 5
};

struct Override {
  // 0 = automatic; G = -1 = force the streaming kernel, and then V = 1 keeps every
  // row on one workgroup, V > 1 splits every row over V workgroups (norm ops), V = 0 with
  // block = 1 sends a norm backward of whole packs to teams of workgroups however few
  // rounds they make
  int G = 0, V = 0, block = 0, bpc = 0;
};

// Rows on whole wavefronts, as many as they need (norm_waves_kernels.hpp): wavefronts a row, packs a
// lane, rows a lane has in its registers, threads the instance is built for, rows a workgroup works on
// at a time, workgroups.  waves 0: not this call.
struct WavesLayout {
  int waves = 0, v = 0, depth = 0, threads = 0, slots = 0, grid = 0;
};

struct Plan {
  bool resident = true;
  bool fast = true;  // N % E == 0: branch-free row access
  int G = 0, V = 0, block = 0, rpb = 0;
  int64_t grid = 0;
  int64_t partial_rows = 0;
  // Split-row path of the norm ops (few rows, each far too long for registers):
  // a row is cut into `split` chunks of `chunk_packs` packs, one workgroup each;
  // 0 or 1 = one workgroup per row.
  int split = 0;
  int64_t chunk_packs = 0;
  // norm backward of few rows beyond the registers (norm_bwd_few_rows_kernel): wavefronts that share a piece of
  // columns; 0: not planned; and the chunks its rows are cut into for their sums.  With a team (`team`) beside it:
  // where the call cannot have that
  int few_waves = 0, few_chunks = 0;
  int64_t few_chunk_packs = 0;
  // softmax backward of rows beyond the registers of two tensors: grad alone fits
  // them (the log_softmax backward then keeps grad resident and streams y)
  bool grad_resident = false;
  // softmax rows of no whole number of packs that one workgroup of tail_g lanes (1024, forward also 512) can hold in
  // tail_v whole packs a lane, tail_packs at most in all (0: not such a row); softmax_tail_serves() says whether it does
  int tail_v = 0, tail_g = 0, tail_packs = 0, tail_cus = 0;
  // a layout was asked for by override: kernels chosen by other means than the
  // layout (softmax of short ragged rows through LDS) stand back
  bool forced = false;
  // norm forward of rows beyond one workgroup's registers held by a team of
  // workgroups (norm_fwd_team_kernel): workgroups a row, packs a lane the kernel is
  // compiled for, packs a workgroup, workgroups launched; team == 0: not planned
  // (softmax: the team that could hold a row, whether it does is softmax_team_serves()'s)
  int team = 0, team_v = 0;
  int64_t team_chunk_packs = 0, team_grid = 0;
  // norm backward of such rows held R = team_v rows at a time by teams of workgroups
  // (norm_bwd_team_kernel): the same fields, one stride of packs a workgroup, and the
  // partial rows of column sums that launch leaves (one a team; partial_rows is what
  // the kernels behind it would use)
  int64_t team_partial_rows = 0;
  // norm forward of such rows with three rows in flight a workgroup, team_v packs of a row
  // a lane and the weights held (norm_fwd_rows_team_kernel): 1; 0: norm_fwd_team_kernel
  int team_r = 0;
  // norm backward / forward on an exact layout (norm_bwd_exact_kernel,
  // norm_fwd_exact_kernel): row blocks a lane keeps in flight, itself included (the
  // forward: 1); GroupNorm on an exact layout (gn_*_exact_kernel): 1; 0 = the
  // general resident kernel
  int exact_depth = 0;
  // what serves the call instead of the resident layout where the row is written in its own type
  // (norm backward: no residual gradient)
  WavesLayout waves;
  // ragged 16-bit norm rows addressed through the 16-byte aligned window that holds
  // each row (norm_row_window()): G * V holds the packs of that window, and a
  // workgroup that walks several row blocks strides by a multiple of 8 rows
  bool window = false;
};

// norm_fwd_team_kernel: threads a workgroup, packs a lane at most, workgroups of
// the grid at most.
constexpr int kTeamBlock = 512;
constexpr int kTeamPerCu = 2;  // workgroups of a team launch a compute unit holds
constexpr int kTeamMaxV = 16;
constexpr int kTeamGroup = 2;  // packs whose weights are requested together
constexpr int kTeamMaxWorkgroups = 512;
// streams with a slot of exchange memory of their own (team_slots.hpp): more than the default
// stream and the 32 of a framework's pool; for the strided softmax, whose slots are 4 MiB, eight
constexpr int kTeamSlots = 64;
constexpr int kTeamColumnSlots = 8;
constexpr int kTeamMinTeams = 8;
// gn_bwd_team_ahead_kernel: packs a lane holds of each tensor and slab (two slabs at a time).
constexpr int kGnTeamAheadPacks = 4;
// norm_bwd_team_kernel: rows a team holds at a time, packs of a row a lane holds of each
// tensor, workgroups a compute unit
constexpr int kTeamBwdRows = 4;
constexpr int kTeamBwdPacks = 2;
constexpr int kTeamBwdPerCu = 1;
// norm_fwd_rows_team_kernel: packs of a row a lane, and the rounds from which it is taken
constexpr int kTeamFwdLongPacks = 10;
constexpr int kTeamFwdMinRounds = 16;
// Ids that team calls draw in turn, from 1 on; as many as the tag of a word has room for (device/team.hpp).
constexpr unsigned int kTeamCallIds = 0x1ffffff;
// One stream's exchange memory (device/team.hpp, team_slots.hpp).
struct TeamEntry {
  // the two-number exchange: (call id << 32) | (round + 1) once s1, s2 are in place, 0 while
  // they change; a workgroup's partial sums (float64 bit patterns)
  unsigned long long tag;
  unsigned long long s1, s2;
  // the exchanges of self-validating words {32 bits of payload, tag}: see device/team.hpp
  // (128 bytes an entry: neighbours' polls go to other memory channels)
  unsigned long long pad[13];
};
struct TeamSlot {
  // [round parity][workgroup]; norm_bwd_team_kernel, which publishes a round before it
  // gathers the one before, goes round all four
  TeamEntry entry[4][kTeamMaxWorkgroups];
  unsigned int gave_up;                    // id of a call one of whose waits ran out (a hint)
  unsigned int pad[3];
};

// Columns (elements of `inner`) a strip of the strided team kernels has at most, and one stream's
// exchange memory there: [round parity][workgroup][number][column] words (softmax_strided_team.hpp).
constexpr int kTeamColumns = 256;
struct TeamColumns {
  unsigned long long word[2][kTeamMaxWorkgroups][2 * kTeamColumns];
  unsigned int gave_up;  // as in TeamSlot
  unsigned int pad[3];
};

// softmax_fwd_team_kernel / softmax_bwd_team_kernel: rows of at least this many packs (64 KiB),
// and the packs a lane the backward holds of each of its two tensors at most.
constexpr int64_t kSoftmaxTeamMinPacks = 4096;
constexpr int kSoftmaxBwdTeamMaxV = 8;

constexpr int kMinG = 8;
constexpr int kMaxG = 1024;
constexpr int kMaxV = 16;
// The 16-bit softmax forward alone goes to 20 packs a lane (163840-element rows:
// the 151936 / 152064-entry vocabularies).
constexpr int kSoftmaxFwdMaxV16 = 20;
// Packs of each of its two tensors a lane of the one-workgroup softmax backward holds at most.
constexpr int kSoftmaxBwdHoldMaxV = 8;
// Packs of grad a lane of the grad-resident log_softmax backward holds at most.
constexpr int kGradResidentMaxV = 20;
// Softmax rows of no whole number of packs beyond the resident layouts: 3 packs a lane at least, on one workgroup of
// 1024 lanes (TAIL in softmax_kernels.hpp).  Against the multi-pass kernels, which read X, or grad and y, twice, bf16
// us: [4096, 128255] log_softmax 453 -> 396, backward 621 -> 587; [4096, 50257] 161 -> 148, 238 -> 225; [515, 50220]
// softmax 26.7 -> 25.4, 40.3 -> 34.5; [2000, 17001] 32.2 -> 26.8, 46.0 -> 37.7.  (The same on packs at the row's own
// alignment: a 16-byte access two bytes off costs twice, [4096, 128255] 479 and 677.)
constexpr int kSoftmaxTailMinV = 3;
// The forward on 512 lanes where more and smaller workgroups a compute unit overlap better: the shortest of these rows
// and calls of few rows (bf16 softmax, 1024 / 512 lanes: [4096, 17001] 54.1 / 50.0 us, [2000, 24570] 39.0 / 37.0, [1000,
// 20005] 18.5 / 14.5, [512, 41003] 16.2 / 15.0, but [4096, 28003] 80.4 / 84.9, [2000, 41003] 61.9 / 62.9).  Rows of the
// resident layouts end at 16384 elements, so a lane holds 5 packs at least (float32: 9).
constexpr int kSoftmaxTailHalfMaxV = 14;
constexpr int softmax_tail_half_min_v(int esize) { return esize == 2 ? 5 : 9; }
constexpr bool softmax_tail_half_lanes(int64_t packs, int64_t M, int num_cus) {
  return packs <= 2560 || (packs <= 4096 && M <= 8 * (int64_t)num_cus) ||
         (packs <= kMaxG / 2 * kSoftmaxTailHalfMaxV && M <= 2 * (int64_t)num_cus);
}
// The log_softmax backward holds grad alone from here on (both tensors: [2000, 49001] 112 us, grad alone 106, the
// multi-pass kernel 106; [1000, 65001] 81.4, 72.7, 74.8; float32 of 5 to 8 packs 0.97 to 1.05 of grad alone's time).
constexpr int kSoftmaxTailGradMinV = 4;
// Bytes of input up to which the two passes gain from the 256 MB cache behind the L2s (a crossover as measured: most
// of a little more than the cache's size still comes out of it).
constexpr int64_t kSoftmaxCachedBytes = (int64_t)288 << 20;
constexpr int max_v_of(OpClass oc, int esize) {
  return oc == OC_SOFTMAX_FWD && esize == 2 ? kSoftmaxFwdMaxV16 : kMaxV;
}
constexpr int kStreamBlock = 1024;
// Split-row path: a chunk is a whole number of workgroup strides and at least
// four of them (32768 16-bit elements); a row is cut into at most 1024 chunks.
constexpr int kSplitMinStrides = 4;
constexpr int kSplitMaxChunks = 1024;
// norm_bwd_few_rows_kernel: rows at most, bytes of a tensor at most, wavefronts a workgroup
constexpr int kFewRowsMax = 128;
constexpr int64_t kFewRowsBytes = int64_t(32) << 20;
constexpr int kFewRowsWaves = 8;

// Preferred packs per lane: what the G ladder aims for.
// Measured on MI355X: 16 elements a lane (two 16-bit packs, four fp32 packs)
// keeps the register count low enough for 8 wavefronts per SIMD, which beats
// fewer, fatter lanes on every op of the family.
constexpr int v_pref(OpClass, int esize) { return esize == 4 ? 4 : 2; }

// Ragged 16-bit rows of the norm forward (every row at another 2-byte alignment,
// where a 128-bit access costs about twice an aligned one) on 256 lanes or more are
// addressed through the 16-byte aligned window that holds the row: it starts up to
// 7 elements before the row and can hold one pack more than the row.  Every whole
// pack of the window is an aligned access, the two end packs are trimmed (loads)
// or written element by element (stores), and gamma / beta are held shifted by the
// window's head: loaded once per workgroup when all its rows have the same head,
// i.e. when it strides by a multiple of 8 rows, which make_plan() sees to (and
// again per row otherwise).  fp16, 8192 rows that start 2 elements into their
// buffers: N = 4097 LayerNorm 43.6 -> 34.6 us, RMSNorm 31.2 -> 29.9 us; 8193: 68.8 ->
// 61.0 and 58.9 -> 51.1 us.  Shorter rows lose (the two end packs weigh more: N =
// 2049 LayerNorm 20.0 -> 20.9 us, RMSNorm 15.3 -> 17.3 us) and keep the row-start
// addressing; so does the backward, which measured no gain (N = 4097 LayerNorm 68.6
// -> 68.1 us) or a loss (RMSNorm 53.8 -> 71.6 us: 132 registers against 127, one
// workgroup a compute unit instead of two).
constexpr bool norm_row_window(int esize, int G, bool fast) {
  return !fast && esize == 2 && G >= 256;
}

// The resident norm forward keeps gamma / beta of a lane's columns in registers
// across its rows while they fit; at 1024 lanes, rows of more packs a lane than
// the table below leave the weights in memory, load each pack of them (from L2)
// where the output needs it, and hold only the row.  esize / wsize: bytes of a
// row / weight element.  Measured, bf16 rows, against the multi-pass kernel that
// served rows beyond 4 packs a lane before (2048 rows): N = 40960 LayerNorm 84 ->
// 65 us (fp32 weights 90 -> 72), RMSNorm 66 -> 59; 65536: 109 -> 101 and 104 ->
// 95; 1024 rows of 131072: 114 -> 105 and 114 -> 98.  Held against looked up, where
// both fit the registers (8192 rows of 40960 / 4096 of 49152 / 8192 of 65536):
// LayerNorm bf16 weights 226 / 143 us against 244 / 153; RMSNorm bf16 weights 240 /
// 147 / 373 against 227 / 144 / 384 (5 and 6 packs held leave one workgroup a
// compute unit where the lookup keeps two); RMSNorm fp32 weights 222 / 136 / 400
// against 236 / 145 / 395.  Up to 4 packs the held weights win by 5-20 %.  The fp32
// LayerNorm with its weights held spilled from 5 packs a lane (N = 20480..32768:
// 209..229 -> 62..104 us); the fp32 RMSNorm holds 8 packs and is 3 % faster so.
constexpr int kNormFwdHoldMaxV = 4;
// With the residual add fused in (a second row in flight a lane) only the lookup
// fits beyond 4 packs, and rows up to norm_fwd_add_max_v() packs a lane.
constexpr bool norm_fwd_holds_weights(int esize, int wsize, int G, int V, bool fast, bool rms,
                                      bool add) {
  if (!fast || G != 1024 || V <= kNormFwdHoldMaxV) return true;
  if (add) return false;
  if (esize == 4) return rms && V <= 8;
  if (wsize == 2) return rms ? V == 8 : V <= 6;
  return rms && V <= 6;
}

constexpr int norm_fwd_add_max_v(int esize, bool rms) { return esize == 4 && !rms ? 10 : 12; }

// Largest packs per lane the register file holds for a G-lane row group.
// G = 1024 means 16 wavefronts per workgroup, i.e. at most 128 VGPRs a lane.
constexpr int v_max(OpClass oc, int esize, int G) {
  int v = 1;
  switch (oc) {
    // (at 1024 lanes without the weights: 16 packs, a 131072-element 16-bit row or
    // a 65536-element fp32 row)
    case OC_NORM_FWD:
      if (G >= 1024) return 16;
      v = esize == 4 ? 16 : 8;
      break;
    // (16-bit rows at 1024 lanes: 4 packs with the dgamma sums in LDS, see
    // norm_bwd_sums_in_lds())
    case OC_NORM_BWD:
      if (G >= 1024 && esize == 2) return 4;
      if (G == 512 && esize == 2) return 5;  // (5: norm_bwd_half_lanes_five())
      v = esize == 4 ? 8 : 4;
      break;
    // the forward keeps long rows in storage format: 16 packs a lane at any
    // G (a 131072-element 16-bit row, a 65536-element fp32 row)
    case OC_SOFTMAX_FWD: return G >= 1024 ? max_v_of(oc, esize) : 16;
    // (16-bit rows at 1024 lanes: 8 packs of each tensor, kept in storage format)
    case OC_SOFTMAX_BWD:
      if (G >= 1024 && esize == 2) return 8;
      v = esize == 4 ? 16 : 8;
      break;
    // GroupNorm lanes hold the row (and dY) only, no weights or column sums, so
    // 16-bit rows keep 8 packs a lane at 1024 lanes (128 VGPRs) and 10 at 512
    // lanes (two workgroups a compute unit); the fp32 forward holds 11 at 1024
    // lanes without spilling, the fp32 backward 4
    case OC_GROUP_FWD: return esize == 4 ? (G >= 1024 ? 11 : 16) : (G == 512 ? 10 : 8);
    case OC_GROUP_BWD: return esize == 4 ? (G >= 1024 ? 4 : 8) : 8;
  }
  if (G >= 1024 && v > 1) v /= 2;
  return v;
}

// Threads per workgroup for a G-lane row group (measured choices):
//   norm forward    256 (BLOCK/G rows per workgroup), G itself above that;
//   norm backward   512 at least: two or more row slots share one partial row
//                   of the dgamma/dbeta reduction;
//   softmax         512 at least;
//   GroupNorm       256 in both directions: its backward keeps no column sums across
//                   rows (the channel sums of a row leave with the row), and with 256
//                   threads bf16 [256, 1024, 14, 14] in 32 groups went 72.0 -> 62.7 us
//                   (dX kernel alone), [256, 2048, 7, 7] 38.8 -> 35.8 us, [64, 1280, 8, 8]
//                   unchanged, [64, 1280, 16, 16] 23.7 -> 24.3 us.
constexpr int block_threads(OpClass oc, int G) {
  const int floor_threads =
      (oc == OC_NORM_FWD || oc == OC_GROUP_FWD || oc == OC_GROUP_BWD) ? 256 : 512;
  return G <= floor_threads ? floor_threads : G;
}

// Whether the resident norm backward requests the rows of its next iteration
// ahead of the current one's arithmetic.  That costs V * 8 registers a lane for
// 16-bit rows.  The two-pack layouts sit just under 128 registers, which keeps
// two 512-thread workgroups on a compute unit, and lose more to a lost
// workgroup than they gain (bf16 [16384, 4096] LayerNorm 78 -> 85 us; with the
// dgamma/dbeta sums moved to LDS to make room, read-add-write 128 bits at a
// time, 78 -> 82 us, and with LDS float atomics ten times that); from three packs
// a lane the kernel holds one workgroup a compute unit anyway and has the
// registers to spare (N = 10240: LayerNorm 208 -> 185 us, RMSNorm 189 -> 176 us;
// with one workgroup a compute unit in the grid as well, see make_plan(), 173
// and 169 us).  The two-pack LayerNorm, whose two sets of column sums make it
// the slower one, gains a little from the prefetch on one workgroup a compute
// unit up to 256 lanes (N = 2048: 44.6 -> 43.3 us, 4096: 78 -> 75 us) and loses a
// little on 512 (N = 7168: 128 -> 130 us, 8192: 142 -> 144 us).
constexpr bool norm_bwd_prefetches(int esize, int G, int V, bool fast, bool rms) {
  if (G >= 1024) return false;  // (3 and 4 packs at 1024 lanes: it spills, 104 -> 172 us)
  return fast && esize == 2 && (V >= 3 || (V == 2 && !rms && G <= 256));
}

// 16-bit backward rows of 16392..32768 elements (hidden sizes 18432, 20480): three
// or four packs a lane on 1024 lanes.  The column sums of such a lane would take
// 48-64 registers beside the row and dY, so the dgamma sums live in LDS (96 / 128
// KB: every lane adds to its own 16-byte slots), the dbeta sums stay in registers
// and gamma stays in memory (L2).  Measured at 4096 rows against the multi-pass
// kernels (two passes over X and dY), bf16: N = 18432 RMSNorm 127 -> 104 us,
// LayerNorm 133 -> 111 us (fp32 weights 147 -> 126 us); 24576: 162 -> 135, 166 ->
// 143, 180 -> 151 us; 32768 RMSNorm 231 -> 175 us.  The LayerNorm with four packs
// spills 29-45 registers and loses (237 -> 302 us): it keeps the multi-pass kernels.
constexpr bool norm_bwd_sums_in_lds(int esize, int G, int V, bool fast) {
  return fast && esize == 2 && G == 1024 && V >= 3;
}
// One case goes through the registers instead: the RMSNorm with 16-bit weights and
// rows of 2049..2560 packs (hidden 18432, 20480) fits 512 lanes x 5 packs with its
// next row on the way in 251 registers, one 512-thread workgroup a compute unit
// (bf16 [16384, 18432] 345 -> 315 us, 72 %; [8192, 20480] 194 -> 176 us).  The
// LayerNorm, fp32 weights and the fused residual gradient spill there (LayerNorm
// 199 -> 351 us) and stay with the LDS sums; so do 6 packs (24576).
constexpr bool norm_bwd_half_lanes_five(int esize, int wsize, int G, int V, bool rms, bool add) {
  return esize == 2 && wsize == 2 && G == 512 && V == 5 && rms && !add;
}
// Exact layouts of the 16-bit norm backward (norm_bwd_exact_kernel): a row of
// `packs` = V * G packs on G lanes, G a whole number of wavefronts.  The table is
// what measured faster than the general resident kernel on MI355X (see the kernel):
// lanes, packs a lane, workgroup threads, row blocks in flight (1 = no prefetch),
// and which calls take it -- LayerNorm / RMSNorm, weights in the row dtype / in
// float32 beside 16-bit rows, with the residual gradient fused in or not.  Two packs
// a lane serve hidden sizes up to 16384; three and four packs a lane keep rows of
// 9216, 18432, 20480 and 24576 elements in registers where the general kernel needs
// its dgamma sums in LDS (bf16 rows x 8192, LayerNorm 18432: 199 -> 165 us, with fp32
// weights 231 -> 166 us; 24576: 258 -> 222 us; RMSNorm with fp32 weights 18432 185 ->
// 158 us, 20480 206 -> 181 us, 24576 231 -> 212 us).
constexpr unsigned kExactLN = 1, kExactLNWide = 2, kExactRMS = 4, kExactRMSWide = 8,
                   kExactAdd = 16;  // (kExactAdd: also with the fused residual gradient)
constexpr unsigned kExactAll = kExactLN | kExactLNWide | kExactRMS | kExactRMSWide;
struct NormBwdExactLayout {
  int G, V, block, depth;
  unsigned calls;
};
constexpr NormBwdExactLayout kNormBwdExact[] = {
    {128, 2, 512, 2, kExactAll | kExactAdd},
    // (the first entry that serves a call is taken: one row slot a workgroup where that
    // measured ahead -- bf16 rows x 16384, LayerNorm 4096 69.4 -> 68.8 us, 5120 88.7 ->
    // 86.5 us, RMSNorm 5120 86.0 -> 83.2 us, 6144 on 384 x 2 instead of 256 x 3 LayerNorm
    // 105.9 -> 102.1 us (fp32 weights 107.3 -> 102.6), RMSNorm 101.9 -> 99.7 us)
    {256, 2, 256, 3, kExactLN | kExactLNWide},
    {256, 2, 512, 3, kExactAll | kExactAdd},
    {320, 2, 320, 3, kExactLN | kExactLNWide},
    {320, 2, 320, 2, kExactRMS | kExactRMSWide},
    {320, 2, 640, 2, kExactAll | kExactAdd},
    {384, 2, 384, 2, kExactAll},
    {448, 2, 448, 2, kExactAll | kExactAdd},
    {512, 2, 512, 3, kExactAll | kExactAdd},
    // (at 896 and 1024 lanes the RMSNorm's general kernel already runs this layout as fast)
    {896, 2, 896, 1, kExactLN | kExactLNWide | kExactAdd},
    {1024, 2, 1024, 1, kExactLN | kExactLNWide | kExactAdd},
    {384, 3, 384, 2, kExactAll},
    {768, 3, 768, 1, kExactLN | kExactLNWide | kExactRMSWide},
    {640, 4, 640, 1, kExactRMSWide},
    {1024, 3, 1024, 1, kExactAll}};
constexpr int kNormBwdExactCount = (int)(sizeof(kNormBwdExact) / sizeof(kNormBwdExact[0]));
constexpr bool norm_bwd_exact_serves(const NormBwdExactLayout& l, bool layer_norm,
                                     bool wide_weights, bool fused_add) {
  const unsigned want = layer_norm ? (wide_weights ? kExactLNWide : kExactLN)
                                   : (wide_weights ? kExactRMSWide : kExactRMS);
  return (l.calls & want) != 0 && (!fused_add || (l.calls & kExactAdd) != 0);
}
// Index into kNormBwdExact of the layout that serves such a call, or -1.
constexpr int norm_bwd_exact_index(int esize, int64_t packs, int64_t M, bool layer_norm,
                                   bool wide_weights, bool fused_add) {
  if (esize != 2) return -1;
  for (int i = 0; i < kNormBwdExactCount; ++i) {
    const NormBwdExactLayout& l = kNormBwdExact[i];
    if (packs == (int64_t)l.V * l.G && norm_bwd_exact_serves(l, layer_norm, wide_weights, fused_add) &&
        M % (l.block / l.G) == 0)
      return i;
  }
  return -1;
}
// Exact two-pack layouts of the 16-bit norm forward (norm_fwd_exact_kernel): lanes,
// workgroup threads, resident workgroups a compute unit.  Hidden 4096 and 5120, where
// it measured 2-5 % ahead of the general resident kernel; not 8192.
struct NormFwdExactLayout {
  int G, block, bpc;
};
constexpr NormFwdExactLayout kNormFwdExact[] = {{256, 512, 2}, {320, 320, 3}};
constexpr int kNormFwdExactCount = (int)(sizeof(kNormFwdExact) / sizeof(kNormFwdExact[0]));
// (up to 128 row blocks a workgroup: at 262144 rows of 4096 the resident grid runs
// at 68 % where the general kernel's grid, which grows with the rows, reaches 75 %)
constexpr int kNormFwdExactMaxIters = 128;
constexpr int norm_fwd_exact_index(int esize, int64_t packs, int64_t M, int num_cus) {
  if (esize != 2) return -1;
  for (int i = 0; i < kNormFwdExactCount; ++i) {
    const int rpb = kNormFwdExact[i].block / kNormFwdExact[i].G;
    if (packs == 2 * (int64_t)kNormFwdExact[i].G && M % rpb == 0 &&
        M / rpb <= (int64_t)num_cus * kNormFwdExact[i].bpc * kNormFwdExactMaxIters)
      return i;
  }
  return -1;
}
// Exact layouts of the 16-bit GroupNorm kernels (gn_fwd_exact_kernel,
// gn_bwd_exact_kernel): one row a workgroup of G lanes with V packs each, for
// rows of exactly G * V packs whose channels are whole runs of 64 packs (the
// 64x64 and 32x32 maps of a diffusion UNet with 32 groups: 10, 20, 30, 40 and 60
// channels a group at 32x32, 10 at 64x64).  Workgroups a compute unit of the
// forward and of the backward grid; 0 = the general resident kernel is faster
// (measured on one MI355X, bf16, 2048 rows; general -> exact, us:
//   1280 packs  forward 14.2 -> 15.0 (kept general)   backward 26.4 -> 22.2
//   2560 packs  forward 29.9 -> 29.3                  backward 49.3 -> 43.0
//   3840 packs  forward 46.6 -> 43.8                  backward 79.4 -> 67.9
//   5120 packs  forward 61.6 -> 58.6                  backward 96.2 -> 84.9 + 3.5
//               (one row a workgroup: 2048 workgroups; a grid of 512 is 2 % behind)
//   7680 packs  forward 94.7 -> 90.2                  backward 140.6 -> 128.0).
struct GroupExactLayout {
  int G, V, bpc_fwd, bpc_bwd;
};
constexpr GroupExactLayout kGroupExact[] = {
    {256, 5, 0, 8}, {512, 5, 3, 2}, {768, 5, 2, 1}, {512, 10, 8, 8}, {960, 8, 1, 1}};
constexpr int kGroupExactCount = (int)(sizeof(kGroupExact) / sizeof(kGroupExact[0]));
constexpr int kGroupExactMaxD = 64;  // channels a group: one lane of a wavefront each
constexpr int group_exact_index(bool backward, int esize, int64_t rows, int64_t L, int64_t HxW,
                                int64_t D) {
  const int E = 8;
  if (esize != 2 || L % E != 0 || HxW % (64 * E) != 0 || D > kGroupExactMaxD ||
      rows > ((int64_t)1 << 31))
    return -1;
  for (int i = 0; i < kGroupExactCount; ++i) {
    const GroupExactLayout& l = kGroupExact[i];
    if (L / E == (int64_t)l.G * l.V && (backward ? l.bpc_bwd : l.bpc_fwd) > 0) return i;
  }
  return -1;
}
// (a 512 x 5 instance exists for that case only)
constexpr bool norm_bwd_instance_ok(int esize, int wsize, int G, int V, bool rms, bool add) {
  return !(esize == 2 && G == 512 && V == 5) || norm_bwd_half_lanes_five(esize, wsize, G, V, rms, add);
}
constexpr bool norm_bwd_lds_layout(int esize, int64_t v_exact, bool layer_norm) {
  return esize == 2 && (v_exact == 3 || (v_exact == 4 && !layer_norm));
}

// Workgroup sizes a G-lane variant is compiled for.
constexpr bool block_built(OpClass oc, int G, int block) {
  if (block < G || block < 256 || block > 1024 || (block & (block - 1))) return false;
  return block == block_threads(oc, G);
}

// How the resident norm backward reads a ragged row.
//   kReadElements: a row's last pack element by element, in a branch of its own.
//   kReadClamped: every lane reads a whole pack, the row's last one where its own would end past
//     the row (load_clamped_pack); takes rows of a pack or more.
//   kReadClampedInside: the same, but lanes wholly past the row read nothing.
// Rows shorter than a pack (N < 8 or 4 elements) run on kMinG lanes, whose kernels keep the element
// loads; make_plan() sees to it that a forced layout does the same.
enum NormBwdRead { kReadElements = 0, kReadClamped = 1, kReadClampedInside = 2 };
constexpr bool norm_bwd_clamps(int G, bool fast) { return !fast && G > kMinG; }
// The clamped form an instance is built for: lanes past the row stay out of it -- their requests
// and the moving of their packs cost up to 8 % of the row loop (fp32 LayerNorm [16384, 4097] 163.5
// -> 148.7 us, fp16 120.8 -> 108.6 at N = 5001) -- except where the branches make the kernel spill
// (the 16-bit LayerNorm on 1024 lanes, which spills without them already: fp16 [8192, 16383] 209 us
// against 226).
constexpr NormBwdRead norm_bwd_read(int esize, int G, bool fast, bool rms) {
  if (!norm_bwd_clamps(G, fast)) return kReadElements;
  return esize == 2 && G >= kMaxG && !rms ? kReadClamped : kReadClampedInside;
}
// The instances that exist with element loads as well, and the calls those serve (us, element loads /
// whole packs):
//   16-bit LayerNorm rows that leave much of 1024 lanes idle -- a wavefront wholly past the row has
//   next to nothing to do there, while the clamped form clears its packs: 16384 fp16 rows of 12289
//   324 / 339, 13001 369 / 354.  In 32nds of the pack slots.  (Plain calls of 1537 to 1600 packs;
//   shorter rows run on whole wavefronts.)
//   Tensors far beyond the caches, rows that fill most of their lanes -- memory-bound, and the
//   requests of the next rows keep the memory busy while one wavefront waits for its elements: fp32
//   LayerNorm [32768, 6143] 460 / 491, [30000, 5001] 341 / 358, RMSNorm [32768, 6143] 454 / 487, [30000,
//   7777] 531 / 567.  (Plain calls beyond 100 million elements; below, whole wavefronts.)
// Calls with a residual gradient go by the same lines, drawn for the plain calls that had these layouts before
// the whole wavefronts did.  There a third tensor is read as well, and the element loads are the faster ones in
// float32 RMSNorm only ([32768, 6143] 634 / 642, [20000, 7777] 485 / 504, but LayerNorm 676 / 599 and [8192, 6143] 180 /
// 157; fp16 LayerNorm [16384, 8193] 648 / 622, [4096, 12289] 213 / 200, with fp32 weights [4096, 8193] 149 / 154; fp16
// RMSNorm on 512 lanes x 3 packs, which no plain call has, [16384, 8193] 311 / 299, [16384, 10001] 395 / 341).
// (add: the call has a residual gradient)
constexpr bool norm_bwd_reads_elements_built(int esize, int G, int V, bool rms, bool add) {
  if (esize == 4) return G == 256 || G == 512;
  return rms ? add && G == 512 && V == 3 : G >= kMaxG;
}
inline bool norm_bwd_reads_elements(int esize, int wsize, int G, int V, bool rms, int64_t M,
                                    int64_t N) {
  if (!norm_bwd_reads_elements_built(esize, G, V, rms, true)) return false;
  const int64_t packs = (N * esize + 15) / 16, slots = (int64_t)G * V;
  if (esize == 4) return packs * 16 > slots * 9 && M * N > 50000000;
  return rms ? M * N > 100000000 : packs * 32 <= slots * (wsize > 2 ? 17 : 25);
}

// Workgroups per compute unit of the grid-stride launch.  The norm kernels keep
// gamma/beta (and the backward column sums) in registers across the rows of a
// workgroup.  Forward: four times as many workgroups as fit on the machine at
// once, so that they drift out of phase (a grid that is exactly resident runs
// its load and store phases in lockstep and loses 5-10% bandwidth) while each
// still amortizes its weight loads over several rows (make_plan() grows this
// grid with the row count).  Backward: every
// workgroup emits one partial row of the dgamma/dbeta reduction, so the grid
// is just what is resident at 1024 threads per CU.  Softmax has no per-column
// state: one workgroup per row block.
constexpr int default_bpc(OpClass oc, int block) {
  if (oc == OC_NORM_FWD) return 4 * (2048 / block);
  if (oc == OC_NORM_BWD) return 1024 / block;
  return 1 << 20;
}

// Which (G, V) kernels exist in the library.  Kept in one place so the
// dispatcher, the planner and the forced-variant check agree.
constexpr bool is_group_class(OpClass oc) { return oc == OC_GROUP_FWD || oc == OC_GROUP_BWD; }

// Kinds of register-resident GroupNorm kernel (see groupnorm_kernels.hpp) and the
// rule that picks one for a shape; E = elements per 16-byte pack of the row dtype.
constexpr int kGnGeneral = 0, kGnUniform = 1, kGnStraddle = 2;
// Channels per group up to which the straddling kernels are taken (their LDS
// array for the parts of packs that belong to the next channel).
constexpr int kGnStraddleMaxD = 512;
constexpr int gn_mode(int64_t L, int64_t HxW, int64_t D, int E) {
  if (HxW % E == 0) return kGnUniform;
  if (L % E == 0 && HxW >= E && D <= kGnStraddleMaxD) return kGnStraddle;
  return kGnGeneral;
}

// GroupNorm rows that would spread over 1024 lanes (one workgroup a compute
// unit, whose load, reduce and store phases then run one after the other) take
// 512 lanes with twice the packs instead while two such workgroups fit a compute
// unit's registers (128 VGPRs a lane): up to 10 packs forward, 7 backward.
// Measured on [64, C, 64, 64] in 32 groups: bf16 forward 71 -> 62 us (C = 320),
// 57 -> 47 us (224); backward 76 -> 63 us (192), 88 -> 71 us (224); fp32
// backward 66 -> 59 us (96).  Eight packs backward spill and gain nothing.
constexpr int group_half_lanes_max_v(OpClass oc) { return oc == OC_GROUP_FWD ? 10 : 7; }

// Masked softmax rows are attention scores: the masked kernels exist up to 32
// elements a lane at 1024 lanes (rows of 32768 elements; the masked 16-bit
// backward, which keeps fp32 copies of both tensors, would spill beyond that
// anyway), and longer masked rows take the multi-pass kernels.
constexpr bool masked_softmax_built(int esize, int G, int V) {
  return !(G == 1024 && V * (16 / esize) > 32);
}

constexpr bool variant_built(OpClass oc, int esize, int G, int V, bool fast) {
  if (G < kMinG || G > kMaxG || (G & (G - 1)) || V < 1 || V > max_v_of(oc, esize)) return false;
  // GroupNorm rows take the packs they have, not the next power of two (a
  // 40960-element bf16 row is 1024 lanes x 5 packs, not x 8): 3 or 5 packs a
  // lane from one wavefront up, anything up to the budget at 1024 lanes
  if (V & (V - 1)) {
    // ragged 16-bit rows just above a power of two (softmax N = 4097: 514 packs of
    // the aligned window) take three packs on half the lanes as well
    if (!fast)
      return (oc == OC_SOFTMAX_FWD || oc == OC_SOFTMAX_BWD || oc == OC_NORM_FWD || oc == OC_NORM_BWD) && esize == 2 &&
             G >= 64 && V == 3 && !(oc == OC_NORM_BWD && G == kMaxG);
    if (V > v_max(oc, esize, G)) return false;
    // softmax rows that need all 1024 lanes (vocabulary-sized) likewise
    // (and the 16-bit forward takes three packs a lane where that fits better)
    if (oc == OC_SOFTMAX_FWD && esize == 2) return G == kMaxG || (G >= 64 && V == 3);
    if (oc == OC_SOFTMAX_FWD || oc == OC_SOFTMAX_BWD) return G == kMaxG;
    // LayerNorm / RMSNorm rows of hidden sizes such as 5120, 6144, 10240, 12288
    // (640, 768, 1280, 1536 16-bit packs): 3 packs a lane; 5 on 512 lanes for the
    // fp32 LayerNorm forward (see norm_layout())
    if (!is_group_class(oc)) {
      if (oc == OC_NORM_BWD && G == 512 && esize == 2 && V == 5) return true;
      // (16-bit forward rows of 2049..3072 packs: 5 or 6 packs on 512 lanes, see make_plan())
      if (oc == OC_NORM_FWD && G == 512 && esize == 2 && (V == 5 || V == 6)) return true;
      if (oc == OC_NORM_FWD && G == kMaxG && V > kNormFwdHoldMaxV)
        return V == 5 || V == 6 || V == 10 || V == 12;
      return G >= 64 && (V == 3 || (V == 5 && oc == OC_NORM_FWD && esize == 4 && G == 512));
    }
    // (and 6..10 packs on 512 lanes, which make_plan() prefers to 1024 lanes)
    return G == kMaxG || (G >= 64 && (V == 3 || V == 5)) ||
           (G == 512 && V <= group_half_lanes_max_v(oc));
  }
  if (V > v_max(oc, esize, G)) return false;
  // ragged rows: the general kernels exist for the preferred packs per lane only;
  // longer ragged rows take the multi-pass kernels (measured faster for softmax
  // at vocabulary sizes such as 50257 than a general kernel with more packs)
  if (!fast) return V == v_pref(oc, esize);
  if (G == kMinG) return V <= v_pref(oc, esize);
  // short rows take one pack a lane on up to one wavefront (see make_plan())
  if ((oc == OC_NORM_FWD || oc == OC_NORM_BWD || oc == OC_SOFTMAX_FWD || oc == OC_SOFTMAX_BWD) &&
      G <= 64 && V == 1)
    return true;
  if (is_group_class(oc) || G == kMaxG) return V >= v_pref(oc, esize);
  // below the lane maximum make_plan() takes the preferred packs a lane (more lanes
  // before more packs), with one measured exception: 16-bit norm rows of 1537..2048
  // packs on 512 lanes x 4.  Other layouts are never selected and are not compiled
  // (a third of the kernels otherwise).
  if ((oc == OC_NORM_FWD || oc == OC_NORM_BWD) && esize == 2 && G == 512 && V == 4) return true;
  return V == v_pref(oc, esize);
}

inline int pow2_ceil(int64_t v) {
  int p = 1;
  while (p < v) p <<= 1;
  return p;
}

// LayerNorm / RMSNorm rows that the power-of-two rule serves badly (measured on
// MI355X at 16384 rows; "slots" = lanes x preferred packs of that rule):
//  * a 16-bit row of 1025..2048 packs would take 1024 lanes, 16 wavefronts around
//    every reduction: 512 lanes with 3 or 4 packs each are faster in the forward
//    (LayerNorm 160 -> 116 us at N = 10240, RMSNorm 2-4 %) and in the LayerNorm
//    backward (250 -> 206 us); the RMSNorm backward gains only with 3 packs
//    (N = 12288: 222 -> 212 us) and keeps 1024 lanes beyond 1536 packs;
//  * a row that fills at most three quarters of the slots takes three packs on a
//    quarter of the slots' lanes instead: hidden sizes such as 1536, 3072, 6144,
//    12288 fit exactly, 2560, 5120, 10240 to 83 % (16-bit forward 3-14 %, fp32
//    LayerNorm backward 5-15 %).  The LayerNorm forward with fp32 weights below
//    512 lanes is the exception, and so is the 16-bit backward below 512 packs;
//  * fp32 LayerNorm forward rows of 2049..2560 packs: 512 lanes x 5 (N = 10240:
//    261 -> 222 us).
// Returns false where the general rule stands.
inline bool norm_layout(OpClass oc, int esize, int64_t packs, bool layer_norm, bool wide_weights,
                        int* G_out, int* V_out) {
  const int vp = v_pref(oc, esize);
  int G2 = pow2_ceil((packs + vp - 1) / vp);
  if (G2 < kMinG) G2 = kMinG;
  if (G2 > kMaxG) G2 = kMaxG;
  const int64_t slots = (int64_t)G2 * vp;
  if (packs > slots) return false;
  const bool fwd = oc == OC_NORM_FWD;
  const bool sparse = packs * 4 <= slots * 3;
  int G = 0, V = 0;
  if (esize == 2) {
    if (G2 == kMaxG) {
      if (sparse) {
        G = 512, V = 3;
      } else if (fwd || layer_norm) {
        G = 512, V = 4;
      }
    } else if (fwd && sparse && !(layer_norm && wide_weights && G2 < 512)) {
      // (fp32 gamma and beta beside 16-bit rows: three packs of each are 48
      // registers, and below 512 lanes the two-pack layout stays ahead)
      G = G2 / 2, V = 3;
    } else if (!fwd && sparse && G2 >= 512) {
      // the backward with three packs a lane requests its next rows ahead:
      // N = 5120: LayerNorm 95 -> 93 us, RMSNorm 92 -> 87 us; 6144: 112 -> 107 us
      // and 108 -> 102 us
      G = G2 / 2, V = 3;
    }
  } else {
    if (fwd && layer_norm && G2 == kMaxG && packs <= 2560) {
      G = 512, V = 5;
    } else if (sparse) {
      G = G2, V = 3;
    }
  }
  if (G == 0 || (int64_t)G * V < packs || !variant_built(oc, esize, G, V, true)) return false;
  *G_out = G;
  *V_out = V;
  return true;
}

// Lanes a ragged 16-bit row of `packs` packs takes in the norm forward (the rule of
// make_plan() below for such rows: two packs a lane, or three on half the lanes when
// the row fills at most three quarters of the two-pack slots), computed ahead of the
// plan because the lanes decide whether `packs` counts the row's window or the row.
inline int ragged_norm_fwd_lanes(int64_t packs, const Override& ov) {
  if (ov.G > 0) return ov.G;
  int G = pow2_ceil((packs + 1) / 2);
  if (G < kMinG) G = kMinG;
  if (G > kMaxG) G = kMaxG;
  if (ov.V == 0 && G >= 128 && packs <= (int64_t)G * 2 && packs * 4 <= (int64_t)G * 2 * 3 &&
      variant_built(OC_NORM_FWD, 2, G / 2, 3, false))
    G /= 2;
  return G;
}

// The layouts on whole wavefronts: instances (packs a lane, rows in registers, threads), forward and
// backward, 16-bit and float32 rows.
struct WavesInstance {
  int v, depth, threads;
};
constexpr WavesInstance kWavesFwd16[] = {{1, 3, 1024}, {2, 3, 1024}};
constexpr WavesInstance kWavesFwd32[] = {{3, 2, 512}};
constexpr WavesInstance kWavesBwd16[] = {{1, 3, 1024}, {2, 2, 768}};
constexpr WavesInstance kWavesBwd32[] = {{3, 3, 512}, {3, 2, 768}};
constexpr int kWavesMax = 16;  // wavefronts a workgroup at most
// LDS floats the backward folds its row slots' column sums through (two slots or more of one pack a lane
// in 16 bits, three in float32, beside a second set of sums)
constexpr int kWavesFoldFloats = 8192;

// Whether a ragged 16-bit backward call has rows enough for them: a workgroup of sixteen wavefronts holds
// several short rows at a time, and where its slots see a row or two each there is nothing to have on its way,
// while the general layout spreads the rows over up to four times as many workgroups.  us, general layout /
// whole wavefronts: up to 128 packs (eight slots) fp16 LayerNorm [881, 739] 8.8 / 9.6, [1830, 869] 10.3 / 11.1,
// bf16 RMSNorm [2395, 547] 10.3 / 11.0, from twelve rows a compute unit on [3100, 850] 13.5 / 13.0; up to 192 (five)
// RMSNorm [1213, 1401] 9.6 / 10.6, fp32 weights [1997, 1317] 10.6 / 11.0, eight rows; up to 256 (four) LayerNorm
// [910, 1807] 11.0 / 11.5, a row for every slot; beyond (three and two) RMSNorm [538, 2249] 9.5 / 10.1, [412, 3791]
// 10.5 / 10.9, likewise.  The LayerNorm, which waits for two sums, gains with five, three and two slots whatever
// the rows ([600, 2201] 12.6 / 10.3).
inline bool norm_waves_bwd_rows(int64_t M, int64_t packs, bool layer_norm, int num_cus) {
  const int64_t waves = (packs + 63) / 64;
  if (waves == 2) return M >= 12 * (int64_t)num_cus;
  if (waves != 4 && layer_norm) return true;
  return M >= (waves == 3 ? 8 : 16 / waves) * num_cus;
}

// Whether a 16-bit backward call of whole packs, 257 to 1024 of them, takes them (us, general layout / whole
// wavefronts).  From 8192 rows on below 513 packs, see below, the LayerNorm beyond 448 up to 200 million elements
// (fp32 weights [40000, 3968] 165 / 163, [104347, 4072] 455 / 478).  Of 513 to 768 packs, where nine to twelve
// wavefronts work of the sixteen that a compute unit's one workgroup has room for, and the general layout has its
// three packs on 256 lanes, calls of up to 50 million elements: beyond, memory is the bound and more wavefronts
// keep it busier (bf16 LayerNorm [8192, 5448] 54 / 53, [36503, 5360] 201 / 215, [52273, 5288] 291 / 320, RMSNorm with
// fp32 weights [104044, 5160] 565 / 636); but not the LayerNorm up to 544, which leaves nearly half of those
// lanes idle ([52000, 4184] 238 / 210).
inline bool norm_waves_bwd_whole(int64_t M, int64_t N, int64_t packs, bool layer_norm) {
  const int64_t n = M * N;
  if (packs <= 512) return M >= 8192 && !(layer_norm && packs > 448 && n > 200000000);
  return packs > 768 || n <= 50000000 || (layer_norm && packs <= 544);
}

// Whether a call on ragged float32 rows of more than 256 packs takes them (us, general layout / whole
// wavefronts).  The forward is the LayerNorm's, from sixteen rows a compute unit on; beyond 60 million elements
// memory is the bound, and four times as many small workgroups out of phase keep it busier ([37590, 4065]
// 228 / 250, [91025, 2949] 388 / 424; up to there 0.78 to 0.98 of the time: [12000, 4097] 73 / 66); of 385 to 512
// packs, which the general layout's 128 lanes hold without a gap, beyond 20 million ([47928, 1559] 116 / 125,
// [8192, 1999] 22.6 / 21.2); not so from 1025 packs on, which leave a third of that layout idle.
// The backward gains up to 100 million elements (0.75 to 0.97 of the time), and up to 768 packs beyond; with more,
// there, the general layout's loads in several workgroups again ([55957, 3777] 483 / 504, [27414, 8269] 521 / 542).
// Rows of more than 1536 packs, one at a time on a compute unit, need a round and a half of them, beyond 2048
// packs two and a half: the general layout works on two at a time ([279, 8061] 21.0 / 21.8, [485, 8743] 25.6 / 27.4,
// RMSNorm [259, 6521] 12.6 / 13.4; [700, 8743] 37.3 / 35.5).
inline bool norm_waves_float_rows(bool backward, int64_t M, int64_t N, int64_t packs, bool layer_norm,
                                  int num_cus) {
  const int64_t n = M * N;
  if (!backward) {
    if (!layer_norm || M < 16 * (int64_t)num_cus) return false;
    return packs > 1024 || n <= (packs > 384 && packs <= 512 ? 20000000 : 60000000);
  }
  if (packs > 1536 && 2 * M < (packs > 2048 ? 5 : 3) * (int64_t)num_cus) return false;
  return packs <= 768 || n <= 100000000;
}

// Whether a ragged 16-bit forward call takes them (us, general layout / whole wavefronts).  The RMSNorm of 577 to
// 768 packs, ten to twelve wavefronts of sixteen, not from four to 31 rows a compute unit ([4832, 4667] 19.3 / 21.3,
// fp32 weights [2687, 5681] 13.8 / 14.8, but [600, 5001] 6.5 / 6.1 and [16384, 4801] 61 / 57), and that of more than
// 896, whose window the general layout's 512 lanes hold without a gap, below four only, with fp32 weights always
// ([21154, 7883] 121 / 129).  The LayerNorm with weights of the rows' type not beyond 60 million elements where row
// slots leave wavefronts of a workgroup idle (161 to 192 and 321 to 384 packs: [30825, 2565] 66 / 72, [94118,
// 1293] 103 / 110, but [16821, 2669] 45 / 40).
inline bool norm_waves_fwd_rows(int64_t M, int64_t N, int64_t packs, bool layer_norm, bool wide_weights,
                                int num_cus) {
  if (layer_norm)
    return wide_weights || M * N <= 60000000 || !(packs <= 192 || (packs > 320 && packs <= 384));
  if (packs > 576 && packs <= 768) return M < 4 * (int64_t)num_cus || M >= 32 * (int64_t)num_cus;
  return packs <= 896 || wide_weights || M < 4 * (int64_t)num_cus;
}

// Which rows take them.  One pack a lane and three rows in registers in 16 bits, with one workgroup of up to
// sixteen wavefronts a compute unit: what is idle of a row's slots is less than a wavefront, and every row
// slot has two rows on their way.  Beyond 1024 packs the backward holds two packs a lane and two rows (ragged
// rows to 1536 packs); float32 rows three packs.  Measured against the general layouts, us, 8192 fp16 rows
// that start 4 bytes off a boundary: LayerNorm backward N = 521 16.6 -> 15.8, 1401 24.9 -> 21.4, 2049 35.6 ->
// 27.0, 4097 57.2 -> 47.2, 8191 103 -> 86, 8193 128 -> 97, 12001 175 -> 131, RMSNorm (bf16) 2049 29.0 -> 25.6,
// 8191 97 -> 82, 1024 rows of 4097 22.8 -> 16.5; LayerNorm forward 1401 14.8 -> 13.8, 2049 19.6 -> 17.6, 4097
// 34.3 -> 27.9, 8191 60.4 -> 48.5; fp32 LayerNorm 2049 forward / backward 33.0 / 46.1 -> 26.7 / 42.6, 4097 55.6
// / 80.9 -> 50.2 / 77.7.  Whole-pack rows that no exact layout serves gain in the backward, where theirs
// leave lanes idle (16384 rows of 2304 48.9 -> 43.6, 4608 84.8 -> 77.9, 6656 117 -> 113; from 513 packs also
// few rows, 2048 of 4608 21.4 -> 19.6, below only many: 2048 of 2560 14.0 -> 14.6).  The other sides of the
// lines: forward rows of 1025 12.1 -> 12.8, RMSNorm 1401 11.8 -> 12.6 and, in float32, 2305 28.3 -> 30.1 (no
// second reduction to wait for); 1024 float32 rows of 4001 8.6 -> 9.4, which are too few to fill three row
// slots a workgroup; whole-pack forward rows, which four times as many small workgroups serve as well.
// Forward rows of 513 to 640 packs would leave seven of sixteen wavefronts without a row: two packs a lane,
// three row slots (4097 30.6 -> 27.9).
inline WavesLayout norm_waves_layout(bool backward, int esize, int64_t M, int64_t N, bool whole_packs,
                                     bool layer_norm, bool wide_weights, int64_t partial_rows, int num_cus) {
  WavesLayout l;
  const int E = 16 / esize;
  const int64_t packs = (N + E - 1) / E;
  int which = -1;
  if (esize == 2) {
    if (backward) {
      if (whole_packs ? packs > 256 && packs <= 1024 && norm_waves_bwd_whole(M, N, packs, layer_norm)
                      : packs > 64 && packs <= 1024 && norm_waves_bwd_rows(M, packs, layer_norm, num_cus))
        which = 0;
      else if (!whole_packs && packs > 1024 && packs <= 1536)
        which = 1;
    } else if (!whole_packs && packs > (layer_norm ? 160 : 320) && packs <= 1024 &&
               norm_waves_fwd_rows(M, N, packs, layer_norm, wide_weights, num_cus)) {
      which = packs > 512 && packs <= 640 && M >= 16 * (int64_t)num_cus ? 1 : 0;
    }
  } else if (!whole_packs && packs > 256 && packs <= (backward ? 2304 : 1152) &&
             norm_waves_float_rows(backward, M, N, packs, layer_norm, num_cus)) {
    which = packs <= 1536 ? 0 : 1;
  }
  // (a row for every compute unit at least: fewer are as fast on either layout, and keep the bits they have in
  // common with the fused add, which has the general one -- 130 rows within 3 % of one another up to 8191)
  if (which < 0 || M < num_cus || M > 0x7fffffff / 2) return l;
  const WavesInstance& in =
      esize == 2 ? (backward ? kWavesBwd16 : kWavesFwd16)[which] : (backward ? kWavesBwd32 : kWavesFwd32)[which];
  const int64_t waves = (packs + 64 * in.v - 1) / (64 * in.v);
  const int most = in.threads / 64;
  // (only the last of a lane's packs may reach past the row)
  if (waves > most || (in.v - 1) * 64 * waves * E > N) return l;
  int64_t grid = (int64_t)num_cus * (!backward && in.threads == 512 ? 2 : 1);
  if (backward && partial_rows > 0 && grid > partial_rows) grid = partial_rows;
  int64_t slots = most / waves;
  const int64_t want = (M + grid - 1) / grid;
  if (slots > want) slots = want;
  const int64_t nrb = (M + slots - 1) / slots;
  l.waves = (int)waves;
  l.v = in.v;
  l.depth = in.depth;
  l.threads = in.threads;
  l.slots = (int)slots;
  l.grid = (int)(grid < nrb ? grid : nrb);
  return l;
}

// Teams of a norm backward whose rows of `packs` packs are beyond one workgroup's registers (norm_bwd_team_kernel):
// workgroups a team, teams (0: none), whether they make enough rounds to be worth it.  whole: what the kernel takes
// (whole packs, no residual gradient).
struct NormBwdTeam {
  int64_t team = 0, teams = 0;
  bool rounds_ok = false;
};
inline NormBwdTeam norm_bwd_team(int64_t M, int64_t packs, bool whole, bool layer_norm, int num_cus) {
  const int64_t cus = num_cus * kTeamBwdPerCu < kTeamMaxWorkgroups ? num_cus * kTeamBwdPerCu : kTeamMaxWorkgroups;
  const int64_t chunk = (int64_t)kTeamBwdPacks * kTeamBlock;
  const int64_t groups = (M + kTeamBwdRows - 1) / kTeamBwdRows;
  NormBwdTeam t;
  t.team = (packs + chunk - 1) / chunk;
  if (!whole || t.team < 2 || t.team > cus) return t;
  t.teams = cus / t.team < groups ? cus / t.team : groups;
  // Worth it from the second round on (a call costs about 25 us beside 9.5-10 us a round,
  // where the two passes of the other kernels cost about 14.6 us for a round's rows); a
  // LayerNorm on large teams (more than 64 workgroups a row) from the fourth.  Measured,
  // bf16, LayerNorm / RMSNorm, team against two passes in us: [512, 401408] (26 rounds)
  // 258 / 243 against 359 / 350; [4096, 65536] (64) 330 / 308 against 478 / 468; [100,
  // 401408] (5) 66 / 59 against 80 / 75; [1024, 40960] (5) 82 / 72 against 81 / 75; [512,
  // 65536] (4) 62 / 52 against 68 / 63; [32, 401408] (2) 34 / 29 against 41 / 37; [64,
  // 262144] (2) 41 / 32 against 41 / 38; [16, 1048576] (2, 128 workgroups a row) 41 / 31
  // against 35 / 34; [8192, 24584] (a row's last workgroup holds a single pack) 327
  // against 380.
  t.rounds_ok = layer_norm && t.team > 64 ? groups >= 4 * t.teams : groups > t.teams;
  return t;
}

// Returns 0, or -5 (ROWNORM_ERR_OVERRIDE) when a forced variant cannot hold the row.
// force_general: take the general (ragged-row) kernels even when N % E == 0.
// layer_norm: the norm op is LayerNorm (statistics of two sums, beta), not RMSNorm.
// wide_weights: fp32 gamma/beta beside 16-bit rows.
// off_line: a tensor of the call does not start on a 128-byte cache line.
// fused_add: the norm forward adds a residual row first (two rows in flight a lane);
// the norm backward adds the residual path's gradient to dX.
// masked: the softmax call reads a mask (see masked_softmax_built()).
// want_dx: the norm backward writes dX (its exact layouts exist for such calls only).
inline int make_plan(OpClass oc, int64_t M, int64_t N, int esize, int num_cus, const Override& ov,
                     bool want_cols, Plan* out, bool force_general = false,
                     bool layer_norm = false, bool wide_weights = false, bool off_line = false,
                     bool fused_add = false, bool masked = false, bool want_dx = true) {
  Plan p;
  const int E = 16 / esize;
  p.fast = (N % E) == 0 && !force_general;
  p.forced = ov.G != 0 || ov.V != 0 || ov.block != 0;
  const bool softmax = oc == OC_SOFTMAX_FWD || oc == OC_SOFTMAX_BWD;
  // the general softmax kernels address a 16-bit row through the 16-byte aligned
  // window that holds it, which starts up to E - 1 elements before the row
  int64_t packs = ((softmax && !p.fast && esize == 2 ? N + E - 1 : N) + E - 1) / E;
  // and so does the general norm forward on 256 lanes or more (norm_row_window()): the
  // lanes a row takes follow from its window's packs (halved below when three packs
  // a lane fit better, hence 512 here)
  if (oc == OC_NORM_FWD && !p.fast && esize == 2 && ov.G >= 0) {
    const int64_t wpacks = (N + E - 1 + E - 1) / E;
    if (norm_row_window(esize, ragged_norm_fwd_lanes(wpacks, ov), false)) {
      p.window = true;
      packs = wpacks;
    }
  }
  if (num_cus <= 0) num_cus = 256;
  bool stream = ov.G < 0;
  if (!stream) {
    int G, V;
    if (ov.G > 0) {
      G = ov.G;
    } else {
      G = pow2_ceil((packs + v_pref(oc, esize) - 1) / v_pref(oc, esize));
      if (G < kMinG) G = kMinG;
      if (G > kMaxG) G = kMaxG;
    }
    // GroupNorm rows of a wavefront or more (measured): about 5 packs a lane on
    // as few lanes as that allows, and exactly the packs the row has
    bool group_exact = false;
    if ((oc == OC_NORM_FWD || oc == OC_NORM_BWD) && p.fast && ov.G == 0 && ov.V == 0)
      group_exact = norm_layout(oc, esize, packs, layer_norm, wide_weights, &G, &V);
    // 16-bit forward rows of 2049..3072 packs (hidden 18432, 20480, 24576) would take
    // 1024 lanes x 3 or 4 packs, one workgroup a compute unit whose load, reduce and
    // store phases run one after the other; two 512-lane workgroups with 5 or 6 packs
    // a lane and their weights held overlap them.  Interleaved A/B at 8192 rows of
    // bf16, LayerNorm: N = 18432 121 -> 107 us (fp32 weights 122 -> 113), 20480 129 ->
    // 116 (133 -> 118), 24576 145 -> 138 (148 -> 136); 8 packs (32768) lose to 1024 x 4.
    // The RMSNorm and the fused residual add (a second row in flight) keep 1024 lanes,
    // with exactly the 3 packs such a row has (below): RMSNorm 18432 98.7 us against
    // 102.8 on 512 x 5 and 105 on 1024 x 4; add + LayerNorm 217 us against 228 on 1024 x 4.
    if (oc == OC_NORM_FWD && p.fast && esize == 2 && layer_norm && !fused_add && ov.G == 0 &&
        ov.V == 0 && packs > 2048 && packs <= 3072) {
      G = 512;
      V = packs <= 2560 ? 5 : 6;
      group_exact = true;
    }
    if (oc == OC_NORM_BWD && p.fast && ov.G == 0 && ov.V == 0 && packs > 2048 && packs <= 2560 &&
        norm_bwd_half_lanes_five(esize, wide_weights ? 4 : esize, 512, 5, !layer_norm, fused_add)) {
      G = 512;
      V = 5;
      group_exact = true;
    }
    // Norm rows of at most one wavefront of packs: with one pack a lane, a load
    // instruction of a wavefront covers one contiguous span of 64 packs (several
    // whole rows), while with V packs a lane it covers 64/G separate pieces of
    // G packs, and every piece that does not start on a cache line touches one
    // line more: 2 instead of 1 at G = 8.  Measured at 2^25 elements (fp32; rows
    // of 64 / 128 / 256 elements that start 8 bytes into a line): LayerNorm
    // forward 160 / 139 / 109 -> 105 / 104 / 105 us, backward 238 / 221 / 178 ->
    // 157 / 156 / 158 us; fp16 rows of 128 elements 78 -> 56 us and 125 -> 83 us.
    // On line-aligned rows the backward gains 4-5 % as well (its column sums take
    // a quarter of the registers), the LayerNorm forward loses 5 %: the forward
    // takes this layout for rows off the line only.
    // Softmax rows behave like the norm forward (off a line, fp32 rows of 64 / 128
    // elements: forward 130 / 138 -> 98 / 95 us, backward 172 / 198 -> 128 / 129 us;
    // on a line the forward loses 5-9 % and the backward is unchanged).
    const bool norm_or_softmax = oc == OC_NORM_FWD || oc == OC_NORM_BWD || softmax;
    if (norm_or_softmax && p.fast && ov.G == 0 && ov.V == 0 && packs <= 64 &&
        (oc == OC_NORM_BWD || off_line)) {
      G = pow2_ceil(packs);
      if (G < kMinG) G = kMinG;
      V = 1;
      group_exact = true;
    }
    // 16-bit softmax forward (its exp makes it the arithmetic-heavy one), ragged
    // 16-bit softmax rows in both directions and ragged 16-bit norm rows:
    // a row that fills at most three quarters of the two-pack slots takes three
    // packs on half the lanes (softmax N = 5120: 62 -> 56 us, 10240: 120 -> 110 us
    // at 16384 rows; at 8192 rows LayerNorm forward N = 4097: 60 -> 52 us; RMSNorm
    // backward 4097: 62 -> 55 us, 8193: 115 -> 97 us).  The ragged LayerNorm backward
    // is the exception: its three-pack kernels take 155 registers (one workgroup a
    // compute unit) where two packs on all the lanes keep two (N = 1025: 60 -> 40 us,
    // 2049: 80 -> 65 us at 16384 rows; 4097: 79 -> 66 us, 5121: 86 -> 76 us at 8192).
    const bool ragged_norm = !p.fast && (oc == OC_NORM_FWD || (oc == OC_NORM_BWD && !layer_norm));
    if (((softmax && (oc == OC_SOFTMAX_FWD || !p.fast)) || ragged_norm) &&
        esize == 2 && ov.G == 0 && ov.V == 0 &&
        G >= 128 && packs <= (int64_t)G * 2 && packs * 4 <= (int64_t)G * 2 * 3 &&
        variant_built(oc, esize, G / 2, 3, p.fast)) {
      G /= 2;
      V = 3;
      group_exact = true;
    }
    if (is_group_class(oc) && p.fast && ov.G == 0 && ov.V == 0) {
      int Gg = pow2_ceil((packs + 4) / 5);
      if (Gg > kMaxG) Gg = kMaxG;
      if (Gg >= 64) {
        int Vg = (int)((packs + Gg - 1) / Gg);
        if (Gg == kMaxG && packs <= 512 * (int64_t)group_half_lanes_max_v(oc) &&
            variant_built(oc, esize, 512, (int)((packs + 511) / 512), true)) {
          Gg = 512;
          Vg = (int)((packs + 511) / 512);
        }
        while (Vg < kMaxV && !variant_built(oc, esize, Gg, Vg, true)) ++Vg;
        if (variant_built(oc, esize, Gg, Vg, true)) {
          G = Gg;
          V = Vg;
          group_exact = true;
        }
      }
    }
    if (ov.V > 0) {
      V = ov.V;
    } else if (!group_exact) {
      V = pow2_ceil((packs + G - 1) / G);
      const int64_t v_exact = (packs + G - 1) / G;
      if (softmax && p.fast && G == kMaxG &&
          v_exact <= max_v_of(oc, esize) && variant_built(oc, esize, G, (int)v_exact, true))
        V = (int)v_exact;
      // norm backward beyond two packs a lane on 1024 lanes: norm_bwd_sums_in_lds()
      if (oc == OC_NORM_BWD && p.fast && G == kMaxG && v_exact > 2 && esize == 2)
        V = norm_bwd_lds_layout(esize, v_exact, layer_norm) ? (int)v_exact : kMaxV + 1;
      // three packs a lane at 1024 lanes, not four with a quarter of them outside the row
      if (oc == OC_NORM_FWD && p.fast && G == kMaxG && v_exact == 3 &&
          variant_built(oc, esize, G, 3, true))
        V = 3;
      // norm forward rows beyond the packs whose weights a lane holds: the next
      // pack count that is built (5, 6, 8, 10, 12, 16)
      if (oc == OC_NORM_FWD && p.fast && G == kMaxG && v_exact > kNormFwdHoldMaxV) {
        int64_t v = v_exact;
        while (v < kMaxV && !variant_built(oc, esize, G, (int)v, true)) ++v;
        V = (int)v;
        if (fused_add && V > norm_fwd_add_max_v(esize, !layer_norm)) V = kMaxV + 1;  // multi-pass
        // a handful of the longest rows: one workgroup takes 15 us for a row of 131072
        // bf16 elements, the split over workgroups 10 us for up to 64 of them (128 rows:
        // 19 us either way; rows of 65536 and fewer are faster here from 16 rows down)
        if (V >= 10 && M < num_cus / 2) V = kMaxV + 1;
      }
      if (!p.fast && V < v_pref(oc, esize)) V = v_pref(oc, esize);
    }
    // masked rows beyond 32 elements a lane at 1024 lanes: the multi-pass kernels
    if (softmax && masked && ov.V == 0 && !masked_softmax_built(esize, G, V)) V = kMaxV + 1;
    const bool holds = (int64_t)G * V >= packs;
    const int block = ov.block > 0 ? ov.block : block_threads(oc, G);
    const bool built = variant_built(oc, esize, G, V, p.fast) && block_built(oc, G, block) &&
                       !(softmax && masked && !masked_softmax_built(esize, G, V)) &&
                       !(oc == OC_NORM_BWD && p.fast &&
                         !norm_bwd_instance_ok(esize, wide_weights ? 4 : esize, G, V, !layer_norm,
                                               fused_add));
    if (ov.G > 0 || ov.V > 0 || ov.block > 0) {
      if (!holds || !built) return -5;
    }
    if (holds && built) {
      p.resident = true;
      p.G = G;
      p.V = V;
      p.block = block;
      if (oc == OC_NORM_BWD && N < E && norm_bwd_clamps(G, p.fast)) {
        p.G = kMinG;
        p.V = v_pref(oc, esize);
        p.block = block_threads(oc, kMinG);
      }
      p.rpb = p.block / p.G;
      // 16-bit forward rows likewise (plain calls: no residual add, no output cast)
      if (oc == OC_NORM_FWD && p.fast && !fused_add && !p.forced && ov.bpc == 0) {
        const int xi = norm_fwd_exact_index(esize, packs, M, num_cus);
        if (xi >= 0) {
          p.G = kNormFwdExact[xi].G;
          p.V = 2;
          p.block = kNormFwdExact[xi].block;
          p.rpb = p.block / p.G;
          p.exact_depth = 1;
        }
      }
      // 16-bit backward rows that fill a two-pack layout of whole wavefronts
      if (oc == OC_NORM_BWD && p.fast && want_dx && !p.forced) {
        const int xi = norm_bwd_exact_index(esize, packs, M, layer_norm, wide_weights, fused_add);
        if (xi >= 0) {
          p.G = kNormBwdExact[xi].G;
          p.V = kNormBwdExact[xi].V;
          p.block = kNormBwdExact[xi].block;
          p.rpb = p.block / p.G;
          p.exact_depth = kNormBwdExact[xi].depth;
        }
      }

    } else {
      stream = true;
    }
  }
  if (stream) {
    p.resident = false;
    p.G = kStreamBlock;
    p.V = 0;
    p.block = kStreamBlock;
    p.rpb = 1;
  }
  const int64_t nrb = (M + p.rpb - 1) / p.rpb;
  int bpc = ov.bpc > 0 ? ov.bpc : default_bpc(oc, p.block);
  // LayerNorm forward with fp32 gamma/beta beside 16-bit rows: every workgroup
  // loads twice the weight bytes, so 256-thread workgroups take half the grid
  // (16384 rows of bf16: N = 4096 53.0 -> 50.7 us, 5120 64.4 -> 62.0 us, 6144
  // 75.7 -> 73.3 us; RMSNorm and 512-thread workgroups measured no gain)
  if (ov.bpc == 0 && oc == OC_NORM_FWD && p.resident && layer_norm && wide_weights &&
      p.block == 256)
    bpc /= 2;
  // The backward that prefetches its next rows holds one workgroup a compute unit:
  // a grid of that size halves the partial rows of the dgamma/dbeta reduction
  // (bf16 [16384, 12288]: LayerNorm 222 -> 208 us, RMSNorm 210 -> 204 us)
  if (ov.bpc == 0 && oc == OC_NORM_BWD && p.resident &&
      (p.exact_depth > 0 || norm_bwd_prefetches(esize, p.G, p.V, p.fast, !layer_norm)))
    bpc = 1;
  int64_t grid = (int64_t)num_cus * bpc;
  // The norm forward beyond a few tens of thousands of rows (measured on bf16 rows
  // of 2048..8192 elements, 65536 and 262144 rows): a workgroup that walks more
  // than a handful of row blocks loses bandwidth (32 iterations: 65 % against
  // 76 %), one that walks too few reloads gamma/beta too often.  The grid grows
  // with the row count so that a workgroup makes about 2 (RMSNorm) or 4
  // (LayerNorm) iterations, twice that with fp32 weights beside 16-bit rows.
  if (oc == OC_NORM_FWD && p.resident && ov.bpc == 0) {
    const int iters = (layer_norm ? 4 : 2) * (wide_weights ? 2 : 1);
    const int64_t want = (nrb + iters - 1) / iters;
    if (grid < want) grid = want;
    // Up to a few tens of thousands of rows, fp32 weights beside 16-bit rows (and
    // LayerNorm on 512 lanes with any weights) take the other regime: three
    // 256-thread or two 512-thread workgroups a compute unit, all resident at once,
    // each walking up to 32 row blocks -- the weights are loaded once per 4..32 rows
    // and no second wave of workgroups leaves a tail.  Interleaved A/B runs, bf16
    // rows, LayerNorm with fp32 weights at 2048 / 4096 / 16384 rows: N = 4096 9.8 /
    // 17.4 / 48.9 -> 8.2 / 13.5 / 46.0 us, N = 8192 17.7 / 33.2 / 93.3 -> 14.2 / 24.3 /
    // 88.6 us; 16384 rows of 5120 / 6144: 61.2 / 72.1 -> 58.9 / 67.6 us (four
    // workgroups of 256 instead of three: 60.1 / 72.3 us).  RMSNorm with fp32 weights,
    // 16384 rows: N = 5120 56.8 -> 54.8, 7168 80.0 -> 76.0, 8192 89.3 -> 85.3, 12288
    // 135.2 -> 128.3 us.  LayerNorm with bf16 weights on 512 lanes: 7168 80.9 -> 77.4,
    // 8192 89.2 -> 86.9, 12288 136.3 -> 131.6 us (10240: 115.3 -> 117.1).  With bf16
    // weights on 256 lanes, and for RMSNorm with bf16 weights, the two regimes are
    // within 1 % at 4096-6144 and the small grid loses 3 % at 10240; the
    // residual-add forward, with twice the bytes in flight, loses 7 % on it: they
    // keep the grid above.  Rows on fewer than 256 lanes (two row slots a workgroup)
    // do not gain (N = 3072: 38.1 -> 40.0 us).  At 65536 rows and beyond (64+ row
    // blocks a workgroup) the small grid loses 3-10 %.  Grids in between (6-8
    // workgroups a compute unit, where a second wave starts) were the slowest at
    // every row count.
    if ((wide_weights || (layer_norm && p.block == 512)) && p.block <= 512 && p.rpb == 1) {
      const int64_t cap = (int64_t)num_cus * (p.block == 512 ? 2 : 3);
      if (nrb <= cap * 32) grid = cap;
    }
  }
  if (oc == OC_NORM_FWD && p.resident && p.exact_depth > 0) {
    const int xi = norm_fwd_exact_index(esize, packs, M, num_cus);
    grid = (int64_t)num_cus * kNormFwdExact[xi].bpc;
  }
  // Rows whose weights are not held gain nothing from a workgroup that walks
  // several rows: one workgroup a row (8192 rows of 40960 bf16: LayerNorm 253 ->
  // 243 us, with fp32 weights 270 -> 254 us, RMSNorm 235 -> 227 us).
  if (oc == OC_NORM_FWD && p.resident && ov.bpc == 0 &&
      !norm_fwd_holds_weights(esize, wide_weights ? 4 : esize, p.G, p.V, p.fast, !layer_norm,
                              fused_add))
    grid = nrb;
  if (!p.resident) p.window = false;
  // windowed rows: 1024 threads a compute unit, all resident at once, so that a
  // workgroup loads its shifted weights once for all its rows (fp16 [8192, 4097]
  // LayerNorm: 4 workgroups of 256 a compute unit 34.6 us, 2: 45.9, 8: 40.0, one row a
  // workgroup 52.3; [8192, 8193] on 512 threads: 2 a compute unit 61.0 us, 1: 83.9, 4: 69.5)
  if (p.window && ov.bpc == 0) grid = (int64_t)num_cus * (1024 / p.block);
  if (grid > nrb) grid = nrb;
  if (grid > 0x7fffffff) grid = 0x7fffffff;
  if (grid < 1) grid = 1;
  // (the kernel takes the window from its lanes: the two must agree)
  if (p.resident && oc == OC_NORM_FWD && p.window != norm_row_window(esize, p.G, p.fast)) return -5;
  // windowed rows: a workgroup that walks several row blocks strides by a multiple of
  // 8 rows, so that every row of a lane group has the same window head
  if (p.window && grid < nrb && grid % 8 != 0) grid = grid > 8 ? grid - grid % 8 : (nrb < 8 ? nrb : 8);
  p.grid = grid;
  p.partial_rows = 0;
  if (oc == OC_NORM_BWD && want_cols) {
    // resident: one partial row per workgroup; streaming: a separate column-sum
    // kernel whose grid.y is the partial-row count.
    if (p.resident) {
      p.partial_rows = grid;
    } else {
      // enough partial rows that the column-sum grid (256 lanes, one pack each,
      // across; partial rows down) gives a compute unit about four workgroups
      const int64_t across = (packs + 255) / 256;
      int64_t pr = (4 * (int64_t)num_cus + across - 1) / across;
      if (pr > 64) pr = 64;
      // rows so long that the columns alone give every compute unit two workgroups: one
      // partial row, which the column-sum kernels then write as dgamma / dbeta themselves
      // (no second stage; bf16 LayerNorm backward [2, 1310720] 25.8 -> 13.9 us, [16, 1048576] 40.7 ->
      // 34.1 us)
      if (across >= 2 * (int64_t)num_cus) pr = 1;
      if (pr > M) pr = M;
      p.partial_rows = pr < 1 ? 1 : pr;
    }
  }
  // (the column sums alone run on the layout they run on beside dX: the same bits)
  if ((oc == OC_NORM_FWD || oc == OC_NORM_BWD) && p.resident && p.exact_depth == 0 && !fused_add &&
      !force_general && !p.forced && ov.bpc == 0 &&
      !(oc == OC_NORM_BWD && p.fast && norm_bwd_exact_index(esize, packs, M, layer_norm, wide_weights, false) >= 0))
    p.waves = norm_waves_layout(oc == OC_NORM_BWD, esize, M, N, p.fast, layer_norm, wide_weights, p.partial_rows,
                                num_cus);
  // Backward of few rows beyond the registers, dX and column sums: two launches, no partial rows
  // (norm_bwd_few_rows_kernel).  Wavefronts that share a piece of 64 packs of columns, a part of the rows each:
  // as many as leave every compute unit one workgroup (us, 1 / 2 / 4 / 8 of them: bf16 LayerNorm [28, 70144] 28.0 /
  // 18.8 / 13.5 / 10.4, [16, 200000] 20.6 / 15.1 / 12.1 / 14.7, [48, 385536] 50.8 / 40.1 / 44.3 / 44.9).  Against the
  // four launches, or teams of workgroups and a second stage: [28, 70144] 27.9 -> 10.4, [3, 87936] 12.5 -> 7.4, [8,
  // 292096] 25.5 -> 11.9, [64, 60000] 28.5 -> 16.9, [57, 156800] 34.2 -> 27.4.  The other sides of the lines: [251,
  // 51584] 37.1 / 46.0, [100, 400000] 67 / 82, and rows that alone give every compute unit two workgroups, which
  // the column-sum kernels serve without partial rows as well ([3, 1451648] 16.6 / 21.4, [7, 1413504] 29.3 / 32.3).
  // An RMSNorm of whole packs keeps its teams, which have half the sums to exchange and to add, from half as many rows
  // and bytes on ([24, 194976] 23.6 -> 14.7, but [75, 162328] 28.3 / 33.8, [108, 38472] 20.6 / 24.2, [19, 659856] 27.5
  // / 30.8), a LayerNorm that has teams from 16 (float32), 21 (float32 weights) and 24 MB a tensor on, where dY and X
  // no longer come out of the L2s, 32 MB together, when they are read again: time over that of the teams, float32 [40,
  // 112000] 17 MB 0.91, [48, 112000] 20 MB 1.06, [48, 160000] 29 MB 1.37; bf16 with float32 weights [64, 160000] 20 MB
  // 0.92, [80, 160000] 24 MB 1.11; bf16 [80, 160000] 24 MB 1.02, [48, 320000] 29 MB 1.07; rows without teams, float32
  // [24, 320000] 29 MB 0.95, [80, 79997] 24 MB 0.78.  Such a LayerNorm call that teams cannot take (captured, dX over an
  // input, no slot) keeps the two launches, the plan has both (dX over dY, four launches / these: float32 [48, 112000]
  // 32.7 / 26.3, [48, 160000] 38.4 / 34.1, bf16 [48, 320000] 40.2 / 37.0, [100, 150000] 42.0 / 43.2).
  const int64_t few_part = layer_norm || !p.fast ? 1 : 2;
  const int64_t few_team_bytes = layer_norm ? (int64_t)(esize == 4 ? 16 : wide_weights ? 21 : 24) << 20 : kFewRowsBytes;
  if (oc == OC_NORM_BWD && !p.resident && want_cols && want_dx && p.partial_rows > 1 && M * few_part <= kFewRowsMax &&
      M * packs * 16 * few_part <= kFewRowsBytes && ov.G == 0 && ov.V == 0 && ov.bpc == 0 && ov.block == 0) {
    const int64_t pieces = (packs + 63) / 64;
    p.few_waves = kFewRowsWaves;
    while (p.few_waves > 1 && pieces * p.few_waves > kFewRowsWaves * (int64_t)num_cus) p.few_waves /= 2;
    // (chunks of whole strides, about four a compute unit; their sums fit the memory of the partial rows, which
    // this call has none of: at most a 16th of one)
    const int64_t most = (4 * (int64_t)num_cus + M - 1) / M;
    const int64_t cp = ((packs + most - 1) / most + kStreamBlock - 1) / kStreamBlock * kStreamBlock;
    p.few_chunk_packs = cp;
    p.few_chunks = (int)((packs + cp - 1) / cp);
  }
  // Rows beyond the registers, and too few of them to give every compute unit a
  // workgroup (the regime of the reference's split-row kernels, Norm.h:632-812):
  // cut each row into chunks so that about four workgroups per compute unit
  // exist.  The partial sums of a row cross workgroups through memory, in a fixed
  // order, between two launches.
  if ((oc == OC_NORM_FWD || oc == OC_NORM_BWD) && !p.resident) {
    const int64_t min_chunk = (int64_t)kSplitMinStrides * kStreamBlock;
    int64_t want = 1;
    if (ov.G < 0 && ov.V > 0)
      want = ov.V;
    else if (M > 0 && M < 2 * (int64_t)num_cus)
      want = (4 * (int64_t)num_cus + M - 1) / M;
    if (want > kSplitMaxChunks) want = kSplitMaxChunks;
    if (want > 1) {
      int64_t cp = (packs + want - 1) / want;
      cp = (cp + kStreamBlock - 1) / kStreamBlock * kStreamBlock;
      if (cp < min_chunk && !(ov.G < 0 && ov.V > 0)) cp = min_chunk;
      int64_t chunks = (packs + cp - 1) / cp;
      // a remainder of less than one workgroup stride joins the chunk before it, so
      // every chunk holds at least kStreamBlock packs (the forward keeps a chunk's
      // partial sums in the first bytes of the chunk's own output)
      if (chunks > 1 && packs - (chunks - 1) * cp < kStreamBlock) --chunks;
      if (chunks > 1) {
        p.split = (int)chunks;
        p.chunk_packs = cp;
      }
    }
  }
  // Forward rows beyond one workgroup's registers: a team of workgroups holds the
  // row (one pass over X).  As few workgroups a row as hold it with 16 packs a lane,
  // then as many teams as there are rows and compute units, and a row spread over
  // all the workgroups its team can have (down to one stride of 1024 packs each).
  // (GroupNorm forward slabs likewise; the caller takes the team only where the channels
  // are whole packs)
  // (also rows that one workgroup still holds, 16 packs a lane on 1024 lanes, when there are
  // too few of them for the compute units: bf16 [128, 131072] LayerNorm 17.4 -> 13.8 us, fp32
  // [128, 65536] 19.2 -> 13.3 us; from 8192 packs down the resident kernel is as fast or faster,
  // its 4-6 us against the team's 6-8)
  const bool few_rows = oc == OC_NORM_FWD && p.resident && 2 * M <= num_cus &&
                        packs >= (int64_t)kMaxG * kMaxV;
  if ((oc == OC_NORM_FWD || oc == OC_GROUP_FWD) && (!p.resident || few_rows) && p.fast && !fused_add &&
      ov.G == 0 && ov.V == 0 && ov.bpc == 0 && ov.block == 0) {
    const int64_t cus = num_cus * kTeamPerCu < kTeamMaxWorkgroups ? num_cus * kTeamPerCu : kTeamMaxWorkgroups;
    const int64_t per_wg = (int64_t)kTeamBlock * kTeamMaxV;
    const int64_t team_min = (packs + per_wg - 1) / per_wg;
    int64_t teams = team_min <= cus ? cus / team_min : 0;
    if (teams > M) teams = M;
    // Fewer than 8 teams run their load, wait and store phases nearly in step, and
    // the wait (about 8 us a round) is not hidden by other teams: bf16 [128, 9834496]
    // (3 teams of 85, 43 rounds) took 1740 us against 1500 us for the two-pass kernel
    // whose second pass comes out of the memory-side cache; 8 teams ([8, 4194304], one
    // round) 35.1 against 40.5 us, 64 teams ([512, 401408], 8 rounds) 177 against 196 us.
    // Fewer than 8 rows, all at once: teams of at most an eighth of the machine, whose exchange is a single
    // round trip ([2, 1310720] 10.7 us in three launches, 12.0 on teams of 256 workgroups, 9.4 on 64; [7, 1413504]
    // 24.1, 13.4; [3, 87936] 10.3, 6.9; and one launch, where three bound such a call: [4, 506752] with its
    // backward 26.6 -> 20.0 us).  More than eight packs a lane for one or two rows leave too much of the machine
    // idle: [1, 4000000] 12.7, 16.8, but [5, 3000000] 25.6, 24.7.
    // (GroupNorm slabs have no split-row kernels to fall back on: with fewer slabs than 8
    // teams, all at once, the alternative is one workgroup a slab)
    const int64_t strides = (packs + kTeamBlock - 1) / kTeamBlock, eighth = cus / kTeamMinTeams;
    const bool at_once = teams >= 1 && teams == M;
    const bool small_teams = oc == OC_NORM_FWD && !p.resident && at_once && M < kTeamMinTeams &&
                             strides <= eighth * (M < 3 ? kTeamMaxV / 2 : kTeamMaxV);
    if (teams >= kTeamMinTeams || ((oc == OC_GROUP_FWD || few_rows) && at_once) || small_teams) {
      // a chunk is a whole number of workgroup strides, exactly the packs a lane the
      // kernel is compiled for: every workgroup but a row's last runs straight-line code
      auto packs_a_lane = [&](int64_t n) {
        int64_t most = cus / n < strides ? cus / n : strides;
        if (small_teams && most > eighth) most = eighth;
        return (strides + most - 1) / most;
      };
      // Two or three rounds, the last of them not full: as many teams as give every round the same rows, each
      // row over more workgroups, where that is less work in a row.  A last round of at most half the teams
      // takes about three tenths of a round's time (two tenths beside float32 weights of 16-bit rows), its
      // workgroups having a compute unit's bandwidth each; a fuller one nine (norm forward, bf16 LayerNorm:
      // [140, 216576] 128 teams of 4 -> 70 of 7 35.3 -> 28.5 us, [33, 1103488] 44.8 -> 36.5, [256, 188416] 52.3
      // -> 42.5, [358, 163840] 58.5 -> 52.2, [64, 1345664] 92.0 -> 80.8; 0.90 of the time over 900 shapes that the
      // rule takes, at worst 1.07).  The other sides of the lines: more packs than that ([389, 188800] 66.9
      // -> 74.5, [112, 686560] 3 x 16 -> 3 x 13 packs 68 -> 77, fp16 with fp32 weights [241, 133440] 35 -> 40); four
      // rounds or more, where the last leaves little idle ([216, 468864] 84.5 -> 89.0, [110, 1526656] 143 -> 181);
      // less than 15 of 16 workgroups used in every round where the last one was a quarter full or more ([148,
      // 291328] 39.4 -> 44.1).  And the weights: workgroup b runs on XCD b % 8, which so meets every gcd(team,
      // 8)-th chunk of gamma and beta; beyond three quarters of its L2 they come from further out every round
      // ([71, 1284480] teams of 20 -> 21 79.7 -> 94.4; fp16 with fp32 weights [20, 2036640] 32 -> 50 41 -> 62).
      const int64_t rounds = (M + teams - 1) / teams;
      if (oc == OC_NORM_FWD && (rounds == 2 || rounds == 3)) {
        const int64_t even = (M + rounds - 1) / rounds, ve = packs_a_lane(even), members = (strides + ve - 1) / ve;
        const int64_t last = M - (rounds - 1) * teams, tenths = 2 * last > teams ? 9 : wide_weights ? 2 : 3;
        const bool less = 10 * rounds * ve <= packs_a_lane(teams) * (10 * (rounds - 1) + tenths);
        const bool fills = 16 * even * members >= 15 * cus || 4 * last < teams;
        const int64_t shared = members % 8 == 0 ? 8 : members % 4 == 0 ? 4 : members % 2 == 0 ? 2 : 1;
        const int64_t weights = (layer_norm || shared == 1 ? 2 : 1) * (wide_weights ? 32 : 16) * packs;
        if (even >= kTeamMinTeams && less && fills && weights <= shared * (3 << 20)) teams = even;
      }
      const int64_t v = packs_a_lane(teams);
      const int64_t team = (strides + v - 1) / v;
      p.team = (int)team;
      p.team_v = (int)v;
      p.team_chunk_packs = v * kTeamBlock;
      p.team_grid = teams * team;
    }
  }
  // Forward rows too long for at least eight such teams (beyond 256 / 8 * 16 * 512 packs),
  // many of them, weights no wider than the rows: one team over the machine, one workgroup a
  // compute unit, kTeamFwdLongPacks packs a lane, three rows in flight a workgroup and gamma /
  // beta held for the whole call (norm_fwd_rows_team_kernel).
  // (override G = -1 with block = 1: whatever the rounds and the other teams, for tests)
  const bool team_rows_forced = ov.G == -1 && ov.V == 0 && ov.block == 1 && ov.bpc == 0;
  if (oc == OC_NORM_FWD && !p.resident && p.fast && !fused_add && !wide_weights &&
      ((ov.G == 0 && ov.V == 0 && ov.bpc == 0 && ov.block == 0 && p.team == 0) || team_rows_forced)) {
    const int64_t cus = num_cus < kTeamMaxWorkgroups ? num_cus : kTeamMaxWorkgroups;
    const int64_t chunk = (int64_t)kTeamFwdLongPacks * kTeamBlock;
    const int64_t team = (packs + chunk - 1) / chunk;
    if (team >= 2 && team <= cus) {
      int64_t teams = cus / team;
      if (teams > M) teams = M;
      const bool rounds_ok = M >= kTeamFwdMinRounds * teams;
      const bool full_ok = 5 * packs >= 4 * team * chunk;
      if (teams >= 1 && ((rounds_ok && full_ok) || team_rows_forced)) {
        p.team = (int)team;
        p.team_v = kTeamFwdLongPacks;
        p.team_r = 1;
        p.team_chunk_packs = chunk;
        p.team_grid = teams * team;
      }
    }
  }
  // Backward rows beyond one workgroup's registers (whole packs, dX wanted, no residual
  // gradient): teams of workgroups hold kTeamBwdRows rows at a time, kTeamBwdPacks strides of
  // packs a workgroup, dY and X read once (norm_bwd_team_kernel).
  // (override G = -1 with block = 1: the team launch whatever the rounds, for tests)
  const bool team_bwd_forced = ov.G == -1 && ov.V == 0 && ov.block == 1 && ov.bpc == 0;
  if (oc == OC_NORM_BWD && !p.resident && p.fast && !fused_add && want_dx &&
      (p.few_waves == 0 || M * packs * 16 > few_team_bytes) &&
      ((ov.G == 0 && ov.V == 0 && ov.bpc == 0 && ov.block == 0) || team_bwd_forced)) {
    const NormBwdTeam t = norm_bwd_team(M, packs, p.fast, layer_norm, num_cus);
    if (t.teams >= 1 && (t.rounds_ok || team_bwd_forced)) {
      p.team = (int)t.team;
      p.team_v = kTeamBwdPacks;
      p.team_chunk_packs = (int64_t)kTeamBwdPacks * kTeamBlock;
      p.team_grid = t.teams * t.team;
      p.team_partial_rows = want_cols ? t.teams : 0;
    }
  }
  // Softmax forward / backward of few, very long rows: one workgroup a row
  // would leave most compute units idle, so each row is held by a team of workgroups
  // (softmax_fwd_team_kernel / softmax_bwd_team_kernel): as few workgroups a row as hold it
  // with 16 (backward: 8 of each tensor) packs a lane, then as many teams as there are rows
  // and room, and a row spread over all the workgroups its team can have.  More rows than
  // teams run in rounds; even then, and with few teams whose waits nothing hides, one
  // workgroup a row is several times slower (fp32 [2, 16777216]: 4800 us).
  // (Before teams and held rows the ragged ones went through softmax_*_stream_kernel, bf16 us: forward [32, 36002] 7.9,
  // [64, 60004] 11.5, [16, 110001] 17.7 -> 7.4; backward [32, 32769] 7.4, [100, 60004] 10.4, [128, 80001] 19.9 -> 16.2.)
  const int64_t row_packs = (N + E - 1) / E;
  if (softmax && !force_general && !masked && ov.G == 0 && ov.V == 0 && ov.bpc == 0 && ov.block == 0 &&
      2 * M <= num_cus && row_packs >= kSoftmaxTeamMinPacks) {
    const int64_t cus = num_cus * kTeamPerCu < kTeamMaxWorkgroups ? num_cus * kTeamPerCu : kTeamMaxWorkgroups;
    const int max_v = oc == OC_SOFTMAX_FWD ? kTeamMaxV : kSoftmaxBwdTeamMaxV;
    const int64_t per_wg = (int64_t)kTeamBlock * max_v;
    const int64_t team_min = (row_packs + per_wg - 1) / per_wg;
    int64_t teams = team_min <= cus ? cus / team_min : 0;
    if (teams > M) teams = M;
    if (teams >= 1) {
      int64_t team_max = cus / teams;
      const int64_t strides = (row_packs + kTeamBlock - 1) / kTeamBlock;
      if (team_max > strides) team_max = strides;
      const int64_t v = (strides + team_max - 1) / team_max;
      const int64_t team = (strides + v - 1) / v;
      if (team >= 2) {
        p.team = (int)team;
        p.team_v = (int)v;
        p.team_chunk_packs = v * kTeamBlock;
        p.team_grid = teams * team;
      }
    }
  }
  if (softmax && !p.resident && !p.fast && !masked && !p.forced && ov.G == 0) {
    const int64_t held = (N + 2 * (E - 1)) / E;  // packs of the window, whatever its head
    const bool on_half = oc == OC_SOFTMAX_FWD && softmax_tail_half_lanes(held, M, num_cus);
    const int64_t v = (held + (on_half ? kMaxG / 2 : kMaxG) - 1) / (on_half ? kMaxG / 2 : kMaxG);
    const int most = oc == OC_SOFTMAX_FWD ? max_v_of(oc, esize) : kGradResidentMaxV;
    if (v >= kSoftmaxTailMinV && v <= most) {
      p.tail_v = (int)v;
      p.tail_packs = (int)held;
      p.tail_cus = num_cus;
      p.tail_g = on_half ? kMaxG / 2 : kMaxG;
    }
  }
  if (oc == OC_SOFTMAX_BWD && !p.resident && p.fast && ov.G == 0 &&
      packs <= (int64_t)kMaxG * kGradResidentMaxV)
    p.grad_resident = true;
  *out = p;
  return 0;
}

// Calls of few softmax rows of kSoftmaxTeamMinPacks packs or more: whether one workgroup a row (`whole`: whole packs,
// in registers; otherwise held, see softmax_tail_serves()) is faster than teams, whose exchange is longer than its way
// through a short row and shorter than through a long one.  The more rows, the longer they may be: teams get smaller
// and their loads are no longer the only ones under way.  Teams of four and less (more rows than 2 / 5 of the compute
// units) gain last.  Measured on the same buffers:
//   whole packs, us, one workgroup / team, bf16 forward [30, 32768] 5.7 / 5.5, [48, 32768] 5.8 / 6.4, [48, 36032] 7.2 /
//     6.6, [64, 40000] 7.5 / 7.6, [64, 45056] 8.2 / 7.6, [100, 50048] 9.4 / 8.6, [128, 50048] 9.5 / 9.6, [128, 65536]
//     10.0 / 9.8; float32 forward [64, 20480] 6.5 / 7.3, [64, 22528] 8.1 / 7.4; bf16 backward [8, 32768] 3.5 / 4.8,
//     [48, 33792] 6.4 / 6.1, [64, 36032] 6.7 / 7.0, [64, 45056] 7.6 / 7.1, [128, 50048] 8.9 / 9.6, [128, 60032] 11.0 /
//     9.9
//   ragged, time over that of the two passes which served such rows before, one workgroup / team, bf16 at 64 rows:
//     forward of 5 packs a lane of 1024 0.88 / 0.96, of 8 0.81 / 0.73; backward 5 0.78 / 1.01, 8 0.78 / 0.87;
//     log_softmax backward 10 0.70 / 0.91, 16 0.67 / 0.59.  At 128 rows: forward 10 0.76 / 0.89, 18 0.68 / 0.68;
//     backward 6 0.92 / 1.24, 8 0.79 / 1.03; log_softmax backward 7 0.73 / 1.10, 16 0.77 / 0.88
inline bool softmax_one_workgroup(bool backward, bool is_log, bool whole, int esize, int64_t M, int64_t packs,
                                  int num_cus) {
  const int64_t m = M * 256 / num_cus;
  const bool small_teams = 5 * M > 2 * (int64_t)num_cus;
  const int64_t from = kSoftmaxTeamMinPacks;
  auto least = [](int64_t a, int64_t b) { return a < b ? a : b; };
  if (whole) {
    if (!backward && esize == 4) return packs <= 5120;
    if (packs <= from) return backward || m >= 40;
    return packs <= (small_teams ? 7168 : m >= 60 ? 5120 : 0);
  }
  if (!backward) {
    if (esize == 4) return packs <= from + (is_log ? least(90 * m - 300, 3072) : 32 * (m - 32));
    return packs <= (small_teams ? 17 * kMaxG : from + (is_log ? 90 * m : 50 * (m - 8)));
  }
  if (!is_log) return esize == 4 || packs <= from + 100 * m;
  if (esize == 4) return packs <= from + least(256 * m, 3072);
  return small_teams || packs <= least(from + 160 * m, 12000);
}

// Whether a softmax row of no whole number of packs is held by one workgroup (p.tail_v) rather than read twice.
// widened: a float32 output of 16-bit rows.  The two passes, two workgroups a compute unit at different places of their
// rows, keep (us, two passes / held; measured over 200 to 8192 rows, three fills of every pack count):
inline bool softmax_tail_serves(const Plan& p, bool backward, bool is_log, bool widened, int esize, int64_t M,
                                int64_t N) {
  const int v = p.tail_v;
  const int64_t cus = p.tail_cus, bytes = M * N * esize;
  if (v == 0) return false;
  if (backward) {
    if (!is_log && v > kSoftmaxBwdHoldMaxV) return false;
    // 16-bit rows that leave much of 4 or 5 packs a lane empty while a second pass comes out of the cache: both tensors
    // in registers are one workgroup a compute unit ([2000, 29483] 62.1 / 66.9, [2000, 31939] 66.7 / 70.2, but [2000,
    // 32515] 80.3 / 70.7, [300, 29483] 12.7 / 11.9; float32 gains there too: [2000, 16791] 88.4 / 69.6)
    if (!is_log && esize == 2 && M > 2 * cus && 2 * bytes <= kSoftmaxCachedBytes &&
        ((v == 4 && p.tail_packs <= 4032) || (v == 5 && p.tail_packs <= 4704)))
      return false;
    // float32 rows whose last lane round is nearly empty, many of them, grad alone held: [4096, 16791] 139 / 149,
    // [3000, 20887] 130 / 135, with a float16 gradient 102 / 111; but [4096, 18839] 0.96 of the time
    if (is_log && esize == 4 && v <= 7 && M > 7 * cus && p.tail_packs <= (v - 1) * kMaxG + 320) return false;
    return true;
  }
  if (v == 17 || v == 19) return false;  // (not built: 0.91 to 1.12 of the two passes, worst at 300 rows)
  if (widened)
    // few rows, whose stores go out at the kernel's end ([130, 53243] 19.3 / 20.6, [200, 36859] 15.8 / 17.2, but [200,
    // 53243] 25.7 / 22.7, [300, 36859] 33.7 / 27.7; log_softmax gains everywhere)
    return is_log || !((4 * M <= 3 * cus && p.tail_packs > 4096) ||
                       (M <= cus && p.tail_packs > 3500 && p.tail_packs <= 4800));
  // log_softmax, whose second pass is short, out of the cache: 16-bit [2000, 48323] 65.5 / 70.2, [2000, 54875] 73.6 /
  // 80.5 (at 1500 rows 1.0 to 1.06 of the time), float32 [3000, 18431] 71.1 / 76.7; but out of it [3000, 53243] 123 /
  // 115, float32 [4096, 18431] 113 / 103
  if (is_log && p.tail_g == kMaxG && M > 4 * cus &&
      (esize == 2 ? v >= 6 && v <= 10 && bytes <= kSoftmaxCachedBytes : v <= 6 && bytes <= kSoftmaxCachedBytes * 7 / 8))
    return false;
  // 1024 lanes, one workgroup a compute unit.  A few rows more than compute units are a second round: 16-bit of 20
  // packs a lane [300, 159739] 57.9 / 58.4, log_softmax 51.7 / 55.5, float32 of 10 to 16 [300, 65123] 45.3 / 48.3 (at
  // 400 rows 0.94 to 1.03 of the time, at 200 0.8)
  if (p.tail_g == kMaxG && M > cus && 2 * M <= 3 * cus && (esize == 2 ? v == 20 : v >= 10)) return false;
  // float32 of 10 to 12 packs, the least that fill it: [1000, 37271] 66.0 / 69.2, [2000, 37271] 129 / 135, log_softmax
  // [700, 45463] 55.4 / 58.2, but [2000, 38911] 131 / 127, of 11 packs [2000, 43007] 150 / 147
  if (p.tail_g == kMaxG && esize == 4 && M > cus &&
      ((v == 10 && !is_log) || (v <= 12 && v >= 10 && M <= 3 * cus)))
    return false;
  return true;
}

// (the held backward reads y through grad's window)
inline bool softmax_tail_aligned(const void* grad, const void* y) {
  return (((uintptr_t)grad ^ (uintptr_t)y) & 15u) == 0;
}

// Whether a softmax call without a mask, with its output apart from its inputs, goes to teams of workgroups (p.team).
// held: nothing but softmax_tail_serves() is in the way of the held form.
inline bool softmax_team_serves(const Plan& p, bool backward, bool is_log, bool widened, int esize, int64_t M,
                                int64_t N, int num_cus, bool held = true) {
  if (p.team == 0 || widened) return p.team > 0;
  const bool one = p.resident || (held && softmax_tail_serves(p, backward, is_log, widened, esize, M, N));
  const int64_t E = 16 / esize;
  return !(one && softmax_one_workgroup(backward, is_log, p.fast, esize, M, (N + E - 1) / E, num_cus));
}

// GroupNorm backward of slabs beyond the registers held by teams of workgroups, one workgroup or
// several (`wpc`) a channel: gn_bwd_team_kernel (v packs a lane and tensor), or the one that has a
// team's next slab on its way meanwhile, gn_bwd_team_ahead_kernel (ahead; v = kGnTeamAheadPacks).
// team 0: not this shape.
struct GnBwdTeam {
  int team = 0, wpc = 0, v = 0;
  bool ahead = false;
  int64_t grid = 0;
};

// rows slabs of D channels of cp packs each.  As few packs a lane (4 or 8 of each tensor) as hold a
// channel on one workgroup, else 8 and several workgroups a channel.
inline GnBwdTeam gn_bwd_team(int64_t rows, int64_t D, int64_t cp, int esize, int num_cus) {
  if (num_cus <= 0) num_cus = 256;
  const int64_t wgs = (int64_t)num_cus * kTeamPerCu < kTeamMaxWorkgroups
                          ? (int64_t)num_cus * kTeamPerCu
                          : (int64_t)kTeamMaxWorkgroups;
  GnBwdTeam none, t;
  // (channels of at most 1024 packs -- one or two packs a lane -- move too little between two
  // exchanges: bf16 [2, 2048, 64, 64] in 32 groups, 8 rounds of 8 KB a workgroup and tensor, 56.6
  // us against 35.0 us for the two launches)
  if (rows < 1 || D < 1 || cp <= 2 * kTeamBlock) return none;
  auto layout = [&](int v) {
    const int64_t chunk = (int64_t)v * kTeamBlock;
    const int64_t wpc = (cp + chunk - 1) / chunk, team = D * wpc;
    GnBwdTeam l;
    if (team < 2 || team > wgs) return l;
    const int64_t teams = wgs / team < rows ? wgs / team : rows;
    l.team = (int)team;
    l.wpc = (int)wpc;
    l.v = v;
    l.grid = teams * team;
    return l;
  };
  t = layout(cp <= 4 * kTeamBlock ? 4 : 8);
  if (t.team == 0) return none;
  // A team that works through several slabs with the next one on its way.  Where four packs a lane
  // hold a channel that costs nothing, and any second slab gains (bf16, 32 groups, us, without /
  // with: [4, 256, 128, 128], two slabs a team, 26.8 / 24.5; [7, 512, 120, 120] 77.3 / 67.6).
  // Where eight did, half as many slabs are held at a time and there are twice as many exchanges:
  // from four slabs a team, on a grid that leaves no more than a sixteenth of the machine idle
  // ([1, 512, 416, 416], 352 workgroups, 122 / 150; [1, 256, 448, 448], 416, 75.6 / 81.1), and only
  // if a channel fits four packs a lane clearly better ([2, 512, 200, 200], three workgroups a
  // channel for two, 69.6 / 63.4; fp32 [8, 128, 136, 136] 62.0 / 55.0; [4, 512, 152, 152], four
  // for two, 65.3 / 75.5), or fills its workgroups (fp32 [4, 256, 256, 256] 154.6 / 144.3, bf16
  // [1, 256, 512, 512] 87.6 / 86.9; [7, 128, 248, 248], 94 % filled, 67.6 / 71.4), or nearly does
  // over eight slabs a team ([1, 512, 496, 496] 173.9 / 166.6; four: [1, 256, 496, 496] 85.4 / 87.2).
  // fp32, half the arithmetic a pack, gains from four slabs if it nearly does ([1, 512, 248, 248]
  // 80.4 / 76.3, [1, 384, 232, 232] 60.3 / 55.0; [7, 384, 104, 104], two thirds filled, 75.9 / 84.9).
  const int64_t teams = t.grid / t.team;
  if (t.v == kGnTeamAheadPacks) {
    t.ahead = rows > teams;
    return t;
  }
  const GnBwdTeam h = layout(kGnTeamAheadPacks);
  if (h.team == 0 || rows <= 3 * teams || h.grid * 16 < wgs * 15) return t;
  const int64_t slots = (int64_t)h.wpc * kGnTeamAheadPacks * kTeamBlock;
  if (3 * h.wpc <= 5 * t.wpc || cp * 100 >= slots * 98 ||
      (cp * 16 >= slots * 15 && (esize == 4 || rows > 7 * teams))) {
    t = h;
    t.ahead = true;
  }
  return t;
}

// Whether the teams of gn_bwd_team_kernel write dgamma / dbeta themselves: a team then takes whole groups, all
// samples of one after the other, which must not make more rounds than slabs dealt out one by one, nor rounds
// of more teams: a last round of at most half the teams is a cheap one, and whole groups put all of a group's
// samples behind it (fp16 [2, 128, 560, 560] in 64 groups, 25 teams, 107 -> 116 us, [2, 256, 296, 296] in 8, 5
// teams, 69 -> 73, bf16 [2, 256, 304, 304] in 64, 42 teams, 66 -> 70; the shapes taken 0.90 to 1.005 of the time).
// (The kernel that has the next slab on its way lost what it gained: [4, 256, 128, 128] 24.0 -> 25.3 us.)
inline bool gn_team_sums_columns(int64_t rows, int64_t groups, int64_t teams) {
  const int64_t samples = rows / groups, rounds = (rows + teams - 1) / teams;
  if (teams > groups || samples > 0xffffff || (groups + teams - 1) / teams * samples > rounds) return false;
  return samples == 1 || 2 * (rows - (rounds - 1) * teams) > teams;
}

// ---- softmax over a non-innermost dimension: [outer, D, inner] ----------------
//
// A group of TX * TY threads owns one tile: TX lanes along `inner` (one 16-byte
// pack each) by TY threads along D, each holding V packs, so the registers
// cover D <= TY * V rows.  The rule: at most 8 packs a lane (4 for the 16-bit
// backward of D <= 32), TY = the power of two that then covers D, V = ceil(D / TY), and TX = as many lanes
// as a row of `inner` has packs, capped so that a group is one wavefront where
// that leaves at least 8 lanes (128-byte segments) per row, and 256 threads
// otherwise.  A group of one wavefront reduces with shuffles alone.  D beyond
// 64 rows x 8 packs x 4 lanes takes the multi-pass kernel.  Strips of whole packs are
// held by teams of workgroups instead where the call allows it and they are faster.
struct StridedPlan {
  bool resident = true;
  bool fast = true;  // inner % E == 0
  int tx_log2 = 0, ty_log2 = 0, V = 0, block = 0;
  int64_t grid = 0;
  // multi-pass kernels with too few tiles for the machine: the D rows are cut into
  // `chunks` chunks of `chunk_rows` rows, one workgroup each (0 or 1: not split)
  int chunks = 0, chunk_rows = 0;
  // strips held by teams of workgroups, two a compute unit (softmax_strided_team.hpp); team 0: not
  // this call.  team_grid = teams * team workgroups, team_tx_log2 = log2 of the packs a strip is
  // wide, team_v = packs a lane
  int team = 0, team_v = 0, team_tx_log2 = 0;
  int64_t team_grid = 0;
  // the same strips by workgroups that have a compute unit to themselves (strided_large_team());
  // large_team 0: two a compute unit
  int large_team = 0, large_v = 0, large_tx_log2 = 0;
  int64_t large_grid = 0;
  // Workgroups of the team a call by teams runs on (0: no teams): one waits for nobody, more exchange.
  int team_size() const { return large_team > 0 ? large_team : team; }
};

// The packs a lane the strided team kernels are built for: the forward holds one tensor, the
// backward two.
constexpr int kStridedTeamV[2][10] = {{1, 2, 3, 4, 6, 8, 10, 12, 14, 16}, {1, 2, 3, 4, 5, 6, 7, 8}};
constexpr int kStridedLargeV[2][4] = {{40, 48, 56, 64}, {20, 24, 28, 32}};
constexpr int strided_team_max_v(bool backward) { return backward ? 8 : 16; }
constexpr int strided_large_max_v(bool backward) { return backward ? 32 : 64; }
// Workgroups of an instance a compute unit holds, and the packs a lane keeps in LDS: up to 48 packs
// of a lane (the backward 24 of each tensor) fit 256 registers, the rest 16 bytes a thread each.  (Beside
// 16 packs in LDS the forward spills 9 to 11 registers, in bfloat16 beside 8 packs 3, outside the loops over the
// packs.)
constexpr int strided_team_per_cu(bool backward, int v) {
  return v > strided_team_max_v(backward) ? 1 : kTeamPerCu;
}
constexpr int strided_team_parked(bool backward, int v) {
  return v > (backward ? 24 : 48) ? v - (backward ? 24 : 48) : 0;
}
// Lanes along `inner` at most: 256-byte row segments, or 512-byte ones.
constexpr int kStridedTeamTx = 16;
constexpr int kStridedTeamWideTx = 32;
constexpr int64_t kStridedTeamMinD = 256;
constexpr int64_t kStridedTeamWideMaxD = 4096;

constexpr int kStridedSplitUnroll = 4;  // rows a lane of the split kernels requests at a time

constexpr int kStridedBlock = 256;
constexpr int kStridedMaxV = 8;

inline int log2_of_pow2(int v) {
  int l = 0;
  while ((1 << l) < v) ++l;
  return l;
}

// Strips of tx packs held by teams (large: on workgroups that have a compute unit each): as few workgroups
// a strip as hold its D rows, as many teams as strips and compute units allow, evened out over the rounds;
// then a strip is spread over the workgroups its team can have.
struct StridedTeam {
  int team = 0, v = 0, tx = 0;
  bool capped = false;  // there were workgroups for a larger team
  int64_t rounds = 0, grid = 0;
};
inline StridedTeam strided_team_of(bool backward, int64_t outer, int64_t D, int64_t packs, int esize, int tx,
                                   int num_cus, bool large = false) {
  const int64_t per_cu = large ? 1 : kTeamPerCu, at_most = kTeamMaxWorkgroups / kTeamPerCu * per_cu;
  const int64_t wgs = num_cus * per_cu < at_most ? num_cus * per_cu : at_most;
  // A team is an eighth of the machine at most: larger ones gain nothing, their exchange takes longer (bf16 [1, 8192,
  // 136] forward on 64 workgroups 11.8 us, on 256 27.5).  A large workgroup enters an empty compute unit only, and
  // other launches' workgroups may take any that has room; but what is not a team ends by itself, and team launches of
  // other streams run before or after (TeamOrder).
  // Beside two streams of calls that fill the machine 20 forward / backward calls of [1, 8192, 8192] took 8.7 /
  // 7.7 ms, on two workgroups a compute unit 8.8 / 9.2, and no wait ran out.
  const int64_t most_wgs = wgs / kTeamMinTeams > 0 ? wgs / kTeamMinTeams : 1;
  const int64_t ty = kTeamBlock / tx, vmax = large ? strided_large_max_v(backward) : strided_team_max_v(backward);
  const int64_t need = (D + ty * vmax - 1) / (ty * vmax);
  const int64_t strips = outer * ((packs + tx - 1) / tx);
  StridedTeam t;
  // (byte offsets of a lane inside a workgroup's rows are 32 bits wide; a float32 output of a 16-bit
  // tensor has twice the bytes)
  if (need > most_wgs || ty * vmax * packs * (esize == 2 ? 32 : 16) >= (int64_t(1) << 31)) return t;
  int64_t teams = wgs / need < strips ? wgs / need : strips;
  t.rounds = (strips + teams - 1) / teams;
  teams = (strips + t.rounds - 1) / t.rounds;
  const int64_t most = (D + ty - 1) / ty;
  int64_t team = wgs / teams < most ? wgs / teams : most;
  t.capped = team > most_wgs;
  if (t.capped) team = most_wgs;
  // (one pack a lane on most of the machine: half as many workgroups with two exchange sooner --
  // bf16 [8, 8192, 32] 12.2 -> 10.2 us)
  if (team > most_wgs / 2 && ty * team >= D && 2 * teams * team > wgs) team = (team + 1) / 2;
  // (a float32 forward of at most 16 columns: a column's thread merges its team's pairs one after the
  // other, two exponentials each -- [8, 8192, 16] on 64 workgroups a team 15.2 us, 32 13.1, 16 11.4;
  // not where that makes it more than eight packs a lane: [1, 30000, 16] 14.2, on 16 19.2)
  if (!backward && esize == 4 && tx <= 4 && team > 16 && D <= ty * 16 * 8) team = 16;
  int64_t v = (D + ty * team - 1) / (ty * team);
  auto built = [&](const auto& list) {
    for (int c : list)
      if (c >= v) return c;
    return 0;
  };
  v = large ? built(kStridedLargeV[backward ? 1 : 0]) : built(kStridedTeamV[backward ? 1 : 0]);
  team = (D + ty * v - 1) / (ty * v);
  t.team = (int)team;
  t.v = (int)v;
  t.tx = tx;
  t.grid = teams * team;
  return t;
}

// The strip's width: 16 packs (256-byte segments), fewer where D needs more workgroups than a team
// may have, or where one round of such teams leaves workgroups over (bf16 [1, 8192, 136] 11.8 us
// with 16 packs, 10.4 with 8; backward of [1, 16384, 136] 11.7, 10.1).
// Or 32 packs, half as many strips to exchange ([35, 1000, 1904] forward / backward 77 / 96 us, 16
// packs 95 / 111), but not
//   where a team holds the strips all at once or D needs large teams, whose exchange grows with the
//   columns ([1, 8192, 8192] 77 / 106, 16 packs 71 / 104);
//   where the last strip, mostly past the row, makes more rounds of packs of it ([200, 700, 320],
//   5/8 of two strips: 62 us, 16 packs 54; [200, 257, 800] 62, 41).  Rows that are not whole
//   128-byte lines share a line with either neighbour, which narrow strips read twice as often: there
//   only if the rounds are a third more (backward: over a third; [200, 700, 264] 64 / 70, 16 packs
//   64 / 76; fp32 [200, 1025, 132] backward 98, 103);
//   where 16 packs take one workgroup a strip, nothing to exchange, and no more rounds ([200, 257,
//   512] 35, 16 packs 27; off the lines only short strips: [200, 512, 264] 47, 54).
// One round of workgroups that each hold a strip alone and are too few to fill two thirds of the
// machine ([40, 257, 800] 14.5 us) take 32 packs too (12.4).
inline StridedTeam strided_team(bool backward, int64_t outer, int64_t D, int64_t packs, int esize, int num_cus) {
  const int px = packs >= 64 ? 64 : pow2_ceil(packs);
  int tx = px < kStridedTeamTx ? px : kStridedTeamTx;
  StridedTeam n = strided_team_of(backward, outer, D, packs, esize, tx, num_cus);
  while (tx > 4 && n.team == 0) {
    n = strided_team_of(backward, outer, D, packs, esize, tx /= 2, num_cus);
    // (narrow segments in many rounds lose to the launches without teams: bf16 backward of [1, 30000,
    // 1904], four rounds, 152 us against 124; [8, 30000, 136], three, 91 against 98)
    if (n.rounds > 3) return StridedTeam{};
  }
  if (n.capped && tx > 8 && n.rounds == 1) {
    const StridedTeam h = strided_team_of(backward, outer, D, packs, esize, tx / 2, num_cus);
    if (h.team > 0 && h.rounds == 1) return h;
  }
  if (n.team == 0 || tx < kStridedTeamTx || px <= kStridedTeamTx || D > kStridedTeamWideMaxD) return n;
  if (n.rounds == 1 && !(n.team == 1 && n.grid > kTeamMaxWorkgroups / 2 && 3 * n.grid < 2 * kTeamMaxWorkgroups)) return n;
  const StridedTeam w = strided_team_of(backward, outer, D, packs, esize, kStridedTeamWideTx, num_cus);
  if (w.team == 0) return n;
  const int64_t nc = n.rounds * n.v, wc = w.rounds * w.v;
  const bool lines = packs % 8 == 0;
  if (n.team == 1 && wc >= nc && (lines || n.v <= 10)) return n;
  return (lines ? 8 * wc > 9 * nc : backward ? 3 * wc > 4 * nc : 3 * wc >= 4 * nc) ? n : w;
}

// The same strips held by workgroups that have a compute unit each: 48 packs a lane in registers and up
// to 16 in LDS (the backward 24 and 8 of each tensor) hold twice what two workgroups hold in registers
// alone, so there are half the rounds and a quarter of the members to a team.  Taken where that makes
// fewer rounds of no more than a sixteenth more packs (a workgroup's packs come in coarser steps) and
// the teams it replaces have twelve members or more; below, two workgroups a compute unit that run out
// of step do as well as fewer rounds (us, two a compute unit / one: bf16 forward of [1, 8192, 8192]
// 70.5 / 59.1, [1, 12899, 3872] 58.4 / 50.1, but [50, 954, 920], teams of 5, 50.5 / 59.4 and [6, 820,
// 10296], of 4, 58.3 / 61.1; backward of [1, 8192, 8192] 103.7 / 82.9, [12, 9602, 200] 46.2 / 30.0,
// [92, 2206, 256] 66.2 / 60.5, but [36, 2844, 384] with 4/3 of the packs 48.1 / 51.5).  Rows of an odd
// number of packs, whose 512-byte pieces start off 32 bytes, gain from teams of 24 on (forward of [4,
// 3419, 3912], 16 members, 58.5 / 67.9, of [2, 13960, 1272], 44, 57.0 / 47.6).  A backward whose strips
// then need no exchange and make one round gains whatever the teams were ([6, 323, 10280] 31.8 / 29.3,
// fp32 [4, 325, 7136] 24.7 / 18.4).
// Part of the gain is the wider strip, 32 packs for 16, half as many strips to exchange.  Where the small
// teams have strips of 32 packs as well there is none in the forward (560 shapes of 20 to 600 MB each: bf16
// 0.97 of the time, a quarter of them slower: [48, 3983, 592] 126 / 149, [18, 4088, 2736] 219 / 239; fp32
// 1.03: [47, 3854, 472] 189 / 218), and in the backward only from eight members on (below: bf16 [14, 3068,
// 1336] 85 / 93, fp32 [45, 3068, 488] 177 / 197), in float32 rows of an odd number of packs where it halves the
// rounds (otherwise 0.98 of the time over 68 shapes, 15 of them slower: [9, 4084, 524] 58.6 / 63.5, [53, 3929,
// 236] 143 / 154; where it does 0.91).  Nor in a forward of rows of 16 packs at most, whose strips stay as they
// are: not in float32 ([34, 12457, 60] 52 / 59, [62, 14919, 56] 112 / 123), in 16 bits for a single round only
// (0.91 of the time; two 1.03: bf16 [55, 14117, 120] 98 / 107, [56, 15618, 104] 99 / 108).
// The other part is the lines of 128 bytes that neighbouring strips of other rows share, and that are read
// twice.  Forward rows of whole lines share none: they take large teams in 16 bits, for a single round, with no
// other to be out of step with (0.93 of the time; of several rounds 1.02: bf16 [62, 6587, 256] 90 / 99, [4, 9431,
// 2304] 80 / 84), and never in float32 (one round 1.00, a quarter of 37 shapes slower: [16, 11602, 128] 44.3 /
// 48.5, [2, 5884, 1824] 42.3 / 45.3; several 1.00: [40, 10726, 128] 94 / 107).
// Workgroup b runs on XCD b % 8: in teams of a multiple of eight members the same rows of neighbouring strips, and
// so the lines they share, meet in one L2.  Float32 forward rows of more than 32 packs on such teams gain from
// large ones of several rounds and a multiple of eight members alone (0.96 of the time; other teams 1.02 over 93
// shapes: [14, 6942, 376] 88 / 98; a single round 1.02 over 62: [4, 8964, 632] 50 / 58, [4, 12060, 492] 56 / 60).
// Never a float16 forward with a float32 output (widened): its stores are twice the bytes of its loads and its
// exponentials are the long ones, and with one workgroup a compute unit neither runs under the other's reads
// (560 shapes of 20 to 600 MB, 1.14 times the time: [59, 3360, 192] 73 / 113, [6, 5912, 1536] 100 / 143, [2,
// 13179, 6336] 320 / 389).
inline StridedTeam strided_large_team(bool backward, int64_t outer, int64_t D, int64_t packs, int esize,
                                      const StridedTeam& t, int num_cus, bool widened) {
  if (t.team == 0 || t.rounds < 2 || widened) return StridedTeam{};
  const StridedTeam l = strided_team_of(backward, outer, D, packs, esize,
                                        packs > kStridedTeamTx ? kStridedTeamWideTx : kStridedTeamTx, num_cus, true);
  if (l.team == 0 || l.rounds >= t.rounds || 8 * l.rounds * l.v > 17 * t.rounds * t.v) return StridedTeam{};
  if (l.team == 1) return backward && l.rounds == 1 ? l : StridedTeam{};
  if (t.tx > kStridedTeamTx && (!backward || l.team < 8)) return StridedTeam{};
  if (t.tx > kStridedTeamTx && esize == 4 && packs % 2 != 0 && 2 * l.rounds > t.rounds) return StridedTeam{};
  if (!backward && (packs <= kStridedTeamTx || packs % 8 == 0) && (esize == 4 || l.rounds > 1)) return StridedTeam{};
  if (!backward && esize == 4 && packs > kStridedTeamWideTx && t.team % 8 == 0 && (l.team % 8 != 0 || l.rounds == 1))
    return StridedTeam{};
  return t.team >= (packs % 2 == 0 ? 12 : 24) ? l : StridedTeam{};
}

// Whether teams serve a shape that the one-workgroup tile (TX lanes along `inner`) holds.  D <=
// 256 is the tile's (at D = 200 [20, 200, 4096] 20.5 / 22.5 us, teams 23.2 / 25.5), and so is a
// tile that spans the row or eight lanes of it: one pass, no exchange (bf16 [2000, 512, 16] 14.1
// us, teams 26.3).  Beyond, the tile's segments are 64 bytes: teams where bandwidth counts, from
// about 7 MB (bf16 forward / backward, tile -> teams: [4, 512, 8192] 28.6 / 38.1 -> 16.2 / 19.0
// us, [64, 300, 800] 23.5 / 29.9 -> 15.8 / 25.8; below, [8, 257, 512] 8.0 / 6.8 against 9.0 /
// 7.5); later for a forward whose rows those segments divide (bf16 [200, 320, 64], 8.2 MB, 9.7
// against 10.1; [40, 384, 320], 9.8 MB, 11.3 against 10.4) and for a float32 forward, whose
// arithmetic the tile hides better ([200, 257, 68], 14 MB, 16.5 against 14.9); and a forward of
// such rows never where teams would leave half of their packs empty, a quarter in float32, a
// little more where nothing is exchanged (bf16 [200, 257, 320] 24.4 against 26.6, [40, 257, 576]
// 11.6 against 12.4, but [200, 257, 192], one workgroup a strip, 18.6 against 14.5; fp32 [40,
// 384, 288] 11.0 against 12.9, [40, 384, 256] 13.9 against 11.5, [2000, 257, 32], one workgroup
// a strip, 37.8 against 34.9). Smaller calls on more than eight packs go by the length of the
// tile's serial part, if they are few tiles or their rows are not divided by the segments (bf16
// [8, 384, 136] 9.9 -> 8.4 forward, [8, 384, 64], eight packs, 8.5 -> 7.8, [1, 512, 512] 8.3 ->
// 6.6 backward, but [8, 512, 576] 9.4 against 9.9; fp32 [1, 512, 132] 7.2 -> 6.5 backward, [8,
// 512, 256] 8.7 -> 7.8, [8, 512, 160] 6.8 against 7.5).
inline bool strided_team_beats_tile(bool backward, int64_t outer, int64_t D, int64_t packs, int esize, int TX,
                                    const StridedTeam& t) {
  if (D <= kStridedTeamMinD || TX >= 8 || TX >= packs) return false;
  const int64_t bytes = outer * D * packs * 16, tiles = outer * ((packs + TX - 1) / TX);
  const bool divided = packs % TX == 0, few = tiles <= 64;
  // packs of the teams' rounds that hold an element, in 64ths
  const int64_t held = outer * D * packs * 64 / (t.rounds * t.v * kTeamMaxWorkgroups * kTeamBlock);
  if (!backward && divided && !few && held < (esize == 4 ? (t.team > 1 ? 48 : 40) : t.team > 1 ? 32 : 29))
    return false;
  if (bytes >= (backward ? 7000000 : esize == 4 ? 13500000 : divided ? 9000000 : 7000000)) return true;
  if (packs < 8 || (packs == 8 && (backward || !few)) || (esize == 4 && !backward)) return false;
  const bool even = tiles <= 128 && packs % 16 == 0;
  if (backward) return divided ? D >= 448 && (even || (few && esize == 2)) : D >= (esize == 4 ? 448 : 320);
  return divided ? D >= 384 && few : D >= 320;
}

// Override: G = lanes along inner (power of two 1..64; -1 forces the multi-pass
// kernel, and then V = 1 keeps all D rows of a tile on one workgroup, V > 1 cuts
// them into that many chunks), V = packs per lane.  Returns 0 or -5.
// widened: the output's elements are wider than the input's.
inline int make_strided_plan(bool backward, int64_t outer, int64_t D, int64_t inner, int esize,
                             int num_cus, const Override& ov, StridedPlan* out, bool widened = false) {
  StridedPlan p;
  const int E = 16 / esize;
  const int64_t packs = (inner + E - 1) / E;
  p.fast = (inner % E) == 0;
  p.block = kStridedBlock;
  // an empty tensor launches nothing (the entry points return before they plan; the
  // plan query gets a plan with no workgroups)
  if (outer < 1 || D < 1 || inner < 1) {
    *out = p;
    return 0;
  }
  if (num_cus <= 0) num_cus = 256;
  const int px = packs >= 64 ? 64 : pow2_ceil(packs);  // lanes a row of `inner` can use
  // packs a lane may hold: 8, or 4 for the 16-bit backward (two packed rows per
  // lane) while a wavefront still covers D -- measured faster
  int vcap = kStridedMaxV;
  if (backward && esize == 2 && D > 4 && D <= 32) vcap = 4;
  if (ov.V > 0 && ov.G >= 0) vcap = ov.V;
  if (vcap < 1 || vcap > kStridedMaxV) return -5;
  // TY = the power of two that covers D with at most vcap rows a thread; V = the
  // rows a thread then really has (not rounded up: D = 21 is 4 x 6, not 4 x 8)
  const int64_t ty_need = pow2_ceil((D + vcap - 1) / vcap);
  int V = (ov.V > 0 && ov.G >= 0) ? ov.V : (int)((D + ty_need - 1) / ty_need);
  int TX = 0, TY = 0;
  // rows are never cut below 4 lanes (64 bytes) to make room for a larger D
  const int ty_max = kStridedBlock / (px < 4 ? px : 4);
  bool stream = ov.G < 0 || (ov.G == 0 && ty_need > ty_max) || ty_need > kStridedBlock;
  if (!stream) {
    TY = (int)ty_need;
    if (ov.G > 0) {
      if (ov.G > 64 || (ov.G & (ov.G - 1))) return -5;
      TX = ov.G;
    } else {
      int cap = 64 / TY;                 // one wavefront per group ...
      if (cap < 8) cap = 8;              // ... unless rows would shrink below 128 bytes
      if (cap * TY > kStridedBlock) cap = kStridedBlock / TY;
      TX = px < cap ? px : cap;
    }
    if ((int64_t)TX * TY > kStridedBlock || TX < 1) {
      if (ov.G > 0 || ov.V > 0) return -5;
      stream = true;
    }
  } else if (ov.G > 0 || (ov.V > 0 && ov.G >= 0)) {
    return -5;
  }
  if (stream) {
    // one group per workgroup, rows of up to 16 lanes (256 bytes; [8192, 8192] over dim 0,
    // forward / backward: 8 lanes 81.6 / 120.9 us, 16 lanes 80.1 / 113.9, 32 lanes 84.2 / 115.2)
    TX = px < 16 ? px : 16;
    TY = kStridedBlock / TX;
    V = 0;
    // Too few tiles to fill the machine (softmax over dim 0 of [8192, 8192] is 128
    // tiles): cut the D rows into chunks of whole TY * unroll strides so that
    // about four workgroups per compute unit exist; a short remainder joins the
    // chunk before it.
    const int64_t tiles = outer * ((packs + TX - 1) / TX);
    const int64_t min_rows = (int64_t)TY * kStridedSplitUnroll;
    int64_t want = 1;
    if (ov.G < 0 && ov.V > 0)
      want = ov.V;
    else if (tiles < 2 * (int64_t)num_cus)
      want = (4 * (int64_t)num_cus + tiles - 1) / tiles;
    if (want > 1) {
      int64_t rows = (D + want - 1) / want;
      rows = (rows + TY - 1) / TY * TY;
      if (rows < min_rows && !(ov.G < 0 && ov.V > 0)) rows = min_rows;
      int64_t chunks = (D + rows - 1) / rows;
      if (chunks > 1 && D - (chunks - 1) * rows < TY) --chunks;
      if (chunks > 65535) chunks = 1;
      if (chunks > 1) {
        p.chunks = (int)chunks;
        p.chunk_rows = (int)rows;
      }
    }
    if (p.chunks <= 1 && !(ov.G < 0 && ov.V > 0)) {
      // not split: fewer lanes along inner while the problem has less than two
      // workgroups per compute unit
      while (TX > 4 && outer * ((packs + TX - 1) / TX) < 2 * (int64_t)num_cus) TX >>= 1;
      TY = kStridedBlock / TX;
    }
  }
  // Strips held by teams of workgroups, where D is beyond the one-workgroup tile or teams are faster
  // than that.  Rows of no whole number of packs too (softmax_strided_team.hpp), by the rules of those rounded
  // up: without teams they were read two and three times, each row's last pack element by element (forward /
  // backward us: bf16 [93, 616, 723] 160 / 194 -> 52 / 67, [1, 6246, 78] 47.0 / 30.3 -> 10.1 / 8.0, fp16 [28, 3452,
  // 239] 80.6 / 90.0 -> 33.4 / 31.3; 400 calls of random shapes 0.57 and 0.52 of the time, none slower).
  if (inner >= E && ov.G == 0 && ov.V == 0 && ov.bpc == 0) {
    const StridedTeam t = strided_team(backward, outer, D, packs, esize, num_cus);
    if (t.team > 0 && (stream || strided_team_beats_tile(backward, outer, D, packs, esize, TX, t))) {
      p.team = t.team;
      p.team_v = t.v;
      p.team_tx_log2 = log2_of_pow2(t.tx);
      p.team_grid = t.grid;
      const StridedTeam l = strided_large_team(backward, outer, D, packs, esize, t, num_cus, widened);
      p.large_team = l.team;
      p.large_v = l.v;
      p.large_tx_log2 = log2_of_pow2(l.tx);
      p.large_grid = l.grid;
    }
  }
  p.resident = !stream;
  p.tx_log2 = log2_of_pow2(TX);
  p.ty_log2 = log2_of_pow2(TY);
  p.V = V;
  const int64_t xtiles = (packs + TX - 1) / TX;
  const int64_t ntiles = outer * xtiles;
  const int groups = kStridedBlock / (TX * TY);
  const int64_t nblocks = (ntiles + groups - 1) / groups;
  const int bpc = ov.bpc > 0 ? ov.bpc : (1 << 20);
  int64_t grid = (int64_t)num_cus * bpc;
  if (grid > nblocks) grid = nblocks;
  if (grid > 0x7fffffff) grid = 0x7fffffff;
  if (grid < 1) grid = 1;
  p.grid = grid;
  *out = p;
  return 0;
}

}  // namespace rownorm
