// softmax / log_softmax over a dimension that is not innermost, where D is beyond the one-workgroup
// tile of softmax_strided_kernels.hpp or teams are faster than that (strided_team_beats_tile()): every
// element crosses the memory interface once.
//
// The tensor is [outer, D, inner], inner a 16-byte pack or more (any alignment); a strip is
// TX consecutive packs of `inner` (up to 32: 512 bytes) and all D rows under them.  A team of `team`
// workgroups of 512 threads holds a strip in registers (and, one workgroup a compute unit, in LDS:
// strided_large_team()): workgroup c the rows [c * TY * V, (c + 1) * TY * V), thread (ty, tx) the V packs
// of rows ty, ty + TY, ... of pack column tx.  A workgroup reduces its rows per column (each
// lane over its packs, a wavefront by shuffles, the eight wavefronts through LDS), publishes the
// C = TX * E columns' numbers -- running maximum and sum of exp(x - maximum), or the sum the
// backward needs --, gathers its team's, merges them in a fixed order and writes its rows out of
// its registers.  A team of one exchanges nothing.  Teams walk the strips in rounds.
//
// What bounds it.  The split over launches that served these shapes reads the inputs twice and
// pays three launches; the multi-pass kernel reads them three times.  Here it is HBM plus what
// does not run under it: the forward's two exponentials an element (31 us of vector ALU time a
// [8192, 8192] call) and the exchange, whose rounds run in step.  Two workgroups a compute unit hold
// 64 MB in registers, so that call made two (forward) or four rounds; one workgroup of 256 registers a
// lane with 16 packs a lane more in LDS holds 128 MB: one or two rounds of teams a quarter as large,
// 70.5 / 103.7 -> 59.1 / 82.9 us (of the 59, the loads alone take 28, the exchange 7).  The exponentials of
// a group of packs are formed while the next groups are on their way: the rows past D are replaced group
// by group, not all at once, which waited for every load (71 -> 68 us).  bf16 forward / backward us,
// without -> with teams of two workgroups a compute unit: [8192, 8192] over dim 0 78.3 / 115 -> 67.8 / 102;
// [4000, 16384] 75.9 / 112 -> 64.6 / 83.6; [8192, 64] 17.6 / 12.1 -> 9.8 / 7.5; [8, 1000, 1024] 22.8 / 17.9 ->
// 12.0 / 12.3; [35, 1000, 1904] 150 / 176 -> 76.6 / 95.7; [100, 2000, 128] 38.6 / 45.6 -> 22.8 / 32.0.
// Requesting the next strip ahead of the exchange (half the packs a lane, twice the rounds)
// measured slower (84-90 us on [8192, 8192]), as did rows dealt out in bands over the team.
//
// The exchange.  A column's number travels as a self-validating 64-bit word {float32, tag} in
// library-owned memory (TeamColumns; tags, the bounded wait, the lost tag and the hint word as
// described in device/team.hpp): the writer orders nothing, a reader accepts a word whose tag is
// the round's.  The first wavefront polls one word a member (all threads polling their own words
// would be 16 MB of memory traffic a poll); once they are there every thread gathers: thread
// (q, column) reads members q, q + Q, ... of its team, Q = 512 / C.  Two buffers suffice: a
// workgroup publishes round r + 2 only after it has gathered round r + 1, which every mate
// published after it had gathered round r.
// A workgroup whose wait runs out walks all D rows of the strip itself (the output must not
// overlap an input) and publishes the lost tag from then on.
#pragma once
#include "device/team.hpp"
#include "softmax_strided_kernels.hpp"

namespace rownorm {

struct StridedTeamShape {
  int64_t strips, xtiles;  // outer * xtiles strips, xtiles of them side by side along inner
  int D, inner, tx_log2, team;
};

// A thread's place in a strip: pack column tx, rows ty, ty + TY, ...; the element of `inner` its
// packs start at.  A pack that would end past the row is the row's last whole pack instead: where the row is
// not a whole number of packs, its first elements are the neighbouring lane's as well, and both store the
// same result (their columns' numbers are formed alike; the neighbour may be another team's, so the output
// must then overlap no input); where the strip is wider than what is left of `inner`, the lane has no column
// of its own and stores nothing (in == false).
template <int E>
struct StridedTeamPlace {
  int tx, ty, TY, e0;
  bool in;
  __device__ __forceinline__ StridedTeamPlace(const StridedTeamShape& s, int tid, int64_t strip) {
    tx = tid & ((1 << s.tx_log2) - 1);
    ty = tid >> s.tx_log2;
    TY = kTeamBlock >> s.tx_log2;
    const int64_t e = (((strip % s.xtiles) << s.tx_log2) + tx) * E;
    in = e < s.inner;
    e0 = e + E <= s.inner ? (int)e : s.inner - E;
  }
};

// Packs [K0, K1) of this thread's V: rows r0 + ty + k * TY, pack column e0 (an element index inside
// the row), into p[0 .. K1 - K0).  One straight line for every workgroup (two versions of it would
// each want the packs in registers of their own): rows past D - 1 read row D - 1;
// strided_team_fill replaces them by `fill`.
template <class T, int E, int K0, int K1>
__device__ __forceinline__ void strided_team_load(Pack<T, E>* p, const T* strip, int r0, int ty,
                                                  int TY, int e0, int D, int inner) {
  const T* base = strip + (int64_t)r0 * inner;
  const int last = D - 1 - r0;
  // (offsets and bounds of the packs are formed here, not ahead of the strips, and one after the other)
  int row = lane_again(ty) + K0 * TY;
#pragma unroll
  for (int k = K0; k < K1; ++k, row += TY) {
    const int rc = row < last ? row : last;
    p[k - K0] = Pack<T, E>::load_stream(
        global_at(base, ((uint32_t)rc * (uint32_t)inner + (uint32_t)e0) * (uint32_t)sizeof(T)));
  }
}
template <class T, int E, int K0, int K1>
__device__ __forceinline__ void strided_team_fill(Pack<T, E>* p, int last, int ty, int TY, float fill) {
  const Pack<T, E> f = Pack<T, E>::splat(fill);
  int row = lane_again(ty) + K0 * TY;
#pragma unroll
  for (int k = K0; k < K1; ++k, row += TY)
    if (row > last) p[k - K0] = f;
}

// NF words a column: publishes v[0..NF) of the C columns (threads below C hold them).
template <int NF>
__device__ __forceinline__ void columns_publish(unsigned long long* mine, int C, bool lost,
                                                unsigned int call_id, unsigned int round,
                                                const float (&v)[NF]) {
  if ((int)threadIdx.x < C) {
    const unsigned long long tag =
        (unsigned long long)(lost ? team_lost_tag(call_id) : team_word_tag(call_id, round)) << 32;
#pragma unroll
    for (int k = 0; k < NF; ++k)
      team_store(&mine[k * kTeamColumns + (int)threadIdx.x],
                 tag | (unsigned long long)__builtin_bit_cast(unsigned int, v[k]));
  }
}

constexpr int kGatherWords = 8;  // words a thread requests before it looks at the first

// Merges N (maximum, sum) pairs into (m, s): one maximum, then N + 1 independent exponentials
// (pair by pair each merge would wait for the one before).
template <bool PRECISE, int N>
__device__ __forceinline__ void merge_pairs(float& m, float& s, const float (&vm)[N],
                                            const float (&vs)[N]) {
  float nm = m;
#pragma unroll
  for (int b = 0; b < N; ++b) nm = fmaxf(nm, vm[b]);
  // (nothing finite: the sums are 0, or NaN if an operand carries one, whatever they are scaled by)
  const float ref = nm == -INFINITY ? 0.0f : nm;
  s *= row_exp<PRECISE>(m - ref);
#pragma unroll
  for (int b = 0; b < N; ++b) s = fmaf(vs[b], row_exp<PRECISE>(vm[b] - ref), s);
  m = nm;
}

// Gathers this thread's share of the team: merge(v) is called with v[number][member] for members
// q, q + Q, ..., B at a time, after reset(); -inf / 0 stand for members past the team's end.  Every
// thread of the workgroup calls it; the result is uniform: true when
// all words of the round were there, false when the wait ran out or the call is lost.
template <int NF, class Reset, class Merge>
__device__ __forceinline__ bool columns_gather(TeamColumns* slot, const unsigned long long* mates,
                                               int C, int team,
                                               unsigned int call_id, unsigned int round,
                                               unsigned long long wait_ticks,
                                               int (&votes)[2][kTeamBlock / 64 + 1], Reset reset,
                                               Merge merge) {
  constexpr int B = kGatherWords / NF;
  const int col = (int)threadIdx.x & (C - 1), q = (int)threadIdx.x / C, Q = kTeamBlock / C;
  const unsigned int expect = team_word_tag(call_id, round);
  const unsigned long long t0 = wall_clock64();
  for (unsigned int polls = 0;; ++polls) {
    int status = 0;  // 1, a word is missing; 2, a lost tag, a hint or the end of the wait
    if (threadIdx.x < 64) {
      // one word of every member, until they are all there
      for (unsigned int n = 0;; ++n) {
        bool ok = true;
        status = 0;
        for (int j = (int)threadIdx.x; j < team; j += 64) {
          const unsigned int tag =
              (unsigned int)(team_load(&mates[(int64_t)j * (2 * kTeamColumns) + C - 1]) >> 32);
          ok = ok && tag == expect;
          if (team_tag_is_lost(tag, call_id)) status = 2;
        }
        const bool late = wall_clock64() - t0 > wait_ticks;
        if (__ballot(ok) == __ballot(true) && !(polls > 0 && late)) break;
        // (the hint word is one address for the whole grid: looked at every 16th time)
        if ((n & 15u) == 0 && __hip_atomic_load(&slot->gave_up, __ATOMIC_RELAXED,
                                                __HIP_MEMORY_SCOPE_AGENT) == call_id)
          status = 2;
        if (late) status = 2;
        if (__ballot(status != 0) != 0) break;
        __builtin_amdgcn_s_sleep(8);
      }
    }
    int (&vote)[kTeamBlock / 64 + 1] = votes[polls & 1u];
    if (threadIdx.x < 64) {
      const bool stop = __ballot(status != 0) != 0;
      if (threadIdx.x == 0) vote[kTeamBlock / 64] = stop ? 2 : 0;
    }
    __syncthreads();
    if (vote[kTeamBlock / 64] != 0) break;
    reset();
    status = 0;
    for (int j0 = q; j0 < team; j0 += B * Q) {
      unsigned long long w[B][NF];
#pragma unroll
      for (int b = 0; b < B; ++b) {
        const int j = j0 + b * Q;
#pragma unroll
        for (int k = 0; k < NF; ++k) w[b][k] = 0;
        if (j < team) {
#pragma unroll
          for (int k = 0; k < NF; ++k)
            w[b][k] = team_load(&mates[((int64_t)j * 2 + k) * kTeamColumns + col]);
        }
      }
      float v[NF][B];
#pragma unroll
      for (int b = 0; b < B; ++b) {
#pragma unroll
        for (int k = 0; k < NF; ++k) v[k][b] = NF == 2 && k == 0 ? -INFINITY : 0.0f;
        if (j0 + b * Q < team) {
#pragma unroll
          for (int k = 0; k < NF; ++k) {
            if ((unsigned int)(w[b][k] >> 32) != expect) status = 1;
            v[k][b] = __builtin_bit_cast(float, (unsigned int)(w[b][k] & 0xffffffffull));
          }
        }
      }
      merge(v);
    }
    const bool missing = __ballot(status != 0) != 0;
    if ((threadIdx.x & 63) == 0) vote[threadIdx.x >> 6] = missing ? 1 : 0;
    __syncthreads();
    int all = 0;
#pragma unroll
    for (int w = 0; w < kTeamBlock / 64; ++w) all |= vote[w];
    if (all == 0) return true;
    // (the words that were missing are on their way, or the wait ends above)
  }
  if (threadIdx.x == 0)
    __hip_atomic_store(&slot->gave_up, call_id, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return false;
}

// A wavefront's (m, s) per column, in every lane, from the lanes' own pairs.
template <int E, bool PRECISE>
__device__ __forceinline__ void wave_columns_merge(float (&m)[E], float (&s)[E], int TX) {
  float own[E];
#pragma unroll
  for (int i = 0; i < E; ++i) own[i] = m[i];
  for (int off = TX; off < 64; off <<= 1)
#pragma unroll
    for (int i = 0; i < E; ++i) m[i] = fmaxf(m[i], __shfl_xor(m[i], off, 64));
#pragma unroll
  for (int i = 0; i < E; ++i) s[i] = m[i] == -INFINITY ? s[i] : s[i] * row_exp<PRECISE>(own[i] - m[i]);
  for (int off = TX; off < 64; off <<= 1)
#pragma unroll
    for (int i = 0; i < E; ++i) s[i] += __shfl_xor(s[i], off, 64);
}

constexpr int kStridedTeamGroup = 4;

// A lane's packs in LDS: a slot of 16 bytes a thread and pack, which only that thread uses.
template <class T, int E, int L>
struct StridedTeamPark {
  typename Pack<T, E>::vec_t v[L > 0 ? L : 1][L > 0 ? kTeamBlock : 1];
  __device__ __forceinline__ void put(int k, const Pack<T, E>& p) { v[k][threadIdx.x] = p.v; }
  __device__ __forceinline__ Pack<T, E> get(int k) const {
    Pack<T, E> p;
    p.v = v[k][threadIdx.x];
    return p;
  }
};

template <class TI, class TO, int V>
__global__ void __launch_bounds__(kTeamBlock, strided_team_per_cu(false, V) * kTeamBlock / 256)
softmax_strided_team_fwd_kernel(const TI* __restrict__ x, TO* __restrict__ y, StridedTeamShape sh,
                                int flags, TeamColumns* slot, unsigned int call_id,
                                unsigned long long wait_ticks) {
  constexpr int E = elems_per_pack<TI>::value;
  constexpr bool PRECISE = sizeof(TO) == 4;
  constexpr int NW = kTeamBlock / 64;
  constexpr int L = strided_team_parked(false, V), R = V - L;  // packs of a lane in LDS, in registers
  constexpr int GR = kStridedTeamGroup;
  static_assert(L % GR == 0 && L <= R, "parked packs pass through registers group by group");
  __shared__ float wm[NW * kTeamColumns], ws[NW * kTeamColumns];  // the wavefronts' pairs
  __shared__ int votes[2][kTeamBlock / 64 + 1];
  __shared__ float gm[kTeamBlock], gs[kTeamBlock];                // the gathering threads' pairs
  __shared__ __align__(16) float fm[kTeamColumns], fk[kTeamColumns];  // maximum, 1/sum or log(sum)
  __shared__ StridedTeamPark<TI, E, L> park;
  const bool is_log = (flags & kSoftmaxLog) != 0;
  const bool is_safe = (flags & kSoftmaxSafe) != 0;
  const int D = sh.D, inner = sh.inner, team = sh.team;
  const int TX = 1 << sh.tx_log2, C = TX * E;
  const int tm = (int)blockIdx.x / team;
  const int teams = (int)gridDim.x / team;
  const int r0 = ((int)blockIdx.x - tm * team) * (kTeamBlock >> sh.tx_log2) * V;
  const int lane = (int)threadIdx.x & 63, wave = (int)threadIdx.x >> 6;
  bool lost = false;
  unsigned int round = 0;
  for (int64_t strip = tm; strip < sh.strips; strip += teams, ++round) {
    // packs 0 .. L - 1 go to LDS, packs L .. V - 1 to xp[0 .. R - 1]
    Pack<TI, E> xp[R];
    // The lane's running maxima and sums, kGroup packs at a time: the exponentials of one group are
    // formed while the next ones are still on their way.
    float m[E], s[E];
#pragma unroll
    for (int i = 0; i < E; ++i) {
      m[i] = -INFINITY;
      s[i] = 0.0f;
    }
    auto absorb = [&](Pack<TI, E>* p, auto k_first, auto n) {
      constexpr int KN = decltype(n)::value;
      float ref[E];
#pragma unroll
      for (int i = 0; i < E; ++i) ref[i] = m[i];
#pragma unroll
      for (int k = 0; k < KN; ++k) {
#pragma unroll
        for (int i = 0; i < E; ++i) ref[i] = fmaxf(ref[i], p[k].get(i));
        keep_packed(p[k]);
      }
      // (nothing finite so far: against 0, -inf elements add 0 and NaN still poisons)
#pragma unroll
      for (int i = 0; i < E; ++i) {
        const float own = m[i];
        m[i] = ref[i];
        ref[i] = ref[i] == -INFINITY ? 0.0f : ref[i];
        if constexpr (decltype(k_first)::value > 0) s[i] *= row_exp<PRECISE>(own - ref[i]);
      }
#pragma unroll
      for (int k = 0; k < KN; ++k) {
#pragma unroll
        for (int i = 0; i < E; ++i) s[i] += row_exp<PRECISE>(p[k].get(i) - ref[i]);
        keep_packed(p[k]);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    {
      const StridedTeamPlace<E> t(sh, lane_again((int)threadIdx.x), strip);
      const TI* xs = x + (strip / sh.xtiles) * (int64_t)D * inner;
      const int last = D - 1 - r0;
      // the parked packs first, through the registers of the last L packs, which are requested as
      // the groups are put away
      if constexpr (L > 0)
        strided_team_load<TI, E, 0, L>(xp + (R - L), xs, r0, t.ty, t.TY, t.e0, D, inner);
      strided_team_load<TI, E, L, V - L>(xp, xs, r0, t.ty, t.TY, t.e0, D, inner);
      static_for<0, L / GR>([&](auto g) {
        constexpr int K = decltype(g)::value * GR;
        Pack<TI, E>* p = xp + (R - L + K);
        strided_team_fill<TI, E, K, K + GR>(p, last, t.ty, t.TY, -INFINITY);
        absorb(p, std::integral_constant<int, K>{}, std::integral_constant<int, GR>{});
#pragma unroll
        for (int k = 0; k < GR; ++k) park.put(K + k, p[k]);
        strided_team_load<TI, E, V - L + K, V - L + K + GR>(p, xs, r0, t.ty, t.TY, t.e0, D, inner);
        __builtin_amdgcn_sched_barrier(0);
      });
      static_for<0, (R + GR - 1) / GR>([&](auto g) {
        constexpr int K = decltype(g)::value * GR, K1 = K + GR < R ? K + GR : R;
        strided_team_fill<TI, E, L + K, L + K1>(xp + K, last, t.ty, t.TY, -INFINITY);
        absorb(xp + K, std::integral_constant<int, L + K>{}, std::integral_constant<int, K1 - K>{});
      });
    }
    // (formed here: moved behind the reduction of the maxima it would need a copy of the packs)
#pragma unroll
    for (int i = 0; i < E; ++i) asm volatile("" : "+v"(s[i]));
    // the pair of column threadIdx.x < C: the workgroup's, then the strip's
    float pm = -INFINITY, ps = 0.0f;
    auto merge_workgroup = [&]() {
      wave_columns_merge<E, PRECISE>(m, s, TX);
      if (lane < TX) {
#pragma unroll
        for (int i = 0; i < E; ++i) {
          wm[wave * kTeamColumns + lane * E + i] = m[i];
          ws[wave * kTeamColumns + lane * E + i] = s[i];
        }
      }
      __syncthreads();
      if ((int)threadIdx.x < C) {
        float vm[NW], vs[NW];
#pragma unroll
        for (int w = 0; w < NW; ++w) {
          vm[w] = wm[w * kTeamColumns + threadIdx.x];
          vs[w] = ws[w * kTeamColumns + threadIdx.x];
        }
        pm = -INFINITY;
        ps = 0.0f;
        merge_pairs<PRECISE>(pm, ps, vm, vs);
      }
    };
    merge_workgroup();
    unsigned long long* words = &slot->word[round & 1u][0][0];
    if (team > 1)
      columns_publish<2>(words + (int64_t)blockIdx.x * (2 * kTeamColumns), C, lost, call_id, round,
                         {pm, ps});
    if (team > 1) {
      float am = -INFINITY, as = 0.0f;
      if (!lost)
        lost = !columns_gather<2>(
            slot, words + (int64_t)tm * team * (2 * kTeamColumns), C, team, call_id, round,
            wait_ticks, votes,
            [&]() {
              am = -INFINITY;
              as = 0.0f;
            },
            [&](const auto& v) { merge_pairs<PRECISE>(am, as, v[0], v[1]); });
      if (!lost) {
        gm[threadIdx.x] = am;
        gs[threadIdx.x] = as;
        __syncthreads();
        if ((int)threadIdx.x < C) {
          pm = gm[threadIdx.x];
          ps = gs[threadIdx.x];
          const int n = kTeamBlock / C < team ? kTeamBlock / C : team;
          for (int g = 1; g < n; ++g)
            online_merge<PRECISE>(pm, ps, gm[g * C + threadIdx.x], gs[g * C + threadIdx.x]);
        }
      } else {
        // the team did not come together: all rows of the strip, then this workgroup's again
        const StridedTeamPlace<E> t(sh, (int)threadIdx.x, strip);
        const TI* xs = x + (strip / sh.xtiles) * (int64_t)D * inner + t.e0;
#pragma unroll
        for (int i = 0; i < E; ++i) {
          m[i] = -INFINITY;
          s[i] = 0.0f;
        }
        for (int d = t.ty; d < D; d += t.TY) {
          const Pack<TI, E> p = Pack<TI, E>::load(xs + (int64_t)d * inner);
#pragma unroll
          for (int i = 0; i < E; ++i) {
            const float nm = fmaxf(m[i], p.get(i));
            const float rf = nm == -INFINITY ? 0.0f : nm;
            s[i] = s[i] * row_exp<PRECISE>(m[i] - rf) + row_exp<PRECISE>(p.get(i) - rf);
            m[i] = nm;
          }
        }
        __syncthreads();  // (wm / ws have been read)
        merge_workgroup();
      }
    }
    if ((int)threadIdx.x < C) {
      fm[threadIdx.x] = pm;
      fk[threadIdx.x] = is_log ? logf(ps) : 1.0f / ps;
    }
    __syncthreads();
    // (the lane's place again, after the exchange: offsets and bounds of its rows are not
    // carried through it)
    const StridedTeamPlace<E> t(sh, lane_again((int)threadIdx.x), strip);
    float kf[E];
#pragma unroll
    for (int i = 0; i < E; ++i) {
      m[i] = fm[t.tx * E + i];
      kf[i] = fk[t.tx * E + i];
    }
    TO* yb = y + ((strip / sh.xtiles) * (int64_t)D + r0) * inner;
    const bool full = r0 + t.TY * V <= D;
    auto store_rows = [&](auto value) {
      const uint32_t off = ((uint32_t)t.ty * (uint32_t)inner + (uint32_t)t.e0) * (uint32_t)sizeof(TO);
      const int64_t step = (int64_t)t.TY * inner;
      int left = D - r0 - t.ty;  // (counted down pack by pack: a bound each would hold a register each)
      auto store_row = [&](const Pack<TI, E>& p) {
        Pack<TO, E> out;
#pragma unroll
        for (int i = 0; i < E; ++i) out.set(i, value(p.get(i), i));
        if (full || left > 0) out.store_stream(global_at(yb, off));
        yb = scalar_again(yb + step);
        left = lane_again(left - t.TY);
        __builtin_amdgcn_sched_barrier(0);
      };
      if constexpr (L > 0) {
        // (the next parked pack is read while one is worked on)
        Pack<TI, E> next = park.get(0);
#pragma unroll
        for (int k = 0; k < L; ++k) {
          const Pack<TI, E> p = next;
          if (k + 1 < L) next = park.get(k + 1);
          store_row(p);
        }
      }
#pragma unroll
      for (int k = 0; k < R; ++k) store_row(xp[k]);
    };
    if (t.in) {
      if (is_log) {
        ROWNORM_UNIFORM_ARM("log_softmax, a strip held by a team");
        store_rows([&](float v, int i) { return (v - m[i]) - kf[i]; });
      } else {
        ROWNORM_UNIFORM_ARM("softmax, a strip held by a team");
        if (is_safe) {
#pragma unroll
          for (int i = 0; i < E; ++i)
            if (m[i] == -INFINITY) m[i] = kf[i] = 0.0f;  // exp(-inf - 0) * 0
        }
        store_rows([&](float v, int i) { return row_exp<PRECISE>(v - m[i]) * kf[i]; });
      }
    }
  }
}

// Backward: V packs a lane of grad and of y; the columns' sums of y * grad (log_softmax: of grad)
// cross the team.
template <class TG, class TO, int V>
__global__ void __launch_bounds__(kTeamBlock, strided_team_per_cu(true, V) * kTeamBlock / 256)
softmax_strided_team_bwd_kernel(const TG* __restrict__ grad, const TG* __restrict__ y,
                                TO* __restrict__ gi, StridedTeamShape sh, int flags,
                                TeamColumns* slot, unsigned int call_id,
                                unsigned long long wait_ticks) {
  constexpr int E = elems_per_pack<TG>::value;
  constexpr bool PRECISE = sizeof(TO) == 4 && sizeof(TG) == 4;
  constexpr int NW = kTeamBlock / 64;
  constexpr int L = strided_team_parked(true, V), R = V - L;  // as in the forward, of each tensor
  constexpr int GR = kStridedTeamGroup;
  static_assert(L % GR == 0 && L <= R, "parked packs pass through registers group by group");
  __shared__ float ws[NW * kTeamColumns];
  __shared__ int votes[2][kTeamBlock / 64 + 1];
  __shared__ float gs[kTeamBlock];
  __shared__ __align__(16) float fs[kTeamColumns];
  __shared__ StridedTeamPark<TG, E, L> gpark, ypark;
  const bool is_log = (flags & kSoftmaxLog) != 0;
  const int D = sh.D, inner = sh.inner, team = sh.team;
  const int TX = 1 << sh.tx_log2, C = TX * E;
  const int tm = (int)blockIdx.x / team;
  const int teams = (int)gridDim.x / team;
  const int r0 = ((int)blockIdx.x - tm * team) * (kTeamBlock >> sh.tx_log2) * V;
  const int lane = (int)threadIdx.x & 63, wave = (int)threadIdx.x >> 6;
  bool lost = false;
  unsigned int round = 0;
  for (int64_t strip = tm; strip < sh.strips; strip += teams, ++round) {
    Pack<TG, E> gp[R], yp[R];
    float s[E];
#pragma unroll
    for (int i = 0; i < E; ++i) s[i] = 0.0f;
    // (no branch on the variant: two arms would each want the packs in registers of their own)
    {
      const StridedTeamPlace<E> t(sh, lane_again((int)threadIdx.x), strip);
      const int64_t slab = (strip / sh.xtiles) * (int64_t)D * inner;
      const TG *gs_ = grad + slab, *ys_ = y + slab;
      auto load = [&](int at, auto k0, auto k1) {
        constexpr int K0 = decltype(k0)::value, K1 = decltype(k1)::value;
        strided_team_load<TG, E, K0, K1>(gp + at, gs_, r0, t.ty, t.TY, t.e0, D, inner);
        strided_team_load<TG, E, K0, K1>(yp + at, ys_, r0, t.ty, t.TY, t.e0, D, inner);
      };
      int left = D - r0 - t.ty;  // (as in the stores below)
      auto absorb = [&](Pack<TG, E>& g, Pack<TG, E>& v) {
#pragma unroll
        for (int i = 0; i < E; ++i) {
          const float sum = fmaf(is_log ? 1.0f : v.get(i), g.get(i), s[i]);
          s[i] = left > 0 ? sum : s[i];
        }
        left = lane_again(left - t.TY);
        keep_packed(g);
        keep_packed(v);
        __builtin_amdgcn_sched_barrier(0);
      };
      // the parked packs first, as in the forward; the two tensors group by group where there are
      // many packs, so that sums are formed while the rest is on its way
      static_for<0, L / GR>([&](auto g) {
        constexpr int K = decltype(g)::value * GR;
        load(R - L + K, std::integral_constant<int, K>{}, std::integral_constant<int, K + GR>{});
      });
      constexpr int LG = V > strided_team_max_v(true) ? GR : R;
      static_assert((R - L) % LG == 0, "whole groups");
      static_for<0, (R - L) / LG>([&](auto g) {
        constexpr int K = decltype(g)::value * LG;
        load(K, std::integral_constant<int, L + K>{}, std::integral_constant<int, L + K + LG>{});
      });
      static_for<0, L / GR>([&](auto g) {
        constexpr int K = decltype(g)::value * GR, AT = R - L + K, K1 = V - L + K;
        static_for<0, GR>([&](auto k) {
          constexpr int J = decltype(k)::value;
          absorb(gp[AT + J], yp[AT + J]);
          gpark.put(K + J, gp[AT + J]);
          ypark.put(K + J, yp[AT + J]);
        });
        load(AT, std::integral_constant<int, K1>{}, std::integral_constant<int, K1 + GR>{});
        __builtin_amdgcn_sched_barrier(0);
      });
      static_for<0, R>([&](auto k) { absorb(gp[decltype(k)::value], yp[decltype(k)::value]); });
    }
#pragma unroll
    for (int i = 0; i < E; ++i) asm volatile("" : "+v"(s[i]));
    float ps = 0.0f;  // the sum of column threadIdx.x < C: the workgroup's, then the strip's
    auto merge_workgroup = [&]() {
      for (int off = TX; off < 64; off <<= 1)
#pragma unroll
        for (int i = 0; i < E; ++i) s[i] += __shfl_xor(s[i], off, 64);
      if (lane < TX) {
#pragma unroll
        for (int i = 0; i < E; ++i) ws[wave * kTeamColumns + lane * E + i] = s[i];
      }
      __syncthreads();
      if ((int)threadIdx.x < C) {
        ps = ws[threadIdx.x];
#pragma unroll
        for (int w = 1; w < NW; ++w) ps += ws[w * kTeamColumns + threadIdx.x];
      }
    };
    merge_workgroup();
    unsigned long long* words = &slot->word[round & 1u][0][0];
    if (team > 1)
      columns_publish<1>(words + (int64_t)blockIdx.x * (2 * kTeamColumns), C, lost, call_id, round,
                         {ps});
    if (team > 1) {
      float as = 0.0f;
      if (!lost)
        lost = !columns_gather<1>(
            slot, words + (int64_t)tm * team * (2 * kTeamColumns), C, team, call_id, round,
            wait_ticks, votes, [&]() { as = 0.0f; }, [&](const auto& v) {
#pragma unroll
              for (float f : v[0]) as += f;
            });
      if (!lost) {
        gs[threadIdx.x] = as;
        __syncthreads();
        if ((int)threadIdx.x < C) {
          ps = gs[threadIdx.x];
          const int n = kTeamBlock / C < team ? kTeamBlock / C : team;
          for (int g = 1; g < n; ++g) ps += gs[g * C + threadIdx.x];
        }
      } else {
        // the team did not come together: all rows of the strip, then this workgroup's again
        const StridedTeamPlace<E> t(sh, (int)threadIdx.x, strip);
        const int64_t at = (strip / sh.xtiles) * (int64_t)D * inner + t.e0;
#pragma unroll
        for (int i = 0; i < E; ++i) s[i] = 0.0f;
        for (int d = t.ty; d < D; d += t.TY) {
          const Pack<TG, E> pg = Pack<TG, E>::load(grad + at + (int64_t)d * inner);
          const Pack<TG, E> py = Pack<TG, E>::load(y + at + (int64_t)d * inner);
#pragma unroll
          for (int i = 0; i < E; ++i) s[i] += is_log ? pg.get(i) : py.get(i) * pg.get(i);
        }
        __syncthreads();  // (ws has been read)
        merge_workgroup();
      }
    }
    if ((int)threadIdx.x < C) fs[threadIdx.x] = ps;
    __syncthreads();
    const StridedTeamPlace<E> t(sh, lane_again((int)threadIdx.x), strip);
#pragma unroll
    for (int i = 0; i < E; ++i) s[i] = fs[t.tx * E + i];
    TO* ob = gi + ((strip / sh.xtiles) * (int64_t)D + r0) * inner;
    const bool full = r0 + t.TY * V <= D;
    auto store_rows = [&](auto value) {
      const uint32_t off = ((uint32_t)t.ty * (uint32_t)inner + (uint32_t)t.e0) * (uint32_t)sizeof(TO);
      const int64_t step = (int64_t)t.TY * inner;
      int left = D - r0 - t.ty;  // (counted down pack by pack: a bound each would hold a register each)
      auto store_row = [&](const Pack<TG, E>& g, const Pack<TG, E>& v) {
        Pack<TO, E> out;
#pragma unroll
        for (int i = 0; i < E; ++i) out.set(i, value(g.get(i), v.get(i), s[i]));
        if (full || left > 0) out.store_stream(global_at(ob, off));
        ob = scalar_again(ob + step);
        left = lane_again(left - t.TY);
        __builtin_amdgcn_sched_barrier(0);
      };
      if constexpr (L > 0) {
        Pack<TG, E> ng = gpark.get(0), nv = ypark.get(0);
#pragma unroll
        for (int k = 0; k < L; ++k) {
          const Pack<TG, E> g = ng, v = nv;
          if (k + 1 < L) {
            ng = gpark.get(k + 1);
            nv = ypark.get(k + 1);
          }
          store_row(g, v);
        }
      }
#pragma unroll
      for (int k = 0; k < R; ++k) store_row(gp[k], yp[k]);
    };
    if (t.in) {
      if (is_log) {
        ROWNORM_UNIFORM_ARM("log_softmax backward, a strip held by a team");
        store_rows([](float g, float v, float sum) { return g - row_exp<PRECISE>(v) * sum; });
      } else {
        ROWNORM_UNIFORM_ARM("softmax backward, a strip held by a team");
        store_rows([](float g, float v, float sum) { return v * (g - sum); });
      }
    }
  }
}

}  // namespace rownorm
