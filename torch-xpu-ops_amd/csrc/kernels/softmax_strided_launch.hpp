// Host dispatch of the non-innermost-dimension softmax kernels: plan -> template instance.
#pragma once
#include "launch.hpp"
#include "softmax_strided_kernels.hpp"
#include "softmax_strided_team.hpp"

namespace rownorm {

// Launches the instance whose packs a lane the plan names: go(packs, shape, grid); false if there is
// none.
template <bool BACKWARD, bool LARGE, size_t I = 0, class Go>
bool launch_strided_team_v(int v, Go go) {
  constexpr auto& list = [] () -> auto& {
    if constexpr (LARGE) return kStridedLargeV[BACKWARD ? 1 : 0];
    else return kStridedTeamV[BACKWARD ? 1 : 0];
  }();
  if (v == list[I]) {
    go(std::integral_constant<int, list[I]>{});
    return true;
  }
  if constexpr (list[I] < (LARGE ? strided_large_max_v(BACKWARD) : strided_team_max_v(BACKWARD)))
    return launch_strided_team_v<BACKWARD, LARGE, I + 1>(v, go);
  return false;
}
// (LARGE: the instances with a compute unit a workgroup are built, see strided_large_team())
template <bool BACKWARD, int E, bool LARGE, class Go>
bool launch_strided_team(const StridedPlan& p, int64_t outer, int D, int inner, Go go) {
  const bool large = p.large_team > 0;
  const int tx_log2 = large ? p.large_tx_log2 : p.team_tx_log2;
  const int64_t xtiles = ((inner + E - 1) / E + (1 << tx_log2) - 1) >> tx_log2;
  const StridedTeamShape sh{outer * xtiles, xtiles, D, inner, tx_log2, large ? p.large_team : p.team};
  const dim3 grid((unsigned)(large ? p.large_grid : p.team_grid));
  if (large) {
    if constexpr (LARGE)
      return launch_strided_team_v<BACKWARD, true>(p.large_v, [&](auto v) { go(v, sh, grid); });
    return false;
  }
  return launch_strided_team_v<BACKWARD, false>(p.team_v, [&](auto v) { go(v, sh, grid); });
}

// Whether the kernels that move whole packs alone serve rows of `inner` elements: rows of whole packs, and others
// where nobody reads what the last packs' neighbours write (strided_tile(), StridedTeamPlace).  On the one-workgroup
// tile an element at a time in a row's last pack costs up to a fifth more (bf16 [26, 26, 16182] backward 21.1 ->
// 17.9 us, fp32 [29, 91, 3854] 42.4 -> 36.3).
inline bool strided_whole_packs(const StridedPlan& p, int inner, int E, bool apart) {
  return p.fast || (inner >= E && apart);
}

template <class TI, class TO, int V, bool FAST>
void launch_strided_fwd_v(const StridedPlan& p, const SoftmaxStridedFwdArgs& a, hipStream_t s) {
  hipLaunchKernelGGL((softmax_strided_fwd_kernel<TI, TO, V, kStridedBlock, FAST>),
                     dim3((unsigned)p.grid), dim3(kStridedBlock), 0, s, (const TI*)a.x, (TO*)a.y,
                     a.outer, a.D, a.inner, StridedLayout{p.tx_log2, p.ty_log2}, a.flags);
}

template <class TI, class TO, bool FAST>
bool launch_strided_fwd_f(const StridedPlan& p, const SoftmaxStridedFwdArgs& a, hipStream_t s) {
  switch (p.V) {
    case 1: launch_strided_fwd_v<TI, TO, 1, FAST>(p, a, s); return true;
    case 2: launch_strided_fwd_v<TI, TO, 2, FAST>(p, a, s); return true;
    case 3: launch_strided_fwd_v<TI, TO, 3, FAST>(p, a, s); return true;
    case 4: launch_strided_fwd_v<TI, TO, 4, FAST>(p, a, s); return true;
    case 5: launch_strided_fwd_v<TI, TO, 5, FAST>(p, a, s); return true;
    case 6: launch_strided_fwd_v<TI, TO, 6, FAST>(p, a, s); return true;
    case 7: launch_strided_fwd_v<TI, TO, 7, FAST>(p, a, s); return true;
    case 8: launch_strided_fwd_v<TI, TO, 8, FAST>(p, a, s); return true;
  }
  return false;
}

template <class TI, class TO>
int launch_softmax_strided_fwd(const StridedPlan& p, const SoftmaxStridedFwdArgs& a,
                               hipStream_t s) {
  const int64_t n = a.outer * (int64_t)a.D * a.inner;
  const bool apart = regions_disjoint(a.y, n * (int64_t)sizeof(TO), a.x, n * (int64_t)sizeof(TI));
  const bool whole = strided_whole_packs(p, a.inner, elems_per_pack<TI>::value, apart);
  if ((p.team_size() == 1 && whole) || (p.team_size() > 1 && a.team_slot != nullptr)) {
    const bool ok = launch_strided_team<false, elems_per_pack<TI>::value, sizeof(TO) <= sizeof(TI)>(
        p, a.outer, a.D, a.inner, [&](auto v, const StridedTeamShape& sh, dim3 grid) {
          hipLaunchKernelGGL((softmax_strided_team_fwd_kernel<TI, TO, decltype(v)::value>), grid,
                             dim3(kTeamBlock), 0, s, (const TI*)a.x, (TO*)a.y, sh, a.flags,
                             (TeamColumns*)a.team_slot, a.team_id, a.team_wait_ticks);
        });
    if (!ok) return (int)hipErrorInvalidConfiguration;
  } else if (p.resident) {
    const bool ok = whole ? launch_strided_fwd_f<TI, TO, true>(p, a, s)
                          : launch_strided_fwd_f<TI, TO, false>(p, a, s);
    if (!ok) return (int)hipErrorInvalidConfiguration;
  } else if (p.chunks > 1 && apart) {
    // the D rows of a tile are split over workgroups; the per-column values cross the
    // three launches inside y, which therefore must not be x
    constexpr int E = elems_per_pack<TI>::value;
    const StridedLayout lay{p.tx_log2, p.ty_log2};
    const dim3 grid((unsigned)p.grid, (unsigned)p.chunks);
    hipLaunchKernelGGL((softmax_strided_split_partial_kernel<TI, TO, kStridedBlock>), grid,
                       dim3(kStridedBlock), 0, s, (const TI*)a.x, (TO*)a.y, a.outer, a.D, a.inner,
                       lay, p.chunk_rows);
    hipLaunchKernelGGL((softmax_strided_split_combine_kernel<TO, E, 2, kStridedBlock>),
                       dim3((unsigned)p.grid), dim3(kStridedBlock), 0, s, (TO*)a.y, a.outer, a.D,
                       a.inner, lay, p.chunk_rows, p.chunks);
    hipLaunchKernelGGL((softmax_strided_split_apply_kernel<TI, TO, kStridedBlock>), grid,
                       dim3(kStridedBlock), 0, s, (const TI*)a.x, (TO*)a.y, a.outer, a.D, a.inner,
                       lay, p.chunk_rows, a.flags);
  } else {
    hipLaunchKernelGGL((softmax_strided_fwd_stream_kernel<TI, TO, kStridedBlock>),
                       dim3((unsigned)p.grid), dim3(kStridedBlock), 0, s, (const TI*)a.x,
                       (TO*)a.y, a.outer, a.D, a.inner, StridedLayout{p.tx_log2, p.ty_log2},
                       a.flags);
  }
  return (int)hipGetLastError();
}

template <class TG, class TO, int V, bool FAST>
void launch_strided_bwd_v(const StridedPlan& p, const SoftmaxStridedBwdArgs& a, hipStream_t s) {
  hipLaunchKernelGGL((softmax_strided_bwd_kernel<TG, TO, V, kStridedBlock, FAST>),
                     dim3((unsigned)p.grid), dim3(kStridedBlock), 0, s, (const TG*)a.grad,
                     (const TG*)a.y, (TO*)a.gi, a.outer, a.D, a.inner,
                     StridedLayout{p.tx_log2, p.ty_log2}, a.flags);
}

template <class TG, class TO, bool FAST>
bool launch_strided_bwd_f(const StridedPlan& p, const SoftmaxStridedBwdArgs& a, hipStream_t s) {
  switch (p.V) {
    case 1: launch_strided_bwd_v<TG, TO, 1, FAST>(p, a, s); return true;
    case 2: launch_strided_bwd_v<TG, TO, 2, FAST>(p, a, s); return true;
    case 3: launch_strided_bwd_v<TG, TO, 3, FAST>(p, a, s); return true;
    case 4: launch_strided_bwd_v<TG, TO, 4, FAST>(p, a, s); return true;
    case 5: launch_strided_bwd_v<TG, TO, 5, FAST>(p, a, s); return true;
    case 6: launch_strided_bwd_v<TG, TO, 6, FAST>(p, a, s); return true;
    case 7: launch_strided_bwd_v<TG, TO, 7, FAST>(p, a, s); return true;
    case 8: launch_strided_bwd_v<TG, TO, 8, FAST>(p, a, s); return true;
  }
  return false;
}

template <class TG, class TO>
int launch_softmax_strided_bwd(const StridedPlan& p, const SoftmaxStridedBwdArgs& a,
                               hipStream_t s) {
  const int64_t n = a.outer * (int64_t)a.D * a.inner;
  const int64_t ob = n * (int64_t)sizeof(TO), ib = n * (int64_t)sizeof(TG);
  const bool apart = regions_disjoint(a.gi, ob, a.grad, ib) && regions_disjoint(a.gi, ob, a.y, ib);
  const bool whole = strided_whole_packs(p, a.inner, elems_per_pack<TG>::value, apart);
  if ((p.team_size() == 1 && whole) || (p.team_size() > 1 && a.team_slot != nullptr)) {
    const bool ok = launch_strided_team<true, elems_per_pack<TG>::value, true>(
        p, a.outer, a.D, a.inner, [&](auto v, const StridedTeamShape& sh, dim3 grid) {
          hipLaunchKernelGGL((softmax_strided_team_bwd_kernel<TG, TO, decltype(v)::value>), grid,
                             dim3(kTeamBlock), 0, s, (const TG*)a.grad, (const TG*)a.y, (TO*)a.gi,
                             sh, a.flags, (TeamColumns*)a.team_slot, a.team_id, a.team_wait_ticks);
        });
    if (!ok) return (int)hipErrorInvalidConfiguration;
  } else if (p.resident) {
    const bool ok = whole ? launch_strided_bwd_f<TG, TO, true>(p, a, s)
                          : launch_strided_bwd_f<TG, TO, false>(p, a, s);
    if (!ok) return (int)hipErrorInvalidConfiguration;
  } else if (p.chunks > 1 && apart) {
    constexpr int E = elems_per_pack<TG>::value;
    const StridedLayout lay{p.tx_log2, p.ty_log2};
    const dim3 grid((unsigned)p.grid, (unsigned)p.chunks);
    hipLaunchKernelGGL((softmax_strided_split_bwd_partial_kernel<TG, TO, kStridedBlock>), grid,
                       dim3(kStridedBlock), 0, s, (const TG*)a.grad, (const TG*)a.y, (TO*)a.gi,
                       a.outer, a.D, a.inner, lay, p.chunk_rows, a.flags);
    hipLaunchKernelGGL((softmax_strided_split_combine_kernel<TO, E, 1, kStridedBlock>),
                       dim3((unsigned)p.grid), dim3(kStridedBlock), 0, s, (TO*)a.gi, a.outer, a.D,
                       a.inner, lay, p.chunk_rows, p.chunks);
    hipLaunchKernelGGL((softmax_strided_split_bwd_apply_kernel<TG, TO, kStridedBlock>), grid,
                       dim3(kStridedBlock), 0, s, (const TG*)a.grad, (const TG*)a.y, (TO*)a.gi,
                       a.outer, a.D, a.inner, lay, p.chunk_rows, a.flags);
  } else {
    hipLaunchKernelGGL((softmax_strided_bwd_stream_kernel<TG, TO, kStridedBlock>),
                       dim3((unsigned)p.grid), dim3(kStridedBlock), 0, s, (const TG*)a.grad,
                       (const TG*)a.y, (TO*)a.gi, a.outer, a.D, a.inner,
                     StridedLayout{p.tx_log2, p.ty_log2}, a.flags);
  }
  return (int)hipGetLastError();
}

}  // namespace rownorm
