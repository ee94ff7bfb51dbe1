// LayerNorm / RMSNorm of rows that fit no power of two of lanes, forward and backward (gfx950, wave64).
//
// A row is held by `waves` wavefronts (a launch argument, 1 to 16), V packs a lane, and a workgroup by as
// many such groups (row slots) as it has wavefronts for.  Pack c of lane l is number c * 64 * waves + l;
// a pack that would end past the row is the row's last whole pack instead, read from E elements before
// the row's end, so that every access of the row loop is one unconditional 128-bit load or store inside
// the row, whatever its length: its first elements are then another lane's as well.  They count in the
// other lane only (the row sums leave them out by a select, the column sums are not written), and both
// lanes store the same result.  Only the last of a lane's packs can be such a one.  With nothing
// conditional between them, the next rows' loads are on their way while one is worked on, in register
// sets of their own (as in norm_bwd_exact_kernel, whose layouts fill their lanes exactly).
//
// What bounds the general kernels on such rows is memory latency: a row of 4097 16-bit elements is 513
// packs, on 512 lanes of two packs half of the requests a compute unit can hold are for nothing, and the
// next row is not asked for before the last one has been stored.
#pragma once
#include <type_traits>

#include "device/pack.hpp"
#include "device/reduce.hpp"
#include "plan.hpp"

namespace rownorm {

// A lane's place: pack c at element at[c] (in bytes, from the row's start); the first `skip` elements of
// its last pack are another lane's.
template <class T, int V>
struct WavesPlace {
  uint32_t off[V];
  int skip;
  // The offset of pack c, formed anew where it is used: widened to 64 bits ahead of the row loop it would
  // hold two registers and the accesses could not take it beside a scalar pointer.
  __device__ __forceinline__ uint32_t operator[](int c) const { return (uint32_t)lane_again((int)off[c]); }
  __device__ __forceinline__ WavesPlace(int lane, int G, int N) {
    constexpr int E = elems_per_pack<T>::value;
#pragma unroll
    for (int c = 0; c < V; ++c) {
      const int e0 = (c * G + lane) * E;
      const int e = e0 < N - E ? e0 : N - E;
      off[c] = (uint32_t)e * (uint32_t)sizeof(T);
      if (c == V - 1) skip = e0 - e;
    }
  }
};

// All-reduce of K sums over the `waves` wavefronts of a row slot (every thread of the workgroup calls it).
// red: two buffers, used in turn.
template <int K>
__device__ __forceinline__ void waves_allreduce(float (&v)[K], float (*red)[16][2], int& phase, int wave,
                                                int first_wave, int waves) {
#pragma unroll
  for (int k = 0; k < K; ++k) v[k] = wave_group_allreduce<64, SumOp>(v[k]);
  if ((threadIdx.x & 63) == 0) {
#pragma unroll
    for (int k = 0; k < K; ++k) red[phase][wave][k] = v[k];
  }
  __syncthreads();
  const int j = (int)threadIdx.x & 15;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const float p = red[phase][(first_wave + j) & 15][k];
    v[k] = wave_group_allreduce<16, SumOp>(j < waves ? p : 0.0f);
  }
  phase ^= 1;
}

// (as keep_packed, for float32 packs too: what was formed of the pack before is formed again, not held)
template <class T, int E>
__device__ __forceinline__ void waves_keep(Pack<T, E>& p) {
  typedef uint32_t raw_t __attribute__((ext_vector_type(4)));
  raw_t r = __builtin_bit_cast(raw_t, p.v);
  asm volatile("" : "+v"(r));
  p.v = __builtin_bit_cast(typename Pack<T, E>::vec_t, r);
}

template <class T, int E, int V>
struct WavesRow {
  float mu, rs;
  Pack<T, E> x[V], d[V];
};

// Forward; arithmetic of norm_fwd_resident_kernel.  The weights of a lane's columns are held for all rows.
template <class T, class WT, int V, int D, int THREADS, bool RMS>
__global__ void __launch_bounds__(THREADS)
norm_fwd_waves_kernel(const T* __restrict__ x, const WT* __restrict__ gamma, const WT* __restrict__ beta,
                      T* __restrict__ y, float* __restrict__ mean, float* __restrict__ rstd, int M, int N,
                      float eps, int waves) {
  constexpr int E = elems_per_pack<T>::value;
  static_assert(D >= 2, "one row set is worked on, the others are on their way");
  __shared__ float red[2][16][2];
  int phase = 0;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int slot = __builtin_amdgcn_readfirstlane(wave / waves), slots = (int)(blockDim.x >> 6) / waves;
  const int G = waves * 64, lane = (int)threadIdx.x - slot * G;
  const float fN = (float)N, inv_n = 1.0f / fN;
  const WavesPlace<T, V> at(lane, G, N);
  constexpr bool kWideWeights = V * E <= 8;
  Pack<WT, E> gp[V], bp[RMS ? 1 : V];
#pragma unroll
  for (int c = 0; c < V; ++c) {
    gp[c] = gamma ? Pack<WT, E>::load(gamma + at.off[c] / sizeof(T)) : Pack<WT, E>::splat(1.0f);
    if constexpr (!RMS)
      bp[c] = beta ? Pack<WT, E>::load(beta + at.off[c] / sizeof(T)) : Pack<WT, E>::zero();
  }

  const int nfull = M / slots, nrb = nfull + (nfull * slots < M ? 1 : 0), step = (int)gridDim.x;
  struct Row {
    Pack<T, E> x[V];
    float k;  // the centre of a 16-bit LayerNorm row
  };
  Row ring[D];
  auto row_of = [&](int rb) {
    const int row = (rb < nrb ? rb : 0) * slots + slot;
    return __builtin_amdgcn_readfirstlane(row < M ? row : M - 1);
  };
  auto fetch = [&](int rb, Row& o) {
    const T* xr = scalar_again(x + (int64_t)row_of(rb) * N);
#pragma unroll
    for (int c = 0; c < V; ++c) o.x[c] = Pack<T, E>::load_stream(global_at(xr, at[c]));
    if constexpr (!RMS && sizeof(T) == 2) {
      // the median of the row's first three elements (norm_fwd_resident_kernel)
      const float a = UniformElem<T>::load(xr, 0).value(), b = UniformElem<T>::load(xr, 1).value(),
                  c3 = UniformElem<T>::load(xr, 2).value();
      o.k = fmaxf(fminf(a, b), fminf(fmaxf(a, b), c3));
    }
  };
  auto work = [&](int rb, Row& w, auto last) {
    constexpr bool LAST = decltype(last)::value;
    const int row = __builtin_amdgcn_readfirstlane(rb * slots + slot);
    const bool real = !LAST || row < M;
    float mean0 = 0.0f, m1 = 0.0f, rs;
    auto mine = [&](int c, int i) { return c < V - 1 || i >= at.skip; };
    if constexpr (RMS) {
      float acc[1] = {0.0f};
#pragma unroll
      for (int c = 0; c < V; ++c)
#pragma unroll
        for (int i = 0; i < E; ++i) {
          const float v = w.x[c].get(i);
          const float a = fmaf(v, v, acc[0]);
          acc[0] = mine(c, i) ? a : acc[0];
        }
      waves_allreduce<1>(acc, red, phase, wave, slot * waves, waves);
      rs = row_rstd_of<T>(row_mean_of<T>(acc[0], fN, inv_n) + eps);
    } else {
      if constexpr (sizeof(T) == 2) {
        mean0 = w.k;
      } else {
        float acc[1] = {0.0f};
#pragma unroll
        for (int c = 0; c < V; ++c)
#pragma unroll
          for (int i = 0; i < E; ++i) acc[0] += mine(c, i) ? w.x[c].get(i) : 0.0f;
        waves_allreduce<1>(acc, red, phase, wave, slot * waves, waves);
        mean0 = acc[0] / fN;
      }
      // (an element that is another lane's counts as the centre: it adds nothing)
      float acc[2] = {0.0f, 0.0f};
#pragma unroll
      for (int c = 0; c < V; ++c) {
        waves_keep(w.x[c]);
#pragma unroll
        for (int i = 0; i < E; ++i) {
          const float d = mine(c, i) ? w.x[c].get(i) - mean0 : 0.0f;
          acc[0] += d;
          acc[1] = fmaf(d, d, acc[1]);
        }
      }
      waves_allreduce<2>(acc, red, phase, wave, slot * waves, waves);
      m1 = row_mean_of<T>(acc[0], fN, inv_n);
      float var = row_mean_of<T>(acc[1] - acc[0] * m1, fN, inv_n);
      var = var < 0.0f ? 0.0f : var;  // a select, not v_max_f32: a NaN row keeps NaN statistics
      rs = row_rstd_of<T>(var + eps);
    }
    if (!real) return;
    const float nm1rs = -m1 * rs;
    T* yr = scalar_again(y + (int64_t)row * N);
#pragma unroll
    for (int c = 0; c < V; ++c) {
      waves_keep(w.x[c]);
      if constexpr (!kWideWeights) {
        keep_packed(gp[c]);
        if constexpr (!RMS) keep_packed(bp[c]);
      }
      Pack<T, E> o;
#pragma unroll
      for (int i = 0; i < E; ++i) {
        const float v = w.x[c].get(i), g = gp[c].get(i);
        if constexpr (RMS)
          o.set(i, (v * rs) * g);
        else if constexpr (sizeof(T) == 2)
          o.set(i, fmaf(v - mean0, rs, nm1rs) * g + bp[c].get(i));
        else
          o.set(i, (((v - mean0) - m1) * rs) * g + bp[c].get(i));
      }
      o.store_stream(global_at(yr, at[c]));
    }
    if (lane == 0) {
      if constexpr (!RMS)
        if (mean) mean[row] = rs == rs ? mean0 + m1 : rs;
      if (rstd) rstd[row] = rs;
    }
  };

#pragma unroll
  for (int k = 0; k < D - 1; ++k) fetch((int)blockIdx.x + k * step, ring[k]);
  int rb = (int)blockIdx.x;
  while (rb + (D - 1) * step < nfull) {
#pragma unroll
    for (int k = 0; k < D; ++k) {
      fetch(rb + (D - 1) * step, ring[(k + D - 1) % D]);
      work(rb, ring[k], std::false_type{});
      rb += step;
    }
  }
  if (rb + (D - 1) * step < nrb) fetch(rb + (D - 1) * step, ring[D - 1]);
#pragma unroll
  for (int k = 0; k < D; ++k) {
    if (rb < nrb) {  // uniform
      work(rb, ring[k], std::true_type{});
      rb += step;
    }
  }
}

// Backward; arithmetic of norm_bwd_resident_kernel.  DX: dX is wanted, otherwise the column sums alone
// (with the same bits).  D register sets of rows; rows of a workgroup's slots
// past M read row M - 1 and only take part in the barrier.
template <class T, class WT, int V, int D, int THREADS, bool RMS, bool DX>
__global__ void __launch_bounds__(THREADS)
norm_bwd_waves_kernel(const T* __restrict__ dy, const T* __restrict__ x, const float* __restrict__ mean,
                      const float* __restrict__ rstd, const WT* __restrict__ gamma, T* dx,
                      float* __restrict__ part_dg, float* __restrict__ part_db, int M, int N,
                      int waves) {
  constexpr int E = elems_per_pack<T>::value;
  constexpr int NS = RMS ? 1 : 2;
  static_assert(D >= 2, "one row set is worked on, the others are on their way");
  __shared__ float red[2][16][2];
  __shared__ __align__(16) float fold[kWavesFoldFloats];
  int phase = 0;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int slot = __builtin_amdgcn_readfirstlane(wave / waves), slots = (int)(blockDim.x >> 6) / waves;
  const int G = waves * 64, lane = (int)threadIdx.x - slot * G;
  const float fN = (float)N, inv_n = 1.0f / fN;
  const bool want_cols = part_dg != nullptr;
  const WavesPlace<T, V> at(lane, G, N);
  // (weights of 16 elements a lane are widened once, more of them per row)
  constexpr bool kWideWeights = V * E <= 16;
  Pack<WT, E> gp[V];
  float dg[V][E], db[RMS ? 1 : V][RMS ? 1 : E];
#pragma unroll
  for (int c = 0; c < V; ++c) {
    gp[c] = gamma ? Pack<WT, E>::load(gamma + at.off[c] / sizeof(T)) : Pack<WT, E>::splat(1.0f);
#pragma unroll
    for (int i = 0; i < E; ++i) {
      dg[c][i] = 0.0f;
      if constexpr (!RMS) db[c][i] = 0.0f;
    }
  }

  // (32-bit row numbers: the scalar unit has no 64-bit comparisons, and rows chosen on the vector unit
  // would take two registers an address)
  const int nfull = M / slots, nrb = nfull + (nfull * slots < M ? 1 : 0), step = (int)gridDim.x;
  WavesRow<T, E, V> ring[D];
  auto fetch = [&](int rb, WavesRow<T, E, V>& o) {
    int row = (rb < nrb ? rb : 0) * slots + slot;
    row = __builtin_amdgcn_readfirstlane(row < M ? row : M - 1);
    o.mu = RMS ? 0.0f : uniform_load<float>(mean + row);
    o.rs = uniform_load<float>(rstd + row);
    // (scalar pointers the compiler cannot fold the lane's offset into: it would hold and add 64 bits a
    // lane, pack and tensor)
    const T* xr = scalar_again(x + (int64_t)row * N);
    const T* gr = scalar_again(dy + (int64_t)row * N);
#pragma unroll
    for (int c = 0; c < V; ++c) {
      o.x[c] = Pack<T, E>::load_stream(global_at(xr, at[c]));
      o.d[c] = Pack<T, E>::load_stream(global_at(gr, at[c]));
    }
  };
  auto work = [&](int rb, WavesRow<T, E, V>& w, auto last) {
    constexpr bool LAST = decltype(last)::value;
    const int row = __builtin_amdgcn_readfirstlane(rb * slots + slot);
    const bool real = !LAST || row < M;
    const float mu = w.mu, rs = w.rs, nmr = -mu * rs;
    auto xhat = [&](float v) { return RMS ? v * rs : (sizeof(T) == 2 ? fmaf(v, rs, nmr) : (v - mu) * rs); };
    float acc[2] = {0.0f, 0.0f};
    if (real) {
#pragma unroll
      for (int c = 0; c < V; ++c) {
        if constexpr (!kWideWeights) keep_packed(gp[c]);
#pragma unroll
        for (int i = 0; i < E; ++i) {
          const float xh = xhat(w.x[c].get(i)), gy = w.d[c].get(i);
          const float g = gy * gp[c].get(i);
          const bool mine = c < V - 1 || i >= at.skip;
          const float a0 = acc[0] + g, a1 = fmaf(g, xh, acc[1]);
          if constexpr (!RMS) acc[0] = mine ? a0 : acc[0];
          acc[1] = mine ? a1 : acc[1];
          dg[c][i] = fmaf(gy, xh, dg[c][i]);
          if constexpr (!RMS) db[c][i] += gy;
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if constexpr (!DX) return;
    waves_allreduce<2>(acc, red, phase, wave, slot * waves, waves);
    if (!real) return;
    T* dr = scalar_again(dx + (int64_t)row * N);
    // (the forms of norm_bwd_resident_kernel: float32 rows in the order that cancels exactly, 16-bit
    // rows regrouped)
    const float s1 = acc[0], s2 = acc[1];
    const float term1 = row_mean_of<T>(rs, fN, inv_n);
    const float ra = rs * (s2 * term1);
    const float cc = mu * ra - (RMS ? 0.0f : s1 * term1);
#pragma unroll
    for (int c = 0; c < V; ++c) {
      waves_keep(w.x[c]);
      waves_keep(w.d[c]);
      if constexpr (!kWideWeights) keep_packed(gp[c]);
      Pack<T, E> o;
#pragma unroll
      for (int i = 0; i < E; ++i) {
        const float g = w.d[c].get(i) * gp[c].get(i);
        float f;
        if constexpr (sizeof(T) == 2) {
          f = fmaf(w.x[c].get(i), -ra, fmaf(g, rs, cc));
        } else {
          f = fN * g;
          f -= xhat(w.x[c].get(i)) * s2;
          if constexpr (!RMS) f -= s1;
          f *= term1;
        }
        o.set(i, f);
      }
      o.store_stream(global_at(dr, at[c]));
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // (row blocks with a row in every slot as straight-line code: a test around a store would make the
  // waits for the rows on their way waits for the store)
#pragma unroll
  for (int k = 0; k < D - 1; ++k) fetch((int)blockIdx.x + k * step, ring[k]);
  int rb = (int)blockIdx.x;
  while (rb + (D - 1) * step < nfull) {
#pragma unroll
    for (int k = 0; k < D; ++k) {
      fetch(rb + (D - 1) * step, ring[(k + D - 1) % D]);
      work(rb, ring[k], std::false_type{});
      rb += step;
    }
  }
  // at most D row blocks are left, the last of them perhaps with rows missing
  if (rb + (D - 1) * step < nrb) fetch(rb + (D - 1) * step, ring[D - 1]);
#pragma unroll
  for (int k = 0; k < D; ++k) {
    if (rb < nrb) {  // uniform
      work(rb, ring[k], std::true_type{});
      rb += step;
    }
  }

  if (!want_cols) return;
  // The slots' column sums meet in the first slot's registers, one slot after the other through LDS
  // (16 bytes a lane and half pack, lanes side by side), which writes the workgroup's partial row.
  constexpr int Q = E / 4;
  float4* f4 = reinterpret_cast<float4*>(fold);
  for (int u = 1; u < slots; ++u) {
    __syncthreads();
    if (slot == u) {
#pragma unroll
      for (int c = 0; c < V; ++c)
#pragma unroll
        for (int h = 0; h < Q; ++h) {
          f4[(c * Q + h) * G + lane] =
              float4{dg[c][4 * h], dg[c][4 * h + 1], dg[c][4 * h + 2], dg[c][4 * h + 3]};
          if constexpr (!RMS)
            f4[((V + c) * Q + h) * G + lane] =
                float4{db[c][4 * h], db[c][4 * h + 1], db[c][4 * h + 2], db[c][4 * h + 3]};
        }
    }
    __syncthreads();
    if (slot == 0) {
#pragma unroll
      for (int c = 0; c < V; ++c)
#pragma unroll
        for (int h = 0; h < Q; ++h) {
          const float4 a = f4[(c * Q + h) * G + lane];
          dg[c][4 * h] += a.x, dg[c][4 * h + 1] += a.y, dg[c][4 * h + 2] += a.z, dg[c][4 * h + 3] += a.w;
          if constexpr (!RMS) {
            const float4 b = f4[((V + c) * Q + h) * G + lane];
            db[c][4 * h] += b.x, db[c][4 * h + 1] += b.y, db[c][4 * h + 2] += b.z, db[c][4 * h + 3] += b.w;
          }
        }
    }
  }
  if (slot != 0) return;
#pragma unroll
  for (int k = 0; k < NS; ++k) {
    float* out = (k == 0 ? part_dg : part_db) + (int64_t)blockIdx.x * N;
#pragma unroll
    for (int c = 0; c < V; ++c) {
      Pack<float, E> p;
#pragma unroll
      for (int i = 0; i < E; ++i) p.set(i, k == 0 ? dg[c][i] : db[RMS ? 0 : c][RMS ? 0 : i]);
      float* to = out + at.off[c] / sizeof(T);
      if (c < V - 1 || at.skip == 0) {
        p.store(to);
      } else {
#pragma unroll
        for (int i = 0; i < E; ++i)
          if (i >= at.skip) to[i] = p.get(i);
      }
    }
  }
}

}  // namespace rownorm
