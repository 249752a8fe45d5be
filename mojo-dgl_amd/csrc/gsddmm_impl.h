// Edge-parallel kernel behind gsddmm (included once per dtype).
//
// Elementwise ops: G consecutive lanes (power of two covering the output
// row's lanes, at most 64) own one edge, so a wavefront writes 64 / G
// consecutive output rows with coalesced stores; each lane gathers its VEC
// columns from the two operand rows selected by the targets (u[e], v[e] or
// e itself). As in gspmm the row is cut into runs of columns over which each
// operand is consecutive or one value, and a run's last lane ends with it, so
// every access is a whole vector at element alignment. One IEEE operation per element, so the result is bit-identical
// to the reference's (src/ported.mojo:295-328).
//
// dot: G lanes own one (edge, output column) pair and split the contracted
// axis `red` between them (VEC consecutive elements per lane per step; the
// last lane's end with the axis, the ones its neighbour holds counting as
// zero: 67 columns took 64 lanes of one float and 2.5 times as long), then
// add the G lane partials with a butterfly; each wavefront
// serves DOT_U rounds of pairs with their loads issued together. The reference keeps
// W lane partials and reduces them once (ported.mojo:273-293), so the two
// agree to rounding, not bit for bit.
#pragma once

#include "mdgl_kernels.h"

namespace mdgl {

template <class T>
struct GsddmmArgs {
  const int32_t* uids;
  const int32_t* vids;
  const T* lhs;
  const T* rhs;
  T* out;
  int64_t num_edges, dl, dr, dout, red;
  Bcast bc;
  int lt, rt, lmode, rmode, G, S;
  int run_len, lpg, nvec;  // columns per run, lanes per run, lanes per row
  int64_t num_tasks, num_waves, num_blocks;
};

__device__ __forceinline__ int64_t target_row(int t, const int32_t* u, const int32_t* v, int64_t e) {
  return t == TGT_U ? (int64_t)u[e] : (t == TGT_V ? (int64_t)v[e] : e);
}

template <class T, int VEC>
__device__ __forceinline__ void fetch_rt(const T* __restrict__ row, int mode, int off,
                                         T (&x)[VEC]) {
  if (mode == M_CONTIG) {
    load_any<false, T, VEC>(row + off, x);
  } else {
    const T s = row[off];
#pragma unroll
    for (int v = 0; v < VEC; ++v) x[v] = s;
  }
}

// A wavefront takes EW_U rounds of 64 / G edges (one slab of columns) and
// requests every round's operand rows before it computes, so each lane has
// 2 * EW_U row loads in flight.
constexpr int EW_U = 4;

template <class T, int OP, int VEC>
__global__ __launch_bounds__(BLOCK) void gsddmm_kernel(GsddmmArgs<T> a) {
  const int64_t blk = xcd_remap(blockIdx.x, a.num_blocks);
  const int lane = threadIdx.x & (WAVE - 1);
  const int64_t wave = blk * WAVES_PER_BLOCK + (threadIdx.x >> 6);
  if (wave >= a.num_waves) return;
  const int G = a.G;
  const int grp = lane / G, gl = lane % G;
  const int64_t slab = a.S > 1 ? wave % a.S : 0;
  const int64_t per_round = WAVE / G;
  const int64_t e0 = (a.S > 1 ? wave / a.S : wave) * EW_U * per_round + grp;
  const int li = (int)slab * G + gl;
  if (li >= a.nvec) return;
  const int run = a.lpg == a.nvec ? 0 : li / a.lpg, j = li - run * a.lpg;
  const int c = j * VEC < a.run_len - VEC ? j * VEC : a.run_len - VEC;
  const int64_t k0 = (int64_t)run * a.run_len + c;
  const int loff = (int)bcast_off(a.bc, k0, true), roff = (int)bcast_off(a.bc, k0, false);
  T x[EW_U][VEC], y[EW_U][VEC];
#pragma unroll
  for (int r = 0; r < EW_U; ++r) {
    const int64_t e = e0 + r * per_round;
    if (e < a.num_edges) {
      if constexpr (OP != OP_COPY_RHS)
        fetch_rt<T, VEC>(a.lhs + target_row(a.lt, a.uids, a.vids, e) * a.dl, a.lmode, loff, x[r]);
      if constexpr (OP != OP_COPY_LHS)
        fetch_rt<T, VEC>(a.rhs + target_row(a.rt, a.uids, a.vids, e) * a.dr, a.rmode, roff, y[r]);
    }
  }
#pragma unroll
  for (int r = 0; r < EW_U; ++r) {
    const int64_t e = e0 + r * per_round;
    if (e >= a.num_edges) break;
    T o[VEC];
#pragma unroll
    for (int v = 0; v < VEC; ++v) {
      T xv = T(0), yv = T(0);
      if constexpr (OP != OP_COPY_RHS) xv = x[r][v];
      if constexpr (OP != OP_COPY_LHS) yv = y[r][v];
      o[v] = message<OP>(xv, yv);
    }
    const int64_t base = e * a.dout + k0;
    store_stream_any<T, VEC>(a.out + base, o);
  }
}

// dot: tasks are (edge, output column) pairs, G lanes per task. A wavefront
// takes DOT_U rounds of 64 / G tasks; when the contracted axis fits in one
// vector per lane (red <= G * VEC) the loads of all rounds are issued before
// the first product, so each lane has 2 * DOT_U row loads in flight.
constexpr int DOT_U = 4;

// VEC elements of two rows from k on; with TAIL (an axis that VEC does not divide,
// red >= VEC) from min(k, red - VEC) on, those before k zero. For floats fixed at
// compile time: one register over 64 is a wavefront per SIMD less (20M dots of 128
// floats: 3,289 us with the test at run time, 3,121 without; doubles take more than
// 64 either way and are 1 to 5 % faster tested at run time).
enum { TAIL_NO = 0, TAIL_YES = 1, TAIL_ASK = 2 };
template <class T, int VEC, int TAIL>
__device__ __forceinline__ void dot_load(const T* __restrict__ l, const T* __restrict__ r, int64_t k,
                                         int64_t red, T (&x)[VEC], T (&y)[VEC]) {
  const bool tail = TAIL == TAIL_YES || (TAIL == TAIL_ASK && red % VEC != 0);
  const int64_t at = tail && k > red - VEC ? red - VEC : k;
  typedef T V __attribute__((ext_vector_type(VEC == 1 ? 2 : VEC), aligned(sizeof(T))));
  typedef const __attribute__((address_space(1))) V GV;
  if constexpr (VEC == 1) {
    x[0] = load_global(l + at);
    y[0] = load_global(r + at);
  } else {
    const V a = *(GV*)(l + at), b = *(GV*)(r + at);
#pragma unroll
    for (int v = 0; v < VEC; ++v) {
      x[v] = a[v];
      y[v] = b[v];
    }
    if (tail) {
      const int dup = (int)(k - at);
#pragma unroll
      for (int v = 0; v < VEC; ++v) {
        x[v] = v < dup ? T(0) : x[v];
        y[v] = v < dup ? T(0) : y[v];
      }
    }
  }
}

template <class T, int VEC, int TAIL>
__device__ __forceinline__ T dot_part(const T* __restrict__ l, const T* __restrict__ r,
                                      int64_t k0, int64_t red, int64_t step) {
  T part = T(0);
  for (int64_t k = k0; k < red; k += step) {
    T xv[VEC], yv[VEC];
    dot_load<T, VEC, TAIL>(l, r, k, red, xv, yv);
#pragma unroll
    for (int v = 0; v < VEC; ++v) part = part + xv[v] * yv[v];
  }
  return part;
}

template <class T, int VEC, int TAIL>
__global__ __launch_bounds__(BLOCK) void gsddmm_dot_kernel(GsddmmArgs<T> a) {
  const int64_t blk = xcd_remap(blockIdx.x, a.num_blocks);
  const int lane = threadIdx.x & (WAVE - 1);
  const int64_t wave = blk * WAVES_PER_BLOCK + (threadIdx.x >> 6);
  if (wave >= a.num_waves) return;  // uniform per wavefront
  const int G = a.G;
  const int grp = lane / G, gl = lane % G;
  const int64_t per_round = WAVE / G;
  const int64_t k0 = (int64_t)gl * VEC;
  int64_t task[DOT_U];
  const T* lp[DOT_U];
  const T* rp[DOT_U];
#pragma unroll
  for (int u = 0; u < DOT_U; ++u) {
    task[u] = (wave * DOT_U + u) * per_round + grp;
    lp[u] = rp[u] = nullptr;
    if (task[u] < a.num_tasks) {
      if (a.dout == 1) {
        // one output column per edge (u_dot_v on (n, d) rows): the task is
        // the edge and the broadcast offsets are 0 -- no 64-bit divides
        lp[u] = a.lhs + target_row(a.lt, a.uids, a.vids, task[u]) * a.dl;
        rp[u] = a.rhs + target_row(a.rt, a.uids, a.vids, task[u]) * a.dr;
      } else {
        // (32-bit where it fits: a 64-bit divide is several times the instructions)
        const int64_t e = a.num_tasks < (int64_t(1) << 32)
                              ? (int64_t)((uint32_t)task[u] / (uint32_t)a.dout)
                              : task[u] / a.dout;
        const int64_t col = task[u] - e * a.dout;
        lp[u] = a.lhs + target_row(a.lt, a.uids, a.vids, e) * a.dl +
                bcast_off(a.bc, col, true) * a.red;
        rp[u] = a.rhs + target_row(a.rt, a.uids, a.vids, e) * a.dr +
                bcast_off(a.bc, col, false) * a.red;
      }
    }
  }
  T part[DOT_U];
  if (a.red <= (int64_t)G * VEC) {
    T xv[DOT_U][VEC], yv[DOT_U][VEC];
#pragma unroll
    for (int u = 0; u < DOT_U; ++u) {
      if (lp[u] && k0 < a.red) {
        dot_load<T, VEC, TAIL>(lp[u], rp[u], k0, a.red, xv[u], yv[u]);
      } else {
#pragma unroll
        for (int v = 0; v < VEC; ++v) xv[u][v] = yv[u][v] = T(0);
      }
    }
#pragma unroll
    for (int u = 0; u < DOT_U; ++u) {
      T pu = T(0);
#pragma unroll
      for (int v = 0; v < VEC; ++v) pu = pu + xv[u][v] * yv[u][v];
      part[u] = pu;
    }
  } else {
#pragma unroll
    for (int u = 0; u < DOT_U; ++u)
      part[u] = lp[u] ? dot_part<T, VEC, TAIL>(lp[u], rp[u], k0, a.red, (int64_t)G * VEC) : T(0);
  }
  // butterfly inside the lane group; every lane of the wavefront runs it
#pragma unroll
  for (int u = 0; u < DOT_U; ++u) part[u] = group_sum(part[u], G);
  if (G >= DOT_U) {
    // the wavefront's DOT_U * 64 / G tasks are consecutive: lane t takes
    // task wave * nt + t from its group's lanes and the results leave as one
    // coalesced store (one partial-line store per round wrote every output
    // line back about five times)
    const int pr = WAVE / G, nt = DOT_U * pr;
    const int su = lane / pr, src = (lane % pr) * G;
    T val = T(0);
#pragma unroll
    for (int u = 0; u < DOT_U; ++u) {
      const T s = __shfl(part[u], src);
      if (su == u) val = s;
    }
    const int64_t t = wave * nt + lane;
    if (lane < nt && t < a.num_tasks) a.out[t] = val;
  } else {
#pragma unroll
    for (int u = 0; u < DOT_U; ++u)
      if (lp[u] && gl == 0) __builtin_nontemporal_store(part[u], a.out + task[u]);
  }
}

template <class T, int VEC>
hipError_t launch_gsddmm_vec(const GsddmmParams& p) {
  GsddmmArgs<T> a;
  a.uids = p.uids;
  a.vids = p.vids;
  a.lhs = static_cast<const T*>(p.lhs);
  a.rhs = static_cast<const T*>(p.rhs);
  a.out = static_cast<T*>(p.out);
  a.num_edges = p.num_edges;
  a.dl = p.dl;
  a.dr = p.dr;
  a.dout = p.dout;
  a.red = p.red;
  a.bc = p.bc;
  a.lt = p.lt;
  a.rt = p.rt;
  a.lmode = p.lmode;
  a.rmode = p.rmode;
  a.run_len = (int)p.run_len;
  a.lpg = p.lpg;
  a.nvec = p.run_len > 0 ? (int)(p.dout / p.run_len * p.lpg) : 0;
  if (p.op == OP_DOT) {
    const int64_t nvec = (p.red + VEC - 1) / VEC;
    int G = 1;
    while (G < nvec && G < WAVE) G <<= 1;
    a.G = G;
    a.S = 1;
    a.num_tasks = p.num_edges * p.dout;
    const int64_t per_wave = (WAVE / G) * DOT_U;
    a.num_waves = (a.num_tasks + per_wave - 1) / per_wave;
  } else {
    const int64_t nvec = a.nvec;
    int G = 1;
    while (G < nvec && G < WAVE) G <<= 1;
    a.G = G;
    a.S = (int)((nvec + G - 1) / G);
    a.num_tasks = p.num_edges;
    const int64_t per_wave = (WAVE / G) * EW_U;
    a.num_waves = ((p.num_edges + per_wave - 1) / per_wave) * a.S;
  }
  a.num_blocks = (a.num_waves + WAVES_PER_BLOCK - 1) / WAVES_PER_BLOCK;
  if (a.num_blocks == 0) return hipSuccess;
  const dim3 grid((unsigned)a.num_blocks), block(BLOCK);
  switch (p.op) {
    case OP_ADD: hipLaunchKernelGGL((gsddmm_kernel<T, OP_ADD, VEC>), grid, block, 0, p.stream, a); break;
    case OP_SUB: hipLaunchKernelGGL((gsddmm_kernel<T, OP_SUB, VEC>), grid, block, 0, p.stream, a); break;
    case OP_MUL: hipLaunchKernelGGL((gsddmm_kernel<T, OP_MUL, VEC>), grid, block, 0, p.stream, a); break;
    case OP_DIV: hipLaunchKernelGGL((gsddmm_kernel<T, OP_DIV, VEC>), grid, block, 0, p.stream, a); break;
    case OP_COPY_LHS:
      hipLaunchKernelGGL((gsddmm_kernel<T, OP_COPY_LHS, VEC>), grid, block, 0, p.stream, a);
      break;
    case OP_COPY_RHS:
      hipLaunchKernelGGL((gsddmm_kernel<T, OP_COPY_RHS, VEC>), grid, block, 0, p.stream, a);
      break;
    case OP_DOT:
      if constexpr (VEC == 1 || sizeof(T) == 8)
        hipLaunchKernelGGL((gsddmm_dot_kernel<T, VEC, VEC == 1 ? TAIL_NO : TAIL_ASK>), grid, block,
                           0, p.stream, a);
      else if (p.red % VEC == 0)
        hipLaunchKernelGGL((gsddmm_dot_kernel<T, VEC, TAIL_NO>), grid, block, 0, p.stream, a);
      else
        hipLaunchKernelGGL((gsddmm_dot_kernel<T, VEC, TAIL_YES>), grid, block, 0, p.stream, a);
      break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

template <class T>
hipError_t launch_gsddmm(const GsddmmParams& p) {
  if (p.vec == VecOf<T>::n) return launch_gsddmm_vec<T, VecOf<T>::n>(p);
  if constexpr (VecOf<T>::n == 4) {
    if (p.vec == 2) return launch_gsddmm_vec<T, 2>(p);
  }
  return launch_gsddmm_vec<T, 1>(p);
}

}  // namespace mdgl

#define MDGL_INSTANTIATE_GSDDMM(T) \
  template hipError_t mdgl::launch_gsddmm<T>(const mdgl::GsddmmParams&);
