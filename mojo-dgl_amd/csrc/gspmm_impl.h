// CSR reduce kernel behind gspmm (included once per (dtype, reducer)
// translation unit).
//
// Work list. A "unit" is either a chunk of a heavy row (written as a
// partial) or a whole row (rows longer than chunk_len are skipped there).
// The first chunk_blocks workgroups take the chunks (so they start first),
// the remaining workgroups the rows; both ranges go through the XCD remap,
// so each XCD serves a contiguous run of units and the rows of a block of
// neighbouring destinations share its L2 (a community graph's chunks dealt
// round-robin over the XCDs held its L2 hit rate at 70 %). A unit is processed
// by G consecutive lanes (G = the power of two covering the row's lanes, at
// most 64 and at least 16, or 2 or 4 for rows of few edges), so a wavefront packs
// 64 / G units; output rows wider than
// 64 lanes are cut into S slabs, one wavefront per slab.
//
// Lane columns. A row is made of dout / L runs of L columns over which each
// operand is either consecutive or one value (run_len, from the broadcast;
// one run when nothing broadcasts). Each run takes `lpg` lanes of VEC columns;
// when VEC does not divide L the run's last lane starts VEC columns before its
// end and so shares some with its neighbour (both compute and store the same
// values). Every load and store is then a whole vector, at element alignment:
// one float per lane made 47-column rows (47 lanes, 4 bytes each) move a
// quarter of the bytes per instruction.
//
// Fold order. Each lane owns VEC output columns and folds its unit's CSR
// slots one after the other, in CSR order: for a row that is not split this
// is exactly the reference's sequential fold (src/ported.mojo:392-422), so
// sum, mean, max and min values are bit-identical to the CPU kernel in the
// same precision. Split rows fold each chunk in order and then fold the
// chunk partials in chunk order; max/min remain exact (strict comparison,
// the earlier chunk wins ties, so the arg is still the first edge in CSR
// order reaching the value).
//
// Memory. U edges are in flight per lane, their ids loaded a batch ahead.
// How the ids reach a unit's lanes depends on G:
//   G = 64      64 ids per load, one per lane, broadcast by v_readlane into
//               scalar registers;
//   G = 16, 32  16 ids per load, the same 16 in each DPP row of the unit, row
//               offsets formed once by the lane that loaded the id and
//               broadcast by DPP (row_newbcast, one VALU operation per word;
//               ds_bpermute with a 64-bit multiply per lane and edge took 45
//               instructions per two edges).
//   G < 16      every lane loads the ids of its own row, U at a time (one load
//               each, the same address across a unit).
// The caller says which of the last two a row of fewer than 16 lanes takes, by
// the edges its rows have on average. With many, 16 lanes, those past the row
// repeating its last columns: a wavefront of 8 to 64 rows waits for the longest
// of them (4 columns on 4.9M edges of a power-law graph, 16 a row: 1,121 us with
// an edge in flight per lane of a packed row, 398 with 8, 192 at 16 lanes). With
// few, the lanes it needs, at least 2 or 4: most rows end within the first U
// edges, and 16 lanes would be 4 rows a wavefront where 16 or 32 fit (one column,
// 2 edges a row, 4M rows: 311 us for copy_u, 113 with 2 lanes, 118 with one lane
// and one edge in flight; 4 random edges a row: 362 and 223; MDGL_ROW_LANES_2 and
// _4, whose caller has the line and both sides).
// Ids past a row repeat its last one, so id loads need no branch; operand rows
// are requested and folded without one except in the batch that ends a row.
#pragma once

#include <type_traits>
#include <utility>

#include "mdgl_kernels.h"

namespace mdgl {

constexpr int M_DYN = 3;
constexpr int M_SCALAR = 4;  // edge operand of one value per edge (dr == 1)

template <class T>
struct GspmmArgs {
  const int32_t* indptr;
  const int32_t* indices;
  const int32_t* eid;
  const int32_t* deg;
  const T* lhs;
  const T* rhs;
  T* out;
  int32_t* arg_u;
  int32_t* arg_e;
  int64_t num_rows, dl, dr, dout;
  int64_t lstride;  // elements between lhs rows
  Bcast bc;
  int lmode, rmode, flags, gshift, S;
  int run_len, lpg, nvec;  // columns per run, lanes per run, lanes per row
  int64_t num_chunks;
  const int32_t* chunk_row;
  const int32_t* chunk_start;
  int chunk_len;
  T* part_val;
  int32_t* part_u;
  int32_t* part_e;
  int64_t chunk_waves, row_waves, chunk_blocks, num_blocks;
  int64_t first_block;  // of this launch (launch_gspmm_op)
  // waves per slab (with several, every unit's slab s comes before slab s + 1,
  // so the rows of neighbouring units share cache lines across wavefronts)
  int64_t chunk_uwaves, row_uwaves;
  const int32_t* sel;  // selected sum (see GspmmParams), else null
  const T* rowop;  // dot output (see GspmmParams), else null
  T* dot_out;
  int dot_lanes;
  const int32_t* rows;  // listed rows (see GspmmParams), else null
  int64_t row_limit;
};

// Edge rows of consecutive columns from this many bytes on are read past the
// caches: each is read once, and so does not displace source rows that other
// edges will gather. Narrower ones share their lines with other edges' rows,
// which the caches may still hold when those are read. Time of streamed reads
// over cached ones, float32 sums by edge id, copy_e and u_mul_e, each warm and
// after the caches were overwritten:
//   bytes        1M edges                6M edges                60M edges
//     16   1.33 1.14  1.31 1.13    1.31 1.29  1.26 1.16    1.05 1.23  1.01 1.01
//     64   1.29 0.92  1.28 0.90    1.23 0.96  1.03 0.92    0.99 1.03  0.90 0.90
//     96   1.23 0.90  1.06 0.90    1.12 0.94  0.96 0.91    0.97 1.01  0.87 0.87
//    128   1.25 0.65  1.21 0.76    0.96 0.81  0.97 0.89    0.96 0.98  0.85 0.86
//    256   1.19 0.55  0.94 0.67    0.96 0.87  0.99 0.92      -
// (100,000 edges: 1.0 warm at any width, after an overwrite 1.09 at 16 bytes, 0.98
// at 96, 0.74 at 256.)
constexpr int64_t STREAM_ROW_BYTES = 96;

// The VEC columns a lane reads from an operand row (off: their offsets; only
// off[0] unless the mode is gather), past the caches with STREAM; rows of
// consecutive columns not with NEAR.
template <class T, int VEC, int M, bool STREAM, bool NEAR>
__device__ __forceinline__ void fetch(const T* __restrict__ row, int mode_rt, const int (&off)[VEC],
                                      T (&x)[VEC]) {
  const int m = (M == M_DYN) ? mode_rt : M;
  if (m == M_CONTIG) {
    load_any<STREAM && !NEAR, T, VEC>(row + off[0], x);
  } else if (m == M_SPLAT) {
    const T s = STREAM ? __builtin_nontemporal_load(row + off[0]) : row[off[0]];
#pragma unroll
    for (int v = 0; v < VEC; ++v) x[v] = s;
  } else {
#pragma unroll
    for (int v = 0; v < VEC; ++v)
      x[v] = STREAM ? __builtin_nontemporal_load(row + off[v]) : row[off[v]];
  }
}

// Lane N of each DPP row of 16 lanes, to all 16 of them.
template <int N>
__device__ __forceinline__ int row_bcast(int v) {
  return __builtin_amdgcn_mov_dpp(v, 0x150 + N, 0xF, 0xF, false);
}
template <int N>
__device__ __forceinline__ float row_bcast(float v) {
  return __int_as_float(row_bcast<N>(__float_as_int(v)));
}
typedef int32_t int_pair __attribute__((ext_vector_type(2)));
template <int N>
__device__ __forceinline__ int64_t row_bcast(int64_t v) {
  const int_pair p = __builtin_bit_cast(int_pair, v);  // a register pair, no shifts
  const int_pair q = {row_bcast<N>(p[0]), row_bcast<N>(p[1])};
  return __builtin_bit_cast(int64_t, q);
}
template <int N>
__device__ __forceinline__ double row_bcast(double v) {
  return __longlong_as_double(row_bcast<N>((int64_t)__double_as_longlong(v)));
}

// A lambda kept out of line would put the arrays it captures in memory.
#define MDGL_INLINE __attribute__((always_inline))

// f(0), ..., f(N - 1) with the number known to the compiler.
template <int... I, class F>
__device__ __forceinline__ void for_each_of(std::integer_sequence<int, I...>, F f) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void for_each(F f) {
  for_each_of(std::make_integer_sequence<int, N>{}, f);
}

// How ids reach the lanes of a unit (see the top): by G.
enum { LAY_ROW = 0, LAY_WIDE = 1, LAY_LANE = 2 };

// DOT: 1 beside the sum, 2 alone (nothing folded or written but the dots).
// NEAR: edge rows are read through the caches.
template <class T, int OP, int RED, int VEC, int LM, int RM, int LAY, int DOT = 0,
          bool SEL = false, bool NEAR = false>
__device__ __forceinline__ void gspmm_body(const GspmmArgs<T>& a, bool chunk, int64_t wave,
                                           int lane) {
  // edges in flight per lane: 8 (4 in the dot pass, whose per-edge
  // butterflies already hide the loads; 8 there cost 14 %)
  constexpr int U = DOT == 1 ? 4 : 8;
  constexpr bool ARG = (RED == RED_MAX || RED == RED_MIN);
  constexpr bool HAS_L = OP != OP_COPY_RHS, HAS_R = OP != OP_COPY_LHS;
  const int G = LAY == LAY_WIDE ? WAVE : 1 << a.gshift;
  const int grp = LAY == LAY_WIDE ? 0 : lane >> a.gshift, gl = lane & (G - 1);
  // (a 64-bit divide is about a hundred instructions, and rows of a few
  // edges run few more: none where one slab or one run makes it 1)
  int slab = 0;
  if (a.S > 1) {
    const int64_t uw = chunk ? a.chunk_uwaves : a.row_uwaves;
    slab = (int)(wave / uw);
    wave -= slab * uw;
  }
  const int64_t unit = LAY == LAY_WIDE ? wave : (wave << (6 - a.gshift)) + grp;

  // ---- resolve the unit to a CSR slot range
  bool ok = unit < (chunk ? a.num_chunks : a.num_rows);
  int64_t row = 0;
  int start = 0, stop = 0;
  if (ok) {
    if (chunk) {
      row = a.chunk_row[unit];
      start = a.chunk_start[unit];
      const int end = a.indptr[row + 1];
      stop = (end - start > a.chunk_len) ? start + a.chunk_len : end;
    } else {
      row = unit;
      if (a.rows) {
        row = a.rows[unit];
        if (row < 0 || row >= a.row_limit) ok = false;  // not a row of the graph: skipped
      }
      if (ok) {
        start = a.indptr[row];
        stop = a.indptr[row + 1];
        if (stop - start > a.chunk_len) ok = false;  // heavy: done by chunks + combine
      }
    }
  }

  // ---- this lane's output columns and operand offsets
  int li = slab * G + gl;
  const bool feat_ok = li < a.nvec;
  if (!feat_ok) li = a.nvec - 1;  // a lane past the row repeats its last one, unwritten
  int64_t k0 = 0;
  int dup = 0;  // leading columns that the run's previous lane also holds
  {
    const int run = a.lpg == a.nvec ? 0 : li / a.lpg, j = li - run * a.lpg;
    const int c = j * VEC < a.run_len - VEC ? j * VEC : a.run_len - VEC;
    k0 = (int64_t)run * a.run_len + c;
    dup = j * VEC - c < VEC ? j * VEC - c : VEC;
  }
  int loff[VEC], roff[VEC];
#pragma unroll
  for (int v = 0; v < VEC; ++v) {
    const bool each = (LM == M_DYN && RM == M_DYN);
    loff[v] = roff[v] = 0;
    if (a.bc.nd == 1) {
      loff[v] = (int)((k0 + v) * a.bc.lstride[0]);
      roff[v] = (int)((k0 + v) * a.bc.rstride[0]);
    } else if (v == 0 || each) {
      loff[v] = (int)bcast_off(a.bc, k0 + v, true);
      roff[v] = (int)bcast_off(a.bc, k0 + v, false);
    }
  }

  // DOT: this row's own feature columns, dotted with every gathered lhs row
  T rowv[VEC];
  if constexpr (DOT) {
#pragma unroll
    for (int v = 0; v < VEC; ++v) rowv[v] = T(0);
    if (ok) load_any<false, T, VEC>(a.rowop + row * a.dout + k0, rowv);
  }

  T acc[VEC];
  int at[VEC];  // max / min: the CSR slot selected (-1: none yet)
#pragma unroll
  for (int v = 0; v < VEC; ++v) {
    acc[v] = seed<T>(RED);
    at[v] = -1;
  }

  const bool ident = a.flags & F_EID_IDENTITY;
  const int n = ok ? stop - start : 0;
  // a scalar edge operand (one value per edge, splatted over the columns) is
  // loaded with the ids, one edge per lane, and broadcast like them
  constexpr bool SCALAR = RM == M_SCALAR && HAS_R;
  constexpr bool ROW_R = HAS_R && !SCALAR;
  // the edge operand may come in CSR slot order (row i of rhs for slot i)
  const bool rhs_csr = a.flags & F_RHS_CSR;
  const bool need_e = SEL || (HAS_R && !rhs_csr && !ident);

  const char* const lbase = reinterpret_cast<const char*>(a.lhs + loff[0]);
  const char* const rbase = reinterpret_cast<const char*>(a.rhs + roff[0]);
  // SEL: the selection's rows lie as the lhs rows do (int32, dl == dout)
  const char* const sbase = reinterpret_cast<const char*>(a.sel + (SEL ? k0 : 0));
#pragma unroll
  for (int v = VEC - 1; v >= 0; --v) {  // from here on relative to the lane's first column
    loff[v] -= loff[0];
    roff[v] -= roff[0];
  }

  // One batch is the edges of U slots, of which the first `rem` are the
  // unit's (all U with FULL: no branch per edge). `lo_of` / `ro_of` give the
  // byte offset of edge u's operand rows, `w_of` its value of a scalar edge
  // operand, `e_of` its edge id (SEL only). A broadcast right
  // before its request keeps one offset live instead of U of them (32
  // registers, and with them two wavefronts per SIMD).
  auto batch = [&](auto full, int slot0, int rem, auto lo_of, auto ro_of, auto w_of,
                   auto e_of) MDGL_INLINE {
    constexpr bool FULL = decltype(full)::value;
    T x[U][VEC], y[U][VEC], w[U];
    int32_t sel[U][VEC];
    auto request = [&](auto iu) MDGL_INLINE {
      constexpr int u = decltype(iu)::value;
      if constexpr (HAS_L) {
        const int64_t lo = lo_of(iu);
        fetch<T, VEC, LM, false, false>(reinterpret_cast<const T*>(lbase + lo), a.lmode, loff, x[u]);
        if constexpr (SEL)
          load_any<false, int32_t, VEC>(
              reinterpret_cast<const int32_t*>(sbase + lo / (int64_t)(sizeof(T) / 4)), sel[u]);
      }
      if constexpr (ROW_R)
        fetch<T, VEC, RM, true, NEAR>(reinterpret_cast<const T*>(rbase + ro_of(iu)), a.rmode, roff,
                                      y[u]);
    };
    auto fold = [&](auto iu) MDGL_INLINE {
      constexpr int u = decltype(iu)::value;
      int eid = 0;
      if constexpr (SEL) eid = e_of(iu);
#pragma unroll
      for (int v = 0; v < VEC; ++v) {
        T xv = T(0), yv = T(0);
        if constexpr (HAS_L) xv = x[u][v];
        if constexpr (SCALAR) yv = w[u];
        else if constexpr (HAS_R) yv = y[u][v];
        T m = message<OP>(xv, yv);
        if constexpr (SEL) m = sel[u][v] == eid ? m : T(0);
        if constexpr (RED == RED_MAX) {
          if (m > acc[v]) { acc[v] = m; at[v] = slot0 + u; }
        } else if constexpr (RED == RED_MIN) {
          if (m < acc[v]) { acc[v] = m; at[v] = slot0 + u; }
        } else {
          acc[v] = acc[v] + m;
        }
      }
    };
    // DOT: the lanes' partial dots per edge and column group, then the sum
    // over the group's lanes; the group's first lane writes
    auto dot = [&](auto iu) MDGL_INLINE {
      constexpr int u = decltype(iu)::value;
      T pd = T(0);
#pragma unroll
      for (int v = 0; v < VEC; ++v) pd = v < dup ? pd : pd + x[u][v] * rowv[v];
      pd = group_sum(pd, a.dot_lanes);
      if (feat_ok && (gl & (a.dot_lanes - 1)) == 0)
        a.dot_out[(int64_t)(slot0 + u) * a.dr + li / a.dot_lanes] = pd;
    };
    for_each<U>([&](auto iu) MDGL_INLINE {
      if (FULL || decltype(iu)::value < rem) request(iu);
    });
    if constexpr (SCALAR)
      for_each<U>([&](auto iu) MDGL_INLINE { w[decltype(iu)::value] = w_of(iu); });
    if constexpr (DOT)
      for_each<U>([&](auto iu) MDGL_INLINE {
        if (FULL || decltype(iu)::value < rem) dot(iu);
      });
    if constexpr (DOT != 2)
      for_each<U>([&](auto iu) MDGL_INLINE {
        if (FULL || decltype(iu)::value < rem) fold(iu);
      });
  };
  const int64_t lbytes = a.lstride * (int64_t)sizeof(T), rbytes = a.dr * (int64_t)sizeof(T);

  if constexpr (LAY == LAY_ROW) {
    // ---- 16 ids per load, broadcast by DPP: a unit's lanes (whole DPP rows)
    // take every branch together, so the lane that holds an id is active
    const int nmax = wave_max_int(n);
    int my_s = 0, my_e = 0;
    // past the unit's slots its last one; slot 0 for a unit without any
    auto fill = [&](int base) MDGL_INLINE {
      const int p = base + (lane & 15);
      const int i = n > 0 ? start + (p < n ? p : n - 1) : 0;
      if constexpr (HAS_L) my_s = a.indices[i];
      if constexpr (HAS_R || SEL) {
        my_e = i;
        if (need_e) my_e = a.eid[i];
      }
    };
    if (nmax > 0) fill(0);
    for (int base = 0; base < nmax; base += 16) {
      int64_t my_lo = 0, my_ro = 0;
      T my_w = T(0);
      const int cur_e = my_e;
      if constexpr (HAS_L) my_lo = (int64_t)my_s * lbytes;
      if constexpr (SCALAR) my_w = a.rhs[my_e];
      else if constexpr (HAS_R) my_ro = (int64_t)my_e * rbytes;
      if (base + 16 < nmax) fill(base + 16);
      for_each<16 / U>([&](auto part) MDGL_INLINE {
        constexpr int F = decltype(part)::value * U;
        const int rem = n - base - F;
        if (rem <= 0) return;
        auto lo_of = [&](auto iu) MDGL_INLINE { return row_bcast<F + decltype(iu)::value>(my_lo); };
        auto ro_of = [&](auto iu) MDGL_INLINE { return row_bcast<F + decltype(iu)::value>(my_ro); };
        auto w_of = [&](auto iu) MDGL_INLINE { return row_bcast<F + decltype(iu)::value>(my_w); };
        auto e_of = [&](auto iu) MDGL_INLINE { return row_bcast<F + decltype(iu)::value>(cur_e); };
        // a divide is a dozen instructions: one body for all rows of the wavefront
        // (elsewhere the rows with a whole batch save its tests)
        const bool whole = OP == OP_DIV ? __builtin_amdgcn_ballot_w64(rem < U) == 0 : rem >= U;
        if (whole)
          batch(std::true_type{}, start + base + F, U, lo_of, ro_of, w_of, e_of);
        else
          batch(std::false_type{}, start + base + F, rem, lo_of, ro_of, w_of, e_of);
      });
    }
  } else if constexpr (LAY == LAY_LANE) {
    // ---- every lane loads its own row's ids, those of a batch at a time
    for (int base = 0; base < n; base += U) {
      int32_t s[U], e[U];
      T w[U];
      const int rem = n - base;
      for_each<U>([&](auto iu) MDGL_INLINE {
        constexpr int u = decltype(iu)::value;
        s[u] = e[u] = 0;
        w[u] = T(0);
        if (u < rem) {
          const int i = start + base + u;
          if constexpr (HAS_L) s[u] = a.indices[i];
          if constexpr (HAS_R || SEL) {
            e[u] = i;
            if (need_e) e[u] = a.eid[i];
          }
        }
      });
      if constexpr (SCALAR)
        for_each<U>([&](auto iu) MDGL_INLINE {
          if (decltype(iu)::value < rem) w[decltype(iu)::value] = a.rhs[e[decltype(iu)::value]];
        });
      auto lo_of = [&](auto iu) MDGL_INLINE { return (int64_t)s[decltype(iu)::value] * lbytes; };
      auto ro_of = [&](auto iu) MDGL_INLINE { return (int64_t)e[decltype(iu)::value] * rbytes; };
      auto w_of = [&](auto iu) MDGL_INLINE { return w[decltype(iu)::value]; };
      auto e_of = [&](auto iu) MDGL_INLINE { return e[decltype(iu)::value]; };
      batch(std::false_type{}, start + base, rem, lo_of, ro_of, w_of, e_of);
    }
  } else {
    // ---- 64 ids per load, broadcast by v_readlane (n is uniform here)
    const int un = __builtin_amdgcn_readfirstlane(n);
    const int ustart = __builtin_amdgcn_readfirstlane(start);
    int my_s = 0, my_e = 0;
    auto fill = [&](int base) MDGL_INLINE {
      const int p = base + lane;
      const int i = ustart + (p < un ? p : un - 1);
      if constexpr (HAS_L) my_s = __builtin_nontemporal_load(a.indices + i);
      if constexpr (HAS_R || SEL) {
        my_e = i;
        if (need_e) my_e = __builtin_nontemporal_load(a.eid + i);
      }
    };
    if (un > 0) fill(0);
    for (int base = 0; base < un; base += WAVE) {
      const int cs = my_s, ce = my_e;
      T my_w = T(0);
      if constexpr (SCALAR) my_w = a.rhs[ce];
      if (base + WAVE < un) fill(base + WAVE);
      const int cnt = un - base < WAVE ? un - base : WAVE;
      for (int j = 0; j < cnt; j += U) {
        auto lo_of = [&](auto iu) MDGL_INLINE {
          return (int64_t)readlane_int(cs, j + decltype(iu)::value) * lbytes;
        };
        auto ro_of = [&](auto iu) MDGL_INLINE {
          return (int64_t)readlane_int(ce, j + decltype(iu)::value) * rbytes;
        };
        auto w_of = [&](auto iu) MDGL_INLINE {
          return readlane_val(my_w, (j + decltype(iu)::value) & (WAVE - 1));
        };
        auto e_of = [&](auto iu) MDGL_INLINE { return readlane_int(ce, j + decltype(iu)::value); };
        if (cnt - j >= U)
          batch(std::true_type{}, ustart + base + j, U, lo_of, ro_of, w_of, e_of);
        else
          batch(std::false_type{}, ustart + base + j, cnt - j, lo_of, ro_of, w_of, e_of);
      }
    }
  }

  if (DOT == 2 || !ok || !feat_ok) return;
  if (chunk) {
    const int64_t o = unit * a.dout + k0;
#pragma unroll
    for (int v = 0; v < VEC; ++v) {
      a.part_val[o + v] = acc[v];
      if constexpr (ARG) {
        a.part_u[o + v] = at[v] >= 0 && a.indices ? a.indices[at[v]] : -1;
        a.part_e[o + v] = at[v] >= 0 && a.eid ? a.eid[at[v]] : -1;
      }
    }
    return;
  }
  if ((a.flags & F_MEAN) && n > 0) {
    T sc = a.deg ? T(a.deg[row]) : T(n);
    if (sc < T(1)) sc = T(1);
#pragma unroll
    for (int v = 0; v < VEC; ++v) acc[v] = acc[v] / sc;
  }
  if (a.flags & F_REPLACE_INF) {
#pragma unroll
    for (int v = 0; v < VEC; ++v)
      if (is_inf(acc[v])) {
        acc[v] = T(0);  // a replaced value has no message behind it
        at[v] = -1;
      }
  }
  const int64_t o = row * a.dout + k0;
  store_stream_any<T, VEC>(a.out + o, acc);
  if constexpr (ARG) {
    auto put = [&](int32_t* dst, const int32_t* id) {
      int32_t x[VEC];
#pragma unroll
      for (int v = 0; v < VEC; ++v) x[v] = at[v] >= 0 ? id[at[v]] : -1;
      store_stream_any<int32_t, VEC>(dst + o, x);
    };
    if (a.arg_u) put(a.arg_u, a.indices);
    if (a.arg_e) put(a.arg_e, a.eid);
  }
}

// Kernel variants, one body each so that every launch only carries the
// registers of its own path: per id layout, with both operands contiguous,
// with a splatted edge operand, with a scalar edge operand (one value per
// edge), or any modes. The scalar one is loaded with the ids and broadcast like
// them: read per lane and edge through the any-modes path it cost a GCN
// aggregation over 128 columns 4x the time of the same gather without it.
// P_DOT (copy / sum) writes only the dots of every gathered row with the row's
// own. P_SEL (copy / sum) adds a gathered value only where the selection's entry is
// the edge itself: the gradient of a max or min without a tensor of per-edge
// gradients in between. The _NEAR ones read edge rows through the caches (see
// STREAM_ROW_BYTES).
enum { P_CC = 0, P_CS = 1, P_DYN = 2, P_CS_DOT = 3, P_CW = 4, P_SEL = 5, P_DOT = 6, P_CC_NEAR = 7,
       P_DYN_NEAR = 8 };

// Wavefronts per SIMD asked of the register allocation: what each path needs
// plus a few registers would otherwise round down to one wavefront less (98
// registers for both operands contiguous: 4 instead of 5, and 9 % of the time
// on rows of 5 edges of two 256-byte rows).
// Sums only: the other reducers' selected slots and a divide's temporaries
// would spill.
constexpr int gspmm_waves(int op, int red, int path, int lay, int vec, int size) {
  if (red != RED_SUM || op == OP_DIV || path == P_DYN || path == P_DYN_NEAR || vec * size > 16)
    return 1;
  if (path == P_SEL) return size == 8 ? 4 : 5;
  if ((path == P_CC || path == P_CC_NEAR) && op != OP_COPY_LHS && op != OP_COPY_RHS) return lay == LAY_WIDE ? 6 : 5;
  return size == 8 ? 6 : 7;
}

template <class T, int OP, int RED, int VEC, int PATH, int LAY>
__global__ __launch_bounds__(BLOCK, gspmm_waves(OP, RED, PATH, LAY, VEC, sizeof(T))) void
gspmm_kernel(GspmmArgs<T> a) {
  const int64_t b = a.first_block + blockIdx.x;
  const bool chunk = b < a.chunk_blocks;
  const int64_t blk =
      chunk ? xcd_remap(b, a.chunk_blocks) : xcd_remap(b - a.chunk_blocks, a.num_blocks - a.chunk_blocks);
  const int lane = threadIdx.x & (WAVE - 1);
  // every lane of a wavefront takes the same path below, so DPP moves and
  // readlanes always see a full wavefront
  const int64_t wave = blk * WAVES_PER_BLOCK + (threadIdx.x >> 6);
  if (wave >= (chunk ? a.chunk_waves : a.row_waves)) return;
  if constexpr (PATH == P_CC)
    gspmm_body<T, OP, RED, VEC, M_CONTIG, M_CONTIG, LAY>(a, chunk, wave, lane);
  else if constexpr (PATH == P_CC_NEAR)
    gspmm_body<T, OP, RED, VEC, M_CONTIG, M_CONTIG, LAY, 0, false, true>(a, chunk, wave, lane);
  else if constexpr (PATH == P_CS)
    gspmm_body<T, OP, RED, VEC, M_CONTIG, M_SPLAT, LAY>(a, chunk, wave, lane);
  else if constexpr (PATH == P_CW)
    gspmm_body<T, OP, RED, VEC, M_CONTIG, M_SCALAR, LAY>(a, chunk, wave, lane);
  else if constexpr (PATH == P_SEL)
    gspmm_body<T, OP, RED, VEC, M_CONTIG, M_CONTIG, LAY, 0, true>(a, chunk, wave, lane);
  else if constexpr (PATH == P_DOT)
    gspmm_body<T, OP, RED, VEC, M_CONTIG, M_CONTIG, LAY, 2>(a, chunk, wave, lane);
  else if constexpr (PATH == P_CS_DOT)
    gspmm_body<T, OP, RED, VEC, M_CONTIG, M_SPLAT, LAY, 1>(a, chunk, wave, lane);
  else if constexpr (PATH == P_DYN_NEAR)
    gspmm_body<T, OP, RED, VEC, M_DYN, M_DYN, LAY, 0, false, true>(a, chunk, wave, lane);
  else
    gspmm_body<T, OP, RED, VEC, M_DYN, M_DYN, LAY>(a, chunk, wave, lane);
}

// Folds the chunk partials of each heavy row in chunk (= CSR) order.
template <class T, int RED>
__global__ __launch_bounds__(BLOCK) void gspmm_combine_kernel(
    const int32_t* __restrict__ heavy_rows, const int32_t* __restrict__ heavy_ptr,
    const int32_t* __restrict__ indptr, const int32_t* __restrict__ deg,
    const T* __restrict__ part_val, const int32_t* __restrict__ part_u,
    const int32_t* __restrict__ part_e, T* __restrict__ out, int32_t* __restrict__ arg_u,
    int32_t* __restrict__ arg_e, int64_t num_heavy, int64_t dout, int flags) {
  const int64_t t = (int64_t)blockIdx.x * BLOCK + threadIdx.x;
  if (t >= num_heavy * dout) return;
  const int64_t h = t / dout, k = t % dout;
  const int64_t row = heavy_rows[h];
  T acc = seed<T>(RED);
  int au = -1, ae = -1;
  // C partials requested at once (a chain of single loads made a hub of
  // hundreds of chunks wait for each of them in turn); past the end the last
  // one again, not folded
  constexpr int C = 16;
  const int c1 = heavy_ptr[h + 1];
  int sel = -1;  // max / min: the chunk selected
  for (int c = heavy_ptr[h]; c < c1; c += C) {
    T v[C];
#pragma unroll
    for (int j = 0; j < C; ++j) {
      const int cc = c + j < c1 ? c + j : c1 - 1;
      v[j] = part_val[(int64_t)cc * dout + k];
    }
#pragma unroll
    for (int j = 0; j < C; ++j) {
      const bool in = c + j < c1;
      if constexpr (RED == RED_MAX) {
        if (in && v[j] > acc) { acc = v[j]; sel = c + j; }
      } else if constexpr (RED == RED_MIN) {
        if (in && v[j] < acc) { acc = v[j]; sel = c + j; }
      } else {
        acc = in ? acc + v[j] : acc;
      }
    }
  }
  if constexpr (RED == RED_MAX || RED == RED_MIN) {
    if (sel >= 0) {
      au = part_u[(int64_t)sel * dout + k];
      ae = part_e[(int64_t)sel * dout + k];
    }
  }
  if (flags & F_MEAN) {
    T sc = deg ? T(deg[row]) : T(indptr[row + 1] - indptr[row]);
    if (sc < T(1)) sc = T(1);
    acc = acc / sc;
  }
  if ((flags & F_REPLACE_INF) && is_inf(acc)) {
    acc = T(0);
    au = ae = -1;
  }
  out[row * dout + k] = acc;
  if constexpr (RED == RED_MAX || RED == RED_MIN) {
    if (arg_u) arg_u[row * dout + k] = au;
    if (arg_e) arg_e[row * dout + k] = ae;
  }
}

template <class T, int OP, int RED, int VEC, int LAY>
void launch_path(const GspmmArgs<T>& a, dim3 grid, dim3 block, int lm, int rm, hipStream_t st) {
  if constexpr (OP == OP_COPY_LHS && RED == RED_SUM) {
    if (a.sel) {
      hipLaunchKernelGGL((gspmm_kernel<T, OP, RED, VEC, P_SEL, LAY>), grid, block, 0, st, a);
      return;
    }
  }
  const bool near = a.dr * (int64_t)sizeof(T) < STREAM_ROW_BYTES;
  auto go = [&](auto path) {
    hipLaunchKernelGGL((gspmm_kernel<T, OP, RED, VEC, decltype(path)::value, LAY>), grid, block, 0,
                       st, a);
  };
#define MDGL_PATH(P) go(std::integral_constant<int, P>{})
  if constexpr (OP == OP_COPY_LHS) {
    MDGL_PATH(P_CC);
  } else if constexpr (OP == OP_COPY_RHS) {
    if (near) MDGL_PATH(P_CC_NEAR);
    else MDGL_PATH(P_CC);
  } else if (lm == M_CONTIG && rm == M_CONTIG) {
    if (near) MDGL_PATH(P_CC_NEAR);
    else MDGL_PATH(P_CC);
  } else if (lm == M_CONTIG && rm == M_SCALAR) {
    MDGL_PATH(P_CW);
  } else if (lm == M_CONTIG && rm == M_SPLAT) {
    MDGL_PATH(P_CS);
  } else if (near) {
    MDGL_PATH(P_DYN_NEAR);
  } else {
    MDGL_PATH(P_DYN);
  }
#undef MDGL_PATH
}

// (lanes of 32 bytes are for rows of more than 64 of 16)
template <class T, int OP, int RED, int VEC>
void launch_lane(const GspmmArgs<T>& a, dim3 grid, dim3 block, int lm, int rm, hipStream_t st) {
  if constexpr (VEC <= VecOf<T>::n)
    launch_path<T, OP, RED, VEC, LAY_LANE>(a, grid, block, lm, rm, st);
}

template <class T, int OP, int RED, int VEC>
hipError_t launch_gspmm_op(const GspmmParams& p) {
  GspmmArgs<T> a;
  a.indptr = p.indptr;
  a.indices = p.indices;
  a.eid = p.eid;
  a.deg = p.deg;
  a.lhs = static_cast<const T*>(p.lhs);
  a.rhs = static_cast<const T*>(p.rhs);
  a.out = static_cast<T*>(p.out);
  a.arg_u = p.arg_u;
  a.arg_e = p.arg_e;
  a.num_rows = p.num_rows;
  a.dl = p.dl;
  a.lstride = p.lstride > 0 ? p.lstride : p.dl;
  a.dr = p.dr;
  a.dout = p.dout;
  a.bc = p.bc;
  a.lmode = p.lmode;
  a.rmode = p.rmode;
  a.flags = p.flags;
  a.run_len = (int)p.run_len;
  a.lpg = p.lpg;
  const int64_t nvec = p.dout / p.run_len * p.lpg;
  a.nvec = (int)nvec;
  const int G = p.group;  // chosen by the host (gspmm_group)
  a.gshift = 0;
  while ((1 << a.gshift) < G) ++a.gshift;
  a.S = (int)((nvec + G - 1) / G);
  a.num_chunks = p.num_chunks;
  a.chunk_row = p.chunk_row;
  a.chunk_start = p.chunk_start;
  a.chunk_len = p.num_chunks > 0 ? p.chunk_len : 0x7fffffff;
  a.part_val = static_cast<T*>(p.part_val);
  a.part_u = p.part_u;
  a.part_e = p.part_e;
  const int64_t per_wave = WAVE / G;
  a.chunk_uwaves = (p.num_chunks + per_wave - 1) / per_wave;
  a.row_uwaves = (p.num_rows + per_wave - 1) / per_wave;
  a.chunk_waves = a.chunk_uwaves * a.S;
  a.row_waves = a.row_uwaves * a.S;
  a.chunk_blocks = (a.chunk_waves + WAVES_PER_BLOCK - 1) / WAVES_PER_BLOCK;
  a.num_blocks = a.chunk_blocks + (a.row_waves + WAVES_PER_BLOCK - 1) / WAVES_PER_BLOCK;
  a.sel = p.sel;
  a.rowop = static_cast<const T*>(p.rowop);
  a.dot_out = static_cast<T*>(p.dot_out);
  a.dot_lanes = p.dot_lanes;
  a.rows = p.rows;
  a.row_limit = p.row_limit;
  const bool copy_l = OP == OP_COPY_LHS, copy_r = OP == OP_COPY_RHS;
  const int lm = copy_r ? a.rmode : a.lmode;
  const int rm = copy_l ? a.lmode : (!copy_r && a.rmode == M_SPLAT && a.dr == 1 ? M_SCALAR : a.rmode);
  const dim3 block(BLOCK);
  // HIP refuses a launch of 2**32 or more work-items, which 16 lanes a row
  // reach at 2**28 rows and 64 at 2**26: longer work lists take several
  // (of whole rounds over the XCDs, so the remap holds)
  for (a.first_block = 0; a.first_block < a.num_blocks; a.first_block += MAX_LAUNCH_BLOCKS) {
    const int64_t left = a.num_blocks - a.first_block;
    const dim3 grid((unsigned)(left < MAX_LAUNCH_BLOCKS ? left : MAX_LAUNCH_BLOCKS));
    bool launched = false;
    if constexpr ((OP == OP_MUL || OP == OP_COPY_LHS) && RED == RED_SUM && VEC == VecOf<T>::n) {
      if (p.dot_out) {
        // the caller checked: contiguous lhs rows, rhs splat over the groups
        constexpr int PATH = OP == OP_MUL ? P_CS_DOT : P_DOT;
        if (G == WAVE)
          hipLaunchKernelGGL((gspmm_kernel<T, OP, RED, VEC, PATH, LAY_WIDE>), grid, block, 0,
                             p.stream, a);
        else if (G < 16)
          hipLaunchKernelGGL((gspmm_kernel<T, OP, RED, VEC, PATH, LAY_LANE>), grid, block, 0,
                             p.stream, a);
        else
          hipLaunchKernelGGL((gspmm_kernel<T, OP, RED, VEC, PATH, LAY_ROW>), grid, block, 0,
                             p.stream, a);
        launched = true;
      }
    }
    if (!launched) {
      if (G == WAVE)
        launch_path<T, OP, RED, VEC, LAY_WIDE>(a, grid, block, lm, rm, p.stream);
      else if (G < 16)
        launch_lane<T, OP, RED, VEC>(a, grid, block, lm, rm, p.stream);
      else
        launch_path<T, OP, RED, VEC, LAY_ROW>(a, grid, block, lm, rm, p.stream);
    }
    hipError_t err = hipGetLastError();
    if (err != hipSuccess) return err;
  }
  if (OP == OP_COPY_LHS && p.dot_out) return hipSuccess;  // no partials to fold
  if (p.num_heavy > 0) {
    const int64_t n = p.num_heavy * p.dout;
    hipLaunchKernelGGL((gspmm_combine_kernel<T, RED>), dim3((unsigned)((n + BLOCK - 1) / BLOCK)),
                       dim3(BLOCK), 0, p.stream, p.heavy_rows, p.heavy_ptr, p.indptr, p.deg,
                       static_cast<const T*>(p.part_val), p.part_u, p.part_e,
                       static_cast<T*>(p.out), p.arg_u, p.arg_e, p.num_heavy, p.dout, p.flags);
    return hipGetLastError();
  }
  return hipSuccess;
}

template <class T, int RED, int VEC>
hipError_t launch_gspmm_vec(const GspmmParams& p) {
  switch (p.op) {
    case OP_ADD: return launch_gspmm_op<T, OP_ADD, RED, VEC>(p);
    case OP_SUB: return launch_gspmm_op<T, OP_SUB, RED, VEC>(p);
    case OP_MUL: return launch_gspmm_op<T, OP_MUL, RED, VEC>(p);
    case OP_DIV: return launch_gspmm_op<T, OP_DIV, RED, VEC>(p);
    case OP_COPY_LHS: return launch_gspmm_op<T, OP_COPY_LHS, RED, VEC>(p);
    case OP_COPY_RHS: return launch_gspmm_op<T, OP_COPY_RHS, RED, VEC>(p);
    default: return hipErrorInvalidValue;
  }
}

template <class T, int RED>
hipError_t launch_gspmm_red(const GspmmParams& p) {
  if (p.vec == VecOf<T>::n) return launch_gspmm_vec<T, RED, VecOf<T>::n>(p);
  if constexpr (VecOf<T>::n == 4) {
    if (p.vec == 2) return launch_gspmm_vec<T, RED, 2>(p);  // 8-byte lanes (even widths)
  } else {
    if (p.vec == 4) return launch_gspmm_vec<T, RED, 4>(p);  // 32-byte float64 lanes
  }
  return launch_gspmm_vec<T, RED, 1>(p);
}

}  // namespace mdgl

#define MDGL_INSTANTIATE_GSPMM(T, RED) \
  template hipError_t mdgl::launch_gspmm_red<T, RED>(const mdgl::GspmmParams&);
