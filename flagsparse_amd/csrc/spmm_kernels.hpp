// CSR SpMM C = A B on gfx950 (B, C row-major).
//
// Lane layout of a wave: [rows of the wave][nonzero slots][G lanes along N].
// The G lanes of a slot each own VEC consecutive columns (one 16-byte access
// of a B row when VEC*sizeof(T) == 16), so a slot streams whole B rows with
// coalesced loads.  The S = 64/(G*rows) slots of a row take nonzeros
// begin+slot, begin+slot+S, ..., UNROLL of them per trip (UNROLL B-row loads in
// flight per lane), and are summed by a lane-xor exchange at the end.  The
// row bins pick S by row length so that short rows share a wave and long rows
// get all 64/G slots; rows longer than the last bin are cut into segments whose
// partial rows a second pass adds in segment order (atomic-free).
// Over a CSC with perm != NULL the same kernel computes A^T B, reading the
// values as data[perm[q]] (no transposed copy of A).
//
// SDD (the differentiable SpMM's backward, over A's CSC): while a slot
// accumulates dB[j] += a_q dC[i] it also has the gathered row dC[i] in
// registers, so the same pass writes dvalues at the nonzero's CSR position,
// dvalues[pos[q]] = <dC[i], B[j]> (B the forward's dense operand, its row j
// loaded once per item).  One gather of dC rows serves both gradients.
//
// The loop is software-pipelined: while the B-row loads of one trip are in
// flight a lane already loads the column ids / values of its next trip -- of
// the same row, or the first trip of its next row -- so the index stream's
// latency hides behind the gathers.  When every operand fits in 4 GiB
// (OFF32), addresses are 32-bit byte offsets from the (uniform) base
// pointers: one VGPR per address, which keeps occupancy at 8 waves/SIMD.
#pragma once

#include "fsp_device.hpp"
#include "fsp_host.hpp"
#include "fsp_plan.hpp"

namespace fsp {

// <x, y> over a lane's VEC columns in the accumulation type.  16-bit values
// go through v_dot2_f32_{bf16,f16}: two products and the running sum per
// instruction, where converting each element and an FMA would take four.
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
template <typename A, typename T, int VEC>
__device__ __forceinline__ A row_dot(const vec_t<T, VEC>& x, const vec_t<T, VEC>& y) {
  if constexpr (std::is_same<T, __bf16>::value && VEC % 2 == 0) {
    float t = 0.0f;
#pragma unroll
    for (int v = 0; v < VEC; v += 2) {
      const bf16x2_t a = {x.v[v], x.v[v + 1]};
      const bf16x2_t c = {y.v[v], y.v[v + 1]};
      t = __builtin_amdgcn_fdot2_f32_bf16(a, c, t, false);
    }
    return t;
  } else if constexpr (std::is_same<T, _Float16>::value && VEC % 2 == 0) {
    float t = 0.0f;
#pragma unroll
    for (int v = 0; v < VEC; v += 2) {
      const f16x2_t a = {x.v[v], x.v[v + 1]};
      const f16x2_t c = {y.v[v], y.v[v + 1]};
      t = __builtin_amdgcn_fdot2(a, c, t, false);
    }
    return t;
  } else {
    A t = A(0);
#pragma unroll
    for (int v = 0; v < VEC; ++v) t += static_cast<A>(x.v[v]) * static_cast<A>(y.v[v]);
    return t;
  }
}

// The backward's extra operands (SDD): the forward's B (row j of the item),
// each nonzero's CSR position, and the dvalues output in CSR order.
template <typename T, typename QT>
struct sdd_args {
  const T* Bj;
  int64_t ldbj;
  const QT* pos;
  T* dvals;
};

// TAIL (SDD only): VEC does not divide n_dense, see `ov`.  Its own
// instantiation: as a branch on a uniform flag the masks cost the whole-vector
// backward 9 % (bf16, N = 128).
// TV: type of A's values, T itself or the wider type the COO product computes
// in (f64 over f32, f32 over f16 / bf16).  Sums are kept in TV's accumulation
// type either way; B and C stay in T, so what is gathered and written is half
// the bytes of a product over widened copies of B and C, and the copies'
// passes are gone: f32, 150001 x 90001, 3 M nonzeros, N = 100: 457 -> 207 us.
template <typename T, typename TV, typename IT, typename PT, typename QT, int VEC, int UNROLL, bool PERM, bool OFF32, bool SDD,
          bool TAIL>
__global__ __launch_bounds__(FSP_WG_THREADS) void spmm_slots_kernel(
    const PT* __restrict__ indptr, const IT* __restrict__ indices, const TV* __restrict__ data,
    const QT* __restrict__ perm, const T* __restrict__ B, int64_t ldb, T* __restrict__ C, int64_t ldc,
    int64_t n_dense, int g_log2, typename acc_of<TV>::type* __restrict__ partials, launch_table tab,
    sdd_args<T, QT> sd) {
  using A = typename acc_of<TV>::type;
  using O = typename addr<OFF32>::off_t;  // element / byte offsets
  using P = typename std::conditional<OFF32, int32_t, int64_t>::type;  // nonzero positions
  // A column id.  B's offsets fit 32 bits, and so do its rows' numbers: of an
  // int64 id the low half is loaded.  Loading both, the compiler gave the unused
  // half's register to the next load's address and waited for every load in
  // flight between the two (10000 x 86679, power-law rows, f32 N = 128, int64
  // indices: 40 us, 30 with int32 indices or 64-bit offsets).
  using I = typename std::conditional<OFF32, uint32_t, IT>::type;
  constexpr int kIdStride = sizeof(IT) / sizeof(I);
  const int k = find_bin(tab, blockIdx.x);
  const launch_bin lb = tab.b[k];  // a copy: the fields stay in registers
  const int s_log2 = lb.lanes_log2;
  const int G = 1 << g_log2;
  const int S = 1 << s_log2;
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int gl = lane & (G - 1);
  const int slot = (lane >> g_log2) & (S - 1);
  const int sub = lane >> (g_log2 + s_log2);
  const int64_t per_wave = 64 >> (g_log2 + s_log2);
  const int64_t per_block = per_wave * FSP_WAVES;
  // A lane's VEC columns.  When VEC does not divide n_dense the last lane's
  // vector is moved back to end at n_dense (the host picks VEC <= n_dense):
  // its first `ov` columns are the previous lane's too, both lanes sum them in
  // the same order and store the same bits, and no access leaves the row.
  const int64_t colv = (static_cast<int64_t>(blockIdx.y) * G + gl) * VEC;
  const bool col_ok = colv < n_dense;
  const O col0 = static_cast<O>(colv + VEC <= n_dense ? colv : n_dense - VEC);
  const int ov = col_ok ? static_cast<int>(colv - static_cast<int64_t>(col0)) : 0;
  // this workgroup's tiles: first, first + step, ... < end
  const tile_range tr = bin_tiles(lb, per_block);
  const int64_t rr_step = tr.step * per_block;
  const O ldb_o = static_cast<O>(ldb);
  const O ldc_o = static_cast<O>(ldc);
  const O nd_o = static_cast<O>(n_dense);

  // Every load below is unconditional (indices clamped into range, results
  // masked by selects) so the compiler can count outstanding loads exactly
  // and wait only for the B rows before the FMAs, not for the prefetch.
  const O col_ld = col_ok ? col0 : O(0);  // lanes past n_dense read column 0
  const int64_t last_item = lb.count - 1;  // bins in the table are non-empty

  // Item (row or segment) of this lane: output slot, nonzero range, and the
  // row it belongs to (its B row under SDD).  Under SDD the lanes past
  // n_dense run their slot's nonzeros too (reading column 0, contributing 0
  // to the dots): a dot's lane-group sum needs every lane of the group.
  auto item = [&](int64_t r, O& out, P& beg, P& end, O& jrow) {
    const bool live = r < lb.count && (SDD || col_ok);
    const int64_t rc = r < lb.count ? r : last_item;
    O o, jr;
    P b, e;
    if (lb.is_segment) {
      o = static_cast<O>(rc);
      jr = SDD ? static_cast<O>(tab.seg_row[rc]) : O(0);
      b = static_cast<P>(tab.seg_begin[rc]);
      e = static_cast<P>(tab.seg_end[rc]);
    } else {
      const int64_t row = lb.rows ? static_cast<int64_t>(lb.rows[rc]) : rc;
      o = static_cast<O>(row);
      jr = o;
      b = static_cast<P>(indptr[row]);
      e = static_cast<P>(indptr[row + 1]);
    }
    out = o;
    jrow = jr;
    beg = live ? b : P(0);
    end = live ? e : P(0);
  };
  // Column ids and values of nonzeros p, p+S, ...; past `end` the loads
  // repeat the item's last nonzero (a valid column of the same row).  They
  // stay raw: masking or converting them here would make the compiler wait
  // for every load in flight (the B rows included) right after the prefetch,
  // so the mask and the conversion are applied where they are consumed.
  auto trip = [&](P p, P end, I (&c)[UNROLL], TV (&a)[UNROLL], QT (&pq)[UNROLL]) {
    const P last = end > 0 ? end - 1 : P(0);
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      const P q = p + static_cast<P>(u) * S;
      const O qc = static_cast<O>(q < end ? q : last);
      c[u] = elem<OFF32>(reinterpret_cast<const I*>(indices), qc * static_cast<O>(kIdStride));
      const O qv = PERM ? static_cast<O>(elem<OFF32>(perm, qc)) : qc;
      a[u] = elem<OFF32>(data, qv);
      if constexpr (SDD) pq[u] = elem<OFF32>(sd.pos, qc);
    }
  };
  // Row j of the forward's B for this lane's columns (zero past n_dense).
  auto b_row = [&](O j) {
    vec_t<T, VEC> r;
    if constexpr (SDD) {
      r = *addr<OFF32>::at(reinterpret_cast<const vec_t<T, VEC>*>(sd.Bj),
                           (j * static_cast<O>(sd.ldbj) + col_ld) * static_cast<O>(sizeof(T)));
    }
    return r;
  };

  int64_t rr = tr.first * per_block + wave * per_wave + sub;
  O out, jrow;
  P beg, end;
  item(rr, out, beg, end, jrow);
  I c[UNROLL];
  TV a[UNROLL];
  QT pq[UNROLL];
  trip(beg + slot, end, c, a, pq);

  for (int64_t tile = tr.first; tile < tr.end; tile += tr.step) {  // wave-uniform
    const bool active = rr < lb.count && col_ok;
    const int64_t rr_next = rr + rr_step;
    // the next item is prefetched only when this workgroup will process it
    const bool has_next = tile + tr.step < tr.end;  // wave-uniform
    O out_n = 0, jrow_n = 0;
    P beg_n = 0, end_n = 0;
    if (has_next) item(rr_next, out_n, beg_n, end_n, jrow_n);
    vec_t<T, VEC> bj;
    if constexpr (SDD) bj = b_row(jrow);
    A acc[VEC];
#pragma unroll
    for (int v = 0; v < VEC; ++v) acc[v] = A(0);
    bool prefetched = false;
    for (P p = beg + slot; p < end; p += static_cast<P>(S) * UNROLL) {
      vec_t<T, VEC> b[UNROLL];
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) {
        const O boff = (static_cast<O>(c[u]) * ldb_o + col_ld) * static_cast<O>(sizeof(T));
        b[u] = *addr<OFF32>::at(reinterpret_cast<const vec_t<T, VEC>*>(B), boff);
      }
      // prefetch: the next trip of this item, else the first trip of the next
      const P pn = p + static_cast<P>(S) * UNROLL;
      const bool same = pn < end;
      prefetched = prefetched || !same;
      TV an[UNROLL];
      I cn[UNROLL];
      QT pqn[UNROLL];
      if constexpr (SDD) {
        // unconditional (with nothing next it reloads this trip's nonzeros,
        // unused): with loads and stores under branches the compiler cannot
        // count what is outstanding and waits for all of it, the dvalue
        // stores included, every trip.  Without SDD the branch stays: there
        // the B loads issue as each pair of column ids arrives (5 % faster on
        // the 4096-matrix batch's short rows).
        trip(same ? pn : (has_next ? beg_n + slot : p), same ? end : (has_next ? end_n : end), cn, an, pqn);
      } else if (same || has_next) {
        trip(same ? pn : beg_n + slot, same ? end : end_n, cn, an, pqn);
      }
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) {
        const bool ok = p + static_cast<P>(u) * S < end;
        const A av = ok ? static_cast<A>(a[u]) : A(0);
#pragma unroll
        for (int v = 0; v < VEC; ++v) {
          const A bv = ok ? static_cast<A>(b[u].v[v]) : A(0);
          acc[v] += av * bv;
        }
      }
      if constexpr (SDD) {
        // dvalues of this trip's nonzeros: a lane's VEC products, then the
        // sum over the slot's G lanes (all of them run this trip)
        // Every lane of the slot stores the slot's total, unconditionally (a
        // store under a branch has the same effect on the waits as a load).
        // Past the item's end a lane's loads were clamped to the item's last
        // nonzero, so it writes that nonzero's own value to its own place.
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
          vec_t<T, VEC> bu = b[u], bv = bj;
          if constexpr (TAIL) {  // the shared columns count once, in the previous lane
#pragma unroll
            for (int v = 0; v < VEC - 1; ++v) {
              if (v < ov) bu.v[v] = bv.v[v] = T(0);
            }
          }
          const A d = group_sum(col_ok ? row_dot<A>(bu, bv) : A(0), G);
          *addr<OFF32>::at(sd.dvals, static_cast<O>(pq[u]) * static_cast<O>(sizeof(T))) = static_cast<T>(d);
        }
      }
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) {
        c[u] = cn[u];
        a[u] = an[u];
        if constexpr (SDD) pq[u] = pqn[u];
      }
    }
    if (!prefetched && has_next) trip(beg_n + slot, end_n, c, a, pq);
    // Sum the S slots of a row: lanes that differ only in the slot bits.
    for (int j = 0; j < s_log2; ++j) {
#pragma unroll
      for (int v = 0; v < VEC; ++v) acc[v] += shfl_xor(acc[v], G << j);
    }
    if (active && slot == 0) {
      if (lb.is_segment) {
        A* dst = addr<OFF32>::at(partials, (out * nd_o + col0) * static_cast<O>(sizeof(A)));
#pragma unroll
        for (int v = 0; v < VEC; ++v) dst[v] = acc[v];
      } else {
        vec_t<T, VEC> o;
#pragma unroll
        for (int v = 0; v < VEC; ++v) o.v[v] = static_cast<T>(acc[v]);
        *addr<OFF32>::at(reinterpret_cast<vec_t<T, VEC>*>(C), (out * ldc_o + col0) * static_cast<O>(sizeof(T))) = o;
      }
    }
    out = out_n;
    jrow = jrow_n;
    beg = beg_n;
    end = end_n;
    rr = rr_next;
  }
}

// n elements of E (below 4 GiB) as a buffer: element kAbsent reads as zero and
// touches no memory.
constexpr uint32_t kAbsent = ~0u;

// Where B's rows come across the fabric, more gathers in flight lower its
// throughput, and the loop whose lanes load their nonzeros each for themselves
// (spmm_slots_kernel) paces them; below that the faster issue of
// spmm_bins_kernel wins.  Time of the former over the latter, int32 indices,
// rows of power-law length (mean 24) with uniform columns / graphs with hub
// columns (mean 14), which the caches keep:
//                                   24 MiB       32           40           48           56           64
//   16 lanes  f32  N =  64      0.995/1.064  0.997/1.035  0.986/1.030  0.987/1.011  0.979/1.016  0.989/1.007
//             bf16 N = 128      1.012/1.096  0.991/1.064  1.009/1.040  0.992/1.035  0.986/1.040  1.004/1.027
//   32 lanes  f32  N = 128      0.995/1.057  0.991/1.037  0.990/1.027  0.963/1.007  0.975/1.015  0.983/0.992
//             f64  N =  64      1.014/1.106  0.989/1.106  0.975/1.050  0.953/1.038  0.960/1.034  0.972/1.020
//   64 lanes  f64  N = 128      1.085/1.249  1.036/1.160  1.007/1.121  0.994/1.072  0.994/1.044  0.981/1.086
//   38 of 64  f64  N =  75      1.072/1.324  1.078/1.252  1.058/1.201  1.066/1.160  1.033/1.128  1.047/1.135
// Uniform columns gain from the eight L2s' 32 MiB on, graphs from twice that.
// The limit of rows that fill a group of 32 lanes (seven lanes in eight) is where
// the former begin to gain, which is the most there is to gain, 5 %; that of other
// groups of 16 or 32 and of full ones of 64 lies between, where one gains what the
// other loses.  A 64-lane group with idle lanes is not paced (38 of 64 up to 400
// MiB: 1.01-1.14), nor are groups of 8 lanes (f32 N = 32, 32 to 128 MiB: 1.00-1.02,
// f64 N = 16 0.99-1.08) and the backward (32 to 256 MiB: f32 N = 64 1.01-1.12, bf16
// N = 128 1.01-1.08, f64 N = 64 1.09-1.27).
constexpr int64_t kPacedBytes = int64_t(56) << 20;
constexpr int64_t kPacedFullBytes = int64_t(32) << 20;
static inline bool spmm_paced(int64_t elem_bytes, int g_log2, int64_t n_dense, int64_t b_bytes, bool backward) {
  const bool full = n_dense * elem_bytes * 8 >= int64_t(16 * 7) << g_log2;
  if (backward || g_log2 < 4 || (g_log2 == 6 && !full)) return false;
  return b_bytes >= (g_log2 == 5 && full ? kPacedFullBytes : kPacedBytes);
}

// Whether a launch of whole vectors with 32-bit offsets shares its nonzeros
// between lanes (spmm_bins_kernel): groups of four lanes or more whose gathers
// are not paced.  (B's bytes and a row stay below the offset that marks an
// absent nonzero.)
static inline bool spmm_shares_nonzeros(int64_t elem_bytes, int g_log2, int64_t n_dense, int64_t ldb, int64_t b_rows,
                                        bool backward) {
  const int64_t b_bytes = b_rows * ldb * elem_bytes;
  return g_log2 >= 2 && b_bytes <= (int64_t(1) << 32) - 1 - ldb * elem_bytes &&
         !spmm_paced(elem_bytes, g_log2, n_dense, b_bytes, backward);
}

template <typename E>
struct buffer {
  __amdgpu_buffer_rsrc_t rsrc;
  __device__ __forceinline__ buffer(const E* p, uint32_t n)
      : rsrc(__builtin_amdgcn_make_buffer_rsrc(const_cast<E*>(p), 0, n * static_cast<uint32_t>(sizeof(E)), kRawBuffer)) {}
  __device__ __forceinline__ E load(uint32_t i) const {
    const uint32_t off = i == kAbsent ? kAbsent : i * static_cast<uint32_t>(sizeof(E));
    if constexpr (sizeof(E) == 2) {
      return __builtin_bit_cast(E, __builtin_amdgcn_raw_buffer_load_b16(rsrc, off, 0, 0));
    } else if constexpr (sizeof(E) == 4) {
      return __builtin_bit_cast(E, __builtin_amdgcn_raw_buffer_load_b32(rsrc, off, 0, 0));
    } else {
      return __builtin_bit_cast(E, __builtin_amdgcn_raw_buffer_load_b64(rsrc, off, 0, 0));
    }
  }
};

// Workgroups per CU (waves per SIMD) the registers must allow: the most that
// spills nothing (eight vectors of 16-bit elements need 95 registers; held to 80
// they spill, and 200000 nodes, N = 128, unroll 8 took 116 us, 87 without; with
// the values behind a permutation unroll 4 needs 66, and held to 64 a bf16 product of
// N = 256 took 55 us, 50 without).
template <int UNROLL, bool SDD, bool PERM, int ELEM>
constexpr int kMinBlocks = UNROLL <= 4 ? (SDD ? 5 : (PERM && ELEM == 2 ? 7 : 8)) : (SDD ? 4 : (ELEM == 2 ? 5 : 6));

// The same layout and summation order as spmm_slots_kernel (bitwise equal),
// with the id and value of a nonzero loaded once per quad (LANES 4) or row of
// 16 lanes (LANES 16) instead of once per lane: lane q holds nonzero q of the
// trip, computes its B row offset, and one DPP move per nonzero hands offset
// and value to the group.  A wave load costs the CU's address unit 18 clocks
// whatever its lanes ask for (measured: all lanes, half masked off, half out
// of range), so two of every three loads, and the offset arithmetic of every
// lane, are what goes.  Nonzeros past a row's end read as value zero and have
// their B row outside the buffer: it reads as zeros without memory traffic, so
// nothing is masked and no load is repeated, and the batches of UNROLL rows
// that no lane needs are skipped.  That takes both zeros: the next rows'
// nonzeros are loaded in the wave's last trip and no sooner, or an infinite
// value among them would meet the zeros of a row that has ended.  Against
// spmm_slots_kernel, vector instructions per launch fall from 44.6 to 23.8
// million and loads from 6.0 to 2.6 million (262144 x 229376, f32 N = 64, either
// side of the limit above).  100003 x 70001 f64, N = 75: 290 -> 240 us;
// 1024-matrix batch, N = 32: 687 -> 665 us; 200000-node graph, bf16 N = 128, by
// kernel: 84.6 -> 80.7 us, its backward 130.5 -> 127.1 us.
template <typename T, typename TV, typename IT, typename PT, typename QT, int VEC, int UNROLL, int LANES, bool PERM,
          bool SDD, bool TAIL>
__global__ __launch_bounds__(FSP_WG_THREADS, (kMinBlocks<UNROLL, SDD, PERM, static_cast<int>(sizeof(T))>)) void spmm_bins_kernel(
    const PT* __restrict__ indptr, const IT* __restrict__ indices, const TV* __restrict__ data,
    const T* __restrict__ B, int64_t ldb, uint32_t b_bytes, T* __restrict__ C, int64_t ldc, int64_t n_dense, uint32_t nnz,
    int g_log2, typename acc_of<TV>::type* __restrict__ partials, launch_table tab, sdd_args<T, QT> sd) {
  using A = typename acc_of<TV>::type;
  constexpr bool OFF32 = true;
  using O = uint32_t;  // element / byte offsets
  using P = int32_t;   // nonzero positions
  using V = vec_t<T, VEC>;
  constexpr int kRegs = UNROLL > LANES ? UNROLL / LANES : 1;  // nonzeros a lane holds
  constexpr int kTrip = LANES * kRegs;                         // nonzeros of a slot per trip
  const launch_bin lb = tab.b[find_bin(tab, blockIdx.x)];  // a copy: the fields stay in registers
  const int s_log2 = lb.lanes_log2;
  const int G = 1 << g_log2;
  const int S = 1 << s_log2;
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int gl = lane & (G - 1);
  const int slot = (lane >> g_log2) & (S - 1);
  const int sub = lane >> (g_log2 + s_log2);
  const int ql = lane & (LANES - 1);
  const int64_t per_wave = 64 >> (g_log2 + s_log2);
  const int64_t per_block = per_wave * FSP_WAVES;
  // A lane's VEC columns, see spmm_slots_kernel.
  const int64_t colv = (static_cast<int64_t>(blockIdx.y) * G + gl) * VEC;
  const bool col_ok = colv < n_dense;
  const O col0 = static_cast<O>(colv + VEC <= n_dense ? colv : n_dense - VEC);
  const int ov = col_ok ? static_cast<int>(colv - static_cast<int64_t>(col0)) : 0;
  const O col_off = (col_ok ? col0 : O(0)) * static_cast<O>(sizeof(T));  // lanes past n_dense read column 0
  const tile_range tr = bin_tiles(lb, per_block);
  const int64_t rr_step = tr.step * per_block;
  const O row_bytes = static_cast<O>(ldb) * static_cast<O>(sizeof(T));
  const int64_t last_item = lb.count - 1;  // bins in the table are non-empty
  // B as a buffer of b_bytes: a load from `outside` (plus any column) reads
  // zeros and touches no memory.
  const auto brsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(B), 0, b_bytes, kRawBuffer);
  const O outside = ~O(0) - row_bytes;
  const buffer<IT> indices_b(indices, nnz);
  const buffer<TV> data_b(data, nnz);
  const buffer<QT> pos_b(sd.pos, nnz);

  // Item (row or segment) of this lane; every lane of a group keeps the
  // nonzero range, also past n_dense: the group's broadcasts read all of them.
  auto item = [&](int64_t r, O& out, P& beg, P& end, O& jrow) {
    const bool live = r < lb.count;
    const int64_t rc = live ? r : last_item;
    P b, e;
    if (lb.is_segment) {
      out = static_cast<O>(rc);
      jrow = SDD ? static_cast<O>(tab.seg_row[rc]) : O(0);
      b = static_cast<P>(tab.seg_begin[rc]);
      e = static_cast<P>(tab.seg_end[rc]);
    } else {
      const int64_t row = lb.rows ? static_cast<int64_t>(lb.rows[rc]) : rc;
      out = jrow = static_cast<O>(row);
      b = static_cast<P>(indptr[row]);
      e = static_cast<P>(indptr[row + 1]);
    }
    beg = live ? b : P(0);
    end = live ? e : P(0);
  };
  // This lane's nonzeros of a trip that starts at the slot's nonzero p; past
  // `end` they read as zero.
  auto trip = [&](P p, P end, IT (&c)[kRegs], TV (&a)[kRegs], QT (&pq)[kRegs]) {
#pragma unroll
    for (int r = 0; r < kRegs; ++r) {
      const P q = p + (static_cast<P>(r * LANES + ql) << s_log2);
      const O at = q < end ? static_cast<O>(q) : kAbsent;
      c[r] = indices_b.load(at);
      if constexpr (!PERM) a[r] = data_b.load(at);
      if constexpr (PERM || SDD) pq[r] = pos_b.load(at);
    }
  };

  int64_t rr = tr.first * per_block + wave * per_wave + sub;
  O out, jrow;
  P beg, end;
  item(rr, out, beg, end, jrow);
  IT c[kRegs];
  TV a[kRegs];
  QT pq[kRegs];
  trip(beg + slot, end, c, a, pq);

  for (int64_t tile = tr.first; tile < tr.end; tile += tr.step) {  // wave-uniform
    const bool active = rr < lb.count && col_ok;
    const int64_t rr_next = rr + rr_step;
    // the next item is prefetched only when this workgroup will process it
    const bool has_next = tile + tr.step < tr.end;  // wave-uniform
    O out_n = 0, jrow_n = 0;
    P beg_n = 0, end_n = 0;
    if (has_next) item(rr_next, out_n, beg_n, end_n, jrow_n);
    V bj;
    if constexpr (SDD) {  // row j of the forward's B
      bj = *addr<OFF32>::at(reinterpret_cast<const V*>(sd.Bj),
                            jrow * static_cast<O>(sd.ldbj) * static_cast<O>(sizeof(T)) + col_off);
      if constexpr (TAIL) {
#pragma unroll
        for (int v = 0; v < VEC - 1; ++v) bj.v[v] = v < ov ? T(0) : bj.v[v];
      }
    }
    A acc[VEC];
#pragma unroll
    for (int v = 0; v < VEC; ++v) acc[v] = A(0);
    P p = beg + slot;
    bool prefetched = false;  // wave-uniform
    // wave-uniform: every lane takes part in the broadcasts.  (`more` says the same
    // as the ballot of the plain product, which makes the compiler keep a first trip
    // apart from the others, whose B rows then wait for the ids alone and not for
    // the values too: 26841 x 89266, f32 N = 57 21.4 -> 20.5 us.  In the backward
    // the second copy spills: training step on 200000 nodes, bf16 252 us with it,
    // 243 without.)
    bool more = __ballot(p < end) != 0;
    while (SDD ? more : __ballot(p < end) != 0) {
      O off[kRegs];
      A av[kRegs];
#pragma unroll
      for (int r = 0; r < kRegs; ++r) {
        const bool ok = p + (static_cast<P>(r * LANES + ql) << s_log2) < end;
        off[r] = ok ? static_cast<O>(c[r]) * row_bytes : outside;
        // the permuted value's random read runs beside the B rows' gathers
        if constexpr (PERM) a[r] = data_b.load(ok ? static_cast<O>(pq[r]) : kAbsent);
      }
      const P pn = p + (static_cast<P>(kTrip) << s_log2);
      const bool more_n = __ballot(pn < end) != 0;
      if constexpr (SDD) more = more_n;
      IT cn[kRegs];
      TV an[kRegs];
      QT pqn[kRegs];
      A dots[kRegs];
      static_for<kTrip / UNROLL>([&](auto batch) {
        constexpr int u0 = decltype(batch)::value * UNROLL;
        if (u0 > 0 && __ballot(p + (static_cast<P>(u0) << s_log2) < end) == 0) return;  // wave-uniform
        V b[UNROLL];
        static_for<UNROLL>([&](auto u) {
          constexpr int n = u0 + decltype(u)::value;
          b[u] = __builtin_bit_cast(
              V, __builtin_amdgcn_raw_buffer_load_b128(brsrc, bcast<LANES, n % LANES>(off[n / LANES]) + col_off, 0, 0));
        });
        // prefetch: the next trip of the wave's items, after the last one the
        // first trip of the next items.  Unconditional (past an item's end, and
        // with nothing next, it touches no memory): under a branch the compiler
        // could not count the loads in flight, and the last B row of the batch
        // would wait for the prefetch too.
        if constexpr (u0 == 0) trip(more_n ? pn : beg_n + slot, more_n ? end : end_n, cn, an, pqn);
        if constexpr (u0 == 0) {
#pragma unroll
          for (int r = 0; r < kRegs; ++r) av[r] = static_cast<A>(a[r]);
        }
        static_for<UNROLL>([&](auto u) {
          constexpr int n = u0 + decltype(u)::value;
          const A x = bcast<LANES, n % LANES>(av[n / LANES]);
#pragma unroll
          for (int v = 0; v < VEC; ++v) acc[v] += x * static_cast<A>(b[u].v[v]);
        });
        if constexpr (SDD) {
          // the dots of this batch: a lane's VEC products, then the sum over
          // the slot's G lanes; the lane that holds the nonzero keeps it
          static_for<UNROLL>([&](auto u) {
            constexpr int n = u0 + decltype(u)::value;
            V bu = b[u];
            if constexpr (TAIL) {  // the shared columns count once, in the previous lane
#pragma unroll
              for (int v = 0; v < VEC - 1; ++v) bu.v[v] = v < ov ? T(0) : bu.v[v];
            }
            const A d = group_sum(col_ok ? row_dot<A>(bu, bj) : A(0), G);
            dots[n / LANES] = ql == n % LANES ? d : dots[n / LANES];
          });
        }
      });
      if constexpr (SDD) {
#pragma unroll
        for (int r = 0; r < kRegs; ++r) {
          const bool ok = p + (static_cast<P>(r * LANES + ql) << s_log2) < end;
          if (ok && gl < LANES) {
            *addr<OFF32>::at(sd.dvals, static_cast<O>(pq[r]) * static_cast<O>(sizeof(T))) = static_cast<T>(dots[r]);
          }
        }
      }
#pragma unroll
      for (int r = 0; r < kRegs; ++r) {
        c[r] = cn[r];
        if constexpr (!PERM) a[r] = an[r];
        if constexpr (PERM || SDD) pq[r] = pqn[r];
      }
      p = pn;
      prefetched = true;
    }
    if (!prefetched && has_next) trip(beg_n + slot, end_n, c, a, pq);
    // Sum the S slots of a row: lanes that differ only in the slot bits.
    for (int j = 0; j < s_log2; ++j) {
#pragma unroll
      for (int v = 0; v < VEC; ++v) acc[v] += shfl_xor(acc[v], G << j);
    }
    if (active && slot == 0) {
      if (lb.is_segment) {
        A* dst = addr<OFF32>::at(partials, (out * static_cast<O>(n_dense) + col0) * static_cast<O>(sizeof(A)));
#pragma unroll
        for (int v = 0; v < VEC; ++v) dst[v] = acc[v];
      } else {
        V o;
#pragma unroll
        for (int v = 0; v < VEC; ++v) o.v[v] = static_cast<T>(acc[v]);
        *addr<OFF32>::at(reinterpret_cast<V*>(C),
                         (out * static_cast<O>(ldc) + col0) * static_cast<O>(sizeof(T))) = o;
      }
    }
    out = out_n;
    jrow = jrow_n;
    beg = beg_n;
    end = end_n;
    rr = rr_next;
  }
}

// C[long_rows[i], :] = sum of the row's segment partials, in segment order.
// One wave per long row (a grid-stride loop over rows): the row's segment
// range and output row are wave-uniform loads, lane l takes columns l,
// l + 64, ..., and each segment's partial row is one coalesced read whose
// address does not depend on the previous one.
template <typename T, typename A>
__global__ __launch_bounds__(FSP_WG_THREADS) void spmm_long_reduce_kernel(
    const A* __restrict__ partials, const int32_t* __restrict__ long_rows,
    const int64_t* __restrict__ seg_ptr, int64_t n_long, int64_t n_dense, T* __restrict__ C, int64_t ldc) {
  const int lane = threadIdx.x & 63;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * FSP_WAVES + (threadIdx.x >> 6); i < n_long;
       i += static_cast<int64_t>(gridDim.x) * FSP_WAVES) {
    const int64_t s0 = seg_ptr[i], s1 = seg_ptr[i + 1];
    T* __restrict__ c_row = C + static_cast<int64_t>(long_rows[i]) * ldc;
    for (int64_t col = lane; col < n_dense; col += 64) {
      const A* __restrict__ p = partials + s0 * n_dense + col;
      A acc = A(0);
#pragma unroll 4
      for (int64_t sg = s0; sg < s1; ++sg, p += n_dense) acc += *p;
      c_row[col] = static_cast<T>(acc);
    }
  }
}

// C[r, :n_dense] = 0 for every row (the matrix has no nonzeros).
template <typename T>
__global__ __launch_bounds__(FSP_WG_THREADS) void fill_zero_rows_kernel(T* __restrict__ C, int64_t ldc,
                                                                        int64_t n_rows, int64_t n_dense) {
  const int64_t total = n_rows * n_dense;
  for (int64_t t = static_cast<int64_t>(blockIdx.x) * FSP_WG_THREADS + threadIdx.x; t < total;
       t += static_cast<int64_t>(gridDim.x) * FSP_WG_THREADS) {
    const int64_t r = t / n_dense;
    C[r * ldc + (t - r * n_dense)] = T(0);
  }
}

struct spmm_args {
  const void* indptr;
  const void* indices;
  const void* data;
  const void* perm;
  const void* B;
  int64_t ldb;
  void* C;
  int64_t ldc;
  int64_t n_rows;
  int64_t n_dense;
  int lanes_n;
  int64_t nnz;
  int64_t b_rows;
  // the fused backward (SDD): forward B, CSR position per nonzero, dvalues
  const void* Bj = nullptr;
  int64_t ldbj = 0;
  const void* pos = nullptr;
  void* dvals = nullptr;
};

template <typename T, typename TV, typename IT, typename PT, typename QT, int VEC, int UNROLL, bool PERM, bool OFF32,
          bool SDD>
static void launch_bins(const spmm_args& x, dim3 grid, int g_log2, typename acc_of<TV>::type* partials,
                        const launch_table& tab, hipStream_t s) {
  const sdd_args<T, QT> sd{static_cast<const T*>(x.Bj), x.ldbj, static_cast<const QT*>(SDD ? x.pos : x.perm),
                           static_cast<T*>(x.dvals)};
  // Groups of 4 or more lanes of whole vectors share their nonzeros through
  // broadcasts; narrower groups load them per lane.
  const int64_t b_bytes = x.b_rows * x.ldb * (int64_t)sizeof(T);
  if constexpr (VEC > 1 && OFF32) {
    const auto bins = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, grid, dim3(FSP_WG_THREADS), 0, s, static_cast<const PT*>(x.indptr),
                         static_cast<const IT*>(x.indices), static_cast<const TV*>(x.data),
                         static_cast<const T*>(x.B), x.ldb, static_cast<uint32_t>(b_bytes), static_cast<T*>(x.C), x.ldc,
                         x.n_dense, static_cast<uint32_t>(x.nnz), g_log2, partials, tab, sd);
    };
    const auto width = [&](auto tail) {
      constexpr bool TAIL = decltype(tail)::value;
      if (g_log2 >= 4) {
        bins(spmm_bins_kernel<T, TV, IT, PT, QT, VEC, UNROLL, 16, PERM, SDD, TAIL>);
      } else {
        bins(spmm_bins_kernel<T, TV, IT, PT, QT, VEC, UNROLL, 4, PERM, SDD, TAIL>);
      }
    };
    if (spmm_shares_nonzeros(sizeof(T), g_log2, x.n_dense, x.ldb, x.b_rows, SDD)) {
      if constexpr (SDD) {
        if (x.n_dense % VEC != 0) {
          width(std::true_type{});
          return;
        }
      }
      width(std::false_type{});
      return;
    }
  }
  const auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(FSP_WG_THREADS), 0, s, static_cast<const PT*>(x.indptr),
                       static_cast<const IT*>(x.indices), static_cast<const TV*>(x.data),
                       static_cast<const QT*>(x.perm), static_cast<const T*>(x.B), x.ldb, static_cast<T*>(x.C),
                       x.ldc, x.n_dense, g_log2, partials, tab, sd);
  };
  if constexpr (SDD && VEC > 1) {
    if (x.n_dense % VEC != 0) {
      launch(spmm_slots_kernel<T, TV, IT, PT, QT, VEC, UNROLL, PERM, OFF32, SDD, true>);
      return;
    }
  }
  launch(spmm_slots_kernel<T, TV, IT, PT, QT, VEC, UNROLL, PERM, OFF32, SDD, false>);
}

template <typename T, typename TV, typename IT, typename PT, typename QT, int VEC, bool PERM, bool SDD>
static int launch_spmm(const spmm_args& x, const fsp_csr_plan* plan, hipStream_t s) {
  using A = typename acc_of<TV>::type;
  const int64_t vcols = ceil_div(x.n_dense, VEC);
  int G = x.lanes_n;
  if (G <= 0) {
    G = 1;
    while (G < 64 && G < vcols) G <<= 1;
  }
  if (G > 64 || !is_pow2(G)) return fail(FSP_ERR_ARG, "fsp_spmm_csr: lanes_n %d must be a power of two <= 64", G);
  const int g_log2 = ilog2(G);
  const int max_s_log2 = 6 - g_log2;
  launch_table tab;
  const int64_t blocks = build_launch_table(
      plan, max_s_log2, max_s_log2,
      [g_log2](int sl, int) { return int64_t(FSP_WAVES) * (int64_t(64) >> (g_log2 + sl)); }, &tab);
  const int64_t partial_bytes = plan->n_segments * x.n_dense * (int64_t)sizeof(A);
  if (plan->n_segments > 0 && (plan->partials_dev == nullptr || plan->partials_bytes < partial_bytes)) {
    return fail(FSP_ERR_WORKSPACE, "fsp_spmm_csr: partials need %lld bytes", (long long)partial_bytes);
  }
  A* partials = static_cast<A*>(plan->partials_dev);
  const int64_t ytiles = ceil_div(vcols, G);
  if (ytiles > 65535) return fail(FSP_ERR_ARG, "fsp_spmm_csr: n_dense %lld too large", (long long)x.n_dense);
  if (SDD && ytiles != 1) {  // a dot needs all of a row's columns in one lane group
    return fail(FSP_ERR_ARG, "fsp_spmm_csr_trans_sddmm: n_dense %lld exceeds one lane group (%d columns)",
                (long long)x.n_dense, G * VEC);
  }
  if (blocks > 0) {
    const dim3 grid(static_cast<unsigned>(blocks), static_cast<unsigned>(ytiles));
    // 32-bit byte offsets when every array the kernel addresses fits in 4 GiB,
    // whatever the row pointer's type (its values fit then too).  With 64-bit
    // pointers and 64-bit offsets the f64 N = 75 product above took 301 us
    // against 290 us, the K = 128 f32 SDDMM 192 against 189 us.  Groups of one
    // or two lanes are the other way round or even (int64 indices, 64-bit offsets
    // / 32-bit ones: 104608-node graph, bf16 N = 16 20.7 / 21.4 us, f32 N = 8 21.2
    // / 21.2; 150000 uniform rows, f64 N = 4 34.1 / 35.4).
    const int64_t lim = int64_t(1) << 32;
    const bool off32 = (std::is_same<PT, int32_t>::value || G >= 4) && (!(PERM || SDD) || std::is_same<QT, int32_t>::value) &&
                       x.nnz * (int64_t)sizeof(TV) < lim && x.nnz * (int64_t)sizeof(IT) < lim &&
                       x.nnz * (int64_t)sizeof(QT) < lim && x.b_rows * x.ldb * (int64_t)sizeof(T) < lim &&
                       x.n_rows * x.ldc * (int64_t)sizeof(T) < lim && partial_bytes < lim &&
                       (!SDD || x.n_rows * x.ldbj * (int64_t)sizeof(T) < lim);
    if (off32) {
      using Q32 = int32_t;
      if (plan->unroll >= 8) {
        launch_bins<T, TV, IT, PT, Q32, VEC, 8, PERM, true, SDD>(x, grid, g_log2, partials, tab, s);
      } else {
        launch_bins<T, TV, IT, PT, Q32, VEC, 4, PERM, true, SDD>(x, grid, g_log2, partials, tab, s);
      }
    } else {
      launch_bins<T, TV, IT, PT, QT, VEC, 4, PERM, false, SDD>(x, grid, g_log2, partials, tab, s);
    }
    const int st = check_launch("spmm_bins");
    if (st) return st;
  }
  if (plan->n_long_rows > 0) {
    int64_t g = ceil_div(plan->n_long_rows, FSP_WAVES);
    if (g > 65536) g = 65536;
    hipLaunchKernelGGL((spmm_long_reduce_kernel<T, A>), dim3(static_cast<unsigned>(g)), dim3(FSP_WG_THREADS), 0, s,
                       partials, plan->long_rows_dev, plan->long_seg_ptr_dev, plan->n_long_rows, x.n_dense,
                       static_cast<T*>(x.C), x.ldc);
    return check_launch("spmm_long_reduce");
  }
  return FSP_OK;
}

template <typename T, typename TV, typename IT, typename PT, typename QT, bool PERM, bool SDD = false>
static int launch_spmm_vec(spmm_args x, const fsp_csr_plan* plan, hipStream_t s) {
  // 16 bytes per lane whatever the width, stride and alignment of the dense
  // rows, as long as a row holds one vector.  The element-wise form (VEC 1)
  // needs a lane per column: 75 f64 columns took two 64-lane column tiles of
  // 8-byte loads, 503 us against 301 us here (100003 x 70001, 2.4 M nonzeros).
  constexpr int V = 16 / sizeof(T);
  if (x.n_dense >= V) return launch_spmm<T, TV, IT, PT, QT, V, PERM, SDD>(x, plan, s);
  x.lanes_n = 0;
  return launch_spmm<T, TV, IT, PT, QT, 1, PERM, SDD>(x, plan, s);
}

// Kernel launches of one value type over the index types.  Each value type is
// instantiated in a translation unit of its own (spmm_<type>.hip): together
// they take minutes to compile, side by side one and a half.
template <typename T>
int spmm_launch(int32_t index_type, int32_t indptr_type, int32_t perm_type, const spmm_args& x,
                const fsp_csr_plan* plan, hipStream_t s) {
  FSP_DISPATCH_INDEX(index_type, IT, {
    FSP_DISPATCH_INDEX(indptr_type, PT, {
      if (x.perm == nullptr) return launch_spmm_vec<T, T, IT, PT, int32_t, false>(x, plan, s);
      FSP_DISPATCH_INDEX(perm_type, QT, { return launch_spmm_vec<T, T, IT, PT, QT, true>(x, plan, s); });
    });
  });
  return FSP_OK;
}

template <typename T>
int spmm_sdd_launch(int32_t index_type, int32_t indptr_type, int32_t pos_type, const spmm_args& x,
                    const fsp_csr_plan* plan, hipStream_t s) {
  FSP_DISPATCH_INDEX(index_type, IT, {
    FSP_DISPATCH_INDEX(indptr_type, PT, {
      FSP_DISPATCH_INDEX(pos_type, QT, {
        if (x.perm != nullptr) return launch_spmm_vec<T, T, IT, PT, QT, true, true>(x, plan, s);
        return launch_spmm_vec<T, T, IT, PT, QT, false, true>(x, plan, s);
      });
    });
  });
  return FSP_OK;
}

// Values in the wider type TV (see spmm_bins_kernel).
template <typename T, typename TV>
int spmm_wide_launch(int32_t index_type, int32_t indptr_type, const spmm_args& x, const fsp_csr_plan* plan,
                     hipStream_t s) {
  FSP_DISPATCH_INDEX(index_type, IT, {
    FSP_DISPATCH_INDEX(indptr_type, PT, { return launch_spmm_vec<T, TV, IT, PT, int32_t, false>(x, plan, s); });
  });
  return FSP_OK;
}

#define FSP_SPMM_WIDE_INSTANCE(EXTERN, T, TV) \
  EXTERN template int spmm_wide_launch<T, TV>(int32_t, int32_t, const spmm_args&, const fsp_csr_plan*, hipStream_t);

#define FSP_SPMM_INSTANCES(EXTERN, T)                                                                          \
  EXTERN template int spmm_launch<T>(int32_t, int32_t, int32_t, const spmm_args&, const fsp_csr_plan*, hipStream_t); \
  EXTERN template int spmm_sdd_launch<T>(int32_t, int32_t, int32_t, const spmm_args&, const fsp_csr_plan*, hipStream_t);

}  // namespace fsp
