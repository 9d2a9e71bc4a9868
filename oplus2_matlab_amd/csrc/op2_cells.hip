// One Runge-Kutta stage of a captured graph on cell tiles: res_calc,
// bres_calc, update and, where they follow, save_soln and adt_calc, one
// thread per cell.
#include <algorithm>
#include <type_traits>

#include "op2_cells.h"

namespace op2 {

namespace {

// Square roots and the division by cfl of adt_calc without the scaling and
// the special cases that the library's carry (a third of their instructions),
// for arguments whose exponents lie in Range: Goldschmidt's iteration for the
// root and Markstein's correction of a quotient from the reciprocal rounded to
// nearest, with the residuals exact in fused operations, so that both are
// correctly rounded as the library's are.  Compared with the library's, no
// difference: the roots of all floats of two binades and the quotients of one
// binade by 8 divisors; 4.0e8 random doubles over the whole of Range, roots
// and quotients by 6 divisors.
__device__ __forceinline__ unsigned high_bits(double v) { return (unsigned)__double2hiint(v); }
__device__ __forceinline__ unsigned high_bits(float v) { return __float_as_uint(v); }
template <typename T>
struct Range;  // positive normal numbers far from both ends, as high_bits
template <>
struct Range<double> {
  static constexpr unsigned lo = (1023u - 400u) << 20, hi = (1023u + 400u) << 20;
};
template <>
struct Range<float> {
  static constexpr unsigned lo = (127u - 50u) << 23, hi = (127u + 50u) << 23;
};
__device__ __forceinline__ double near_root(double v) {
  const double y = __builtin_amdgcn_rsq(v);
  double g = v * y, h = 0.5 * y;
  const double r = fma(-h, g, 0.5);
  g = fma(g, r, g);
  h = fma(h, r, h);
  g = fma(fma(-g, g, v), h, g);
  return fma(fma(-g, g, v), h, g);
}
__device__ __forceinline__ float near_root(float v) {
  const float y = __builtin_amdgcn_rsqf(v);
  float g = v * y, h = 0.5f * y;
  const float r = fmaf(-h, g, 0.5f);
  g = fmaf(g, r, g);
  h = fmaf(h, r, h);
  return fmaf(fmaf(-g, g, v), h, g);
}
// v / d, rd = 1 / d rounded to nearest
template <typename T>
__device__ __forceinline__ T near_quotient(T v, T d, T rd) {
  T q = v * rd;
  q = __builtin_elementwise_fma(__builtin_elementwise_fma(-d, q, v), rd, q);
  return __builtin_elementwise_fma(__builtin_elementwise_fma(-d, q, v), rd, q);
}

// adt_of (the same bits), rcfl = 1 / cfl rounded to nearest, or 0 to call
// adt_of always
template <typename T>
__device__ __forceinline__ T adt_near(const T x1[2], const T x2[2], const T x3[2], const T x4[2],
                                      const T q[4], const AirfoilConsts<T> &k, T rcfl) {
  const T ri = T(1) / q[0];
  const T u = ri * q[1], v = ri * q[2];
  const T cc = k.gam * k.gm1 * (ri * q[3] - T(0.5) * (u * u + v * v));
  const T c = near_root(cc);
  unsigned lo = high_bits(cc), hi = lo;
  T s = T(0);
  auto side = [&](const T a[2], const T b[2]) {
    const T dx = b[0] - a[0], dy = b[1] - a[1];
    const T l = dx * dx + dy * dy;
    lo = min(lo, high_bits(l));
    hi = max(hi, high_bits(l));
    return fabs(u * dy - v * dx) + c * near_root(l);
  };
  s = side(x1, x2);
  s += side(x2, x3);
  s += side(x3, x4);
  s += side(x4, x1);
  lo = min(lo, high_bits(s));
  hi = max(hi, high_bits(s));
  if (lo >= Range<T>::lo && hi <= Range<T>::hi && rcfl != T(0))
    return near_quotient(s, k.cfl, rcfl);
  return adt_of(x1, x2, x3, x4, q, k);
}

// a state's four reals, kept out of the caches if `stream`
template <typename T>
__device__ __forceinline__ void store_state(T *p, const T v[4], bool stream) {
  if (!stream) {
    Vec<T>::store4(p, v);
    return;
  }
  typedef T v16 __attribute__((ext_vector_type(16 / sizeof(T))));
#pragma unroll
  for (int j = 0; j < 4 * (int)sizeof(T) / 16; j++) {
    v16 u;
    __builtin_memcpy(&u, v + j * (16 / sizeof(T)), 16);
    __builtin_nontemporal_store(u, reinterpret_cast<v16 *>(p) + j);
  }
}

// LDS of a tile: per cell the state q, adt, and 1 / q[0] and the pressure,
// which every edge of the cell needs (computed once per cell of the tile
// instead of once per edge side), in rows of 16-byte vectors, CAP cells each,
// so that reads of neighbouring cells touch every bank once and one address
// (16 times the cell's number) with constant offsets reaches them all; then
// the nodes' coordinates.
template <typename T, int CAP>
struct TileLds {
  static constexpr int kRows = 4 * sizeof(T) / 16;  // 16-byte vectors of a state
  static constexpr int kVec = 16 / sizeof(T);       // reals of one
  typedef T v16 __attribute__((ext_vector_type(kVec)));
  typedef T v2 __attribute__((ext_vector_type(2)));
  unsigned char *base;
  __device__ __forceinline__ v16 *row(int j, unsigned at) const {
    return reinterpret_cast<v16 *>(base + j * CAP * 16 + at);
  }
  __device__ __forceinline__ void put(unsigned at, const T v[4], T adt, T gm1) const {
#pragma unroll
    for (int j = 0; j < kRows; j++) {
      v16 u;
      __builtin_memcpy(&u, v + j * kVec, 16);
      *row(j, at) = u;
    }
    const T ri = T(1) / v[0];
    const T t[4] = {ri, gm1 * (v[3] - T(0.5) * ri * (v[1] * v[1] + v[2] * v[2])), adt, T(0)};
    v16 u;
    __builtin_memcpy(&u, t, 16);
    *row(kRows, at) = u;
    if (kVec == 2) *reinterpret_cast<T *>(row(kRows + 1, at)) = adt;
  }
  __device__ __forceinline__ void get(unsigned at, T v[4], T &ri, T &p, T &adt) const {
#pragma unroll
    for (int j = 0; j < kRows; j++) {
      const v16 u = *row(j, at);
      __builtin_memcpy(v + j * kVec, &u, 16);
    }
    const v16 u = *row(kRows, at);
    ri = u[0];
    p = u[1];
    adt = kVec == 2 ? *reinterpret_cast<const T *>(row(kRows + 1, at)) : u[kVec - 2];
  }
  // (at: sizeof(v2) times the node's number)
  __device__ __forceinline__ v2 *node(unsigned at) const {
    return reinterpret_cast<v2 *>(base + cells_row_bytes(sizeof(T)) * CAP + at);
  }
  __device__ __forceinline__ void put_x(int i, const T v[2]) const {
    *node(i * sizeof(v2)) = v2{v[0], v[1]};
  }
};

// v plus the value that DPP control CTRL brings (0 from outside, and in rows
// not in ROWS)
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_add(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, ROWS, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, ROWS, 0xf, true);
  return v + __hiloint2double(hi, lo);
}
// The sum of a wavefront in its last lane, in registers alone: rows of 16
// lanes by shifts, then from row to row (18 instructions; the butterfly
// through the LDS takes 35 and 12 permutations).
__device__ __forceinline__ double wave_sum(double v) {
  v = dpp_add<0x111, 0xf>(v);  // row_shr 1, 2, 4, 8
  v = dpp_add<0x112, 0xf>(v);
  v = dpp_add<0x114, 0xf>(v);
  v = dpp_add<0x118, 0xf>(v);
  v = dpp_add<0x142, 0xa>(v);  // row_bcast 15: rows 1 and 3
  return dpp_add<0x143, 0xc>(v);  // row_bcast 31: rows 2 and 3
}

// The bytes of a cell's nodes (four 16-bit offsets in two words) that a
// neighbour's code picks, as v_perm selects them: node i in the low half and
// i + 1 in the high half for code i, the other way round for code 4 + i.
__device__ __forceinline__ unsigned node_selector(unsigned code) {
  const unsigned a = code & 3u, b = (code + 1) & 3u;
  const unsigned pa = 2 * a | (2 * a + 1) << 8, pb = 2 * b | (2 * b + 1) << 8;
  return code & 4u ? pb | pa << 16 : pa | pb << 16;
}

}  // namespace

// One workgroup per tile (after the s.nfold leading workgroups, which fold
// the previous stages' partials), one thread per cell that it finishes:
//  1. stage q and adt of the tile's cells (its own, consecutive in memory
//     on a renumbered mesh, then the rings through its list) and x of its
//     nodes in LDS;
//  2. after a barrier each thread finishes its cell: the fluxes of the
//     cell's edges in the plan's increment order, boundary fluxes, update,
//     and adt_calc of the new state from the cell's four nodes.
// A launch of S stages repeats 2 on the new states, which go back to LDS
// after a barrier: the first stage finishes the owned cells and S - 1 rings,
// each further stage a ring less, the last the owned cells alone, which are
// stored.  Cells in rings are finished by several tiles, with the same bits.
// (1.24 cells finished in the first stage per owned one with 256-cell tiles.)
// An edge between two cells is evaluated by both, so nothing is exchanged
// after the barrier, and the edges need no records of their own.  A cell
// sums exactly what res_calc adds to it, in the same order and with the same
// rounding: the flux is the half sum h of the two cells' fluxes along the
// side plus the dissipation d = mu (q1 - q2); h is odd in the side vector
// and d in the cells, and negation is exact, so -flux of the edge's second
// cell is h of the reversed side plus mu (own - other).  Only the order in
// which h adds its momentum terms depends on which cell is first (`second`).
// MULTI: any number of stages; else one, without the loop (FP64 2.88M cells
// 196 us an iteration as the loop's single pass, 179 without).
template <typename T, bool MULTI, int CAP>
__global__ __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(6, 8))) void k_cells(
    CellArgs<T> s, BresIdx<T> bi, AirfoilConsts<T> k, CarriedFold fold) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ double red[1024 / kWave];
  __shared__ unsigned selector[8];
  if ((int)blockIdx.x < s.nfold) {
    if (carries_fold(fold)) carried_fold<kFixedBlock>(fold, red);
    if (s.nseg > 0 && s.log_count && blockIdx.x == 0 && threadIdx.x == 0)
      *s.log_base = atomicAdd(s.log_count, (unsigned)(s.nseg * s.stages));
    return;
  }
  const int b = xcd_block(blockIdx.x - s.nfold, s.nblk);
  const int *tile = s.tile + kTileInts * b;
  const int *ring = tile + 6;  // ring[j]: cells up to ring j + 1
  const int stages = MULTI ? s.stages : 1;
  const int rings = min(stages, kMaxRings);
  const int o0 = tile[0], no = tile[1], l0 = tile[2];
  const int first_node = tile[3], run = tile[4];
  const int nc = ring[rings - 1], nx = ring[kMaxRings + rings - 1];
  const int done = rings > 1 ? ring[rings - 2] : no;  // cells finished in the first stage
  const int lx = l0 + ring[kMaxRings - 1] - no;       // listed nodes
  const int tid = threadIdx.x, nt = blockDim.x;
  using v2 = typename TileLds<T, CAP>::v2;
  const TileLds<T, CAP> L{smem};

  // One pass over the tile, every load issued before the first is used (no
  // branches: idle threads repeat another's load), the lists first, since the
  // gathers through them are the longest chain.  A thread loads its cell, a
  // node of the run, and a cell of the last ring or a listed node.
  const int nh = nc - done, nl = nh + nx;
  const int own = min(tid, done - 1);
  const int ocell = s.list[l0 + max(own - no, 0)];
  const int li = min(tid, max(nl - 1, 0));
  const int item = s.list[li < nh ? l0 + done - no + li : lx + li - nh];
  const int mine = s.owned ? s.owned[o0 + min(own, no - 1)] : o0 + own;
  int c = own < no ? mine : ocell;
  T vq[4], hq[4], vx[2], hx[2];
  Vec<T>::load2(s.x + 2 * (size_t)(first_node + min(tid, run - 1)), vx);
  const uint4 rec = s.rec[tile[5] + own];
  unsigned w0 = rec.x, w1 = rec.y, w2 = rec.z, w3 = rec.w;
  Vec<T>::load4(s.q_in + 4 * (size_t)c, vq);
  const T va = s.adt_in[c];
  const int hc = tid < nh ? item : c;
  const int hn = tid >= nh && tid < nl ? item : first_node;
  Vec<T>::load4(s.q_in + 4 * (size_t)hc, hq);
  const T ha = s.adt_in[hc];
  Vec<T>::load2(s.x + 2 * (size_t)hn, hx);
  int bidx = -1;
  if (s.bres) {
    const uint2 w = bi.word[c >> 5];
    const unsigned bit = 1u << (c & 31);
    bidx = (w.x & bit) ? (int)(w.y + __popc(w.x & (bit - 1u))) : -1;
  }
  if (tid < 8) selector[tid] = node_selector(tid);
  if (tid < run) L.put_x(tid, vx);
  if (tid < done) L.put(16 * tid, vq, va, k.gm1);
  if (tid < nh)
    L.put(16 * (done + tid), hq, ha, k.gm1);
  else if (tid < nl)
    L.put_x(run + tid - nh, hx);
  // (tiles of more nodes, or of more cells in the last ring, than threads)
  for (int i = tid + nt; i < run; i += nt) {
    Vec<T>::load2(s.x + 2 * (size_t)(first_node + i), vx);
    L.put_x(i, vx);
  }
  for (int i = tid + nt; i < nl; i += nt) {
    if (i < nh) {
      const int g = s.list[l0 + done - no + i];
      Vec<T>::load4(s.q_in + 4 * (size_t)g, hq);
      L.put(16 * (done + i), hq, s.adt_in[g], k.gm1);
    } else {
      Vec<T>::load2(s.x + 2 * (size_t)s.list[lx + i - nh], hx);
      L.put_x(run + i - nh, hx);
    }
  }
  // The cell's (first) boundary edge does not change over the stages: its
  // nodes' difference and its kind are read once, not as a chain of three
  // loads per stage.
  T bd[2] = {T(0), T(0)};
  int bkind = 0, bmesh = 0;
  bool bmore = false;
  if (MULTI && bidx >= 0) {
    const int4 rec = bi.rec[2 * bidx];
    bmore = bi.rec[2 * bidx + 1].z >= 0;
    bkind = bi.bound[rec.z];
    bmesh = rec.w;
    T x1[2], x2[2];
    Vec<T>::load2(bi.x + 2 * (size_t)rec.x, x1);
    Vec<T>::load2(bi.x + 2 * (size_t)rec.y, x2);
    bd[0] = x1[0] - x2[0];
    bd[1] = x1[1] - x2[1];
  }
  // a launch that logs its sums itself takes its slots at once
  unsigned slot = 0;
  if (s.log && tid == 0) slot = atomicAdd(s.log_count, (unsigned)stages);
  // where the state before the iteration is, read again for each stage but
  // the iteration's first (8 registers held over the FP64 edge loop spill)
  // (the iterations of a whole mesh keep it where the first one's was)
  const T *before = s.qold ? s.qold : s.q_in;
  bool first = !s.qold;
  __syncthreads();

#pragma unroll 1
  for (int t = 0; t < stages; t++) {
    // the record stays packed: what is unpacked from it is not to be kept
    // over the stages (43 registers spilled)
    if (MULTI) asm volatile("" : "+v"(w0), "+v"(w1), "+v"(w2), "+v"(w3), "+v"(c));
    const bool last = t + 1 == stages;
    // stages still to come take a ring each
    const int left = min(stages - 1 - t, kMaxRings - 1);
    const int now = left > 0 ? ring[left - 1] : no;
    double acc = 0.0;
    T qn[4], an;
    if (tid < now) {
      T qc[4], rc, pc, ac;
      L.get(16 * tid, qc, rc, pc, ac);
      // twice the sum of the fluxes (res_calc's halves are taken at the end:
      // exact)
      T sum[4] = {T(0), T(0), T(0), T(0)};
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const unsigned w = e < 2 ? w0 : w1, h = e & 1 ? w >> 16 : w;
        const unsigned nb = (h >> 2) & 0x3ff0u;
        if (nb == 16 * kNoCell) break;
        // the side's two nodes, read again from LDS (holding the four side
        // vectors in registers costs a wave per SIMD)
        const unsigned sel =
            *reinterpret_cast<const unsigned *>(reinterpret_cast<const unsigned char *>(selector) +
                                                (h & 0x1cu));
        const unsigned ends = __builtin_amdgcn_perm(w3, w2, sel);
        T qb[4], rb, pb, ab;
        L.get(nb, qb, rb, pb, ab);
        const v2 xa = *L.node(ends & 0xffffu), xb = *L.node(ends >> 16);
        const T dx = xa.x - xb.x, dy = xa.y - xb.y;
        const bool second = h & 1u;
        const T vc = rc * (qc[1] * dy - qc[2] * dx);
        const T vn = rb * (qb[1] * dy - qb[2] * dx);
        const T mu = (ac + ab) * k.eps;
        sum[0] += vc * qc[0] + vn * qb[0] + mu * (qc[0] - qb[0]);
        {
          const T c1 = vc * qc[1], c2 = pc * dy, n1 = vn * qb[1], n2 = pb * dy;
          const T a1 = second ? n1 : c1, a2 = second ? n2 : c2, b1 = second ? c1 : n1,
                  b2 = second ? c2 : n2;
          sum[1] += a1 + a2 + b1 + b2 + mu * (qc[1] - qb[1]);
        }
        {
          const T c1 = vc * qc[2], c2 = pc * dx, n1 = vn * qb[2], n2 = pb * dx;
          const T a1 = second ? n1 : c1, a2 = second ? n2 : c2, b1 = second ? c1 : n1,
                  b2 = second ? c2 : n2;
          sum[2] += a1 - a2 + b1 - b2 + mu * (qc[2] - qb[2]);
        }
        sum[3] += vc * (qc[3] + pc) + vn * (qb[3] + pb) + mu * (qc[3] - qb[3]);
      }
      T r[4] = {T(0), T(0), T(0), T(0)};
      if (t == 0 && !s.zero_res) Vec<T>::load4(s.res + 4 * (size_t)c, r);
#pragma unroll
      for (int d = 0; d < 4; d++) r[d] = r[d] + T(0.5) * sum[d];
      if (MULTI && bidx >= 0) {
        T qi[4] = {k.qinf[0], k.qinf[1], k.qinf[2], k.qinf[3]}, f[4];
        if (bi.qinf_dat) Vec<T>::load4(bi.qinf_dat + 4 * (size_t)bmesh, qi);
        const T at0[2] = {T(0), T(0)};
        boundary_flux(bd, at0, qc, ac, bkind, qi, k, f);
#pragma unroll
        for (int d = 0; d < 4; d++) r[d] += f[d];
      }
      if (MULTI ? bmore : bidx >= 0) {
#pragma unroll 1
        for (int m = MULTI ? 1 : 0; m < 2; m++) {
          const int4 rec = bi.rec[2 * bidx + m];
          if (rec.z < 0) break;
          T x1[2], x2[2], f[4];
          Vec<T>::load2(bi.x + 2 * (size_t)rec.x, x1);
          Vec<T>::load2(bi.x + 2 * (size_t)rec.y, x2);
          T qi[4] = {k.qinf[0], k.qinf[1], k.qinf[2], k.qinf[3]};
          if (bi.qinf_dat) Vec<T>::load4(bi.qinf_dat + 4 * (size_t)rec.w, qi);
          boundary_flux(x1, x2, qc, ac, bi.bound[rec.z], qi, k, f);
#pragma unroll
          for (int d = 0; d < 4; d++) r[d] += f[d];
        }
      }
      T qo[4] = {qc[0], qc[1], qc[2], qc[3]};
      if (!first) Vec<T>::load4(before + 4 * (size_t)c, qo);
      const double adti = 1.0 / (double)ac;
#pragma unroll
      for (int d = 0; d < 4; d++) {
        const double del = adti * (double)r[d];
        qn[d] = (T)((double)qo[d] - del);
        acc += del * del;
      }
      an = ac;
      if (s.adt || !last) {
        T xs[4][2];
#pragma unroll
        for (int n = 0; n < 4; n++) {
          const unsigned w = n < 2 ? w2 : w3;
          const v2 u = *L.node(n & 1 ? w >> 16 : w & 0xffffu);
          xs[n][0] = u.x;
          xs[n][1] = u.y;
        }
        an = adt_near(xs[0], xs[1], xs[2], xs[3], qn, k, s.rcfl);
      }
      if (tid >= no) acc = 0.0;  // (the cell's owner counts it)
      if (!last && (s.saves >> t & 1)) Vec<T>::store4(s.q_in + 4 * (size_t)c, qn);
      if (last) {
        store_state(s.q_out + 4 * (size_t)c, qn, s.stream);
        if (s.qold_out) Vec<T>::store4(s.qold_out + 4 * (size_t)c, qn);
        s.adt_out[c] = an;
        if (s.store_res) {
          const T z[4] = {T(0), T(0), T(0), T(0)};
          Vec<T>::store4(s.res + 4 * (size_t)c, z);
        }
      }
    }
    // the tile's squared moves: wavefronts, then over the wavefronts
    acc = wave_sum(acc);
    if (tid % kWave == kWave - 1) red[tid / kWave] = acc;
    __syncthreads();  // (every old state has been read)
    if (!last && tid < now) L.put(16 * tid, qn, an, k.gm1);
    if (tid == 0) {
      acc = red[0];
      for (int w = 1; w < nt / kWave; w++) acc += red[w];
      if (s.log) {
        *s.out = acc;
        s.log[(slot + t) & (kLogCap - 1)] = acc;
      } else {
        s.partials[(size_t)t * s.nblk + b] = acc;
      }
    }
    if (!last) __syncthreads();
    first = s.saves >> t & 1;
  }
}

template <typename T>
void launch_cells(int threads, const CellArgs<T> &a, const BresIdx<T> &bi,
                  const AirfoilConsts<T> &k, const CarriedFold &fold, size_t lds,
                  hipStream_t stream) {
  const bool multi = a.stages > 1;
  auto pick = [&](auto cap) {
    return multi ? k_cells<T, true, decltype(cap)::value> : k_cells<T, false, decltype(cap)::value>;
  };
  auto kern = a.cells == 256   ? pick(std::integral_constant<int, 256>{})
              : a.cells == 384 ? pick(std::integral_constant<int, 384>{})
              : a.cells == 512 ? pick(std::integral_constant<int, 512>{})
              : a.cells == 768 ? pick(std::integral_constant<int, 768>{})
                               : pick(std::integral_constant<int, 1024>{});
  if (lds > 64 * 1024)
    OP2_HIP_CHECK(hipFuncSetAttribute((const void *)kern,
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  hipLaunchKernelGGL(kern, dim3(a.nblk + a.nfold), dim3(threads), lds, stream, a, bi, k,
                     fold);
}

template void launch_cells<double>(int, const CellArgs<double> &, const BresIdx<double> &,
                                   const AirfoilConsts<double> &, const CarriedFold &, size_t,
                                   hipStream_t);
template void launch_cells<float>(int, const CellArgs<float> &, const BresIdx<float> &,
                                  const AirfoilConsts<float> &, const CarriedFold &, size_t,
                                  hipStream_t);

// The tiles of owner-gather plan p (a res_calc's: arguments 0 and 1 the
// edge's nodes, 6 and 7 its cells) with the nodes of pcell; whole: all cells
// as one tile; wide: aligned pairs of blocks as one tile.
CellTilesHost build_cell_tiles(const Plan &p, op_map pcell, size_t real_bytes, bool whole,
                               bool wide, int depth) {
  CellTilesHost t;
  if (p.ell.empty() || p.perm.empty() || p.maps.size() != 8 || pcell->dim != 4) return t;
  const op_map pedge = p.maps[0], pecell = p.maps[6];
  if (!pedge || p.maps[1] != pedge || !pecell || p.maps[7] != pecell || pcell->from != pecell->to ||
      pcell->to != pedge->to || pedge->dim != 2 || pecell->dim != 2 || p.idxs[0] != 0 ||
      p.idxs[1] != 1 || p.idxs[6] != 0 || p.idxs[7] != 1)
    return t;
  const int *en = map_host(pedge), *ec = map_host(pecell), *cn = map_host(pcell);
  const size_t ncell = pecell->to->size;

  // per cell: its neighbours (-1 after the last) and their side bits
  std::vector<int> nbr(4 * ncell, -1);
  std::vector<uint16_t> bits(ncell, 0);
  for (int b = 0; b < p.nblocks; b++)
    for (int i = p.owned_off[b]; i < p.owned_off[b + 1]; i++) {
      const int c = p.owned[i];
      unsigned used = 0;
      for (int m = 0; m < 4; m++) {
        const unsigned e = p.ell[4 * (size_t)i + m];
        if (e == 0xffffu) break;
        const size_t edge = p.perm[p.blk_off[b] + (e >> 2)];
        const unsigned second = e & 3u;
        if (second > 1 || ec[2 * edge + second] != c) return t;
        const int n1 = en[2 * edge], n2 = en[2 * edge + 1];
        unsigned sd = 4, reversed = 0;
        for (unsigned q = 0; q < 4 && sd == 4; q++) {
          if (used >> q & 1) continue;
          const int u = cn[4 * (size_t)c + q], v = cn[4 * (size_t)c + (q + 1) % 4];
          if (n1 == u && n2 == v) {
            sd = q;
          } else if (n1 == v && n2 == u) {
            sd = q;
            reversed = 1;
          }
        }
        if (sd == 4) return t;
        used |= 1u << sd;
        nbr[4 * (size_t)c + m] = ec[2 * edge + 1 - second];
        bits[c] |= (sd | (reversed ^ second) << 2 | second << 3) << (4 * m);
      }
    }

  // local number of each cell and node in the tile that numbered it last
  std::vector<int> cell_tile(ncell, -1), node_tile(pedge->to->size, -1);
  std::vector<short> cell_loc(ncell), node_loc(pedge->to->size);
  std::vector<int> cells, nodes;
  const int all_nodes = pedge->to->size;
  int stamp = 0;
  t.first_of_block.assign(p.nblocks + 1, 0);

  // one tile of owned cells [lo, hi); false: does not fit
  auto tile = [&](int lo, int hi, int max_done, int max_cells) {
    const int no = hi - lo, id = stamp++;
    int ring[kMaxRings], ring_nodes[kMaxRings], run0 = 0, run = 0;
    cells.assign(p.owned.begin() + lo, p.owned.begin() + hi);
    nodes.clear();
    for (int i = 0; i < no; i++) {
      cell_tile[cells[i]] = id;
      cell_loc[cells[i]] = (short)std::min(i, 0x7fff);
    }
    for (int j = 0, from = 0; j < kMaxRings; j++) {
      if (j >= depth) {
        ring[j] = ring[j - 1];
        ring_nodes[j] = ring_nodes[j - 1];
        continue;
      }
      // the nodes and neighbours of the cells of ring j (0: the owned cells)
      const int to = (int)cells.size();
      if (to > kMaxLocal) return false;
      for (int i = from; i < to; i++) {
        const size_t c = cells[i];
        for (int m = 0; m < 4; m++) {
          const int n = cn[4 * c + m], o = nbr[4 * c + m];
          if (node_tile[n] != id) {
            node_tile[n] = id;
            nodes.push_back(n);
          }
          if (o >= 0 && cell_tile[o] != id) {
            cell_tile[o] = id;
            cell_loc[o] = (short)std::min<size_t>(cells.size(), 0x7fff);
            cells.push_back(o);
          }
        }
      }
      if (j == 0)
        // the longest run of consecutive nodes is read without the list
        for (int n : nodes) {
          if (n > 0 && node_tile[n - 1] == id) continue;  // not the first of its run
          int end = n + 1;
          while (end < all_nodes && node_tile[end] == id) end++;
          if (end - n > run) {
            run0 = n;
            run = end - n;
          }
        }
      from = to;
      ring[j] = (int)cells.size();
      ring_nodes[j] = (int)nodes.size();
    }
    const int done = depth > 1 ? ring[depth - 2] : no;
    const int nc = ring[kMaxRings - 1], nn = ring_nodes[kMaxRings - 1];
    if (nc > kMaxLocal || nn > kMaxLocal) return false;
    if ((done > max_done || std::max(nc, nn) > max_cells) && no > kWave) return false;

    t.tile.insert(t.tile.end(),
                  {lo, no, (int)t.list.size(), run0, run, (int)(t.rec.size() / 4)});
    for (int j = 0; j < kMaxRings; j++) {
      t.tile.push_back(ring[j]);
      t.max_cells[j] = std::max(t.max_cells[j], ring[j]);
      t.max_nodes[j] = std::max(t.max_nodes[j], ring_nodes[j]);
      t.max_done[j] = std::max(t.max_done[j], j < depth ? (j ? ring[j - 1] : no) : done);
    }
    for (int j = 0; j < kMaxRings; j++) t.tile.push_back(ring_nodes[j] - run);
    t.list.insert(t.list.end(), cells.begin() + no, cells.end());
    int listed = run;
    for (int n : nodes) {
      if (n >= run0 && n < run0 + run) {
        node_loc[n] = (short)(n - run0);
      } else {
        node_loc[n] = (short)listed++;
        t.list.push_back(n);
      }
    }
    for (int i = 0; i < done; i++) {
      const size_t c = cells[i];
      unsigned nd[4], half[4];
      for (int m = 0; m < 4; m++) {
        const int o = nbr[4 * c + m];
        nd[m] = (unsigned)node_loc[cn[4 * c + m]] * 2 * (unsigned)real_bytes;
        const unsigned nb = o >= 0 ? (unsigned)cell_loc[o] : kNoCell, sd = bits[c] >> (4 * m) & 15u;
        half[m] = nb << 6 | (sd & 7u) << 2 | sd >> 3;
      }
      for (int m = 0; m < 4; m += 2) t.rec.push_back(half[m] | half[m + 1] << 16);
      for (int m = 0; m < 4; m += 2) t.rec.push_back(nd[m] | nd[m + 1] << 16);
    }
    return true;
  };
  if (whole) {
    if (!tile(0, (int)p.owned.size(), kMaxLocal, kMaxLocal)) return CellTilesHost{};
    t.whole = true;
    std::fill(t.first_of_block.begin() + 1, t.first_of_block.end(), 1);
    t.list.push_back(0);  // (read by tiles without a list)
    return t;
  }
  t.rec.reserve(5 * ncell);
  const int part = wide ? 2 * p.part_size : p.part_size;
  const int most = depth > 1 ? part * 3 / 2 : part;
  const int max_done = std::max((most + kWave - 1) / kWave, 4) * kWave;
  const int max_cells = std::max(depth > 1 ? 2 * part : part * 3 / 2, 256);
  std::vector<std::pair<int, int>> todo;
  // the pieces of the renumbered cells: a pair of blocks lies in one
  const auto segs = rt().set_segments.find(pecell->to);
  const bool pairs = wide && p.owned_identity && segs != rt().set_segments.end();
  size_t sg = 0;
  int base = 0;
  for (int b = 0; b < p.nblocks; b++) {
    t.first_of_block[b] = t.ntiles();
    const int first = p.owned_off[b];
    int end = p.owned_off[b + 1];
    if (pairs) {
      const std::vector<int> &st = segs->second;
      while (sg < st.size() && st[sg] <= first) base = st[sg++];
      const int piece_end = sg < st.size() ? st[sg] : (int)ncell;
      if ((first - base) % part == 0 && end - first == p.part_size && b + 1 < p.nblocks &&
          p.owned_off[b + 2] <= piece_end) {
        end = p.owned_off[b + 2];
        t.first_of_block[++b] = -1;
      }
    }
    todo.assign(1, {first, end});
    while (!todo.empty()) {
      const auto [lo, hi] = todo.back();
      todo.pop_back();
      if (tile(lo, hi, max_done, max_cells)) continue;
      if (hi - lo <= kWave) return CellTilesHost{};
      // halves, the first one next; cut at a multiple of the wavefront
      const int mid = lo + std::max((hi - lo) / 2 / kWave, 1) * kWave;
      todo.push_back({mid, hi});
      todo.push_back({lo, mid});
    }
  }
  t.first_of_block[p.nblocks] = t.ntiles();
  t.list.push_back(0);  // (read by a last tile without a list)
  return t;
}

}  // namespace op2
