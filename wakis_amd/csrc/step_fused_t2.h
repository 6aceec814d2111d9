// Two leapfrog steps per launch (temporal blocking) for the wakefield step:
// material codes, masks folded into the coefficients (zero_masked), the beam
// line fed from the beam table, with or without conduction (COND: J = sigma E
// everywhere, recomputed from E as in k_fused4 and stored by the last launch
// of a call).
//
// A workgroup owns T rows of OW cells (both chosen by the host for the grid)
// and a chunk of z-planes and marches up in z like k_fused4, but carries two
// time levels, the second one plane behind the first: at plane k it computes
// step n+1 (level 1: H1(k), E1(k)) and step n+2 at plane k-1 (level 2: H2(k-1),
// E2(k-1)), and stores only level 2. Level 2 on the own rows needs level-1
// values on rows j0-1 .. j0+T (E1) and j0-2 .. j0+T (H1), so the workgroup
// holds T + 4 rows, row r = j0-2+r (the last one only stages E0 of row
// j0+T+1); along x it holds one lane (V cells) more on each side of the own
// cells, unless one tile spans the row. Halo values are recomputed, never
// exchanged. Every value is formed by the same expression as in k_fused4
// (h_row, e_sum, the coefficient recomputation from the codes), so both levels
// are bit-identical to two single steps.
//
// Thread t holds the V cells of lane t % Q of row t / Q, so rows of any length
// fill the waves; a lane that the row end cuts loads and stores its cells one
// at a time, the others with 16-byte accesses at the alignment the row has.
// A staged row is Q lanes, the first of them without cells where a tile starts
// at the row's first cell (its zeros are the cells before this row and after
// the previous one), and lies in LDS in thread order: 64 lanes then take 64
// consecutive words (a gap between the rows of a wave cost a second pass of
// every access). Rows of exactly whole waves keep the gap instead of the lane.
//
// Per plane, with a barrier after P1 and one after P2:
//   P1 H1(k) on rows 0..T+2; stage H1(k); issue the loads of H0(k+1) and of the
//      metric rows of plane k+1
//   P2 E1(k) on rows 1..T+2; H2(k-1) on rows 1..T+1 (reads E1(k-1) staged in
//      the previous P3); stage H2(k-1), E0(k+1) and the metric rows; issue the
//      loads of E0(k+2) and of the codes of plane k+1
//   P3 E2(k-1) on rows 2..T+1, stores; stage E1(k)
// P3 and the next P1 touch different buffers and need no barrier between them.
// The loads of H0 are in flight over a plane, those of E0 over P3 (issued with
// E0's, H0 cost 641 / 596 ms a pass at 256x256x512 FP32, 172 / 153 with
// conduction at 200x200x400, 93 / 83 at 160x160x200 FP64; E0 a plane earlier,
// in 12 more registers, gave nothing). No register is
// copied from a load before its use, and the per-plane scalars (Lz, tLz, the
// beam) are staged in LDS once per launch, so the waves rarely wait for
// memory. LDS holds one block per component and cell of a lane, rows end to
// end in it, so a single-word read takes consecutive words in consecutive
// lanes (no bank conflicts). E and H are read once and written once per two
// steps.
//
// On weight codes (FP32, weight_codes.h) a cell's code names a row of finished
// weights in LDS: 6 values for its H rows and 6 for its E rows in two reads
// each, no metric values, rings or scalars beside them; the row 0 of zeros stands
// for cells off the grid.
//
// What bounds it: memory on large FP32 grids (256x256x512: 1.70 GB per launch at
// 5.1 TB/s, the rate of a device copy); elsewhere the chain of a plane, LDS passes
// and the instructions its 12 waves issue between two barriers (a wave and plane, by
// the counters at 256x256x512: 383 VALU and 79 LDS on weight codes, 555 and 94 on
// material codes). One branch per update and none per cell, buffer loads that return zeros
// off the grid, own neighbours from registers. us per step, one step per launch (or
// rows of one wave and a branch per cell, *) -> this form on material codes -> now:
// 256x256x512 FP32 197* -> 188 -> 165, 200x200x400 FP32 with conduction 149* -> 111
// -> 85, 300x220x180 FP32 270 -> 99 -> 66, 91x75x161 FP32 35 -> 17.6 -> 12.4,
// 160x160x200 FP64 267 -> 66 -> 58, 48x48x128 FP64 17.2 -> 9.4 -> 8.6.
#pragma once
#include "step_fused4.h"
#include "t2_limits.h"
#include "weight_codes.h"

namespace wf {

// One launch of the two-step kernel over a grid.
struct T2Aux {
  int ixs, iys;
  int cap_ix0, cap_iy0, cap_nx, cap_ny;
  int64_t cap_samples, cap_sample;
  int KZ, ntx, nty, ntz;  // planes per chunk, tiles
  int T, OW;              // own rows and cells of a tile
  int Q, QS;              // lanes and LDS slots of a staged row
  int l0, ln;             // own lanes of a row: l0 .. l0 + ln - 1, lane l0 at the tile's first cell
  int stream;             // FP32: stores are streamed past the caches
  int skip_j;             // COND: 1 = J is stored by a later launch of the call
};

// Threads of a workgroup at most, and LDS slots per block of the staged E0, H1,
// E1, H2 (a buffer of R rows takes R * QS + 1 slots): 126.7 KB FP32, 132.6 KB FP64
// of the CU's 160
constexpr int T2_NT = 768;
struct T2Slots {
  static constexpr int E0 = 832, H1 = 768, E1 = 704, H2 = 704;
};

// An array behind a buffer descriptor: a lane addresses it with a byte offset
// of its own plus a uniform one (plane and component), so a plane's accesses
// need no address arithmetic, and a lane whose own offset is OOB reads zeros
// and writes nothing, so they need no branch (t2_limits.h).
typedef __amdgpu_buffer_rsrc_t Buf;
__device__ __forceinline__ Buf buf_of(const void *p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, (int)bytes, 0x00020000);
}
template <typename S>
__device__ __forceinline__ S buf_ld1(Buf b, uint32_t v, uint32_t s) {
  if constexpr (sizeof(S) == 4) {
    return __builtin_bit_cast(S, __builtin_amdgcn_raw_buffer_load_b32(b, (int)v, (int)s, 0));
  } else {
    return __builtin_bit_cast(S, __builtin_amdgcn_raw_buffer_load_b64(b, (int)v, (int)s, 0));
  }
}
// The byte offsets of a lane's V cells: v for a whole lane; with RAG a lane that
// the row end cuts has v = OOB and one offset per cell instead.
template <int V>
struct Offs {
  uint32_t v, c[V - 1];
  bool cut;
};
// V cells of each of NC components (cstep bytes apart), 16 bytes at the
// alignment the row has; zeros unless `in` (uniform: a select costs less here
// than a branch, which the loads could not be scheduled across)
template <bool RAG, typename S, int NC, int V>
__device__ __forceinline__ void buf_ld(Buf b, const Offs<V> &o, bool in, uint32_t s,
                                       uint32_t cstep, S (&d)[NC][V]) {
  typedef S vec __attribute__((ext_vector_type(V)));
  const uint32_t v = in ? o.v : OOB;
  s = in ? s : 0;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const vec t = __builtin_bit_cast(
        vec, __builtin_amdgcn_raw_buffer_load_b128(b, (int)v, (int)(s + c * cstep), 0));
#pragma unroll
    for (int q = 0; q < V; ++q) d[c][q] = t[q];
  }
  if (RAG && o.cut && in) {
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int q = 0; q < V - 1; ++q) d[c][q] = buf_ld1<S>(b, o.c[q], s + c * cstep);
  }
}
// the same for stores, with cache policy POL (2: non-temporal)
template <int POL, bool RAG, typename S, int NC, int V>
__device__ __forceinline__ void buf_st_pol(Buf b, const Offs<V> &o, uint32_t s, uint32_t cstep,
                                           const S (&d)[NC][V]) {
  typedef S vec __attribute__((ext_vector_type(V)));
  typedef unsigned int u4 __attribute__((ext_vector_type(4)));
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    vec t;
#pragma unroll
    for (int q = 0; q < V; ++q) t[q] = d[c][q];
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4, t), b, (int)o.v,
                                           (int)(s + c * cstep), POL);
  }
  if (RAG && o.cut) {
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int q = 0; q < V - 1; ++q) {
        if constexpr (sizeof(S) == 4)
          __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned int, d[c][q]), b,
                                                (int)o.c[q], (int)(s + c * cstep), POL);
        else
          __builtin_amdgcn_raw_buffer_store_b64(
              __builtin_bit_cast(decltype(__builtin_amdgcn_raw_buffer_load_b64(b, 0, 0, 0)),
                                 d[c][q]),
              b, (int)o.c[q], (int)(s + c * cstep), POL);
      }
  }
}

// FP64 is always streamed past the caches, FP32 on the host's rule (t2_aux)
template <bool RAG, typename S, int NC, int V>
__device__ __forceinline__ void buf_st(bool stream, Buf b, const Offs<V> &o, uint32_t s,
                                       uint32_t cstep, const S (&d)[NC][V]) {
  if (sizeof(S) == 8 || stream) buf_st_pol<2, RAG>(b, o, s, cstep, d);
  else buf_st_pol<0, RAG>(b, o, s, cstep, d);
}

// Dynamic LDS of a workgroup in values of S: the ring of iAy / itAy rows, the
// x metric, the ring of iAx / itAx values, the per-plane scalars, the material
// table; on weight codes the table of weights and the beam.
__host__ __device__ inline int t2_dyn_values(int V, int Q, int T, int KZ, int nmat, bool wc) {
  if (wc) return WC_ROW * nmat + 2 * (KZ + 3);
  return 8 * Q * V + 6 * (T + 4) + 4 * (KZ + 3) + 9 * nmat;
}

// The rows of h_row and e_sum with their weights given (w0 of terms 0 and 1, w1
// of terms 2 and 3) and without the first addition to zero, which changes no
// value but the sign of a zero sum: an H or E that is not -0 itself stays the
// same bit for bit.
template <bool DESC, typename S>
__device__ __forceinline__ S t2_h(S h, S w0, S w1, S e0, S e1, S e2, S e3, int s0, int s2) {
  const S p0 = w0 * e0, p1 = w0 * e1, p2 = w1 * e2, p3 = w1 * e3;
  S acc;
  if (!DESC) {
    acc = s0 > 0 ? p0 - p1 : p1 - p0;
    acc = s2 > 0 ? acc + p2 : acc - p2;
    acc = s2 > 0 ? acc - p3 : acc + p3;
  } else {
    acc = s2 > 0 ? p2 - p3 : p3 - p2;
    acc = s0 > 0 ? acc - p1 : acc + p1;
    acc = s0 > 0 ? acc + p0 : acc - p0;
  }
  return h - acc;
}
template <typename S>
__device__ __forceinline__ S t2_e(S w0, S w1, S h0, S h1, S h2, S h3, int s0, int s2) {
  const S p0 = w0 * h0, p1 = w0 * h1, p2 = w1 * h2, p3 = w1 * h3;
  S acc = s0 > 0 ? p0 - p1 : p1 - p0;
  acc = s2 > 0 ? acc + p2 : acc - p2;
  return s2 > 0 ? acc - p3 : acc + p3;
}

template <typename S, bool COND, bool DESC, bool RAG, bool WC, bool MON = false>
__device__ __forceinline__ void
t2_tile(const GridDev &g, const MetricDev<S> &m, const S *__restrict__ Ein,
        const S *__restrict__ Hin, S *__restrict__ Eout, S *__restrict__ Hout,
        S *__restrict__ J, const Coefs<S> &cf, S dt, const T2Aux &x,
        const S *__restrict__ beam1, const S *__restrict__ beam2, S *__restrict__ cap,
        const int tile, S *__restrict__ E1out = nullptr) {
  using I = uint32_t;  // byte offsets: every 3N array within 4 GiB
  constexpr int V = 16 / sizeof(S);
  // a row of the table: 9 material values, or (WC) 12 weights, ieps, sigma
  constexpr int NM = WC ? WC_ROW : 9, IE = WC ? 12 : 3, SG = WC ? 15 : 6;
  constexpr int CE0 = T2Slots::E0, CH1 = T2Slots::H1, CE1 = T2Slots::E1, CH2 = T2Slots::H2;
  // blocks [component][cell of the lane][slot]; the slot of lane ln of row r is
  // r * QS + ln + 1; a slot that no lane owns stays 0. Of H_y only the last
  // cell of a lane is read by another one: one block.
  __shared__ S sE0_[3 * V * CE0];        // E0(k), rows j0-2 .. j0+T+1
  __shared__ S sH1_[(2 * V + 1) * CH1];  // H1(k), rows j0-2 .. j0+T
  __shared__ S sE1_[3 * V * CE1];        // E1(k-1) until P3 stages E1(k), rows j0-1 .. j0+T
  __shared__ S sH2_[(2 * V + 1) * CH2];  // H2(k-1), rows j0-1 .. j0+T-1
  extern __shared__ __align__(16) unsigned char s_dyn[];
  const int Q = x.Q, QS = x.QS, T = x.T;
  S *sDyn = reinterpret_cast<S *>(s_dyn);
  S *sCy = sDyn;                          // [plane % 3][iAy, itAy][Q * V]
  S *sX = sCy + 3 * 2 * Q * V;            // [Lx, tLx][Q * V]
  S *sRow = sX + 2 * Q * V;               // [plane % 3][iAx, itAx][T + 4]
  // [Lz, tLz, beam 1, beam 2][KZ + 3], the beams alone on weight codes
  S *sPl = WC ? sDyn + NM * cf.nmat : sRow + 3 * 2 * (T + 4);
  S *sMat = WC ? sDyn : sPl + 4 * (x.KZ + 3);  // [nmat][NM]
  typedef S vec __attribute__((ext_vector_type(V)));
  const auto ldsv = [&](const S *p, S (&o)[V]) {
    const vec v = *reinterpret_cast<const vec *>(p);
#pragma unroll
    for (int q = 0; q < V; ++q) o[q] = v[q];
  };

  for (int t = threadIdx.x; t < cf.nmat * NM; t += blockDim.x) sMat[t] = cf.mat[t];
  // the slots that no lane owns: the one before the first row, and the gaps
  for (int t = threadIdx.x; t <= (QS > Q ? T + 4 : 0); t += blockDim.x) {
    const int s = t * QS;
#pragma unroll
    for (int b = 0; b < 3 * V; ++b) {
      if (t <= T + 4) sE0_[b * CE0 + s] = S(0);
      if (b < 2 * V + 1 && t <= T + 3) sH1_[b * CH1 + s] = S(0);
      if (t <= T + 2) sE1_[b * CE1 + s] = S(0);
      if (b < 2 * V + 1 && t <= T + 1) sH2_[b * CH2 + s] = S(0);
    }
  }

  const int tx = tile % x.ntx, tyz = tile / x.ntx;
  const int tz = tyz / x.nty, ty = tyz - tz * x.nty;
  const int j0 = ty * T, k0 = tz * x.KZ;
  const int kend = min(k0 + x.KZ, g.Nz);
  const int r = (int)threadIdx.x / Q;  // row of the workgroup
  const int ln = (int)threadIdx.x - r * Q;
  const bool act = r < T + 4;
  const int j = j0 - 2 + r;
  const bool rowok = act && (j >= 0) && (j < g.Ny);
  const int xi = tx * x.OW + V * (ln - x.l0);
  // cells of this lane inside the row
  const int nvx = (xi >= 0 && xi < g.Nx) ? (RAG ? min(V, g.Nx - xi) : V) : 0;  // of any row
  const int nv = rowok ? nvx : 0;
  const bool lact = nv > 0;
  const I ES = (I)sizeof(S), NB = (I)g.N * ES, sz = (I)g.sz;
  const I cell = lact ? (I)xi + (I)g.sy * (I)j : (I)0;  // in its plane
  const bool doH1 = r <= T + 2, doE1 = r >= 1 && r <= T + 2;
  const bool doH2 = r >= 1 && r <= T + 1;
  const bool own = lact && r >= 2 && r <= T + 1 && ln >= x.l0 && ln < x.l0 + x.ln;
  // byte offsets of this lane's cells in a plane
  const auto offs = [&](int n, I at_cell, bool on) {
    Offs<V> o;
    o.v = (on && n == V) ? at_cell * ES : OOB;
    o.cut = RAG && on && n > 0 && n < V;
#pragma unroll
    for (int q = 0; q < V - 1; ++q) o.c[q] = (o.cut && q < n) ? (at_cell + (I)q) * ES : OOB;
    return o;
  };
  const Offs<V> of = offs(nv, cell, true);
  Offs<V> ofh = of, ofs = of;  // H0 (not read on the last row); stores
  if (!doH1) ofh.v = OOB;
  if (!own) {
    ofs.v = OOB;
    ofs.cut = false;
  }
  const I vc = (doH1 && nv == V) ? cell : OOB;                 // codes
  // the 2-D metric tables lie in one array, iAx first: rows 0 and 1 read the
  // iAy and itAy of their cells, the first lane of a row its iAx and itAx
  const I yz = (I)g.Ny * (I)g.Nz, xz = (I)g.Nx * (I)g.Nz, xy = (I)g.Nx * (I)g.Ny;
  const Offs<V> ofy = offs(r < 2 ? nvx : 0, (I)xi + (r == 0 ? yz : 2 * yz + xz + xy), r < 2);
  const I vx = (ln == 0 && rowok) ? (I)j * ES : OOB;
  const Buf bEi = buf_of(Ein, 3 * NB), bHi = buf_of(Hin, 3 * NB);
  const Buf bEo = buf_of(Eout, 3 * NB), bHo = buf_of(Hout, 3 * NB);
  const Buf bC = buf_of(cf.code, (I)g.N), bM = buf_of(cf.iAx, 2 * (yz + xz + xy) * ES);
  // slots of this lane: own row in E0 and H1 (P), the rows of the other buffers
  // start one row later
  const int P = r * QS + ln + 1, Pu = P + QS, Pd = P - QS, Pdd = Pd - QS;
  // cell xi + q (0 <= q <= V) of component c at slot s of a buffer
  const auto e0 = [&](int c, int s, int q) -> S & {
    return q >= V ? sE0_[(c * V) * CE0 + s + 1] : sE0_[(c * V + q) * CE0 + s];
  };
  const auto e1 = [&](int c, int s, int q) -> S & {
    return q >= V ? sE1_[(c * V) * CE1 + s + 1] : sE1_[(c * V + q) * CE1 + s];
  };
  // blocks of H: x, z, then the last cell of y
  const auto hb = [](int c, int q) { return c == 0 ? q : c == 2 ? V + q : 2 * V; };
  const auto h1 = [&](int c, int s, int q) -> S & { return sH1_[hb(c, q) * CH1 + s]; };
  const auto h2 = [&](int c, int s, int q) -> S & { return sH2_[hb(c, q) * CH2 + s]; };

  if (!WC && r < 2) {
#pragma unroll
    for (int q = 0; q < V; ++q)
      sX[(r * Q + ln) * V + q] = q < nvx ? (r == 0 ? m.Lx : m.tLx)[xi + q] : S(0);
  }
  S iAz[1][V] = {}, itAz[1][V] = {};
  S Ly = S(0), tLy = S(0);
  if constexpr (!WC) {
    buf_ld<RAG>(bM, of, true, (yz + xz) * ES, 0, iAz);
    buf_ld<RAG>(bM, of, true, (2 * (yz + xz) + xy) * ES, 0, itAz);
    if (rowok) { Ly = m.Ly[j]; tLy = m.tLy[j]; }
  }
  const int qbeam = (lact && j == x.iys && x.ixs >= xi && x.ixs < xi + nv) ? x.ixs - xi : -1;
  // Ez window capture: own cells only, one sample per level
  int capq0 = V, capq1 = 0;
  int64_t capb1 = 0;
  if (cap && own && j >= x.cap_iy0 && j < x.cap_iy0 + x.cap_ny) {
    const int lo = max(xi, x.cap_ix0), hi = min(xi + nv, x.cap_ix0 + x.cap_nx);
    if (lo < hi) {
      capq0 = lo - xi; capq1 = hi - xi;
      capb1 = ((int64_t)(j - x.cap_iy0) * x.cap_samples + x.cap_sample) * g.Nz;
    }
  }
  const auto capture = [&](int64_t at_plane, const S (&ez)[V]) {
    const int64_t capl = (int64_t)x.cap_ny * x.cap_samples * g.Nz;  // stride of one x line
#pragma unroll
    for (int q = 0; q < V; ++q)
      if (q >= capq0 && q < capq1) cap[capb1 + at_plane + (int64_t)(q + xi - x.cap_ix0) * capl] = ez[q];
  };

  const int kstart = max(k0 - 2, 0);
  // per-plane values of planes kstart .. kend, staged once: Lz, tLz, the beam
  // of both levels
  const int NP = x.KZ + 3;
  constexpr int PL0 = WC ? 2 : 0;  // the first of the four that is staged
  for (int t = threadIdx.x; t < (4 - PL0) * NP; t += blockDim.x) {
    const int which = PL0 + t / NP, kk = kstart + t % NP;
    S v = S(0);
    if (kk < g.Nz && kk <= kend) {
      if (which == 0) v = m.Lz[kk];
      else if (which == 1) v = m.tLz[kk];
      else if (which == 2) v = beam1 ? beam1[kk] : S(0);
      else v = beam2 ? beam2[kk] : S(0);
    }
    sPl[t] = v;
  }
  const auto plv = [&](int which, int kk) { return sPl[(which - PL0) * NP + kk - kstart]; };
  const auto ring = [](int kk) { return (kk + 3) % 3; };
  const auto cyv = [&](int which, int slot) { return sCy + ((slot * 2 + which) * Q + ln) * V; };
  // planes past the grid are zeros
  const auto load_e = [&](int kk, S (&o)[3][V]) {
    buf_ld<RAG>(bEi, of, kk < g.Nz, (I)kk * sz * ES, NB, o);
  };
  const auto load_h = [&](int kk, S (&o)[3][V]) {
    buf_ld<RAG>(bHi, ofh, kk < g.Nz, (I)kk * sz * ES, NB, o);
  };
  const auto load_code = [&](int kk) -> uint32_t {
    const bool in = kk < g.Nz;
    const int v = (int)(in ? vc : OOB), s = in ? (int)((I)kk * sz) : 0;
    uint32_t c;
    if constexpr (V == 4) c = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(bC, v, s, 0);
    else c = (uint32_t)(uint16_t)__builtin_amdgcn_raw_buffer_load_b16(bC, v, s, 0);
    if (RAG && of.cut && in) {
      c = 0;
#pragma unroll
      for (int q = 0; q < V - 1; ++q)
        c |= (uint32_t)(uint8_t)__builtin_amdgcn_raw_buffer_load_b8(
                 bC, (int)(q < nv ? cell + (I)q : OOB), s, 0) << (8 * q);
    }
    return c;
  };
  // the weights of cell q's H rows (x: Ly, Lz; y: Lx, Lz; z: Lx, Ly) and E rows
  // (the same of tL) at a lane's codes: from the table, or formed from the
  // material values and the metric rows of the plane at ring slot rs
  struct Metric {
    S ax, z, cy[V], x[V];
  };
  const auto trow = [&](uint32_t cd, int q) {
    return sMat + NM * (int)((cd >> (8 * q)) & 0xffu);
  };
  // which: 0 for H (iA, L), 1 for E (itA, tL)
  const auto metric = [&](int which, int rs, int kk) {
    Metric o = {};
    if constexpr (!WC) {
      o.ax = sRow[(rs * 2 + which) * (T + 4) + r];
      o.z = sPl[which * NP + kk - kstart];
      ldsv(sCy + ((rs * 2 + which) * Q + ln) * V, o.cy);
      ldsv(sX + (which * Q + ln) * V, o.x);
    }
    return o;
  };
  const auto h_w = [&](const S *t, int q, const Metric &o, S (&w)[6]) {
    if constexpr (WC) {
      typedef S v4 __attribute__((ext_vector_type(4)));
      typedef S v2 __attribute__((ext_vector_type(2)));
      const v4 u = *reinterpret_cast<const v4 *>(t);
      const v2 y = *reinterpret_cast<const v2 *>(t + 4);
      w[0] = u[0]; w[1] = u[1]; w[2] = u[2]; w[3] = u[3]; w[4] = y[0]; w[5] = y[1];
    } else {
      const S a0 = (S)(o.ax * t[0]), a1 = (S)(o.cy[q] * t[1]), a2 = (S)(iAz[0][q] * t[2]);
      w[0] = dt * (S)(a0 * Ly); w[1] = dt * (S)(a0 * o.z);
      w[2] = dt * (S)(a1 * o.x[q]); w[3] = dt * (S)(a1 * o.z);
      w[4] = dt * (S)(a2 * o.x[q]); w[5] = dt * (S)(a2 * Ly);
    }
  };
  const auto e_w = [&](const S *t, int q, const Metric &o, S (&w)[6]) {
    if constexpr (WC) {
      typedef S v4 __attribute__((ext_vector_type(4)));
      typedef S v2 __attribute__((ext_vector_type(2)));
      const v2 y = *reinterpret_cast<const v2 *>(t + 6);
      const v4 u = *reinterpret_cast<const v4 *>(t + 8);
      w[0] = y[0]; w[1] = y[1]; w[2] = u[0]; w[3] = u[1]; w[4] = u[2]; w[5] = u[3];
    } else {
      const S b0 = (S)(t[3] * o.ax), b1 = (S)(t[4] * o.cy[q]), b2 = (S)(t[5] * itAz[0][q]);
      w[0] = b0 * tLy; w[1] = b0 * o.z;
      w[2] = b1 * o.x[q]; w[3] = b1 * o.z;
      w[4] = b2 * o.x[q]; w[5] = b2 * tLy;
    }
  };
  struct Row {
    S cy[1][V], ax, bx;
  };
  // the metric rows of plane kk, and their place in the rings
  const auto load_row = [&](int kk, Row &o) {
    if constexpr (WC) return;
    const bool in = kk < g.Nz;
    buf_ld<RAG>(bM, ofy, in, (I)kk * (I)g.Nx * ES, 0, o.cy);
    const I v = in ? vx : OOB, s = in ? (I)kk * (I)g.Ny * ES : 0;
    o.ax = buf_ld1<S>(bM, v, s);
    o.bx = buf_ld1<S>(bM, v, s + (yz + xz + xy) * ES);
  };
  const auto put_row = [&](int kk, const Row &o) {
    if constexpr (WC) return;
    const int slot = ring(kk);
    if (r < 2) {
      vec v;
#pragma unroll
      for (int q = 0; q < V; ++q) v[q] = o.cy[0][q];
      *reinterpret_cast<vec *>(cyv(r, slot)) = v;
    }
    if (ln == 0 && act) {
      sRow[(slot * 2 + 0) * (T + 4) + r] = o.ax;
      sRow[(slot * 2 + 1) * (T + 4) + r] = o.bx;
    }
  };

  S Ek1[3][V], h0[3][V];  // E0(k+1), H0(k)
  uint32_t code = load_code(kstart), codep = 0;
  {
    S Ek[3][V];
    Row row;
    load_e(kstart, Ek);
    load_row(kstart, row);
    load_e(kstart + 1, Ek1);
    load_h(kstart, h0);
    if (act) {
#pragma unroll
      for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int q = 0; q < V; ++q) e0(c, P, q) = Ek[c][q];
    }
    put_row(kstart, row);
  }
  // carried between planes: H1(k-1), H2(k-2) (x, y) and the codes of plane
  // k-1 (level 2's coefficients; its metric values come from the rings). A
  // lane outside the grid holds zeros: its fields and metric values are 0.
  S H1[3][V], E1[3][V], H2[3][V], H1p[3][V], H2p[2][V];
#pragma unroll
  for (int q = 0; q < V; ++q) {
#pragma unroll
    for (int c = 0; c < 3; ++c) H1[c][q] = E1[c][q] = H2[c][q] = H1p[c][q] = S(0);
    H2p[0][q] = H2p[1][q] = S(0);
  }
  __syncthreads();

  for (int k = kstart; k <= kend; ++k) {
    const int p = k - 1;                   // level-2 plane
    const bool l2e = p >= k0 && p < kend;  // E2(p) and H2(p) stored
    const int rk = ring(k), rp = ring(p);

    // ---- P1: H1(k)
    if (doH1) {
      const Metric o = metric(0, rk, k);
      S EX[V], EY[V + 1], EZ[V + 1];
#pragma unroll
      for (int q = 0; q < V + 1; ++q) {
        if (q < V) EX[q] = e0(0, P, q);
        EY[q] = e0(1, P, q); EZ[q] = e0(2, P, q);
      }
#pragma unroll
      for (int q = 0; q < V; ++q) {
        S w[6];
        h_w(trow(code, q), q, o, w);
        H1[0][q] = t2_h<DESC>(h0[0][q], w[0], w[1], EY[q], Ek1[1][q], EZ[q], e0(2, Pu, q),
                              +1, -1);
        H1[1][q] = t2_h<DESC>(h0[1][q], w[2], w[3], EX[q], Ek1[0][q], EZ[q], EZ[q + 1], -1, +1);
        H1[2][q] = t2_h<DESC>(h0[2][q], w[4], w[5], EX[q], e0(0, Pu, q), EY[q], EY[q + 1],
                              +1, -1);
        h1(0, P, q) = H1[0][q];
        h1(2, P, q) = H1[2][q];
        if (q == V - 1) h1(1, P, q) = H1[1][q];
      }
    }
    const int kn = k < kend ? k + 1 : g.Nz;  // nothing is read after the last plane
    Row row;
    load_row(kn, row);
    load_h(kn, h0);
    __syncthreads();

    // ---- P2: E1(k), then H2(k-1)
    if (doE1) {
      const S bm = plv(2, k);
      const Metric o = metric(1, rk, k);
      const S HYm = h1(1, P - 1, V - 1), HZm = h1(2, P - 1, V - 1);  // -x neighbours
      S s2[V];
#pragma unroll
      for (int q = 0; q < V; ++q) {
        const S *t = trow(code, q);
        S w[6];
        e_w(t, q, o, w);
        S d0 = t2_e(w[0], w[1], H1p[1][q], H1[1][q], h1(2, Pd, q), H1[2][q], +1, -1);
        S d1 = t2_e(w[2], w[3], H1p[0][q], H1[0][q], q ? H1[2][q - 1] : HZm, H1[2][q], -1, +1);
        S d2 = t2_e(w[4], w[5], h1(0, Pd, q), H1[0][q], q ? H1[1][q - 1] : HYm, H1[1][q],
                    +1, -1);
        s2[q] = d2;
        const S o0 = e0(0, P, q), o1 = e0(1, P, q), o2 = e0(2, P, q);  // E0(k) as staged
        if (COND) {  // J = sigma E0
          d0 = d0 - t[IE] * (S)(t[SG] * o0);
          d1 = d1 - t[IE + 1] * (S)(t[SG + 1] * o1);
          d2 = d2 - t[IE + 2] * (S)(t[SG + 2] * o2);
        }
        E1[0][q] = (S)(o0 + dt * d0);
        E1[1][q] = (S)(o1 + dt * d1);
        E1[2][q] = (S)(o2 + dt * d2);
      }
      if (qbeam >= 0) {  // the beam's current instead on its line
#pragma unroll
        for (int q = 0; q < V; ++q) {
          const S d2 = s2[q] - trow(code, q)[IE + 2] * bm;
          if (q == qbeam) E1[2][q] = (S)(e0(2, P, q) + dt * d2);
        }
      }
      if (capq0 < capq1 && x.cap_sample < x.cap_samples && k >= k0 && k < kend)
        capture(k, E1[2]);
      if (MON && k >= k0 && k < kend)  // E of the first step, for a field monitor
        buf_st<RAG>(x.stream != 0, buf_of(E1out, 3 * NB), ofs, (I)k * sz * ES, NB, E1);
    }
    if (doH2 && p >= kstart) {  // H2 below plane 0 stays 0
      const Metric o = metric(0, rp, p);
      // E1(p): own row from slot Pd (x neighbour at q = V), row j+1 from slot P
      S EX[V], EY[V + 1], EZ[V + 1];
#pragma unroll
      for (int q = 0; q < V + 1; ++q) {
        if (q < V) EX[q] = e1(0, Pd, q);
        EY[q] = e1(1, Pd, q); EZ[q] = e1(2, Pd, q);
      }
#pragma unroll
      for (int q = 0; q < V; ++q) {
        S w[6];
        h_w(trow(codep, q), q, o, w);
        H2[0][q] = t2_h<DESC>(H1p[0][q], w[0], w[1], EY[q], E1[1][q], EZ[q], e1(2, P, q), +1, -1);
        H2[1][q] = t2_h<DESC>(H1p[1][q], w[2], w[3], EX[q], E1[0][q], EZ[q], EZ[q + 1], -1, +1);
        H2[2][q] = t2_h<DESC>(H1p[2][q], w[4], w[5], EX[q], e1(0, P, q), EY[q], EY[q + 1],
                              +1, -1);
        h2(0, Pd, q) = H2[0][q];
        h2(2, Pd, q) = H2[2][q];
        if (q == V - 1) h2(1, Pd, q) = H2[1][q];
      }
      // H2(k-1) of the own rows is final
      if (l2e) buf_st<RAG>(x.stream != 0, bHo, ofs, (I)p * sz * ES, NB, H2);
    }
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int q = 0; q < V; ++q) H1p[c][q] = H1[c][q];
    // stage E0(k+1): other lanes read this lane's slots in P1 only
    if (act) {
#pragma unroll
      for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int q = 0; q < V; ++q) e0(c, P, q) = Ek1[c][q];
    }
    put_row(k + 1, row);
    // the loads of E0(k+2) before the barrier, FP64 after it (ms a pass: 91x75x161
    // FP32 16.4 against 16.5, 300x220x180 72.4 / 73.7, 160x160x200 FP64 85.2 / 82.6)
    constexpr bool LATE = sizeof(S) == 8;
    uint32_t coden;
    const auto loads = [&]() {
      coden = load_code(kn);
      load_e(k < kend ? k + 2 : g.Nz, Ek1);
    };
    if (!LATE) loads();
    __syncthreads();

    // ---- P3: E2(k-1) on the own rows, stores; stage E1(k). No barrier before
    // the next P1, which reads E0(k+1) and writes H1(k+1) only
    if (LATE) loads();
    if (own && l2e) {
      const S bv2 = plv(3, p);
      const Metric o = metric(1, rp, p);
      const S HYm = h2(1, Pd - 1, V - 1), HZm = h2(2, Pd - 1, V - 1);
      S E2[3][V], s2[V], Jn[3][V];
#pragma unroll
      for (int q = 0; q < V; ++q) {
        const S *t = trow(codep, q);
        S w[6];
        e_w(t, q, o, w);
        S d0 = t2_e(w[0], w[1], H2p[1][q], H2[1][q], h2(2, Pdd, q), H2[2][q], +1, -1);
        S d1 = t2_e(w[2], w[3], H2p[0][q], H2[0][q], q ? H2[2][q - 1] : HZm, H2[2][q], -1, +1);
        S d2 = t2_e(w[4], w[5], h2(0, Pdd, q), H2[0][q], q ? H2[1][q - 1] : HYm, H2[1][q],
                    +1, -1);
        s2[q] = d2;
        const S o0 = e1(0, Pd, q), o1 = e1(1, Pd, q), o2 = e1(2, Pd, q);  // E1(k-1)
        if (COND) {
          d0 = d0 - t[IE] * (S)(t[SG] * o0);
          d1 = d1 - t[IE + 1] * (S)(t[SG + 1] * o1);
          d2 = d2 - t[IE + 2] * (S)(t[SG + 2] * o2);
        }
        E2[0][q] = (S)(o0 + dt * d0);
        E2[1][q] = (S)(o1 + dt * d1);
        E2[2][q] = (S)(o2 + dt * d2);
      }
      if (qbeam >= 0) {
#pragma unroll
        for (int q = 0; q < V; ++q) {
          const S d2 = s2[q] - trow(codep, q)[IE + 2] * bv2;
          if (q == qbeam) E2[2][q] = (S)(e1(2, Pd, q) + dt * d2);
        }
        if (!COND) J[2 * g.N + (int64_t)p * g.sz + cell + qbeam] = bv2;
      }
      if (capq0 < capq1 && x.cap_sample + 1 < x.cap_samples) capture(g.Nz + p, E2[2]);
      buf_st<RAG>(x.stream != 0, bEo, ofs, (I)p * sz * ES, NB, E2);
      if (COND && !x.skip_j) {  // J = sigma E2 by the call's last launch
        const Buf bJ = buf_of(J, 3 * NB);
#pragma unroll
        for (int q = 0; q < V; ++q) {
          const S *t = trow(codep, q);
#pragma unroll
          for (int c = 0; c < 3; ++c) Jn[c][q] = (S)(t[SG + c] * E2[c][q]);
        }
        buf_st<RAG>(x.stream != 0, bJ, ofs, (I)p * sz * ES, NB, Jn);
      }
    }
#pragma unroll
    for (int q = 0; q < V; ++q) { H2p[0][q] = H2[0][q]; H2p[1][q] = H2[1][q]; }
    if (doE1) {
#pragma unroll
      for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int q = 0; q < V; ++q) e1(c, Pd, q) = E1[c][q];
    }
    // level 2 of the next plane uses this plane's coefficients
    codep = code;
    code = coden;
  }
}

template <typename S, bool COND, bool DESC, bool RAG, bool WC>
__global__ void __launch_bounds__(T2_NT)
k_fused4_t2(GridDev g, MetricDev<S> m, const S *__restrict__ Ein, const S *__restrict__ Hin,
            S *__restrict__ Eout, S *__restrict__ Hout, S *__restrict__ J, Coefs<S> cf, S dt,
            T2Aux x, const S *__restrict__ beam1, const S *__restrict__ beam2,
            S *__restrict__ cap) {
  t2_tile<S, COND, DESC, RAG, WC>(g, m, Ein, Hin, Eout, Hout, J, cf, dt, x, beam1, beam2, cap,
                             xcd_tile(blockIdx.x, x.ntx * x.nty * x.ntz));
}

// The same, the E of the first step stored too (E1out).
template <typename S, bool COND, bool DESC, bool RAG, bool WC>
__global__ void __launch_bounds__(T2_NT)
k_fused4_t2_mon(GridDev g, MetricDev<S> m, const S *__restrict__ Ein, const S *__restrict__ Hin,
                S *__restrict__ Eout, S *__restrict__ Hout, S *__restrict__ J, Coefs<S> cf, S dt,
                T2Aux x, const S *__restrict__ beam1, const S *__restrict__ beam2,
                S *__restrict__ cap, S *__restrict__ E1out) {
  t2_tile<S, COND, DESC, RAG, WC, true>(g, m, Ein, Hin, Eout, Hout, J, cf, dt, x, beam1, beam2, cap,
                                    xcd_tile(blockIdx.x, x.ntx * x.nty * x.ntz), E1out);
}

// One grid of a batch that takes its steps in pairs (BatchDesc) and its tiles.
template <typename S>
struct T2Batch {
  BatchDesc<S> b;
  T2Aux x;    // cap_sample is set per launch
  int tile0;  // its first tile in the numbering of the pair launches
};

// Steps s and s + 1 of every grid that takes both in a pair, in one launch. The
// run covers the steps [step0, end); `flip`: the launch reads E2/H2. Each grid has
// its share of the CUs, one workgroup each. 24 grids of 28 to 160 cells a side
// (5.3 million cells), FP32: about 100 us per launch, 50 a step, against 92 + 4.5
// of the one-step kernel and its step counter.
template <typename S, bool COND, bool DESC, bool RAG, bool WC>
__global__ void __launch_bounds__(T2_NT)
k_fused4_t2_batch(const T2Batch<S> *__restrict__ d, int ninst, int ntiles, int s, int step0,
                  int end, int flip) {
  const int tile = xcd_tile(blockIdx.x, ntiles);
  int lo = 0, hi = ninst - 1;  // last descriptor with tile0 <= tile
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (d[mid].tile0 <= tile) lo = mid;
    else hi = mid - 1;
  }
  const T2Batch<S> &e = d[lo];
  if (s >= batch_single0(e.b.nsteps, step0, end, 1)) return;  // whole workgroup
  T2Aux x = e.x;
  x.cap_sample = e.b.cap_sample0 + s;
  x.skip_j = 1;  // J is stored by the single steps at a grid's end
  const GridDev g = e.b.g;
  const MetricDev<S> m = e.b.m;
  const Coefs<S> cf = e.b.cf;
  const S *row = e.b.beam_table + (e.b.beam_row0 + s) * g.Nz;
  t2_tile<S, COND, DESC, RAG, WC>(g, m, flip ? e.b.E2 : e.b.E, flip ? e.b.H2 : e.b.H,
                              flip ? e.b.E : e.b.E2, flip ? e.b.H : e.b.H2, e.b.J, cf, e.b.dt, x,
                              row, row + g.Nz, e.b.cap, tile - e.tile0);
}

}  // namespace wf
