// Marching PCG rounds: the two-iteration round of a MIXED cavity that has
// several regions per workgroup, evaluated by waves that march up strips of
// 128 columns instead of by workgroups that stage regions in LDS.
//
// A wave owns PfCav::mown columns of a strip (two cells per lane, a 4-column
// halo each side) and mlen rows. It reads p, r and x row by row, a few rows
// ahead, and carries the chain of the round in registers: with row t of p come
//   a = A p at row t-1;  c = A M a, e = A z, the two steps and the stores at
//   row t-2;  a' = A p'' at row t-3;  c', e' and the Gram sums at row t-4.
// Vertical neighbours are registers, horizontal ones come from the adjacent
// lane (DPP), and a difference of neighbours is formed once and used at both
// of its cells. Cell expressions are those of region_ca and give its bits;
// only the order of the Gram sums follows the strips. There is no barrier and
// no LDS in the loop.
//
// A region's round takes 353 vector instructions a cell (six stencils of five
// LDS reads each, their addresses, a frame of a quarter of its cells) and waits
// at five barriers; a strip's takes 100. What bounds it: at 4096^2 with an
// FP64 iterate the 537 MB it reads and writes (5 TB/s of a copy's rate: 110 us
// of a round; regions took 175, 2.2 times the vector work), below 1536^2 the
// vector work of its short segments. Two cells a lane: with one, 8 of 64 lanes
// would be halo; four do not fit the 128 registers of a 16-wave workgroup.
// Rounds of a 400-iteration solve, solve start included, regions -> strips:
// 1040^2 25.9 -> 22.6 us, 1535^2 45.3 -> 31.7, 2048^2 (FP32 iterate) 46.0 -> 36.1,
// 2560^2 (FP64 iterate) 97.9 -> 61.2, 4096^2 184.7 -> 123.5.
#pragma once

namespace pf {

typedef float MF2 __attribute__((ext_vector_type(2), aligned(4)));
typedef double MD2 __attribute__((ext_vector_type(2), aligned(8)));

constexpr int kStripCols = 2 * TX;           // columns a wave reads
constexpr int kStripOwn = kStripCols - 8;    // of which it may own

// The lane above's (below's) value; 0 in the last (first) lane.
__device__ __attribute__((always_inline)) inline float lane_up(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x130, 0xF, 0xF, true));  // wave_shl:1
}
__device__ __attribute__((always_inline)) inline float lane_down(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x138, 0xF, 0xF, true));  // wave_shr:1
}

// r and p are read again in the next round and stored as usual; an FP64 x goes
// past the caches both ways (4096^2: 123.5 us a round against 126.5 with every
// store streaming and 142.3 with none; 2560^2: 61.2, 63.6, 58.2).
//
// One strip segment. EDGE: it reads or owns cells on or beyond the domain's
// boundary, where neighbours are missing, weights are 1, rows may be
// identity rows, and loads go cell by cell to clamped places.
template <bool XD, bool EDGE>
__device__ __attribute__((always_inline)) inline void march_strip(const PfCav& C, const PhaseArgs& A, int strip, int seg,
                                                                  double (&acc)[NP]) {
  using XT = std::conditional_t<XD, double, float>;
  constexpr int kAhead = (XD && EDGE) ? 1 : 2;  // rows read ahead
  const int nx = __builtin_amdgcn_readfirstlane(C.nx), ny = __builtin_amdgcn_readfirstlane(C.ny);
  const int lane = threadIdx.x;
  const bool init = __builtin_amdgcn_readfirstlane(A.ca_init) != 0;
  const int par = __builtin_amdgcn_readfirstlane(A.par);
  const PF_GLOBAL float* const R = uniform((const float*)mixed_r(C, init ? (par ^ 1) : par));
  const PF_GLOBAL float* const P = uniform((const float*)mixed_p(C, par ^ 1));
  PF_GLOBAL float* const Rn = uniform(mixed_r(C, par ^ 1));
  PF_GLOBAL float* const Pn = uniform(mixed_p(C, par));
  PF_GLOBAL XT* const X = uniform((XT*)(XD ? (void*)C.x64 : C.x));
  const int mown = __builtin_amdgcn_readfirstlane(C.mown), mlen = __builtin_amdgcn_readfirstlane(C.mlen);
  const int i0 = strip * mown, s0 = i0 - 4;  // first own column, first column
  const int i1 = min(i0 + mown, nx);
  const int j0 = seg * mlen, j1 = min(j0 + mlen, ny);
  const int col = s0 + 2 * lane;
  const bool own0 = col >= i0 && col < i1, own1 = col + 1 >= i0 && col + 1 < i1;
  const bool pinned = (C.op == 0);
  const float scx = uniform(pinned ? -A.cx : A.cx), scy = uniform(pinned ? -A.cy : A.cy);
  const float wi = uniform(C.jacobi ? A.minvf : 1.0f);  // interior weight
  // EDGE: no neighbour to the east of a cell (or the cell is left of the domain).
  const bool noE0 = EDGE && (col == nx - 1 || col == -1), noE1 = EDGE && (col + 1 == nx - 1 || col + 1 == -1);
  const bool bc0 = EDGE && (col == 0 || col == nx - 1), bc1 = EDGE && (col + 1 == 0 || col + 1 == nx - 1);
  const float w0 = bc0 ? 1.0f : wi, w1 = bc1 ? 1.0f : wi;
  // EDGE: pairs beyond the domain are read at its first or last two columns; a
  // pair that the east boundary cuts takes its cell from there.
  const unsigned k0 = EDGE ? (unsigned)min(max(col, 0), nx - 2) : (unsigned)col;
  const bool cut = EDGE && col == nx - 1;
  unsigned o4 = 4u * k0, ox = (unsigned)sizeof(XT) * k0;  // byte offsets in a row
  // A place in a row: scalar row address, 32-bit lane offset.
  auto at = [](auto* row, unsigned o, auto kind) {
    using V = decltype(kind);
    return (PF_GLOBAL V*)((const PF_GLOBAL char*)row + o);
  };
  const int tlo = max(j0 - 4, 0), thi = min(j1 + 3, ny - 1);  // rows that are read

  auto load2 = [&](const PF_GLOBAL float* B, int row) -> MF2 {
    const PF_GLOBAL float* q = B + (size_t)min(max(row, tlo), thi) * nx;
    MF2 v = *at(q, o4, MF2{});
    if constexpr (EDGE) v.x = cut ? v.y : v.x;
    return v;
  };
  auto loadx = [&](int row, XT (&v)[2]) {
    const PF_GLOBAL XT* q = X + (size_t)min(max(row, tlo), thi) * nx;
    if constexpr (XD) {
      const MD2 d = __builtin_nontemporal_load(at(q, ox, MD2{}));
      v[0] = d.x;
      v[1] = d.y;
    } else {
      const MF2 d = *at(q, ox, MF2{});
      v[0] = d.x;
      v[1] = d.y;
    }
    if constexpr (EDGE) v[0] = cut ? v[1] : v[0];
  };
  // A's value at a row's two cells f, from the differences to the row above
  // (dn) and below (ds).
  auto lap = [&](int row, MF2 f, MF2 dn, MF2 ds) -> MF2 {
    float d0 = f.y - f.x;
    float d1 = lane_up(f.x) - f.y;
    if constexpr (EDGE) {
      d0 = noE0 ? 0.0f : d0;
      d1 = noE1 ? 0.0f : d1;
    }
    const float dw = lane_down(d1);
    MF2 v;
    v.x = __fmul_rn(d0 - dw, scx) + __fmul_rn(dn.x - ds.x, scy);
    v.y = __fmul_rn(d1 - d0, scx) + __fmul_rn(dn.y - ds.y, scy);
    if constexpr (EDGE) {
      const bool br = row == 0 || row == ny - 1;
      const bool id0 = pinned ? (row == 0 && col == 0) : (br || bc0);
      const bool id1 = pinned ? false : (br || bc1);
      v.x = id0 ? f.x : v.x;
      v.y = id1 ? f.y : v.y;
    }
    return v;
  };
  // Difference of the rows above and at `row`; none across the domain's edges.
  auto diff = [&](int row, MF2 up, MF2 f) -> MF2 {
    MF2 d;
    d.x = up.x - f.x;
    d.y = up.y - f.y;
    if constexpr (EDGE) {
      if (row == ny - 1 || row == -1) d.x = d.y = 0.0f;
    }
    return d;
  };
  auto weigh = [&](int row, MF2 f) -> MF2 {
    MF2 v;
    if constexpr (EDGE) {
      const bool br = row == 0 || row == ny - 1;
      v.x = (br ? 1.0f : w0) * f.x;
      v.y = (br ? 1.0f : w1) * f.y;
    } else {
      v.x = wi * f.x;
      v.y = wi * f.y;
    }
    return v;
  };

  const MF2 zero = {0.0f, 0.0f};
  const float a0 = uniform(A.ca0f), b0 = uniform(A.cb0f), a1 = uniform(A.ca1f), b1 = uniform(A.cb1f);
  const double da0 = XD ? uniform(A.ca0) : 0.0, da1 = XD ? uniform(A.ca1) : 0.0;
  MF2 p1 = zero, p2 = zero, dsP = zero;              // p at rows t-1, t-2; its differences
  MF2 q2 = zero, dsM = zero;                         // a at row t-2; differences of M a
  MF2 r2 = zero, dsZ = zero;                         // r at row t-2; differences of z
  MF2 np3 = zero, np4 = zero, dsNP = zero;           // new p at rows t-3, t-4
  MF2 nr3 = zero, nr4 = zero, dsNZ = zero;           // new r
  MF2 na4 = zero, dsNM = zero;                       // new a at row t-4
  MF2 pf[kAhead], rf[kAhead];
  XT xf[kAhead][2];
  const int t0 = j0 - 4, tend = j1 + 4;
#pragma unroll
  for (int d = 0; d < kAhead; ++d) {
    pf[d] = load2(P, t0 + d);
    rf[d] = load2(R, t0 + d - 1);
    loadx(t0 + d - 2, xf[d]);
  }
  auto step = [&](int t, int d) {
    asm volatile("" : "+v"(o4), "+v"(ox));  // not to be added to the bases ahead of the loop
    MF2 p0 = pf[d];
    const MF2 r1 = rf[d];
    const XT x0 = xf[d][0], x1 = xf[d][1];
    pf[d] = load2(P, t + kAhead);
    rf[d] = load2(R, t + kAhead - 1);
    loadx(t + kAhead - 2, xf[d]);
    if (init) p0 = zero;
    // a at row t-1.
    const MF2 dnP = diff(t - 1, p0, p1);
    const MF2 q1 = lap(t - 1, p1, dnP, dsP);
    dsP = dnP;
    // c and e at row t-2, the two steps (ca_steps).
    const MF2 m1 = weigh(t - 1, q1), m2 = weigh(t - 2, q2);
    const MF2 z1 = weigh(t - 1, r1), z2 = weigh(t - 2, r2);
    const MF2 dnM = diff(t - 2, m1, m2), dnZ = diff(t - 2, z1, z2);
    const MF2 c = lap(t - 2, m2, dnM, dsM), e = lap(t - 2, z2, dnZ, dsZ);
    dsM = dnM;
    dsZ = dnZ;
    MF2 s1, nr2, np2;  // p between the steps; new r and p
    s1.x = (z2.x - a0 * m2.x) + b0 * p2.x;
    s1.y = (z2.y - a0 * m2.y) + b0 * p2.y;
    nr2.x = (r2.x - a0 * q2.x) - a1 * ((e.x - a0 * c.x) + b0 * q2.x);
    nr2.y = (r2.y - a0 * q2.y) - a1 * ((e.y - a0 * c.y) + b0 * q2.y);
    const MF2 nz2 = weigh(t - 2, nr2);
    np2.x = nz2.x + b1 * s1.x;
    np2.y = nz2.y + b1 * s1.y;
    if (t - 2 >= j0 && t - 2 < j1) {
      const size_t rb = (size_t)(t - 2) * nx;
      XT y0, y1;
      if constexpr (XD) {
        y0 = (x0 + da0 * (double)p2.x) + da1 * (double)s1.x;
        y1 = (x1 + da0 * (double)p2.y) + da1 * (double)s1.y;
      } else {
        y0 = (x0 + a0 * p2.x) + a1 * s1.x;
        y1 = (x1 + a0 * p2.y) + a1 * s1.y;
      }
      if (EDGE ? own0 && own1 : own0) {
        *at(Pn + rb, o4, MF2{}) = np2;
        if (!init) {
          *at(Rn + rb, o4, MF2{}) = nr2;
          if constexpr (XD) {
            const MD2 y = {y0, y1};
            pcg_store(y, at(X + rb, ox, MD2{}));
          } else {
            const MF2 y = {y0, y1};
            pcg_store(y, at(X + rb, ox, MF2{}));
          }
        }
      } else if (EDGE && cut) {
        *at(Pn + rb + 1, o4, float{}) = np2.x;
        if (!init) {
          *at(Rn + rb + 1, o4, float{}) = nr2.x;
          pcg_store(y0, at(X + rb + 1, ox, XT{}));
        }
      }
    }
    // The new a at row t-3.
    const MF2 dnNP = diff(t - 3, np2, np3);
    const MF2 na3 = lap(t - 3, np3, dnNP, dsNP);
    dsNP = dnNP;
    // The new c and e at row t-4, and the Gram sums there.
    const MF2 nm3 = weigh(t - 3, na3), nm4 = weigh(t - 4, na4);
    const MF2 nz3 = weigh(t - 3, nr3), nz4 = weigh(t - 4, nr4);
    const MF2 dnNM = diff(t - 4, nm3, nm4), dnNZ = diff(t - 4, nz3, nz4);
    if (t - 4 >= j0 && t - 4 < j1) {
      const MF2 nc = lap(t - 4, nm4, dnNM, dsNM), ne = lap(t - 4, nz4, dnNZ, dsNZ);
      const MF2 mc = weigh(t - 4, nc), me = weigh(t - 4, ne);
      auto gram = [&](float fp, float fz, float fr, float fa, float fma, float fc, float fmc, float fe, float fme) {
        const double dp = fp, dz = fz, dr = fr, da = fa, dma = fma, dc = fc, dmc = fmc, de = fe, dme = fme;
        acc[0] = __fma_rn(dp, da, acc[0]);
        acc[1] = __fma_rn(dp, dc, acc[1]);
        acc[2] = __fma_rn(dp, de, acc[2]);
        acc[3] = __fma_rn(da, dma, acc[3]);
        acc[4] = __fma_rn(da, dmc, acc[4]);
        acc[5] = __fma_rn(da, dz, acc[5]);
        acc[6] = __fma_rn(da, dme, acc[6]);
        acc[7] = __fma_rn(dc, dmc, acc[7]);
        acc[8] = __fma_rn(dc, dz, acc[8]);
        acc[9] = __fma_rn(dc, dme, acc[9]);
        acc[10] = __fma_rn(dr, dz, acc[10]);
        acc[11] = __fma_rn(dz, de, acc[11]);
        acc[12] = __fma_rn(de, dme, acc[12]);
        acc[13] = __fma_rn(dr, dr, acc[13]);
      };
      if constexpr (EDGE) {  // by selects: branches would cost a copy of the sums
        auto u = [&](float v) -> float { return own0 ? v : 0.0f; };
        auto v = [&](float w) -> float { return own1 ? w : 0.0f; };
        gram(u(np4.x), u(nz4.x), u(nr4.x), u(na4.x), u(nm4.x), u(nc.x), u(mc.x), u(ne.x), u(me.x));
        gram(v(np4.y), v(nz4.y), v(nr4.y), v(na4.y), v(nm4.y), v(nc.y), v(mc.y), v(ne.y), v(me.y));
      } else if (own0) {
        gram(np4.x, nz4.x, nr4.x, na4.x, nm4.x, nc.x, mc.x, ne.x, me.x);
        gram(np4.y, nz4.y, nr4.y, na4.y, nm4.y, nc.y, mc.y, ne.y, me.y);
      }
    }
    dsNM = dnNM;
    dsNZ = dnNZ;
    p2 = p1;
    p1 = p0;
    q2 = q1;
    r2 = r1;
    np4 = np3;
    np3 = np2;
    nr4 = nr3;
    nr3 = nr2;
    na4 = na3;
  };
  for (int t = t0; t < tend; t += kAhead) {
#pragma unroll
    for (int d = 0; d < kAhead; ++d) step(t + d, d);  // a row beyond tend is nobody's
  }
}

// The round of workgroup b: the Gram sums of its waves' strips.
template <bool XD>
__device__ __attribute__((always_inline)) inline void march_ca(const PfCav& C, const PhaseArgs& A, int b,
                                                               double (&acc)[NP]) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.y);
  const int task = b * C.mwaves + wave;
  if (wave >= C.mwaves || task >= C.mstrips * C.msegs) return;
  const int seg = __builtin_amdgcn_readfirstlane(task / C.mstrips);
  const int strip = __builtin_amdgcn_readfirstlane(task - seg * C.mstrips);
  const int s0 = strip * C.mown - 4, j0 = seg * C.mlen;
  if (s0 >= 1 && s0 + kStripCols <= C.nx - 1 && j0 - 4 >= 1 && j0 + C.mlen + 4 <= C.ny - 1)
    march_strip<XD, false>(C, A, strip, seg, acc);
  else
    march_strip<XD, true>(C, A, strip, seg, acc);
}

}  // namespace pf
