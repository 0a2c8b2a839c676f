// Windowed environment sweep (sequential.py:452-505), the dominant kernel.
//
// A window is a run of consecutive sweep steps (gates in reverse circuit
// order) whose qubits fit in a 4-bit set U.  For the window starting at gate k
// the pass kernel streams (T', phi) once:
//   T'  <- G'^dagger T' for the previous window's updated gates (in order)
//   phi <- G_k^dagger phi
//   R[x][y] = sum_{r not in U} conj(T'[x, r]) phi[y, r]     (16 x 16, MFMA f64)
//   phi <- G_j^dagger phi for the window's other gates
// and the finalize kernel replays the window on the 16-dim space: for each
// gate j the environment is the partial trace of R over U's other bits,
// G'_j = conj(polar(E_j)), then R <- G'_j^T R (target side) and
// R <- R conj(G_{j+1}) (state side).  This equals the gate-by-gate sweep
// exactly (every step of it is local to U), with one pass over HBM per window
// instead of one per gate.
//
// MFMA v_mfma_f64_16x16x4f64 operand layout (checked on gfx950):
//   A[i][k] lane i + 16k,  B[k][j] lane j + 16k,  D[i][j] lane j + 16(i%4), item i/4.
#include "qmx_device.h"
#include "qmx_internal.h"

namespace qmx {

typedef double d4v __attribute__((ext_vector_type(4)));

QMX_DEV uint64_t wdeposit(uint64_t x, uint64_t mask) {
  uint64_t r = 0;
  while (mask) {
    uint64_t low = mask & (~mask + 1ull);
    if (x & 1ull) r |= low;
    x >>= 1;
    mask &= mask - 1ull;
  }
  return r;
}

QMX_DEV int wlocal(uint64_t pmask, int gb) { return __popcll(pmask & ((1ull << gb) - 1ull)); }

template <typename S>
QMX_DEV double2 lds_get(const S* s, int l) { return to_c(s[l]); }

// gate (adjoint) on an LDS tile of storage type S, local bits m1 (site) / m0 (site+1)
template <typename S>
QMX_DEV void wtile_gate_adj(S* s, int t, int width, int m1, int m0, const double2* gm) {
  if (width == 2) {
    const int ng = 1 << (t - 2);
    const int s0 = 1 << m0, s1 = 1 << m1;
    for (int q = threadIdx.x; q < ng; q += blockDim.x) {
      int l0 = (int)insert_zero(insert_zero((uint64_t)q, m0), m1);
      double2 x0 = to_c(s[l0]), x1 = to_c(s[l0 + s0]), x2 = to_c(s[l0 + s1]), x3 = to_c(s[l0 + s0 + s1]);
#pragma unroll
      for (int o = 0; o < 4; ++o) {
        double2 acc = cmulc(gm[0 * 4 + o], x0);
        acc = cfmac(gm[1 * 4 + o], x1, acc);
        acc = cfmac(gm[2 * 4 + o], x2, acc);
        acc = cfmac(gm[3 * 4 + o], x3, acc);
        int idx = o == 0 ? l0 : (o == 1 ? l0 + s0 : (o == 2 ? l0 + s1 : l0 + s0 + s1));
        s[idx] = from_c<S>(acc);
      }
    }
  } else {
    const int ng = 1 << (t - 1);
    const int s1 = 1 << m1;
    for (int q = threadIdx.x; q < ng; q += blockDim.x) {
      int l0 = (int)insert_zero((uint64_t)q, m1);
      double2 x0 = to_c(s[l0]), x1 = to_c(s[l0 + s1]);
      double2 y0 = cfmac(gm[1 * 4 + 0], x1, cmulc(gm[0 * 4 + 0], x0));
      double2 y1 = cfmac(gm[1 * 4 + 1], x1, cmulc(gm[0 * 4 + 1], x0));
      s[l0] = from_c<S>(y0);
      s[l0 + s1] = from_c<S>(y1);
    }
  }
}

// complex64 tiles: gate arithmetic in FP32 (the storage precision)
QMX_DEV float2 fcmulc(float2 a, float2 b) {
  return make_float2(fmaf(a.x, b.x, a.y * b.y), fmaf(a.x, b.y, -a.y * b.x));
}
QMX_DEV float2 fcfmac(float2 a, float2 b, float2 acc) {
  acc.x = fmaf(a.x, b.x, acc.x);
  acc.x = fmaf(a.y, b.y, acc.x);
  acc.y = fmaf(a.x, b.y, acc.y);
  acc.y = fmaf(-a.y, b.x, acc.y);
  return acc;
}

QMX_DEV void wtile_gate_adj_f32(float2* s, int t, int width, int m1, int m0, const float2* gm) {
  if (width == 2) {
    const int ng = 1 << (t - 2);
    const int s0 = 1 << m0, s1 = 1 << m1;
    for (int q = threadIdx.x; q < ng; q += blockDim.x) {
      int l0 = (int)insert_zero(insert_zero((uint64_t)q, m0), m1);
      float2 x0 = s[l0], x1 = s[l0 + s0], x2 = s[l0 + s1], x3 = s[l0 + s0 + s1];
      float2 y[4];
#pragma unroll
      for (int o = 0; o < 4; ++o) {
        float2 acc = fcmulc(gm[0 * 4 + o], x0);
        acc = fcfmac(gm[1 * 4 + o], x1, acc);
        acc = fcfmac(gm[2 * 4 + o], x2, acc);
        acc = fcfmac(gm[3 * 4 + o], x3, acc);
        y[o] = acc;
      }
      s[l0] = y[0]; s[l0 + s0] = y[1]; s[l0 + s1] = y[2]; s[l0 + s0 + s1] = y[3];
    }
  } else {
    const int ng = 1 << (t - 1);
    const int s1 = 1 << m1;
    for (int q = threadIdx.x; q < ng; q += blockDim.x) {
      int l0 = (int)insert_zero((uint64_t)q, m1);
      float2 x0 = s[l0], x1 = s[l0 + s1];
      s[l0] = fcfmac(gm[1 * 4 + 0], x1, fcmulc(gm[0 * 4 + 0], x0));
      s[l0 + s1] = fcfmac(gm[1 * 4 + 1], x1, fcmulc(gm[0 * 4 + 1], x0));
    }
  }
}

template <typename S>
QMX_DEV void wgate(S* s, int t, int width, int m1, int m0, const double2* gm, const float2* gmf);
template <>
QMX_DEV void wgate<float2>(float2* s, int t, int width, int m1, int m0, const double2*, const float2* gmf) {
  wtile_gate_adj_f32(s, t, width, m1, m0, gmf);
}
template <>
QMX_DEV void wgate<double2>(double2* s, int t, int width, int m1, int m0, const double2* gm, const float2*) {
  wtile_gate_adj<double2>(s, t, width, m1, m0, gm);
}

QMX_DEV int wsane(int n, int site, int w) { return (w == 2 && site < n - 1) ? 2 : 1; }

// step -> (layer, site) of the sweep order (reverse circuit order)
QMX_DEV void step_gate(int n, int s, int& layer, int& site) {
  layer = s / n;
  site = n - 1 - s % n;
}

// ---- register-group gate application ------------------------------------
// A lane holds the 16 amplitudes of one group over a 4-bit set (index x, bit
// m of x = m-th lowest bit of the set).  Gate adjoints act on bits (HB, LB)
// of x (LB < 0: one-qubit gate on HB); indices are compile-time.
template <typename C> struct CT;
template <> struct CT<float> {
  using c2 = float2;
  static QMX_DEV c2 mk(double2 v) { return make_float2((float)v.x, (float)v.y); }
  static QMX_DEV c2 mulc(c2 a, c2 b) { return make_float2(fmaf(a.x, b.x, a.y * b.y), fmaf(a.x, b.y, -a.y * b.x)); }
  static QMX_DEV c2 fmac(c2 a, c2 b, c2 acc) {
    acc.x = fmaf(a.x, b.x, acc.x); acc.x = fmaf(a.y, b.y, acc.x);
    acc.y = fmaf(a.x, b.y, acc.y); acc.y = fmaf(-a.y, b.x, acc.y);
    return acc;
  }
};
template <> struct CT<double> {
  using c2 = double2;
  static QMX_DEV c2 mk(double2 v) { return v; }
  static QMX_DEV c2 mulc(c2 a, c2 b) { return cmulc(a, b); }
  static QMX_DEV c2 fmac(c2 a, c2 b, c2 acc) { return cfmac(a, b, acc); }
};

template <typename C, int HB, int LB>
QMX_DEV void grp_adj(typename CT<C>::c2 (&a)[16], const typename CT<C>::c2* g) {
  using T = CT<C>;
  if (LB >= 0) {
#pragma unroll
    for (int x = 0; x < 16; ++x) {
      if (((x >> HB) & 1) || ((x >> (LB < 0 ? 0 : LB)) & 1)) continue;
      const int i0 = x, i1 = x | (1 << (LB < 0 ? 0 : LB)), i2 = x | (1 << HB), i3 = i1 | (1 << HB);
      typename T::c2 x0 = a[i0], x1 = a[i1], x2 = a[i2], x3 = a[i3];
      typename T::c2 y[4];
#pragma unroll
      for (int o = 0; o < 4; ++o) {
        typename T::c2 acc = T::mulc(g[0 * 4 + o], x0);
        acc = T::fmac(g[1 * 4 + o], x1, acc);
        acc = T::fmac(g[2 * 4 + o], x2, acc);
        acc = T::fmac(g[3 * 4 + o], x3, acc);
        y[o] = acc;
      }
      a[i0] = y[0]; a[i1] = y[1]; a[i2] = y[2]; a[i3] = y[3];
    }
  } else {
#pragma unroll
    for (int x = 0; x < 16; ++x) {
      if ((x >> HB) & 1) continue;
      const int i0 = x, i1 = x | (1 << HB);
      typename T::c2 x0 = a[i0], x1 = a[i1];
      a[i0] = T::fmac(g[1 * 4 + 0], x1, T::mulc(g[0 * 4 + 0], x0));
      a[i1] = T::fmac(g[1 * 4 + 1], x1, T::mulc(g[0 * 4 + 1], x0));
    }
  }
}

// code = hb * 2 + (width == 2): width-2 gates have lb = hb - 1
template <typename C>
QMX_DEV void grp_apply(int code, typename CT<C>::c2 (&a)[16], const typename CT<C>::c2* g) {
  switch (code) {
    case 3: grp_adj<C, 1, 0>(a, g); break;
    case 5: grp_adj<C, 2, 1>(a, g); break;
    case 7: grp_adj<C, 3, 2>(a, g); break;
    case 0: grp_adj<C, 0, -1>(a, g); break;
    case 2: grp_adj<C, 1, -1>(a, g); break;
    case 4: grp_adj<C, 2, -1>(a, g); break;
    case 6: grp_adj<C, 3, -1>(a, g); break;
    default: break;
  }
}

// LDS element swizzle: low 5 bits XOR a fold of the higher bits (bijective)
QMX_DEV int swz(int l) { return l ^ (((l >> 5) ^ (l >> 10)) & 31); }

template <typename S> struct StoreC;
template <> struct StoreC<float2> { using C = float; };
template <> struct StoreC<double2> { using C = double; };

// deposit of the low bits of x into the set bits of mask (32-bit)
QMX_DEV uint32_t dep32(uint32_t x, uint32_t mask) {
  uint32_t r = 0;
  while (mask) {
    uint32_t low = mask & (~mask + 1u);
    if (x & 1u) r |= low;
    x >>= 1;
    mask &= mask - 1u;
  }
  return r;
}

// offset of group element x from the 4 positions p[] of its set
QMX_DEV uint32_t xoffs(const int* p, int x) {
  return (((uint32_t)x & 1u) << p[0]) | ((((uint32_t)x >> 1) & 1u) << p[1]) |
         ((((uint32_t)x >> 2) & 1u) << p[2]) | ((((uint32_t)x >> 3) & 1u) << p[3]);
}

QMX_DEV uint32_t group_roffg(const GroupMap& m, int g) { return (uint32_t)wdeposit((uint64_t)g, m.restg); }
QMX_DEV int group_roffl(const GroupMap& m, int g) { return (int)dep32((uint32_t)g, m.restl); }

// gate code of (site, width) inside a 4-bit group set: hb * 2 + (width == 2)
QMX_DEV int gate_code(uint64_t mask, int n, int site, int w) {
  int hb = __popcll(mask & ((1ull << (n - 1 - site)) - 1ull));
  return hb * 2 + (w == 2 ? 1 : 0);
}

// Support of phi in a state's last n steps (its first circuit layer, whose
// gates act on |0..0>): once the gates of steps up to s are removed, the bits
// below s % n are in |0>.  They are set to exactly zero there, which leaves the
// environments' null columns exact, and tiles that have such a bit set are not
// visited: neither phi nor T', which only ever meets phi, is needed there again.
QMX_DEV uint64_t dead_bits(int n, int kb, int s0) {
  return s0 > kb - n && s0 > 0 ? (1ull << ((s0 - 1) % n)) - 1ull : 0ull;
}
// place inside the set `mask` of the bit that the removal of step s's gate
// leaves in |0>, or -1
QMX_DEV int dead_after(uint64_t mask, int n, int kb, int s) {
  const int h = s % n;
  return s >= kb - n && h > 0 ? __popcll(mask & ((1ull << (h - 1)) - 1ull)) : -1;
}

// complex64 fits 4 waves per SIMD without spills; complex128 runs at 2 (a
// 4-wave budget would spill its FP64 groups)
// STAGED: the tiles of T' and phi are copied between HBM and LDS in tile
// order by all threads (coalesced runs of 2^c0 amplitudes, c0 = number of
// lowest state bits inside the tile) and the register groups are read from
// and written to LDS.  The host selects it for windows whose groups stride
// the state by 4 or more amplitudes per lane (gate bits at the lowest state
// bits), where direct group loads would scatter every wave-wide access.
template <typename S, int WPE, bool STAGED>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(WPE))) void window_pass_kernel(
    WinPassArgs<S> a) {
  using C = typename StoreC<S>::C;
  using T = CT<C>;
  using c2 = typename T::c2;
  extern __shared__ char wsm[];
  __shared__ c2 gmat[2 * kMaxWindow][16];
  __shared__ int gcode[2 * kMaxWindow], gdead[2 * kMaxWindow];
  // group element offsets, [side][x]: side 0 = T' over the previous set,
  // side 1 = phi over the current set; global (state) and tile-local
  __shared__ uint32_t xog[2][16];
  __shared__ int xol[2][16];
  __shared__ int rdep[8];
  __shared__ uint32_t hoff[STAGED ? 256 : 1];
  const int b = a.list ? a.list[blockIdx.y] : blockIdx.y;
  const int n = a.n;
  if (a.skip && a.skip[b]) return;
  const int kb = a.layers[b] * n;
  if (a.s0 >= kb) return;
  const int nc = min(a.s1, kb) - a.s0;
  const int np = a.p1 - a.p0;   // previous window (all valid: p1 == s0 < kb)
  if (threadIdx.x >= 64 && threadIdx.x < 96) {
    const int x = threadIdx.x & 15, side = (threadIdx.x >> 4) & 1;
    xog[side][x] = side ? xoffs(a.gu.ubit, x) : xoffs(a.gp.ubit, x);
    xol[side][x] = (int)(side ? xoffs(a.gu.ux, x) : xoffs(a.gp.ux, x));
    if (threadIdx.x < 72) rdep[x] = group_roffl(a.gu, 4 * x);
  }
  // one gate entry per thread ((np + nc) * 16 <= 256)
  if ((int)threadIdx.x < (np + nc) * 16) {
    const int j = threadIdx.x >> 4, e = threadIdx.x & 15;
    const int s = j < np ? a.p0 + j : a.s0 + (j - np);
    int layer, site;
    step_gate(n, s, layer, site);
    const size_t gi = ((size_t)b * a.lmax + layer) * n + site;
    gmat[j][e] = T::mk(a.gates[gi * 16 + e]);
    if (e == 0) {
      gcode[j] = gate_code(j < np ? a.gp.mask : a.gu.mask, n, site, wsane(n, site, a.widths[gi]));
      gdead[j] = j < np ? -1 : dead_after(a.gu.mask, n, kb, s);
    }
  }
  // staged copies: tile-local index l -> state offset (l & lomask) + hoff[l >> c0]
  const uint64_t pbits = ((1ull << n) - 1ull) & ~a.qmask;
  const int c0 = STAGED ? __builtin_ctzll(~pbits) : 0;
  if (STAGED) {
    for (int h = threadIdx.x; h < (1 << (a.t - c0)); h += blockDim.x)
      hoff[h] = (uint32_t)wdeposit((uint64_t)h << c0, pbits);
  }
  __syncthreads();
  const int t = a.t;
  const size_t len = (size_t)1 << n;
  S* sT = reinterpret_cast<S*>(wsm);
  S* sP = sT + (1 << t);
  const bool first = (np == 0);
  // T' is first written by window 1: windows 0 and 1 read the target
  const S* tsrc = (a.p0 == 0 ? a.target : a.tprime) + (size_t)b * len;
  S* tdst = a.tprime + (size_t)b * len;
  S* phi = a.phi + (size_t)b * len;
  const uint64_t qmask = a.qmask & ~dead_bits(n, kb, a.s0);   // the live tiles' bits
  const long ntiles = 1l << __popcll(qmask);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int ngroups = 1 << (t - 4);
  // lanes [0, ngroups): T' groups over the previous set; [ngroups, 2 ngroups): phi groups
  const int task = threadIdx.x;
  const bool tside = task < ngroups;
  const bool active = task < 2 * ngroups;
  const int grp = tside ? task : task - ngroups;
  // One code path for both sides: this lane's set (bit positions in the state
  // and in the tile), source/destination, gate range and the point at which
  // the group is deposited in LDS (after all previous-window gates for T',
  // after the first current-window gate for phi).
  const uint64_t restg = tside ? a.gp.restg : a.gu.restg;
  const uint32_t restl = tside ? a.gp.restl : a.gu.restl;
  const uint32_t roffg = active ? (uint32_t)wdeposit((uint64_t)grp, restg) : 0u;
  const int roffl = active ? (int)dep32((uint32_t)grp, restl) : 0;
  const uint32_t* xg = xog[tside ? 0 : 1];
  const int* xl = xol[tside ? 0 : 1];
  const S* src = tside ? tsrc : phi;
  S* dst = tside ? tdst : phi;
  S* lds = tside ? sT : sP;
  const bool store_dst = a.store && (tside ? !first : true);
  const int g0 = tside ? 0 : np;
  const int ngate = tside ? np : nc;
  const int lds_after = tside ? np : 1;
  // R phase: wave w takes rest indices [w kper, (w + 1) kper), 4 per k-step
  const int kper = ngroups / 4;
  const int xl_i = (int)xoffs(a.gu.ux, lane & 15);
  // rest index of this lane at k-step k: r = wave kper + 4k + lane / 16, three
  // disjoint bit fields (kper = 2^(t-6) >= 4), so its tile offset is the OR of
  // a per-lane part and the per-step part rdep[k]
  const int rlane = xl_i + group_roffl(a.gu, wave * kper + (lane >> 4));
  d4v acc_r = {0, 0, 0, 0}, acc_i = {0, 0, 0, 0};
  const uint32_t lomask = (1u << c0) - 1u;
  // Direct loads: a group is dead once stored, so the next tile's group is
  // loaded into the same registers right then and its loads stay in flight
  // through the barriers and the R phase.  The next tile is this block's
  // alone (tiles go round-robin over the blocks), so no other block writes it.
  c2 v[16];
  auto load_group = [&](uint32_t g) {
#pragma unroll
    for (int x = 0; x < 16; ++x) v[x] = T::mk(to_c(src[g + xg[x]]));
  };
  if (!STAGED && active && (long)blockIdx.x < ntiles)
    load_group((uint32_t)wdeposit((uint64_t)blockIdx.x, qmask) + roffg);
  // Staged tiles of 2^kWinTileBits amplitudes over 256 threads: the 128
  // T'-side threads copy the T' tile (16 amplitudes each, tile order), the
  // 128 phi-side threads the phi tile, through the group registers v.  The
  // next tile's loads are issued into v once v is dead (T' side: after the
  // group phase; phi side: once its final values are back in LDS), and v is
  // written to LDS at the next tile's start.
  // With a contiguous low run of c0 >= 7 bits, tile index sl0 + 128 i
  // (sl0 < 128) sits at state offset sl0 + ((128 i) & lomask) + hoff[(128 i)
  // >> c0]: a per-lane part and a block-uniform part.
  const bool fast_stage = STAGED && t == kWinTileBits && blockDim.x == 256 && c0 >= 7;
  const int sl0 = threadIdx.x & 127;
  uint32_t ust[16];
#pragma unroll
  for (int i = 0; i < 16; ++i)
    ust[i] = fast_stage ? __builtin_amdgcn_readfirstlane(((128u * i) & lomask) + hoff[(128 * i) >> c0]) : 0u;
  auto load_stage = [&](uint32_t tb) {
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = T::mk(to_c(src[tb + ust[i] + sl0]));
  };
  if (fast_stage && (long)blockIdx.x < ntiles) load_stage((uint32_t)wdeposit((uint64_t)blockIdx.x, qmask));
  for (long tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
    const uint32_t base = (uint32_t)wdeposit((uint64_t)tile, qmask);
    const uint32_t gb = base + roffg;
    const long nxt = tile + gridDim.x;
    if (STAGED) {
      if (fast_stage) {
#pragma unroll
        for (int i = 0; i < 16; ++i) lds[swz(sl0 + 128 * i)] = from_c<S>(make_double2(v[i].x, v[i].y));
      } else {
        for (int l = threadIdx.x; l < (1 << t); l += blockDim.x) {
          const uint32_t off = base + ((uint32_t)l & lomask) + hoff[l >> c0];
          sT[swz(l)] = tsrc[off];
          sP[swz(l)] = phi[off];
        }
      }
      __syncthreads();
    }
    if (active) {
      if (STAGED) {
#pragma unroll
        for (int x = 0; x < 16; ++x) v[x] = T::mk(to_c(lds[swz(roffl + xl[x])]));
      }
      for (int j = 0; j <= ngate; ++j) {
        if (j == lds_after) {
#pragma unroll
          for (int x = 0; x < 16; ++x)
            lds[swz(roffl + xl[x])] = from_c<S>(make_double2(v[x].x, v[x].y));
        }
        if (j < ngate) {
          grp_apply<C>(gcode[g0 + j], v, gmat[g0 + j]);
          const int z = gdead[g0 + j];
          if (z >= 0) {
#pragma unroll
            for (int x = 0; x < 16; ++x)
              if ((x >> z) & 1) v[x] = c2{0, 0};
          }
        }
      }
      if (!STAGED && store_dst) {
#pragma unroll
        for (int x = 0; x < 16; ++x) dst[gb + xg[x]] = from_c<S>(make_double2(v[x].x, v[x].y));
      }
      if (!STAGED) {
        if (nxt < ntiles) load_group((uint32_t)wdeposit((uint64_t)nxt, qmask) + roffg);
      }
      if (fast_stage && tside && nxt < ntiles) load_stage((uint32_t)wdeposit((uint64_t)nxt, qmask));
    }
    __syncthreads();
    // R += conj(T') phi^T over this tile: A[x][k] = conj(T'[x, r]), B[k][y] = phi[y, r]
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      if (4 * k >= kper) break;
      const int li = swz(rlane | rdep[k]);
      double2 tv = to_c(sT[li]);
      double2 pv = to_c(sP[li]);
      // Re R += Re T Re phi + Im T Im phi,  Im R += Re T Im phi - Im T Re phi
      acc_r = __builtin_amdgcn_mfma_f64_16x16x4f64(tv.x, pv.x, acc_r, 0, 0, 0);
      acc_r = __builtin_amdgcn_mfma_f64_16x16x4f64(tv.y, pv.y, acc_r, 0, 0, 0);
      acc_i = __builtin_amdgcn_mfma_f64_16x16x4f64(tv.x, pv.y, acc_i, 0, 0, 0);
      acc_i = __builtin_amdgcn_mfma_f64_16x16x4f64(-tv.y, pv.x, acc_i, 0, 0, 0);
    }
    __syncthreads();
    if (STAGED) {
      // phi's final values (all window gates) replace its R operand in LDS,
      // then both tiles go back to HBM in tile order (T' holds its final
      // values since the group phase)
      if (a.store && active && !tside) {
#pragma unroll
        for (int x = 0; x < 16; ++x) sP[swz(roffl + xl[x])] = from_c<S>(make_double2(v[x].x, v[x].y));
      }
      if (fast_stage && !tside && nxt < ntiles) load_stage((uint32_t)wdeposit((uint64_t)nxt, qmask));
    }
    if (STAGED && a.store) {
      __syncthreads();
      if (fast_stage) {
        if (store_dst) {
#pragma unroll
          for (int i = 0; i < 16; ++i) dst[base + ust[i] + sl0] = lds[swz(sl0 + 128 * i)];
        }
      } else {
        for (int l = threadIdx.x; l < (1 << t); l += blockDim.x) {
          const uint32_t off = base + ((uint32_t)l & lomask) + hoff[l >> c0];
          if (!first) tdst[off] = sT[swz(l)];
          phi[off] = sP[swz(l)];
        }
      }
      __syncthreads();
    }
  }
  // combine waves: D[i][j] at lane j + 16 (i % 4), item i / 4
  double* red = reinterpret_cast<double*>(wsm);   // 4 waves x 512
  {
    const int j = lane & 15, ib = lane >> 4;
#pragma unroll
    for (int it = 0; it < 4; ++it) {
      int i = it * 4 + ib;
      red[wave * 512 + (i * 16 + j) * 2] = acc_r[it];
      red[wave * 512 + (i * 16 + j) * 2 + 1] = acc_i[it];
    }
  }
  __syncthreads();
  double* pb = a.part + ((size_t)b * gridDim.x + blockIdx.x) * 512;
  for (int e = threadIdx.x; e < 512; e += blockDim.x)
    pb[e] = ((red[e] + red[512 + e]) + (red[1024 + e] + red[1536 + e]));
}

// ---- forward circuit pass ------------------------------------------------
// Applies the gates of up to kMaxStages stages (stage k: forward circuit
// positions fpos[gstart[k] .. gstart[k+1]), gate (layer L_b - 1 - f / N,
// site f % N), positions f >= L_b N skipped) to every state.  Stage 0 reads
// HBM, the last stage writes HBM, intermediate stages exchange through the
// LDS tile.
// Support: the circuit starts from |0..0>, and a gate only spreads the state
// over its own bits, so before the pass every amplitude at an index with a
// bit outside live_in is zero (not read: the memory there may be stale) and
// after it every amplitude outside live_out is.  Only tiles inside live_out
// are visited (tmask: the tile-index bits), and only amplitudes inside
// live_out are written, except in a full pass, which writes every amplitude.
// from_basis0: the input is |0..0> itself (psi is not read).
template <typename S>
__global__ __launch_bounds__(256) void fwd_pass_kernel(FwdArgs<S> a) {
  using C = typename StoreC<S>::C;
  using T = CT<C>;
  using c2 = typename T::c2;
  extern __shared__ char wsm[];
  __shared__ c2 gmat[kMaxFwdGates][16];
  __shared__ int gcode[kMaxFwdGates];
  const int b = a.list ? a.list[blockIdx.y] : blockIdx.y;
  const int n = a.n;
  if (a.skip && a.skip[b]) return;
  const int lb = a.layers[b];
  const int ng = a.gstart[a.nstage];
  // one gate entry per thread (kMaxFwdGates * 16 <= 4 * 256); positions past
  // this state's circuit get code -1 (no gate)
  for (int t = threadIdx.x; t < ng * 16; t += blockDim.x) {
    const int e = t & 15, j = t >> 4;
    const int f = a.fpos[j];
    if (f < lb * n) {
      int st = 0;
      while (a.gstart[st + 1] <= j) ++st;
      const int layer = lb - 1 - f / n, site = f % n;
      const size_t gi = ((size_t)b * a.lmax + layer) * n + site;
      // grp_apply applies the adjoint of what it is given: stage G^dagger
      const double2 gv = a.gates[gi * 16 + (e & 3) * 4 + (e >> 2)];
      gmat[j][e] = T::mk(make_double2(gv.x, -gv.y));
      if (e == 0) gcode[j] = gate_code(a.gs[st].mask, n, site, wsane(n, site, a.widths[gi]));
    } else if (e == 0) {
      gcode[j] = -1;
    }
  }
  __syncthreads();
  int total = 0;
  for (int j = 0; j < ng; ++j) total += a.fpos[j] < lb * n ? 1 : 0;
  const uint64_t all = (1ull << n) - 1ull;
  // a dense pass without gates leaves the state as it is
  if (total == 0 && !a.from_basis0 && a.live_in == all) return;
  const int t = a.t;
  const size_t len = (size_t)1 << n;
  S* lds = reinterpret_cast<S*>(wsm);
  S* psi = a.psi + (size_t)b * len;
  const long ntiles = 1l << __popcll(a.tmask);
  const int ngroups = 1 << (t - 4);
  const uint32_t dead_in = (uint32_t)(~a.live_in & all), dead_out = (uint32_t)(~a.live_out & all);
  // One group per thread (ngroups <= 256 = blockDim for tiles of <= 2^12
  // amplitudes).  Stage 0 always uses the same group map, so the next tile's
  // stage-0 loads are issued as soon as this tile's are consumed and stay in
  // flight while this tile's stages run.
  const bool has = (int)threadIdx.x < ngroups;
  const GroupMap& g0m = a.gs[0];
  const uint32_t roffg0 = has ? group_roffg(g0m, threadIdx.x) : 0u;
  c2 pre[16];
  auto load0 = [&](uint32_t bse) {
#pragma unroll
    for (int x = 0; x < 16; ++x) {
      const uint32_t ad = bse + roffg0 + xoffs(g0m.ubit, x);
      if (ad & dead_in)
        pre[x] = T::mk(make_double2(0.0, 0.0));
      else if (a.from_basis0)
        pre[x] = T::mk(make_double2(ad == 0u ? 1.0 : 0.0, 0.0));
      else
        pre[x] = T::mk(to_c(psi[ad]));
    }
  };
  if (has && (long)blockIdx.x < ntiles) load0((uint32_t)wdeposit((uint64_t)blockIdx.x, a.tmask));
  for (long tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
    const uint32_t base = (uint32_t)wdeposit((uint64_t)tile, a.tmask);
    for (int st = 0; st < a.nstage; ++st) {
      const GroupMap& gm = a.gs[st];
      const bool last = (st + 1 == a.nstage);
      if (has) {
        const int grp = threadIdx.x;
        const uint32_t roffg = st == 0 ? roffg0 : group_roffg(gm, grp);
        const int roffl = group_roffl(gm, grp);
        c2 v[16];
        if (st == 0) {
#pragma unroll
          for (int x = 0; x < 16; ++x) v[x] = pre[x];
          const long nxt = tile + gridDim.x;
          if (nxt < ntiles) load0((uint32_t)wdeposit((uint64_t)nxt, a.tmask));
        } else {
#pragma unroll
          for (int x = 0; x < 16; ++x) v[x] = T::mk(to_c(lds[swz(roffl + (int)xoffs(gm.ux, x))]));
        }
        for (int j = a.gstart[st]; j < a.gstart[st + 1]; ++j) grp_apply<C>(gcode[j], v, gmat[j]);
        if (last) {
#pragma unroll
          for (int x = 0; x < 16; ++x) {
            const uint32_t ad = base + roffg + xoffs(gm.ubit, x);
            if (a.full || !(ad & dead_out)) psi[ad] = from_c<S>(make_double2(v[x].x, v[x].y));
          }
        } else {
#pragma unroll
          for (int x = 0; x < 16; ++x) lds[swz(roffl + (int)xoffs(gm.ux, x))] = from_c<S>(make_double2(v[x].x, v[x].y));
        }
      }
      // stage exchange, and the next tile's stage 0 must not overwrite LDS early
      if (a.nstage > 1) __syncthreads();
    }
  }
}

// The forward pass on the matrix cores (tiles of 2^12 amplitudes; complex64
// states with N <= 28, complex128 with N <= 27): each stage's gates are fused
// into one 16 x 16 complex matrix M (column c = the stage's gates applied in
// order to the unit vector e_c of the stage's 4-bit group index), and each
// wave applies M to its groups, 16 at a time, as complex products on
// v_mfma_f32_16x16x4f32 or v_mfma_f64_16x16x4f64 (three real products per
// k-step, below).  Operand layouts (checked on gfx950): A[i][k] in lane
// i + 16 k and B[k][j] in lane j + 16 k for both; D[i][j] in lane
// j + 16 (i / 4), item i % 4 for f32 and in lane j + 16 (i % 4), item i / 4
// for f64.  Lane jl + 16 kq of a wave therefore holds, for column block cb,
// the amplitudes P(kq, s) (s < 4) of one group as B operands and receives the
// amplitudes P(kq, r) (r < 4) of the same group in item r, when the rows of M
// are ordered by MfmaT::row; P and the group's rest bits follow the stage's
// lane roles (MfmaMap, chosen on the host).  Loads, support (live_in /
// live_out) and the LDS exchange between stages are those of fwd_pass_kernel.
typedef float f4v __attribute__((ext_vector_type(4)));

// Per-type parts of the matrix-core pass.  A tile holds 256 groups, run by
// 8 waves of 2 column blocks (16 groups each): complex64 at 6 waves per SIMD
// (3 blocks per CU while their LDS fits; 4 waves of 4 column blocks ran 3%
// slower at 4 per SIMD), complex128 at 2 (its 64 KiB tile leaves room for
// one block per CU).
template <typename S> struct MfmaT;
template <> struct MfmaT<float2> {
  using R = float;
  using V4 = f4v;
  static constexpr int kWaves = 8;
  static constexpr int kShift = 3;   // log2 bytes per amplitude
  static QMX_DEV V4 mfma(R x, R y, V4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(x, y, c, 0, 0, 0); }
  static QMX_DEV float2 mk(double x, double y) { return make_float2((float)x, (float)y); }
  static QMX_DEV int row(int q, int r) { return 4 * q + r; }
};
template <> struct MfmaT<double2> {
  using R = double;
  using V4 = d4v;
  static constexpr int kWaves = 8;
  static constexpr int kShift = 4;
  static QMX_DEV V4 mfma(R x, R y, V4 c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(x, y, c, 0, 0, 0); }
  static QMX_DEV double2 mk(double x, double y) { return make_double2(x, y); }
  static QMX_DEV int row(int q, int r) { return q + 4 * r; }
};

// index parts of the matrix-core pass (positions from MfmaMap words, one
// per byte): the lane's (jl at j[0..3], kq at ks[0..1]), the wave's (w at
// h[NB..3]), and the uniform (cb at h[0..NB-1], s at ks[2..3]), NB = 2 with 4
// column blocks per wave and 1 with 2; the three are disjoint bit fields
QMX_DEV uint32_t pos8(uint32_t w, int i) { return (w >> (8 * i)) & 255u; }
QMX_DEV uint32_t lanepart(uint32_t j, uint32_t ks, int jl, int kq) {
  return ((uint32_t)(jl & 1) << pos8(j, 0)) | ((uint32_t)((jl >> 1) & 1) << pos8(j, 1)) |
         ((uint32_t)((jl >> 2) & 1) << pos8(j, 2)) | ((uint32_t)(jl >> 3) << pos8(j, 3)) |
         ((uint32_t)(kq & 1) << pos8(ks, 0)) | ((uint32_t)(kq >> 1) << pos8(ks, 1));
}
template <int NB> QMX_DEV uint32_t wavepart(uint32_t h, int w) {
  uint32_t r = 0;
#pragma unroll
  for (int i = NB; i < 4; ++i) r |= (uint32_t)((w >> (i - NB)) & 1) << pos8(h, i);
  return r;
}
template <int NB> QMX_DEV uint32_t unipart(uint32_t h, uint32_t ks, int cb, int s) {
  uint32_t r = ((uint32_t)(s & 1) << pos8(ks, 2)) | ((uint32_t)(s >> 1) << pos8(ks, 3));
#pragma unroll
  for (int i = 0; i < NB; ++i) r |= (uint32_t)((cb >> i) & 1) << pos8(h, i);
  return r;
}

template <typename S>
__attribute__((always_inline)) QMX_DEV void fwd_mfma_body(const FwdArgs<S>& a) {
  using M = MfmaT<S>;
  using R = typename M::R;
  using V4 = typename M::V4;
  constexpr int kCB = 16 / M::kWaves;       // column blocks of 16 groups per wave
  constexpr int kNB = kCB == 4 ? 2 : 1;     // their index bits
  extern __shared__ char wsm[];
  __shared__ int gcode[kMaxFwdGates];
  __shared__ uint32_t mmw[kMaxStages][3];  // per stage: jl, hl, ksl of MfmaMap
  const int b = a.list ? a.list[blockIdx.y] : blockIdx.y;
  const int n = a.n;
  if (a.skip && a.skip[b]) return;
  const int lb = a.layers[b];
  const int ng = a.gstart[a.nstage];
  const int t = a.t;   // kFwdTileBits: 256 groups of 16, 16 * kCB per wave
  S* lds = reinterpret_cast<S*>(wsm);
  // the stage matrices after the tile, in A-operand order: with P(q, s) the
  // amplitude index whose bits kx are q and bits sx are s (lane roles),
  // mst[st][s][row(q, r) + 16 kq] = M[P(q, r)][P(kq, s)], so that a wave's
  // A load is contiguous
  S* mst = lds + ((size_t)1 << t);
  // gates (as G^dagger, which grp_apply applies as G) in the tile area, which
  // stage 0 only writes after the matrices are built
  S(*gmat)[16] = reinterpret_cast<S(*)[16]>(wsm);
  for (int e2 = threadIdx.x; e2 < ng * 16; e2 += blockDim.x) {
    const int e = e2 & 15, j = e2 >> 4;
    const int f = a.fpos[j];
    if (f < lb * n) {
      int st = 0;
      while (a.gstart[st + 1] <= j) ++st;
      const int layer = lb - 1 - f / n, site = f % n;
      const size_t gi = ((size_t)b * a.lmax + layer) * n + site;
      const double2 gv = a.gates[gi * 16 + (e & 3) * 4 + (e >> 2)];
      gmat[j][e] = M::mk(gv.x, -gv.y);
      if (e == 0) gcode[j] = gate_code(a.gs[st].mask, n, site, wsane(n, site, a.widths[gi]));
    } else if (e == 0) {
      gcode[j] = -1;
    }
  }
  __syncthreads();
  int total = 0;
  for (int j = 0; j < ng; ++j) total += a.fpos[j] < lb * n ? 1 : 0;
  const uint64_t all = (1ull << n) - 1ull;
  if (total == 0 && !a.from_basis0 && a.live_in == all) return;
  if ((int)threadIdx.x < a.nstage * 16) {
    const int st = threadIdx.x >> 4, c = threadIdx.x & 15;
    const MfmaMap& mm = a.mm[st];
    S v[16];
#pragma unroll
    for (int x = 0; x < 16; ++x) v[x] = M::mk(x == c ? 1.0 : 0.0, 0.0);
    for (int j = a.gstart[st]; j < a.gstart[st + 1]; ++j) grp_apply<R>(gcode[j], v, gmat[j]);
    // amplitude index x <-> (q, s): q = its bits kx, s = its bits sx
    const uint32_t kx0 = pos8(mm.kxsx, 0), kx1 = pos8(mm.kxsx, 1), sx0 = pos8(mm.kxsx, 2), sx1 = pos8(mm.kxsx, 3);
    auto qof = [&](int x) { return (int)(((x >> kx0) & 1) | (((x >> kx1) & 1) << 1)); };
    auto sof = [&](int x) { return (int)(((x >> sx0) & 1) | (((x >> sx1) & 1) << 1)); };
    const int kc = qof(c), sc = sof(c);
#pragma unroll
    for (int x = 0; x < 16; ++x) mst[(st * 4 + sc) * 64 + 16 * kc + M::row(qof(x), sof(x))] = v[x];
    if (c == 0) {
      mmw[st][0] = mm.jl;
      mmw[st][1] = mm.hl;
      mmw[st][2] = mm.ksl;
    }
  }
  __syncthreads();
  const size_t len = (size_t)1 << n;
  // 32-bit byte offsets from a scalar base (below 2^32 for N <= 28 in
  // complex64 and N <= 27 in complex128)
  char* pbytes = reinterpret_cast<char*>(a.psi + (size_t)b * len);
  const long ntiles = 1l << __popcll(a.tmask);
  const uint32_t dead_in = (uint32_t)(~a.live_in & all), dead_out = (uint32_t)(~a.live_out & all);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int jl = lane & 15, kq = lane >> 4;
  // Every index below is an OR of disjoint bit fields, split into a per-lane
  // part (jl: the 4 low bits of the group index, kq: 2 bits of the amplitude
  // index) and a part that is uniform over the wave (wave, cb, s4 / r).  The
  // deposits and xoffs are linear over disjoint fields and the LDS swizzle is
  // linear over XOR, so an access costs one OR or XOR of the two parts.
  const MfmaMap& m0 = a.mm[0];
  const MfmaMap& mL = a.mm[a.nstage - 1];
  const uint32_t h0g = __builtin_amdgcn_readfirstlane(m0.hg), k0g = __builtin_amdgcn_readfirstlane(m0.ksg);
  const uint32_t hLg = __builtin_amdgcn_readfirstlane(mL.hg), kLg = __builtin_amdgcn_readfirstlane(mL.ksg);
  const uint32_t g0lane = lanepart(m0.jg, k0g, jl, kq);
  const uint32_t gLlane = lanepart(mL.jg, kLg, jl, kq);
  const uint32_t g0w = wavepart<kNB>(h0g, wave), gLw = wavepart<kNB>(hLg, wave);
  // B operands of stage 0 for one tile: [cb * 4 + s] = amplitude P(kq, s)
  S pre[4 * kCB];
  auto load0 = [&](uint32_t bse) {
#pragma unroll
    for (int cb = 0; cb < kCB; ++cb)
#pragma unroll
      for (int s4 = 0; s4 < 4; ++s4) {
        const uint32_t ad = bse + (g0w | unipart<kNB>(h0g, k0g, cb, s4)) + g0lane;
        S v;
        if (ad & dead_in)
          v = M::mk(0.0, 0.0);
        else if (a.from_basis0)
          v = M::mk(ad == 0u ? 1.0 : 0.0, 0.0);
        else
          v = *reinterpret_cast<const S*>(pbytes + (ad << M::kShift));
        pre[cb * 4 + s4] = v;
      }
  };

  for (long tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
    const uint32_t base = (uint32_t)wdeposit((uint64_t)tile, a.tmask);
    // stage 0's operands come from HBM at the tile's start: a prefetch of
    // the next tile's would cost the occupancy that hides the load latency
    // (measured with 4 column blocks per wave: 3 instead of 4 waves per
    // SIMD, slower)
    load0(base);
    for (int st = 0; st < a.nstage; ++st) {
      // lane roles of the stage (uniform: LDS broadcast, then scalar)
      const uint32_t mjl = __builtin_amdgcn_readfirstlane(mmw[st][0]);
      const uint32_t mhl = __builtin_amdgcn_readfirstlane(mmw[st][1]);
      const uint32_t mksl = __builtin_amdgcn_readfirstlane(mmw[st][2]);
      const bool last = (st + 1 == a.nstage);
      // tile-local offsets: per lane (jl, kq, swizzled once per stage) and
      // per (wave, cb, s or r)
      const int lsw = swz((int)lanepart(mjl, mksl, jl, kq));
      const uint32_t lw = wavepart<kNB>(mhl, wave);
      S xv[4 * kCB];
      if (st == 0) {
#pragma unroll
        for (int q = 0; q < 4 * kCB; ++q) xv[q] = pre[q];
      } else {
#pragma unroll
        for (int cb = 0; cb < kCB; ++cb)
#pragma unroll
          for (int s4 = 0; s4 < 4; ++s4) xv[cb * 4 + s4] = lds[lsw ^ swz((int)(lw | unipart<kNB>(mhl, mksl, cb, s4)))];
      }
      // A operands: M[jl][4 s + kq]
      S am[4];
#pragma unroll
      for (int s4 = 0; s4 < 4; ++s4) am[s4] = mst[(st * 4 + s4) * 64 + lane];
      // one column block at a time, each complex product as three real ones
      // (Gauss): k1 = Re M Re x, k2 = Im M Im x, k3 = (Re M + Im M)(Re x +
      // Im x); Re y = k1 - k2, Im y = k3 - k1 - k2.  The three accumulators
      // alternate, so consecutive products are independent.
      R asum[4];
#pragma unroll
      for (int s4 = 0; s4 < 4; ++s4) asum[s4] = am[s4].x + am[s4].y;
#pragma unroll
      for (int cb = 0; cb < kCB; ++cb) {
        V4 k1 = {0, 0, 0, 0}, k2 = {0, 0, 0, 0}, k3 = {0, 0, 0, 0};
#pragma unroll
        for (int s4 = 0; s4 < 4; ++s4) {
          const S x = xv[cb * 4 + s4];
          k1 = M::mfma(am[s4].x, x.x, k1);
          k2 = M::mfma(am[s4].y, x.y, k2);
          k3 = M::mfma(asum[s4], x.x + x.y, k3);
        }
        const V4 yr = k1 - k2, yi = k3 - k1 - k2;
        if (last) {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const uint32_t ad = base + (gLw | unipart<kNB>(hLg, kLg, cb, r)) + gLlane;
            if (a.full || !(ad & dead_out))
              *reinterpret_cast<S*>(pbytes + (ad << M::kShift)) = M::mk(yr[r], yi[r]);
          }
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            lds[lsw ^ swz((int)(lw | unipart<kNB>(mhl, mksl, cb, r)))] = M::mk(yr[r], yi[r]);
        }
      }
      // stage exchange, and the next tile's stage 0 must not overwrite LDS early
      if (a.nstage > 1) __syncthreads();
    }
  }
}

__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(6, 6))) void fwd_mfma_kernel(FwdArgs<float2> a) {
  fwd_mfma_body(a);
}
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void fwd_mfma64_kernel(FwdArgs<double2> a) {
  fwd_mfma_body(a);
}

// Replay the window on the 16-dim space of U (one block per state).  A chain
// of dependent small steps, bound by their latency: wave 0 takes each gate's
// environment and polar factor without a barrier inside, the other waves apply
// the next gate to the state side of Q at the same time (the two sides
// commute), and two barriers per gate are left.  13.2 us per window of one
// N=10 complex128 state (3.3 gates), against 48.3 us with a barrier around each
// of the gate's steps and the 16-lane pivoted polar.
// It runs beside the other half-batch's window pass, whose waves fill the
// SIMDs; its own waves take the highest issue priority so that this short,
// latency-bound chain is not slowed down by them.
__global__ __launch_bounds__(256) void window_finalize_kernel(WinFinArgs a) {
  __builtin_amdgcn_s_setprio(3);
  __shared__ double2 q[256];
  __shared__ double2 qn[256];
  __shared__ double2 gm[kMaxWindow][16];
  __shared__ int gw[kMaxWindow], gh[kMaxWindow], gl[kMaxWindow], gz[kMaxWindow];
  __shared__ double2 gnew[16];
  __shared__ double2 es[16];
  __shared__ double2 rm[16];
  __shared__ double part_sum[512];
  const int b = a.list ? a.list[blockIdx.x] : blockIdx.x;
  const int n = a.n;
  if (a.skip && a.skip[b]) return;
  const int kb = a.layers[b] * n;
  if (a.s0 >= kb) return;
  const int nc = min(a.s1, kb) - a.s0;
  // the window's gates, one entry per thread (nc * 16 <= 128), and the
  // positions of each gate's bits inside U (rank among U's bits); issued
  // before the partial sum so that both latencies overlap
  if ((int)threadIdx.x < nc * 16) {
    const int j = threadIdx.x >> 4, e = threadIdx.x & 15;
    int layer, site;
    step_gate(n, a.s0 + j, layer, site);
    const size_t gi = ((size_t)b * a.lmax + layer) * n + site;
    gm[j][e] = a.gates[gi * 16 + e];
    if (e == 0) {
      const int w = wsane(n, site, a.widths[gi]);
      gw[j] = w;
      const int hb = n - 1 - site;
      gh[j] = __popcll(a.umask & ((1ull << hb) - 1ull));
      gl[j] = w == 2 ? __popcll(a.umask & ((1ull << (hb - 1)) - 1ull)) : 0;
      gz[j] = dead_after(a.umask, n, kb, a.s0 + j);
    }
  }
  // R = sum of the block partials (slots 0, ps, 2 ps, ...) in a fixed order
  const double* pb = a.part + (size_t)b * a.nblk * 512;
  const int ps = a.pstride > 0 ? a.pstride : 1;
  const size_t st4 = (size_t)ps * 512;
  // (8 partials per step, all loads issued before the adds: the partials
  // come from L2 / HBM and the sum is latency-bound)
  for (int e = threadIdx.x; e < 512; e += blockDim.x) {
    double s = 0.0;
    int qq = 0;
#pragma unroll 2
    for (; qq + 7 * ps < a.nblk; qq += 8 * ps) {
      const double* q0 = pb + (size_t)qq * 512 + e;
      double v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = q0[u * st4];
      s += (((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7])));
    }
    for (; qq < a.nblk; qq += ps) s += pb[(size_t)qq * 512 + e];
    part_sum[e] = s;
  }
  __syncthreads();
  q[threadIdx.x] = make_double2(part_sum[2 * threadIdx.x], part_sum[2 * threadIdx.x + 1]);
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int j = 0; j < nc; ++j) {
    const int w = gw[j], hb = gh[j], lb = gl[j];
    const int d = w == 2 ? 4 : 2;
    const bool more = j + 1 < nc;
    if (wave == 0) {
      // E[o][i] = sum_z Q[(o,z)][(i,z)] over the U bits outside gate j, one
      // entry per lane (the four rows of 16 lanes alike)
      const int o = (lane >> 2) & 3, i = lane & 3;
      const int gmask = w == 2 ? (1 << hb) | (1 << lb) : 1 << hb;
      const int xo = w == 2 ? ((o >> 1) << hb) | ((o & 1) << lb) : (o & 1) << hb;
      const int yi = w == 2 ? ((i >> 1) << hb) | ((i & 1) << lb) : (i & 1) << hb;
      double2 acc = cz();
      if (o < d && i < d) {
        int z = 0;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          if (k >= 16 / d) break;
          acc = cadd(acc, q[(z | xo) * 16 + (z | yi)]);
          z = ((z | gmask) + 1) & ~gmask & 15;   // the next pattern of the other bits
        }
      }
      if (lane < 16) es[lane] = acc;
      const bool last = a.s0 + j == kb - 1 && a.overlap;
      const double nuc = update_gate_wave(d, a.omega_m1, gm[j], es, rm, gnew, lane, last);
      if (lane < 16) {
        int layer, site;
        step_gate(n, a.s0 + j, layer, site);
        const size_t gi = ((size_t)b * a.lmax + layer) * n + site;
        a.gates[gi * 16 + lane] = gnew[lane];
      }
      if (lane == 0 && last) a.overlap[(size_t)b * a.overlap_stride] = nuc;
    } else if (more) {
      // the other waves apply the next gate on the state side meanwhile:
      // Q[x][y] <- sum_{y'} Q[x][y'] conj(G_{j+1}[y'_g][y_g])
      const int w2 = gw[j + 1], hb2 = gh[j + 1], lb2 = gl[j + 1];
      const int m2 = w2 == 2 ? (1 << hb2) | (1 << lb2) : 1 << hb2;
      for (int e = threadIdx.x - 64; e < 256; e += 192) {
        const int x = e >> 4, y = e & 15;
        const int yg = w2 == 2 ? (((y >> hb2) & 1) << 1) | ((y >> lb2) & 1) : ((y >> hb2) & 1);
        double2 s = cz();
#pragma unroll
        for (int pg = 0; pg < 4; ++pg) {
          if (pg >= 2 && w2 != 2) break;
          const int yp = (y & ~m2) | (w2 == 2 ? ((pg >> 1) << hb2) | ((pg & 1) << lb2) : pg << hb2);
          s = cfmac(gm[j + 1][pg * 4 + yg], q[x * 16 + yp], s);
        }
        const int z2 = gz[j + 1];
        qn[e] = z2 >= 0 && ((y >> z2) & 1) ? cz() : s;
      }
    }
    if (!more) break;   // Q is not read after the window's last gate
    __syncthreads();
    // target side: Q[x][y] <- sum_{x'} G'[x'_g][x_g] Q[x'][y]
    {
      const int x = threadIdx.x >> 4, y = threadIdx.x & 15;
      const int gmask = w == 2 ? (1 << hb) | (1 << lb) : 1 << hb;
      const int xg = w == 2 ? (((x >> hb) & 1) << 1) | ((x >> lb) & 1) : ((x >> hb) & 1);
      double2 s = cz();
#pragma unroll
      for (int pg = 0; pg < 4; ++pg) {
        if (pg >= 2 && w != 2) break;
        const int xp = (x & ~gmask) | (w == 2 ? ((pg >> 1) << hb) | ((pg & 1) << lb) : pg << hb);
        s = cfma(gnew[pg * 4 + xg], qn[xp * 16 + y], s);
      }
      q[threadIdx.x] = s;
    }
    __syncthreads();
  }
}

// ---- all sweeps of a small state in one block -------------------------------
// T' and phi (up to 2^12 complex128 or 2^13 complex64 amplitudes) stay in LDS
// from the first sweep to the last.  The sweep is a serial chain of polar
// factors, so everything else is taken off that chain: in phase p of a sweep
// wave 0, the lead, turns the cross matrix of step p - 1 into its environment
// and new gate G'_{p-1}, while waves 1 to 4 prepare step p without it,
//   T'  <- G'_{p-2}^dagger T',   phi <- G_p^dagger phi,
//   R_p[x][y] = sum_r conj(T'[x, r]) phi[y, r]
// over the set V of the bits of steps p - 1 and p (three of them, the steps
// descend one site at a time), an 8 x 8 matrix.  G'_{p-1}, which R_p still
// lacks, acts inside V, so the next phase's environment is
//   E_p[o][i] = sum_z sum_x' G'_{p-1}[x'_g][x_g] R_p[x'][y],  x = (o, z), y = (i, z).
// Each worker owns a quarter of the indices r outside U = V and step p - 2's
// bits in a phase, so updates and products need no barrier between them, and
// one barrier per step is left.  Gate p + 2 is fetched two phases ahead.
// After the gate of site i of the first circuit layer is removed, the sites
// behind i are in |0>: phi is set to exactly zero where they are not.
// Bound by the issue of the lead's chain and of the worker that shares its SIMD
// up to 2^10 complex128 amplitudes (6.2k cycles a step at N = 6, environment
// 1.7k and polar factor 4.2k, and 7.0k at N = 10), by the workers' updates and
// products above (17k at N = 12).  The code of a step has to stay inside the 64
// KiB instruction cache that two CUs share: paths that are cold cost more to
// fetch than to run.  One state, 4 layers, 4 sweeps: 0.30 ms against 0.86 gate
// by gate at N = 5, 0.70 against 1.25 in windows at N = 10; 16 states of N = 12
// 1.8 ms against 3.1.
constexpr int kLdsWorkers = 4;
constexpr int kLdsThreads = 64 * (1 + kLdsWorkers);
constexpr int kLdsChunk = 32;   // gates per stage of the circuit rebuild (the partials' space)

// Place of amplitude l in LDS: its banks, 8 double2 or 16 float2 wide, take the
// XOR of l's 3-bit or 4-bit digits, so that the three neighbouring bits which
// the lanes of a product run over never share a bank.  (Linear over XOR.)
template <typename S> QMX_DEV int lds_at(int l) {
  if constexpr (sizeof(S) == 16) return l ^ (((l >> 3) ^ (l >> 6) ^ (l >> 9) ^ (l >> 12)) & 7);
  else return l ^ (((l >> 4) ^ (l >> 8) ^ (l >> 12)) & 15);
}
// x with a zero bit inserted at position p
QMX_DEV int zero_at(int x, int p) { return x + (x & ~((1 << p) - 1)); }
// the low bits of z at the set bits of mask (at most three of them)
QMX_DEV int spread3(int z, uint32_t mask) {
  const uint32_t f0 = mask & (~mask + 1u), r1 = mask ^ f0, f1 = r1 & (~r1 + 1u), f2 = r1 ^ f1;
  return (z & 1 ? f0 : 0) | (z & 2 ? f1 : 0) | (z & 4 ? f2 : 0);
}

// the four amplitudes at i0, i0 ^ sl, i0 ^ sh, i0 ^ sl ^ sh, and G^dagger of them
template <typename S, typename C2> QMX_DEV void quad_load(const S* s, int i0, int sl, int sh, C2 (&x)[4]) {
  using T = CT<typename StoreC<S>::C>;
  x[0] = T::mk(to_c(s[i0]));
  x[1] = T::mk(to_c(s[i0 ^ sl]));
  x[2] = T::mk(to_c(s[i0 ^ sh]));
  x[3] = T::mk(to_c(s[i0 ^ sl ^ sh]));
}
template <typename S, typename C2>
QMX_DEV void quad_adj(S* s, int i0, int sl, int sh, const C2 (&g)[16], const C2 (&x)[4]) {
  using T = CT<typename StoreC<S>::C>;
  C2 y[4];
#pragma unroll
  for (int o = 0; o < 4; ++o) {
    C2 acc = T::mulc(g[o], x[0]);
    acc = T::fmac(g[4 + o], x[1], acc);
    acc = T::fmac(g[8 + o], x[2], acc);
    y[o] = T::fmac(g[12 + o], x[3], acc);
  }
  s[i0] = from_c<S>(make_double2(y[0].x, y[0].y));
  s[i0 ^ sl] = from_c<S>(make_double2(y[1].x, y[1].y));
  s[i0 ^ sh] = from_c<S>(make_double2(y[2].x, y[2].y));
  s[i0 ^ sl ^ sh] = from_c<S>(make_double2(y[3].x, y[3].y));
}

// y = G^dagger x on amplitude quads (w = 2: bits h, h - 1) or pairs (w = 1: bit
// h) of an LDS state: this lane's patterns are base ^ su(u), u < nu (swizzled
// indices with the gate's bits zero; every index map here is linear over bit
// fields and the swizzle over XOR), if `on`.
template <typename S, typename F>
QMX_DEV void lds_gate(S* s, int w, int h, const double2* g, int nu, bool on, int base, F su) {
  using T = CT<typename StoreC<S>::C>;
  using c2 = typename T::c2;
  const int sh = lds_at<S>(1 << h);
  if (!on) return;
  if (w == 2) {
    const int sl = lds_at<S>(1 << (h - 1));
    c2 gc[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) gc[k] = T::mk(g[k]);
    auto load = [&](int i0, c2 (&x)[4]) { quad_load<S>(s, i0, sl, sh, x); };
    auto apply = [&](int i0, const c2 (&x)[4]) { quad_adj<S>(s, i0, sl, sh, gc, x); };
    // two patterns at a time: one's loads are in flight under the other's work
    int u = 0;
    for (; u + 1 < nu; u += 2) {
      const int ia = base ^ su(u), ib = base ^ su(u + 1);
      c2 xa[4], xb[4];
      load(ia, xa);
      load(ib, xb);
      apply(ia, xa);
      apply(ib, xb);
    }
    if (u < nu) {
      const int ia = base ^ su(u);
      c2 xa[4];
      load(ia, xa);
      apply(ia, xa);
    }
  } else {
    const c2 g00 = T::mk(g[0]), g01 = T::mk(g[1]), g10 = T::mk(g[4]), g11 = T::mk(g[5]);
    for (int u = 0; u < nu; ++u) {
      const int i0 = base ^ su(u), i1 = i0 ^ sh;
      const c2 x0 = T::mk(to_c(s[i0])), x1 = T::mk(to_c(s[i1]));
      const c2 y0 = T::fmac(g10, x1, T::mulc(g00, x0)), y1 = T::fmac(g11, x1, T::mulc(g01, x0));
      s[i0] = from_c<S>(make_double2(y0.x, y0.y));
      s[i1] = from_c<S>(make_double2(y1.x, y1.y));
    }
  }
}

template <typename S>
__global__ __launch_bounds__(kLdsThreads) void lds_sweep_kernel(LdsSweepArgs<S> a) {
  using T = CT<typename StoreC<S>::C>;
  using c2 = typename T::c2;
  extern __shared__ char wsm[];
  __shared__ double2 gold[4][16];            // old gates of steps p - 1 .. p + 1
  __shared__ double2 gnew[3][16];            // new gates of steps p - 3 .. p - 1
  __shared__ double2 es[16], rm[16];
  __shared__ int wold[4];                    // widths of gold (and of the new gates)
  __shared__ int wch[kLdsChunk];
  __shared__ uint32_t uset[16], vset[16];
  __shared__ double red[2 * (1 + kLdsWorkers)];
  const int b = blockIdx.x, n = a.n;
  const size_t len = (size_t)1 << n;
  S* sT = reinterpret_cast<S*>(wsm);
  S* sP = sT + len;
  double2* part = reinterpret_cast<double2*>(sP + len);   // 2 phases x kLdsWorkers x 64; gate stages
  int4* tab = reinterpret_cast<int4*>(part + 2 * kLdsWorkers * 64);   // n x 64
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lb = min(max(a.layers[b], 0), a.lmax), K = lb * n;
  double2* gates = a.gates + (size_t)b * a.lmax * n * 16;
  const int* widths = a.widths + (size_t)b * a.lmax * n;
  const double2* ref = a.psi_ref && a.fidelity ? a.psi_ref + (size_t)b * len : nullptr;
  const int mu = n < 4 ? n : 4, mv = n < 3 ? n : 3;   // bits of U and V
  // C|0..0> into sP, gates in forward order (their adjoints into the stage:
  // lds_gate conjugates back)
  auto rebuild = [&]() {
    for (int l = tid; l < (int)len; l += kLdsThreads) sP[lds_at<S>(l)] = from_c<S>(make_double2(l == 0 ? 1.0 : 0.0, 0.0));
    for (int f0 = 0; f0 < K; f0 += kLdsChunk) {
      const int nf = min(kLdsChunk, K - f0);
      __syncthreads();
      for (int e = tid; e < nf * 16; e += kLdsThreads) {
        const int f = f0 + (e >> 4);
        const size_t gi = (size_t)(lb - 1 - f / n) * n + f % n;
        part[e] = cconj(gates[gi * 16 + (e & 3) * 4 + ((e >> 2) & 3)]);
        if ((e & 15) == 0) wch[e >> 4] = wsane(n, f % n, widths[gi]);
      }
      __syncthreads();
      int h = n - 1 - f0 % n;
      for (int g = 0; g < nf; ++g) {
        // one wave per SIMD: wave 0 would be the fifth
        if (wave) {
          const int w = __builtin_amdgcn_readfirstlane(wch[g]);
          const int cnt = (int)(len >> w), t0 = tid - 64;
          auto at = [&](int t) { return lds_at<S>(w == 2 ? zero_at(zero_at(t, h - 1), h) : zero_at(t, h)); };
          lds_gate<S>(sP, w, h, part + g * 16, (cnt + kLdsThreads - 65) / (kLdsThreads - 64), t0 < cnt, at(t0),
                      [&](int u) { return at(u * (kLdsThreads - 64)); });
        }
        h = h ? h - 1 : n - 1;
        __syncthreads();
      }
    }
    __syncthreads();
  };
  // <psi_ref|C|0..0> of sP, on every thread (fixed order)
  auto overlap_ref = [&]() {
    double re = 0.0, im = 0.0;
    for (int l = tid; l < (int)len; l += kLdsThreads) {
      const double2 r = ref[l], p = to_c(sP[lds_at<S>(l)]);
      re = fma(r.x, p.x, fma(r.y, p.y, re));
      im = fma(r.x, p.y, fma(-r.y, p.x, im));
    }
    re = rows_sum(sum16(re));
    im = rows_sum(sum16(im));
    if (lane == 0) {
      red[2 * wave] = re;
      red[2 * wave + 1] = im;
    }
    __syncthreads();
    double2 t = cz();
#pragma unroll
    for (int w = 0; w <= kLdsWorkers; ++w) t = cadd(t, make_double2(red[2 * w], red[2 * w + 1]));
    __syncthreads();
    return t;
  };
  auto snapshot = [&](int done) {
    if (!a.snaps || done < a.snap_first || done > a.snap_first + 1) return;
    double2* dst = a.snaps + (size_t)(done - a.snap_first) * a.snap_stride + (size_t)b * a.lmax * n * 16;
    for (int e = tid; e < a.lmax * n * 16; e += kLdsThreads) dst[e] = gates[e];
  };
  // Step p acts on bit r = p % n (site n - 1 - r) and, with two qubits, on
  // bit r - 1.  By residue: U, the worst-case bits of steps p, p - 1 and p - 2,
  // and V, those of p and p - 1 (before the sweep's start any bits will do),
  // padded with the lowest free ones (V inside U).
  if (tid < n) {
    uint32_t u = 0, v = 0;
    for (int k = 0; k < 3; ++k) {
      const int r = (tid + 2 * n - k) % n;
      u |= 1u << r | (r > 0 ? 1u << (r - 1) : 0u);
      if (k == 1) v = u;
    }
    for (int bit = 0; bit < n && __popc(u) < mu; ++bit) u |= 1u << bit;
    for (int bit = 0; bit < n && __popc(v) < mv; ++bit) v |= u & (1u << bit);
    uset[tid] = u;
    vset[tid] = v;
  }
  auto prev = [&](int r) { return r == 0 ? n - 1 : r - 1; };
  auto rank_in = [](uint32_t u, int bit) { return __popc(u & ((1u << bit) - 1u)); };
  auto gate_at = [&](int r, int layer) { return (size_t)layer * n + (n - 1 - r); };
  // A worker's indices r outside U: r0 .. r0 + G - 1 (G a power of two, r0 a
  // multiple of it).  U's bits in rising order; deposit of r outside U.
  const int rest = 1 << (n - mu), G = rest >= kLdsWorkers ? rest / kLdsWorkers : 1, glog = __ffs(G) - 1;
  auto deposit = [&](uint32_t u, int r) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if (k < mu) r = zero_at(r, u ? __ffs(u) - 1 : 31);
      u &= u - 1u;
    }
    return r;
  };
  // The lanes' places per residue, which would take a third of a step to form
  // again each time: of the first pattern of T's and phi's gate (of two qubits),
  // and of T' and phi in the products below
  __syncthreads();
  for (int e = tid; e < 64 * n; e += kLdsThreads) {
    const int r = e >> 6, ln = e & 63, ht = prev(prev(r));
    const uint32_t u = uset[r], v = vset[r], far = u & ~v;
    const int at = deposit(u, ln & (G - 1)), q = ln >> glog;
    const uint32_t gt = ht ? 3u << (ht - 1) : 1u, gc = r ? 3u << (r - 1) : 1u;
    const int kk = ln & 7, x0 = 2 * ((ln >> 3) & 3), y0 = 4 * (ln >> 5);
    const int base = deposit(u, kk & (G - 1)) | ((kk >> glog) & 1 ? (int)far : 0);
    tab[e] = make_int4(lds_at<S>(at | spread3(q, u & ~gt)), lds_at<S>(at | spread3(q, u & ~gc)),
                       lds_at<S>(base | spread3(x0, v)), lds_at<S>(base | spread3(y0, v)));
  }
  snapshot(0);
  const bool use_goal = a.goal && ref;
  int done = 0;
  double2 fid = cz();
  int s = 0;
  for (; s < a.nsweeps; ++s) {
    rebuild();
    if (ref) {
      fid = overlap_ref();
      if (tid == 0) a.fidelity[(size_t)b * (a.nsweeps + 1) + s] = fid;
    }
    if (use_goal && sqrt(fid.x * fid.x + fid.y * fid.y) >= a.goal[b]) break;
    ++done;
    const S* tsrc = a.target + (size_t)b * len;
    for (int l = tid; l < (int)len; l += kLdsThreads) sT[lds_at<S>(l)] = tsrc[l];
    // old gates: step 0 now, step p + 1 written in phase p, where step p + 2 is
    // fetched into a worker's registers
    if (tid < 16 && K > 0) {
      gold[0][tid] = gates[gate_at(0, 0) * 16 + tid];
      if (tid == 0) wold[0] = wsane(n, n - 1, widths[gate_at(0, 0)]);
    }
    const bool fetcher = wave == 1 && lane < 16;
    double2 gnext = cz();
    int wnext = 0;
    int fr = 1, fl = 0;   // residue and layer of the step to fetch next (n >= 2)
    if (fetcher && K > 1) {
      gnext = gates[gate_at(fr, fl) * 16 + lane];
      wnext = wsane(n, n - 1 - fr, widths[gate_at(fr, fl)]);
    }
    int rp = 0, layer_prev = 0;   // p % n; the layer of step p - 1
    __syncthreads();
    for (int p = 0; p <= K && K > 0; ++p) {
      if (wave == 0) {
        if (p > 0) {
          // ---- lead: the environment and the new gate of step k = p - 1
          __builtin_amdgcn_s_setprio(3);
          const int k = p - 1, hbit = prev(rp), kp = k - 1, hpbit = prev(hbit);
          const int lv = vset[hbit], lw = wold[k & 3], lwp = wold[kp & 3];   // (one wait for the three)
          const uint32_t v = __builtin_amdgcn_readfirstlane(lv);
          const int w = __builtin_amdgcn_readfirstlane(lw), d = w == 2 ? 4 : 2;
          const int hb = rank_in(v, hbit), gl = w == 2 ? hb - 1 : hb;   // the gate's lowest bit in V
          // the pending gate of step k - 1
          const int wp = kp >= 0 ? __builtin_amdgcn_readfirstlane(lwp) : 0, np = 1 << wp;
          const int pl = rank_in(v, hpbit) - (wp == 2 ? 1 : 0);
          const int pmask = (np - 1) << pl;
          const double2* gp = gnew[(kp + 3) % 3];
          const int o = (lane >> 2) & 3, i = lane & 3, row = lane >> 4;
          const uint32_t fm = ((1u << mv) - 1u) & ~((uint32_t)(d - 1) << gl);   // V's bits beside the gate's
          const int nt = ((1 << mv) / d) << wp;
          // terms (z, x'_g), one in four per row of lanes: two each, four for a
          // one-qubit gate after one of two qubits
          double2 acc = cz();
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            if (u == 2 && nt <= 8) break;
            const int t = row + 4 * u;
            const int pg = t & (np - 1), z = spread3(t >> wp, fm);
            const int x = z | (o & (d - 1)) << gl, y = z | (i & (d - 1)) << gl;
            const int at = (wp ? (x & ~pmask) | pg << pl : x) * 8 + y;
            const double2* q = part + (k & 1) * kLdsWorkers * 64 + at;
            const double2 c = gp[pg * 4 + ((x >> pl) & (np - 1))];
            const double2 e = cadd(cadd(q[0], q[64]), cadd(q[128], q[192]));
            const double2 f = wp ? cmul(c, e) : e;
            acc = t < nt ? cadd(acc, f) : acc;
          }
          acc = make_double2(rows_sum(acc.x), rows_sum(acc.y));
          if (lane < 16) es[lane] = o < d && i < d ? acc : cz();
          const bool last = k == K - 1 && a.overlap;
          const double nuc = update_gate_wave(d, a.omega_m1, gold[k & 3], es, rm, gnew[k % 3], lane, last);
          if (lane < 16) gates[gate_at(hbit, layer_prev) * 16 + lane] = gnew[k % 3][lane];
          if (lane == 0 && last) a.overlap[(size_t)b * a.nsweeps + s] = nuc;
          __builtin_amdgcn_s_setprio(0);
        }
      } else if (p < K) {
        // ---- workers: step p without G'_{p-1}
        const int wid = wave - 1;
        if (fetcher && p + 1 < K) {
          gold[(p + 1) & 3][lane] = gnext;
          if (lane == 0) wold[(p + 1) & 3] = wnext;
          if (++fr == n) {
            fr = 0;
            ++fl;
          }
          if (p + 2 < K) {
            gnext = gates[gate_at(fr, fl) * 16 + lane];
            wnext = wsane(n, n - 1 - fr, widths[gate_at(fr, fl)]);
          }
        }
        const uint32_t u = __builtin_amdgcn_readfirstlane(uset[rp]), v = __builtin_amdgcn_readfirstlane(vset[rp]);
        const int4 places = tab[rp * 64 + lane];
        auto roff = [&](int r) { return deposit(u, r); };
        const int r0 = wid * G, nr = r0 < rest ? G : 0;
        const int sr0 = lds_at<S>(roff(r0));
        auto update = [&](S* s, int w, int h, int first, const double2* g) {
          const uint32_t om = u & ~(w == 2 ? 3u << (h - 1) : 1u << h);   // U's bits beside the gate's
          const int cnt = nr << (mu - w);
          auto at = [&](int t) { return lds_at<S>(roff(t & (G - 1)) | spread3(t >> glog, om)); };
          lds_gate<S>(s, w, h, g, (cnt + 63) >> 6, lane < cnt, sr0 ^ (w == 2 ? first : at(lane)),
                      [&](int k) { return at(64 * k); });
        };
        const int kt = p - 2, h = rp;
        auto width_of = [&](int k) { return __builtin_amdgcn_readfirstlane(wold[k & 3]); };
        const int wt = kt >= 0 ? width_of(kt) : 0, wc = width_of(p), ht = prev(prev(rp));
        if (wt == 2 && wc == 2 && nr << (mu - 2) <= 64) {
          // one pattern a lane: the loads of both sides are in flight together
          const int lt = lds_at<S>(1 << (ht - 1)), mt = lds_at<S>(1 << ht), lc = lds_at<S>(1 << (h - 1)),
                    mc = lds_at<S>(1 << h);
          if (lane < nr << (mu - 2)) {
            const int it = sr0 ^ places.x, ic = sr0 ^ places.y;
            c2 xt[4], xc[4], g[16];
            quad_load<S>(sT, it, lt, mt, xt);
            quad_load<S>(sP, ic, lc, mc, xc);
#pragma unroll
            for (int k = 0; k < 16; ++k) g[k] = T::mk(gnew[kt % 3][k]);
            quad_adj<S>(sT, it, lt, mt, g, xt);
#pragma unroll
            for (int k = 0; k < 16; ++k) g[k] = T::mk(gold[p & 3][k]);
            quad_adj<S>(sP, ic, lc, mc, g, xc);
          }
        } else {
          if (wt) update(sT, wt, ht, places.x, gnew[kt % 3]);
          update(sP, wc, h, places.y, gold[p & 3]);
        }
        __builtin_amdgcn_wave_barrier();
        if (p >= K - n && h > 0) {
          // the sites behind step p's are in |0> once this gate of the first
          // circuit layer is gone
          const uint32_t om = u & ~(1u << (h - 1));
          for (int t = lane; t < nr << (mu - 1); t += 64)
            sP[sr0 ^ lds_at<S>(roff(t & (G - 1)) | spread3(t >> glog, om) | 1 << (h - 1))] = from_c<S>(cz());
          __builtin_amdgcn_wave_barrier();
        }
        // R over V by vector FMA (the 4 x 4 x 4 matrix instruction measured 80
        // cycles here, four times the vector unit's for the same products): lane
        // bits 0-2 take eight indices (r and U's bit outside V), bits 3-4 two x
        // of T' and bit 5 four y of phi
        const uint32_t far = u & ~v;                   // one bit, none for n < 4
        const int cnt = far ? 2 * nr : nr, kk = lane & 7, x0 = 2 * ((lane >> 3) & 3), y0 = 4 * (lane >> 5);
        auto at = [&](int t) { return lds_at<S>(roff(t & (G - 1)) | ((t >> glog) & 1 ? (int)far : 0)); };
        // (lanes beyond V read valid places too: spread3 drops the bits that V lacks)
        const int bt = sr0 ^ places.z, bp = sr0 ^ places.w;
        const int v0 = lds_at<S>(spread3(1, v)), v1 = lds_at<S>(spread3(2, v));
        double2 acc[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] = cz();
#pragma unroll 2
        for (int k0 = 0; k0 < cnt; k0 += 8) {
          const int off = at(k0);
          double2 tv[2], pv[4];
#pragma unroll
          for (int j = 0; j < 2; ++j) tv[j] = to_c(sT[bt ^ off ^ (j ? v0 : 0)]);
#pragma unroll
          for (int j = 0; j < 4; ++j) pv[j] = to_c(sP[bp ^ off ^ (j & 1 ? v0 : 0) ^ (j & 2 ? v1 : 0)]);
#pragma unroll
          for (int e = 0; e < 8; ++e) acc[e] = cfmac(tv[e >> 2], pv[e & 3], acc[e]);
        }
        if (kk >= cnt)
#pragma unroll
          for (int e = 0; e < 8; ++e) acc[e] = cz();
        // sum over the eight lanes; each keeps one entry: (x0 + kk % 2, y0 + kk / 2)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const double2 keep = kk & 1 ? acc[4 + e] : acc[e], send = kk & 1 ? acc[e] : acc[4 + e];
          acc[e] = make_double2(keep.x + dpp<0xB1>(send.x), keep.y + dpp<0xB1>(send.y));
        }
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const double2 keep = kk & 2 ? acc[2 * e + 1] : acc[2 * e], send = kk & 2 ? acc[2 * e] : acc[2 * e + 1];
          acc[e] = make_double2(keep.x + dpp<0x4E>(send.x), keep.y + dpp<0x4E>(send.y));
        }
        {
          // lanes i and i ^ 4 through the mirrored halves: their low bits flip, so
          // the quad is turned back first
          const double2 keep = kk & 4 ? acc[1] : acc[0], send = kk & 4 ? acc[0] : acc[1];
          acc[0] = make_double2(keep.x + dpp<0x141>(dpp<0x1B>(send.x)), keep.y + dpp<0x141>(dpp<0x1B>(send.y)));
        }
        part[((p & 1) * kLdsWorkers + wid) * 64 + (x0 + (kk & 1)) * 8 + y0 + ((kk >> 1) & 1) + 2 * (kk >> 2)] = acc[0];
      }
      __syncthreads();
      if (p > 0 && rp == 0) ++layer_prev;   // step p starts a layer
      rp = rp + 1 == n ? 0 : rp + 1;
    }
    snapshot(s + 1);
  }
  if (s == a.nsweeps) {
    rebuild();
    if (ref) fid = overlap_ref();
  }
  if (ref && tid == 0) a.fidelity[(size_t)b * (a.nsweeps + 1) + a.nsweeps] = fid;
  if (a.sweeps_done && tid == 0) a.sweeps_done[b] = a.goal ? (use_goal ? done : 0) : a.nsweeps;
  if (a.circuit_out)
    for (int l = tid; l < (int)len; l += kLdsThreads) a.circuit_out[(size_t)b * len + l] = sP[lds_at<S>(l)];
}

template <typename S>
hipError_t launch_lds_sweep(const LdsSweepArgs<S>& a, int batch, hipStream_t st) {
  constexpr size_t parts = 2 * kLdsWorkers * 64 * sizeof(double2);
  static_assert(parts >= kLdsChunk * 16 * sizeof(double2), "a stage of gates fits the partials' space");
  // the limit is set to the largest need, so that launches from several host
  // threads never lower it under each other
  constexpr int nmax = lds_sweep_qubits(sizeof(S));
  const size_t most = (2 * sizeof(S) << nmax) + parts + nmax * 64 * sizeof(int4);
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(lds_sweep_kernel<S>),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)most);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(lds_sweep_kernel<S>, dim3(batch), dim3(kLdsThreads),
                     (2 * sizeof(S) << a.n) + parts + a.n * 64 * sizeof(int4), st, a);
  return hipGetLastError();
}
template hipError_t launch_lds_sweep<float2>(const LdsSweepArgs<float2>&, int, hipStream_t);
template hipError_t launch_lds_sweep<double2>(const LdsSweepArgs<double2>&, int, hipStream_t);

template <typename S>
void launch_fwd_pass(const FwdArgs<S>& a, int nblk, int batch, hipStream_t st) {
  size_t shm = sizeof(S) << a.t;
  // the host fills a.mm under the same condition (fwd_mfma_applies)
  if (fwd_mfma_applies(a.mfma, a.t, a.n, sizeof(S))) {
    // the tile, then one 16 x 16 complex matrix per stage
    shm += (size_t)a.nstage * 256 * sizeof(S);
    if constexpr (sizeof(S) == 8) {
      hipLaunchKernelGGL(fwd_mfma_kernel, dim3(nblk, batch), dim3(512), shm, st, a);
      return;
    } else {
      // above the default 64 KiB of dynamic LDS; the limit is always set to
      // the kernel's largest need (tile + kMaxStages matrices), so that
      // launches from several host threads never lower it under each other
      const size_t most = (sizeof(S) << kFwdTileBits) + (size_t)kMaxStages * 256 * sizeof(S);
      if (hipFuncSetAttribute(reinterpret_cast<const void*>(fwd_mfma64_kernel),
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)most) == hipSuccess) {
        hipLaunchKernelGGL(fwd_mfma64_kernel, dim3(nblk, batch), dim3(512), shm, st, a);
        return;
      }
      shm = sizeof(S) << a.t;
    }
  }
  hipLaunchKernelGGL(fwd_pass_kernel<S>, dim3(nblk, batch), dim3(256), shm, st, a);
}
template void launch_fwd_pass<float2>(const FwdArgs<float2>&, int, int, hipStream_t);
template void launch_fwd_pass<double2>(const FwdArgs<double2>&, int, int, hipStream_t);

template <typename S>
void launch_window_pass(const WinPassArgs<S>& a, int nblk, int batch, hipStream_t st) {
  int t = a.t;
  size_t shm = 2 * (sizeof(S) << t);
  const size_t red = 4 * 512 * sizeof(double);
  if (shm < red) shm = red;
  constexpr int wpe = sizeof(S) == 8 ? 4 : 2;
  if (a.staged)
    hipLaunchKernelGGL((window_pass_kernel<S, wpe, true>), dim3(nblk, batch), dim3(256), shm, st, a);
  else
    hipLaunchKernelGGL((window_pass_kernel<S, wpe, false>), dim3(nblk, batch), dim3(256), shm, st, a);
}
template void launch_window_pass<float2>(const WinPassArgs<float2>&, int, int, hipStream_t);
template void launch_window_pass<double2>(const WinPassArgs<double2>&, int, int, hipStream_t);

void launch_window_finalize(const WinFinArgs& a, int batch, hipStream_t st) {
  hipLaunchKernelGGL(window_finalize_kernel, dim3(batch), dim3(256), 0, st, a);
}

// block k of state b sums partial slots [k group, min((k + 1) group, nblk))
// into slot k group (each thread owns elements e, e + 256 of every slot)
__global__ __launch_bounds__(256) void window_reduce_kernel(double* part, int nblk, int group, const int* list) {
  double* pb = part + (size_t)(list ? list[blockIdx.y] : blockIdx.y) * nblk * 512;
  const int q0 = blockIdx.x * group, q1 = min(q0 + group, nblk);
  for (int e = threadIdx.x; e < 512; e += blockDim.x) {
    double s = 0.0;
    int q = q0;
    for (; q + 3 < q1; q += 4)
      s += ((pb[(size_t)q * 512 + e] + pb[(size_t)(q + 1) * 512 + e]) +
            (pb[(size_t)(q + 2) * 512 + e] + pb[(size_t)(q + 3) * 512 + e]));
    for (; q < q1; ++q) s += pb[(size_t)q * 512 + e];
    pb[(size_t)q0 * 512 + e] = s;
  }
}

void launch_window_reduce(double* part, int nblk, int group, int batch, const int* list, hipStream_t st) {
  hipLaunchKernelGGL(window_reduce_kernel, dim3((nblk + group - 1) / group, batch), dim3(256), 0, st, part,
                     nblk, group, list);
}

}  // namespace qmx
