// Replica-batch kernels: one force evaluation of many independent periodic
// boxes of one force field (LJ + erfc Coulomb pairs with RBL or a full pair
// set, sampled or Ewald k-space), every stage one launch over a range of
// replicas:
//
//   kb_bin       wrap, cell of every atom, per-cell counts (atomics)
//   kb_scan      per-cell offsets of atoms and charged atoms (a workgroup per
//                replica)
//   kb_scatter   cell buckets in arrival order
//   kb_cellsort  per cell: charged atoms first, then by caller index (a
//                deterministic order); sorted positions, types, ids, and the
//                charged atoms' compact copy
//   kb_eval      three kinds of workgroups in one launch: the k-space of a
//                replica (S(k), energy, virial, force of its charged atoms),
//                the LJ pairs of a brick (persistent over the (replica, brick)
//                work list, the brick's neighbourhood staged in LDS) and the
//                Coulomb pairs of a run of charged atoms; FP64 energy, virial
//                and force sum per replica
//   kb_finish    the three force rows added in caller order, mean pair force
//                removed (RBL)
//
// Cells are rebuilt every evaluation (no skin, no stored lists), so an
// evaluation has no host-side decisions and the whole sequence replays as
// one captured graph.  A dimension of fewer than three cells is staged once
// and pairs take the minimum image; elsewhere stage coordinates are shifted
// across the box edges.
#include <hip/hip_runtime.h>

#include "batch.hpp"
#include "device.hpp"

namespace rbmdx {
namespace {

__device__ __forceinline__ float wrap_coord(float x, float lo, float L, float invL,
                                            float& s) {
  s = (x - lo) * invL;
  const float f = floorf(s);
  s -= f;
  return f != 0.f ? x - f * L : x;
}

__device__ __forceinline__ int batch_cell(const RepInfo& p, float x, float y, float z,
                                          float w[3]) {
  float s[3];
  w[0] = wrap_coord(x, p.box.lo[0], p.box.L[0], p.box.invL[0], s[0]);
  w[1] = wrap_coord(y, p.box.lo[1], p.box.L[1], p.box.invL[1], s[1]);
  w[2] = wrap_coord(z, p.box.lo[2], p.box.L[2], p.box.invL[2], s[2]);
  int c[3];
#pragma unroll
  for (int d = 0; d < 3; ++d)
    c[d] = max(0, min((int)(s[d] * (float)p.nc[d]), p.nc[d] - 1));
  return p.c0 + (c[2] * p.nc[1] + c[1]) * p.nc[0] + c[0];
}

__global__ __launch_bounds__(256) void kb_bin(BatchDev d, BatchRange rg) {
  const int i = rg.a0 + blockIdx.x * blockDim.x + threadIdx.x;
  // per-replica sums are accumulated with atomics by later stages
  for (int q = blockIdx.x * blockDim.x + threadIdx.x; q < (rg.r1 - rg.r0) * kBatchAcc;
       q += gridDim.x * blockDim.x)
    d.racc[(size_t)rg.r0 * kBatchAcc + q] = 0.0;
  for (int q = blockIdx.x * blockDim.x + threadIdx.x; q < (rg.r1 - rg.r0) * kBatchKAcc;
       q += gridDim.x * blockDim.x)
    d.kacc[(size_t)rg.r0 * kBatchKAcc + q] = 0.0;
  if (i >= rg.a1) return;
  const RepInfo& p = d.rep[d.rep_of[i]];
  float w[3];
  const int cell = batch_cell(p, d.px[i], d.py[i], d.pz[i], w);
  d.cell_of[i] = cell;
  // one atomic for both counts: atoms in the low half, charged in the high
  const unsigned long long one = d.charge[i] != 0.f ? (1ull << 32) + 1ull : 1ull;
  d.slot[i] = (int)(unsigned)atomicAdd(&d.cnt[cell], one);
}

// Exclusive offsets of one replica's cells, a workgroup each (atoms from a0,
// charged atoms from q0: both are known per replica, so no scan crosses
// replicas); the counters are cleared for the next evaluation.  One workgroup
// over all cells took 240 us for the 49,000 cells of 256 replicas, this 5.
__global__ __launch_bounds__(256) void kb_scan(BatchDev d, BatchRange rg) {
  __shared__ int sm[33];
  const RepInfo& p = d.rep[rg.r0 + blockIdx.x];
  const int c0 = p.c0, nc = p.nc[0] * p.nc[1] * p.nc[2];
  int ra = p.a0, rq = p.q0;
  for (int base = 0; base < nc; base += blockDim.x) {
    const int c = base + (int)threadIdx.x;
    const unsigned long long v = c < nc ? d.cnt[c0 + c] : 0ull;
    int ta, tq;
    const int ea = block_excl_scan((int)(unsigned)v, ta, sm);
    const int eq = block_excl_scan((int)(v >> 32), tq, sm);
    if (c < nc) {
      d.start[c0 + c] = ra + ea;
      d.qstart[c0 + c] = rq + eq;
      d.cnt[c0 + c] = 0ull;
    }
    ra += ta;
    rq += tq;
  }
  // (the next replica's first cell: the same values its own workgroup writes)
  if (threadIdx.x == 0) {
    d.start[c0 + nc] = ra;
    d.qstart[c0 + nc] = rq;
  }
}

// Sort key of a caller atom inside its cell: charged first, then by index.
constexpr int kNeutralKey = 1 << 30;
__global__ __launch_bounds__(256) void kb_scatter(BatchDev d, BatchRange rg) {
  const int i = rg.a0 + blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= rg.a1) return;
  d.tmp[d.start[d.cell_of[i]] + d.slot[i]] = (d.charge[i] != 0.f ? 0 : kNeutralKey) + i;
}

// One thread per atom: its rank among the keys of its cell (the lanes of a
// wave read the same few buckets), then its rows of the sorted arrays and,
// for a charged atom, of the compact charged copy.
__global__ __launch_bounds__(256) void kb_cellsort(BatchDev d, BatchRange rg) {
  const int b = rg.a0 + blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= rg.a1) return;
  const int kv = d.tmp[b], i = kv & (kNeutralKey - 1);
  const int c = d.cell_of[i];
  const int s0 = d.start[c], s1 = d.start[c + 1];
  int r = 0;
  for (int q = s0; q < s1; ++q) r += d.tmp[q] < kv ? 1 : 0;
  const int k = s0 + r;
  const RepInfo& p = d.rep[d.rep_of[i]];
  float w[3];
  batch_cell(p, d.px[i], d.py[i], d.pz[i], w);
  const int g = d.gid[i];
  // .w: the byte offset of the type's entry in one row of the LJ table
  d.xs[k] = make_float4(w[0], w[1], w[2], __int_as_float(d.type[i] << 4));
  d.gid_s[k] = g;
  d.perm[k] = i;
  if (kv < kNeutralKey) {
    const int q = d.qstart[c] + r;
    d.xqc[q] = make_float4(w[0], w[1], w[2], d.charge[i]);
    d.qi[q] = make_int4(g, d.qpos[i], c, i);
  }
}

// Slot tables of one brick's neighbourhood (the brick widened by one cell;
// a dimension of fewer than three cells taken whole).
struct BrickNb {
  int o[3], w[3];      // brick cells [o, o + w)
  int rs[3], rn[3];    // neighbourhood start (may be -1) and count
  int full[3];
  int nslots;
  int mi;
};

// With three cells or more, every owner's window of three cells holds each
// cell once, shifted by +-L across the edges.  For a pair two cells apart of
// a three-cell dimension the shifted distance may exceed L/2, but then its
// other image is at least one cell away, beyond the cutoff, as is this one:
// every pair inside the cutoff is met exactly once, at its minimum image.
__device__ __forceinline__ BrickNb batch_brick(const RepInfo& p, int b) {
  BrickNb h;
  const int bc[3] = {b % p.nb[0], (b / p.nb[0]) % p.nb[1], b / (p.nb[0] * p.nb[1])};
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    h.o[d] = bc[d] * p.bw;
    h.w[d] = min(p.bw, p.nc[d] - h.o[d]);
    h.full[d] = p.nc[d] < 3;
    h.rs[d] = h.full[d] ? 0 : h.o[d] - 1;
    h.rn[d] = h.full[d] ? p.nc[d] : h.w[d] + 2;
  }
  h.nslots = h.rn[0] * h.rn[1] * h.rn[2];
  h.mi = h.full[0] | h.full[1] | h.full[2];
  return h;
}

// The CVFF special-bond row of caller atom i.
template <bool GEN>
__device__ __forceinline__ SpecRow batch_spec_row(const BatchDev& d, int ms, int i) {
  SpecRow r;
  if (GEN && ms > 0) {
    const int4 c = d.spn[i];
    r.n12 = c.x;
    r.n13 = c.y;
    r.n14 = c.z;
    r.ids = d.spid + (size_t)i * ms;
  }
  return r;
}

// LDS of kb_eval's workgroups: one buffer for the three roles.
//   LJ: the stage (position and LJ-row offset), 64 entries of padding that
//       the unrolled tests may read past a row, then the per-lane lists of
//       accepted stage positions [LjList][block] and, with GEN, the staged
//       global ids;
//   Coulomb: per-lane lists of accepted charged atoms [kQList][block];
//   k-space: the atom tile, per-k coefficients and rho, and partial sums.
constexpr int kEvalBlock = 256;
// Accepted stage positions per lane between two evaluations of the list: the
// force pass, whose registers allow 4 waves per SIMD, takes as few as let a
// fourth workgroup into a CU's LDS; with energies or CVFF registers allow 3.
template <bool LEAN>
struct LjList {
  static constexpr int value = LEAN ? 24 : 44;
  static constexpr size_t bytes = (size_t)value * 256 * sizeof(unsigned short);
};
constexpr int kStagePad = 64;
constexpr int kQList = 8;
constexpr int kKsTile = 256;
constexpr size_t kStageBytes = (size_t)(kBatchStageCap + kStagePad) * sizeof(float4);
constexpr size_t kGidBytes = (size_t)kBatchStageCap * sizeof(int);
constexpr size_t kKsBytes = kKsTile * sizeof(float4) + 2 * (size_t)kBatchMaxK * sizeof(float4) +
                            (size_t)kBatchMaxK * sizeof(double2) +
                            2 * (size_t)kEvalBlock * sizeof(double);
static_assert(kEvalBlock == 256 && kKsBytes <= kStageBytes + LjList<true>::bytes, "k-space LDS");

// r^2 with room for the rounding of a test that shifts another operand across
// the box edge than the evaluation does: coordinates are within |lo| + L of 0,
// so the two d differ by at most 1.8e-7 (|lo| + L) per dimension and d^2 at
// the cutoff by 3.7e-7 r times the sum of these.
__device__ __forceinline__ float test_r2(const Box<float>& b, float r2) {
  const float s = fabsf(b.lo[0]) + b.L[0] + fabsf(b.lo[1]) + b.L[1] + fabsf(b.lo[2]) + b.L[2];
  return r2 + 1e-6f * sqrtf(r2) * s;
}

// Dimensions (a bit each) across whose edge a pair of charged atoms, the first
// in cell `own`, takes its image as r_j shifted by L before the subtraction;
// in the others L comes off r_j - r_i, which rounds differently: the last bit
// decides the class of a pair at a cutoff.  Shifted: the dimensions that a
// two-cell brick widened by ext_c on both sides does not cover, if that
// neighbourhood has at most kCoulImageCells cells.  Nothing here stages such a
// neighbourhood: the rule only fixes the rounding of an image, in the form in which
// stored results and trajectories have it, so that a pair at a cutoff keeps its
// class.  It follows the owner's cell, so the two directions of a pair within
// rounding of a boundary (about one in a million) may differ in class.
constexpr int kCoulImageCells = 512;
__device__ __forceinline__ int coul_shifted(const RepInfo& p, const int own[3]) {
  int m = 0, cells = 1;
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    const int w = min(2, p.nc[q] - (own[q] & ~1)) + 2 * p.ext_c[q];
    if (w < p.nc[q]) m |= 1 << q;
    cells *= min(w, p.nc[q]);
  }
  return cells <= kCoulImageCells ? m : 0;
}

// Where an owner's rows wrap (MODE 2 of lj_lane): per dimension the first
// neighbourhood cell, and the cell count of a dimension of three or four cells
// (0: its neighbourhood is staged shifted).
struct WrapLane {
  int rs[3], nc[3];
  // image shift of the owner against neighbourhood cell k
  __device__ __forceinline__ float shift(int q, int k, const Box<float>& b) const {
    const int u = rs[q] + k;
    return nc[q] == 0 ? 0.f : (u < 0 ? -b.L[q] : (u >= nc[q] ? b.L[q] : 0.f));
  }
};

// A charged owner near a box edge: dimensions (bits) staged in shifted images
// in which its pairs with charged atoms take L off r_j - r_i (coul_shifted).
// Only a distance within rounding of a cutoff is affected, so the stage stays
// as it is and such a pair, about one in a million, is looked up again.
struct QEdge {
  int mask, nslots;
  const int *soff, *sfirst;
  const float4* xs;
  const int* perm;
  const float* charge;
  // d^2 and d of the pair with the neighbourhood's atom l
  __device__ float image(const float4& xi, int l, const Box<float>& b, float& dx, float& dy,
                         float& dz) const {
    int s = 0;
    for (int k = 1; k < nslots; ++k) s = soff[k] <= l ? k : s;
    const int j = sfirst[s] + (l - soff[s]);
    if (charge[perm[j]] != 0.f) {
      const float4 x = xs[j];
      const float tx = x.x - xi.x, ty = x.y - xi.y, tz = x.z - xi.z;
      if (mask & 1) dx = fma_r(-rint(tx * b.invL[0]), b.L[0], tx);
      if (mask & 2) dy = fma_r(-rint(ty * b.invL[1]), b.L[1], ty);
      if (mask & 4) dz = fma_r(-rint(tz * b.invL[2]), b.L[2], tz);
    }
    return fma_r(dz, dz, fma_r(dy, dy, mul_rn(dx, dx)));
  }
};

// LJ pairs of one owner lane over the part [w0, w1) of the neighbourhood that
// the stage holds.  Two phases, so that the pair terms run on lanes that hold
// a pair: the candidates of each stencil row are tested 8 at a time without
// branches (d^2 - r^2's sign shifted into a mask: eight VALU instructions a
// test), the accepted stage positions go to the lane's list, and the list is
// evaluated at the end of the window (or when it would overflow).  The lpo
// lanes of an owner each take a contiguous part of every row.
// Bound by VALU issue.  256 electrolytes (777,841 atoms): 3352 us with every
// candidate's terms evaluated in one pass at the default shape, 512 to 537 us
// for the whole of kb_eval (Coulomb and k-space blocks beside it) with the lists.
//
// MODE 0: every dimension is staged in shifted images.  MODE 2: some dimension
// has three or four cells.  It is staged unshifted and its pairs take the
// minimum image as one subtraction of L from r_j - r_i, so that a pair at a
// cutoff falls on the side the single-box path puts it; the tests shift the
// owner instead (per row, and in x per side of the wrapped cell: two
// instructions a test) against test_r2, and the evaluation decides.  MODE 1:
// some dimension has fewer than three cells, and the tests take the minimum
// image as well.
template <bool RBL, bool EFLAG, bool GEN, int MODE>
__device__ __forceinline__ void lj_lane(const PairConst<float>& pc, const Box<float>& b,
                                        const float* s_lj, const float4* sx,
                                        const int* sgid, const int* soff,
                                        unsigned short* list, int T, const int lo3[3],
                                        const int hi3[3], int rn0, int rn1, int w0, int w1,
                                        bool live, const float4& xi, int li,
                                        const WrapLane& wl, const QEdge& qe, int sub, int lsh,
                                        bool shell, unsigned long long hi, const SpecRow& sr,
                                        float& fx, float& fy, float& fz, Acc<float>& a) {
  const float r2 = (EFLAG || GEN) ? fminf(pc.rclj2, pc.rc2) : pc.a_hi;
  const char* lj_row =
      reinterpret_cast<const char*>(s_lj) + (__float_as_int(xi.w) * pc.ntypes);
  const float r2t = test_r2(b, r2);
  // distances within rounding of a class boundary (none unless qe says so): the
  // cutoff, which without energies is the core's, and otherwise the core's as well
  const float near = qe.mask ? r2t - r2 : -1.f;
  auto d2_of = [&](const float4& xj, float& dx, float& dy, float& dz) {
    return MODE ? pair_d2_list<float>(b, xi.x, xi.y, xi.z, xj.x, xj.y, xj.z, dx, dy, dz)
                : pair_d2<float, false>(b, xi.x, xi.y, xi.z, xj.x, xj.y, xj.z, dx, dy, dz);
  };
  int cnt = 0;
  // entry k of the list; past its end a stand-in (the stage's first atom)
  // whose terms are dropped
  auto eval = [&](int k) {
    const bool on = k < cnt;
    const int l = on ? list[k * T] : 0;
    const float4 xj = sx[l];
    float dx, dy, dz;
    float d2 = d2_of(xj, dx, dy, dz);
    bool edge = fabsf(d2 - r2) <= near;
    if (RBL && (EFLAG || GEN)) edge = edge || fabsf(d2 - pc.t_core) <= near;
    if (RBL && GEN)  // the shell's bounds
      edge = edge || fabsf(d2 - pc.rs2) <= near || fabsf(d2 - pc.t_shell) <= near;
    if (__builtin_expect(edge, 0)) d2 = qe.image(xi, l + w0, b, dx, dy, dz);
    const float2 lj = *reinterpret_cast<const float2*>(lj_row + __float_as_int(xj.w));
    const float inv = pair_rcp(d2);
    const float s2 = lj.y * inv;
    const float s6 = s2 * s2 * s2;
    float flj = lj.x * (2.f * s6 - 1.f) * s6 * inv;
    if (!EFLAG && !GEN) {
      const float f = (on & (d2 < r2) & (d2 > pc.a_lo)) ? flj : 0.f;
      fx = fma_r(f, dx, fx);
      fy = fma_r(f, dy, fy);
      fz = fma_r(f, dz, fz);
      return;
    }
    const bool in = on & (d2 < r2);
    float ws = 1.f;
    if (GEN && in && sr.n14 > 0) ws = special_w<float>(sr, sgid[l], pc);
    flj *= ws;
    float w = 1.f;
    if (RBL) {
      const bool core = d2 < pc.t_core;
      w = (core && d2 < pc.rs2 && d2 > pc.eps_min) ? 1.f : 0.f;
      if (GEN && shell && in && !core && d2 < pc.t_shell && d2 > pc.rs2 &&
          rbl_keep(pc.ifreq, pc.fmask, pc.c32, pc.epoch, hi, rbl_hj(sgid[l])))
        w = pc.freq;
    }
    const float f = (in && w != 0.f) ? w * flj : 0.f;
    fx = fma_r(f, dx, fx);
    fy = fma_r(f, dy, fy);
    fz = fma_r(f, dz, fz);
    if (EFLAG) {
      const float eps = *reinterpret_cast<const float*>(lj_row + __float_as_int(xj.w) + 8);
      a.e_lj += in ? (double)(ws * (2.f * eps * (s6 - 1.f) * s6)) : 0.0;
      add_virial<float, EFLAG>(a, dx, dy, dz, in ? flj : 0.f);
    }
  };
  auto drain = [&]() {
    for (int k = 0; __any(k < cnt); k += 2) {
      eval(k);
      eval(k + 1);
    }
    cnt = 0;
  };
  for (int kz = lo3[2]; kz <= hi3[2]; ++kz)
    for (int ky = lo3[1]; ky <= hi3[1]; ++ky) {
      const int srow = (kz * rn1 + ky) * rn0;
      const int l0 = max(soff[srow + lo3[0]], w0) - w0;
      const int l1 = min(soff[srow + hi3[0] + 1], w1) - w0;
      const int len = max(l1 - l0, 0), part = (len + (1 << lsh) - 1) >> lsh;
      const int b0 = l0 + sub * part;
      const int n = live ? min(part, len - sub * part) : 0;
      // MODE 2: the owner's position as the tests of this row see it, on the
      // first xn candidates of the lane's part (x0) and on the rest (x1)
      float x0 = xi.x, x1 = xi.x, yr = xi.y, zr = xi.z;
      int xn = 0;
      if (MODE == 2) {
        yr -= wl.shift(1, ky, b);
        zr -= wl.shift(2, kz, b);
        x0 -= wl.shift(0, lo3[0], b);
        x1 -= wl.shift(0, hi3[0], b);
        // the wrapped cell is the row's first (x0) or its last (x1)
        const int sp = x0 != xi.x ? lo3[0] + 1 : hi3[0];
        xn = soff[srow + sp] - w0 - b0;
      }
      for (int k0 = 0; __any(k0 < n); k0 += 32) {
        unsigned m = 0;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          if (!__any(k0 + 8 * g < n)) {
            m <<= 8;
            continue;
          }
          // a lane whose row is over reads its row's start (masked below)
          const float4* xp = sx + (k0 + 8 * g < n ? b0 + k0 + 8 * g : 0);
#pragma unroll
          for (int u = 0; u < 8; ++u) {
            float dx, dy, dz, s;
            if (MODE == 2)
              s = pair_d2<float, false>(b, u + 8 * g + k0 < xn ? x0 : x1, yr, zr, xp[u].x,
                                        xp[u].y, xp[u].z, dx, dy, dz) - r2t;
            else
              s = d2_of(xp[u], dx, dy, dz) - r2t;
            m = __builtin_amdgcn_alignbit(m, __float_as_uint(s), 31);
          }
        }
        // candidates past the row's part and the owner itself
        const int rem = min(max(n - k0, 0), 32);
        m &= (unsigned)(0xffffffff00000000ull >> rem);
        const int so = li - b0 - k0;
        if ((unsigned)so < 32u) m &= ~(0x80000000u >> so);
        auto take = [&](int room) {
          while (m && cnt < room) {
            const int u = __clz((int)m);
            m &= ~(0x80000000u >> u);
            list[cnt * T] = (unsigned short)(b0 + k0 + u);
            ++cnt;
          }
        };
        constexpr int kRoom = LjList<!EFLAG && !GEN>::value;
        if (kRoom >= 32) {
          if (__any(cnt + __popc(m) > kRoom)) drain();
          take(kRoom);
        } else {
          // evaluated when some lane's list is full
          for (;;) {
            take(kRoom);
            if (!__any(m != 0)) break;
            drain();
          }
        }
      }
    }
  drain();
}

// LJ pairs of one brick: every atom of the brick against its 27 cells.
template <bool RBL, bool EFLAG, bool GEN>
__device__ __forceinline__ void lj_brick(const BatchDev& d, const PairConst<float>& pc,
                                         const RepInfo& p, int brick, const float* s_lj,
                                         char* buf, int* soff, int* sfirst, int* sedge,
                                         float fs[3], Acc<float>& a) {
  float4* sx = reinterpret_cast<float4*>(buf);
  unsigned short* list = reinterpret_cast<unsigned short*>(buf + kStageBytes) + threadIdx.x;
  int* sgid = reinterpret_cast<int*>(buf + kStageBytes + LjList<!EFLAG && !GEN>::bytes);
  const Box<float> b = p.box;
  const BrickNb h = batch_brick(p, brick);
  if (threadIdx.x < 64) {
    int cnt = 0;
    const int s = threadIdx.x;
    if (s < h.nslots) {
      const int k[3] = {s % h.rn[0], (s / h.rn[0]) % h.rn[1], s / (h.rn[0] * h.rn[1])};
      int cw[3], e = 0;
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        const int u = h.rs[q] + k[q];
        cw[q] = wrapi(u, p.nc[q]);
        e |= (u < 0 ? 0 : (u >= p.nc[q] ? 2 : 1)) << (2 * q);
      }
      const int cell = p.c0 + (cw[2] * p.nc[1] + cw[1]) * p.nc[0] + cw[0];
      sfirst[s] = d.start[cell];
      cnt = d.start[cell + 1] - d.start[cell];
      sedge[s] = e;
    }
    const int inc = wave_incl_scan(cnt);
    if (s < h.nslots) soff[s] = inc - cnt;
    if (s == 63) soff[h.nslots] = inc;
  }
  __syncthreads();
  const int total = soff[h.nslots];
  // the brick's own cells u = 0..own_n-1 (x-fastest within the brick) and
  // their atoms' running offsets (at most 8 cells)
  const int own_n = h.w[0] * h.w[1] * h.w[2];
  int own_end[8];
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    int len = 0;
    if (u < own_n) {
      const int k[3] = {u % h.w[0], (u / h.w[0]) % h.w[1], u / (h.w[0] * h.w[1])};
      const int s = ((h.o[2] - h.rs[2] + k[2]) * h.rn[1] + (h.o[1] - h.rs[1] + k[1])) *
                        h.rn[0] +
                    (h.o[0] - h.rs[0] + k[0]);
      len = soff[s + 1] - soff[s];
    }
    own_end[u] = (u > 0 ? own_end[u - 1] : 0) + len;
  }
  const int nown = own_end[7];
  // lpo adjacent lanes per owner (up to 8, as many as the block leaves idle)
  int lsh = 0;
  while (lsh < 3 && (nown << (lsh + 1)) <= (int)blockDim.x) ++lsh;
  const int lpo = 1 << lsh;
  const bool shell = RBL && pc.rclj2 > pc.rs2;
  // a neighbourhood beyond the stage goes in windows of kBatchStageCap atoms
  // (staged again for every pass over the owners)
  const bool one = total <= kBatchStageCap;
  WrapLane wl;
  bool unsh = false;
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    wl.rs[q] = h.rs[q];
    wl.nc[q] = p.nc[q] < 5 ? p.nc[q] : 0;
    unsh = unsh || p.nc[q] < 5;
  }
  for (int t0 = 0; t0 < (nown << lsh); t0 += blockDim.x) {
    const int tt = t0 + (int)threadIdx.x;
    const bool live = tt < (nown << lsh);
    const int t = live ? tt >> lsh : 0, sub = tt & (lpo - 1);
    int u = 0, ub = 0;
#pragma unroll
    for (int q = 0; q < 7; ++q)
      if (own_end[q] <= t) {
        u = q + 1;
        ub = own_end[q];
      }
    const int j0 = t - ub;
    const int k[3] = {u % h.w[0], (u / h.w[0]) % h.w[1], u / (h.w[0] * h.w[1])};
    int ko[3], lo3[3], hi3[3];
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      ko[q] = h.o[q] - h.rs[q] + k[q];
      lo3[q] = h.full[q] ? 0 : ko[q] - 1;
      hi3[q] = h.full[q] ? h.rn[q] - 1 : ko[q] + 1;
    }
    const int s_own = (ko[2] * h.rn[1] + ko[1]) * h.rn[0] + ko[0];
    const int i = sfirst[s_own] + j0;
    const int li = soff[s_own] + j0;
    const float4 xi = d.xs[i];
    const int ci = d.perm[i];
    const unsigned long long hi = (RBL && GEN) ? rbl_hi(d.gid_s[i]) : 0ull;
    const SpecRow sr = batch_spec_row<GEN>(d, pc.ms, ci);
    QEdge qe{0, h.nslots, soff, sfirst, d.xs, d.perm, d.charge};
    if (d.charge[ci] != 0.f) {
      const int own[3] = {h.o[0] + k[0], h.o[1] + k[1], h.o[2] + k[2]};
      qe.mask = ~coul_shifted(p, own) &
                ((p.nc[0] < 5 ? 0 : 1) | (p.nc[1] < 5 ? 0 : 2) | (p.nc[2] < 5 ? 0 : 4));
    }
    float fx = 0.f, fy = 0.f, fz = 0.f;
    for (int w0 = 0; w0 < total; w0 += kBatchStageCap) {
      const int w1 = min(total, w0 + kBatchStageCap);
      if (!one || t0 == 0) {
        if (!one) __syncthreads();  // the previous window's readers are done
        const int lane = threadIdx.x & 15;
        for (int s = threadIdx.x >> 4; s < h.nslots; s += blockDim.x >> 4) {
          const int o = soff[s], f = sfirst[s], e = sedge[s];
          float sh[3];
#pragma unroll
          for (int q = 0; q < 3; ++q) {
            const int c = (e >> (2 * q)) & 3;
            sh[q] = p.nc[q] < 5 ? 0.f : (c == 0 ? -b.L[q] : (c == 2 ? b.L[q] : 0.f));
          }
          const int le = min(soff[s + 1], w1);
          for (int l = max(o, w0) + lane; l < le; l += 16) {
            float4 v = d.xs[f + (l - o)];
            v.x += sh[0];
            v.y += sh[1];
            v.z += sh[2];
            sx[l - w0] = v;
            if (GEN) sgid[l - w0] = d.gid_s[f + (l - o)];
          }
        }
        __syncthreads();
      }
      if (h.mi)
        lj_lane<RBL, EFLAG, GEN, 1>(pc, b, s_lj, sx, sgid, soff, list, blockDim.x, lo3, hi3,
                                     h.rn[0], h.rn[1], w0, w1, live, xi, li - w0, wl, qe,
                                     sub, lsh, shell, hi, sr, fx, fy, fz, a);
      else if (unsh)
        lj_lane<RBL, EFLAG, GEN, 2>(pc, b, s_lj, sx, sgid, soff, list, blockDim.x, lo3, hi3,
                                     h.rn[0], h.rn[1], w0, w1, live, xi, li - w0, wl, qe,
                                     sub, lsh, shell, hi, sr, fx, fy, fz, a);
      else
        lj_lane<RBL, EFLAG, GEN, 0>(pc, b, s_lj, sx, sgid, soff, list, blockDim.x, lo3, hi3,
                                     h.rn[0], h.rn[1], w0, w1, live, xi, li - w0, wl, qe,
                                     sub, lsh, shell, hi, sr, fx, fy, fz, a);
    }
    fs[0] += fx;
    fs[1] += fy;
    fs[2] += fz;
    for (int o = lpo / 2; o > 0; o >>= 1) {
      fx += __shfl_xor(fx, o, 64);
      fy += __shfl_xor(fy, o, 64);
      fz += __shfl_xor(fz, o, 64);
    }
    if (live && sub == 0) d.fs[ci] = make_float4(fx, fy, fz, 0.f);
  }
}

// Coulomb pairs of the charged atoms [c0, c0 + block / qlanes) of a replica,
// qlanes lanes per atom, over the charged atoms of the cells within ext_c:
// the cells of one stencil row are consecutive in the compact charged order
// (two runs where the row wraps), read from cache.  Tested first, then the
// accepted ones (per-lane list) take the erfc terms and the RBL hash.
template <bool RBL, bool EFLAG, bool GEN>
__device__ __forceinline__ void coul_run(const BatchDev& d, const PairConst<float>& pc,
                                         const RepInfo& p, int c0, int qlanes, char* buf,
                                         float fs[3], Acc<float>& a) {
  int* list = reinterpret_cast<int*>(buf) + threadIdx.x;
  const int T = (int)blockDim.x;
  const Box<float> b = p.box;
  const int grp = threadIdx.x / qlanes, gl = threadIdx.x % qlanes;
  const int c = c0 + grp;
  const bool live = c < p.q0 + p.nq;
  const int cc = live ? c : p.q0 + p.nq - 1;
  const float4 xi = d.xqc[cc];
  const int4 qi = d.qi[cc];
  const unsigned long long hi = RBL ? rbl_hi(qi.x) : 0ull;
  const SpecRow sr = batch_spec_row<GEN>(d, pc.ms, qi.w);
  const int cl = qi.z - p.c0;
  const int cx = cl % p.nc[0], cy = (cl / p.nc[0]) % p.nc[1], cz = cl / (p.nc[0] * p.nc[1]);
  const Span sy = make_span(cy, p.ext_c[1], p.nc[1]), sz = make_span(cz, p.ext_c[2], p.nc[2]);
  // x cells of a row: [x0, x1] and, where the window wraps, [y0, y1]
  const Span sxs = make_span(cx, p.ext_c[0], p.nc[0]);
  const int x0 = max(sxs.start, 0), x1 = min(sxs.start + sxs.count, p.nc[0]) - 1;
  int y0 = 0, y1 = -1;
  if (sxs.start < 0) {
    y0 = sxs.start + p.nc[0];
    y1 = p.nc[0] - 1;
  } else if (sxs.start + sxs.count > p.nc[0]) {
    y1 = sxs.start + sxs.count - 1 - p.nc[0];
  }
  const int nrow = sy.count * sz.count;
  // lanes over candidates within a row (cw) and over rows, by the mean run
  int cw = 1;
  const float run = (float)p.nq * (float)sxs.count / (float)(p.nc[0] * p.nc[1] * p.nc[2]);
  while (cw < qlanes && run > 8.f * (float)cw) cw *= 2;
  const int rw = qlanes / cw, rl = gl / cw, ql = gl % cw;
  float fx = 0.f, fy = 0.f, fz = 0.f;
  int cnt = 0;
  // The nearest image of r_j - r_i (coul_shifted); the tests, which always
  // shift r_j - r_i, go against test_r2.
  const int own[3] = {cx, cy, cz};
  const int sm = coul_shifted(p, own);
  const bool shifted[3] = {(sm & 1) != 0, (sm & 2) != 0, (sm & 4) != 0};
  auto image = [&](int q, float x, float y) {
    const float t = y - x, k = rint(t * b.invL[q]);
    return fma_r(-k, b.L[q], shifted[q] ? y : t) - (shifted[q] ? x : 0.f);
  };
  const float rc2t = test_r2(b, pc.rc2);
  auto drain = [&]() {
    for (int k = 0; __any(k < cnt); ++k) {
      if (k < cnt) {
        const int j = list[k * T];
        const float4 xj = d.xqc[j];
        const float dx = image(0, xi.x, xj.x), dy = image(1, xi.y, xj.y),
                    dz = image(2, xi.z, xj.z);
        const float d2 = fma_r(dz, dz, fma_r(dy, dy, mul_rn(dx, dx)));
        if (!(d2 < pc.rc2)) continue;  // the list's test has slack
        float w = 1.f, ws = 1.f;
        if (RBL || GEN) {
          const int gj = d.qi[j].x;
          w = pair_weight<float, RBL>(pc, d2, hi, [&] { return rbl_hj(gj); });
          if (GEN && sr.n14 > 0) ws = special_w<float>(sr, gj, pc);
        }
        const float qq = xi.w * xj.w;
        const float rinv = pair_rsqrt(d2), inv = pair_rcp(d2);
        float fc, ec;
        coul<float>(pc, d2, rinv, inv, qq, fc, ec);
        // a special pair removes (1 - ws) of the full Coulomb force from
        // every kept pair, without the RBL multiplier
        const float corr = GEN ? (1.f - ws) * (-pc.qqr2e * qq * rinv * rinv * rinv) : 0.f;
        const float f = w * fc - (w != 0.f ? corr : 0.f);
        fx = fma_r(f, dx, fx);
        fy = fma_r(f, dy, fy);
        fz = fma_r(f, dz, fz);
        if (EFLAG) {
          a.e_c += (double)(ec - (GEN ? (1.f - ws) * (0.5f * pc.qqr2e * qq * rinv) : 0.f));
          add_virial<float, EFLAG>(a, dx, dy, dz, fc - corr);
        }
      }
    }
    cnt = 0;
  };
  for (int r = rl; __any(r < nrow); r += rw) {
    const int row = p.c0 + (sz.at(min(r, nrow - 1) / sy.count) * p.nc[1] +
                            sy.at(min(r, nrow - 1) % sy.count)) * p.nc[0];
    for (int seg = 0; seg < 2; ++seg) {
      const int e0 = seg ? y0 : x0, e1 = seg ? y1 : x1;
      if (!__any(e1 >= e0)) break;
      const bool on = live && r < nrow && e1 >= e0;
      const int j0 = on ? d.qstart[row + e0] : 0;
      const int j1 = on ? d.qstart[row + e1 + 1] : 0;
      for (int j = j0 + ql; __any(j < j1); j += 4 * cw) {
        float4 xj[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) xj[u] = d.xqc[j + u * cw < j1 ? j + u * cw : cc];
        if (__any(cnt + 4 > kQList)) drain();
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          float dx, dy, dz;
          const float d2 = pair_d2_list<float>(b, xi.x, xi.y, xi.z, xj[u].x, xj[u].y, xj[u].z,
                                               dx, dy, dz);
          if (j + u * cw < j1 && j + u * cw != c && d2 < rc2t) {
            list[cnt * T] = j + u * cw;
            ++cnt;
          }
        }
      }
    }
  }
  drain();
  fs[0] += fx;
  fs[1] += fy;
  fs[2] += fz;
  for (int o = qlanes / 2; o > 0; o >>= 1) {
    fx += __shfl_xor(fx, o, 64);
    fy += __shfl_xor(fy, o, 64);
    fz += __shfl_xor(fz, o, 64);
  }
  if (live && gl == 0) d.fq[qi.y] = make_float4(fx, fy, fz, 0.f);
}

// k-space of one replica: S(k) (one k per thread; with K at most half the
// block, the atoms of a tile split over block / K groups; FP32 within a tile
// and FP64 across), the energy and virial (FP64), then the force on every
// charged atom (several lanes per atom, each a part of the k's, when the
// replica has few).  RBE and EWALD: the k's of m, weights kw or
// exp(-k^2 / 4 alpha), virial E_k (delta_ab - 2 k_a k_b (1/(4 alpha) + 1/k^2)).
// RBSOG: the P sampled k's (weight kw) and the nd direct vectors (per-replica
// weights kwd), every k in the RBE form E_k = qqr2e (2 pi / V) w |rho|^2 / k^2;
// virial W_aa += E_k and W_ab += tau_k |rho_s|^2 k_s,a k_s,b with s the
// virial-chain source of a sampled k (tau = ktau, over |k_s|^4) or the direct
// vector itself (tau = kvd) (kspace_calculator_op.hip.cu:1133-1222, :1308-1352).
template <bool EFLAG>
__device__ __forceinline__ void kspace_replica(const BatchDev& d, const PairConst<float>& pc,
                                               const RepInfo& p, int r, char* buf,
                                               double* smem) {
  float4* sa = reinterpret_cast<float4*>(buf);
  float4* kf0 = sa + kKsTile;
  float4* kf1 = kf0 + kBatchMaxK;
  double2* srho = reinterpret_cast<double2*>(kf1 + kBatchMaxK);
  double* spart = reinterpret_cast<double*>(srho + kBatchMaxK);  // [2 * block]
  const double two_pi = 6.283185307179586476925;
  const int P = d.P, T = (int)blockDim.x;
  const bool sog = d.kmode == 2;
  const int K = P + (sog ? d.nd : 0);
  const int* m = d.m + (size_t)r * d.mstride;
  // integer vector of k: sampled (replica's m) or direct (shared table)
  auto mvec = [&](int k) { return k < P ? m + 3 * k : d.dm + 3 * (k - P); };
  double kv[kBatchKAcc] = {0, 0, 0, 0, 0, 0, 0};
  int kw = T;  // threads over k; T / kw groups over the atoms
  while (K <= kw / 2 && kw > 32) kw /= 2;
  const int ng = T / kw, grp = (int)threadIdx.x / kw, kt = (int)threadIdx.x % kw;
  for (int k0 = 0; k0 < K; k0 += kw) {
    const int k = k0 + kt;
    const int* mk = mvec(k < K ? k : 0);
    const float mx = (float)mk[0], my = (float)mk[1], mz = (float)mk[2];
    double re = 0.0, im = 0.0;
    for (int t0 = 0; t0 < p.nq; t0 += kKsTile) {
      const int tn = min(kKsTile, p.nq - t0);
      __syncthreads();
      for (int j = threadIdx.x; j < tn; j += T) {
        const float4 x = d.xqc[p.q0 + t0 + j];
        sa[j] = make_float4((x.x - p.box.lo[0]) * p.box.invL[0],
                            (x.y - p.box.lo[1]) * p.box.invL[1],
                            (x.z - p.box.lo[2]) * p.box.invL[2], x.w);
      }
      __syncthreads();
      float fr = 0.f, fi = 0.f;
#pragma unroll 4
      for (int j = grp; j < tn; j += ng) {
        const float4 a = sa[j];
        float sn, cs;
        sincos_rev(fma_r(mx, a.x, fma_r(my, a.y, mz * a.z)), sn, cs);
        fr = fma_r(a.w, cs, fr);
        fi = fma_r(a.w, sn, fi);
      }
      re += (double)fr;
      im += (double)fi;
    }
    if (ng > 1) {  // K <= kw: a single pass
      spart[2 * threadIdx.x] = re;
      spart[2 * threadIdx.x + 1] = im;
      __syncthreads();
      re = im = 0.0;
      for (int g = 0; g < ng; ++g) {
        re += spart[2 * (g * kw + kt)];
        im += spart[2 * (g * kw + kt) + 1];
      }
    }
    if (k < K && grp == 0) {
      const double kx = two_pi * mk[0] / (double)p.box.L[0];
      const double ky = two_pi * mk[1] / (double)p.box.L[1];
      const double kz = two_pi * mk[2] / (double)p.box.L[2];
      const double k2 = kx * kx + ky * ky + kz * kz;
      const double wk = d.kmode == 1 ? exp(-k2 / (4.0 * (double)pc.alpha))
                        : (k < P ? p.kw : d.kwd[(size_t)r * d.nd + (k - P)]);
      const double A = wk * (-4.0 * 3.141592653589793238463 * (double)pc.qqr2e) /
                       (p.volume * k2);
      kf0[k] = make_float4((float)mk[0], (float)mk[1], (float)mk[2], (float)(A * re));
      kf1[k] = make_float4((float)kx, (float)ky, (float)kz, (float)(A * im));
      srho[k] = make_double2(re, im);
      if (EFLAG) {
        const double base =
            (double)pc.qqr2e * two_pi / p.volume * wk * (re * re + im * im) / k2;
        kv[0] += base;
        if (sog) {
          kv[1] += base;
          kv[2] += base;
          kv[3] += base;
        } else {
          const double cc = 2.0 * (1.0 / (4.0 * (double)pc.alpha) + 1.0 / k2);
          kv[1] += base * (1.0 - cc * kx * kx);
          kv[2] += base * (1.0 - cc * ky * ky);
          kv[3] += base * (1.0 - cc * kz * kz);
          kv[4] += base * (-cc * kx * ky);
          kv[5] += base * (-cc * kx * kz);
          kv[6] += base * (-cc * ky * kz);
        }
      }
    }
  }
  __syncthreads();  // srho of every k is written
  if (EFLAG) {
    if (sog)
      for (int k = threadIdx.x; k < K; k += T) {
        const int src = k < P ? m[3 * P + k] : k;
        const int* ms = mvec(src);
        const double kx = two_pi * ms[0] / (double)p.box.L[0];
        const double ky = two_pi * ms[1] / (double)p.box.L[1];
        const double kz = two_pi * ms[2] / (double)p.box.L[2];
        const double2 rs = srho[src];
        double t = (k < P ? p.ktau : d.kvd[(size_t)r * d.nd + (k - P)]) *
                   (rs.x * rs.x + rs.y * rs.y);
        if (k < P) {
          const double k2 = kx * kx + ky * ky + kz * kz;
          t /= k2 * k2;
        }
        kv[1] += t * kx * kx;
        kv[2] += t * ky * ky;
        kv[3] += t * kz * kz;
        kv[4] += t * kx * ky;
        kv[5] += t * kx * kz;
        kv[6] += t * ky * kz;
      }
    block_sum<kBatchKAcc>(kv, smem);
    if (threadIdx.x == 0)
      for (int q = 0; q < kBatchKAcc; ++q) d.kacc[(size_t)r * kBatchKAcc + q] = kv[q];
  }
  // nl lanes per atom, lane s the k's s, s + nl, ...
  int nl = 1;
  while (nl < 16 && 2 * nl * p.nq <= T) nl *= 2;
  const int s = (int)threadIdx.x % nl, per = T / nl;
  for (int c0 = 0; c0 < p.nq; c0 += per) {
    const int c = c0 + (int)threadIdx.x / nl;
    const bool live = c < p.nq;
    const float4 x = d.xqc[p.q0 + (live ? c : 0)];
    const float sx = (x.x - p.box.lo[0]) * p.box.invL[0];
    const float sy = (x.y - p.box.lo[1]) * p.box.invL[1];
    const float sz = (x.z - p.box.lo[2]) * p.box.invL[2];
    float fx = 0.f, fy = 0.f, fz = 0.f;
#pragma unroll 4
    for (int k = s; k < K; k += nl) {
      const float4 a = kf0[k];
      const float4 e = kf1[k];
      float sn, cs;
      sincos_rev(fma_r(a.x, sx, fma_r(a.y, sy, a.z * sz)), sn, cs);
      const float gg = fma_r(cs, e.w, -sn * a.w);
      fx = fma_r(gg, e.x, fx);
      fy = fma_r(gg, e.y, fy);
      fz = fma_r(gg, e.z, fz);
    }
    for (int o = nl / 2; o > 0; o >>= 1) {
      fx += __shfl_xor(fx, o, 64);
      fy += __shfl_xor(fy, o, 64);
      fz += __shfl_xor(fz, o, 64);
    }
    if (live && s == 0)
      d.fk[d.qi[p.q0 + c].y] = make_float4(x.w * fx, x.w * fy, x.w * fz, 0.f);
  }
}

// Blocks [0, nk): the k-space of one replica each (first, since a large
// replica's takes longest); [nk, nk + npg): LJ, persistent over the bricks of
// the range; the rest: Coulomb, one run of charged atoms each.  Nothing
// depends on another block's result, so the k-space latency and the short
// Coulomb runs fill the machine beside the LJ bricks.
// GEN: CVFF special bonds, or an LJ cutoff beyond r_core (RBL shell pairs in
// the LJ pass), which need the candidates' global ids.
template <bool RBL, bool EFLAG, bool GEN>
__global__ __launch_bounds__(kEvalBlock) void kb_eval(BatchDev d, PairConst<float> pc_arg,
                                                      BatchRange rg, int nk, int npg,
                                                      int qlanes) {
  __shared__ __align__(16) char buf[kStageBytes + LjList<!EFLAG && !GEN>::bytes +
                                      (GEN ? kGidBytes : 0)];
  __shared__ int soff[kBatchMaxSlots + 1];
  __shared__ int sfirst[kBatchMaxSlots];
  __shared__ int sedge[kBatchMaxSlots];
  __shared__ float s_lj[4 * kBatchMaxTypes * kBatchMaxTypes];
  __shared__ double smem[(kEvalBlock / 64) * kBatchAcc];
  const int blk = (int)blockIdx.x;
  if (blk < nk) {
    const int r = rg.r0 + blk;
    kspace_replica<EFLAG>(d, pc_arg, d.rep[r], r, buf, smem);
    return;
  }
  const bool lj = blk < nk + npg;
  if (lj) {
    const int nt = pc_arg.ntypes;
    for (int q = threadIdx.x; q < 4 * nt * nt; q += blockDim.x) s_lj[q] = d.lj[q];
  }
  const long long epoch = *d.epoch;
  const int w1 = lj ? rg.w1 : rg.x1;
  for (int wi = lj ? rg.w0 + (blk - nk) : rg.x0 + (blk - nk - npg); wi < w1;
       wi += lj ? npg : w1) {
    const BatchWork wk = lj ? d.work[wi] : d.qwork[wi];
    const RepInfo& p = d.rep[wk.rep];
    PairConst<float> pc = pc_arg;
    if (RBL) {
      pc.epoch = epoch;
      pc.freq = p.freq;
      pc.ifreq = p.ifreq;
      pc.fmask = p.fmask;
      pc.c32 = p.c32;
    }
    Acc<float> a;
    float fs[3] = {0.f, 0.f, 0.f};  // this thread's share of the force sum
    if (lj) {
      __syncthreads();  // the previous item's readers of the tables are done
      lj_brick<RBL, EFLAG, GEN>(d, pc, p, wk.brick, s_lj, buf, soff, sfirst, sedge, fs, a);
    } else {
      coul_run<RBL, EFLAG, GEN>(d, pc, p, wk.brick, qlanes, buf, fs, a);
    }
    if (EFLAG) {
      double v[kBatchAcc] = {(double)fs[0], (double)fs[1], (double)fs[2], a.e_lj, a.e_c,
                             a.v[0],        a.v[1],        a.v[2],        a.v[3], a.v[4],
                             a.v[5]};
      block_sum<kBatchAcc>(v, smem);
      if (threadIdx.x == 0)
        for (int q = 0; q < kBatchAcc; ++q)
          if (v[q] != 0.0) atomicAdd(&d.racc[(size_t)wk.rep * kBatchAcc + q], v[q]);
    } else if (RBL) {  // the mean pair force
      double v[3] = {(double)fs[0], (double)fs[1], (double)fs[2]};
      block_sum<3>(v, smem);
      if (threadIdx.x == 0)
        for (int q = 0; q < 3; ++q)
          if (v[q] != 0.0) atomicAdd(&d.racc[(size_t)wk.rep * kBatchAcc + q], v[q]);
    }
  }
}

// The force rows added in caller order; the RBL mean pair force of each
// replica removed.
__global__ __launch_bounds__(256) void kb_finish(BatchDev d, BatchRange rg, int mean_fix,
                                                 int has_q, int has_k) {
  const int i = rg.a0 + blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= rg.a1) return;
  float4 f = d.fs[i];
  if (mean_fix) {
    const int r = d.rep_of[i];
    const double* acc = d.racc + (size_t)r * kBatchAcc;
    const double inv = 1.0 / (double)d.rep[r].n;
    f.x -= (float)(acc[0] * inv);
    f.y -= (float)(acc[1] * inv);
    f.z -= (float)(acc[2] * inv);
  }
  const int q = has_q ? d.qpos[i] : -1;
  if (q >= 0) {
    const float4 c = d.fq[q];
    f.x += c.x;
    f.y += c.y;
    f.z += c.z;
    if (has_k) {
      const float4 k = d.fk[q];
      f.x += k.x;
      f.y += k.y;
      f.z += k.z;
    }
  }
  d.fx[i] = f.x;
  d.fy[i] = f.y;
  d.fz[i] = f.z;
}

__global__ void kb_epoch(long long* e, long long step) { *e = step; }

inline int cdiv(int a, int b) { return (a + b - 1) / b; }

}  // namespace

hipError_t batch_set_epoch(long long* epoch, long long step, hipStream_t s) {
  hipLaunchKernelGGL(kb_epoch, dim3(1), dim3(1), 0, s, epoch, step);
  return hipGetLastError();
}

hipError_t batch_launch(const BatchDev& d, const PairConst<float>& pc, int rbl,
                        int coulomb, int eflag, int special, const BatchRange& rg,
                        const BatchTune& t, int num_cu, hipStream_t s) {
  const int na = rg.a1 - rg.a0, nw = rg.w1 - rg.w0;
  if (na <= 0) return hipSuccess;
  hipLaunchKernelGGL(kb_bin, dim3(cdiv(na, 256)), dim3(256), 0, s, d, rg);
  hipLaunchKernelGGL(kb_scan, dim3(rg.r1 - rg.r0), dim3(256), 0, s, d, rg);
  hipLaunchKernelGGL(kb_scatter, dim3(cdiv(na, 256)), dim3(256), 0, s, d, rg);
  hipLaunchKernelGGL(kb_cellsort, dim3(cdiv(na, 256)), dim3(256), 0, s, d, rg);
  const int npg = std::max(1, std::min(nw, t.grid_per_cu * num_cu));
  const int nk = coulomb && d.P > 0 ? rg.r1 - rg.r0 : 0;
  const int nq = coulomb ? rg.x1 - rg.x0 : 0;
  const bool gen = special || (rbl && pc.rclj2 > pc.rs2);
#define RBMDX_KB_EVAL(RB, EF, GE)                                                        \
  hipLaunchKernelGGL((kb_eval<RB, EF, GE>), dim3(nk + npg + nq), dim3(t.pair_block), 0, s, \
                     d, pc, rg, nk, npg, t.qlanes)
#define RBMDX_KB_EVAL2(RB, EF)   \
  if (gen)                       \
    RBMDX_KB_EVAL(RB, EF, true); \
  else                           \
    RBMDX_KB_EVAL(RB, EF, false)
  if (rbl && eflag) {
    RBMDX_KB_EVAL2(true, true);
  } else if (rbl) {
    RBMDX_KB_EVAL2(true, false);
  } else if (eflag) {
    RBMDX_KB_EVAL2(false, true);
  } else {
    RBMDX_KB_EVAL2(false, false);
  }
#undef RBMDX_KB_EVAL2
#undef RBMDX_KB_EVAL
  hipLaunchKernelGGL(kb_finish, dim3(cdiv(na, 256)), dim3(256), 0, s, d, rg, rbl,
                     coulomb ? 1 : 0, nk > 0 ? 1 : 0);
  return hipGetLastError();
}

}  // namespace rbmdx
