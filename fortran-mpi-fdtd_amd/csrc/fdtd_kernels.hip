// fdtd_kernels.hip -- gfx950 kernels of the 3D Yee time step.
//
// Field layout: one array per component, x fastest, with a one-cell ghost
// ring on every axis (index 0..n+1, the reference's (0:N+1) bounds,
// sim3/program.f90:77).  Offset of (i,j,k) = i + px*j + pxy*k, px padded.
// Non-periodic ghosts stay zero (PEC); periodic axes keep the ghost planes
// that the reference's halo exchange fills (sim3/include/mympi_func.f90:
// 241-690) up to date from inside the kernels: the E writer of plane 1
// also writes ghost n+1, the H writer of plane n also writes ghost 0.
//
// Two engines:
//  FUSED  (production): E = E + Ku*gax*curl H per cell (D is kept only in
//         dispersive cells), split-field PML cells in the same kernel,
//         source folded in.  A step is an E and an H launch, the
//         dispersive cells and the monitors beside the cells (k_step_e,
//         k_step_h), or one pass over two copies of the fields (k_march,
//         k_gen_e, k_gen_h); Lorentz groups have launches of their own.
//  STAGED (reference order): updateD, source, material E = D*gax,
//         dispersive ADE, y-slab PML with interface copies, updateH,
//         y-slab PML H -- the reference's stages in two launches
//         (k_staged_e, k_staged_h), D kept everywhere.
#include <hip/hip_runtime.h>

#include <cmath>

#include "fdtd_internal.h"

namespace fdtd {

// Exact quotient by a divisor known on the host, of any 31-bit number (m =
// ceil(2^(31+s) / d), s = ceil(log2 d): Granlund and Montgomery, "Division by
// invariant integers using multiplication", 1994): a scalar multiply and a
// shift for the wave-uniform indices, which hardware divides in vector
// floating point otherwise.
struct FastDiv {
  uint32_t m, sh;
  int32_t d;
};
inline FastDiv fast_div(int d) {
  FastDiv f;
  f.d = d;
  uint32_t sc = 0;
  while (((uint64_t)1 << sc) < (uint64_t)d) ++sc;
  f.sh = 31 + sc;
  f.m = (uint32_t)((((uint64_t)1 << f.sh) + (uint64_t)d - 1) / (uint64_t)d);
  return f;
}
__device__ __forceinline__ int fast_quot(const FastDiv& f, int v) {
  return (int)(((uint64_t)(uint32_t)v * f.m) >> f.sh);
}

template <typename real>
struct FieldArgs {
  real* e[3];
  real* h[3];
  real* d[3];
  const uint8_t* matid;
  const Vec4<real>* coef;   // Ku*gax x,y,z, PML medium gax
  const Vec4<real>* gaxe;   // gax x,y,z, energy eps
  const uint32_t* flags;    // bit q: a dielectric writes E_q
  const int32_t* rowmat;    // per ghosted (j,k) row: uniform id or -1 (dword: scalar loads)
  int32_t nx, ny, nz;
  int32_t per[3];
  int32_t px, pxy;          // offsets fit 31 bits (checked at commit)
  FastDiv by_px, by_pxy;    // i, j, k of an offset
  real ku;
  int32_t xcdmap;  // deal blocks to the 8 XCDs (one L2 each) in contiguous runs
};

// element at byte offset `off` of the row or plane that starts at p; with p
// wave-uniform the access takes a scalar address and the 32-bit offset, and
// no address arithmetic per access
template <typename real>
__device__ __forceinline__ real ld_at(const real* p, uint32_t off) {
  return *(const real*)((const char*)p + off);
}
// NT: a nontemporal store (streams_past_llc)
template <bool NT, typename real>
__device__ __forceinline__ void put(real* p, real v) {
  if constexpr (NT)
    __builtin_nontemporal_store(v, p);
  else
    *p = v;
}

// A launch of several parts gives each a whole number of rounds over the
// XCDs, so that the dealing of a part's blocks does not depend on the parts
// before it.
__host__ __device__ __forceinline__ int round8(int n) { return (n + 7) & ~7; }

// Logical block of block b of a part of nb blocks (padded to 8 * tper):
// each XCD takes a contiguous run of tper.
__device__ __forceinline__ int deal(int b, int tper, int xcdmap) { return xcdmap ? (b & 7) * tper + (b >> 3) : b; }

template <typename real>
struct PmlArgs {
  int32_t P[3];
  real* s[S_N];
  const real* f1[3];
  const real* f2[3];
  const real* g1[3];
  const real* g2[3];
  real kup;  // f2 and g2 outside an axis's slabs (f1 and g1 are 1 there)
};

template <typename real>
struct RefPmlArgs {
  int32_t P, jb;
  int64_t sx, sxy;  // slab strides: i + sx*jl + sxy*k
  real* s[2][S_N];
  const real* prof[2];  // 12 profiles per slab, stride ps
  int32_t ps;
};

// i, j, k of offset c
template <typename real>
__device__ __forceinline__ void cell_of(const FieldArgs<real>& a, int c, int& i, int& j, int& k) {
  k = fast_quot(a.by_pxy, c);
  const int r = c - k * a.pxy;
  j = fast_quot(a.by_px, r);
  i = r - j * a.px;
}

// ---------------------------------------------------------------------------
// ghost maintenance for periodic axes
template <typename real>
__device__ __forceinline__ void put_e_ghost(real* f, real v, int i, int j, int k, int64_t c,
                                            const FieldArgs<real>& a) {
  if (a.per[0] && i == 1) f[c + a.nx] = v;
  if (a.per[1] && j == 1) f[c + a.px * a.ny] = v;
  if (a.per[2] && k == 1) f[c + a.pxy * a.nz] = v;
}
template <typename real>
__device__ __forceinline__ void put_h_ghost(real* f, real v, int i, int j, int k, int64_t c,
                                            const FieldArgs<real>& a) {
  if (a.per[0] && i == a.nx) f[c - a.nx] = v;
  if (a.per[1] && j == a.ny) f[c - a.px * a.ny] = v;
  if (a.per[2] && k == a.nz) f[c - a.pxy * a.nz] = v;
}

__device__ __forceinline__ bool in_pml(const int32_t* P, int i, int j, int k, int nx, int ny, int nz) {
  return i <= P[0] || i > nx - P[0] || j <= P[1] || j > ny - P[1] || k <= P[2] || k > nz - P[2];
}

// cell v of an axis of n cells lies in one of the axis's two PML slabs
__device__ __forceinline__ bool in_slab(int P, int v, int n) { return v <= P || v > n - P; }

// Split parts of an ALL_FACES PML cell before the update.  A component is
// the sum of two parts, one per transverse axis (Ex = Exy + Exz, Ey = Eyz +
// Eyx, Ez = Ezx + Ezy; H alike); only a part whose axis's slab holds the
// cell is stored (sx, sy, sz), since the other axis's profile there is that
// of the interior (f1 = 1, f2 = Ku).  A part not stored is the old
// component less its other part, or, with neither part stored, the first
// part of the sum is the whole old component and the second 0 -- in exact
// arithmetic the same step, and a face cell moves 13 words a half step
// instead of 18.  sp: stored parts in the order yx, zx, xy, zy, xz, yz
// (the x parts, the y parts, the z parts); f: the old components; o: the
// parts in that order.
template <typename real>
__device__ __forceinline__ void pml_parts(bool sx, bool sy, bool sz, const real* sp, const real* f, real* o) {
  o[0] = sx ? sp[0] : (sz ? f[1] - sp[5] : (real)0);  // yx, second of y = yz + yx
  o[1] = sx ? sp[1] : (sy ? f[2] - sp[3] : f[2]);     // zx, first of z = zx + zy
  o[2] = sy ? sp[2] : (sz ? f[0] - sp[4] : f[0]);     // xy, first of x = xy + xz
  o[3] = sy ? sp[3] : (sx ? f[2] - sp[1] : (real)0);  // zy
  o[4] = sz ? sp[4] : (sy ? f[0] - sp[2] : (real)0);  // xz
  o[5] = sz ? sp[5] : (sx ? f[1] - sp[0] : f[1]);     // yz
}

// The six split updates of an ALL_FACES PML cell (mod3/BERpmly_mod.f90:150-155
// for E, :186-191 for H) from the parts o (pml_parts order) and the
// neighbouring fields: f1/g1 and f2/g2 are the cell's profiles along each
// axis (1 and Ku outside that axis's slabs), r the medium's 1/eps.  Every
// update of a PML cell, whichever kernel makes it, goes through these, so
// all of them round alike.
template <typename real>
__device__ __forceinline__ void e_pml_split(real fx1, real fx2, real fy1, real fy2, real fz1, real fz2, real r,
                                            const real* o, real hx, real hy, real hz, real hz_jm, real hx_jm,
                                            real hy_km, real hx_km, real hz_im, real hy_im, real* n) {
  n[0] = fx1 * o[0] + (fx2 * r) * (-hz + hz_im);    // yx
  n[1] = fx1 * o[1] + (fx2 * r) * (hy + (-hy_im));  // zx
  n[2] = fy1 * o[2] + (fy2 * r) * (hz + (-hz_jm));  // xy
  n[3] = fy1 * o[3] + (fy2 * r) * (-hx + hx_jm);    // zy
  n[4] = fz1 * o[4] + (fz2 * r) * (-hy + hy_km);    // xz
  n[5] = fz1 * o[5] + (fz2 * r) * (hx + (-hx_km));  // yz
}

template <typename real>
__device__ __forceinline__ void h_pml_split(real gx1, real gx2, real gy1, real gy2, real gz1, real gz2, const real* o,
                                            real ex, real ey, real ez, real ey_kp, real ex_kp, real ez_jp, real ex_jp,
                                            real ez_ip, real ey_ip, real* n) {
  n[0] = gx1 * o[0] + gx2 * (-ez + ez_ip);    // yx
  n[1] = gx1 * o[1] + gx2 * (ey + (-ey_ip));  // zx
  n[2] = gy1 * o[2] + gy2 * (ez + (-ez_jp));  // xy
  n[3] = gy1 * o[3] + gy2 * (-ex + ex_jp);    // zy
  n[4] = gz1 * o[4] + gz2 * (-ey + ey_kp);    // xz
  n[5] = gz1 * o[5] + gz2 * (ex + (-ex_kp));  // yz
}

// Compact index of an ALL_FACES PML cell: z slabs (full xy planes), then y
// slabs of the middle planes (full x rows), then the low and then the high
// x slab of the rest, each of those row after row (Px cells a row), so the
// rows a workgroup of one x slab updates are contiguous in every split
// array.  The count of PML cells is below the ghosted cell count, which
// fits 31 bits.
__device__ __forceinline__ int pml_index(const int32_t* P, int i, int j, int k, int nx, int ny, int nz) {
  const int Px = P[0], Py = P[1], Pz = P[2];
  if (k <= Pz || k > nz - Pz) {
    const int kk = k <= Pz ? k - 1 : Pz + (k - (nz - Pz + 1));
    return kk * nx * ny + (j - 1) * nx + (i - 1);
  }
  const int baseY = 2 * Pz * nx * ny;
  const int km = k - Pz - 1;
  if (j <= Py || j > ny - Py) {
    const int jj = j <= Py ? j - 1 : Py + (j - (ny - Py + 1));
    return baseY + (km * 2 * Py + jj) * nx + (i - 1);
  }
  const int nym = ny - 2 * Py;
  const int baseX = baseY + (nz - 2 * Pz) * 2 * Py * nx;
  const int jm = j - Py - 1;
  const bool hi = i > Px;
  const int ii = hi ? i - (nx - Px + 1) : i - 1;
  return baseX + (hi ? (nz - 2 * Pz) * nym * Px : 0) + (km * nym + jm) * Px + ii;
}

// ---------------------------------------------------------------------------
// FUSED engine: E half step (myfdtd_func.f90:19-41 in E-form, material
// update_E folded in, ALL_FACES split-field PML, plane sources).
//
// Every load is issued before the first store (e_cell_load, then
// e_cell_store): the field pointers may alias as far as the compiler knows,
// so a load placed after a store would wait for it and cost one more memory
// round trip.  The two phases are apart so that a thread marching a column
// can issue the next plane's loads before this plane's arithmetic.  UNI:
// the row has one material id `rm` (wave-uniform, the table entry read with
// scalar loads); otherwise the id is gathered per cell.
//
// z march: with use_carry, Hy and Hx of plane k-1 come from cy, cx (the
// previous plane of the same thread) instead of memory.
//
// In place (the two-kernel step) EO* are E* and pw is p.  Over two copies
// (the general tiles of the one-pass step, pp): the old E comes from EO*,
// the old splits from p, the new E goes to E* and the new splits to pw, and
// components no material writes are copied over.
template <typename real>
struct ECellIn {
  int c, s;
  bool pml, sx, sy, sz, any_src;
  uint32_t fl, id;
  Vec4<real> cf;
  real hx, hy, hz, hz_jm, hx_jm, hy_km, hx_km, hz_im, hy_im;
  real e0[3], sp[6], fx1, fx2, fy1, fy2, fz1, fz2;
};

template <typename real, bool UNI, int FACE = 0>
__device__ __forceinline__ void e_cell_load(const FieldArgs<real>& a, const PmlArgs<real>& p,
                                            const int* sa, int rm, int i, int j, int k, bool use_carry, real cy,
                                            real cx, const real* H0, const real* H1, const real* H2,
                                            const real* EO0, const real* EO1, const real* EO2, ECellIn<real>& in) {
  const int c = i + a.px * j + a.pxy * k;
  in.c = c;
  in.hx = H0[c]; in.hy = H1[c]; in.hz = H2[c];
  in.hz_jm = H2[c - a.px]; in.hx_jm = H0[c - a.px];
  in.hy_km = use_carry ? cy : H1[c - a.pxy];
  in.hx_km = use_carry ? cx : H0[c - a.pxy];
  in.hz_im = H2[c - 1]; in.hy_im = H1[c - 1];
  const unsigned id = UNI ? (unsigned)__builtin_amdgcn_readfirstlane(rm) : (unsigned)a.matid[c];
  in.id = id;
  in.fl = a.flags[id];
  in.cf = a.coef[id];
  in.pml = FACE ? true : in_pml(p.P, i, j, k, a.nx, a.ny, a.nz);
  in.any_src = sa[0] >= 0 || sa[1] >= 0 || sa[2] >= 0;
  in.s = 0;
  in.sx = in.sy = in.sz = false;
  for (int q = 0; q < 6; ++q) in.sp[q] = 0;
  in.e0[0] = in.e0[1] = in.e0[2] = 0;
  in.fx1 = in.fx2 = in.fy1 = in.fy2 = in.fz1 = in.fz2 = 0;
  if (in.pml) {
    const int s = pml_index(p.P, i, j, k, a.nx, a.ny, a.nz);
    bool sx, sy, sz;
    if constexpr (FACE == 0) {
      sx = in_slab(p.P[0], i, a.nx);
      sy = in_slab(p.P[1], j, a.ny);
      sz = in_slab(p.P[2], k, a.nz);
      in.fx1 = p.f1[0][i]; in.fx2 = p.f2[0][i];
      in.fy1 = p.f1[1][j]; in.fy2 = p.f2[1][j];
      in.fz1 = p.f1[2][k]; in.fz2 = p.f2[2][k];
    } else {  // a face cell of the y (FACE 1) or z (FACE 2) slabs: the other axes' profiles are 1, Ku
      sx = false;
      sy = FACE == 1;
      sz = FACE == 2;
      in.fx1 = (real)1; in.fx2 = p.kup;
      in.fy1 = sy ? p.f1[1][j] : (real)1; in.fy2 = sy ? p.f2[1][j] : p.kup;
      in.fz1 = sz ? p.f1[2][k] : (real)1; in.fz2 = sz ? p.f2[2][k] : p.kup;
    }
    in.s = s;
    in.sx = sx;
    in.sy = sy;
    in.sz = sz;
    // only the parts along the axes whose slabs hold the cell are stored
    // (pml_parts); the old component is read where a part is not
    if (sx) { in.sp[0] = p.s[S_EYX][s]; in.sp[1] = p.s[S_EZX][s]; }
    if (sy) { in.sp[2] = p.s[S_EXY][s]; in.sp[3] = p.s[S_EZY][s]; }
    if (sz) { in.sp[4] = p.s[S_EXZ][s]; in.sp[5] = p.s[S_EYZ][s]; }
    if (!(sy && sz)) in.e0[0] = EO0[c];
    if (!(sz && sx)) in.e0[1] = EO1[c];
    if (!(sx && sy)) in.e0[2] = EO2[c];
  } else {
    in.e0[0] = EO0[c]; in.e0[1] = EO1[c]; in.e0[2] = EO2[c];
  }
}

template <typename real>
__device__ __forceinline__ void e_cell_store(const FieldArgs<real>& a, const PmlArgs<real>& pw, bool pp,
                                             const real* sv, const int* sa, int i, int j, int k,
                                             const ECellIn<real>& in, real* E0, real* E1, real* E2) {
  const int c = in.c;
  const real* e0 = in.e0;
  const real hx = in.hx, hy = in.hy, hz = in.hz, hz_jm = in.hz_jm, hx_jm = in.hx_jm, hy_km = in.hy_km,
             hx_km = in.hx_km, hz_im = in.hz_im, hy_im = in.hy_im;
  if (in.pml) {
    // mod3/BERpmly_mod.f90:150-155 with the splits driven by total H
    const real r = in.cf.v[3];
    const int s = in.s;
    real o[6];
    pml_parts(in.sx, in.sy, in.sz, in.sp, e0, o);
    real n[6];
    e_pml_split(in.fx1, in.fx2, in.fy1, in.fy2, in.fz1, in.fz2, r, o, hx, hy, hz, hz_jm, hx_jm, hy_km, hx_km, hz_im,
                hy_im, n);
    real eyx = n[0], ezx = n[1], exy = n[2], ezy = n[3], exz = n[4], eyz = n[5];
    // a source plane through the PML feeds the split along its normal
    if (sa[0] == 1) exy = exy + sv[0] * r;
    if (sa[0] == 2) exz = exz + sv[0] * r;
    if (sa[1] == 0) eyx = eyx + sv[1] * r;
    if (sa[1] == 2) eyz = eyz + sv[1] * r;
    if (sa[2] == 0) ezx = ezx + sv[2] * r;
    if (sa[2] == 1) ezy = ezy + sv[2] * r;
    if (in.sx) { pw.s[S_EYX][s] = eyx; pw.s[S_EZX][s] = ezx; }
    if (in.sy) { pw.s[S_EXY][s] = exy; pw.s[S_EZY][s] = ezy; }
    if (in.sz) { pw.s[S_EXZ][s] = exz; pw.s[S_EYZ][s] = eyz; }
    const real ex = exy + exz, ey = eyz + eyx, ez = ezx + ezy;
    E0[c] = ex;
    E1[c] = ey;
    E2[c] = ez;
    // a periodic axis without PML of its own still meets the slabs of the
    // other axes at its boundary
    put_e_ghost(E0, ex, i, j, k, c, a);
    put_e_ghost(E1, ey, i, j, k, c, a);
    put_e_ghost(E2, ez, i, j, k, c, a);
    return;
  }
  // E_q += Ku*gax_q*curl_q (+ gax_q * source) for every component a
  // dielectric writes
  const real cur[3] = {(hz - hz_jm) + (-hy + hy_km),   // curlhzy + curlhyz
                       (hx - hx_km) + (-hz + hz_im),   // curlhxz + curlhzx
                       (hy - hy_im) + (-hx + hx_jm)};  // curlhyx + curlhxy
  const uint32_t fl = in.fl;
  // the source scale: loaded here, source planes are few
  Vec4<real> gx;
  if (in.any_src) gx = a.gaxe[in.id];
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    if (!(fl & (1u << q))) {
      if (pp && !(fl & (16u << q))) {  // no writer: the value carries over
        real* Eq = q == 0 ? E0 : (q == 1 ? E1 : E2);
        Eq[c] = e0[q];
        put_e_ghost(Eq, e0[q], i, j, k, c, a);
      }
      continue;
    }
    real ev = e0[q] + in.cf.v[q] * cur[q];
    if (sa[q] >= 0) ev = ev + gx.v[q] * sv[q];
    real* Eq = q == 0 ? E0 : (q == 1 ? E1 : E2);
    Eq[c] = ev;
    put_e_ghost(Eq, ev, i, j, k, c, a);
  }
}

template <typename real, bool UNI>
__device__ __forceinline__ void fused_e_cell(const FieldArgs<real>& a, const PmlArgs<real>& p,
                                             const PmlArgs<real>& pw, bool pp, const real* sv, const int* sa, int rm,
                                             int i, int j, int k, real& cy, real& cx, bool use_carry,
                                             const real* H0, const real* H1, const real* H2, const real* EO0,
                                             const real* EO1, const real* EO2, real* E0, real* E1, real* E2) {
  ECellIn<real> in;
  e_cell_load<real, UNI>(a, p, sa, rm, i, j, k, use_carry, cy, cx, H0, H1, H2, EO0, EO1, EO2, in);
  cy = in.hy;
  cx = in.hx;
  e_cell_store(a, pw, pp, sv, sa, i, j, k, in, E0, E1, E2);
}

// plane sources through cell (i,j,k): value and normal axis per E
// component (-1: none here).  Called before any memory load is in flight (a
// loop carrying per-lane values past outstanding loads makes the compiler
// wait for them).
template <typename real>
__device__ __forceinline__ void plane_sources(const SrcArgs<real>& src, int nsrc, int i, int j, int k, real* sv,
                                              int* sa) {
  for (int q = 0; q < nsrc; ++q) {
    const int ax = src.axis[q];
    const int pos = ax == 0 ? i : (ax == 1 ? j : k);
    if (pos == src.index[q]) {
      const int cq = src.comp[q];
      const real v = src_value(src, q);
      if (cq == 0) { sv[0] += v; sa[0] = ax; }
      else if (cq == 1) { sv[1] += v; sa[1] = ax; }
      else { sv[2] += v; sa[2] = ax; }
    }
  }
}

// The z march of one (i,j) column over planes tz*KZ+1 .. tz*KZ+KZ.  The
// field arrays come in as restrict pointers: no H array is written here and
// no E array is read through another pointer, so the compiler may issue the
// loads of the next plane before the stores of this one.
template <typename real, int KZ>
__device__ __forceinline__ void e_column(const FieldArgs<real>& a, const PmlArgs<real>& p, const SrcArgs<real>& src,
                                         int nsrc, int i, int j, int tz, const real* __restrict__ H0,
                                         const real* __restrict__ H1, const real* __restrict__ H2,
                                         real* __restrict__ E0, real* __restrict__ E1, real* __restrict__ E2) {
  real cy = 0, cx = 0;
  bool have = false;
#pragma unroll
  for (int r = 0; r < KZ; ++r) {
    const int k = tz * KZ + r + 1;
    if (k > a.nz) break;
    const int rm = a.rowmat[__builtin_amdgcn_readfirstlane(j + (a.ny + 2) * k)];
    if (rm < 0) {  // a mixed row: e_mixed_block updates it
      have = false;
      continue;
    }
    real sv[3] = {0, 0, 0};
    int sa[3] = {-1, -1, -1};
    plane_sources(src, nsrc, i, j, k, sv, sa);
    fused_e_cell<real, true>(a, p, p, false, sv, sa, rm, i, j, k, cy, cx, have, H0, H1, H2, E0, E1, E2, E0, E1, E2);
    have = true;
  }
}

// Row segments of the cell-parallel launches: a wavefront takes 64 cells of
// one (j,k) row (or of a tile of planes above it), four consecutive segments
// (x fastest) a workgroup, so j and k are wave-uniform and row data are
// scalar loads.  w counts segments; false: past the end.
struct SegGrid {
  int32_t n, tper;     // segments in all, blocks per XCD run
  FastDiv ntx, ny;     // by the segments a row, by the rows a plane
};
__device__ __forceinline__ bool seg_of(const SegGrid& g, int b, int xcdmap, int& tx, int& row) {
  const int w = deal(b, g.tper, xcdmap) * 4 + __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  if (w >= g.n) return false;
  row = fast_quot(g.ntx, w);
  tx = w - row * g.ntx.d;
  return true;
}

// Rows that mix material ids: wavefront w updates segment w % ntx of row
// rows[w / ntx] (row index j + (ny+2)*k), gathering table entries per cell.
template <typename real>
__device__ __forceinline__ void e_mixed_block(const FieldArgs<real>& a, const PmlArgs<real>& p,
                                              const SrcArgs<real>& src, int nsrc, const int32_t* rows,
                                              const SegGrid& g, int b) {
  int tx, q;
  if (!seg_of(g, b, 0, tx, q)) return;
  const int r = rows[q];
  const int i = tx * 64 + ((int)threadIdx.x & 63) + 1;
  const int j = r % (a.ny + 2), k = r / (a.ny + 2);
  if (i > a.nx) return;
  real sv[3] = {0, 0, 0};
  int sa[3] = {-1, -1, -1};
  plane_sources(src, nsrc, i, j, k, sv, sa);
  real cy = 0, cx = 0;
  fused_e_cell<real, false>(a, p, p, false, sv, sa, -1, i, j, k, cy, cx, false, a.h[0], a.h[1], a.h[2], a.e[0],
                            a.e[1], a.e[2], a.e[0], a.e[1], a.e[2]);
}

// ---------------------------------------------------------------------------
// FUSED engine: H half step (myfdtd_func.f90:45-64 + split-field H) of one
// cell, as the E step in a load phase (h_cell_load) and an arithmetic and
// store phase (h_cell_store), with 64-bit lane addresses: from row addresses
// and 32-bit offsets, as the march does, two-kernel H takes 175 against 165 us
// at 203^3 FP64, 79.9 against 79.2 in FP32, and k_gen_h 251 against 246 us at
// 320^3 FP64, 82.8 against 77.9 in FP32.  z march: with use_carry, Ex and Ey of plane
// k come from cex, cey (loaded as plane k+1 by the previous plane of the
// same thread).  In place HO* are H* and pw is p; over two copies the old
// H and splits come from HO* and p, the new ones go to H* and pw.
template <typename real>
struct HCellIn {
  int c, s;
  bool pml, sx, sy, sz;
  real ex, ey, ez, ey_kp, ex_kp, ez_jp, ex_jp, ez_ip, ey_ip;
  real h0[3], sp[6], gx1, gx2, gy1, gy2, gz1, gz2;
};

template <typename real, int FACE = 0>
__device__ __forceinline__ void h_cell_load(const FieldArgs<real>& a, const PmlArgs<real>& p, int i, int j, int k,
                                            bool use_carry, real cex, real cey, const real* E0, const real* E1,
                                            const real* E2, const real* HO0, const real* HO1, const real* HO2,
                                            HCellIn<real>& in) {
  const int c = i + a.px * j + a.pxy * k;
  in.c = c;
  in.ex = use_carry ? cex : E0[c];
  in.ey = use_carry ? cey : E1[c];
  in.ez = E2[c];
  in.ey_kp = E1[c + a.pxy]; in.ex_kp = E0[c + a.pxy];
  in.ez_jp = E2[c + a.px]; in.ex_jp = E0[c + a.px];
  in.ez_ip = E2[c + 1]; in.ey_ip = E1[c + 1];
  in.pml = FACE ? true : in_pml(p.P, i, j, k, a.nx, a.ny, a.nz);
  in.s = 0;
  in.sx = in.sy = in.sz = false;
  for (int q = 0; q < 6; ++q) in.sp[q] = 0;
  in.h0[0] = in.h0[1] = in.h0[2] = 0;
  in.gx1 = in.gx2 = in.gy1 = in.gy2 = in.gz1 = in.gz2 = 0;
  if (in.pml) {
    const int s = pml_index(p.P, i, j, k, a.nx, a.ny, a.nz);
    bool sx, sy, sz;
    if constexpr (FACE == 0) {
      sx = in_slab(p.P[0], i, a.nx);
      sy = in_slab(p.P[1], j, a.ny);
      sz = in_slab(p.P[2], k, a.nz);
      in.gx1 = p.g1[0][i]; in.gx2 = p.g2[0][i];
      in.gy1 = p.g1[1][j]; in.gy2 = p.g2[1][j];
      in.gz1 = p.g1[2][k]; in.gz2 = p.g2[2][k];
    } else {
      sx = false;
      sy = FACE == 1;
      sz = FACE == 2;
      in.gx1 = (real)1; in.gx2 = p.kup;
      in.gy1 = sy ? p.g1[1][j] : (real)1; in.gy2 = sy ? p.g2[1][j] : p.kup;
      in.gz1 = sz ? p.g1[2][k] : (real)1; in.gz2 = sz ? p.g2[2][k] : p.kup;
    }
    in.s = s;
    in.sx = sx;
    in.sy = sy;
    in.sz = sz;
    if (sx) { in.sp[0] = p.s[S_HYX][s]; in.sp[1] = p.s[S_HZX][s]; }
    if (sy) { in.sp[2] = p.s[S_HXY][s]; in.sp[3] = p.s[S_HZY][s]; }
    if (sz) { in.sp[4] = p.s[S_HXZ][s]; in.sp[5] = p.s[S_HYZ][s]; }
    if (!(sy && sz)) in.h0[0] = HO0[c];
    if (!(sz && sx)) in.h0[1] = HO1[c];
    if (!(sx && sy)) in.h0[2] = HO2[c];
  } else {
    in.h0[0] = HO0[c]; in.h0[1] = HO1[c]; in.h0[2] = HO2[c];
  }
}

template <typename real>
__device__ __forceinline__ void h_cell_store(const FieldArgs<real>& a, const PmlArgs<real>& pw, int i, int j, int k,
                                             const HCellIn<real>& in, real* H0, real* H1, real* H2) {
  const int c = in.c;
  const real ex = in.ex, ey = in.ey, ez = in.ez, ey_kp = in.ey_kp, ex_kp = in.ex_kp, ez_jp = in.ez_jp,
             ex_jp = in.ex_jp, ez_ip = in.ez_ip, ey_ip = in.ey_ip;
  if (in.pml) {
    // mod3/BERpmly_mod.f90:186-191 with the splits driven by total E
    const int s = in.s;
    real o[6];
    pml_parts(in.sx, in.sy, in.sz, in.sp, in.h0, o);
    real n[6];
    h_pml_split(in.gx1, in.gx2, in.gy1, in.gy2, in.gz1, in.gz2, o, ex, ey, ez, ey_kp, ex_kp, ez_jp, ex_jp, ez_ip, ey_ip,
                n);
    const real hyx = n[0], hzx = n[1], hxy = n[2], hzy = n[3], hxz = n[4], hyz = n[5];
    if (in.sx) { pw.s[S_HYX][s] = hyx; pw.s[S_HZX][s] = hzx; }
    if (in.sy) { pw.s[S_HXY][s] = hxy; pw.s[S_HZY][s] = hzy; }
    if (in.sz) { pw.s[S_HXZ][s] = hxz; pw.s[S_HYZ][s] = hyz; }
    const real hx = hxy + hxz, hy = hyz + hyx, hz = hzx + hzy;
    H0[c] = hx;
    H1[c] = hy;
    H2[c] = hz;
    put_h_ghost(H0, hx, i, j, k, c, a);
    put_h_ghost(H1, hy, i, j, k, c, a);
    put_h_ghost(H2, hz, i, j, k, c, a);
    return;
  }
  const real curleyz = ey_kp - ey, curlezy = -ez_jp + ez;
  const real curlezx = ez_ip - ez, curlexz = -ex_kp + ex;
  const real curlexy = ex_jp - ex, curleyx = -ey_ip + ey;
  const real hx = in.h0[0] + a.ku * (curleyz + curlezy);
  const real hy = in.h0[1] + a.ku * (curlezx + curlexz);
  const real hz = in.h0[2] + a.ku * (curlexy + curleyx);
  H0[c] = hx;
  H1[c] = hy;
  H2[c] = hz;
  put_h_ghost(H0, hx, i, j, k, c, a);
  put_h_ghost(H1, hy, i, j, k, c, a);
  put_h_ghost(H2, hz, i, j, k, c, a);
}

template <typename real>
__device__ __forceinline__ void fused_h_cell(const FieldArgs<real>& a, const PmlArgs<real>& p,
                                             const PmlArgs<real>& pw, int i, int j, int k, real& cex, real& cey,
                                             bool use_carry, const real* E0, const real* E1, const real* E2,
                                             const real* HO0, const real* HO1, const real* HO2, real* H0, real* H1,
                                             real* H2) {
  HCellIn<real> in;
  h_cell_load(a, p, i, j, k, use_carry, cex, cey, E0, E1, E2, HO0, HO1, HO2, in);
  cex = in.ex_kp;
  cey = in.ey_kp;
  h_cell_store(a, pw, i, j, k, in, H0, H1, H2);
}

// H over tiles of KZ planes, each thread marching its (i,j) column; restrict
// pointers as in e_column (no E array is written here).
template <typename real, int KZ>
__device__ __forceinline__ void h_column(const FieldArgs<real>& a, const PmlArgs<real>& p, int i, int j, int tz,
                                         const real* __restrict__ E0, const real* __restrict__ E1,
                                         const real* __restrict__ E2, real* __restrict__ H0, real* __restrict__ H1,
                                         real* __restrict__ H2) {
  real cex = 0, cey = 0;
#pragma unroll
  for (int r = 0; r < KZ; ++r) {
    const int k = tz * KZ + r + 1;
    if (k > a.nz) break;
    fused_h_cell(a, p, p, i, j, k, cex, cey, r > 0, E0, E1, E2, H0, H1, H2, H0, H1, H2);
  }
}

// ---------------------------------------------------------------------------
// x-face tiles exist in FP32 (build_march_tiles)
template <typename real>
constexpr bool kXface = sizeof(real) == 4;

// One-pass step (FUSED engine): the E and the H half step of a time step
// read from one copy of the fields and written to the other (old: m.eo,
// m.ho and the splits p.s; new: a.e, a.h and pw.s), so no cell reads a value
// another workgroup has already replaced, whatever order they run in.  The
// grid is cut into tiles of 64 x R cells over z ranges of at most kc/4 planes
// (lists built on the host, fdtd_api.hip build_march_tiles):
//
//  plain tiles (one dielectric material, no PML cell among the cells they
//  own, no x- or y-normal source plane; z-normal sources are added per
//  plane) go to march_block: one wavefront marches the tile through its
//  planes and does E and H in one pass, so each field crosses HBM once per
//  step (12 words per cell where the two-kernel step moves 18).  A plain
//  tile owns the cells of its x range [xlo, xhi]; every cell whose new E
//  it computes (its own, the row, plane and column after them) is a
//  non-PML cell of its material.
//
//  x-face tiles (FP32): plain tiles whose lanes reach into an x PML slab;
//  those lanes keep the x slab's parts (yx, zx) of E and H and take the
//  split-field update of a face cell (e_pml_split / h_pml_split, as the
//  general kernels do), the other lanes the plain one.  They share the
//  plain tiles' launch (k_march).
//
//  general tiles (PML, dispersive or mixed materials, other sources, and
//  the x-slab parts of plain tiles) go to k_gen_e and then k_gen_h, the
//  fused cell updates of the two-kernel step over the two copies.
//  Dispersive components are written into the new E in k_gen_e's launch.
//
// The arithmetic of every cell is that of the two-kernel step term for
// term, so both forms give the same bits.
//
// Everything of a tile but its lanes' columns is wave-uniform (tile index
// through readfirstlane): loop control, row and plane tests and addresses
// are scalar, an access is a scalar plane address plus a 32-bit lane offset.
// Against per-lane 64-bit addresses the FP32 kernel of 4 rows went from 195
// to 144 registers and from 1610 to 816 vector instructions; the large grids,
// bound by HBM, gained 0-2 % (320^3 FP64 113.0 -> 111.1 ms per 96 steps), the
// registers let the x-face tiles share the launch.
template <typename real>
struct MarchArgs {
  const real* eo[3];      // E after the previous step
  const real* ho[3];      // H after the previous step
};

// 8 words per entry; plain tiles: i0, j0, k0, k1, xlo, xhi (owned x range),
// material id, x face; general workgroups: x0, x1, j0, j1, k0, width, k1, face
struct TileList {
  const int32_t* tiles;
  int32_t n, tper;
  int32_t nsplit;  // general workgroups: workgroups per entry (its planes, the E update) or 1
};


// lane l receives lane l-1 (lane 0: 0) / lane l+1 (lane 63: 0); every lane
// of the wavefront must be active
template <typename real>
__device__ __forceinline__ real lane_prev(real v) {
  if constexpr (sizeof(real) == 4) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x138, 0xf, 0xf, false));
  } else {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)(b & 0xffffffffll), 0x138, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), 0x138, 0xf, 0xf, false);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
  }
}
template <typename real>
__device__ __forceinline__ real lane_next(real v) {
  if constexpr (sizeof(real) == 4) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x130, 0xf, 0xf, false));
  } else {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)(b & 0xffffffffll), 0x130, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), 0x130, 0xf, 0xf, false);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
  }
}
// value of lane l (wave-uniform l)
template <typename real>
__device__ __forceinline__ real lane_at(real v, int l) {
  if constexpr (sizeof(real) == 4) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
  } else {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffll), l);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
  }
}

// cell index v of an axis of n cells as a tile sees it: v <= n is the cell
// itself; v = n+1 is cell 1 on a periodic axis and a dead (zero) ghost
// otherwise
template <bool PER>
__device__ __forceinline__ int march_map(int v, int n, int per, bool& live) {
  live = v <= n || (PER && v == n + 1 && per);
  return v <= n ? v : 1;
}

// What a wavefront marches: its columns and rows (physical cells after the
// periodic wrap) and which of them are live / owned.  Everything but ip,
// the offsets and the lane flags is wave-uniform (scalar registers and
// branches).  The offsets are byte offsets inside a plane, fixed over the
// march: an access is a scalar plane address plus one of them, no address
// arithmetic per load (a plane is below 4 GiB: fdtd_api.hip onepass_fits).
template <int R>
struct MarchTile {
  int ip, i0, j0, jyh, jrow[R], k0, k1;
  uint32_t o[R], oyl, oyh, oxh, oxl;  // rows, row j0-1, row j0+R, columns i0+64 and i0-1
  bool lane_live, lane_own, xh_need, xg_live, yh_live, yh_need;
  bool row_live[R], row_own[R];
  bool ghosts;  // the tile owns cells on a periodic boundary
};

// Keeps an offset's widening to 64 bits inside the loop that uses it: hoisted
// out, the compiler forgets that the offset is an unsigned 32-bit one and
// adds it to the plane's address per access (a 64-bit VALU add each) instead
// of letting the access do it.  No instruction.
__device__ __forceinline__ void opaque(uint32_t& off) { asm volatile("" : "+v"(off)); }

// Old fields of one plane of a plain tile, loaded a plane ahead of use.
template <typename real, int R>
struct PlainPlane {
  real ex[R], ey[R], ez[R], hx[R], hy[R], hz[R];
  real yl_hz, yl_hx;                       // row j0-1
  real yh_ex, yh_ez, yh_hx, yh_hy, yh_hz;  // row j0+R
  real xh_ey, xh_ez, xh_hx, xh_hy, xh_hz;  // column i0+64, lane q: row j0-1+q
  real xl_hz, xl_hy;                       // column i0-1, lane q: tile row q (q = R: row j0+R)
  // x-slab lanes of x-face tiles: the kept parts (yx, zx) of the old E and H
  real pe_yx[R], pe_zx[R], ph_yx[R], ph_zx[R];
  real yh_pe_zx;  // row j0+R: old Ezx
};

// x-slab face cells in the march (tiles at the ends of a row of tiles whose
// lanes reach into an x slab, list word 7 set): the x slabs' kept parts yx,
// zx over the two copies, the x profiles, and the compact index of the x
// slabs (pml_index: base, then Px cells a row over the rows and planes
// between the y and z slabs, the high slab hioff after the low one).
template <typename real>
struct XfArgs {
  const real* eo[2];  // old Eyx, Ezx
  const real* ho[2];  // old Hyx, Hzx
  real* en[2];        // new Eyx, Ezx
  real* hn[2];        // new Hyx, Hzx
  const real *f1, *f2, *g1, *g2;
  real kup;
  int32_t Px, Py, Pz, nym, nzm, base, hioff;
};

// a lane of an x-face tile: in an x slab (on), where its row of parts
// starts, its x profiles
template <typename real>
struct XfLane {
  bool on;
  int sb;
  real f1, f2, g1, g2;
};

// offset of row j, plane k in an x slab's parts (clamped to the slab's rows
// and planes: rows and planes a tile only loads for, never stores, stay in
// bounds)
template <typename real>
__device__ __forceinline__ int xf_row(const XfArgs<real>& x, int j, int k) {
  const int km = min(max(k - x.Pz - 1, 0), x.nzm - 1);
  const int jm = min(max(j - x.Py - 1, 0), x.nym - 1);
  return (km * x.nym + jm) * x.Px;
}

// Every address below lies inside the ghosted box (rows, columns and planes
// are mapped to 0..n+1 before use), so the loads are unconditional.  A value
// loaded for a dead lane, row or plane is read only by that position's own
// new E, which is zeroed; nothing consumes the loaded registers early, so
// the loads stay in flight until the plane that uses them.
template <typename real, int R, bool XF>
__device__ __forceinline__ void plain_load(const FieldArgs<real>& a, const MarchArgs<real>& m, const XfArgs<real>& x,
                                           const XfLane<real>& xl, MarchTile<R>& w, int k,
                                           PlainPlane<real, R>& P) {
  const int64_t kb = (int64_t)a.pxy * k;
#pragma unroll
  for (int r = 0; r < R; ++r) opaque(w.o[r]);
  opaque(w.oyl);
  opaque(w.oyh);
  opaque(w.oxh);
  opaque(w.oxl);
  const real *e0 = m.eo[0] + kb, *e1 = m.eo[1] + kb, *e2 = m.eo[2] + kb;
  const real *h0 = m.ho[0] + kb, *h1 = m.ho[1] + kb, *h2 = m.ho[2] + kb;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    P.ex[r] = ld_at(e0, w.o[r]);
    P.ey[r] = ld_at(e1, w.o[r]);
    P.ez[r] = ld_at(e2, w.o[r]);
    P.hx[r] = ld_at(h0, w.o[r]);
    P.hy[r] = ld_at(h1, w.o[r]);
    P.hz[r] = ld_at(h2, w.o[r]);
  }
  // row j0-1 (a real row or the ghost row 0)
  P.yl_hz = ld_at(h2, w.oyl);
  P.yl_hx = ld_at(h0, w.oyl);
  if (w.yh_need) {  // row j0+R
    P.yh_ex = ld_at(e0, w.oyh);
    P.yh_ez = ld_at(e2, w.oyh);
    P.yh_hx = ld_at(h0, w.oyh);
    P.yh_hy = ld_at(h1, w.oyh);
    P.yh_hz = ld_at(h2, w.oyh);
  }
  if (w.xh_need) {  // column i0+64, one row per lane 0..R (lane 0: row j0-1, Hx only)
    P.xh_hx = ld_at(h0, w.oxh);
    P.xh_ey = ld_at(e1, w.oxh);
    P.xh_ez = ld_at(e2, w.oxh);
    P.xh_hy = ld_at(h1, w.oxh);
    P.xh_hz = ld_at(h2, w.oxh);
  }
  // column i0-1 (a real column or the ghost column 0), one row per lane
  P.xl_hz = ld_at(h2, w.oxl);
  P.xl_hy = ld_at(h1, w.oxl);
  if constexpr (XF) {
    if (xl.on) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int sc = xl.sb + xf_row(x, w.jrow[r], k);
        P.pe_yx[r] = x.eo[0][sc];
        P.pe_zx[r] = x.eo[1][sc];
        P.ph_yx[r] = x.ho[0][sc];
        P.ph_zx[r] = x.ho[1][sc];
      }
      P.yh_pe_zx = w.yh_need ? x.eo[1][xl.sb + xf_row(x, w.jyh, k)] : (real)0;
    } else {
#pragma unroll
      for (int r = 0; r < R; ++r) P.pe_yx[r] = P.pe_zx[r] = P.ph_yx[r] = P.ph_zx[r] = 0;
      P.yh_pe_zx = 0;
    }
  }
}

// registers carried from plane k-1 to plane k
template <typename real, int R>
struct PlainCarry {
  real hx[R], hy[R], hz[R];  // old H of plane k-1
  real ex[R], ey[R], ez[R];  // new E of plane k-1
  real yh_hy, yh_ex, yh_ez;  // row j0+R: old Hy, new Ex, Ez of plane k-1
  real xh_hx, xh_ey, xh_ez;  // column i0+64 (lane q: row j0-1+q): old Hx, new Ey, Ez of plane k-1
  real ph_yx[R], ph_zx[R];   // x-slab lanes: old H parts of plane k-1
};

// material coefficients of a plain tile (wave-uniform) and this plane's
// z-normal source terms, as fused_e_cell applies them to a dielectric cell
template <typename real>
struct PlainCoef {
  real c[3];   // Ku*gax
  real g[3];   // gax (source scaling)
  real r;      // 1/eps (the PML update's medium)
  real sv[3];  // sources of this plane per component
  bool sa[3];
};

template <typename real>
__device__ __forceinline__ real plain_e(const PlainCoef<real>& q, int c, real e0, real cur) {
  real ev = e0 + q.c[c] * cur;
  if (q.sa[c]) ev = ev + q.g[c] * q.sv[c];
  return ev;
}

template <typename real, int R, bool XF, bool PER, bool NT>
__device__ __forceinline__ void plain_plane(const FieldArgs<real>& a, const MarchArgs<real>& m,
                                            const XfArgs<real>& x, const XfLane<real>& xl,
                                            const SrcArgs<real>& src, int nsrc, PlainCoef<real> q,
                                            MarchTile<R>& w, int lane, int k,
                                            const PlainPlane<real, R>& cur, PlainPlane<real, R>& nxt,
                                            PlainCarry<real, R>& c) {
  if (k + 1 <= w.k1 + 1) {
    bool lv;
    plain_load<real, R, XF>(a, m, x, xl, w, march_map<PER>(k + 1, a.nz, a.per[2], lv), nxt);
  }
  bool live_k;
  const int kk = march_map<PER>(k, a.nz, a.per[2], live_k);
  const bool store_k = k <= w.k1;
  // this plane's z-normal sources (wave-uniform), in source order
  q.sv[0] = q.sv[1] = q.sv[2] = 0;
  q.sa[0] = q.sa[1] = q.sa[2] = false;
  for (int s = 0; s < nsrc; ++s)
    if (src.axis[s] == 2 && src.index[s] == kk) {
      const int cq = src.comp[s];
      const real v = src_value(src, s);
      if (cq == 0) { q.sv[0] += v; q.sa[0] = true; }
      else if (cq == 1) { q.sv[1] += v; q.sa[1] = true; }
      else { q.sv[2] += v; q.sa[2] = true; }
    }
  // new E of plane k on the tile's rows
  real exn[R], eyn[R], ezn[R];
  real pyx[R], pzx[R];  // x-slab lanes: the new E parts yx, zx
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const real hz_jm = r ? cur.hz[r - 1] : cur.yl_hz;
    const real hx_jm = r ? cur.hx[r - 1] : cur.yl_hx;
    real hz_im = lane_prev(cur.hz[r]);
    real hy_im = lane_prev(cur.hy[r]);
    const real lz = lane_at(cur.xl_hz, r), ly = lane_at(cur.xl_hy, r);
    if (lane == 0) {
      hz_im = lz;
      hy_im = ly;
    }
    const bool live = live_k && w.lane_live && w.row_live[r];
    const real hx = cur.hx[r], hy = cur.hy[r], hz = cur.hz[r];
    real ex = plain_e(q, 0, cur.ex[r], (hz - hz_jm) + (-hy + c.hy[r]));  // curlhzy + curlhyz
    real ey = plain_e(q, 1, cur.ey[r], (hx - c.hx[r]) + (-hz + hz_im));  // curlhxz + curlhzx
    real ez = plain_e(q, 2, cur.ez[r], (hy - hy_im) + (-hx + hx_jm));    // curlhyx + curlhxy
    pyx[r] = pzx[r] = 0;
    if constexpr (XF) {
      if (xl.on) {  // a face cell of an x slab: the split update, its x parts kept
        const real f[3] = {cur.ex[r], cur.ey[r], cur.ez[r]};
        const real sp[6] = {cur.pe_yx[r], cur.pe_zx[r], 0, 0, 0, 0};
        real o[6], n[6];
        pml_parts(true, false, false, sp, f, o);
        e_pml_split(xl.f1, xl.f2, (real)1, x.kup, (real)1, x.kup, q.r, o, hx, hy, hz, hz_jm, hx_jm, c.hy[r], c.hx[r],
                    hz_im, hy_im, n);
        ex = n[2] + n[4];
        ey = n[5] + n[0];
        ez = n[1] + n[3];
        pyx[r] = n[0];
        pzx[r] = n[1];
      }
    }
    exn[r] = live ? ex : (real)0;
    eyn[r] = live ? ey : (real)0;
    ezn[r] = live ? ez : (real)0;
  }
  // new Ex, Ez of row j0+R
  real yex = 0, yez = 0;
  if (w.yh_need) {
    real hy_im = lane_prev(cur.yh_hy);
    const real ly = lane_at(cur.xl_hy, R);
    if (lane == 0) hy_im = ly;
    const bool live = live_k && w.lane_live && w.yh_live;
    real ex = plain_e(q, 0, cur.yh_ex, (cur.yh_hz - cur.hz[R - 1]) + (-cur.yh_hy + c.yh_hy));
    real ez = plain_e(q, 2, cur.yh_ez, (cur.yh_hy - hy_im) + (-cur.yh_hx + cur.hx[R - 1]));
    if constexpr (XF) {
      if (xl.on) {  // Ex = Exy + Exz, Ez = Ezx + Ezy (the Ey inputs are not needed)
        const real f[3] = {cur.yh_ex, (real)0, cur.yh_ez};
        const real sp[6] = {(real)0, cur.yh_pe_zx, 0, 0, 0, 0};
        real o[6], n[6];
        pml_parts(true, false, false, sp, f, o);
        e_pml_split(xl.f1, xl.f2, (real)1, x.kup, (real)1, x.kup, q.r, o, cur.yh_hx, cur.yh_hy, cur.yh_hz,
                    cur.hz[R - 1], cur.hx[R - 1], c.yh_hy, (real)0, (real)0, hy_im, n);
        ex = n[2] + n[4];
        ez = n[1] + n[3];
      }
    }
    yex = live ? ex : (real)0;
    yez = live ? ez : (real)0;
  }
  // new Ey, Ez of column i0+64 (lanes 1..R: row j0-1+lane)
  real xey = 0, xez = 0;
  if (w.xh_need) {
    real hzl = 0, hyl = 0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const real vz = lane_at(cur.hz[r], 63), vy = lane_at(cur.hy[r], 63);
      if (lane == r + 1) {
        hzl = vz;
        hyl = vy;
      }
    }
    const real hx_jm = lane_prev(cur.xh_hx);
    const bool live = live_k && w.xg_live && lane >= 1 && lane <= R;
    const real ey = plain_e(q, 1, cur.xh_ey, (cur.xh_hx - c.xh_hx) + (-cur.xh_hz + hzl));
    const real ez = plain_e(q, 2, cur.xh_ez, (cur.xh_hy - hyl) + (-cur.xh_hx + hx_jm));
    xey = live ? ey : (real)0;
    xez = live ? ez : (real)0;
  }
  // stores of the new E of plane k
  if (store_k && w.lane_own) {
    const int64_t kb = (int64_t)a.pxy * kk;
    real *e0 = a.e[0] + kb, *e1 = a.e[1] + kb, *e2 = a.e[2] + kb;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if (!w.row_own[r]) continue;
      put<NT>((real*)((char*)e0 + w.o[r]), exn[r]);
      put<NT>((real*)((char*)e1 + w.o[r]), eyn[r]);
      put<NT>((real*)((char*)e2 + w.o[r]), ezn[r]);
      if (PER && w.ghosts) {
        const int64_t cc = w.ip + a.px * w.jrow[r] + kb;
        put_e_ghost(a.e[0], exn[r], w.ip, w.jrow[r], kk, cc, a);
        put_e_ghost(a.e[1], eyn[r], w.ip, w.jrow[r], kk, cc, a);
        put_e_ghost(a.e[2], ezn[r], w.ip, w.jrow[r], kk, cc, a);
      }
      if constexpr (XF) {
        if (xl.on) {
          const int sc = xl.sb + xf_row(x, w.jrow[r], kk);
          x.en[0][sc] = pyx[r];
          x.en[1][sc] = pzx[r];
        }
      }
    }
  }
  // new H of plane k-1 (myfdtd_func.f90:45-64)
  if (k > w.k0) {
    const int64_t kb = (int64_t)a.pxy * (k - 1);
    real *h0 = a.h[0] + kb, *h1 = a.h[1] + kb, *h2 = a.h[2] + kb;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const real ez_jp = r < R - 1 ? c.ez[r + 1] : c.yh_ez;
      const real ex_jp = r < R - 1 ? c.ex[r + 1] : c.yh_ex;
      real ez_ip = lane_next(c.ez[r]);
      real ey_ip = lane_next(c.ey[r]);
      const real xz = lane_at(c.xh_ez, r + 1), xy = lane_at(c.xh_ey, r + 1);
      if (lane == 63) {
        ez_ip = xz;
        ey_ip = xy;
      }
      if (!(w.lane_own && w.row_own[r])) continue;
      real hx = c.hx[r] + a.ku * ((eyn[r] - c.ey[r]) + (-ez_jp + c.ez[r]));
      real hy = c.hy[r] + a.ku * ((ez_ip - c.ez[r]) + (-exn[r] + c.ex[r]));
      real hz = c.hz[r] + a.ku * ((ex_jp - c.ex[r]) + (-ey_ip + c.ey[r]));
      const int kh = k - 1;
      if constexpr (XF) {
        if (xl.on) {
          const real f[3] = {c.hx[r], c.hy[r], c.hz[r]};
          const real sp[6] = {c.ph_yx[r], c.ph_zx[r], 0, 0, 0, 0};
          real o[6], n[6];
          pml_parts(true, false, false, sp, f, o);
          h_pml_split(xl.g1, xl.g2, (real)1, x.kup, (real)1, x.kup, o, c.ex[r], c.ey[r], c.ez[r], eyn[r], exn[r],
                      ez_jp, ex_jp, ez_ip, ey_ip, n);
          hx = n[2] + n[4];
          hy = n[5] + n[0];
          hz = n[1] + n[3];
          const int sc = xl.sb + xf_row(x, w.jrow[r], kh);
          x.hn[0][sc] = n[0];
          x.hn[1][sc] = n[1];
        }
      }
      put<NT>((real*)((char*)h0 + w.o[r]), hx);
      put<NT>((real*)((char*)h1 + w.o[r]), hy);
      put<NT>((real*)((char*)h2 + w.o[r]), hz);
      if (PER && w.ghosts) {
        const int64_t cc = w.ip + a.px * w.jrow[r] + kb;
        put_h_ghost(a.h[0], hx, w.ip, w.jrow[r], kh, cc, a);
        put_h_ghost(a.h[1], hy, w.ip, w.jrow[r], kh, cc, a);
        put_h_ghost(a.h[2], hz, w.ip, w.jrow[r], kh, cc, a);
      }
    }
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    c.hx[r] = cur.hx[r];
    c.hy[r] = cur.hy[r];
    c.hz[r] = cur.hz[r];
    c.ex[r] = exn[r];
    c.ey[r] = eyn[r];
    c.ez[r] = ezn[r];
    if constexpr (XF) {
      c.ph_yx[r] = cur.ph_yx[r];
      c.ph_zx[r] = cur.ph_zx[r];
    }
  }
  c.yh_hy = cur.yh_hy;
  c.yh_ex = yex;
  c.yh_ez = yez;
  c.xh_hx = cur.xh_hx;
  c.xh_ey = xey;
  c.xh_ez = xez;
}

// Plain tiles, four independent wavefronts per workgroup (one tile each):
// the wavefront owns the 64 x R cells of its tile over planes k0..k1; per
// plane k it computes the new E of plane k and the new H of plane k-1,
// carrying the old H and the new E of the plane below in registers while
// the loads of plane k+1 are in flight.  Neighbours come from the row
// before / after (registers), from lanes l-1 / l+1 (DPP wave shifts), and
// from halos it loads and recomputes itself: row j0-1 (old Hz, Hx), row
// j0+R (its new Ex, Ez), column i0-1 (old Hz, Hy: lanes 0..R gather one
// row each), column i0+64 (its new Ey, Ez: lanes 1..R), plane k1+1 (its new
// E).  No LDS and no barrier.  PER: some axis is periodic (the ghost stores
// and the wrapped maps cost registers and scalar branches per row and plane,
// so the handles without a periodic axis run a kernel without them).
template <typename real, int R, bool XF, bool PER, bool NT>
__device__ __forceinline__ void march_block(const FieldArgs<real>& a, const MarchArgs<real>& m, const TileList& tl,
                                            const SrcArgs<real>& src, int nsrc, const XfArgs<real>& x, int b) {
  const int lane = threadIdx.x & 63;
  const int tile = deal(b, tl.tper, a.xcdmap) * 4 + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  if (tile >= tl.n) return;  // whole wavefront
  const int32_t* T = tl.tiles + 8 * tile;
  MarchTile<R> w;
  w.i0 = __builtin_amdgcn_readfirstlane(T[0]);
  w.j0 = __builtin_amdgcn_readfirstlane(T[1]);
  w.k0 = __builtin_amdgcn_readfirstlane(T[2]);
  w.k1 = __builtin_amdgcn_readfirstlane(T[3]);
  const int xlo = __builtin_amdgcn_readfirstlane(T[4]), xhi = __builtin_amdgcn_readfirstlane(T[5]);
  const int mid = __builtin_amdgcn_readfirstlane(T[6]);
  PlainCoef<real> q;
  {
    const Vec4<real> cf = a.coef[mid], gx = a.gaxe[mid];
    for (int d = 0; d < 3; ++d) {
      q.c[d] = cf.v[d];
      q.g[d] = gx.v[d];
    }
    q.r = cf.v[3];
  }
  constexpr uint32_t ws = sizeof(real);
  const uint32_t pxb = (uint32_t)a.px * ws;
  // lanes xlo..xhi are owned; lane xhi+1 supplies the new E after the
  // range (the next cell, or the wrapped cell 1)
  w.ip = march_map<PER>(w.i0 + lane, a.nx, a.per[0], w.lane_live);
  w.lane_live = w.lane_live && w.i0 + lane >= xlo && w.i0 + lane <= xhi + 1;
  w.lane_own = w.i0 + lane >= xlo && w.i0 + lane <= xhi;
  const uint32_t ib = (uint32_t)w.ip * ws;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    w.jrow[r] = march_map<PER>(w.j0 + r, a.ny, a.per[1], w.row_live[r]);
    w.row_own[r] = w.j0 + r <= a.ny;
    w.o[r] = ib + pxb * (uint32_t)w.jrow[r];
  }
  w.oyl = ib + pxb * (uint32_t)(w.j0 - 1);
  // halo row j0+R: needed when the last tile row is owned
  w.yh_need = w.j0 + R - 1 <= a.ny;
  w.jyh = march_map<PER>(w.j0 + R, a.ny, a.per[1], w.yh_live);
  w.oyh = ib + pxb * (uint32_t)w.jyh;
  // halo column i0+64: needed when lane 63 is owned
  w.xh_need = xhi == w.i0 + 63;
  bool xh_live;
  const int ixh = march_map<PER>(w.i0 + 64, a.nx, a.per[0], xh_live);
  // gather rows: column i0+64 lane q -> row j0-1+q (q = 0..R; lane 0 only
  // supplies Hx), column i0-1 lane q -> tile row q (q < R) or the halo row
  {
    const int g = min(lane, R);
    bool lv;
    const int jxg = g == 0 ? w.j0 - 1 : march_map<PER>(w.j0 + g - 1, a.ny, a.per[1], lv);
    w.xg_live = xh_live && (g == 0 || lv);
    w.oxh = (uint32_t)ixh * ws + pxb * (uint32_t)jxg;
    const int jxl = march_map<PER>(w.j0 + g, a.ny, a.per[1], lv);
    w.oxl = (uint32_t)(w.i0 - 1) * ws + pxb * (uint32_t)jxl;
  }
  w.ghosts = PER && ((a.per[0] && (xlo == 1 || xhi == a.nx)) || (a.per[1] && (w.j0 == 1 || w.j0 + R > a.ny)) ||
             (a.per[2] && (w.k0 == 1 || w.k1 == a.nz)));
  PlainCarry<real, R> c;
  {
    // old Hx, Hy of plane k0-1 (a real plane or the ghost plane 0) for the
    // k-1 terms of plane k0
    const int64_t kb = (int64_t)a.pxy * (w.k0 - 1);
    const real *h0 = m.ho[0] + kb, *h1 = m.ho[1] + kb;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      c.hx[r] = ld_at(h0, w.o[r]);
      c.hy[r] = ld_at(h1, w.o[r]);
      c.hz[r] = 0;
      c.ex[r] = c.ey[r] = c.ez[r] = 0;
    }
    c.yh_hy = ld_at(h1, w.oyh);
    c.yh_ex = c.yh_ez = 0;
    c.xh_hx = ld_at(h0, w.oxh);
    c.xh_ey = c.xh_ez = 0;
#pragma unroll
    for (int r = 0; r < R; ++r) c.ph_yx[r] = c.ph_zx[r] = 0;
  }
  // x-face tiles (word 7): lanes in an x slab take the split update; their
  // column of the x slab's parts and their x profiles are fixed per lane
  XfLane<real> xl{};
  if constexpr (XF) {
    const int i = w.ip;
    xl.on = __builtin_amdgcn_readfirstlane(T[7]) != 0 && (i <= x.Px || i > a.nx - x.Px);
    if (xl.on) {
      const bool hi = i > x.Px;  // as pml_index (the slabs never overlap: 2 Px <= nx)
      xl.sb = x.base + (hi ? x.hioff + (i - (a.nx - x.Px + 1)) : i - 1);
      xl.f1 = x.f1[i];
      xl.f2 = x.f2[i];
      xl.g1 = x.g1[i];
      xl.g2 = x.g2[i];
    }
  }
  PlainPlane<real, R> A, B;
  plain_load<real, R, XF>(a, m, x, xl, w, w.k0, A);
  for (int k = w.k0; k <= w.k1 + 1; k += 2) {
    plain_plane<real, R, XF, PER, NT>(a, m, x, xl, src, nsrc, q, w, lane, k, A, B, c);
    if (k + 1 <= w.k1 + 1) plain_plane<real, R, XF, PER, NT>(a, m, x, xl, src, nsrc, q, w, lane, k + 1, B, A, c);
  }
}

// General work: workgroup = 256 threads over cells x0..x1 x j0..j1 of
// planes k0..k1 (list entry: x0, x1, j0, j1, k0, width, k1, face), 64 x 4 cells
// (a wavefront is one row), 32 x 8 or 16 x 16 (narrow boxes: the x edges),
// the fused cell updates over the two copies.  gen_e_block reads the old H and
// E and writes the new E, one cell per thread, a workgroup per plane (the
// planes of an entry dealt to neighbouring workgroups, so a plane's
// neighbour below is still in L2);
// k_gen_h then reads the new E and the old H and writes the new H, each
// thread marching its (i, j) column up through the planes, pipelined by
// hand: the loads of plane k+1 are issued before the arithmetic and stores
// of plane k (no plane reads what the kernel writes, so the order is
// free), and E of the plane above comes from registers (10 % faster than a
// cell per thread; the E update marched so holds too many registers and
// runs slower).
template <typename real>
__device__ __forceinline__ bool gen_cell(const FieldArgs<real>& a, const TileList& tl, int b, int& i, int& j, int& k0,
                                         int& k1, bool& wide, int& pl, int& face) {
  int lb = deal(b, tl.tper, a.xcdmap);
  if (lb >= tl.n * tl.nsplit) return false;
  pl = lb % tl.nsplit;
  lb /= tl.nsplit;
  const int32_t* T = tl.tiles + 8 * lb;
  const int bw = T[5];
  wide = bw == 64;
  const int t = (int)threadIdx.x;
  i = T[0] + (t & (bw - 1));
  j = T[2] + (wide ? __builtin_amdgcn_readfirstlane(t >> 6) : t / bw);
  k0 = T[4];
  k1 = T[6];
  face = T[7];
  return i <= T[1] && j <= T[3];
}

// a.h: the old H, a.e: the new E
template <typename real>
__device__ __forceinline__ void gen_e_block(const FieldArgs<real>& a, const PmlArgs<real>& p, const PmlArgs<real>& pw,
                                            const MarchArgs<real>& m, const TileList& tl, const SrcArgs<real>& src,
                                            int nsrc, int b) {
  int i, j, k0, k1, pl, face;
  bool wide;
  if (!gen_cell(a, tl, b, i, j, k0, k1, wide, pl, face)) return;
  const int k = k0 + pl;
  if (k > k1) return;
  real sv[3] = {0, 0, 0};
  int sa[3] = {-1, -1, -1};
  real cy = 0, cx = 0;
  const int rm = wide ? a.rowmat[__builtin_amdgcn_readfirstlane(j + (a.ny + 2) * k)] : -1;
  // face cells of one slab in rows of one dielectric, no source plane
  // (build_march_tiles); the row's id is read with scalar loads, so only
  // 64-wide rows with an id take this path
  if (face && wide && rm >= 0) {
    ECellIn<real> in;
    if (face == 2)
      e_cell_load<real, true, 2>(a, p, sa, rm, i, j, k, false, cy, cx, a.h[0], a.h[1], a.h[2], m.eo[0], m.eo[1],
                                 m.eo[2], in);
    else
      e_cell_load<real, true, 1>(a, p, sa, rm, i, j, k, false, cy, cx, a.h[0], a.h[1], a.h[2], m.eo[0], m.eo[1],
                                 m.eo[2], in);
    e_cell_store(a, pw, true, sv, sa, i, j, k, in, a.e[0], a.e[1], a.e[2]);
    return;
  }
  plane_sources(src, nsrc, i, j, k, sv, sa);
  if (rm >= 0)
    fused_e_cell<real, true>(a, p, pw, true, sv, sa, rm, i, j, k, cy, cx, false, a.h[0], a.h[1], a.h[2], m.eo[0],
                             m.eo[1], m.eo[2], a.e[0], a.e[1], a.e[2]);
  else
    fused_e_cell<real, false>(a, p, pw, true, sv, sa, -1, i, j, k, cy, cx, false, a.h[0], a.h[1], a.h[2], m.eo[0],
                              m.eo[1], m.eo[2], a.e[0], a.e[1], a.e[2]);
}

// one (i, j) column of planes k0..k1, pipelined by hand (see above)
template <typename real, int FACE>
__device__ __forceinline__ void gen_h_column(const FieldArgs<real>& a, const PmlArgs<real>& p, const PmlArgs<real>& pw,
                                             const MarchArgs<real>& m, int i, int j, int k0, int k1) {
  HCellIn<real> cur, nxt;
  h_cell_load<real, FACE>(a, p, i, j, k0, false, (real)0, (real)0, a.e[0], a.e[1], a.e[2], m.ho[0], m.ho[1],
                          m.ho[2], cur);
  for (int k = k0; k <= k1; ++k) {
    const int kn = min(k + 1, k1);
    h_cell_load<real, FACE>(a, p, i, j, kn, kn > k, cur.ex_kp, cur.ey_kp, a.e[0], a.e[1], a.e[2], m.ho[0],
                            m.ho[1], m.ho[2], nxt);
    h_cell_store(a, pw, i, j, k, cur, a.h[0], a.h[1], a.h[2]);
    cur = nxt;
  }
}

template <typename real>
__global__ __launch_bounds__(256) void k_gen_h(FieldArgs<real> a, PmlArgs<real> p, PmlArgs<real> pw,
                                               MarchArgs<real> m, TileList tl) {
  int i, j, k0, k1, pl, face;
  bool wide;
  if (!gen_cell(a, tl, (int)blockIdx.x, i, j, k0, k1, wide, pl, face)) return;
  if (face == 2)
    gen_h_column<real, 2>(a, p, pw, m, i, j, k0, k1);
  else if (face == 1)
    gen_h_column<real, 1>(a, p, pw, m, i, j, k0, k1);
  else
    gen_h_column<real, 0>(a, p, pw, m, i, j, k0, k1);
}

// ---------------------------------------------------------------------------
// Dispersive cells: Drude + up to 4 critical points + Raman
// (mod3/gold_mod.f90:61-83, mod3/graphene_mod.f90:70-100).  State SoA:
// word w of component q for cell e at state[(w*3+q)*n + e];
// words: [D (FUSED only)], I, S, g_p re, g_p im (p < ncp), sn, snm2 (Raman).
// The state and the update are FP64 in both precisions: inside a metal E is
// the small difference of the large D and I, which FP32 would cancel away
// (an FP32 state gave 6e-5 relative spectra error on the 16-disk case);
// E is stored in field precision.
// STAGED rows: D advances on rows j0..j1 (updateD between the y slabs); on
// the slabs' inner rows ja and jb the split fields write Ex and Ez (0: no
// such row).
struct StagedRows {
  int32_t j0, j1, ja, jb;
  __device__ __forceinline__ bool main(int j) const { return j >= j0 && j <= j1; }
  __device__ __forceinline__ bool pml_writes(int j, int q) const { return q != 1 && (j == ja || j == jb); }
};

// New D of a cell: updateD, sim3/include/myfdtd_func.f90:19-41, on the main
// rows, then the plane sources through it one after the other,
// sim3/program.f90:396-406 (the TFSF consistency terms among them).  False:
// D stays as it is.
template <typename real, bool NT = false>
__device__ __forceinline__ bool staged_d(const FieldArgs<real>& a, const SrcArgs<real>& src, int nsrc,
                                         const StagedRows& rows, int i, int j, int k, int c, real* d) {
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    if constexpr (NT)
      d[q] = __builtin_nontemporal_load(a.d[q] + c);
    else
      d[q] = a.d[q][c];
  }
  bool wrote = rows.main(j);
  if (wrote) {
    const real hx = a.h[0][c], hy = a.h[1][c], hz = a.h[2][c];
    const real curlhzy = hz - a.h[2][c - a.px];
    const real curlhyz = -hy + a.h[1][c - a.pxy];
    const real curlhxz = hx - a.h[0][c - a.pxy];
    const real curlhzx = -hz + a.h[2][c - 1];
    const real curlhyx = hy - a.h[1][c - 1];
    const real curlhxy = -hx + a.h[0][c - a.px];
    d[0] = d[0] + a.ku * (curlhzy + curlhyz);
    d[1] = d[1] + a.ku * (curlhxz + curlhzx);
    d[2] = d[2] + a.ku * (curlhyx + curlhxy);
  }
  for (int q = 0; q < nsrc; ++q) {
    const int pos = src.axis[q] == 0 ? i : (src.axis[q] == 1 ? j : k);
    if (pos != src.index[q]) continue;
    wrote = true;
    const int cq = src.comp[q];
    const real v = src_value(src, q);
    if (cq == 0) d[0] = d[0] + v;
    else if (cq == 1) d[1] = d[1] + v;
    else d[2] = d[2] + v;
  }
  return wrote;
}

template <typename real, bool FUSED>
__device__ __forceinline__ void ade_cell(const FieldArgs<real>& a, const AdeCoef<double>& co, const int32_t* cells,
                                         const uint8_t* masks, double* state, int64_t n, const SrcArgs<real>& src,
                                         int nsrc, int64_t e, const StagedRows& rows) {
  const int c = cells[e];
  const int mask = masks[e];
  int i, j, k;
  cell_of(a, c, i, j, k);
  double cur[3] = {0, 0, 0};
  double sv[3] = {0, 0, 0};
  real dn[3];
  if (FUSED) {
    const double hx = a.h[0][c], hy = a.h[1][c], hz = a.h[2][c];
    cur[0] = (hz - (double)a.h[2][c - a.px]) + (-hy + (double)a.h[1][c - a.pxy]);
    cur[1] = (hx - (double)a.h[0][c - a.pxy]) + (-hz + (double)a.h[2][c - 1]);
    cur[2] = (hy - (double)a.h[1][c - 1]) + (-hx + (double)a.h[0][c - a.px]);
    for (int q = 0; q < nsrc; ++q) {
      const int pos = src.axis[q] == 0 ? i : (src.axis[q] == 1 ? j : k);
      if (pos == src.index[q]) sv[src.comp[q]] += (double)src_value(src, q);
    }
  } else {
    staged_d(a, src, nsrc, rows, i, j, k, c, dn);
  }
  const int w0 = FUSED ? 1 : 0;  // word offset of I
  const int ncp = co.ncp;
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    if (!(mask & (1 << q))) continue;
    double dv;
    if (FUSED) {
      double* dp = state + (int64_t)(0 * 3 + q) * n + e;
      dv = *dp + co.ku * cur[q];
      dv = dv + sv[q];
      *dp = dv;
    } else {
      a.d[q][c] = dn[q];  // the rows' part leaves these components' D to this one
      dv = dn[q];
    }
    double* Ip = state + (int64_t)((w0 + 0) * 3 + q) * n + e;
    double* Sp = state + (int64_t)((w0 + 1) * 3 + q) * n + e;
    const double Iv = *Ip, Sv = *Sp;
    double xr = (dv - Iv) + co.ha * Sv;
    double xi = 0;
    double gr[4], gi[4];
#pragma unroll
    for (int pp = 0; pp < 4; ++pp) {
      if (pp >= ncp) break;
      gr[pp] = state[(int64_t)((w0 + 2 + pp) * 3 + q) * n + e];
      gi[pp] = state[(int64_t)((w0 + 2 + ncp + pp) * 3 + q) * n + e];
      xr = xr + (co.gbr[pp] * gr[pp] - co.gbi[pp] * gi[pp]);
      xi = xi + (co.gbr[pp] * gi[pp] + co.gbi[pp] * gr[pp]);
    }
    double snv = 0, snm2 = 0;
    double* snp = nullptr;
    double* snm2p = nullptr;
    if (co.raman) {
      snp = state + (int64_t)((w0 + 2 + 2 * ncp) * 3 + q) * n + e;
      snm2p = state + (int64_t)((w0 + 3 + 2 * ncp) * 3 + q) * n + e;
      snv = *snp;
      snm2 = *snm2p;
    }
    // E = Re[X / (ga + sn)]
    const double dr = co.gar + snv, di = co.gai;
    const double ev = (xr * dr + xi * di) / (dr * dr + di * di);
    if (FUSED || !rows.pml_writes(j, q)) {
      a.e[q][c] = (real)ev;
      put_e_ghost(a.e[q], (real)ev, i, j, k, c, a);
    }
    if (co.raman) {
      const double nsn = co.r1 * snv + co.r2 * snm2 + co.r0 * (ev * ev);
      *snm2p = snv;
      *snp = nsn;
    }
    *Ip = Iv + co.hb * ev;
    *Sp = co.ha * Sv + co.hb * ev;
#pragma unroll
    for (int pp = 0; pp < 4; ++pp) {
      if (pp >= ncp) break;
      state[(int64_t)((w0 + 2 + pp) * 3 + q) * n + e] = (co.gbr[pp] * gr[pp] - co.gbi[pp] * gi[pp]) + co.gcr[pp] * ev;
      state[(int64_t)((w0 + 2 + ncp + pp) * 3 + q) * n + e] =
          (co.gbr[pp] * gi[pp] + co.gbi[pp] * gr[pp]) + co.gci[pp] * ev;
    }
  }
}

// Up to kAdeMulti Drude/CP/Raman groups as a part of an E launch: group q
// takes blocks blk[q] .. blk[q+1]-1.  The FUSED forms advance D here and
// write components no other part writes.  The coefficients come as kernel
// arguments: read through a pointer, they were loaded again after every store
// of the state (11 -> 21 us for one 9,000-cell group alone).
constexpr int kAdeMulti = 4;
struct AdeMulti {
  int32_t ng;
  int32_t blk[kAdeMulti + 1];
  AdeCoef<double> co[kAdeMulti];
  const int32_t* cells[kAdeMulti];
  const uint8_t* masks[kAdeMulti];
  double* state[kAdeMulti];
  int64_t n[kAdeMulti];
};

template <typename real, bool FUSED>
__device__ __forceinline__ void ade_block(const FieldArgs<real>& a, const AdeMulti& g, const SrcArgs<real>& src,
                                          int nsrc, int b, const StagedRows& rows = StagedRows{}) {
  int q = 0;
  while (q + 1 < g.ng && b >= g.blk[q + 1]) ++q;
  const int64_t e = (int64_t)(b - g.blk[q]) * 256 + threadIdx.x;
  if (e >= g.n[q]) return;
  ade_cell<real, FUSED>(a, g.co[q], g.cells[q], g.masks[q], g.state[q], g.n[q], src, nsrc, e, rows);
}

// groups past the first kAdeMulti
template <typename real, bool FUSED>
__global__ __launch_bounds__(256) void k_ade_multi(FieldArgs<real> a, AdeMulti g, SrcArgs<real> src, int nsrc,
                                                   StagedRows rows) {
  ade_block<real, FUSED>(a, g, src, nsrc, (int)blockIdx.x, rows);
}

// ---------------------------------------------------------------------------
// Lorentz poles in D form (mod3/si_mod.f90:46-82): E = D - S_1 - ... - S_np
// with the S of the previous step, then per pole S_l <- ga_l*S_l +
// gb_l*S_l(older) + gc_l*E, in the module's operation order.  FUSED: D is
// kept in state word 0 and advanced here from curl H (E-form engine), as
// ade_cell does.  State SoA, word w of component q for cell e at
// state[(w*3+q)*n + e]; words: [D], S_l (l < np), S_l one step older.  FP64
// in both precisions; E is stored in field precision.
template <typename real, bool FUSED>
__global__ __launch_bounds__(256) void k_lord(FieldArgs<real> a, LordCoef co, const int32_t* cells,
                                              const uint8_t* masks, double* state, int64_t n, SrcArgs<real> src,
                                              int nsrc) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n) return;
  const int c = cells[e];
  const int mask = masks[e];
  int i, j, k;
  cell_of(a, c, i, j, k);
  double cur[3] = {0, 0, 0};
  double sv[3] = {0, 0, 0};
  if (FUSED) {
    const double hx = a.h[0][c], hy = a.h[1][c], hz = a.h[2][c];
    cur[0] = (hz - (double)a.h[2][c - a.px]) + (-hy + (double)a.h[1][c - a.pxy]);
    cur[1] = (hx - (double)a.h[0][c - a.pxy]) + (-hz + (double)a.h[2][c - 1]);
    cur[2] = (hy - (double)a.h[1][c - 1]) + (-hx + (double)a.h[0][c - a.px]);
    for (int q = 0; q < nsrc; ++q) {
      const int pos = src.axis[q] == 0 ? i : (src.axis[q] == 1 ? j : k);
      if (pos == src.index[q]) sv[src.comp[q]] += (double)src_value(src, q);
    }
  }
  const int w0 = FUSED ? 1 : 0;
  const int np = co.npols;
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    if (!(mask & (1 << q))) continue;
    double dv;
    if (FUSED) {
      double* dp = state + (int64_t)q * n + e;
      dv = *dp + co.ku * cur[q];
      dv = dv + sv[q];
      *dp = dv;
    } else {
      dv = a.d[q][c];
    }
    double s1[4], s2[4];
    double ev = dv;
#pragma unroll
    for (int l = 0; l < 4; ++l) {
      if (l >= np) break;
      s1[l] = state[(int64_t)((w0 + l) * 3 + q) * n + e];
      s2[l] = state[(int64_t)((w0 + np + l) * 3 + q) * n + e];
      ev = ev - s1[l];
    }
    a.e[q][c] = (real)ev;
    put_e_ghost(a.e[q], (real)ev, i, j, k, c, a);
#pragma unroll
    for (int l = 0; l < 4; ++l) {
      if (l >= np) break;
      state[(int64_t)((w0 + l) * 3 + q) * n + e] = (co.ga[l] * s1[l] + co.gb[l] * s2[l]) + co.gc[l] * ev;
      state[(int64_t)((w0 + np + l) * 3 + q) * n + e] = s1[l];
    }
  }
}

// ---------------------------------------------------------------------------
// Lorentz-Jp cells, E form (mod3/goldLorentzJp_mod.f90:37-91 and the family:
// grapheneLorentzJp_mod.f90:42-101 adds the third-order oscillator and
// drives Ez with JpT_x).  The pole state is FP64 in both precisions (an FP32
// P would lose the small per-step increments dt*Jp of slow poles); the E
// update is evaluated in FP64 and stored in field precision.  State SoA,
// word w of component q for cell e at state[(w*3+q)*n + e]; words: P_l
// (l < npols), Jp_l, [Q, G].  JpT is the running sum of the Jp_l, summed in
// pole order as the modules accumulate it.
template <typename real>
__global__ __launch_bounds__(256) void k_ljp(FieldArgs<real> a, LjpCoef<double> co, const int32_t* cells,
                                             const uint8_t* masks, double* state, int64_t n, SrcArgs<real> src,
                                             int nsrc) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n) return;
  const int c = cells[e];
  const int mask = masks[e];
  int i, j, k;
  cell_of(a, c, i, j, k);
  const real hx = a.h[0][c], hy = a.h[1][c], hz = a.h[2][c];
  const real cur[3] = {(hz - a.h[2][c - a.px]) + (-hy + a.h[1][c - a.pxy]),   // curlhzy + curlhyz
                       (hx - a.h[0][c - a.pxy]) + (-hz + a.h[2][c - 1]),     // curlhxz + curlhzx
                       (hy - a.h[1][c - 1]) + (-hx + a.h[0][c - a.px])};     // curlhyx + curlhxy
  real sv[3] = {0, 0, 0};
  int hit = 0;  // bit q: a source plane through this cell feeds E_q
  for (int q = 0; q < nsrc; ++q) {
    const int pos = src.axis[q] == 0 ? i : (src.axis[q] == 1 ? j : k);
    if (pos == src.index[q]) {
      sv[src.comp[q]] += src_value(src, q);
      hit |= 1 << src.comp[q];
    }
  }
  const int np = co.npols;
  const int wq = 2 * np;  // word of Q
  double jt[3] = {0, 0, 0};
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    if (!((co.jmask >> q) & 1)) continue;
#pragma unroll
    for (int l = 0; l < 4; ++l) {
      if (l >= np) break;
      jt[q] = jt[q] + state[(int64_t)((np + l) * 3 + q) * n + e];
    }
  }
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    if (!(mask & (1 << q))) continue;
    const double jd = (q == 2 && co.ezjx) ? jt[0] : jt[q];
    double ev = (double)a.e[q][c] + co.kuga * ((double)cur[q] - co.ds * jd);
    if ((hit >> q) & 1) ev = ev + co.ga * (double)sv[q];
    const real er = (real)ev;
    a.e[q][c] = er;
    put_e_ghost(a.e[q], er, i, j, k, c, a);
    double Qv = 0;
    if (co.nl) Qv = state[(int64_t)(wq * 3 + q) * n + e];
#pragma unroll
    for (int l = 0; l < 4; ++l) {
      if (l >= np) break;
      double* Pp = state + (int64_t)(l * 3 + q) * n + e;
      double* Jp = state + (int64_t)((np + l) * 3 + q) * n + e;
      double p0 = (co.xi[l] * ev) / co.c0;
      if (l == 0 && co.nl) p0 = p0 + ((co.xi3 * Qv) * ev) / co.c0;
      const double jn = co.g1[l] * *Jp + co.g2[l] * (p0 - *Pp);
      *Jp = jn;
      *Pp = *Pp + co.dt * jn;
    }
    if (co.nl) {
      double* Gp = state + (int64_t)((wq + 1) * 3 + q) * n + e;
      const double ze = co.z0 * ev;
      const double gn = co.ng1 * *Gp + co.ng2 * (ze * ze - Qv);
      *Gp = gn;
      state[(int64_t)(wq * 3 + q) * n + e] = Qv + co.dt * gn;
    }
  }
}

// ---------------------------------------------------------------------------
// STAGED engine: updateD, the sources and update_E of one cell in one pass
// (each cell's D and E depend on H alone), as the reference's stages compute
// it; E of the dispersive materials and the split fields are other parts of
// the same launch (k_staged_e).
//
// ConstantDielectric%update_E for every cell/component whose last writer is
// a dielectric (mod3/simpledielectric_mod.f90:181-183).  flags bit 8+q: the
// dispersive cells' part advances D_q.
template <typename real, bool NT>
__device__ __forceinline__ void staged_e_cell(const FieldArgs<real>& a, const SrcArgs<real>& src, int nsrc,
                                              const StagedRows& rows, int i, int j, int k, uint32_t fl,
                                              const Vec4<real>& gx) {
  const int c = i + a.px * j + a.pxy * k;
  real d[3];
  const bool wrote = staged_d<real, NT>(a, src, nsrc, rows, i, j, k, c, d);
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    if (wrote && !(fl & (256u << q))) put<NT>(a.d[q] + c, d[q]);
    if (!(fl & (1u << q)) || rows.pml_writes(j, q)) continue;
    const real ev = d[q] * gx.v[q];
    a.e[q][c] = ev;
    put_e_ghost(a.e[q], ev, i, j, k, c, a);
  }
}

// updateH, sim3/include/myfdtd_func.f90:45-64, of one main-row cell; the row
// below the upper slab is copied into the slab's ghost row (ref_pml_e_cell).
template <typename real>
__device__ __forceinline__ void staged_h_cell(const FieldArgs<real>& a, const RefPmlArgs<real>& p,
                                              const StagedRows& rows, int i, int j, int k) {
  const int c = i + a.px * j + a.pxy * k;
  const real ex = a.e[0][c], ey = a.e[1][c], ez = a.e[2][c];
  const real curleyz = a.e[1][c + a.pxy] - ey;
  const real curlezy = -a.e[2][c + a.px] + ez;
  const real curlezx = a.e[2][c + 1] - ez;
  const real curlexz = -a.e[0][c + a.pxy] + ex;
  const real curlexy = a.e[0][c + a.px] - ex;
  const real curleyx = -a.e[1][c + 1] + ey;
  const real hx = a.h[0][c] + a.ku * (curleyz + curlezy);
  const real hy = a.h[1][c] + a.ku * (curlezx + curlexz);
  const real hz = a.h[2][c] + a.ku * (curlexy + curleyx);
  a.h[0][c] = hx;
  a.h[1][c] = hy;
  a.h[2][c] = hz;
  put_h_ghost(a.h[0], hx, i, j, k, c, a);
  put_h_ghost(a.h[1], hy, i, j, k, c, a);
  put_h_ghost(a.h[2], hz, i, j, k, c, a);
  if (j + 1 == rows.jb) {
    const int64_t o = i + p.sxy * k;  // slab row 0
    p.s[1][S_HXY][o] = hx;
    p.s[1][S_HZY][o] = hz;
  }
}

// Reference y-slab PML, E: updateEs (mod3/BERpmly_mod.f90:117-159) driven by
// split H only, then setboundayEya/Eyb (:200-225,255-278).  Slab 0 holds
// rows 0..P+1, slab 1 rows jb-1..ny+1; split ghosts stay zero.  The module
// copies the main fields of the row beyond a slab's inner one into the
// slab's ghost row (E and H of rows P+1 and jb-1).  Two of the copies are
// read.  H of row jb-1, in the next step's E update of row jb: it is the row
// as updateH left it, whatever the TFSF terms or the caller add to H after
// that, so the thread that updates the row keeps the copy (staged_h_cell;
// the slab's H cells, beside it in the launch, do not read it).  E of row
// P+1, in the H update of row P of the same step: nothing writes it in
// between, and the H update takes the main field.
template <typename real>
__device__ __forceinline__ void ref_pml_e_cell(const FieldArgs<real>& a, const RefPmlArgs<real>& p, int i, int jr,
                                               int k) {
  const int sl = jr < p.P ? 0 : 1;
  const int j = sl == 0 ? jr + 1 : p.jb + (jr - p.P);
  const int jl = sl == 0 ? j : j - (p.jb - 1);
  real* const* S = p.s[sl];
  const real* pr = p.prof[sl];
  const int ps = p.ps;
  const int64_t o = i + p.sx * jl + p.sxy * k;
  const int64_t ojm = o - p.sx, okm = o - p.sxy, oim = o - 1;
  const int c = i + a.px * j + a.pxy * k;
  const real curlHzy_p = S[S_HZX][o] + S[S_HZY][o];
  const real curlHzy_m = -S[S_HZX][ojm] - S[S_HZY][ojm];
  const real curlHyz_p = -S[S_HYZ][o] - S[S_HYX][o];
  const real curlHyz_m = S[S_HYZ][okm] + S[S_HYX][okm];
  const real curlHxz_p = S[S_HXY][o] + S[S_HXZ][o];
  const real curlHxz_m = -S[S_HXY][okm] - S[S_HXZ][okm];
  const real curlHzx_p = -S[S_HZX][o] - S[S_HZY][o];
  const real curlHzx_m = S[S_HZX][oim] + S[S_HZY][oim];
  const real curlHyx_p = S[S_HYZ][o] + S[S_HYX][o];
  const real curlHyx_m = -S[S_HYZ][oim] - S[S_HYX][oim];
  const real curlHxy_p = -S[S_HXY][o] - S[S_HXZ][o];
  const real curlHxy_m = S[S_HXY][ojm] + S[S_HXZ][ojm];
  const real f1x = pr[0 * ps + i], f2x = pr[1 * ps + i];
  const real f1y = pr[2 * ps + j], f2y = pr[3 * ps + j];
  const real f1z = pr[4 * ps + k], f2z = pr[5 * ps + k];
  S[S_EYX][o] = f1x * S[S_EYX][o] + f2x * (curlHzx_p + curlHzx_m);
  S[S_EZX][o] = f1x * S[S_EZX][o] + f2x * (curlHyx_p + curlHyx_m);
  const real exy = f1y * S[S_EXY][o] + f2y * (curlHzy_p + curlHzy_m);
  const real ezy = f1y * S[S_EZY][o] + f2y * (curlHxy_p + curlHxy_m);
  S[S_EXY][o] = exy;
  S[S_EZY][o] = ezy;
  S[S_EXZ][o] = f1z * S[S_EXZ][o] + f2z * (curlHyz_p + curlHyz_m);
  S[S_EYZ][o] = f1z * S[S_EYZ][o] + f2z * (curlHxz_p + curlHxz_m);
  if (sl == 0 ? j == p.P : j == p.jb) {
    a.e[0][c] = exy;
    a.e[2][c] = ezy;
  }
}

// Reference y-slab PML, H: updateHs (:161-195) and setboundayHya/Hyb.
template <typename real>
__device__ __forceinline__ void ref_pml_h_cell(const FieldArgs<real>& a, const RefPmlArgs<real>& p, int i, int jr,
                                               int k) {
  const int sl = jr < p.P ? 0 : 1;
  const int j = sl == 0 ? jr + 1 : p.jb + (jr - p.P);
  const int jl = sl == 0 ? j : j - (p.jb - 1);
  real* const* S = p.s[sl];
  const real* pr = p.prof[sl];
  const int ps = p.ps;
  const int64_t o = i + p.sx * jl + p.sxy * k;
  const int64_t ojp = o + p.sx, okp = o + p.sxy, oip = o + 1;
  const int c = i + a.px * j + a.pxy * k;
  const bool edge = sl == 0 && j == p.P;  // the row above is the main one P+1
  const real curlEzy_p = edge ? -a.e[2][c + a.px] : -S[S_EZX][ojp] - S[S_EZY][ojp];
  const real curlEzy_m = S[S_EZX][o] + S[S_EZY][o];
  const real curlEyz_p = S[S_EYZ][okp] + S[S_EYX][okp];
  const real curlEyz_m = -S[S_EYZ][o] - S[S_EYX][o];
  const real curlExz_p = -S[S_EXY][okp] - S[S_EXZ][okp];
  const real curlExz_m = S[S_EXY][o] + S[S_EXZ][o];
  const real curlEzx_p = S[S_EZX][oip] + S[S_EZY][oip];
  const real curlEzx_m = -S[S_EZX][o] - S[S_EZY][o];
  const real curlEyx_p = -S[S_EYZ][oip] - S[S_EYX][oip];
  const real curlEyx_m = S[S_EYZ][o] + S[S_EYX][o];
  const real curlExy_p = edge ? a.e[0][c + a.px] : S[S_EXY][ojp] + S[S_EXZ][ojp];
  const real curlExy_m = -S[S_EXY][o] - S[S_EXZ][o];
  const real g1x = pr[6 * ps + i], g2x = pr[7 * ps + i];
  const real g1y = pr[8 * ps + j], g2y = pr[9 * ps + j];
  const real g1z = pr[10 * ps + k], g2z = pr[11 * ps + k];
  S[S_HYX][o] = g1x * S[S_HYX][o] + g2x * (curlEzx_m + curlEzx_p);
  S[S_HZX][o] = g1x * S[S_HZX][o] + g2x * (curlEyx_m + curlEyx_p);
  const real hxy = g1y * S[S_HXY][o] + g2y * (curlEzy_m + curlEzy_p);
  const real hzy = g1y * S[S_HZY][o] + g2y * (curlExy_m + curlExy_p);
  S[S_HXY][o] = hxy;
  S[S_HZY][o] = hzy;
  S[S_HXZ][o] = g1z * S[S_HXZ][o] + g2z * (curlEyz_m + curlEyz_p);
  S[S_HYZ][o] = g1z * S[S_HYZ][o] + g2z * (curlExz_m + curlExz_p);
  if (sl == 0 ? j == p.P : j == p.jb) {
    a.h[0][c] = hxy;
    a.h[2][c] = hzy;
  }
}

// ---------------------------------------------------------------------------
// Monitors: running DFT on a plane (sim3/program.f90:456-472), time-blocked:
// every gated step copies the plane's selected components into a ring of
// kDftBlock samples; a flush adds dt * sum_b cos/sin(w t_b) F_b, t_b =
// (n_b - 1) dt, to the FP64 accumulators [slot][re|im][m][v][u].
// The samples of up to kMonPlanes DFT planes, each laid out as
// samples[slot][v][u] (u, v the plane's two free axes in x, y, z order), then
// the probes, as a part of a launch that leaves the fields they read alone
// (or a launch of their own at the end of a call or a DFT block).  Plane q
// owns blocks blk[q] .. blk[q+1]-1, (np+255)/256 per sampled component; the
// blocks from blk[nplanes] on write the probes.  The two-kernel step samples
// E in its H launch and H in the next step's E launch.
constexpr int kMonPlanes = 8;
template <typename real>
struct MonList {
  int32_t nplanes, nprobe, nblk;
  int32_t part;            // probes: 1 the time and E, 2 H, 3 all
  int32_t axis[kMonPlanes], index[kMonPlanes], n1[kMonPlanes];
  int64_t np[kMonPlanes];
  uint64_t sel[kMonPlanes];  // byte q: component | slot << 4 of the plane's q-th sample
  real* dst[kMonPlanes];
  int32_t blk[kMonPlanes + 1];
  const int32_t* ppos;
  double* pout;
  double tn;
};

// F(c): array of component c (0..2 E, 3..5 H)
template <typename real, typename Fields>
__device__ __forceinline__ void mon_block(const MonList<real>& m, int px, int pxy, int b, const Fields& F) {
  if (b >= m.nblk) return;
  if (b >= m.blk[m.nplanes]) {  // point probes, sim3/program.f90:445-451 (incident-line probes are written by k_tfsf_h)
    const int p = (b - m.blk[m.nplanes]) * 256 + (int)threadIdx.x;
    if (p >= m.nprobe || m.ppos[3 * p] < 0) return;
    const int64_t c = m.ppos[3 * p] + px * m.ppos[3 * p + 1] + pxy * m.ppos[3 * p + 2];
    double* r = m.pout + 7 * p;
    if (m.part & 1) {
      r[0] = m.tn;
      for (int q = 0; q < 3; ++q) r[1 + q] = (double)F(q)[c];
    }
    if (m.part & 2)
      for (int q = 3; q < 6; ++q) r[1 + q] = (double)F(q)[c];
    return;
  }
  int q = 0;
  while (q + 1 < m.nplanes && b >= m.blk[q + 1]) ++q;
  const int64_t np = m.np[q];
  const int nbx = (int)((np + 255) / 256);
  const int lb = b - m.blk[q];
  const int e = lb / nbx;
  const int64_t o = (int64_t)(lb - e * nbx) * 256 + threadIdx.x;
  if (o >= np) return;
  const int n1 = m.n1[q], axis = m.axis[q];
  const int u = (int)(o % n1) + 1, v = (int)(o / n1) + 1;
  int pc[3];
  const int a1 = axis == 0 ? 1 : 0, a2 = axis == 2 ? 1 : 2;
  pc[axis] = m.index[q];
  pc[a1] = u;
  pc[a2] = v;
  const int64_t c = pc[0] + px * pc[1] + pxy * pc[2];
  const int sel = (int)(m.sel[q] >> (8 * e)) & 0xff;
  m.dst[q][(int64_t)(sel >> 4) * np + o] = F(sel & 7)[c];
}

template <typename real>
__global__ __launch_bounds__(256) void k_monitors(FieldArgs<real> a, MonList<real> m) {
  mon_block(m, a.px, a.pxy, (int)blockIdx.x, [&](int c) -> const real* { return c < 3 ? a.e[c] : a.h[c - 3]; });
}

// ---------------------------------------------------------------------------
// Launches of the FUSED engine.  Each is a list of parts, every part a range
// of workgroups, none of which reads what another part of the launch writes:
// a launch of its own costs a part 4-9 us however little it does (the start
// of its first wavefronts and the drain of its last ones), which is most of
// the step on small grids.  Measured with the parts as launches of their own
// (profiling runs them so, that each has its time) and in two launches a
// step, the two-kernel form, us a step: 64^3 FP32 25.2 / 14.9, 96^3 FP32
// 40.0 / 28.4, 96^3 FP64 55.5 / 40.3, 150 x 137 x 211 FP32 periodic under a
// TFSF wave 103 / 84, 160^3 FP32 91 / 80.
struct Parts {
  int32_t mon, ade, mix, xf, plain, gen;  // blocks of each part (0: not in this launch)
  int32_t line;                           // 8: the incident line's block (before mon), 0: none
};

// The kernel arguments a cell update needs, loaded in one batch: left to the
// compiler, each is loaded where it is first used and waited for there, a
// chain of a dozen scalar loads before the first field load.  No instruction
// beyond the loads.  FP32 H, 160^3: 36.5 -> 35.0 us; the E update and FP64
// lose more to the registers it takes (160^3 E 48 -> 54 us).
template <typename real>
__device__ __forceinline__ void load_args(const FieldArgs<real>& a, const PmlArgs<real>& p) {
  asm volatile("" ::"s"(a.e[0]), "s"(a.e[1]), "s"(a.e[2]), "s"(a.h[0]), "s"(a.h[1]), "s"(a.h[2]), "s"(a.nx), "s"(a.ny),
               "s"(a.nz), "s"(a.px), "s"(a.pxy), "s"(p.P[0]), "s"(p.P[1]), "s"(p.P[2]), "s"(a.per[0]), "s"(a.per[1]),
               "s"(a.per[2]));
}

// Two-kernel step, E half: monitors of the step before (H), dispersive
// cells, rows that mix materials, and the rows with one material id (the
// table entry is then a wave-uniform scalar load).  A wavefront of the
// latter marches its 64 columns through KZ planes, carrying H of the plane
// below in registers (KZ = 1: one plane, nothing carried).
template <typename real, int KZ, bool LISTS>
__global__ __launch_bounds__(256) void k_step_e(FieldArgs<real> a, PmlArgs<real> p, SrcArgs<real> src, int nsrc,
                                                Parts pt, MonList<real> mon, AdeMulti ade, const int32_t* mix,
                                                SegGrid gm, SegGrid gt) {
  int b = (int)blockIdx.x;
  if constexpr (LISTS) {
    if (b < pt.mon) {
      mon_block(mon, a.px, a.pxy, b, [&](int c) -> const real* { return c < 3 ? a.e[c] : a.h[c - 3]; });
      return;
    }
    b -= pt.mon;
    if (b < round8(pt.ade)) {
      if (b < pt.ade) ade_block<real, true>(a, ade, src, nsrc, b);
      return;
    }
    b -= round8(pt.ade);
    if (b < pt.mix) {
      e_mixed_block(a, p, src, nsrc, mix, gm, b);
      return;
    }
    b -= pt.mix;
  }
  int tx, r;
  if (!seg_of(gt, b, a.xcdmap, tx, r)) return;
  const int i = tx * 64 + ((int)threadIdx.x & 63) + 1;
  const int tz = fast_quot(gt.ny, r), j = r - tz * gt.ny.d + 1;
  if (i > a.nx) return;
  e_column<real, KZ>(a, p, src, nsrc, i, j, tz, a.h[0], a.h[1], a.h[2], a.e[0], a.e[1], a.e[2]);
}

// ---------------------------------------------------------------------------
// TFSF incident line (sim1/program.f90:217-262, mod1/BERpmly_ExHz_mod.f90).
// One workgroup walks the line; the PML object's own fields pe, ph live on
// cells 1..npml and n-npml+1..n and hand over at the slab edges.
struct TfsfLine {
  double *e, *h, *pe, *ph;
  const double *f1, *f2, *g1, *g2;
  int32_t n, npml, src, lo, hi, comp, hc, axis, sg;
  double ck, ku;
};

// one workgroup: the line's E half step and its PML
__device__ __forceinline__ void tfsf_line_e(const TfsfLine& L, double g) {
  const int N = L.n, P = L.npml, hi = N - P + 1;
  for (int j = P + 1 + (int)threadIdx.x; j <= hi - 1; j += blockDim.x) {
    double v = L.e[j] + L.ck * (L.h[j] - L.h[j - 1]);
    if (j == L.src) v = v + g;
    L.e[j] = v;
  }
  if (P > 0) {
    for (int j = 1 + (int)threadIdx.x; j <= P; j += blockDim.x)
      L.pe[j] = L.f1[j] * L.pe[j] + L.f2[j] * (L.ph[j] - L.ph[j - 1]);
    for (int j = hi + (int)threadIdx.x; j <= N; j += blockDim.x)
      L.pe[j] = L.f1[j] * L.pe[j] + L.f2[j] * (L.ph[j] - L.ph[j - 1]);
    __syncthreads();
    if (threadIdx.x == 0) {
      L.pe[P + 1] = L.e[P + 1];
      L.e[P] = L.pe[P];
      L.pe[hi - 1] = L.e[hi - 1];
      L.e[hi] = L.pe[hi];
    }
  }
}

// Two-kernel step, H half: monitors of this step (E), every cell; with one
// TFSF the E half step of its incident line too (pt.line, the first block: the
// E launch read the line's H, k_tfsf_h reads its E): as a launch of its own it
// cost 4.8 us of the 85 us a step of 150 x 137 x 211 cells takes.
template <typename real, int KZ>
__global__ __launch_bounds__(256) void k_step_h(FieldArgs<real> a, PmlArgs<real> p, Parts pt, MonList<real> mon,
                                                SegGrid gt, TfsfLine line, double line_g) {
  int b = (int)blockIdx.x;
  if (b < pt.line) {
    if (b == 0) tfsf_line_e(line, line_g);
    return;
  }
  b -= pt.line;
  if (b < pt.mon) {
    mon_block(mon, a.px, a.pxy, b, [&](int c) -> const real* { return c < 3 ? a.e[c] : a.h[c - 3]; });
    return;
  }
  b -= pt.mon;
  if constexpr (sizeof(real) == 4) load_args(a, p);
  int tx, r;
  if (!seg_of(gt, b, a.xcdmap, tx, r)) return;
  const int i = tx * 64 + ((int)threadIdx.x & 63) + 1;
  const int tz = fast_quot(gt.ny, r), j = r - tz * gt.ny.d + 1;
  if (i > a.nx) return;
  h_column<real, KZ>(a, p, i, j, tz, a.e[0], a.e[1], a.e[2], a.h[0], a.h[1], a.h[2]);
}

// One-pass step: what reads the old copies and writes the new ones goes in
// two launches by the registers it needs: the x-face tiles and the plain
// tiles (the longest workgroups first), then the monitors of the step before,
// dispersive cells and E of the general cells; H of the general cells
// (k_gen_h) follows, since it reads E that other workgroups write.  NT: the
// marching tiles' stores nontemporal (streams_past_llc).
template <typename real, int R, bool PER, bool NT>
__global__ __launch_bounds__(256) void k_march(FieldArgs<real> a, MarchArgs<real> m, SrcArgs<real> src, int nsrc,
                                               Parts pt, TileList xf, TileList plain, XfArgs<real> x) {
  int b = (int)blockIdx.x;
  if (b < pt.xf) {
    if constexpr (kXface<real>) march_block<real, 2, true, PER, NT>(a, m, xf, src, nsrc, x, b);
    return;
  }
  b -= pt.xf;
  march_block<real, R, false, PER, NT>(a, m, plain, src, nsrc, x, b);
}

// a.h: the old H, a.e: the new E.  FP32 runs at eight wavefronts per SIMD
// (the compiler keeps some kernel arguments in vector registers to fit): the
// general cells wait on memory for most of their life.
template <typename real>
__global__ __launch_bounds__(256, sizeof(real) == 4 ? 8 : 4) void k_gen_e(
    FieldArgs<real> a, MarchArgs<real> m, PmlArgs<real> p, PmlArgs<real> pw, SrcArgs<real> src, int nsrc, Parts pt,
    MonList<real> mon, AdeMulti ade, TileList gen) {
  int b = (int)blockIdx.x;
  if (b < pt.mon) {
    mon_block(mon, a.px, a.pxy, b, [&](int c) -> const real* { return c < 3 ? m.eo[c] : m.ho[c - 3]; });
    return;
  }
  b -= pt.mon;
  if (b < round8(pt.ade)) {
    if (b < pt.ade) ade_block<real, true>(a, ade, src, nsrc, b);
    return;
  }
  gen_e_block(a, p, pw, m, gen, src, nsrc, b - round8(pt.ade));
}

// STAGED step, E half: monitors of the step before (H), the dispersive cells,
// the y slabs' split E (mix: their blocks), then D, sources and dielectric E
// of every row; H half: monitors (E), split H, H of the main rows.  A row's
// material entry is a scalar load where the row has one id.  The reference
// keeps these as seven loops; as launches of their own they cost the shipped
// case (125 x 1266 x 25, FP64) 174 us a step, D and E alone 52 + 36 us at 15
// words a cell where one pass moves 12; together 148 us.  NT: D, which nothing
// else of the step reads, marked nontemporal on grids past the memory-side
// cache (streams_past_llc), where E and H, 6 of the 9 arrays, then mostly stay
// in it: 126 us.
template <typename real, bool NT>
__global__ __launch_bounds__(256) void k_staged_e(FieldArgs<real> a, RefPmlArgs<real> rp, SrcArgs<real> src, int nsrc,
                                                  StagedRows rows, Parts pt, MonList<real> mon, AdeMulti ade,
                                                  SegGrid gs, SegGrid gt) {
  int b = (int)blockIdx.x;
  if (b < pt.mon) {
    mon_block(mon, a.px, a.pxy, b, [&](int c) -> const real* { return c < 3 ? a.e[c] : a.h[c - 3]; });
    return;
  }
  b -= pt.mon;
  if (b < round8(pt.ade)) {
    if (b < pt.ade) ade_block<real, false>(a, ade, src, nsrc, b, rows);
    return;
  }
  b -= round8(pt.ade);
  int tx, r;
  if (b < pt.mix) {
    if (!seg_of(gs, b, a.xcdmap, tx, r)) return;
    const int i = tx * 64 + ((int)threadIdx.x & 63) + 1, kz = fast_quot(gs.ny, r);
    if (i <= a.nx) ref_pml_e_cell(a, rp, i, r - kz * gs.ny.d, kz + 1);
    return;
  }
  if (!seg_of(gt, b - pt.mix, a.xcdmap, tx, r)) return;
  const int i = tx * 64 + ((int)threadIdx.x & 63) + 1, kz = fast_quot(gt.ny, r);
  const int j = r - kz * gt.ny.d + 1, k = kz + 1;
  if (i > a.nx) return;
  const int rm = a.rowmat[j + (a.ny + 2) * k];
  if (rm >= 0) {
    const uint32_t fl = a.flags[rm];
    bool any = rows.main(j) || (fl & 7u);
    for (int q = 0; q < nsrc; ++q) any |= src.axis[q] != 1 || src.index[q] == j;
    if (!any) return;  // a slab row that nothing here writes
    staged_e_cell<real, NT>(a, src, nsrc, rows, i, j, k, fl, a.gaxe[rm]);
  } else {
    const unsigned id = a.matid[i + a.px * j + a.pxy * k];
    staged_e_cell<real, NT>(a, src, nsrc, rows, i, j, k, a.flags[id], a.gaxe[id]);
  }
}

template <typename real>
__global__ __launch_bounds__(256) void k_staged_h(FieldArgs<real> a, RefPmlArgs<real> rp, StagedRows rows, Parts pt,
                                                  MonList<real> mon, SegGrid gs, SegGrid gt) {
  int b = (int)blockIdx.x;
  if (b < pt.mon) {
    mon_block(mon, a.px, a.pxy, b, [&](int c) -> const real* { return c < 3 ? a.e[c] : a.h[c - 3]; });
    return;
  }
  b -= pt.mon;
  int tx, r;
  if (b < pt.mix) {
    if (!seg_of(gs, b, a.xcdmap, tx, r)) return;
    const int i = tx * 64 + ((int)threadIdx.x & 63) + 1, kz = fast_quot(gs.ny, r);
    if (i <= a.nx) ref_pml_h_cell(a, rp, i, r - kz * gs.ny.d, kz + 1);
    return;
  }
  if (!seg_of(gt, b - pt.mix, a.xcdmap, tx, r)) return;
  const int i = tx * 64 + ((int)threadIdx.x & 63) + 1, kz = fast_quot(gt.ny, r);
  if (i <= a.nx) staged_h_cell(a, rp, rows, i, r - kz * gt.ny.d + rows.j0, kz + 1);
}

// x-face tiles of 4 rows (FDTD_XFACE_BY=4)
template <typename real, bool PER, bool NT>
__global__ __launch_bounds__(256) void k_xface4(FieldArgs<real> a, MarchArgs<real> m, SrcArgs<real> src, int nsrc,
                                                TileList xf, XfArgs<real> x) {
  march_block<real, 4, true, PER, NT>(a, m, xf, src, nsrc, x, (int)blockIdx.x);
}

// cos/sin table of one block of samples: tab[(b*nfreq + m)*2 + {0,1}]
__global__ void k_dft_table(const double* omega, int nfreq, int n_first, int count, double dt, double* tab) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= nfreq * count) return;
  const int b = q / nfreq, m = q - b * nfreq;
  const double t = (double)(n_first + b - 1) * dt;
  double sw, cw;
  sincos(omega[m] * t, &sw, &cw);
  tab[2 * q] = cw;
  tab[2 * q + 1] = sw;
}

// The fold of a block as a matrix product on the FP64 matrix cores:
// D[m][cell] = sum_b T[m][b] F[b][cell] for the cosine and the sine rows,
// then acc += dt * D.  A workgroup stages the table of up to 64
// frequencies (all the block's samples, cosine and sine side by side, rows
// padded against bank conflicts) in LDS once and then walks its share of
// the plane; each wavefront takes 16 cells of one component slot at a
// time, reads their samples, then streams them 4 at a time through 8 16x16
// tiles (4 of cosines, 4
// of sines; v_mfma_f64_16x16x4f64 on gfx950: A[i][k] comes from lane i +
// 16k, B[k][j] from lane j + 16k, and D[i][j] lands in lane j + 16 (i % 4),
// element i / 4).  The samples are not held in registers, so a block can
// be long: each flush reads and writes every accumulator once, so 64
// samples a block move half the accumulator bytes of 32.  The block's sum
// is in another order than a running sum (products fused, four samples at
// a time), a rounding difference the spectra carry at the 1e-16 level.
typedef double v4d __attribute__((ext_vector_type(4)));
constexpr int kDftTabRow = 65;  // double2 entries a sample row of the staged table (64 + 1 pad)
constexpr int kDftFoldGroups = 512;  // workgroups of a fold: two a CU

// One wavefront's share: 16 cells of a slot, NT tiles of 16 frequencies from
// m0.  Every load -- the block's samples, then the accumulators -- is issued
// before the first matrix instruction and without a branch: rows past the
// block's samples, cells past the plane and frequencies past the last are
// clamped to the last one (the table holds zeros for such samples; such cells
// and frequencies are not stored).  Loaded under those tests each sample had a
// wait of its own, and a tile's accumulators were not asked for until its sums
// were done: a fold of 384 x 384 cells, 4 components, 128 frequencies (2.4 GB
// read and written) 1000 us then, 638 us now; 150 x 137 cells, 32 frequencies
// 62 and 35 us; FP64 320 x 320, 64 frequencies 241 and 224 us.  32 frequencies
// a pass with three wavefronts a SIMD instead of two measured 692, 31 and 258.
template <typename real, int NT>
__device__ __forceinline__ void dft_fold_tile(const real* __restrict__ samp, const double2* lt, uint32_t np, int nslots,
                                              int slot, int64_t cell, int nfreq, int m0, int count, double dt,
                                              double* __restrict__ re, double* __restrict__ im, int jj, int kk) {
  const bool cin = cell < (int64_t)np;
  const int64_t cc = cin ? cell : (int64_t)np - 1;
  real f[kDftBlock / 4];  // this lane's samples: b = 4 st + kk
#pragma unroll
  for (int st = 0; st < kDftBlock / 4; ++st) {
    const int b = min(4 * st + kk, count - 1);
    f[st] = samp[(uint64_t)(uint32_t)(b * nslots + slot) * np + cc];
  }
  __builtin_amdgcn_sched_barrier(0);  // the samples first: the sums wait for them alone
  double ar[NT][4], ai[NT][4];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const uint64_t o = (uint64_t)(uint32_t)min(m0 + 16 * t + kk + 4 * v, nfreq - 1) * np + cc;
      ar[t][v] = re[o];
      ai[t][v] = im[o];
    }
  // the samples are in, the accumulators still under way: without this the
  // compiler moves each sample's load to the step below that uses it
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int st = 0; st < kDftBlock / 4; ++st) asm volatile("" : "+v"(f[st]));
  v4d dc[NT], ds[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) dc[t] = ds[t] = (v4d){0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int st = 0; st < kDftBlock / 4; ++st) {  // every lane: the matrix instructions need them all
    if (4 * st >= count) break;
    const double fv = (double)f[st];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const double2 cs = lt[(4 * st + kk) * kDftTabRow + 16 * t + jj];
      dc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(cs.x, fv, dc[t], 0, 0, 0);
      ds[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(cs.y, fv, ds[t], 0, 0, 0);
    }
  }
  if (!cin) return;
  asm volatile("" : "+v"(m0));  // the addresses again, not kept over the sums (registers)
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int m = m0 + 16 * t + kk + 4 * v;
      if (m >= nfreq) continue;
      const uint64_t o = (uint64_t)(uint32_t)m * np + cell;
      re[o] = ar[t][v] + dc[t][v] * dt;
      im[o] = ai[t][v] + ds[t][v] * dt;
    }
}

template <typename real>
__global__ __launch_bounds__(256, 2) void k_dft_accum(const real* __restrict__ samp, int64_t np, int nslots, int nfreq,
                                                   int count, const double* __restrict__ tab, double dt,
                                                   double* __restrict__ acc) {
  __shared__ double2 lt[kDftBlock * kDftTabRow];
  const int lane = (int)threadIdx.x & 63, w = (int)threadIdx.x >> 6;
  const int jj = lane & 15, kk = lane >> 4;
  const int64_t ntile = (np + 15) / 16, nwt = ntile * nslots;
  for (int m0 = 0; m0 < nfreq; m0 += 64) {
    __syncthreads();
    for (int q = (int)threadIdx.x; q < kDftBlock * 64; q += 256) {
      const int b = q >> 6, mm = q & 63;
      double2 v = {0.0, 0.0};
      if (b < count && m0 + mm < nfreq) v = *(const double2*)(tab + 2 * ((int64_t)b * nfreq + m0 + mm));
      lt[b * kDftTabRow + mm] = v;
    }
    __syncthreads();
    // wave tiles of 16 cells of one slot, strided over the grid (the loop
    // count is uniform per wavefront; no barrier inside)
    const int nt = (min(64, nfreq - m0) + 15) / 16;
    for (int64_t wt = (int64_t)blockIdx.x * 4 + w; wt < nwt; wt += (int64_t)gridDim.x * 4) {
      const int slot = (int)(wt / ntile);
      const int64_t cell = (wt - (int64_t)slot * ntile) * 16 + jj;
      double* re = acc + (int64_t)slot * 2 * nfreq * np;
      double* im = re + (int64_t)nfreq * np;
      auto go = [&](auto n) {
        dft_fold_tile<real, decltype(n)::value>(samp, lt, (uint32_t)np, nslots, slot, cell, nfreq, m0, count, dt, re,
                                                im, jj, kk);
      };
      if (nt == 4)
        go(std::integral_constant<int, 4>{});
      else if (nt == 3)
        go(std::integral_constant<int, 3>{});
      else if (nt == 2)
        go(std::integral_constant<int, 2>{});
      else
        go(std::integral_constant<int, 1>{});
    }
  }
}

inline TfsfLine tfsf_line(const Sim* s, const Tfsf& t) {
  TfsfLine L;
  const int64_t m = t.n + 2;
  L.e = t.d_line;
  L.h = t.d_line + m;
  L.pe = t.d_line + 2 * m;
  L.ph = t.d_line + 3 * m;
  L.f1 = t.d_line + 4 * m;
  L.f2 = t.d_line + 5 * m;
  L.g1 = t.d_line + 6 * m;
  L.g2 = t.d_line + 7 * m;
  L.n = t.n;
  L.npml = t.p.npml;
  L.src = t.p.src_index;
  L.lo = t.p.lo;
  L.hi = t.p.hi;
  L.comp = t.p.comp;
  L.hc = t.hc;
  L.axis = t.p.axis;
  L.sg = t.sg;
  L.ck = s->ku * (1.0 / t.p.eps);
  L.ku = s->ku;
  return L;
}

// E half step of the line: ex_inc update (:222-224), the pulse (:228-229),
// mypmly_inc%updateE (:231; updateE_pmy_low/high + setboundaryEa/Eb)
__global__ __launch_bounds__(256) void k_tfsf_line_e(TfsfLine L, double g) { tfsf_line_e(L, g); }

// H half step of the TFSF: block 0 advances the line (hz_inc update :252-254,
// mypmly_inc%updateH :255) and records its probes; the other blocks apply
// the consistency terms on H (:260-262 and, two-sided, the far plane):
// H_h(lo-1) -= s*Ku*e(lo), H_h(hi) += s*Ku*e(hi+1).  ALL_FACES PML cells on
// a plane take the term into the split along the line's axis.
template <typename real>
__global__ __launch_bounds__(256) void k_tfsf_h(FieldArgs<real> a, PmlArgs<real> p, int all_faces, TfsfLine L,
                                                const int32_t* lp, int nlp, double* rec, double tn, int n1, int n2) {
  if (blockIdx.x == 0) {
    const int N = L.n, P = L.npml, hi = N - P + 1;
    for (int j = P + 1 + (int)threadIdx.x; j <= hi - 1; j += blockDim.x) L.h[j] = L.h[j] + L.ku * (L.e[j + 1] - L.e[j]);
    if (P > 0) {
      for (int j = 1 + (int)threadIdx.x; j <= P; j += blockDim.x)
        L.ph[j] = L.g1[j] * L.ph[j] + L.g2[j] * (L.pe[j + 1] - L.pe[j]);
      for (int j = hi + (int)threadIdx.x; j <= N; j += blockDim.x)
        L.ph[j] = L.g1[j] * L.ph[j] + L.g2[j] * (L.pe[j + 1] - L.pe[j]);
      __syncthreads();
      if (threadIdx.x == 0) {
        L.ph[P + 1] = L.h[P + 1];
        L.h[P] = L.ph[P];
        L.ph[hi - 1] = L.h[hi - 1];
        L.h[hi] = L.ph[hi];
      }
    }
    __syncthreads();
    if ((int)threadIdx.x < nlp) {  // sim1/program.f90:272-273
      double* r = rec + 7 * lp[2 * threadIdx.x];
      const int j = lp[2 * threadIdx.x + 1];
      r[0] = tn;
      for (int q = 1; q < 7; ++q) r[q] = 0.0;
      r[1 + L.comp] = L.e[j];
      r[4 + L.hc] = L.sg * L.h[j];
    }
    return;
  }
  const int64_t u = (int64_t)(blockIdx.x - 1) * blockDim.x + threadIdx.x;
  const int64_t np = (int64_t)n1 * n2;
  const int nplanes = L.hi > 0 ? 2 : 1;
  if (u >= np * nplanes) return;
  const int pl = (int)(u / np);
  const int64_t w = u - (int64_t)pl * np;
  const int index = pl == 0 ? L.lo - 1 : L.hi;
  const double ev = pl == 0 ? L.e[L.lo] : L.e[L.hi + 1];
  const double val = (pl == 0 ? -(L.sg * L.ku) : (L.sg * L.ku)) * ev;
  const int a1 = L.axis == 0 ? 1 : 0, a2 = L.axis == 2 ? 1 : 2;
  int c3[3];
  c3[L.axis] = index;
  c3[a1] = (int)(w % n1) + 1;
  c3[a2] = (int)(w / n1) + 1;
  const int i = c3[0], j = c3[1], k = c3[2];
  const int c = i + a.px * j + a.pxy * k;
  const int q = L.hc;
  real hv;
  if (all_faces && in_pml(p.P, i, j, k, a.nx, a.ny, a.nz)) {
    // the part of H_q along the axis takes the value; with both parts of
    // H_q stored, H_q = the two summed as h_cell_store sums them (Hxy+Hxz,
    // Hyz+Hyx, Hzx+Hzy), otherwise H_q takes the value itself (a part not
    // stored is H_q less the other part)
    const int sa = q == 0 ? (L.axis == 1 ? S_HXY : S_HXZ)
                          : (q == 1 ? (L.axis == 0 ? S_HYX : S_HYZ) : (L.axis == 0 ? S_HZX : S_HZY));
    const int s0 = q == 0 ? S_HXY : (q == 1 ? S_HYZ : S_HZX);
    const int s1 = q == 0 ? S_HXZ : (q == 1 ? S_HYX : S_HZY);
    const bool st[3] = {in_slab(p.P[0], i, a.nx), in_slab(p.P[1], j, a.ny), in_slab(p.P[2], k, a.nz)};
    const bool both = st[q == 0 ? 1 : 0] && st[q == 2 ? 1 : 2];
    const int sp = pml_index(p.P, i, j, k, a.nx, a.ny, a.nz);
    if (st[L.axis]) p.s[sa][sp] = p.s[sa][sp] + (real)val;
    hv = both ? p.s[s0][sp] + p.s[s1][sp] : a.h[q][c] + (real)val;
  } else {
    hv = a.h[q][c] + (real)val;
  }
  a.h[q][c] = hv;
  put_h_ghost(a.h[q], hv, i, j, k, c, a);
}

// Flux of a DFT plane, one block per frequency, fixed-order tree reduction.
__global__ __launch_bounds__(256) void k_flux(const double* acc, int64_t np, int nfreq, int shA, int seA, int shB,
                                              int seB, double ds, double* S) {
  __shared__ double red[256];
  const int m = blockIdx.x;
  auto re = [&](int slot) { return acc + (int64_t)slot * 2 * nfreq * np + (int64_t)m * np; };
  auto im = [&](int slot) { return acc + (int64_t)slot * 2 * nfreq * np + (int64_t)nfreq * np + (int64_t)m * np; };
  const double *rhA = re(shA), *ihA = im(shA), *reA = re(seA), *ieA = im(seA);
  const double *rhB = re(shB), *ihB = im(shB), *reB = re(seB), *ieB = im(seB);
  double acc_l = 0.0;
  for (int64_t o = threadIdx.x; o < np; o += blockDim.x)
    acc_l += ((rhA[o] * reA[o]) + (ihA[o] * ieA[o]) - (rhB[o] * reB[o]) - (ihB[o] * ieB[o])) * ds;
  red[threadIdx.x] = acc_l;
  __syncthreads();
  for (int w = blockDim.x / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) S[m] = red[0];
}

// Served-job sentinel: flag = 1 when any of the six field arrays holds a
// NaN or Inf (ghosts and padding are zero).  Lanes that find one store 1
// (the same value, so the race is harmless); the flag is never cleared.
template <typename real>
__global__ __launch_bounds__(256) void k_nonfinite(const real* e0, const real* e1, const real* e2, const real* h0,
                                                   const real* h1, const real* h2, int64_t n, int* flag) {
  const real* f[6] = {e0, e1, e2, h0, h1, h2};
  bool bad = false;
  for (int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; c < n; c += (int64_t)gridDim.x * blockDim.x)
#pragma unroll
    for (int q = 0; q < 6; ++q) bad |= !isfinite(f[q][c]);
  if (bad) flag[0] = 1;
}

// Energy sums over interior cells; one partial pair per block.
template <typename real>
__global__ __launch_bounds__(256) void k_energy(FieldArgs<real> a, double* part) {
  __shared__ double r1[256], r2[256];
  const int64_t n = (int64_t)a.nx * a.ny * a.nz;
  double s1 = 0, s2 = 0;
  for (int64_t o = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; o < n; o += (int64_t)gridDim.x * blockDim.x) {
    const int i = (int)(o % a.nx) + 1;
    const int64_t r = o / a.nx;
    const int j = (int)(r % a.ny) + 1, k = (int)(r / a.ny) + 1;
    const int64_t c = i + a.px * j + a.pxy * k;
    const double ex = a.e[0][c], ey = a.e[1][c], ez = a.e[2][c];
    const double hx = a.h[0][c], hy = a.h[1][c], hz = a.h[2][c];
    s1 += (double)a.gaxe[a.matid[c]].v[3] * (ex * ex + ey * ey + ez * ez);
    s2 += hx * hx + hy * hy + hz * hz;
  }
  r1[threadIdx.x] = s1;
  r2[threadIdx.x] = s2;
  __syncthreads();
  for (int w = blockDim.x / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) {
      r1[threadIdx.x] += r1[threadIdx.x + w];
      r2[threadIdx.x] += r2[threadIdx.x + w];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = r1[0];
    part[2 * blockIdx.x + 1] = r2[0];
  }
}

// periodic ghost refresh of one component after a host write
template <typename real>
__global__ void k_ghosts(FieldArgs<real> a, real* f, int axis) {
  const int n[3] = {a.nx, a.ny, a.nz};
  const int a1 = axis == 0 ? 1 : 0, a2 = axis == 2 ? 1 : 2;
  const int u = blockIdx.x * blockDim.x + threadIdx.x;
  const int v = blockIdx.y;
  if (u > n[a1] + 1) return;
  int p[3];
  p[a1] = u;
  p[a2] = v;
  const int64_t st[3] = {1, a.px, a.pxy};
  p[axis] = 0;
  const int64_t c0 = p[0] + a.px * p[1] + a.pxy * p[2];
  f[c0 + st[axis] * (n[axis] + 1)] = f[c0 + st[axis] * 1];
  f[c0] = f[c0 + st[axis] * n[axis]];
}

// ---------------------------------------------------------------------------
// host-side launchers
namespace {

template <typename real>
FieldArgs<real> field_args(Sim* s) {
  FieldArgs<real> a{};
  for (int q = 0; q < 3; ++q) {
    a.e[q] = (real*)s->E[q];
    a.h[q] = (real*)s->H[q];
    a.d[q] = (real*)s->D[q];
  }
  a.matid = s->d_matid;
  const size_t nt = (size_t)s->ntab;
  a.coef = (const Vec4<real>*)s->d_mattab;
  a.gaxe = a.coef + nt;
  a.flags = (const uint32_t*)(a.gaxe + nt);
  a.rowmat = s->d_rowmat;
  a.nx = s->nx;
  a.ny = s->ny;
  a.nz = s->nz;
  for (int q = 0; q < 3; ++q) a.per[q] = s->g.periodic[q] ? 1 : 0;
  a.px = (int32_t)s->px;
  a.pxy = (int32_t)s->pxy;
  a.by_px = fast_div(a.px);
  a.by_pxy = fast_div(a.pxy);
  a.ku = (real)s->ku;
  a.xcdmap = s->xcdmap;
  return a;
}

template <typename real>
PmlArgs<real> pml_args(Sim* s) {
  PmlArgs<real> p{};
  for (int q = 0; q < 3; ++q) p.P[q] = s->P[q];
  for (int q = 0; q < S_N; ++q) p.s[q] = s->d_split ? (real*)s->d_split + (int64_t)q * s->npml_cells : nullptr;
  p.kup = (real)s->ku_pml;
  if (s->d_prof) {
    const real* base = (const real*)s->d_prof;
    int64_t off = 0;
    const int n[3] = {s->nx, s->ny, s->nz};
    for (int ax = 0; ax < 3; ++ax) {
      p.f1[ax] = base + off; off += n[ax] + 2;
      p.f2[ax] = base + off; off += n[ax] + 2;
      p.g1[ax] = base + off; off += n[ax] + 2;
      p.g2[ax] = base + off; off += n[ax] + 2;
    }
  }
  return p;
}

template <typename real>
RefPmlArgs<real> ref_pml_args(Sim* s) {
  RefPmlArgs<real> p{};
  p.P = s->pml.npml[1];
  p.jb = s->ny - p.P + 1;
  p.sx = s->nx + 2;
  p.sxy = (int64_t)(s->nx + 2) * (p.P + 2);
  for (int sl = 0; sl < 2; ++sl) {
    for (int q = 0; q < S_N; ++q) p.s[sl][q] = (real*)s->d_slab + ((int64_t)sl * S_N + q) * s->slab_cells;
    p.prof[sl] = (const real*)s->d_ref_prof + (int64_t)sl * 12 * s->ref_prof_stride;
  }
  p.ps = s->ref_prof_stride;
  return p;
}

struct Timer {
  Sim* s;
  int kid;
  hipEvent_t a = nullptr, b = nullptr;
  Timer(Sim* s_, int kid_) : s(s_), kid(kid_) {
    if (!s->profiling) return;
    a = get();
    if (a && hipEventRecord(a, s->stream) != hipSuccess) a = nullptr;
  }
  hipEvent_t get() {
    if (!s->event_pool.empty()) {
      hipEvent_t e = s->event_pool.back();
      s->event_pool.pop_back();
      return e;
    }
    hipEvent_t e = nullptr;
    if (hipEventCreate(&e) != hipSuccess) return nullptr;
    return e;
  }
  ~Timer() {
    if (!s->profiling || !a) return;
    b = get();
    if (!b || hipEventRecord(b, s->stream) != hipSuccess) return;
    s->pending.push_back({kid, {a, b}});
  }
};

// FP32: from this many workgroups of plain rows on, the lists of a two-kernel
// E launch have a launch of their own.  Beside them the rows' kernel holds the
// registers of the dispersive update (seven wavefronts a SIMD instead of
// eight), which costs more than a launch once the rows fill the GPU many
// times over.  In FP64 the rows alone hold as many (four wavefronts either
// way), and one launch is the better at every size.  Cubes with a gold sphere,
// one launch against two, us a step: FP32 96 cells a side 27.2 / 33.1, 128: 46.2
// / 50.2, 160: 87.0 / 88.3, 203: 229 / 224, 256: 401 / 389, 320: 747 / 725; FP64
// 96: 43.0 / 48.7, 160: 193 / 197, 203: 403 / 410, 256: 693 / 701, 320: 1320 /
// 1327.
constexpr int kListsApart = 32768;

// the segment grid of `rows` rows of nx cells (SegGrid) and its blocks
inline SegGrid seg_grid(int nx, int ny, int64_t rows, int* blocks) {
  SegGrid g;
  g.ntx = fast_div((nx + 63) / 64);
  g.ny = fast_div(ny);
  g.n = (int32_t)(g.ntx.d * rows);
  const int nb = (g.n + 3) / 4;  // four wavefronts a workgroup
  g.tper = (nb + 7) / 8;
  *blocks = 8 * g.tper;
  return g;
}

// ---- monitors ----------------------------------------------------------------
// What is still to be sampled of the last step made: its DFT planes (the
// components `sel` names) and its probes.
template <typename real>
void mon_add(MonList<real>& m, const MonPend& q) {
  const int n = m.nplanes++;
  m.axis[n] = q.axis;
  m.index[n] = q.index;
  m.n1[n] = q.n1;
  m.np[n] = q.np;
  m.sel[n] = q.sel;
  m.dst[n] = (real*)q.dst;
  m.blk[n + 1] = m.blk[n] + (int32_t)((q.np + 255) / 256) * q.nsel;
}
template <typename real>
void mon_probes(Sim* s, MonList<real>& m, double* out, double tn, int part) {
  m.nprobe = (int)s->probes.size();
  m.ppos = (const int32_t*)s->d_probe_pos;
  m.pout = out;
  m.tn = tn;
  m.part = part;
}
template <typename real>
void mon_close(MonList<real>& m) {
  m.nblk = m.blk[m.nplanes] + (m.nprobe > 0 ? (m.nprobe + 255) / 256 : 0);
}

template <typename real>
void launch_monitors(Sim* s, MonList<real>& m) {
  mon_close(m);
  if (!m.nblk) return;
  Timer tm(s, FDTD_K_MON);
  hipLaunchKernelGGL(k_monitors<real>, dim3((unsigned)m.nblk), dim3(256), 0, s->stream, field_args<real>(s), m);
}

// The pending samples as a list a launch can take along; the planes that do
// not fit the list are sampled by launches of their own.
template <typename real>
MonList<real> take_pending(Sim* s) {
  MonList<real> m{};
  size_t q = 0;
  for (; s->mon_pend.size() - q > (size_t)kMonPlanes;) {
    MonList<real> o{};
    for (int e = 0; e < kMonPlanes; ++e) mon_add(o, s->mon_pend[q++]);
    launch_monitors(s, o);
  }
  for (; q < s->mon_pend.size(); ++q) mon_add(m, s->mon_pend[q]);
  if (s->probe_part) mon_probes(s, m, s->probe_out, s->probe_tn, s->probe_part);
  s->mon_pend.clear();
  s->probe_part = 0;
  mon_close(m);
  return m;
}

template <typename real>
void flush_pending(Sim* s) {
  MonList<real> m = take_pending<real>(s);
  launch_monitors(s, m);
}

template <typename real>
SrcArgs<real> source_args(Sim* s, int n, int* nsrc) {
  SrcArgs<real> sa{};
  sa.n = n;
  const double t = (double)(n - 1) * s->dt;
  int q = 0;
  for (const auto& src : s->srcs) {
    const fdtd_pulse& p = src.p;
    // sim3/program.f90:400
    const double g = p.amplitude * (std::exp(-0.5 * ((t - p.t0) / p.st) * ((t - p.t0) / p.st)) * std::sin(p.w0 * t));
    sa.axis[q] = src.axis;
    sa.index[q] = src.index;
    sa.comp[q] = src.comp;
    sa.val[q] = (real)g;
    sa.dval[q] = nullptr;
    ++q;
  }
  // TFSF consistency terms on D, sim1/program.f90:236-238: D(lo) -= Ku*h(lo-1)
  // and, two-sided, D(hi+1) += Ku*h(hi), h read from the line on the device
  for (const auto& t : s->tfsfs) {
    const double* h = t.d_line + (t.n + 2);
    sa.axis[q] = t.p.axis;
    sa.index[q] = t.p.lo;
    sa.comp[q] = t.p.comp;
    sa.val[q] = 0;
    sa.dval[q] = h + (t.p.lo - 1);
    sa.dscale[q] = -s->ku;
    ++q;
    if (t.p.hi > 0) {
      sa.axis[q] = t.p.axis;
      sa.index[q] = t.p.hi + 1;
      sa.comp[q] = t.p.comp;
      sa.val[q] = 0;
      sa.dval[q] = h + t.p.hi;
      sa.dscale[q] = s->ku;
      ++q;
    }
  }
  *nsrc = q;
  return sa;
}

template <typename real>
void dft_flush_plane(Sim* s, DftPlane& d) {
  if (d.nbuf == 0) return;
  flush_pending<real>(s);
  const int64_t np = (int64_t)d.n1 * d.n2;
  Timer tm(s, FDTD_K_MON);
  const int nt = d.nfreq * d.nbuf;
  hipLaunchKernelGGL(k_dft_table, dim3((unsigned)((nt + 255) / 256)), dim3(256), 0, s->stream, d.d_omega, d.nfreq,
                     d.n_first, d.nbuf, s->dt, d.d_tab);
  // two workgroups a CU (the staged table is 65 KB of LDS), each walking
  // wave tiles of 16 cells of one slot
  const int64_t wgs = ((np + 15) / 16 * d.nslots + 3) / 4;
  hipLaunchKernelGGL(k_dft_accum<real>, dim3((unsigned)std::min<int64_t>(wgs, kDftFoldGroups)), dim3(256), 0,
                     s->stream, (const real*)d.d_samp, np, d.nslots, d.nfreq, d.nbuf, d.d_tab, s->dt, d.d_acc);
  d.nbuf = 0;
}

template <typename real>
int step_impl(Sim* s) {
  const int n = s->n_done + 1;
  FieldArgs<real> a = field_args<real>(s);
  int nsrc = 0;
  SrcArgs<real> src = source_args<real>(s, n, &nsrc);
  if (s->dry) nsrc = 0;
  hipStream_t st = s->stream;
  auto ade_coef = [&](const AdeGroup& g) {  // FP64 in both precisions
    AdeCoef<double> c = g.coef;
    c.ku = s->ku;
    return c;
  };
  auto lord_coef = [&](const AdeGroup& g) {
    LordCoef c = g.ld;
    c.ku = s->ku;
    return c;
  };

  const bool refy = s->pml_mode == FDTD_PML_REF_Y;
  const int Py = refy ? s->pml.npml[1] : 0;
  const StagedRows rows{1 + Py, s->ny - Py, refy ? Py : 0, refy ? s->ny - Py + 1 : 0};
  // the Drude/CP/Raman groups, kAdeMulti at a time: the first list goes with
  // an E launch (their blocks in *blocks), the others have launches of their own
  auto ade_lists = [&](const FieldArgs<real>& af, int* blocks) {
    AdeMulti first{}, g{};
    bool have = false;
    auto done = [&]() {
      if (!g.ng) return;
      if (!have) {
        first = g;
        have = true;
      } else {
        Timer tm(s, FDTD_K_ADE);
        if (s->engine == FDTD_ENGINE_FUSED)
          hipLaunchKernelGGL((k_ade_multi<real, true>), dim3((unsigned)g.blk[g.ng]), dim3(256), 0, st, af, g, src, nsrc,
                             rows);
        else
          hipLaunchKernelGGL((k_ade_multi<real, false>), dim3((unsigned)g.blk[g.ng]), dim3(256), 0, st, af, g, src,
                             nsrc, rows);
      }
      g = AdeMulti{};
    };
    for (auto& G : s->groups) {
      if (G.kind != 0 || !G.ncells) continue;
      const int q = g.ng++;
      g.co[q] = ade_coef(G);
      g.cells[q] = G.d_cells;
      g.masks[q] = G.d_mask;
      g.state[q] = (double*)G.d_state;
      g.n[q] = G.ncells;
      g.blk[q + 1] = g.blk[q] + (int32_t)((G.ncells + 255) / 256);
      if (g.ng == kAdeMulti) done();
    }
    done();
    *blocks = first.blk[first.ng];
    return first;
  };

  // TFSF lines: E half step after the main E stage (the D terms above read
  // h(lo-1) before this step's line H update); H half step, consistency
  // terms on H and the line probes after the main H stage
  auto line_pulse = [&](const fdtd_pulse& pu) {
    const double tt = (double)(n - 1) * s->dt;
    return pu.amplitude * (std::exp(-0.5 * ((tt - pu.t0) / pu.st) * ((tt - pu.t0) / pu.st)) * std::sin(pu.w0 * tt));
  };
  auto tfsf_e = [&](hipStream_t sq) {
    if (s->dry) return;
    for (const auto& t : s->tfsfs) {
      Timer tm(s, FDTD_K_MAT);
      hipLaunchKernelGGL(k_tfsf_line_e, dim3(1), dim3(256), 0, sq, tfsf_line(s, t), line_pulse(t.p.pulse));
    }
  };
  auto tfsf_h = [&](hipStream_t sq, PmlArgs<real> pa, int all_faces) {
    if (s->dry) return;
    const int np = (int)s->probes.size();
    double* row = np ? s->d_probe + (int64_t)7 * np * (s->probe_row0 + (n - 1 - s->call_base)) : nullptr;
    for (const auto& t : s->tfsfs) {
      const int ax = t.p.axis;
      const int nn[3] = {s->nx, s->ny, s->nz};
      const int n1 = nn[ax == 0 ? 1 : 0], n2 = nn[ax == 2 ? 1 : 2];
      const int64_t cells = (int64_t)n1 * n2 * (t.p.hi > 0 ? 2 : 1);
      Timer tm(s, FDTD_K_MAT);
      hipLaunchKernelGGL((k_tfsf_h<real>), dim3((unsigned)(1 + (cells + 255) / 256)), dim3(256), 0, sq, a, pa,
                         all_faces, tfsf_line(s, t), (const int32_t*)t.d_lp, row ? t.nlp : 0, row,
                         (double)n * s->dt, n1, n2);
    }
  };
  // this step's samples: the planes open at step n with their ring slots
  // (dry steps write them too, into the slot the next real step overwrites);
  // comps bit c selects component c
  auto sample = [&](int comps, auto&& take) {
    for (auto& d : s->dfts) {
      if (n < d.n_begin || (d.n_end > 0 && n > d.n_end)) continue;
      MonPend q{};
      int slot = 0;
      for (int c = 0; c < 6; ++c) {
        if (!(d.mask & (1 << c))) continue;
        if (comps & (1 << c)) q.sel |= (uint64_t)(c | slot << 4) << (8 * q.nsel++);
        ++slot;
      }
      if (!q.nsel) continue;
      q.axis = d.axis;
      q.index = d.index;
      q.n1 = d.n1;
      q.np = (int64_t)d.n1 * d.n2;
      q.dst = (real*)d.d_samp + (int64_t)d.nbuf * slot * q.np;
      take(q);
    }
  };
  const bool probes_on = !s->probes.empty() && !s->dry;
  double* probe_row =
      probes_on ? s->d_probe + (int64_t)7 * (int64_t)s->probes.size() * (s->probe_row0 + (n - 1 - s->call_base)) : nullptr;
  auto pend = [&](int comps, int part) {  // left to the next step's first launch, or the end of the call
    sample(comps, [&](const MonPend& q) { s->mon_pend.push_back(q); });
    if (probes_on) {
      s->probe_part = part;
      s->probe_out = probe_row;
      s->probe_tn = (double)n * s->dt;
    }
  };
  // profiling: every part a launch of its own, timed; FDTD_DFT_FUSE=0: the
  // monitors alone
  const bool apart = s->profiling, mon_apart = apart || !s->dft_fuse;
  // in the H launch E is final and H is not: it samples E, the next step's
  // first launch H
  auto e_samples = [&]() {
    MonList<real> mon{};
    if (mon_apart) return mon;
    sample(7, [&](const MonPend& q) {
      if (mon.nplanes == kMonPlanes) {
        launch_monitors(s, mon);
        mon = MonList<real>{};
      }
      mon_add(mon, q);
    });
    if (probes_on) mon_probes(s, mon, probe_row, (double)n * s->dt, 1);
    mon_close(mon);
    return mon;
  };
  if (s->engine == FDTD_ENGINE_FUSED && s->onepass) {
    // new fields go to the second copies, then the copies swap roles
    FieldArgs<real> an = a;
    for (int q = 0; q < 3; ++q) {
      an.e[q] = (real*)s->E2[q];
      an.h[q] = (real*)s->H2[q];
    }
    FieldArgs<real> ae = an;  // E of dispersive and general cells: the old H in, the new E out
    for (int q = 0; q < 3; ++q) ae.h[q] = a.h[q];
    for (auto& g : s->groups) {
      if (g.kind != 2 || !g.ncells) continue;
      Timer tm(s, FDTD_K_ADE);
      hipLaunchKernelGGL((k_lord<real, true>), dim3((unsigned)((g.ncells + 255) / 256)), dim3(256), 0, st, ae,
                         lord_coef(g), g.d_cells, g.d_mask, (double*)g.d_state, g.ncells, src, nsrc);
    }
    {
      int rc = build_march_tiles(s, s->op_by, s->op_kc);
      if (rc) return rc;
    }
    PmlArgs<real> p = pml_args<real>(s);  // old splits
    PmlArgs<real> pw = p;                 // new splits
    for (int q = 0; q < S_N; ++q)
      pw.s[q] = s->d_split2 ? (real*)s->d_split2 + (int64_t)q * s->npml_cells : nullptr;
    MarchArgs<real> m{};
    for (int q = 0; q < 3; ++q) {
      m.eo[q] = a.e[q];
      m.ho[q] = a.h[q];
    }
    const int R = s->op_by;
    const bool per = a.per[0] || a.per[1] || a.per[2];
    // x-face tiles: the split parts of the x slabs, old (p) and new (pw),
    // and the x profiles
    XfArgs<real> xa{};
    if (s->n_tl_xf) {
      const int Px = p.P[0], Py = p.P[1], Pz = p.P[2];
      xa.eo[0] = p.s[S_EYX];
      xa.eo[1] = p.s[S_EZX];
      xa.ho[0] = p.s[S_HYX];
      xa.ho[1] = p.s[S_HZX];
      xa.en[0] = pw.s[S_EYX];
      xa.en[1] = pw.s[S_EZX];
      xa.hn[0] = pw.s[S_HYX];
      xa.hn[1] = pw.s[S_HZX];
      xa.f1 = p.f1[0];
      xa.f2 = p.f2[0];
      xa.g1 = p.g1[0];
      xa.g2 = p.g2[0];
      xa.kup = p.kup;
      xa.Px = Px;
      xa.Py = Py;
      xa.Pz = Pz;
      xa.nym = s->ny - 2 * Py;
      xa.nzm = s->nz - 2 * Pz;
      xa.base = 2 * Pz * s->nx * s->ny + (s->nz - 2 * Pz) * 2 * Py * s->nx;
      xa.hioff = (s->nz - 2 * Pz) * xa.nym * Px;
    }
    // four wavefronts (tiles) a workgroup
    auto tile_list = [&](const int32_t* tiles, int ntl, int per_block, int nsplit, int* blocks) {
      TileList t{tiles, ntl, 0, nsplit};
      const int nb = (ntl * nsplit + per_block - 1) / per_block;
      t.tper = (nb + 7) / 8;
      *blocks = 8 * t.tper;
      return t;
    };
    Parts all{};
    const TileList tp = tile_list(s->d_tl_plain, s->n_tl_plain, 4, 1, &all.plain);
    TileList tx = tile_list(s->d_tl_plain + 8 * (int64_t)s->n_tl_plain, s->n_tl_xf, 4, 1, &all.xf);
    const TileList te = tile_list(s->d_tl_gen, s->n_tl_gen, 1, s->tl_gkc, &all.gen);  // a workgroup per plane
    const AdeMulti ade = ade_lists(ae, &all.ade);
    MonList<real> mon{};
    if (!apart) mon = take_pending<real>(s);
    all.mon = round8(mon.nblk);
    auto march = [&](const Parts& pt) {
      const int nb = pt.xf + pt.plain;
      if (!nb) return;
      auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3((unsigned)nb), dim3(256), 0, st, an, m, src, nsrc, pt, tx, tp, xa);
      };
      auto by_rows = [&](auto prd, auto nt) {
        constexpr bool PER = decltype(prd)::value, NT = decltype(nt)::value;
        if (R == 2)
          go(k_march<real, 2, PER, NT>);
        else if (R == 4)
          go(k_march<real, 4, PER, NT>);
        else if constexpr (sizeof(real) == 4)  // FP64 tiles stop at 4 rows (8 would spill)
          go(k_march<real, 8, PER, NT>);
      };
      auto by_store = [&](auto prd) {
        s->nt_march ? by_rows(prd, std::true_type{}) : by_rows(prd, std::false_type{});
      };
      per ? by_store(std::true_type{}) : by_store(std::false_type{});
    };
    auto gen_e = [&](const Parts& pt) {
      const int nb = pt.mon + round8(pt.ade) + pt.gen;
      if (nb)
        hipLaunchKernelGGL(k_gen_e<real>, dim3((unsigned)nb), dim3(256), 0, st, ae, m, p, pw, src, nsrc, pt, mon,
                           ade, te);
    };
    auto launch_xf4 = [&]() {
      if constexpr (kXface<real>) {
        auto go = [&](auto kern) {
          hipLaunchKernelGGL(kern, dim3((unsigned)all.xf), dim3(256), 0, st, an, m, src, nsrc, tx, xa);
        };
        if (s->nt_march)
          per ? go(k_xface4<real, true, true>) : go(k_xface4<real, false, true>);
        else
          per ? go(k_xface4<real, true, false>) : go(k_xface4<real, false, false>);
      }
    };
    const bool xf4 = s->n_tl_xf && s->tl_bx == 4;
    if (apart) {
      if (all.ade) {
        Timer tm(s, FDTD_K_ADE);
        gen_e(Parts{0, all.ade, 0, 0, 0, 0});
      }
      if (s->n_tl_plain) {
        Timer tm(s, FDTD_K_E);
        march(Parts{0, 0, 0, 0, all.plain, 0});
      }
      if (s->n_tl_xf) {
        Timer tm(s, FDTD_K_XF);
        xf4 ? launch_xf4() : march(Parts{0, 0, 0, all.xf, 0, 0});
      }
      if (s->n_tl_gen) {
        Timer tm(s, FDTD_K_GEN_E);
        gen_e(Parts{0, 0, 0, 0, 0, all.gen});
      }
    } else {
      if (xf4) launch_xf4();
      march(Parts{0, 0, 0, xf4 ? 0 : all.xf, all.plain, 0});
      gen_e(Parts{all.mon, all.ade, 0, 0, 0, all.gen});
    }
    if (s->n_tl_gen) {
      int nb = 0;
      const TileList th = tile_list(s->d_tl_gen, s->n_tl_gen, 1, 1, &nb);
      Timer tm(s, FDTD_K_GEN_H);
      hipLaunchKernelGGL(k_gen_h<real>, dim3((unsigned)nb), dim3(256), 0, st, an, p, pw, m, th);
    }
    for (int q = 0; q < 3; ++q) {
      std::swap(s->E[q], s->E2[q]);
      std::swap(s->H[q], s->H2[q]);
    }
    std::swap(s->d_split, s->d_split2);
    a = field_args<real>(s);
    tfsf_e(st);
    tfsf_h(st, pml_args<real>(s), 1);
    pend(63, 3);
  } else if (s->engine == FDTD_ENGINE_FUSED) {
    PmlArgs<real> p = pml_args<real>(s);
    Parts all{};
    int tiles = 0;
    const SegGrid gt = seg_grid(s->nx, s->ny, (int64_t)s->ny * ((s->nz + s->zm - 1) / s->zm), &tiles);
    const SegGrid gm = seg_grid(s->nx, s->ny, s->nmix, &all.mix);
    const AdeMulti ade = ade_lists(a, &all.ade);
    auto by_zm = [&](auto&& go) {
      if (s->zm == 8)
        go(std::integral_constant<int, 8>{});
      else if (s->zm == 4)
        go(std::integral_constant<int, 4>{});
      else if (s->zm == 2)
        go(std::integral_constant<int, 2>{});
      else
        go(std::integral_constant<int, 1>{});
    };
    {
      MonList<real> mon{};
      if (!apart) mon = take_pending<real>(s);
      all.mon = round8(mon.nblk);
      auto launch = [&](const Parts& pt, int ntile) {
        const int lists = pt.mon + round8(pt.ade) + pt.mix, nb = lists + ntile;
        if (!nb) return;
        auto go = [&](auto kern) {
          hipLaunchKernelGGL(kern, dim3((unsigned)nb), dim3(256), 0, st, a, p, src, nsrc, pt, mon, ade,
                             (const int32_t*)s->d_mixrows, gm, gt);
        };
        by_zm([&](auto kz) {
          lists ? go(k_step_e<real, decltype(kz)::value, true>) : go(k_step_e<real, decltype(kz)::value, false>);
        });
      };
      if (apart) {
        {
          Timer tm(s, FDTD_K_E);
          launch(Parts{}, tiles);
          launch(Parts{0, 0, all.mix, 0, 0, 0}, 0);
        }
        if (all.ade) {
          Timer tm(s, FDTD_K_ADE);
          launch(Parts{0, all.ade, 0, 0, 0, 0}, 0);
        }
      } else if (sizeof(real) == 8 || tiles < kListsApart) {
        launch(all, tiles);
      } else {
        launch(Parts{}, tiles);
        launch(all, 0);
      }
    }
    for (auto& g : s->groups) {
      if (!g.ncells) continue;
      Timer tm(s, FDTD_K_ADE);
      if (g.kind == 1)
        hipLaunchKernelGGL(k_ljp<real>, dim3((unsigned)((g.ncells + 255) / 256)), dim3(256), 0, st, a, g.lj,
                           g.d_cells, g.d_mask, (double*)g.d_state, g.ncells, src, nsrc);
      else if (g.kind == 2)
        hipLaunchKernelGGL((k_lord<real, true>), dim3((unsigned)((g.ncells + 255) / 256)), dim3(256), 0, st, a,
                           lord_coef(g), g.d_cells, g.d_mask, (double*)g.d_state, g.ncells, src, nsrc);
    }
    const bool with_line = !apart && !s->dry && s->tfsfs.size() == 1;
    if (!with_line) tfsf_e(st);
    {
      const MonList<real> mon = e_samples();
      Parts pt{};
      pt.mon = round8(mon.nblk);
      pt.line = with_line ? 8 : 0;  // a whole round of blocks over the XCDs
      const TfsfLine line = with_line ? tfsf_line(s, s->tfsfs[0]) : TfsfLine{};
      const double line_g = with_line ? line_pulse(s->tfsfs[0].p.pulse) : 0.0;
      Timer tm(s, FDTD_K_H);
      by_zm([&](auto kz) {
        hipLaunchKernelGGL((k_step_h<real, decltype(kz)::value>), dim3((unsigned)(pt.line + pt.mon + tiles)), dim3(256),
                           0, st, a, p, pt, mon, gt, line, line_g);
      });
    }
    tfsf_h(st, p, 1);
    mon_apart ? pend(63, 3) : pend(56, 2);
  } else {
    RefPmlArgs<real> rp{};
    if (refy) rp = ref_pml_args<real>(s);
    Parts all{};
    int tiles = 0, main_tiles = 0;
    const SegGrid gt = seg_grid(s->nx, s->ny, (int64_t)s->ny * s->nz, &tiles);
    const SegGrid gh = seg_grid(s->nx, s->ny - 2 * Py, (int64_t)(s->ny - 2 * Py) * s->nz, &main_tiles);
    const SegGrid gs = seg_grid(s->nx, std::max(1, 2 * Py), (int64_t)2 * Py * s->nz, &all.mix);
    const AdeMulti ade = ade_lists(a, &all.ade);
    // the Lorentz cells' launches read E or the new D, and write E the split
    // fields then replace: the slabs' part comes after them
    bool lorentz = false;
    for (const auto& g : s->groups) lorentz |= g.kind != 0 && g.ncells;
    {
      MonList<real> mon{};
      if (!apart) mon = take_pending<real>(s);
      all.mon = round8(mon.nblk);
      auto launch = [&](const Parts& pt, int ntile) {
        const int nb = pt.mon + round8(pt.ade) + pt.mix + ntile;
        auto go = [&](auto kern) {
          hipLaunchKernelGGL(kern, dim3((unsigned)nb), dim3(256), 0, st, a, rp, src, nsrc, rows, pt, mon, ade, gs, gt);
        };
        if (nb) s->nt_d ? go(k_staged_e<real, true>) : go(k_staged_e<real, false>);
      };
      if (apart) {
        {
          Timer tm(s, FDTD_K_E);
          launch(Parts{}, tiles);
        }
        if (all.ade) {
          Timer tm(s, FDTD_K_ADE);
          launch(Parts{0, all.ade, 0, 0, 0, 0}, 0);
        }
      } else if (lorentz) {
        launch(Parts{all.mon, all.ade, 0, 0, 0, 0}, tiles);
      } else {
        launch(all, tiles);
      }
    }
    for (auto& g : s->groups) {
      if (!g.ncells) continue;
      Timer tm(s, FDTD_K_ADE);
      if (g.kind == 1)  // E form from curl H: the plane sources enter here, not through D
        hipLaunchKernelGGL(k_ljp<real>, dim3((unsigned)((g.ncells + 255) / 256)), dim3(256), 0, st, a, g.lj,
                           g.d_cells, g.d_mask, (double*)g.d_state, g.ncells, src, nsrc);
      else if (g.kind == 2)
        hipLaunchKernelGGL((k_lord<real, false>), dim3((unsigned)((g.ncells + 255) / 256)), dim3(256), 0, st, a,
                           lord_coef(g), g.d_cells, g.d_mask, (double*)g.d_state, g.ncells, src, 0);
    }
    if (refy && (apart || lorentz)) {
      Timer tm(s, FDTD_K_PML_E);
      hipLaunchKernelGGL((k_staged_e<real, false>), dim3((unsigned)all.mix), dim3(256), 0, st, a, rp, src, nsrc, rows,
                         Parts{0, 0, all.mix, 0, 0, 0}, MonList<real>{}, AdeMulti{}, gs, gt);
    }
    tfsf_e(st);
    {
      const MonList<real> mon = e_samples();
      auto launch = [&](const Parts& pt, const MonList<real>& m, int ntile) {
        const int nb = pt.mon + pt.mix + ntile;
        if (nb)
          hipLaunchKernelGGL(k_staged_h<real>, dim3((unsigned)nb), dim3(256), 0, st, a, rp, rows, pt, m, gs, gh);
      };
      if (apart) {
        {
          Timer tm(s, FDTD_K_H);
          launch(Parts{}, mon, main_tiles);
        }
        if (refy) {
          Timer tm(s, FDTD_K_PML_H);
          launch(Parts{0, 0, all.mix, 0, 0, 0}, mon, 0);
        }
      } else {
        launch(Parts{round8(mon.nblk), 0, all.mix, 0, 0, 0}, mon, main_tiles);
      }
    }
    tfsf_h(st, PmlArgs<real>{}, 0);
    mon_apart ? pend(63, 3) : pend(56, 2);
  }
  if (mon_apart) flush_pending<real>(s);
  // dry steps (the autotuner's) sample into the ring slot the next real step
  // overwrites, so each step form is timed with its sampling cost, and
  // neither advance the ring, fold nor record probes
  if (s->dry) return 0;
  // fold after this step's samples are written, when the ring is full or
  // the step is a multiple of kDftBlock: the blocks then end at the same
  // steps however the calls that make the steps are cut (a call folds what
  // it buffered at its end), so runs stepped in chunks of kDftBlock
  // multiples, or resumed from a checkpoint, equal runs stepped at once
  for (auto& d : s->dfts) {
    if (n < d.n_begin || (d.n_end > 0 && n > d.n_end)) continue;
    if (d.nbuf == 0) d.n_first = n;
    d.nbuf += 1;
    if (d.nbuf == kDftBlock || n % kDftBlock == 0) dft_flush_plane<real>(s, d);
  }
  return 0;
}

}  // namespace

int launch_step(Sim* s) {
  // launch errors are read back with hipGetLastError, which reports the
  // last failing call of this thread: clear what an earlier, unrelated call
  // left so it is not taken for a launch failure of this step
  (void)hipGetLastError();
  int rc = s->prec == FDTD_FP32 ? step_impl<float>(s) : step_impl<double>(s);
  if (rc) return rc;
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return hip_check(e, "kernel launch");
  return 0;
}

int launch_dft_flush(Sim* s) {
  // the last step's samples and probes, whether or not a plane has a block open
  if (s->prec == FDTD_FP32)
    flush_pending<float>(s);
  else
    flush_pending<double>(s);
  for (auto& d : s->dfts) {
    if (s->prec == FDTD_FP32)
      dft_flush_plane<float>(s, d);
    else
      dft_flush_plane<double>(s, d);
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return hip_check(e, "DFT flush");
  return 0;
}

int flux_check(Sim* s, int id) {
  const DftPlane& d = s->dfts[id];
  const int axis = d.axis;
  const int need[4] = {axis == 1 ? FDTD_HX : (axis == 2 ? FDTD_HY : FDTD_HZ),
                       axis == 1 ? FDTD_EZ : (axis == 2 ? FDTD_EX : FDTD_EY),
                       axis == 1 ? FDTD_HZ : (axis == 2 ? FDTD_HX : FDTD_HY),
                       axis == 1 ? FDTD_EX : (axis == 2 ? FDTD_EY : FDTD_EZ)};
  for (int q = 0; q < 4; ++q)
    if (!(d.mask & (1 << need[q]))) return set_error(FDTD_ERR_ARG, "flux needs the four tangential components");
  return 0;
}

// Interior rows of planes k0.. of a field, as FP64 without the ghosts: a
// wavefront 64 cells of a row, bound by its writes (8 B a cell).
template <typename real>
__global__ __launch_bounds__(256) void k_pack(const real* __restrict__ f, int nx, int ny, int64_t px, int64_t pxy,
                                              int k0, int64_t rows, double* __restrict__ out) {
  const int64_t r = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (r >= rows) return;
  const int64_t k = r / ny, j = r - k * ny;
  const real* row = f + px * (j + 1) + pxy * (k0 + k);
  for (int i = (int)threadIdx.x & 63; i < nx; i += 64) out[r * nx + i] = (double)row[i + 1];
}

int launch_pack(Sim* s, const void* field, int k0, int planes, double* out) {
  FDTD_HIP(hipSetDevice(s->device));
  const int64_t rows = (int64_t)s->ny * planes;
  const dim3 nb((unsigned)((rows + 3) / 4));
  if (s->prec == FDTD_FP32)
    hipLaunchKernelGGL(k_pack<float>, nb, dim3(256), 0, s->stream, (const float*)field, s->nx, s->ny, s->px, s->pxy,
                       k0, rows, out);
  else
    hipLaunchKernelGGL(k_pack<double>, nb, dim3(256), 0, s->stream, (const double*)field, s->nx, s->ny, s->px, s->pxy,
                       k0, rows, out);
  FDTD_HIP(hipGetLastError());
  return 0;
}

int launch_flux(Sim* s, int id, double* S) {
  int rc = flux_check(s, id);
  if (rc) return rc;
  double* dS = reduction_buffer(s, sizeof(double) * (size_t)s->dfts[id].nfreq);
  if (!dS) return set_error(FDTD_ERR_NOMEM, "flux buffer");
  return launch_flux_into(s, id, dS, S);
}

// The flux reduction of plane `id` into the device buffer dS (nfreq
// doubles, each written whole), then copied to the host array S.
int launch_flux_into(Sim* s, int id, double* dS, double* S) {
  DftPlane& d = s->dfts[id];
  int eA, eB, hA, hB;
  if (d.axis == 1) { hA = FDTD_HX; eA = FDTD_EZ; hB = FDTD_HZ; eB = FDTD_EX; }
  else if (d.axis == 2) { hA = FDTD_HY; eA = FDTD_EX; hB = FDTD_HX; eB = FDTD_EY; }
  else { hA = FDTD_HZ; eA = FDTD_EY; hB = FDTD_HY; eB = FDTD_EZ; }
  const int64_t np = (int64_t)d.n1 * d.n2;
  hipLaunchKernelGGL(k_flux, dim3((unsigned)d.nfreq), dim3(256), 0, s->stream, d.d_acc, np, d.nfreq, d.slot[hA],
                     d.slot[eA], d.slot[hB], d.slot[eB], s->ds, dS);
  FDTD_HIP(hipGetLastError());
  FDTD_HIP(hipMemcpyAsync(S, dS, sizeof(double) * (size_t)d.nfreq, hipMemcpyDeviceToHost, s->stream));
  FDTD_HIP(hipStreamSynchronize(s->stream));
  return 0;
}

int launch_energy(Sim* s, double* we, double* wh) {
  const int nb = 1024;
  double* part = reduction_buffer(s, sizeof(double) * 2 * nb);
  if (!part) return set_error(FDTD_ERR_NOMEM, "energy buffer");
  if (s->prec == FDTD_FP32)
    hipLaunchKernelGGL(k_energy<float>, dim3(nb), dim3(256), 0, s->stream, field_args<float>(s), part);
  else
    hipLaunchKernelGGL(k_energy<double>, dim3(nb), dim3(256), 0, s->stream, field_args<double>(s), part);
  FDTD_HIP(hipGetLastError());
  std::vector<double> h(2 * nb);
  FDTD_HIP(hipMemcpyAsync(h.data(), part, sizeof(double) * 2 * nb, hipMemcpyDeviceToHost, s->stream));
  FDTD_HIP(hipStreamSynchronize(s->stream));
  double a = 0, b = 0;
  for (int q = 0; q < nb; ++q) {
    a += h[2 * q];
    b += h[2 * q + 1];
  }
  *we = a;
  *wh = b;
  return 0;
}

int launch_nonfinite(Sim* s, int* d_flag) {
  const int64_t n = s->ncell_alloc;
  const dim3 grid((unsigned)std::min<int64_t>((n + 255) / 256, 4096));
  if (s->prec == FDTD_FP32)
    hipLaunchKernelGGL(k_nonfinite<float>, grid, dim3(256), 0, s->stream, (const float*)s->E[0],
                       (const float*)s->E[1], (const float*)s->E[2], (const float*)s->H[0], (const float*)s->H[1],
                       (const float*)s->H[2], n, d_flag);
  else
    hipLaunchKernelGGL(k_nonfinite<double>, grid, dim3(256), 0, s->stream, (const double*)s->E[0],
                       (const double*)s->E[1], (const double*)s->E[2], (const double*)s->H[0],
                       (const double*)s->H[1], (const double*)s->H[2], n, d_flag);
  FDTD_HIP(hipGetLastError());
  return 0;
}

int launch_set_ghosts(Sim* s, int comp) {
  const int n[3] = {s->nx, s->ny, s->nz};
  for (int ax = 0; ax < 3; ++ax) {
    if (!s->g.periodic[ax]) continue;
    const int a1 = ax == 0 ? 1 : 0, a2 = ax == 2 ? 1 : 2;
    dim3 grid((unsigned)((n[a1] + 2 + 63) / 64), (unsigned)(n[a2] + 2));
    void* f = comp < 3 ? s->E[comp] : (comp < 6 ? s->H[comp - 3] : s->D[comp - 6]);
    if (s->prec == FDTD_FP32)
      hipLaunchKernelGGL(k_ghosts<float>, grid, dim3(64), 0, s->stream, field_args<float>(s), (float*)f, ax);
    else
      hipLaunchKernelGGL(k_ghosts<double>, grid, dim3(64), 0, s->stream, field_args<double>(s), (double*)f, ax);
  }
  FDTD_HIP(hipGetLastError());
  return 0;
}

}  // namespace fdtd
