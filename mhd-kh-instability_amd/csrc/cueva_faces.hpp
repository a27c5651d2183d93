// Face kernel of the CUEVA step: MPx reconstruction of every quantity at the
// x and y faces of a face pair and the HLL / HLLE / HLLC solve, written to
// the face-flux planes.  T is the arithmetic of reconstruction and Riemann
// solve: double (bitwise with the reference) or float (the mixed form, built
// in its own translation unit).
#pragma once

#include <stddef.h>

#include <type_traits>
#include <utility>

#include "cueva_common.hpp"
#include "cueva_update.hpp"

#ifndef CUEVA_XCD_FACES
#define CUEVA_XCD_FACES 1
#endif
// minimum waves per SIMD the marching kernel is compiled for (0: the
// default of march_min_waves)
#ifndef CUEVA_MARCH_F32_WAVES
#define CUEVA_MARCH_F32_WAVES 0
#endif
#ifndef CUEVA_MARCH_F64_WAVES
#define CUEVA_MARCH_F64_WAVES 0
#endif
#ifndef CUEVA_FACES_WAVES_PER_EU
#define FACES_WAVES
#else
#define FACES_WAVES __attribute__((amdgpu_waves_per_eu(CUEVA_FACES_WAVES_PER_EU, CUEVA_FACES_WAVES_PER_EU)))
#endif

namespace cueva {

// Stencils loaded ahead of the one being reconstructed, by the type of the
// planes they are loaded from.  FP64 planes (FP64 form, 2 waves per SIMD, HLLC
// + MP5 at 2048x4096, step with 0 / 1 / 2 / 3): 6.6 / 5.53 / 5.19 / 5.12 ms.
// FP32 planes (mixed form, 3 waves per SIMD, 2 / 3 / 4): 3.49 / 3.40 / 3.37
// (5 at 2 waves 3.37; 4 waves per SIMD with 2 spill, 3.61).
template <typename ST> constexpr int face_ahead() { return sizeof(ST) == 8 ? 3 : 4; }

// launch grid of k_faces over the face pairs [-1,imax] x [-1,jmax]
inline dim3 faces_grid(const Geom& g, dim3 blk) {
  const unsigned tx = (unsigned)((g.imax + 2 + blk.x - 1) / blk.x), ty = (unsigned)((g.jmax + 2 + blk.y - 1) / blk.y);
#if CUEVA_XCD_FACES
  return dim3(8 * ((tx * ty + 7) / 8));
#else
  return dim3(tx, ty);
#endif
}

// ---------------------------------------------------------------------------
// faces: reconstruction + Riemann solve for the face pair (i,j), i.e. the x
// face between (i,j),(i+1,j) and the y face between (i,j),(i,j+1), for
// i in [-1,imax], j in [-1,jmax] (16_*_flow_mpx.f95 face loops)
// ---------------------------------------------------------------------------
// The cell a face solve stands at, split for the addressing of a wavefront:
// its 64 lanes share the row, so a plane's row address is formed on scalar
// registers and each lane adds only its 32-bit byte offset within the row
// (global loads take a scalar base, a 32-bit lane offset and a constant).
struct Cell {
  uint32_t vo;   // byte offset of column i in its row of an FP64 plane
  int64_t ro;    // first element of row j (the same for every lane)
  int pitch;
};
__device__ inline Cell cell_of(const Geom& g, int i, int j) {
  return {(uint32_t)(i + X0) * 8u, (int64_t)(__builtin_amdgcn_readfirstlane(j) + GH) * g.pitch, g.pitch};
}
// element (i + DI, j + dj)
template <int DI = 0, typename ST> __device__ inline ST at_cell(const ST* __restrict__ a, const Cell& c, int dj = 0) {
  const char* row = (const char*)(a + (c.ro + (int64_t)dj * c.pitch));
  return *(const ST*)(row + (sizeof(ST) == 8 ? c.vo : c.vo >> 1) + DI * (int)sizeof(ST));
}

// the NV values of one quantity across the face, as loaded (MPx: 2K+2; MC
// limiter: 4)
template <int NV, typename ST> struct Sten { ST v[NV]; };
template <int DIR, typename ST, int... T>
__device__ inline void sten_load(const ST* __restrict__ a, const Cell& c, Sten<(int)sizeof...(T), ST>& s,
                                 std::integer_sequence<int, T...>) {
  constexpr int K = (int)sizeof...(T) / 2 - 1;
  ((s.v[T] = DIR == 0 ? at_cell<DIR == 0 ? T - K : 0>(a, c) : at_cell(a, c, T - K)), ...);
}

// quantities reconstructed at a face, in the order they are taken: the
// kinematics first (the fallbacks couple the two faces of a pair)
enum { F_VX, F_VY, F_VZ, F_P, F_RHO, F_PSI, F_PHI, F_EX, F_EY, F_EZ, F_BX, F_BY, F_BZ, F_Q, F_D, F_TAU, F_SX, F_SY,
       F_SZ, F_JN, F_NQ };
template <int F, int DIR, bool STAGE_KIN, typename ST> __device__ inline const ST* face_plane(const Planes& P) {
  if constexpr (F <= F_RHO) {
    constexpr int q = F == F_VX ? K_VX : F == F_VY ? K_VY : F == F_VZ ? K_VZ : F == F_P ? K_P : K_RHO;
    return kin_src<ST, STAGE_KIN>(P, q);
  } else {
    constexpr int s[15] = {S_PSI, S_PHI, S_EX, S_EY, S_EZ, S_BX, S_BY, S_BZ, S_Q, S_D, S_TAU, S_SX, S_SY, S_SZ,
                           DIR == 0 ? S_JX : S_JY};
    constexpr int k = s[F - F_PSI];
    return stage_src<ST>(P, k);
  }
}
template <int F, typename T> __device__ inline T& face_slot(Side<T>& o) {
  constexpr T Side<T>::*m[F_NQ] = {&Side<T>::vx, &Side<T>::vy, &Side<T>::vz, &Side<T>::p, &Side<T>::rho,
                                   &Side<T>::psi, &Side<T>::phi, &Side<T>::ex, &Side<T>::ey, &Side<T>::ez,
                                   &Side<T>::bx, &Side<T>::by, &Side<T>::bz, &Side<T>::q, &Side<T>::d,
                                   &Side<T>::tau, &Side<T>::sx, &Side<T>::sy, &Side<T>::sz, &Side<T>::jn};
  return o.*m[F];
}

template <int F, int DIR, bool STAGE_KIN, int NV, typename ST>
__device__ inline void face_load(const Planes& P, const Cell& c, Sten<NV, ST>& s) {
  sten_load<DIR>(face_plane<F, DIR, STAGE_KIN, ST>(P), c, s, std::make_integer_sequence<int, NV>());
}
template <int ORD, int F, int N, typename ST, typename T>
__device__ inline void face_take(const Sten<N, ST>& s, Side<T>& L, Side<T>& R) {
  T v[N];
#pragma unroll
  for (int t = 0; t < N; t++) v[t] = (T)s.v[t];
  if constexpr (F == F_P || F == F_RHO) mp_face_pos<ORD>(v, face_slot<F>(L), face_slot<F>(R));
  else mp_face<ORD>(v, face_slot<F>(L), face_slot<F>(R));
}

// Reconstruct quantities F0 + S... of one face.  The stencils of the next
// quantities are loaded before the current one is reconstructed: the
// limiter's wavefront-wide branch keeps the compiler from moving loads across
// it, and without this every quantity waited for its own loads.
template <int ORD, int F0, int DIR, bool STAGE_KIN, typename ST, typename T, int... S>
__device__ inline void face_fields_seq(const Planes& P, const Cell& c, Side<T>& L, Side<T>& R,
                                       std::integer_sequence<int, S...>) {
  constexpr int N = sizeof...(S), AH = face_ahead<ST>();
  Sten<2 * MPc<ORD>::K + 2, ST> b[AH + 1];
  auto pre = [&](auto t) {
    if constexpr (t() < AH && t() < N) face_load<F0 + t(), DIR, STAGE_KIN>(P, c, b[t()]);
  };
  auto one = [&](auto t) {
    if constexpr (t() + AH < N)
      face_load<F0 + t() + AH, DIR, STAGE_KIN>(P, c, b[(t() + AH) % (AH + 1)]);
    face_take<ORD, F0 + t()>(b[t() % (AH + 1)], L, R);
  };
  (pre(std::integral_constant<int, S>()), ...);
  (one(std::integral_constant<int, S>()), ...);
}
template <int ORD, int F0, int F1, int DIR, bool STAGE_KIN, typename ST, typename T>
__device__ inline void face_fields(const Planes& P, const Cell& c, Side<T>& L, Side<T>& R) {
  face_fields_seq<ORD, F0, DIR, STAGE_KIN, ST>(P, c, L, R, std::make_integer_sequence<int, F1 - F0>());
}

// ---------------------------------------------------------------------------
// HLL with the monotonised-central slope limiter (flux_solver = 2,
// 16_hll_flow_mcl.f95:554-1402, REC_PRIM = 0): second-order face states of
// the stage fields and of the t^n velocity, pressure and density, and the
// Lax-Friedrichs-form HLL flux with signal speed Sp = 1 (const_sp = 0,
// parameters.f95:274).  The x face uses only x-reconstructed states and the
// y face only y-reconstructed ones.
// ---------------------------------------------------------------------------
// mcl(fa, fb) of funciones.f95:57-95 (kind = slop, parameters.f95:17) and
// limiter(ga, gb) of funciones.f95:100-142 (kind = limit, :18): 1 MinMod,
// 2 monotonised central, 3 Superbee; the three-argument min as flang
// evaluates it, min(min(a, b), c)
template <typename T> __device__ inline T mcl_slope(T fa, T fb, int kind = 2) {
  const T s = T(0.5) * (csign(fa) + csign(fb));
  if (kind == 1) return s * mn(fab(fa), fab(fb));
  if (kind == 3) return s * mn(mn(T(2) * fab(fa), T(2) * fab(fb)), mx(fab(fa), fab(fb)));
  // a NaN operand that FP64's minimum drops is NaN in the sum as well
  return s * mn(T(2) * lim_mn(fab(fa), fab(fb)), T(0.5) * fab(fa + fb));
}

// J, FD, Ftau and the three FS of one side: E^2+B^2 (16_hll_flow_mcl.f95:821),
// W (:900), E.v (:995), J (:1033), FD (:1050), eps and h (:1124), Ftau
// (:1181), FS (:1198-1241)
template <int DIR, typename T> __device__ inline void mcl_side_fluxes(T gam, T sigma, Side<T>& o) {
  const T e2b2 = ((((sq(o.ex) + sq(o.ey)) + sq(o.ez)) + sq(o.bx)) + sq(o.by)) + sq(o.bz);
  const T w = T(1) / sqrt(((T(1) - sq(o.vx)) - sq(o.vy)) - sq(o.vz));
  const T edv = (o.ex * o.vx + o.ey * o.vy) + o.ez * o.vz;
  const T eps = o.p / ((gam - T(1)) * o.rho);
  const T h = o.rho * (T(1) + eps) + o.p;
  const T hw2 = h * sq(w);
  if constexpr (DIR == 0) {
    o.jn = (sigma * w) * ((o.ex + (o.bz * o.vy - o.by * o.vz)) - edv * o.vx) + o.q * o.vx;
    o.fd = o.d * o.vx;
    o.ftau = (o.bz * o.ey - o.by * o.ez) + hw2 * o.vx;
    o.fs1 = ((((-sq(o.ex)) - sq(o.bx)) + hw2 * sq(o.vx)) + T(0.5) * e2b2) + o.p;
    o.fs2 = ((-(o.ex * o.ey)) - o.bx * o.by) + (hw2 * o.vx) * o.vy;
    o.fs3 = ((-(o.ex * o.ez)) - o.bx * o.bz) + (hw2 * o.vx) * o.vz;
  } else {
    o.jn = (sigma * w) * ((o.ey + (o.bx * o.vz - o.bz * o.vx)) - edv * o.vy) + o.q * o.vy;
    o.fd = o.d * o.vy;
    o.ftau = (o.bx * o.ez - o.bz * o.ex) + hw2 * o.vy;
    o.fs1 = ((-(o.ex * o.ey)) - o.bx * o.by) + (hw2 * o.vx) * o.vy;
    o.fs2 = ((((-sq(o.ey)) - sq(o.by)) + hw2 * sq(o.vy)) + T(0.5) * e2b2) + o.p;
    o.fs3 = ((-(o.ey * o.ez)) - o.by * o.bz) + (hw2 * o.vy) * o.vz;
  }
}

// One quantity's left and right face values between a cell and its +x (DIR 0)
// or +y (DIR 1) neighbour (u_L = u_i + FAC mcl(.), u_R = u_{i+1} - FAC mcl(.),
// FAC = 0.5), and of the tangential E and B pair the "_m" states: the cell
// value negated, the slope kept (16_hll_flow_mcl.f95:634-655, 708-737)
template <int F, int DIR, int KIND, typename ST, typename T>
__device__ inline void mcl_take(int slop, const Sten<4, ST>& s, Side<T>& L, Side<T>& R) {
  const T um = (T)s.v[0], u0 = (T)s.v[1], u1 = (T)s.v[2], u2 = (T)s.v[3];
  const T sl = T(0.5) * mcl_slope(u1 - u0, u0 - um, KIND ? KIND : slop);
  const T sr = T(0.5) * mcl_slope(u2 - u1, u1 - u0, KIND ? KIND : slop);
  face_slot<F>(L) = u0 + sl;
  face_slot<F>(R) = u1 - sr;
  if constexpr (F == (DIR == 0 ? F_EZ : F_EX)) {
    L.em = (-u0) + sl;
    R.em = (-u1) - sr;
  }
  if constexpr (F == (DIR == 0 ? F_BY : F_BZ)) {
    L.bm = (-u0) + sl;
    R.bm = (-u1) - sr;
  }
}

// The states of one face from the MC limiter with their physical fluxes
// (16_hllc_flow_mcl.f95:1760-2479 forms the same ones).  A quantity's four
// values are loaded MCL_AHEAD quantities before it is reconstructed, and its
// two states are pinned where they are formed: left to itself the compiler put
// the reconstruction where the states are used, which held all nineteen
// stencils in registers (63-168 VGPRs spilled in FP64; none now) and exposed
// the loads.  HLL + MC FP64 step at 2048x4096 / 300x700: 7.1 ms / 188 us
// before; 2 ahead 3.66 / 102.6, 4 ahead 3.47 / 102.1, 6 ahead 3.50 / 102.5.
constexpr int MCL_AHEAD = 4;
template <int DIR, int KIND, bool STAGE_KIN, typename ST, typename T, int... Q>
__device__ inline void mcl_fields(const Planes& P, int slop, const Cell& c, Side<T>& L, Side<T>& R,
                                  std::integer_sequence<int, Q...>) {
  constexpr int N = sizeof...(Q), AH = MCL_AHEAD;
  Sten<4, ST> b[AH + 1];
  auto pre = [&](auto t) {
    if constexpr (t() < AH) face_load<t(), DIR, STAGE_KIN>(P, c, b[t()]);
  };
  auto one = [&](auto t) {
    if constexpr (t() + AH < N) face_load<t() + AH, DIR, STAGE_KIN>(P, c, b[(t() + AH) % (AH + 1)]);
    mcl_take<t(), DIR, KIND>(slop, b[t() % (AH + 1)], L, R);
    asm volatile("" : "+v"(face_slot<t()>(L)), "+v"(face_slot<t()>(R)));
    __builtin_amdgcn_sched_barrier(0);
  };
  (pre(std::integral_constant<int, Q>()), ...);
  (one(std::integral_constant<int, Q>()), ...);
}
template <int F, int DIR, bool STAGE_KIN, typename ST, typename T>
__device__ inline void mcl_one(const Planes& P, int slop, const Cell& c, Side<T>& L, Side<T>& R) {
  Sten<4, ST> s;
  face_load<F, DIR, STAGE_KIN>(P, c, s);
  mcl_take<F, DIR, 0>(slop, s, L, R);
}
template <int DIR, bool STAGE_KIN, typename ST, typename T>
__device__ inline void mcl_sides(const Planes& P, const Scheme& S, const Cell& c, Side<T>& L, Side<T>& R) {
  // the default slope has its own body: chosen per quantity, the compiler
  // evaluated all three slopes and selected
  if (S.slop == 2) mcl_fields<DIR, 2, STAGE_KIN, ST>(P, S.slop, c, L, R, std::make_integer_sequence<int, F_JN>());
  else mcl_fields<DIR, 0, STAGE_KIN, ST>(P, S.slop, c, L, R, std::make_integer_sequence<int, F_JN>());
  mcl_side_fluxes<DIR>((T)S.gamma, (T)S.sigma, L);
  mcl_side_fluxes<DIR>((T)S.gamma, (T)S.sigma, R);
}

// 0.5 (A_L + A_R - Sp (U_R - U_L)) with Sp = 1 (16_hll_flow_mcl.f95:1259-1396)
template <typename T> __device__ inline T mcl_lf(T al, T ar, T ul, T ur) { return T(0.5) * ((al + ar) - (ur - ul)); }

// the fluxes of the face between the cell at c and its +x (DIR 0, FX_* slots)
// or +y neighbour (DIR 1, FY_*)
template <int DIR, bool STAGE_KIN, typename ST, typename T>
__device__ inline void mcl_face(const Planes& P, const Scheme& S, const Cell& c, T* f) {
  Side<T> L, R;
  mcl_sides<DIR, STAGE_KIN, ST>(P, S, c, L, R);
  if constexpr (DIR == 0) {
    f[FX_EXPSI] = mcl_lf(L.ex, R.ex, L.psi, R.psi);
    f[FX_BXPHI] = mcl_lf(L.bx, R.bx, L.phi, R.phi);
    f[FX_PHIBX] = mcl_lf(L.phi, R.phi, L.bx, R.bx);
    f[FX_EZBY] = -mcl_lf(L.em, R.em, L.by, R.by);
    f[FX_EYBZ] = mcl_lf(L.ey, R.ey, L.bz, R.bz);
    f[FX_PSIEX] = mcl_lf(L.psi, R.psi, L.ex, R.ex);
    f[FX_BZEY] = mcl_lf(L.bz, R.bz, L.ey, R.ey);
    f[FX_BYEZ] = -mcl_lf(L.bm, R.bm, L.ez, R.ez);
    f[FX_J] = mcl_lf(L.jn, R.jn, L.q, R.q);
    f[FX_FD] = mcl_lf(L.fd, R.fd, L.d, R.d);
    f[FX_FTAU] = mcl_lf(L.ftau, R.ftau, L.tau, R.tau);
    f[FX_FSX] = mcl_lf(L.fs1, R.fs1, L.sx, R.sx);
    f[FX_FSY] = mcl_lf(L.fs2, R.fs2, L.sy, R.sy);
    f[FX_FSZ] = mcl_lf(L.fs3, R.fs3, L.sz, R.sz);
  } else {
    f[FY_EYPSI] = mcl_lf(L.ey, R.ey, L.psi, R.psi);
    f[FY_BYPHI] = mcl_lf(L.by, R.by, L.phi, R.phi);
    f[FY_EZBX] = mcl_lf(L.ez, R.ez, L.bx, R.bx);
    f[FY_PHIBY] = mcl_lf(L.phi, R.phi, L.by, R.by);
    f[FY_EXBZ] = -mcl_lf(L.em, R.em, L.bz, R.bz);
    f[FY_BZEX] = -mcl_lf(L.bm, R.bm, L.ex, R.ex);
    f[FY_PSIEY] = mcl_lf(L.psi, R.psi, L.ey, R.ey);
    f[FY_BXEZ] = mcl_lf(L.bx, R.bx, L.ez, R.ez);
    f[FY_J] = mcl_lf(L.jn, R.jn, L.q, R.q);
    f[FY_FD] = mcl_lf(L.fd, R.fd, L.d, R.d);
    f[FY_FTAU] = mcl_lf(L.ftau, R.ftau, L.tau, R.tau);
    f[FY_FSX] = mcl_lf(L.fs1, R.fs1, L.sx, R.sx);
    f[FY_FSY] = mcl_lf(L.fs2, R.fs2, L.sy, R.sy);
    f[FY_FSZ] = mcl_lf(L.fs3, R.fs3, L.sz, R.sz);
  }
}

// ---------------------------------------------------------------------------
// Lax-Friedrichs flux splitting (flux_solver = 1, 15_lax_flow.f95:733-1460):
// at every cell the split fluxes F+- = A +- Sp U (Sp = 1) of the stage fields
// and of the cell fluxes flowinit forms (14_flowinit.f95:264-373); the face
// value is 0.5 (L + R), L = F+(i) + FAC mcl(F+(i+1)-F+(i), F+(i)-F+(i-1)),
// R = F-(i+1) - FAC mcl(F+(i+2)-F+(i+1), F+(i+1)-F+(i)) (the slope of R is
// also taken from F+).  flowinit fills only the interior and
// boundary_flux_conserved no ghosts for this solver, so the cell fluxes are
// 0 on ghost cells (cleanvarint, 07_clean_var.f95:341-350).
// ---------------------------------------------------------------------------
// J, FD, Ftau, FS along DIR at cell (i,j) = k, with the t^n W and enthalpy
// of startconvar (06_conserved_var.f95:92-109)
template <int DIR, typename ST, typename T>
__device__ inline void lax_cell_fluxes(const Geom& g, const Planes& P, const Scheme& S, int i, int j, int64_t k,
                                       T* out) {
  if (i < 0 || i > g.imax || j < 0 || j > g.jmax) {
#pragma unroll
    for (int t = 0; t < 6; t++) out[t] = T(0);
    return;
  }
  // flowinit's cell fluxes: of v^n, p^n, rho^n, or with REC_PRIM = 1 of the
  // stage's primitives (14_flowinit.f95:376-489)
  const T vx = (T)kin_src<ST>(P, K_VX)[k], vy = (T)kin_src<ST>(P, K_VY)[k], vz = (T)kin_src<ST>(P, K_VZ)[k];
  const T p = (T)kin_src<ST>(P, K_P)[k], rho = (T)kin_src<ST>(P, K_RHO)[k];
  const T ex = (T)stage_src<ST>(P, S_EX)[k], ey = (T)stage_src<ST>(P, S_EY)[k], ez = (T)stage_src<ST>(P, S_EZ)[k];
  const T bx = (T)stage_src<ST>(P, S_BX)[k], by = (T)stage_src<ST>(P, S_BY)[k], bz = (T)stage_src<ST>(P, S_BZ)[k];
  const T w = T(1) / sqrt(T(1) - ((sq(vx) + sq(vy)) + sq(vz)));
  const T eps = p / (((T)S.gamma - T(1)) * rho);
  const T h = rho * (T(1) + eps) + p;
  const T e2 = (sq(ex) + sq(ey)) + sq(ez), b2 = (sq(bx) + sq(by)) + sq(bz);
  const T hw2 = h * sq(w);
  out[0] = (T)stage_src<ST>(P, DIR == 0 ? S_JX : S_JY)[k];
  if constexpr (DIR == 0) {
    out[1] = (T)stage_src<ST>(P, S_D)[k] * vx;
    out[2] = (bz * ey - by * ez) + hw2 * vx;
    out[3] = ((((-sq(ex)) - sq(bx)) + hw2 * sq(vx)) + T(0.5) * (e2 + b2)) + p;
    out[4] = ((-(ex * ey)) - bx * by) + (hw2 * vx) * vy;
    out[5] = ((-(ex * ez)) - bx * bz) + (hw2 * vx) * vz;
  } else {
    out[1] = (T)stage_src<ST>(P, S_D)[k] * vy;
    out[2] = (bx * ez - bz * ex) + hw2 * vy;
    out[3] = ((-(ex * ey)) - bx * by) + (hw2 * vx) * vy;
    out[4] = ((((-sq(ey)) - sq(by)) + hw2 * sq(vy)) + T(0.5) * (e2 + b2)) + p;
    out[5] = ((-(ey * ez)) - by * bz) + (hw2 * vy) * vz;
  }
}

// the face value from the split flux of cells i-1 .. i+2 (a: the flux, u:
// the field it is split with, sa = -1 for the fluxes the reference splits
// as -X +- U and negates afterwards)
template <typename T> __device__ inline T lax_face_value(int slop, const T* a, const T* u, T sa = T(1)) {
  const T p0 = sa * a[0] + u[0], p1 = sa * a[1] + u[1], p2 = sa * a[2] + u[2], p3 = sa * a[3] + u[3];
  const T m2 = sa * a[2] - u[2];
  const T l = p1 + T(0.5) * mcl_slope(p2 - p1, p1 - p0, slop);
  const T r = m2 - T(0.5) * mcl_slope(p3 - p2, p2 - p1, slop);
  return T(0.5) * (l + r);
}

template <typename T, typename ST> __device__ inline void lax_ld(const ST* __restrict__ a, const int64_t* k, T* v) {
#pragma unroll
  for (int c = 0; c < 4; c++) v[c] = (T)a[k[c]];
}

// the fluxes of the face between cell (i,j) and its +x (DIR 0) or +y
// (DIR 1) neighbour
template <int DIR, typename ST, typename T>
__device__ inline void lax_face(const Geom& g, const Planes& P, const Scheme& S, int i, int j, T* f) {
  int64_t k[4];
  T fl[4][6];
#pragma unroll
  for (int c = 0; c < 4; c++) {
    const int ii = DIR == 0 ? i + c - 1 : i, jj = DIR == 1 ? j + c - 1 : j;
    k[c] = g.at(ii, jj);
    lax_cell_fluxes<DIR, ST>(g, P, S, ii, jj, k[c], fl[c]);
  }
  T psi[4], phi[4], ex[4], ey[4], ez[4], bx[4], by[4], bz[4];
  lax_ld(stage_src<ST>(P, S_PSI), k, psi); lax_ld(stage_src<ST>(P, S_PHI), k, phi);
  lax_ld(stage_src<ST>(P, S_EX), k, ex); lax_ld(stage_src<ST>(P, S_EY), k, ey); lax_ld(stage_src<ST>(P, S_EZ), k, ez);
  lax_ld(stage_src<ST>(P, S_BX), k, bx); lax_ld(stage_src<ST>(P, S_BY), k, by); lax_ld(stage_src<ST>(P, S_BZ), k, bz);
  if constexpr (DIR == 0) {  // 15_lax_flow.f95:930-1180
    f[FX_EXPSI] = lax_face_value(S.slop, ex, psi);
    f[FX_BXPHI] = lax_face_value(S.slop, bx, phi);
    f[FX_PHIBX] = lax_face_value(S.slop, phi, bx);
    f[FX_EZBY] = -lax_face_value(S.slop, ez, by, T(-1));
    f[FX_EYBZ] = lax_face_value(S.slop, ey, bz);
    f[FX_PSIEX] = lax_face_value(S.slop, psi, ex);
    f[FX_BZEY] = lax_face_value(S.slop, bz, ey);
    f[FX_BYEZ] = -lax_face_value(S.slop, by, ez, T(-1));
  } else {
    f[FY_EYPSI] = lax_face_value(S.slop, ey, psi);
    f[FY_BYPHI] = lax_face_value(S.slop, by, phi);
    f[FY_EZBX] = lax_face_value(S.slop, ez, bx);
    f[FY_PHIBY] = lax_face_value(S.slop, phi, by);
    f[FY_EXBZ] = -lax_face_value(S.slop, ex, bz, T(-1));
    f[FY_BZEX] = -lax_face_value(S.slop, bz, ex, T(-1));
    f[FY_PSIEY] = lax_face_value(S.slop, psi, ey);
    f[FY_BXEZ] = lax_face_value(S.slop, bx, ez);
  }
  static_assert((int)FX_J == (int)FY_J && (int)FX_FSZ == (int)FY_FSZ, "fluid slots at the same place");
  const int us[6] = {S_Q, S_D, S_TAU, S_SX, S_SY, S_SZ};
#pragma unroll
  for (int t = 0; t < 6; t++) {
    T a[4], u[4];
#pragma unroll
    for (int c = 0; c < 4; c++) a[c] = fl[c][t];
    lax_ld(stage_src<ST>(P, us[t]), k, u);
    f[FX_J + t] = lax_face_value(S.slop, a, u);
  }
}

// both faces of the face pair (i,j): put_x(Fx(i+1/2,j)) as soon as the x
// face is solved, put_y(Fy(i,j+1/2)) as soon as the y face is; each flux
// array is dead after its put, which keeps the other solve's registers free
// of it.  YFIRST solves the y face first (the two solves are independent
// except under HLLE, whose y solve starts from the x solve's last iterate).
template <int ORD, int SOLVER, typename T, typename ST, bool YFIRST = false, bool STAGE_KIN = true, typename PutX,
          typename PutY>
__device__ __forceinline__ void face_pair(const Geom& g, const Planes& P, const Scheme& S, const StatusRef& st, int i,
                                          int j, PutX put_x, PutY put_y) {
  static_assert(!(YFIRST && SOLVER == 6), "the HLLE y solve needs the x solve first");
  const int64_t c = g.at(i, j);
  const Cell cc = cell_of(g, i, j);
  if constexpr (SOLVER == 3 || SOLVER == 4) {
    // HLLE / HLLC + MC limiter: x solve first (the y solve starts from its last iterate)
    T f[FX_N > FY_N ? FX_N : FY_N];
    const bool seed = S.hllc_seed_ref != 0;
    T xseed = T(0), vlast = T(0);
    Side<T> sl, sr;
    if (seed) {
      mcl_one<F_EX, 1, STAGE_KIN, ST>(P, S.slop, cc, sl, sr);
      mcl_one<F_EZ, 1, STAGE_KIN, ST>(P, S.slop, cc, sl, sr);
      mcl_one<F_BX, 1, STAGE_KIN, ST>(P, S.slop, cc, sl, sr);
      mcl_one<F_BZ, 1, STAGE_KIN, ST>(P, S.slop, cc, sl, sr);
      xseed = hlle_y_ery<T, true>(sl, sr);
    }
    mcl_sides<0, STAGE_KIN, ST>(P, S, cc, sl, sr);
    int code = SOLVER == 3 ? hlle_mcl_face<0>((T)S.gamma, sl, sr, f, seed, xseed, vlast)
                           : hllc_x<T, true>(sl, sr, f, seed, xseed, &vlast);
    if (code) report(st, code, i, j);
    put_x(f);
    mcl_sides<1, STAGE_KIN, ST>(P, S, cc, sl, sr);
    T unused;
    code = SOLVER == 3 ? hlle_mcl_face<1>((T)S.gamma, sl, sr, f, seed, vlast, unused)
                       : hllc_y<T, true>(sl, sr, f, seed, vlast);
    if (code) report(st, code, i, j);
    put_y(f);
    return;
  }
  if constexpr (SOLVER == 1 || SOLVER == 2) {  // second-order solvers: the faces are independent
    T f[FX_N > FY_N ? FX_N : FY_N];
    auto face = [&](auto dir) {
      constexpr int D = decltype(dir)::value;
      if constexpr (SOLVER == 1) lax_face<D, ST>(g, P, S, i, j, f);
      else mcl_face<D, STAGE_KIN, ST>(P, S, cc, f);
      if constexpr (D == 0) put_x(f);
      else put_y(f);
    };
    if constexpr (YFIRST) {
      face(std::integral_constant<int, 1>());
      face(std::integral_constant<int, 0>());
    } else {
      face(std::integral_constant<int, 0>());
      face(std::integral_constant<int, 1>());
    }
    return;
  }
  Side<T> xl, xr, yl, yr;
  // kinematics of both faces first: the fallbacks couple them
  face_fields<ORD, F_VX, F_PSI, 0, STAGE_KIN, ST>(P, cc, xl, xr);
  face_fields<ORD, F_VX, F_PSI, 1, STAGE_KIN, ST>(P, cc, yl, yr);
  // superluminal fallback, 16_hll_flow_mpx.f95:1392-1461 (same in hllc;
  // hlle only prints, 16_hlle_flow_mpx.f95:2270-2300)
  if (SOLVER != 6) {
    T v2xl = (sq(xl.vx) + sq(xl.vy)) + sq(xl.vz);
    T v2xr = (sq(xr.vx) + sq(xr.vy)) + sq(xr.vz);
    T v2yl = (sq(yl.vx) + sq(yl.vy)) + sq(yl.vz);
    T v2yr = (sq(yr.vx) + sq(yr.vy)) + sq(yr.vz);
    if (v2xl >= T(1) || v2xr >= T(1) || v2yl >= T(1) || v2yr >= T(1)) {
      const int64_t cm = g.at(i - 1, j), cj = g.at(i, j - 1);
      xl.vx = (T)P.p[P_VX][c]; xl.vy = (T)P.p[P_VY][c]; xl.vz = (T)P.p[P_VZ][c];
      xr.vx = (T)P.p[P_VX][cm]; xr.vy = (T)P.p[P_VY][cm]; xr.vz = (T)P.p[P_VZ][cm];
      yl.vx = (T)P.p[P_VX][c]; yl.vy = (T)P.p[P_VY][c]; yl.vz = (T)P.p[P_VZ][c];
      yr.vx = (T)P.p[P_VX][cj]; yr.vy = (T)P.p[P_VY][cj]; yr.vz = (T)P.p[P_VZ][cj];
    }
  }
  if (SOLVER == 7) {  // density fix-up, 16_hllc_flow_mpx.f95:2663-2693
    if (yl.rho < T(0) || yr.rho < T(0) || xl.rho < T(0) || xr.rho < T(0)) {
      T rc = (T)(0.1 * P.p[P_RHO][c]);
      if (yl.rho < T(0)) yl.rho = rc;
      else if (yr.rho < T(0)) yr.rho = rc;
      else if (xl.rho < T(0)) xl.rho = rc;
      else xr.rho = rc;
    }
  }
  constexpr bool HW = SOLVER == 6;
  // HLLE: first Newton point of the x contact solve in the reference build
  // is the y face's (E x B)_y; that of the y solve is the x solve's last iterate
  T seed_x = T(0), seed_y = T(0);
  if (SOLVER == 6 && S.hllc_seed_ref) {
    face_fields<ORD, F_EX, F_EX + 1, 1, STAGE_KIN, ST>(P, cc, yl, yr);
    face_fields<ORD, F_EZ, F_EZ + 1, 1, STAGE_KIN, ST>(P, cc, yl, yr);
    face_fields<ORD, F_BX, F_BX + 1, 1, STAGE_KIN, ST>(P, cc, yl, yr);
    face_fields<ORD, F_BZ, F_BZ + 1, 1, STAGE_KIN, ST>(P, cc, yl, yr);
    seed_x = hlle_y_ery(yl, yr);
  }
  auto xface = [&]() {
    face_fields<ORD, F_PSI, F_NQ, 0, STAGE_KIN, ST>(P, cc, xl, xr);
    side_physics<0, HW>((T)S.gamma, xl);
    side_physics<0, HW>((T)S.gamma, xr);
    T f[FX_N];
    if (SOLVER == 7) {
      int code = hllc_x(xl, xr, f, S.hllc_seed_ref != 0);
      if (code) report(st, code, i, j);
    } else if (SOLVER == 6) {
      int code = hlle_face<0>((T)S.gamma, xl, xr, f, S.hllc_seed_ref != 0, seed_x, seed_y);
      if (code) report(st, code, i, j);
    } else {
      hll_x(xl, xr, f);
    }
    put_x(f);
  };
  auto yface = [&]() {
    face_fields<ORD, F_PSI, F_NQ, 1, STAGE_KIN, ST>(P, cc, yl, yr);
    side_physics<1, HW>((T)S.gamma, yl);
    side_physics<1, HW>((T)S.gamma, yr);
    T f[FY_N];
    if (SOLVER == 7) {
      int code = hllc_y(yl, yr, f, S.hllc_seed_ref != 0);
      if (code) report(st, code, i, j);
    } else if (SOLVER == 6) {
      T unused;
      int code = hlle_face<1>((T)S.gamma, yl, yr, f, S.hllc_seed_ref != 0, seed_y, unused);
      if (code) report(st, code, i, j);
    } else {
      hll_y(yl, yr, f);
    }
    put_y(f);
  };
  if constexpr (YFIRST) {
    yface();
    xface();
  } else {
    xface();
    yface();
  }
}

// Waves per SIMD k_faces is built for (a register bound).  The MCL solvers
// need 197 VGPRs in FP64 and 125-143 in FP32 and the bound keeps the compiler
// from taking more than their waves leave; the other solvers fit their waves
// unbounded.
template <typename T, int SOLVER>
constexpr int faces_min_waves() {
  if constexpr (sizeof(T) == 8) return SOLVER >= 2 && SOLVER <= 4 ? 2 : 1;
  else return SOLVER >= 2 && SOLVER <= 4 ? 3 : 1;
}

template <int ORD, int SOLVER, typename T = double>
__global__ void __launch_bounds__(256, (faces_min_waves<T, SOLVER>())) FACES_WAVES
k_faces(Geom g, Planes P, Scheme S, StatusRef st) {
  if (halted(st)) return;
#if CUEVA_XCD_FACES
  int bx, by;
  if (!xcd_tile((g.imax + 2 + (int)blockDim.x - 1) / (int)blockDim.x,
                (g.jmax + 2 + (int)blockDim.y - 1) / (int)blockDim.y, bx, by))
    return;
#else
  const int bx = blockIdx.x, by = blockIdx.y;
#endif
  const int i = bx * blockDim.x + threadIdx.x - 1;
  const int j = by * blockDim.y + threadIdx.y - 1;
  if (i > g.imax || j > g.jmax) return;
  const int64_t c = g.at(i, j);
  face_pair<ORD, SOLVER, T, double>(
      g, P, S, st, i, j,
      [&](const T* f) {
#pragma unroll
        for (int t = 0; t < FX_N; t++) {
          if constexpr (sizeof(T) == 8) P.fx[t][c] = f[t];
          else P.fxf[t][c] = f[t];
        }
      },
      [&](const T* f) {
#pragma unroll
        for (int t = 0; t < FY_N; t++) {
          if constexpr (sizeof(T) == 8) P.fy[t][c] = f[t];
          else P.fyf[t][c] = f[t];
        }
      });
}

// ---------------------------------------------------------------------------
// Marching face kernel: reconstruction + Riemann solve + flux difference in
// one pass.  A block of MW wavefronts owns a strip of MARCH_COLS cell
// columns and a segment of `seg` cell rows (seg = MW m - 1).  Lane L of every
// wavefront computes the face pair of column i0 - 1 + L; per tile step the
// MW wavefronts take MW consecutive face rows.  Fx(i-1/2) is the left lane's x flux (a
// cross-lane shuffle of the registers the x solve leaves; HLLE, which must
// solve x first, goes through LDS); Fy(j-1/2) is the LDS row of the
// wavefront below, or for the lowest wavefront the previous tile step's top
// row.  Lane 0 only supplies Fx(i0-1/2), the segment's first face row only
// Fy(j0-1/2): each face is solved once per strip and segment, plus one
// column and one row per block.
//
// One barrier per tile step: the y rows alternate between two LDS buffers,
// and wavefront 0 copies the top row it needs next into its own row after
// the barrier; a buffer is rewritten two tile steps later, after every
// reader has passed the barrier in between.  HLLE keeps one buffer and
// takes a second barrier at the end of each tile step instead.
//   FINAL false: the stage right-hand side -> rhs[l] (17_fluxandsource.f95),
//                and the next stage's state (sumint, varint, electricvarint,
//                flowinit) -> sn, interior points;
//   FINAL true:  sumfin + varfin + electricfield of the last stage -> U^{n+1}
//                into rhs[l][0..13]; with C2P also the primitive recovery
//                of every point (-> pn, W) and, with args.stage0, the next
//                step's stage-0 state (-> sn); else the recovery pass follows.
// ---------------------------------------------------------------------------
constexpr int MARCH_COLS = 63;

inline int march_strips(const Geom& g) { return (g.imax + 1 + MARCH_COLS - 1) / MARCH_COLS; }

// the marching kernel's one argument (read through the kernel-argument
// pointer inside the loop, so it must be the first and only argument)
struct MarchArgs {
  Planes P;
  Geom g;
  Scheme S;
  int l, seg;
  StatusRef st;
  int stage0;  // C2P: also the next step's stage-0 state
  int strips, segs;  // the tiles of the launch
  int xcd;           // 1D grid in XCD-aware tile order (xcd_tile), else x = strip, y = segment
};
static_assert(offsetof(MarchArgs, P) == 0, "argument block layout");

// Waves per SIMD the marching kernel is built for, a register bound (the
// compiler spills past it).  Measured per step at 2048x4096:
//   FP64: 2 for every solver.  HLL, HLLE (with one y-row buffer, below) and
//     HLLC take 219-222 VGPRs with MP5, 242-246 with MP9, the MCL solvers
//     184-229: they fit 2 unbounded too (within 1 % of the same time).
//     Lax-Friedrichs takes 266 unbounded, 1 wave per SIMD: 7.00 ms, bounded
//     (12 spilled) 5.00.  3 waves (168 VGPRs) spill 22-40 under HLLC and ran
//     12 % slower;
//   FP32: 3 (144-162 VGPRs).  4 waves (128) spill 10-40: HLLC 3.42 against
//     3.29 ms, HLL 3.50 / 3.24, HLL + MC 3.16 / 2.97, HLLE + MP7 at 1024x2048
//     0.985 / 0.914.
template <typename T, int SOLVER>
constexpr int march_min_waves() {
  if constexpr (sizeof(T) == 8) return CUEVA_MARCH_F64_WAVES > 0 ? CUEVA_MARCH_F64_WAVES : 2;
  else return CUEVA_MARCH_F32_WAVES > 0 ? CUEVA_MARCH_F32_WAVES : 3;
}

// y-face row buffers: 2 (one barrier per tile step), or 1 for HLLE (a second
// barrier at the end of the tile step, before the rows are rewritten), whose
// x rows also pass through LDS: 63 KB per FP64 block instead of 91 KB, so
// that two blocks fit a CU's 160 KB
template <int SOLVER>
constexpr int march_y_buffers() {
  return SOLVER == 6 ? 1 : 2;
}

// Wavefronts per block = face rows per tile step: 4.  More re-read fewer halo
// rows (a tile step reads MW + 5), but the barriers then wait for more of
// them: HLLC + MP5 at 2048x4096 with 4 / 6 / 8 waves, FP64 4.99 / 6.24 / 5.41
// ms per step, FP32 3.29 / 4.01 / 3.57.
#ifndef CUEVA_MARCH_F32_BLOCK_WAVES
#define CUEVA_MARCH_F32_BLOCK_WAVES 4
#endif
#ifndef CUEVA_MARCH_F64_BLOCK_WAVES
#define CUEVA_MARCH_F64_BLOCK_WAVES 4
#endif
__host__ __device__ constexpr int march_block_waves(bool fp32, int solver) {
  return solver == 6 ? 4 : (fp32 ? CUEVA_MARCH_F32_BLOCK_WAVES : CUEVA_MARCH_F64_BLOCK_WAVES);
}

template <int ORD, int SOLVER, typename T, bool FINAL, bool C2P = false>
__global__ void __launch_bounds__(64 * march_block_waves(sizeof(T) == 4, SOLVER), (march_min_waves<T, SOLVER>()))
k_faces_march(MarchArgs args) {
  constexpr int MW = march_block_waves(sizeof(T) == 4, SOLVER);
  constexpr bool XLDS = SOLVER == 6;            // x solved first, its fluxes through LDS
  constexpr int YB = march_y_buffers<SOLVER>();
  __shared__ T fyb[YB][MW][FY_N][64];           // y-face rows of this (and the previous) tile step
  __shared__ T fyp[FY_N][64];                   // wavefront 0's row below: previous step's top row
  __shared__ T fxb[XLDS ? MW : 1][FX_N][64];    // x-face rows (HLLE)
  if (halted(args.st)) return;  // uniform over the launch: before any barrier
  int strip = (int)blockIdx.x, segment = (int)blockIdx.y;
  if (args.xcd && !xcd_tile(args.strips, args.segs, strip, segment)) return;  // uniform over the block
  const int lane = threadIdx.x, w = threadIdx.y;
  const int i = strip * MARCH_COLS - 1 + lane;
  const int jc0 = segment * args.seg;
  const int jend = min(jc0 + args.seg - 1, args.g.jmax);
  int b = 0;
  for (int jt = jc0 - 1; jt <= jend; jt += MW, b ^= YB - 1) {  // uniform over the block: the barriers below
    // The arguments (plane pointers, geometry, scheme constants) are read
    // again from the kernel's argument block every tile step rather than
    // held in scalar registers across the loop, where they do not fit and
    // spill into vector-register lanes: kept, the FP32 forms measured 8 %
    // slower at 2048x4096, FP64 HLLC the same.  FP64 HLL keeps them:
    // re-reading measured 16 % slower there.
    constexpr bool REREAD = sizeof(T) == 4 || SOLVER != 5;
    const __attribute__((address_space(4))) MarchArgs* ap =
        (const __attribute__((address_space(4))) MarchArgs*)__builtin_amdgcn_kernarg_segment_ptr();
    if constexpr (REREAD) asm volatile("" : "+s"(ap));
    const MarchArgs& A = REREAD ? *(const MarchArgs*)ap : args;
    const Planes& P = A.P;
    const Geom& g = A.g;
    const Scheme& S = A.S;
    const int l = A.l;
    const StatusRef& st = A.st;
    const int j = jt + w;
    const bool face_ok = i <= g.imax && j <= jend;
    T fx[FX_N];
    auto put_y = [&](const T* f) {
#pragma unroll
      for (int a = 0; a < FY_N; a++) fyb[b][w][a][lane] = f[a];
    };
    auto put_x = [&](const T* f) {
#pragma unroll
      for (int a = 0; a < FX_N; a++) {
        if constexpr (XLDS) fxb[w][a][lane] = f[a];
        else fx[a] = f[a];
      }
    };
    if (face_ok) {
      face_pair<ORD, SOLVER, T, T, !XLDS, false>(g, P, S, st, i, j, put_x, put_y);
    } else {
      T z[FX_N > FY_N ? FX_N : FY_N];
#pragma unroll
      for (int a = 0; a < (FX_N > FY_N ? FX_N : FY_N); a++) z[a] = T(0);
      put_x(z);
      put_y(z);
    }
    T dfx[FX_N];
    if constexpr (!XLDS) {
#pragma unroll
      for (int a = 0; a < FX_N; a++) {
        const T left = __shfl_up(fx[a], 1, 64);
        dfx[a] = ddx<T>(S, fx[a] - left);
      }
    }
    __syncthreads();
    const bool cell_ok = face_ok && lane >= 1 && j >= jc0;
    if (cell_ok) {
      if constexpr (XLDS) {
#pragma unroll
        for (int a = 0; a < FX_N; a++) dfx[a] = ddx<T>(S, fxb[w][a][lane] - fxb[w][a][lane - 1]);
      }
      T dfy[FY_N];
#pragma unroll
      for (int a = 0; a < FY_N; a++) {
        const T below = w == 0 ? fyp[a][lane] : fyb[b][w - 1][a][lane];
        dfy[a] = ddy<T>(S, fyb[b][w][a][lane] - below);
      }
      const int64_t k = g.at(i, j);
      // never with REC_PRIM = 1
      const Rhs r = rhs_of<T, false>(P, S, k, dfx, dfy, sizeof(T) == 4 && l == 0);
      if constexpr (!FINAL) {
        put_planes<R_N>(P.rhs[l], k, r.r, S.stream > 0);
        // the next stage's state of this point (pointwise in U^n and the
        // stage right-hand sides, the last of which is still in registers)
        double sv[S_N];
        stage_point(P, S, l + 1, k, false, P.p[P_VX][k], P.p[P_VY][k], P.p[P_VZ][k], P.p[P_EX][k], P.p[P_EY][k],
                    P.p[P_EZ][k], P.p[P_BX][k], P.p[P_BY][k], P.p[P_BZ][k], P.p[P_RHO][k], P.p[P_P][k],
                    P.p[P_PSI][k], P.p[P_PHI][k], P.p[P_Q][k], sv, &r);
        store_stage<sizeof(T) == 4>(P.sn, P.snf, k, sv, false, S.full != 0, S.stream > 0);
      } else {
        double nu[A_N];
        final_update_from(P, S, k, r, nu);
        put_planes<A_N>(P.rhs[l], k, nu, S.stream > 0);
        if constexpr (C2P) recover_point(P, S, st, i, j, k, nu, A.stage0);
      }
    }
    if (w == 0) {
#pragma unroll
      for (int a = 0; a < FY_N; a++) fyp[a][lane] = fyb[b][MW - 1][a][lane];
    }
    if constexpr (YB == 1) __syncthreads();  // every read of this step's rows before the next step's writes
    else if constexpr (XLDS) __builtin_amdgcn_wave_barrier();  // this step's fxb reads before the next step's writes
  }
}

// kernel of (rec_order, solver, stage kind), for a launch by pointer
template <typename T>
inline const void* march_kernel(int rec_order, int solver, bool final_stage, bool c2p) {
#define CUEVA_MK(O, SV)                                                                          \
  (final_stage ? (c2p ? reinterpret_cast<const void*>(&k_faces_march<O, SV, T, true, true>)      \
                      : reinterpret_cast<const void*>(&k_faces_march<O, SV, T, true, false>))    \
               : reinterpret_cast<const void*>(&k_faces_march<O, SV, T, false, false>))
  if (solver == 1) return CUEVA_MK(5, 1);  // second order: the MP order does not enter
  if (solver == 2) return CUEVA_MK(5, 2);
  if (solver == 3) return CUEVA_MK(5, 3);
  if (solver == 4) return CUEVA_MK(5, 4);
  switch (rec_order * 10 + solver) {
    case 55: return CUEVA_MK(5, 5);
    case 56: return CUEVA_MK(5, 6);
    case 57: return CUEVA_MK(5, 7);
    case 75: return CUEVA_MK(7, 5);
    case 76: return CUEVA_MK(7, 6);
    case 77: return CUEVA_MK(7, 7);
    case 95: return CUEVA_MK(9, 5);
    case 96: return CUEVA_MK(9, 6);
    case 97: return CUEVA_MK(9, 7);
    default: return nullptr;
  }
#undef CUEVA_MK
}

}  // namespace cueva
