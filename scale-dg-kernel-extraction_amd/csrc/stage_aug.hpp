// Stage kernels over augmented pencils (gfx950), one template for two
// precisions:
//  * mixed (HIP_MP): the 1D-operator contractions and the Lift run in FP32 with
//    FP32 accumulation; the state q, the face-flux jumps, the volume fluxes
//    q*u_d and the RK stage combination stay FP64; velocities are read from
//    FP32 copies;
//  * FP64 (HIP, tile candidates): the same data flow in FP64 throughout.
//
// For each direction d the sum-factorised derivative and that direction's two
// Lift faces form one product over the element's "pencils" r (node lines along
// d):
//   out_d(r, c) = sum_l E_d F_d(r, l) D(c, l)
//               + l-(c) flux(face d-, r) + l+(c) flux(face d+, r)
// i.e. A_d = [E_d F_d | flux_d- | flux_d+]  (pencils x (NQ + 2)),
//      B   = [D^T ; l- ; l+]                ((NQ + 2) x NQ), the same for every
// direction and element.  The reference's face-node order (Fmask,
// mod_mesh.f90:278-324) is the pencil order of the face's normal direction, so
// the Lift (tensorprod_Lift_hexahedral, mod_dg_optr_kernel.f90:262-288, in its
// tensor-product form) is two extra rows of the contraction
// (tensorprod_divlike_dirXYZ, mod_dg_optr_kernel.f90:197-258).  The three
// direction results are summed in FP64, dqdt = -((X + Y) + Z), and RK-combined
// in FP64 (main.f90:69-73).
//
// Two forms of the product give the same bits: an MFMA 16x16x4 adds its four
// products to the accumulator one after the other, k ascending, each fused and
// rounded, which is what a chain of FMAs in that order does (both precisions;
// no difference in 2.5e6 results each of random operands, denormals among
// them).
//  * stage_aug, one pencil per lane on the VALU, is the faster one almost
//    everywhere: the pencils never leave the registers, where the MFMA form
//    writes A to LDS, reads it, writes the product and reads that.  us per
//    launch at about 1.7e7 DOF, velocity fields, MFMA -> VALU: mixed p = 2
//    157 -> 140, p = 3 125 -> 113, p = 7 103 -> 96, p = 10 118 -> 104, p = 12
//    129 -> 115, p = 18 155 -> 143; FP64 p = 14 164 -> 152, p = 15 148 -> 143,
//    p = 17 243 -> 199, p = 18 241 -> 178, p = 19 302 -> 197.  Constant
//    velocity: mixed p = 3 112 -> 73, p = 7 79 -> 67, p = 12 91 -> 79; FP64
//    p = 19 168 -> 140.
//  * the MFMA one, direction by direction through one LDS area, where it is
//    faster (by_mfma): mixed p = 16, 17 (fields 140 against 177 and 137 against
//    158) and constant-velocity launches of the mixed form at p >= 16 (101
//    against 139, 104/127, 100/113, 110/130) and of FP64 at p = 16 (123/146),
//    and launches of few elements of the mixed form at p = 13..15 (stage_small).
//    Above p = 15 an element is five to seven wavefronts, and on four SIMDs the VALU
//    form's phases take as long as two of them, while the MFMA form's eight
//    wavefronts share the tiles.
#pragma once

#include <algorithm>
#include <atomic>

#include "contract.hpp"
#include "dgk_internal.hpp"

namespace dgk {

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef double f64x4 __attribute__((ext_vector_type(4)));

// Operand precision of the contraction GEMMs.
// Both MFMAs take A(row = lane%16, k = lane/16) and B(k = lane/16,
// col = lane%16); result value t of a lane lies in column lane%16 and row
// RSTRIDE_Q*(lane/16) + RSTRIDE_T*t (checked on the device for both).
struct PrecMixed {
  using vel_t = float;   // velocity copies read by the kernel
  using op_t = float;    // A, B operands in LDS / registers
  using acc_t = f32x4;   // 16x16 result, 4 values per lane
  static constexpr int RSTRIDE_Q = 4, RSTRIDE_T = 1;
  static __device__ __forceinline__ acc_t mfma(op_t a, op_t b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
};
struct PrecF64 {
  using vel_t = double;
  using op_t = double;
  using acc_t = f64x4;
  static constexpr int RSTRIDE_Q = 1, RSTRIDE_T = 4;
  static __device__ __forceinline__ acc_t mfma(op_t a, op_t b, acc_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
};

__device__ __forceinline__ int xcd_block_mp(int b, int n) {
  const int per = n >> 3, rem = n & 7;
  const int x = b & 7, local = b >> 3;
  return x * per + min(x, rem) + local;
}

__device__ __forceinline__ int64_t uniform_mp(int64_t v) {
  const int lo = __builtin_amdgcn_readfirstlane((int)(v & 0xffffffff));
  const int hi = __builtin_amdgcn_readfirstlane((int)(v >> 32));
  return (int64_t)(((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo);
}

// Whether a shape's product runs on the MFMA (above).
template <class P, int NQ, bool SEQ, bool CVEL>
constexpr bool by_mfma() {
  if (!SEQ || NQ <= 16) return false;
  return sizeof(typename P::op_t) == 4 ? CVEL || NQ <= 18 : CVEL && NQ == 17;
}

// MFMA form: one element per block, one LDS area of A, a direction at a time.
// The block is eight wavefronts, two per SIMD, the idle lanes taking tiles,
// and held to 4 waves per SIMD, so two blocks share a CU (per launch at about
// 1.7e7 DOF, p = 16..19, against 5..7 wavefronts and no cap: mixed
// 171/153/180/209 -> 151/166/176/193 us).
template <class P, int NQ>
struct Seq {
  static constexpr int NQ2 = NQ * NQ;
  static constexpr int NP = NQ2 * NQ;
  static constexpr int THREADS = 512;
  static constexpr int WAVES = THREADS / 64;
  static constexpr int ROWS = ((NQ2 + 15) / 16) * 16;      // pencils per direction
  static constexpr int MTILES = ROWS / 16;
  static constexpr int NT = (NQ + 15) / 16;                // 16-wide column tiles of B
  static constexpr int KAUG = NQ + 2;
  static constexpr int KSTEPS = (KAUG + 3) / 4;
  // Operands per row of A in LDS: KAUG rounded up to odd, so that the lanes
  // that write and read A at a stride of one row (the y and z pencils, the
  // flux columns, the 16 rows of an MFMA operand read) spread over the banks
  // (rows of 4 KSTEPS: 79% of the LDS cycles were conflicts at p = 18).  The K
  // padding is not stored: the operand read puts zeros there.
  static constexpr int STRIDE = KAUG | 1;
  static constexpr int AREA = ROWS * STRIDE;               // A of one direction
  static constexpr size_t LDS_BYTES = (size_t)(AREA + 4) * sizeof(typename P::op_t);
  static constexpr size_t LDS_BYTES_ONCE = (size_t)(3 * AREA + 4) * sizeof(typename P::op_t);
  static constexpr int JPW = (MTILES + WAVES - 1) / WAVES;
};

// VALU form: EPB elements per block, a lane per pencil.
template <class P, int NQ, int EPB, bool CVEL>
struct Aug {
  using vel_t = typename P::vel_t;
  using op_t = typename P::op_t;
  static constexpr int NQ2 = NQ * NQ;
  static constexpr int LANES = EPB * NQ2, THREADS = ((LANES + 63) / 64) * 64;
  // row, slab and element strides: an odd row spreads the lanes of an x pencil
  // read (a row apart) over the banks
  static constexpr int S1 = NQ | 1, S2 = NQ * S1, SE = NQ * S2, BUF = EPB * SE;
  // above p = 7 the v, w and q0 columns are loaded a phase before their use
  static constexpr bool LATE = NQ > 8;
  static constexpr size_t LDS_BYTES = (size_t)BUF * (sizeof(double) + (CVEL ? 0 : sizeof(vel_t)));
  // non-temporal RK base and output, as stage_pencil's
  static constexpr bool NT = !CVEL && (NQ2 % 16 == 0 || NQ > 9);
};

// A shape as launched: block size, LDS, registers.
template <class P, int NQ, int EPB, bool SEQ, bool CVEL>
struct Shape {
  static constexpr bool MFMA = by_mfma<P, NQ, SEQ, CVEL>();
  static constexpr int THREADS = MFMA ? Seq<P, NQ>::THREADS : Aug<P, NQ, EPB, CVEL>::THREADS;
  static constexpr size_t LDS_BYTES =
      MFMA ? Seq<P, NQ>::LDS_BYTES : Aug<P, NQ, EPB, CVEL>::LDS_BYTES;
  // 4 waves per SIMD also for the mixed constant-velocity form at p = 15, which
  // lands at 131 VGPRs otherwise (73.2 -> 71.7 us per launch)
  static constexpr int MIN_WAVES_EU =
      MFMA || (CVEL && NQ == 16 && EPB == 1 && sizeof(typename P::op_t) == 4) ? 4 : 1;
};

// Shapes whose face normals are tested at run time, in one instantiation for
// both: the direction-by-direction and the mixed one-wavefront ones.  The
// others have a compile-time form each.
template <class P, int NQ, int EPB, bool SEQ>
constexpr bool ax_runtime() {
  return SEQ || (sizeof(typename P::op_t) == 4 && EPB * NQ * NQ <= 64);
}

// Candidate kinds per order: for Nq^2 <= 64 one, two or four wavefronts of
// whole elements, then one wavefront direction by direction; above, one
// element, two elements, and one element direction by direction; above
// p = 15 one element, all at once or direction by direction.  The candidates
// 0, 1, ... are the kinds of an order that kind_ok keeps (per-order defaults in
// kMpDefault and kF64Default).  In the VALU form all at once and direction by
// direction are one algorithm; the second tests the face normals at run time where
// velocity fields are read (with a constant velocity they are the same machine code).
// Both stay: candidates are numbered and selected by callers.
constexpr int kKinds = 4;
template <int NQ>
constexpr int kind_epb(int k) {
  constexpr int NQ2 = NQ * NQ;
  if (NQ2 <= 64) {
    const int waves = k == 1 ? 2 : k == 2 ? 4 : 1;
    const int e = 64 * waves / NQ2;
    return e < 1 ? 1 : e;
  }
  return k == 1 ? 2 : 1;
}
template <int NQ>
constexpr bool kind_seq(int k) {
  return NQ * NQ > 64 ? k == 2 : k == 3;
}
// The kinds an order has.  The last line is the LDS that three areas of A all at once
// (one direction by direction) take on the MFMA, which the VALU form does not
// allocate: it keeps the candidates' numbers what they have been (all at once above
// p = 15: FP64 up to p = 17, mixed up to p = 19).
template <class P, int NQ>
constexpr bool kind_ok(int k) {
  if (NQ * NQ > 64 && k == 3) return false;
  if (NQ > kMaxNqValu && k == 1) return false;  // above p = 15: one element per workgroup
  const int rows = ((kind_epb<NQ>(k) * NQ * NQ + 15) / 16) * 16;
  return (size_t)(kind_seq<NQ>(k) ? 1 : 3) * rows * (NQ + 2) * sizeof(typename P::op_t) <=
         160 * 1024;
}
template <class P, int NQ>
constexpr int ncand() {
  return (int)kind_ok<P, NQ>(0) + (int)kind_ok<P, NQ>(1) + (int)kind_ok<P, NQ>(2) +
         (int)kind_ok<P, NQ>(3);
}
// kind of candidate c (-1 if none)
template <class P, int NQ>
constexpr int kind_of(int c) {
  int n = 0;
  for (int k = 0; k < kKinds; ++k) {
    if (!kind_ok<P, NQ>(k)) continue;
    if (n == c) return k;
    ++n;
  }
  return -1;
}

// One 16-pencil tile: A rows (STRIDE operands apart) from `tile`, B (NT column
// tiles) in registers; all A values are read before any result overwrites the
// tile's first NQ columns.  `left` = KAUG - kq * KSTEPS: operands of this
// lane's K range from there on are padding, read as whatever follows the row
// and replaced by zero.
template <class P, int KSTEPS, int KAUG, int STRIDE, int NQ, int NT>
__device__ __forceinline__ void mfma_tile(typename P::op_t *tile,
                                          const typename P::op_t (&bop)[NT][KSTEPS], int rd,
                                          int wr, int col, int left) {
  typename P::op_t a[KSTEPS];
#pragma unroll
  for (int ks = 0; ks < KSTEPS; ++ks) {
    const typename P::op_t v = tile[rd + ks];
    a[ks] = 3 * KSTEPS + ks < KAUG || ks < left ? v : (typename P::op_t)0;
  }
  typename P::acc_t acc[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    acc[nt] = typename P::acc_t{0, 0, 0, 0};
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) acc[nt] = P::mfma(a[ks], bop[nt][ks], acc[nt]);
  }
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    if (16 * nt + col < NQ) {
#pragma unroll
      for (int t4 = 0; t4 < 4; ++t4) tile[wr + 16 * nt + t4 * P::RSTRIDE_T * STRIDE] = acc[nt][t4];
    }
  }
}

// ---- the VALU form ---------------------------------------------------------
// The order in which the MFMA adds the products of a pencil (mfma_tile): step ks
// adds k = 0..3, which are the rows kq KSTEPS + ks, kq = 0..3.
template <int NQ>
struct RowsMfma {
  static constexpr int N = NQ + 2, KSTEPS = (N + 3) / 4;
  static constexpr int l(int n) {
    int m = 0;
    for (int ks = 0; ks < KSTEPS; ++ks)
      for (int kq = 0; kq < 4; ++kq) {
        const int r = kq * KSTEPS + ks;
        if (r < N && m++ == n) return r;
      }
    return 0;
  }
};

template <class P, int NQ, int EPB, bool AXR, bool AXAL, bool CVEL, bool GU>
__device__ __forceinline__ void
stage_aug(const double *__restrict__ q_, const double *q0_,
          const typename P::vel_t *__restrict__ u_, const typename P::vel_t *__restrict__ v_,
          const typename P::vel_t *__restrict__ w_, double *out_,
          const int32_t *__restrict__ nbr_, const int32_t *__restrict__ vmapP_,
          const typename P::op_t *__restrict__ D_, const typename P::op_t *__restrict__ ell_,
          const double *__restrict__ geo_, const uint32_t *__restrict__ geoid_,
          const int32_t *__restrict__ order_, const int64_t Ne_, const double ca_,
          const double cb_, const double dt_, const int mode_, const int axis_aligned_,
          const int dt_geo_, const int rev_, const int64_t zp_) {
  using C = Aug<P, NQ, EPB, CVEL>;
  using vel_t = typename P::vel_t;
  using op_t = typename P::op_t;
  constexpr int NQ2 = C::NQ2, NP = NQ2 * NQ, NFT = 6 * NQ2;
  constexpr int S1 = C::S1, S2 = C::S2;
  constexpr bool HALF = sizeof(op_t) == 4;  // X and Y both fit in q's buffer
  extern __shared__ double smem_mp[];
  const int tid = threadIdx.x;
  const int64_t slot0 = (int64_t)xcd_block_mp(blockIdx.x, gridDim.x) * EPB;
  const bool lane_ok = tid < C::LANES;
  const int el = lane_ok ? tid / NQ2 : 0;
  const int ij = lane_ok ? tid - el * NQ2 : 0;
  const int i = ij % NQ, j = ij / NQ;
  const int64_t slot = slot0 + el;
  const bool active = lane_ok && slot < Ne_;
  int64_t e;
  if (EPB == 1) {
    e = slot < Ne_ ? slot_element(slot, Ne_, order_, rev_, zp_) : 0;
    e = uniform_mp(e);
  } else {
    e = active ? slot_element(slot, Ne_, order_, rev_, zp_) : 0;
  }
  const int64_t ebase = e * NP, base = ebase + ij;
  const bool rk = mode_ == 1;
  const bool use_q0 = rk && ca_ != 0.0;
  const bool axal = CVEL || (AXR ? axis_aligned_ != 0 : AXAL);  // launch_shape

  double qc[NQ], qP[6], q0v[NQ];
  vel_t vP[6], uc[NQ], vc[NQ], wc[NQ];
  auto load_col = [&](vel_t (&c)[NQ], const vel_t *p) {
    if constexpr (!CVEL) {
#pragma unroll
      for (int k = 0; k < NQ; ++k) c[k] = p[base + k * NQ2];
    }
  };
  auto load_q = [&]() {
#pragma unroll
    for (int k = 0; k < NQ; ++k) qc[k] = q_[base + k * NQ2];
  };
  auto load_q0 = [&]() {
    if (use_q0) {
#pragma unroll
      for (int k = 0; k < NQ; ++k)
        q0v[k] = C::NT ? __builtin_nontemporal_load(q0_ + base + k * NQ2) : q0_[base + k * NQ2];
    }
  };
  auto load_trace = [&](int f, int64_t pidx) {
    qP[f] = q_[pidx];
    if constexpr (!CVEL) vP[f] = (kFaceAxis[f] == 0 ? u_ : kFaceAxis[f] == 1 ? v_ : w_)[pidx];
  };
  if (active) {
    constexpr int ford[6] = {3, 1, 0, 2, 4, 5};  // in the order of use
    if (vmapP_) {
      load_q();
      load_col(uc, u_);
#pragma unroll
      for (int n = 0; n < 6; ++n) {
        const int f = ford[n];
        load_trace(f, (int64_t)vmapP_[e * NFT + f * NQ2 + ij]);
      }
    } else {
      int32_t nb[6];
#pragma unroll
      for (int f = 0; f < 6; ++f) nb[f] = nbr_[e * 6 + f];
      load_q();
      load_col(uc, u_);
#pragma unroll
      for (int n = 0; n < 6; ++n) {
        const int f = ford[n];
        load_trace(f, (int64_t)nb[f] * NP + nbr_face_node(f, i, j, NQ));
      }
    }
    if constexpr (!C::LATE) {
      load_col(vc, v_);
      load_col(wc, w_);
      load_q0();
    }
  }
  double *const B1 = smem_mp + el * C::SE;
  vel_t *const B2 = (vel_t *)(smem_mp + C::BUF) + el * C::SE;
  op_t *const X = (op_t *)B1, *const Y = X + (HALF ? C::SE : 0);
  const int zo = i + j * S1, xo = i * S1 + j * S2, yo = i + j * S2;
  const double *g_lane = geo_ + (active && geoid_ ? (int64_t)geoid_[e] * kGeoStride : 0);
  if constexpr (EPB == 1) g_lane = geo_ + (geoid_ ? (int64_t)geoid_[e] * kGeoStride : 0);

  auto body = [&](const double *__restrict__ g) {
    vel_t cv[3] = {(vel_t)0, (vel_t)0, (vel_t)0};
    if constexpr (CVEL) {
      cv[0] = (vel_t)g[kGeoVel];
      cv[1] = (vel_t)g[kGeoVel + 1];
      cv[2] = (vel_t)g[kGeoVel + 2];
    }
    auto face_flux = [&](int f, double qm, vel_t vm) -> op_t {
      double VelM, VelP;
      if (axal) {
        const int ax = kFaceAxis[f];
        const double na = g[kGeoNormal + 3 * f + ax];
        VelM = (double)vm * na;
        VelP = (double)(CVEL ? cv[ax] : vP[f]) * na;
      } else {
        // general normals: all three components on both sides
        const int64_t m = ebase + own_face_node(f, i, j, NQ);
        const int64_t pidx = vmapP_ ? (int64_t)vmapP_[e * NFT + f * NQ2 + ij]
                                    : (int64_t)nbr_[e * 6 + f] * NP + nbr_face_node(f, i, j, NQ);
        const double n1 = g[kGeoNormal + 3 * f], n2 = g[kGeoNormal + 3 * f + 1],
                     n3 = g[kGeoNormal + 3 * f + 2];
        VelM = (double)u_[m] * n1 + (double)v_[m] * n2 + (double)w_[m] * n3;
        VelP = (double)u_[pidx] * n1 + (double)v_[pidx] * n2 + (double)w_[pidx] * n3;
      }
      const double alpha = 0.5 * fabs(VelP + VelM);
      return (op_t)(0.5 * g[kGeoFscale + f] * (qP[f] * VelP - qm * VelM - alpha * (qP[f] - qm)));
    };
    op_t a[NQ + 2], acc[NQ];
    double qy[NQ];
    // ---- x pencils
    if (active) {
#pragma unroll
      for (int k = 0; k < NQ; ++k) {
        B1[zo + k * S2] = qc[k];
        if constexpr (!CVEL) B2[zo + k * S2] = uc[k];
      }
    }
    __syncthreads();
    {
      double qx[NQ];
      if (active) {
#pragma unroll
        for (int l = 0; l < NQ; ++l) qx[l] = B1[xo + l];
#pragma unroll
        for (int l = 0; l < NQ; ++l) qy[l] = B1[yo + l * S1];
      }
      if (active) {
        const double Ex = g[kGeoEscale];
        vel_t v0 = cv[0], v1 = cv[0];
#pragma unroll
        for (int l = 0; l < NQ; ++l) {
          const vel_t vel = CVEL ? cv[0] : B2[xo + l];
          if (l == 0) v0 = vel;
          if (l == NQ - 1) v1 = vel;
          a[l] = (op_t)(Ex * (qx[l] * (double)vel));
        }
        a[NQ] = face_flux(3, qx[0], v0);
        a[NQ + 1] = face_flux(1, qx[NQ - 1], v1);
        if constexpr (C::LATE) load_col(vc, v_);
        Contract<op_t, NQ, RowsMfma<NQ>>().run(D_, ell_, a, acc);
      }
    }
    __syncthreads();
    if (active) {
#pragma unroll
      for (int l = 0; l < NQ; ++l) X[xo + l] = acc[l];
      if constexpr (!CVEL) {
#pragma unroll
        for (int k = 0; k < NQ; ++k) B2[zo + k * S2] = vc[k];
      }
    }
    __syncthreads();
    // ---- y pencils
    if (active) {
      const double Ey = g[kGeoEscale + 1];
      vel_t v0 = cv[1], v1 = cv[1];
#pragma unroll
      for (int l = 0; l < NQ; ++l) {
        const vel_t vel = CVEL ? cv[1] : B2[yo + l * S1];
        if (l == 0) v0 = vel;
        if (l == NQ - 1) v1 = vel;
        a[l] = (op_t)(Ey * (qy[l] * (double)vel));
      }
      a[NQ] = face_flux(0, qy[0], v0);
      a[NQ + 1] = face_flux(2, qy[NQ - 1], v1);
      if constexpr (C::LATE) {
        load_col(wc, w_);
        load_q0();
      }
      Contract<op_t, NQ, RowsMfma<NQ>>().run(D_, ell_, a, acc);
#pragma unroll
      for (int c = 0; c < NQ; ++c) {
        if constexpr (HALF) Y[yo + c * S1] = acc[c];
        else X[yo + c * S1] = X[yo + c * S1] + acc[c];
      }
    }
    __syncthreads();
    // ---- z pencils, RK update (FP64)
    if (active) {
      const double Ez = g[kGeoEscale + 2];
#pragma unroll
      for (int l = 0; l < NQ; ++l) a[l] = (op_t)(Ez * (qc[l] * (double)(CVEL ? cv[2] : wc[l])));
      a[NQ] = face_flux(4, qc[0], CVEL ? cv[2] : wc[0]);
      a[NQ + 1] = face_flux(5, qc[NQ - 1], CVEL ? cv[2] : wc[NQ - 1]);
      Contract<op_t, NQ, RowsMfma<NQ>>().run(D_, ell_, a, acc);
      double res[NQ];
#pragma unroll
      for (int k = 0; k < NQ; ++k) {
        double xy = (double)X[zo + k * S2];
        if constexpr (HALF) xy += (double)Y[zo + k * S2];
        res[k] = -(xy + (double)acc[k]);
      }
      if (rk) {
        const double dtv = dt_geo_ ? g[kGeoDt] : dt_;
#pragma unroll
        for (int k = 0; k < NQ; ++k) {
          const double upd = cb_ * (qc[k] + dtv * res[k]);
          res[k] = use_q0 ? ca_ * q0v[k] + upd : upd;
        }
      }
#pragma unroll
      for (int k = 0; k < NQ; ++k) {
        if constexpr (C::NT) __builtin_nontemporal_store(res[k], out_ + base + (int64_t)k * NQ2);
        else out_[base + (int64_t)k * NQ2] = res[k];
      }
    }
  };
  if constexpr (GU) {
    body(geo_);
  } else if constexpr (EPB > 1) {
    const double *gb = block_record(slot0, EPB, Ne_, geo_, geoid_, order_, rev_, zp_, dt_geo_);
    if (gb) body(gb);
    else body(g_lane);
  } else {
    body(g_lane);
  }
}

// ---- the kernel; the MFMA form, direction by direction ------------------------
//   1. the lane loads its q column (FP64), the own traces of the x/y faces and
//      the neighbour traces straight into registers (coalesced along (i,j));
//   2. FP64 upwind fluxes; per direction, FP64 volume fluxes E_d q u_d (the
//      velocity column loaded when its direction comes up), each rounded once
//      to the operand precision, written into A in LDS, one pencil per row;
//   3. MFMA over 16-pencil tiles; K is permuted so that lane (col, kq) keeps
//      rows l = kq*KSTEPS + ks of B in registers and reads A at fixed offsets
//      from its own base; the result overwrites the tile's rows in place;
//   4. the direction results are summed in FP64 and RK-combined.
// ONCE: the three directions at once, each in an LDS area of its own, their velocity
// columns loaded with the rest.
template <class P, int NQ, bool CVEL, bool ONCE>
__device__ __forceinline__ void
stage_seq(const double *q_, const double *q0_,
          const typename P::vel_t *u_, const typename P::vel_t *v_,
          const typename P::vel_t *w_, double *out_,
          const int32_t *nbr_, const int32_t *vmapP_,
          const typename P::op_t *D_, const typename P::op_t *ell_,
          const double *geo_, const uint32_t *geoid_,
          const int32_t *order_, const int64_t Ne_, const double ca_,
          const double cb_, const double dt_, const int mode_, const int axis_aligned_,
          const int dt_geo_, const int rev_, const int64_t zp_) {
  using C = Seq<P, NQ>;
  using vel_t = typename P::vel_t;
  using op_t = typename P::op_t;
  constexpr int NQ2 = C::NQ2, NP = C::NP, NFT = 6 * NQ2, KSTEPS = C::KSTEPS;
  constexpr int KAUG = C::KAUG, STRIDE = C::STRIDE;
  extern __shared__ double smem_mp[];
  op_t *const As = (op_t *)smem_mp;

  const int tid = threadIdx.x;
  const int wave = tid >> 6, lane = tid & 63;
  const int64_t slot = (int64_t)xcd_block_mp(blockIdx.x, gridDim.x);
  const bool lane_ok = tid < NQ2;
  const int ij = lane_ok ? tid : 0;
  const int i = ij % NQ, j = ij / NQ;
  const bool active = lane_ok && slot < Ne_;
  int64_t e = slot < Ne_ ? slot_element(slot, Ne_, order_, rev_, zp_) : 0;
  e = uniform_mp(e);
  const double *__restrict__ g = geo_ + (geoid_ ? (int64_t)geoid_[e] * kGeoStride : 0);
  const int64_t ebase = e * NP;
  const int64_t base = ebase + ij;
  const bool rk = mode_ == 1;
  const bool use_q0 = rk && ca_ != 0.0;
  const bool axal = CVEL || axis_aligned_ != 0;  // launch_shape
  const vel_t *const velp[3] = {u_, v_, w_};
  vel_t cv[3] = {(vel_t)0, (vel_t)0, (vel_t)0};
  if constexpr (CVEL) {
    cv[0] = (vel_t)g[kGeoVel];
    cv[1] = (vel_t)g[kGeoVel + 1];
    cv[2] = (vel_t)g[kGeoVel + 2];
  }
  auto nbr_at = [&](int f) -> int64_t {
    return vmapP_ ? (int64_t)vmapP_[e * NFT + f * NQ2 + ij]
                  : (int64_t)nbr_[e * 6 + f] * NP + nbr_face_node(f, i, j, NQ);
  };

  // ---- 1. loads straight into registers ------------------------------------
  double qc[NQ], qM[4], qP[6];
  vel_t w0 = cv[2], w1 = cv[2], vM[4], vP[6];  // velocity component along the face axis
  vel_t cols[3][NQ];                           // ONCE: the velocity columns
  if (active) {
#pragma unroll
    for (int k = 0; k < NQ; ++k) qc[k] = q_[base + k * NQ2];
    if constexpr (ONCE && !CVEL) {
#pragma unroll
      for (int d = 0; d < 3; ++d)
#pragma unroll
        for (int k = 0; k < NQ; ++k) cols[d][k] = velp[d][base + k * NQ2];
    }
    if constexpr (!CVEL) {
      w0 = w_[base];
      w1 = w_[base + (NQ - 1) * NQ2];
    }
#pragma unroll
    for (int f = 0; f < 4; ++f) {  // own traces of the x and y faces
      const int64_t m = ebase + own_face_node(f, i, j, NQ);
      qM[f] = q_[m];
      vM[f] = CVEL ? cv[kFaceAxis[f]] : (kFaceAxis[f] == 0 ? u_ : v_)[m];
    }
#pragma unroll
    for (int f = 0; f < 6; ++f) {
      const int64_t pidx = nbr_at(f);
      qP[f] = q_[pidx];
      vP[f] = CVEL ? cv[kFaceAxis[f]]
                   : (kFaceAxis[f] == 0 ? u_ : kFaceAxis[f] == 1 ? v_ : w_)[pidx];
    }
  }

  // ---- 2a. FP64 upwind fluxes -------------------------------------------------
  op_t fl[6];
  auto face_flux = [&](int f) {
    const double qm = f == 4 ? qc[0] : f == 5 ? qc[NQ - 1] : qM[f];
    double VelM, VelP;
    if (axal) {
      const int ax = kFaceAxis[f];
      const double na = g[kGeoNormal + 3 * f + ax];
      const vel_t vm = f == 4 ? w0 : f == 5 ? w1 : vM[f];
      VelM = (double)vm * na;
      VelP = (double)vP[f] * na;
    } else {
      // general normals: all three components on both sides
      const int64_t m = ebase + own_face_node(f, i, j, NQ);
      const int64_t pidx = nbr_at(f);
      const double n1 = g[kGeoNormal + 3 * f], n2 = g[kGeoNormal + 3 * f + 1],
                   n3 = g[kGeoNormal + 3 * f + 2];
      VelM = (double)u_[m] * n1 + (double)v_[m] * n2 + (double)w_[m] * n3;
      VelP = (double)u_[pidx] * n1 + (double)v_[pidx] * n2 + (double)w_[pidx] * n3;
    }
    const double alpha = 0.5 * fabs(VelP + VelM);
    fl[f] = (op_t)(0.5 * g[kGeoFscale + f] * (qP[f] * VelP - qm * VelM - alpha * (qP[f] - qm)));
  };
  if (active) {
#pragma unroll
    for (int f = 0; f < 6; ++f) face_flux(f);
  }

  // B = [D^T ; l- ; l+ ; 0] rows of this lane (k permuted, see above)
  constexpr int NT = C::NT;
  const int col = lane & 15, kq = lane >> 4;
  op_t bop[NT][KSTEPS];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const int c = 16 * nt + col;
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) {
      const int l = kq * KSTEPS + ks;
      bop[nt][ks] = c >= NQ ? (op_t)0 : l < NQ ? D_[c + l * NQ] : l == NQ ? ell_[c]
                    : l == NQ + 1 ? ell_[NQ + c] : (op_t)0;
    }
  }
  const int rd = col * STRIDE + kq * KSTEPS;        // A read offset of this lane in a tile
  const int wr = P::RSTRIDE_Q * kq * STRIDE + col;  // result offset of value 0
  const int left = KAUG - kq * KSTEPS;              // stored operands of the lane's K range
  // Node (i,j,k) sits in the x pencil (j,k) at position i, in the y pencil
  // (i,k) at position j and in the z pencil (i,j) at position k; face node
  // (i,j) of the faces normal to d is pencil ij of direction d.
  const int pos_off[3] = {j * STRIDE + i, i * STRIDE + j, ij * STRIDE};
  const int pos_step[3] = {NQ * STRIDE, NQ * STRIDE, 1};
  const int face_m[3] = {3, 0, 4}, face_p[3] = {1, 2, 5};  // -d and +d faces

  // ---- 2b-4a, one direction at a time through one LDS area -------------------
  // Rows of A beyond the element's pencils hold stale LDS; each output row
  // depends only on its own A row, and those rows are never read back.
  double tend[NQ], q0v[NQ];
  if constexpr (ONCE) {
    if (active) {
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        const double Ed = g[kGeoEscale + d];
        op_t *a = As + d * C::AREA + pos_off[d];
#pragma unroll
        for (int k = 0; k < NQ; ++k)
          a[k * pos_step[d]] = (op_t)(Ed * (qc[k] * (double)(CVEL ? cv[d] : cols[d][k])));
        op_t *r = As + d * C::AREA + ij * STRIDE;
        r[NQ] = fl[face_m[d]];
        r[NQ + 1] = fl[face_p[d]];
      }
      if (use_q0) {
#pragma unroll
        for (int k = 0; k < NQ; ++k) q0v[k] = __builtin_nontemporal_load(q0_ + base + k * NQ2);
      }
    }
    __syncthreads();
#pragma unroll
    for (int t = wave; t < 3 * C::MTILES; t += C::WAVES)  // wave-uniform
      mfma_tile<P, KSTEPS, KAUG, STRIDE, NQ, NT>(As + t * 16 * STRIDE, bop, rd, wr, col, left);
    __syncthreads();
    if (active) {
#pragma unroll
      for (int d = 0; d < 3; ++d)
#pragma unroll
        for (int k = 0; k < NQ; ++k) {
          const double x = (double)As[d * C::AREA + pos_off[d] + k * pos_step[d]];
          tend[k] = d == 0 ? x : tend[k] + x;
        }
    }
  } else {
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      if (active) {
        const double Ed = g[kGeoEscale + d];
        const vel_t *vel = velp[d];
        op_t *a = As + pos_off[d];
        vel_t col_d[NQ];
#pragma unroll
        for (int k = 0; k < NQ; ++k) col_d[k] = CVEL ? cv[d] : vel[base + k * NQ2];
        // all of the column in flight before its first use: left to itself the
        // compiler may load and wait one node at a time (mixed p = 17 fields,
        // 166 us per launch against 138)
        if constexpr (!CVEL) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < NQ; ++k)
          a[k * pos_step[d]] = (op_t)(Ed * (qc[k] * (double)col_d[k]));
        op_t *r = As + ij * STRIDE;
        r[NQ] = fl[face_m[d]];
        r[NQ + 1] = fl[face_p[d]];
      }
      __syncthreads();
#pragma unroll
      for (int jj = 0; jj < C::JPW; ++jj) {
        const int t = wave + jj * C::WAVES;
        if (t >= C::MTILES) break;  // wave-uniform
        mfma_tile<P, KSTEPS, KAUG, STRIDE, NQ, NT>(As + t * 16 * STRIDE, bop, rd, wr, col, left);
      }
      __syncthreads();
      if (active) {
#pragma unroll
        for (int k = 0; k < NQ; ++k) {
          const double x = (double)As[pos_off[d] + k * pos_step[d]];
          tend[k] = d == 0 ? x : tend[k] + x;
        }
      }
      if (d < 2) __syncthreads();  // the next direction overwrites the area
    }
  }

  // ---- 4b. RK epilogue (FP64).  The RK base is read only here: held through
  // the last direction's product it cost p = 16, 17 a wave per SIMD.  In a
  // block of its own, or the allocation spills.
  if (!ONCE && active && use_q0) {
#pragma unroll
    for (int k = 0; k < NQ; ++k) q0v[k] = __builtin_nontemporal_load(q0_ + base + k * NQ2);
  }
  if (active) {
    const double dtv = dt_geo_ ? g[kGeoDt] : dt_;
#pragma unroll
    for (int k = 0; k < NQ; ++k) {
      const double td = -tend[k];
      const int64_t idx = base + (int64_t)k * NQ2;
      double res = td;
      if (rk) {
        const double upd = cb_ * (qc[k] + dtv * td);
        res = use_q0 ? ca_ * q0v[k] + upd : upd;
      }
      __builtin_nontemporal_store(res, out_ + idx);
    }
  }
}

// AXAL: every face normal lies along its face's axis (checked on the host);
// the ax_runtime shapes test it at run time (instantiated as the general form).
// CVEL: constant velocity per element, (u, v, w) = words kGeoVel..+2 of its
// geometry record (batched and served boxes, solvers with constant fields); no
// velocity field is read, and the operand-precision value of a constant is the
// value its per-node copy holds, so the results are the same bits.
// GU: several elements per workgroup and one geometry record for the whole
// launch (no per-element record ids): the record is read through the kernel
// argument itself, i.e. through the scalar cache (as in stage_f64).
template <class P, int NQ, int EPB, bool SEQ, bool AXAL, bool CVEL = false, bool GU = false>
__global__ void
__attribute__((amdgpu_flat_work_group_size(1, Shape<P, NQ, EPB, SEQ, CVEL>::THREADS),
               amdgpu_waves_per_eu(Shape<P, NQ, EPB, SEQ, CVEL>::MIN_WAVES_EU)))
stage_mfma(const double *__restrict__ q_, const double *q0_,
           const typename P::vel_t *__restrict__ u_, const typename P::vel_t *__restrict__ v_,
           const typename P::vel_t *__restrict__ w_, double *out_,
           const int32_t *__restrict__ nbr_, const int32_t *__restrict__ vmapP_,
           const typename P::op_t *__restrict__ D_, const typename P::op_t *__restrict__ ell_,
           const double *__restrict__ geo_, const uint32_t *__restrict__ geoid_,
           const int32_t *__restrict__ order_, const int64_t Ne_, const double ca_,
           const double cb_, const double dt_, const int mode_, const int axis_aligned_,
           const int dt_geo_, const int rev_, const int64_t zp_) {
  static_assert(!GU || EPB > 1, "one element per workgroup reads its record uniformly anyway");
  if constexpr (!Shape<P, NQ, EPB, SEQ, CVEL>::MFMA) {
    stage_aug<P, NQ, EPB, ax_runtime<P, NQ, EPB, SEQ>(), AXAL, CVEL, GU>(
        q_, q0_, u_, v_, w_, out_, nbr_, vmapP_, D_, ell_, geo_, geoid_, order_, Ne_, ca_, cb_,
        dt_, mode_, axis_aligned_, dt_geo_, rev_, zp_);
  } else {
    stage_seq<P, NQ, CVEL, false>(
        q_, q0_, u_, v_, w_, out_, nbr_, vmapP_, D_, ell_, geo_, geoid_, order_, Ne_, ca_, cb_,
        dt_, mode_, axis_aligned_, dt_geo_, rev_, zp_);
  }
}

// Launches of few elements (has_small): the MFMA form, the directions at once.
template <class P, int NQ, bool CVEL>
__global__ void
__attribute__((amdgpu_flat_work_group_size(1, Seq<P, NQ>::THREADS),
               amdgpu_waves_per_eu(CVEL ? 4 : 2)))
stage_small(const double *__restrict__ q_, const double *q0_,
            const typename P::vel_t *__restrict__ u_, const typename P::vel_t *__restrict__ v_,
            const typename P::vel_t *__restrict__ w_, double *out_,
            const int32_t *__restrict__ nbr_, const int32_t *__restrict__ vmapP_,
            const typename P::op_t *__restrict__ D_, const typename P::op_t *__restrict__ ell_,
            const double *__restrict__ geo_, const uint32_t *__restrict__ geoid_,
            const int32_t *__restrict__ order_, const int64_t Ne_, const double ca_,
            const double cb_, const double dt_, const int mode_, const int axis_aligned_,
            const int dt_geo_, const int rev_, const int64_t zp_) {
  stage_seq<P, NQ, CVEL, true>(q_, q0_, u_, v_, w_, out_, nbr_, vmapP_, D_, ell_, geo_, geoid_,
                               order_, Ne_, ca_, cb_, dt_, mode_, axis_aligned_, dt_geo_, rev_,
                               zp_);
}

template <class P, int NQ, int EPB, bool SEQ, bool AXAL, bool CVEL, bool GU>
int prepare_kernel() {
  // set once per device; concurrent callers may both set it (idempotent)
  static std::atomic<int> prepared_dev{-1};
  int dev = 0;
  DGK_HIP(hipGetDevice(&dev));
  if (prepared_dev.load(std::memory_order_acquire) != dev) {
    DGK_HIP(hipFuncSetAttribute((const void *)stage_mfma<P, NQ, EPB, SEQ, AXAL, CVEL, GU>,
                                hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)Shape<P, NQ, EPB, SEQ, CVEL>::LDS_BYTES));
    prepared_dev.store(dev, std::memory_order_release);
  }
  return DGK_OK;
}

// a form with its uniform-geometry variant where a workgroup holds several
// elements
template <class P, int NQ, int EPB, bool SEQ, bool AXAL, bool CVEL = false>
int prepare_form() {
  DGK_TRY((prepare_kernel<P, NQ, EPB, SEQ, AXAL, CVEL, false>()));
  if constexpr (EPB > 1) DGK_TRY((prepare_kernel<P, NQ, EPB, SEQ, AXAL, CVEL, true>()));
  return DGK_OK;
}

// Both face-normal forms of a shape (one, testing at run time, for the
// AX_RUNTIME shapes).
template <class P, int NQ, int EPB, bool SEQ>
int prepare_shape() {
  constexpr bool AXR = ax_runtime<P, NQ, EPB, SEQ>();
  DGK_TRY((prepare_form<P, NQ, EPB, SEQ, false>()));
  if constexpr (!AXR) DGK_TRY((prepare_form<P, NQ, EPB, SEQ, true>()));
  DGK_TRY((prepare_form<P, NQ, EPB, SEQ, !AXR, true>()));
  return DGK_OK;
}

template <class P, int NQ, int EPB, bool SEQ, bool AXAL, bool CVEL, bool GU, class Args>
int launch_kernel(const Args &a, hipStream_t s) {
  using T = Shape<P, NQ, EPB, SEQ, CVEL>;
  const int64_t nblk = (a.Ne + EPB - 1) / EPB;
  if (nblk > INT32_MAX) return set_error(DGK_ERR_UNSUPPORTED, "too many elements");
  DGK_TRY((prepare_kernel<P, NQ, EPB, SEQ, AXAL, CVEL, GU>()));
  hipLaunchKernelGGL((stage_mfma<P, NQ, EPB, SEQ, AXAL, CVEL, GU>), dim3((unsigned)nblk),
                     dim3(T::THREADS), T::LDS_BYTES, s, a.q, a.q0, a.u, a.v, a.w, a.out, a.nbr,
                     a.vmapP, a.D, a.ell, a.geo, a.geoid, a.order, a.Ne, a.ca, a.cb, a.dt,
                     a.mode, a.axis_aligned, a.dt_geo, a.reverse, a.zperiod);
  DGK_HIP(hipGetLastError());
  return DGK_OK;
}

template <class P, int NQ, int EPB, bool SEQ, bool AXAL, class Args, bool CVEL = false>
int launch_form(const Args &a, hipStream_t s) {
  if constexpr (EPB > 1)
    if (!a.geoid) return launch_kernel<P, NQ, EPB, SEQ, AXAL, CVEL, true>(a, s);
  return launch_kernel<P, NQ, EPB, SEQ, AXAL, CVEL, false>(a, s);
}

// Where a launch of few elements takes stage_small: the mixed form at p = 13..15 with
// at most one element per CU, with a constant velocity two.  Such a launch lasts as
// long as one element does, which is four wavefronts in the VALU form and eight here,
// with the three directions between two barriers.  us per launch, stage_aug against
// stage_small: p = 13 8 elements 7.8/7.2, 256 8.7/8.2, constant velocity 256
// 8.7/6.7, 512 11.4/10.5; p = 15 8 elements 8.8/8.2, 256 10.2/9.9, constant
// velocity 256 9.3/7.8, 512 13.8/13.0.  With more elements than that fit at once
// stage_aug has the higher rate: p = 15 320 elements 14.0/17.5, constant velocity
// 768 16.9/19.6.  The same bits.
constexpr int64_t kCus = 256;
template <class P, int NQ, int EPB>
constexpr bool has_small() {
  return sizeof(typename P::op_t) == 4 && NQ >= 14 && NQ <= 16 && EPB == 1;
}

template <class P, int NQ, bool CVEL, class Args>
int launch_small(const Args &a, hipStream_t s) {
  using C = Seq<P, NQ>;
  static_assert(C::LDS_BYTES_ONCE <= 64 * 1024, "no attribute to set");
  hipLaunchKernelGGL((stage_small<P, NQ, CVEL>), dim3((unsigned)a.Ne), dim3(C::THREADS),
                     C::LDS_BYTES_ONCE, s, a.q, a.q0, a.u, a.v, a.w, a.out, a.nbr, a.vmapP, a.D, a.ell,
                     a.geo, a.geoid, a.order, a.Ne, a.ca, a.cb, a.dt, a.mode, a.axis_aligned,
                     a.dt_geo, a.reverse, a.zperiod);
  DGK_HIP(hipGetLastError());
  return DGK_OK;
}

template <class P, int NQ, int EPB, bool SEQ, class Args>
int launch_shape(const Args &a, hipStream_t s) {
  constexpr bool AXR = ax_runtime<P, NQ, EPB, SEQ>();
  // constant velocity: on axis-aligned faces only
  const bool cvel = a.cvel && a.axis_aligned && !a.vmapP;
  if constexpr (has_small<P, NQ, EPB>())
    if (a.Ne <= (cvel ? 2 * kCus : kCus))
      return cvel ? launch_small<P, NQ, true>(a, s) : launch_small<P, NQ, false>(a, s);
  if (cvel)
    return launch_form<P, NQ, EPB, SEQ, !AXR, Args, true>(a, s);
  if constexpr (!AXR)
    if (a.axis_aligned) return launch_form<P, NQ, EPB, SEQ, true>(a, s);
  return launch_form<P, NQ, EPB, SEQ, false>(a, s);
}

// Candidate c of order NQ (compile-time), as a kernel instantiation.
template <class P, int NQ, int CAND>
struct Cand {
  static constexpr int K = kind_of<P, NQ>(CAND);
  static constexpr int EPB = kind_epb<NQ>(K < 0 ? 0 : K);
  static constexpr bool SEQ = kind_seq<NQ>(K < 0 ? 0 : K);
};

template <class P, int NQ>
int prepare_nq_all() {
  DGK_TRY((prepare_shape<P, NQ, Cand<P, NQ, 0>::EPB, Cand<P, NQ, 0>::SEQ>()));
  if constexpr (ncand<P, NQ>() > 1)
    DGK_TRY((prepare_shape<P, NQ, Cand<P, NQ, 1>::EPB, Cand<P, NQ, 1>::SEQ>()));
  if constexpr (ncand<P, NQ>() > 2)
    DGK_TRY((prepare_shape<P, NQ, Cand<P, NQ, 2>::EPB, Cand<P, NQ, 2>::SEQ>()));
  if constexpr (ncand<P, NQ>() > 3)
    DGK_TRY((prepare_shape<P, NQ, Cand<P, NQ, 3>::EPB, Cand<P, NQ, 3>::SEQ>()));
  return DGK_OK;
}

template <class P, int NQ, class Args>
int launch_nq_cand(int cand, const Args &a, hipStream_t s) {
  if constexpr (ncand<P, NQ>() > 1)
    if (cand == 1) return launch_shape<P, NQ, Cand<P, NQ, 1>::EPB, Cand<P, NQ, 1>::SEQ>(a, s);
  if constexpr (ncand<P, NQ>() > 2)
    if (cand == 2) return launch_shape<P, NQ, Cand<P, NQ, 2>::EPB, Cand<P, NQ, 2>::SEQ>(a, s);
  if constexpr (ncand<P, NQ>() > 3)
    if (cand == 3) return launch_shape<P, NQ, Cand<P, NQ, 3>::EPB, Cand<P, NQ, 3>::SEQ>(a, s);
  return launch_shape<P, NQ, Cand<P, NQ, 0>::EPB, Cand<P, NQ, 0>::SEQ>(a, s);
}

template <class P, int NQ>
int shapes_of(int *epb) {
  constexpr int n = ncand<P, NQ>();
  if constexpr (n > 0) epb[0] = Cand<P, NQ, 0>::EPB;
  if constexpr (n > 1) epb[1] = Cand<P, NQ, 1>::EPB;
  if constexpr (n > 2) epb[2] = Cand<P, NQ, 2>::EPB;
  if constexpr (n > 3) epb[3] = Cand<P, NQ, 3>::EPB;
  return n;
}

}  // namespace

#define DGK_NQ_SWITCH(NQV, CALL)                                                         \
  switch (NQV) {                                                                         \
  case 2: return CALL(2); case 3: return CALL(3); case 4: return CALL(4);                \
  case 5: return CALL(5); case 6: return CALL(6); case 7: return CALL(7);                \
  case 8: return CALL(8); case 9: return CALL(9); case 10: return CALL(10);              \
  case 11: return CALL(11); case 12: return CALL(12); case 13: return CALL(13);          \
  case 14: return CALL(14); case 15: return CALL(15); case 16: return CALL(16);          \
  case 17: return CALL(17); case 18: return CALL(18); case 19: return CALL(19);          \
  case 20: return CALL(20);                                                              \
  default: return set_error(DGK_ERR_UNSUPPORTED, "Nq outside 2.." + std::to_string(kMaxNq));                   \
  }

}  // namespace dgk
