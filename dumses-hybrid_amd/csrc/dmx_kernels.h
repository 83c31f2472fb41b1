// dmx_kernels.h -- device data layout and kernels of the MHD step.
//
// Layout in HBM (one context = one ghosted domain, nghost = 3):
//   index(i,j,k) = (i+2) + px*((j+2) + gy*(k+2)),  i in [-2, nx+3] (the
//   reference's uin index range), px = nx+6 rounded up to 16 elements so
//   every x-row starts 128-byte aligned; x is the fastest index (coalesced).
//   U  : 8 planes -- rho, rho*u, rho*v, rho*w in the bulk type T; the total
//        energy E and the left-face fields Bx_L, By_L, Bz_L always in float64
//        (E: the pressure recovery at low beta subtracts the magnetic energy
//        from it; B: the CT face-B accumulation stays float64 in both
//        precisions).  The reference's right faces are implied:
//        B_R(i) = B_L(i+1).
//   S  : 38 (47) values of T per cell, the per-cell trace summary written by the
//        trace kernel for cells [0, n+1]^3 (see TraceSlot), in groups of
//        256 bytes of consecutive cells per slot (s_off in dmx_step.inc).
//   F  : 18 planes of T, x/y/z face fluxes of rho, rho*u, rho*v, rho*w, E
//        (already multiplied by ds*dt as compflux does) and the HLLD star
//        total pressure p_T (raw).
//   EM : 3 planes of T, edge EMFs times dt.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "dmx_tiling.h"

// 1: the trace summary holds the fields of both faces of a cell in each
// direction (47 words) and the states at a face or edge take the mean of the
// two cells' values.  float32 contexts with the learned limiter are built so
// (dmx_f32l.hip): the two values differ by a rounding there, and the limiter's
// branches amplify the last bit of the state (1e-7 to 6e-5 within 30 steps at
// 128^3), so its runs keep the arithmetic they had.  It is not the more accurate
// one: after 30 steps of turbulence from six seeds the relative L1 difference
// from float64 is 3.16e-5 to 3.84e-5 at 64^3 with 47 words and 3.15e-5 to
// 3.84e-5 with 38, 1.90e-5 to 2.36e-5 and 1.92e-5 to 2.36e-5 at 96^3, 1.68e-5
// to 1.87e-5 with both at 128^3, and neither form's largest difference (3e-3 to
// 1.5e-2) is the lesser one on most seeds.  The 38-word form would take 59 us
// instead of 63 in the fused kernel at 64^3, 419 instead of 443 at 128^3 and
// 2570 instead of 2750 at 256^3.  In float64 both forms give the same bits.
#ifndef DMX_BOTH_FACES
#define DMX_BOTH_FACES 0
#endif
// 1: the fused kernel's threads hold one direction each (dmx_fused.inc)
#ifndef DMX_LANE_DIR
#define DMX_LANE_DIR 0
#endif

namespace dmx {

enum TraceSlot {
    S_R = 0, S_U, S_V, S_W, S_P, S_A, S_B, S_C,          // predicted centre state
    S_DRX = 8, S_DUX, S_DVX, S_DWX, S_DPX, S_DBX, S_DCX, // half slopes along x
    S_DRY = 15, S_DUY, S_DVY, S_DWY, S_DPY, S_DAY, S_DCY,
    S_DRZ = 22, S_DUZ, S_DVZ, S_DWZ, S_DPZ, S_DAZ, S_DBZ,
#if DMX_BOTH_FACES
    S_AL = 29, S_AR, S_BL, S_BR, S_CL, S_CR,             // predicted face fields
    S_DALY = 35, S_DARY, S_DALZ, S_DARZ,                 // face-field half slopes
    S_DBLX, S_DBRX, S_DBLZ, S_DBRZ,
    S_DCLX, S_DCRX, S_DCLY, S_DCRY,
    NSLOT = 47
#else
    // predicted left face fields and their transverse half slopes: the right
    // face of a cell is the left one of the next cell, whose predictor forms
    // the same expressions.  Without the right faces a cell has 38 words, not
    // 47: at 256^3 the float64 trace takes 1.79 ms (2.13), the face/edge
    // stage 4.42 (4.88), both bound by the summary's traffic, and the float32
    // fused kernel 2.67 (2.83), whose LDS tile is that much smaller
    S_AL = 29, S_BL, S_CL,
    S_DALY = 32, S_DALZ, S_DBLX, S_DBLZ, S_DCLX, S_DCLY,
    NSLOT = 38
#endif
};

// flux planes: F[d*6 + c], c in {rho, mx, my, mz, E, pstar}
enum { F_R = 0, F_MX, F_MY, F_MZ, F_E, F_PS, NFC = 6 };

struct Geom {
    int nx, ny, nz;
    int px, gy, gz;
    long long nvol;      // elements per plane
    double dx, dy, dz;
    double hdx;          // dx / 2
    double ds[3];        // face areas dy dz, dx dz, dx dy
    double xmin, xmax, ymin, ymax, zmin, zmax;
    __host__ __device__ __forceinline__ long long idx(int i, int j, int k) const
    {
        return (long long)(i + 2) + (long long)px * ((long long)(j + 2) + (long long)gy * (k + 2));
    }
    __device__ __forceinline__ double xc(int i) const { return xmin + hdx + (double)(i - 1) * dx; }
};

struct Phys {
    double gamma, ciso, omega0, courant;
    double nu, eta;
    // formed on the host: there are no scalar float64 instructions, so every
    // thread of a kernel would hold these in vector registers
    double smallp;       // pressure floor, commons.f90:52
    double entho;        // 1 / (gamma - 1), gamma in the bulk type
    int iso, slope_type, riemann, riemann2d, fargo;
    int bc[3];
};

template <typename T> struct Fields {
    T* uh;          // 4 planes: rho, rho*u, rho*v, rho*w
    double* ue;     // total energy E
    double* ub;     // 3 face-B planes
    T* s;           // NSLOT planes
    T* f;           // 18 planes
    T* em;          // 3 planes
    // learned limiter (slope_type 4) only
    float* lq;      // 8 planes: primitive variables of every cell
    float* ls;      // 24 planes: limited slopes [direction][variable]
    const unsigned short* lw;   // packed bf16 weights (see the limiter kernel)
    const float* lb;            // biases b1 (64), b2 (64), b3 (8)
    unsigned int* lcount;       // fallback counter
};

} // namespace dmx
