// nmr_device.h -- device functions shared by the kernel files.  Not part of
// the public ABI.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "nmr_kernels.h"

namespace nmr {

// Harmonic mean 2ab/(a + b) of two (scaled) diffusivities for the face
// between them, with the hardware reciprocal (v_rcp_f32, about 1 ulp) in
// place of an IEEE division.  Sums below 1e-30 -- solids, which the
// reference gives D = 1e-50 -- give 0: their reciprocal would overflow, and
// the exact mean is below 1e-30 there anyway.  Every general kernel uses it,
// so they stay bit-identical.
__device__ __forceinline__ float hmean(float a, float b)
{
    const float s = a + b;
    return s > 1e-30f ? (2.f * a * b) * __builtin_amdgcn_rcpf(s) : 0.f;
}

// Block index -> tile index such that XCD x (blocks x, x+8, x+16, ...) gets
// the contiguous tile range [x*q + min(x,r), ...), q = nb/8, r = nb%8.
__device__ __forceinline__ int xcd_tile(int b, int nb)
{
    const int xcd = b & 7, ib = b >> 3;
    const int q = nb >> 3, r = nb & 7;
    return xcd * q + (xcd < r ? xcd : r) + ib;
}

// Instantaneous RF / gradient pulse: every pore voxel's M is rotated by an
// angle about an axis, as AddImpulse + OrtTransform do it
// (src/NmrRelaxationSolve.cpp:2536-2608).  Angles and the rotation are
// evaluated in FP64 in the reference's order of operations; the state stays
// FP32.  Reference index i maps to x + 1 here (no ghost layer: ghost cells
// are refilled from the interior after every pulse in the reference anyway).
__device__ __forceinline__ void pulse_voxel(const PulseArgs& a, int x, int y, int z, float* mx, float* my, float* mz)
{
    double len = sqrt(a.ax * a.ax + a.ay * a.ay + a.az * a.az);
    if (len == 0.0) len = 1.0;
    const double n0x = a.ax / len, n0y = a.ay / len, n0z = a.az / len;
    const double i = (double)(x + 1), j = (double)(y + 1), k = (double)(z + 1);
    double angle, rx, ry, rz;
    if (a.flag == 1) { // narrow gradient pulse, axis = unit gradient direction
        angle = a.param * a.gamma * ((i - 1) * a.dx * a.ax + (j - 1) * a.dy * a.ay + (k - 1) * a.dz * a.az);
        rx = n0x; ry = n0y; rz = n0z;
    } else if (a.flag == 2) { // RF pulse of angle param about the (unnormalised) axis
        angle = a.param;
        rx = a.ax; ry = a.ay; rz = a.az;
    } else if (a.flag == 3) { // multi-gradient pulse about a far-away origin
        const double distance = 10e+12;
        const double eff = sqrt(a.ax * a.ax + a.ay * a.ay + a.az * a.az);
        const double t = (i - 1.0 - distance) * a.dx * n0x + (j - 1.0 - distance) * a.dy * n0y +
                         (k - 1.0 - distance) * a.dz * n0z;
        angle = a.gamma * eff * sqrt(t * t);
        rx = n0x; ry = n0y; rz = n0z;
    } else { // flag 4: radial phase about the domain centre
        const double tx = (i - 0.5) * a.dx * a.ax - 0.5 * a.nx * a.dx * a.ax;
        const double ty = (j - 0.5) * a.dy * a.ay - 0.5 * a.ny * a.dy * a.ay;
        const double tz = (k - 0.5) * a.dz * a.az - 0.5 * a.nz * a.dz * a.az;
        angle = 0.0 - a.gamma * sqrt(tx * tx + ty * ty + tz * tz);
        rx = a.ax; ry = a.ay; rz = a.az;
    }
    const double c = cos(angle), s = sin(angle);
    const double vx = *mx, vy = *my, vz = mz ? (double)*mz : 0.0;
    const double scal = rx * vx + ry * vy + rz * vz;
    *mx = (float)(vx * c + rx * (1.0 - c) * scal + s * (ry * vz - rz * vy));
    *my = (float)(vy * c + ry * (1.0 - c) * scal + s * (rz * vx - rx * vz));
    if (mz) *mz = (float)(vz * c + rz * (1.0 - c) * scal + s * (rx * vy - ry * vx));
}

} // namespace nmr
