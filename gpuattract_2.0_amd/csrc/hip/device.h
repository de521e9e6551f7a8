// Device-side data descriptors and the per-bead arithmetic of the scoring path.
//
// Every function reproduces the reference CPU path's FP32 operation order
// (no contraction: the library is built with -ffp-contract=off) so that
// per-bead values match the CPU restatement bit for bit; only the per-pose
// sums use a different (wave-tree) order.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "attract_hip.h"
#include "libm_sincosf.h"

namespace att {

constexpr int kWave = 64;
constexpr unsigned kMaxTypesLDS = 32;  // pair table staged in LDS up to 32x32 types

// Interpolation grid (model/IntrplGrid.h:34-209) with the constants its
// constructor derives (model/IntrplGrid.tpp:30-41).  Stored as voxel octets:
// for every (grid, iz, iy, ix) with i < n-1 the eight corner float4 values, in
// the order trilinearInterpolation sums them (000, 100, 010, 001, 101, 011,
// 110, 111), contiguous and 128-byte aligned — one cache line per lookup.
// octE holds the energy channel of the same octets (8 floats, 32 bytes per
// voxel) for the adjoint, which reads no other channel; null for grids without
// a neighbour list (the adjoint never reads those) and where their memory was
// needed elsewhere.
struct DGrid {
    const float4* oct;
    const float4* octE;
    unsigned nx, ny, nz, nxy, nvox, ngrids;
    float lox, loy, loz, hix, hiy, hiz;
    float dVox, dVox_inv, vol_inv;
};

// Neighbour-list grid (model/NLGrid.h:36-202, model/NLGrid.tpp:30-52).
struct DNL {
    const uint2* desc;
    const uint32_t* list;
    unsigned nx, ny, nz;
    float lox, loy, loz, hix, hiy, hiz;
    float dVox_inv, P2, P2_inv;
    float P6_inv;  // P2_inv^3, as lj() forms it
    float ddP[2];  // coulomb()'s distance factor at the plateau, by dielec
    double ratioC; // 1 / (10000 P2), for plateau_ratio_fast
};

// Protein (model/Protein.h:38-167): pos = {x, y, z, charge}.
struct DProt {
    const float4* pos;
    const float* soa;     // [x: ns][y: ns][z: ns][1: ns], zero beyond n: the bead-order reductions
    const unsigned* type;
    const unsigned* mtype;
    const float* modes;   // [c][m][n]: coalesced over beads
    const float4* modesT; // per bead one row {type bits, 3*M floats [m][c]}, padded to a float4 multiple
    const float* modeForce;
    unsigned n, M, rowT;  // rowT = float4 per modesT row
    unsigned ns;          // n rounded up to 64
};

// Basis grids of the parameter derivative (attached to a DGrid of the same
// geometry): per voxel, per basis channel, the 8 corner values in trilinear
// order (two float4).  nb = 2T channels [S_1, S6_1, S_2, S6_2, ...].
struct DBasis {
    const float4* oct;
    unsigned nb;
};

struct DPar {
    const att_pair_params* tab;  // T*T, index T*(recType-1)+(ligType-1)
    unsigned T;
    int shape;   // 8 or 12
    int dielec;  // 0 constant, 1 variable
    float ffelec;
};

struct V3 { float x, y, z; };

// RotMat::operator*(Vec3) (commons/RotMat.h:122-129).
__device__ __forceinline__ V3 matvec(const float* m, float x, float y, float z) {
    V3 o;
    o.x = m[0] * x + m[1] * y + m[2] * z;
    o.y = m[3] * x + m[4] * y + m[5] * z;
    o.z = m[6] * x + m[7] * y + m[8] * z;
    return o;
}

// euler2rotmat (model/matrixFunctions.h:38-77) from the six trig values
// {cSSI, cPHI, sSSI, sPHI, cROT, sROT}.
__device__ __forceinline__ void rotmat_from_trig(float cSSI, float cPHI, float sSSI, float sPHI,
                                                 float cROT, float sROT, float* m) {
    const float cSSI_cPHI = cSSI * cPHI, cSSI_sPHI = cSSI * sPHI;
    const float sSSI_cPHI = sSSI * cPHI, sSSI_sPHI = sSSI * sPHI;
    m[0] = cROT * cSSI_cPHI + sROT * sPHI;
    m[1] = sROT * cSSI_cPHI - cROT * sPHI;
    m[2] = sSSI_cPHI;
    m[3] = cROT * cSSI_sPHI - sROT * cPHI;
    m[4] = sROT * cSSI_sPHI + cROT * cPHI;
    m[5] = sSSI_sPHI;
    m[6] = -cROT * sSSI;
    m[7] = -sROT * sSSI;
    m[8] = cSSI;
}

// euler2torquemat (model/matrixFunctions.h:79-127) contracted with the torque
// tensor T[k][l] as TorqueMat::rotateReduce does (commons/TorqueMat.h:27-37).
__device__ __forceinline__ void torque_reduce(float cSSI, float cPHI, float sSSI, float sPHI,
                                              float cROT, float sROT, const float* T, float* out) {
    const float cSSI_cPHI = cSSI * cPHI, cSSI_sPHI = cSSI * sPHI;
    const float sSSI_cPHI = sSSI * cPHI, sSSI_sPHI = sSSI * sPHI;
    float tm[27];
    tm[0] = -cROT * cSSI_sPHI + sROT * cPHI;
    tm[1] = -sROT * cSSI_sPHI - cROT * cPHI;
    tm[2] = -sSSI_sPHI;
    tm[9] = cROT * cSSI_cPHI + sROT * sPHI;
    tm[10] = sROT * cSSI_cPHI - cROT * sPHI;
    tm[11] = sSSI_cPHI;
    tm[18] = 0.f; tm[19] = 0.f; tm[20] = 0.f;
    tm[3] = -cROT * sSSI_cPHI;
    tm[4] = -sROT * sSSI_cPHI;
    tm[5] = cSSI_cPHI;
    tm[12] = -cROT * sSSI_sPHI;
    tm[13] = -sROT * sSSI_sPHI;
    tm[14] = cSSI_sPHI;
    tm[21] = -cROT * cSSI;
    tm[22] = -sROT * cSSI;
    tm[23] = -sSSI;
    tm[6] = -sROT * cSSI_cPHI + cROT * sPHI;
    tm[7] = cROT * cSSI_cPHI + sROT * sPHI;
    tm[8] = 0.f;
    tm[15] = -sROT * cSSI_sPHI - cROT * cPHI;
    tm[16] = cROT * cSSI_sPHI - sROT * cPHI;
    tm[17] = 0.f;
    tm[24] = sROT * sSSI;
    tm[25] = -cROT * sSSI;
    tm[26] = 0.f;
    float r0 = 0.f, r1 = 0.f, r2 = 0.f;
#pragma unroll
    for (int k = 0; k < 3; ++k)
#pragma unroll
        for (int l = 0; l < 3; ++l) {
            r0 += tm[9 * k + 0 + l] * T[3 * k + l];
            r1 += tm[9 * k + 3 + l] * T[3 * k + l];
            r2 += tm[9 * k + 6 + l] * T[3 * k + l];
        }
    out[0] = r0; out[1] = r1; out[2] = r2;
}

// A value that is the same on every lane, in a scalar register: a pose's
// rotation, translation and amplitudes would otherwise hold some 30 vector
// registers through the walks (the 10-mode adjoint without parameter gradients
// spilled 84 B per lane with them there and spills none now; with them 28-44 B are
// left).
__device__ __forceinline__ float uniform(float v) {
    return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}

// The six trig values of a pose, evaluated once per wave: lanes 0..2 take
// sin and cos of (ssi, phi, rot) with the C library's single-precision values
// (sincosf_libm, as the reference's std::sin/std::cos(float)), then every lane
// reads them back.
__device__ __forceinline__ void pose_trig(float phi, float ssi, float rot, int lane, float* t) {
    float c = 0.f, s = 0.f;
    if (lane < 3) sincosf_libm(lane == 0 ? ssi : lane == 1 ? phi : rot, &s, &c);
    auto at = [](float v, int l) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l)); };
    t[0] = at(c, 0);  // cSSI
    t[1] = at(c, 1);  // cPHI
    t[2] = at(s, 0);  // sSSI
    t[3] = at(s, 1);  // sPHI
    t[4] = at(c, 2);  // cROT
    t[5] = at(s, 2);  // sROT
}

// IntrplGrid::outOfBounds_byPos (model/IntrplGrid.h:113-117).
// Written as "not inside" so that a NaN coordinate counts as outside (the
// reference's form would index the grid with it); identical for finite input.
__device__ __forceinline__ bool grid_out(const DGrid& g, float x, float y, float z) {
    return !((x >= g.lox && x <= g.hix) && (y >= g.loy && y <= g.hiy) && (z >= g.loz && z <= g.hiz));
}

__device__ __forceinline__ unsigned grid_index(float p, float lo, float inv, unsigned n) {
    const unsigned i = (unsigned)floorf((p - lo) * inv);
    return i < n - 2 ? i : n - 2;
}

// getVoxelByIndex + trilinearInterpolation (model/IntrplGrid.h:130-163,
// model/trilinIntrpl.h:28-65): eight float4 corners, weights and summation in
// the reference's order, then scaled by 1/voxelVolume.
__device__ __forceinline__ float4 trilin(const DGrid& g, float px, float py, float pz, unsigned ix,
                                         unsigned iy, unsigned iz, unsigned type) {
    const float mnx = (float)(int)ix * g.dVox + g.lox;
    const float mny = (float)(int)iy * g.dVox + g.loy;
    const float mnz = (float)(int)iz * g.dVox + g.loz;
    const float ax = px - mnx, ay = py - mny, az = pz - mnz;
    const float bx = (mnx + g.dVox) - px, by = (mny + g.dVox) - py, bz = (mnz + g.dVox) - pz;
    const float tmpMax_xy = bx * by;
    const float tmpMin_xy = ax * ay;
    const float w0 = tmpMax_xy * bz;
    const float w1 = (ax * by) * bz;
    const float w2 = (bx * ay) * bz;
    const float w3 = tmpMax_xy * az;
    const float w4 = (ax * by) * az;
    const float w5 = (bx * ay) * az;
    const float w6 = tmpMin_xy * bz;
    const float w7 = tmpMin_xy * az;
    const size_t o = (((size_t)type * (g.nz - 1) + iz) * (g.ny - 1) + iy) * (g.nx - 1) + ix;
    const float4* d = g.oct + 8 * o;
    const float4 c0 = d[0], c1 = d[1], c2 = d[2], c3 = d[3];
    const float4 c4 = d[4], c5 = d[5], c6 = d[6], c7 = d[7];
    float4 V;
    V.x = c0.x * w0; V.y = c0.y * w0; V.z = c0.z * w0; V.w = c0.w * w0;
    V.x = V.x + c1.x * w1; V.y = V.y + c1.y * w1; V.z = V.z + c1.z * w1; V.w = V.w + c1.w * w1;
    V.x = V.x + c2.x * w2; V.y = V.y + c2.y * w2; V.z = V.z + c2.z * w2; V.w = V.w + c2.w * w2;
    V.x = V.x + c3.x * w3; V.y = V.y + c3.y * w3; V.z = V.z + c3.z * w3; V.w = V.w + c3.w * w3;
    V.x = V.x + c4.x * w4; V.y = V.y + c4.y * w4; V.z = V.z + c4.z * w4; V.w = V.w + c4.w * w4;
    V.x = V.x + c5.x * w5; V.y = V.y + c5.y * w5; V.z = V.z + c5.z * w5; V.w = V.w + c5.w * w5;
    V.x = V.x + c6.x * w6; V.y = V.y + c6.y * w6; V.z = V.z + c6.z * w6; V.w = V.w + c6.w * w6;
    V.x = V.x + c7.x * w7; V.y = V.y + c7.y * w7; V.z = V.z + c7.z * w7; V.w = V.w + c7.w * w7;
    V.x = V.x * g.vol_inv; V.y = V.y * g.vol_inv; V.z = V.z * g.vol_inv; V.w = V.w * g.vol_inv;
    return V;
}

// interpolate (model/interpolation.h:26-53).
__device__ __forceinline__ float4 interp(const DGrid& g, float px, float py, float pz,
                                         unsigned type, float charge, int* cell) {
    const unsigned ix = grid_index(px, g.lox, g.dVox_inv, g.nx);
    const unsigned iy = grid_index(py, g.loy, g.dVox_inv, g.ny);
    const unsigned iz = grid_index(pz, g.loz, g.dVox_inv, g.nz);
    if (cell) { cell[0] = (int)ix; cell[1] = (int)iy; cell[2] = (int)iz; }
    float4 pot = trilin(g, px, py, pz, ix, iy, iz, type);
    if (fabsf(charge) > 0.001f) {
        float4 el = trilin(g, px, py, pz, ix, iy, iz, 0);
        el.x = el.x * charge; el.y = el.y * charge; el.z = el.z * charge; el.w = el.w * charge;
        pot.x = pot.x + el.x; pot.y = pot.y + el.y; pot.z = pot.z + el.z; pot.w = pot.w + el.w;
    }
    return pot;
}

// potForce for one bead (model/interpolation.h:56-102): inner grid, else outer
// grid, else zero; mapped type 0 contributes nothing.
__device__ __forceinline__ float4 pot_bead(const DGrid& inner, const DGrid& outer, float px,
                                           float py, float pz, unsigned mtype, float charge,
                                           int* cell) {
    float4 pot = make_float4(0.f, 0.f, 0.f, 0.f);
    if (mtype == 0) return pot;
    if (grid_out(inner, px, py, pz)) {
        if (!grid_out(outer, px, py, pz)) pot = interp(outer, px, py, pz, mtype, charge, cell ? cell + 3 : nullptr);
    } else {
        pot = interp(inner, px, py, pz, mtype, charge, cell);
    }
    return pot;
}

// pot_bead without branches around the lookup: the grid (inner, else outer)
// is selected per lane and its octet always read, the result replaced by zero
// where the bead is in neither grid or has mapped type 0.  The same values as
// pot_bead; a loop over beads can have several lookups in flight.  The read
// stays inside the grid for any coordinate (grid_index clamps to the last
// voxel, NaN included) and type (the scoring entry points refuse bodies with
// a mapped type >= the grid's number of grids).
__device__ __forceinline__ float4 pot_bead_flat(const DGrid& inner, const DGrid& outer, float px,
                                                float py, float pz, unsigned mtype, float charge) {
    const bool in = !grid_out(inner, px, py, pz);
    const bool valid = mtype != 0 && (in || !grid_out(outer, px, py, pz));
    DGrid g;
    g.oct = in ? inner.oct : outer.oct;
    g.nx = in ? inner.nx : outer.nx;
    g.ny = in ? inner.ny : outer.ny;
    g.nz = in ? inner.nz : outer.nz;
    g.lox = in ? inner.lox : outer.lox;
    g.loy = in ? inner.loy : outer.loy;
    g.loz = in ? inner.loz : outer.loz;
    g.dVox = in ? inner.dVox : outer.dVox;
    g.dVox_inv = in ? inner.dVox_inv : outer.dVox_inv;
    g.vol_inv = in ? inner.vol_inv : outer.vol_inv;
    const unsigned ix = grid_index(px, g.lox, g.dVox_inv, g.nx);
    const unsigned iy = grid_index(py, g.loy, g.dVox_inv, g.ny);
    const unsigned iz = grid_index(pz, g.loz, g.dVox_inv, g.nz);
    float4 pot = trilin(g, px, py, pz, ix, iy, iz, mtype);
    if (fabsf(charge) > 0.001f) {  // interp's electrostatic term
        float4 el = trilin(g, px, py, pz, ix, iy, iz, 0);
        el.x = el.x * charge; el.y = el.y * charge; el.z = el.z * charge; el.w = el.w * charge;
        pot.x = pot.x + el.x; pot.y = pot.y + el.y; pot.z = pot.z + el.z; pot.w = pot.w + el.w;
    }
    return valid ? pot : make_float4(0.f, 0.f, 0.f, 0.f);
}

// LJPotForce (model/forcefield.h:28-83) with swi = 1: 6.0*vlj and the force
// factor are evaluated in double, as the reference's FP32 build does.
__device__ __forceinline__ void lj(float dr2, float dr2_inv, float dx, float dy, float dz,
                                   const att_pair_params& p, int shape, float& fx, float& fy,
                                   float& fz, float& e) {
    const float ivor = (float)p.ipon;
    const float rr23 = dr2_inv * dr2_inv * dr2_inv;
    const float rrd = shape == 8 ? dr2_inv : rr23;
    const float shapedelta = shape == 8 ? 2.f : 6.f;
    const float rep = p.rc * rrd;
    const float vlj = (rep - p.ac) * rr23;
    // 6 vlj is exact in double: fma rounds as the product and the sum would
    const double s = __builtin_fma(6.0, (double)vlj, (double)(shapedelta * (rep * rr23)));
    float fb;
    if (dr2 < p.rmin2) {
        e = vlj + (ivor - 1.f) * p.emin;
        fb = (float)s;
    } else {
        e = ivor * vlj;
        fb = (float)((double)ivor * s);
    }
    fx = fb * dx; fy = fb * dy; fz = fb * dz;
}

// ChargePotForce (model/forcefield.h:85-146) with swi = 1.
__device__ __forceinline__ void coulomb(float dr2_inv, float dx, float dy, float dz, float q,
                                        int dielec, float& fx, float& fy, float& fz, float& e) {
    float dd;
    if (dielec == 0) dd = (float)((double)sqrtf(dr2_inv) - 1.0 / 50.0);
    else dd = (float)((double)dr2_inv - 1.0 / (50.0 * 50.0));
    if (dd < 0.f) dd = 0.f;
    e = q * dd;
    if (dd <= 0.f) { fx = 0.f; fy = 0.f; fz = 0.f; return; }
    if (dielec == 0) {
        const float et2 = q * sqrtf(dr2_inv);
        fx = et2 * dx; fy = et2 * dy; fz = et2 * dz;
    } else {
        const float et2 = q * dr2_inv;
        fx = (2.f * et2) * dx; fy = (2.f * et2) * dy; fz = (2.f * et2) * dz;
    }
}

// Neighbour-list cell of a ligand bead (NLGrid bounds and getIndex,
// model/NLGrid.h:100-131, as NLPotForce tests them, model/neighborlist.h:
// 47-63): {numEl, idx} of the cell's list, {0, 0} when the bead has no
// neighbour-list term (type 0 or outside the grid).  cell receives the index.
__device__ __forceinline__ uint2 nl_cell(const DNL& nl, float px, float py, float pz,
                                         unsigned ligType, int* cell = nullptr) {
    if (ligType == 0) return make_uint2(0u, 0u);
    if (!((px >= nl.lox && px <= nl.hix) && (py >= nl.loy && py <= nl.hiy) &&
          (pz >= nl.loz && pz <= nl.hiz)))
        return make_uint2(0u, 0u);
    // NLGrid::getIndex (model/NLGrid.h:100-108): round half away from zero.
    const int ix = (int)roundf((px - nl.lox) * nl.dVox_inv);
    const int iy = (int)roundf((py - nl.loy) * nl.dVox_inv);
    const int iz = (int)roundf((pz - nl.loz) * nl.dVox_inv);
    if (cell) { cell[0] = ix; cell[1] = iy; cell[2] = iz; }
    return nl.desc[nl.nx * (iz * nl.ny + iy) + ix];
}

// The pair table as the list walks read it: the workgroup's LDS copy
// (stage_table) or the table in global memory.  Entries of the LDS copy are
// read through an LDS-typed pointer, so they are LDS loads; through a generic
// pointer they would be flat loads, which also wait for the vector-memory
// loads of the receptor beads in flight.
struct PairTab {
    const att_pair_params* p;
    bool lds;
    __device__ __forceinline__ att_pair_params operator[](unsigned k) const {
        if (lds) {
            typedef const __attribute__((address_space(3))) float* LdsF;
            typedef const __attribute__((address_space(3))) int* LdsI;
            const LdsF f = (LdsF)(const float*)(p + k);
            att_pair_params e;
            e.rc = f[0];
            e.ac = f[1];
            e.ipon = ((LdsI)(const int*)(p + k))[2];
            e.rmin2 = f[3];
            e.emin = f[4];
            return e;
        }
        return p[k];
    }
};

// Pair table into LDS when it fits (kMaxTypesLDS), else read from global.
__device__ __forceinline__ PairTab stage_table(const DPar& par, att_pair_params* s_tab) {
    if (par.T <= kMaxTypesLDS) {
        for (unsigned k = threadIdx.x; k < par.T * par.T; k += blockDim.x) s_tab[k] = par.tab[k];
        return PairTab{s_tab, true};
    }
    return PairTab{par.tab, false};
}

// Entry n of the plateau-ratio table, sqrt(((n + 0.5) / 10000) / P2) in double
// rounded to float (model/NLGrid.tpp:44-51, read by getRatio at n =
// int(dr2 * 10000), model/NLGrid.h:141-143).  Evaluated per pair rather than
// loaded: a division, a division and a square root, each correctly rounded
// in double as on the host, so the value is the table's to the bit (checked
// over every entry), and the walk waits on no load after the distance.
__device__ __forceinline__ float plateau_ratio(unsigned n, float P2) {
    return (float)__builtin_sqrt((((double)n + 0.5) / 10000.0) / (double)P2);
}

// plateau_ratio from one square-root estimate: the entry to a relative error
// below 2^-42 in double (the estimate's 2^-22 squared by one Newton step; c =
// 1 / (10000 P2)), which rounds to the entry's float unless a rounding boundary
// lies that close (one entry in 2^17): those take plateau_ratio.  The same
// bits in 16 instructions instead of about 50.
__device__ __forceinline__ float plateau_ratio_fast(unsigned n, float P2, double c) {
    const double u = __builtin_fma((double)n, c, 0.5 * c);
    const float uf = (float)u;
    const float rs = __builtin_amdgcn_rsqf(uf);
    const double s0 = (double)(uf * rs), h = (double)(0.5f * rs);
    const double s = __builtin_fma(__builtin_fma(-s0, s0, u), h, s0);
    constexpr double eps = 0x1p-42;
    const float lo = (float)__builtin_fma(s, -eps, s), hi = (float)__builtin_fma(s, eps, s);
    return lo == hi ? lo : plateau_ratio(n, P2);  // NaN takes the exact path too
}

// Beads whose neighbour lists are walked one per quad are ordered by list
// length, longest first, bead order inside a class, so that the quads of a
// wave walk lists of similar length.  Nine classes (>= 64, 48, 36, 28, 22, 16,
// 11, 6, 1 pairs) where the order decides which thread sums a bead's receptor
// mode gradients; sixteen by the number of four-entry steps (>= 19, 18, 16,
// 14, 12, then one class per number) where it decides no bit or only the last: the rigid kernels,
// whose walks take 6 % fewer steps for 7 ballots more per 64 beads (1000/300).
// The class of a bead with cnt > 0 listed neighbours:
struct Classes9 {
    static constexpr unsigned kNum = 9;
    static __device__ __forceinline__ unsigned of(unsigned cnt) {
        return (unsigned)(cnt < 64u) + (cnt < 48u) + (cnt < 36u) + (cnt < 28u) + (cnt < 22u) +
               (cnt < 16u) + (cnt < 11u) + (cnt < 6u);
    }
};
struct Classes16 {
    static constexpr unsigned kNum = 16;
    static __device__ __forceinline__ unsigned of(unsigned cnt) {
        const unsigned steps = (min(cnt, 76u) + 3u) / 4u;
        return steps <= 12u ? 16u - steps : (21u - steps) / 2u - (steps == 19u ? 1u : 0u);
    }
};
constexpr unsigned kQueueChunks = 6;  // chunks of 64 beads per wave at most (5 bits each, packed)
template <class Classes>
__host__ __device__ constexpr unsigned queue_counters(unsigned beads) {
    return Classes::kNum * ((beads + 63) / 64) + 1;
}

// The classes of a thread's beads of a super-chunk (beads tid, tid + threads,
// ...: at most kQueueChunks), five bits each.
template <class Classes>
__device__ __forceinline__ unsigned pack_class(unsigned packed, unsigned u, unsigned cnt) {
    return packed | (cnt ? Classes::of(cnt) : Classes::kNum) << (5 * u);
}

// Inclusive prefix sum over the 64 lanes of a wave (DPP: row shifts of 1, 2, 4
// and 8 lanes, then the row totals broadcast).
__device__ __forceinline__ unsigned wave_scan(unsigned v) {
    v += (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false);
    v += (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, false);
    v += (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, false);
    v += (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, false);
    v += (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false);
    v += (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false);
    return v;
}

// The listed beads among beads 0..m-1 of a super-chunk (m <= 64 * CHUNKS per
// wave), in class order, into s_q; returns their number.  Run by WAVES waves
// with sync() a barrier over them; `classes` are each thread's (pack_class);
// s_cc holds queue_counters(m) counters: per (class, chunk of 64 beads) the
// number of listed beads, then their exclusive prefix in (class, chunk) order.
// Bound by latency (14k cycles per super-chunk with a serial scan by one
// thread, 5k so): one set of ballots gives every bead its rank among the
// chunk's beads of its class, and one wave scans the counters.
template <class Classes, int WAVES, unsigned CHUNKS, class Sync>
__device__ __forceinline__ unsigned class_queue(unsigned classes, unsigned m, unsigned short* s_q,
                                                unsigned* s_cc, unsigned tid, Sync sync) {
    constexpr unsigned K = Classes::kNum;
    static_assert(CHUNKS <= kQueueChunks, "packed classes");
    const unsigned lane = tid & (kWave - 1), wv = tid / kWave;
    const unsigned chunks = (m + kWave - 1) / kWave;
    unsigned rank[CHUNKS];
#pragma unroll
    for (unsigned u = 0; u < CHUNKS; ++u) {
        rank[u] = 0;
        const unsigned ch = wv + u * WAVES;
        if (ch >= chunks) continue;  // uniform per wave
        const unsigned cls = ch * kWave + lane < m ? (classes >> (5 * u)) & 31u : K;
        unsigned total = 0;
#pragma unroll
        for (unsigned q = 0; q < K; ++q) {
            const unsigned long long b = __ballot(cls == q);
            const unsigned below = __builtin_amdgcn_mbcnt_hi((unsigned)(b >> 32),
                                                             __builtin_amdgcn_mbcnt_lo((unsigned)b, 0u));
            rank[u] = cls == q ? below : rank[u];
            total = lane == q ? (unsigned)__popcll(b) : total;
        }
        if (lane < K) s_cc[lane * chunks + ch] = total;
    }
    sync();
    const unsigned entries = K * chunks;
    if (wv == 0) {
        constexpr unsigned kPer = (K * CHUNKS * WAVES + kWave - 1) / kWave;  // consecutive, per lane
        unsigned v[kPer], sum = 0;
#pragma unroll
        for (unsigned i = 0; i < kPer; ++i) {
            const unsigned e = lane * kPer + i;
            v[i] = e < entries ? s_cc[e] : 0u;
            sum += v[i];
        }
        const unsigned incl = wave_scan(sum);
        unsigned run = incl - sum;
#pragma unroll
        for (unsigned i = 0; i < kPer; ++i) {
            const unsigned e = lane * kPer + i;
            if (e < entries) s_cc[e] = run;
            run += v[i];
        }
        if (lane == kWave - 1) s_cc[entries] = incl;
    }
    sync();
#pragma unroll
    for (unsigned u = 0; u < CHUNKS; ++u) {
        const unsigned ch = wv + u * WAVES;
        if (ch >= chunks) continue;
        const unsigned cls = ch * kWave + lane < m ? (classes >> (5 * u)) & 31u : K;
        if (cls < K) s_q[s_cc[cls * chunks + ch] + rank[u]] = (unsigned short)(ch * kWave + lane);
    }
    const unsigned total = s_cc[entries];
    sync();
    return total;
}

// The value of lane K of this lane's quad (four consecutive lanes, all active).
template <int K>
__device__ __forceinline__ float quad_lane(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), K * 0x55, 0xf, 0xf, true));
}

// acc + the quad's four values, added one after the other in lane order.
__device__ __forceinline__ float quad_fold(float acc, float v) {
    acc += quad_lane<0>(v);
    acc += quad_lane<1>(v);
    acc += quad_lane<2>(v);
    acc += quad_lane<3>(v);
    return acc;
}

// Butterfly sum over the 64 lanes of a wave (same value on every lane).
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) v += __shfl_xor(v, m);
    return v;
}

// The same over unsigned counters (exact: any order gives the same sum).
__device__ __forceinline__ unsigned wave_sum_u(unsigned v) {
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) v += __shfl_xor(v, m);
    return v;
}

// reducePotForce clamp (model/reduction.h:60-72); x *= 0.01 is a double multiply.
__device__ __forceinline__ void force_clamp(float& x, float& y, float& z) {
#pragma unroll
    for (int it = 0; it < 3; ++it) {
        const float magn2 = x * x + y * y + z * z;
        if (magn2 > 1.0e18f) {
            x = (float)((double)x * 0.01);
            y = (float)((double)y * 0.01);
            z = (float)((double)z * 0.01);
        }
    }
}

// correctModeForce (model/reduction_modes.h:100-115): d += 4 k d^4, the power in double.
__device__ __forceinline__ float correct_mode(float d, float k) {
    const double dd = (double)d, d2 = dd * dd;
    const float cf = (float)((double)(4.f * k) * (d2 * d2));
    return d + cf;
}

// Byte offset of the adjoint's parameter-derivative slices behind the pair
// table in its dynamic LDS.
__host__ __device__ constexpr size_t adjoint_pg_offset(unsigned tabSlots) {
    return (sizeof(att_pair_params) * (size_t)tabSlots + 15) & ~(size_t)15;
}

// Key of a grid-cell record: cells (inner grid first) in buckets of 2^cellBits,
// key = bucket << lowBits | (type - 1) << cellBits | cell in its bucket.  A
// bucket is one cell (cellBits 0) for the run pass.
struct PgKeys {
    unsigned cellsIn, cellBits, lowBits;
    unsigned invalid;  // number of buckets << lowBits: no grid term
    __host__ __device__ unsigned key(unsigned cell, unsigned type) const {
        return (cell >> cellBits) << lowBits | (type - 1u) << cellBits | (cell & ((1u << cellBits) - 1u));
    }
};

constexpr unsigned kQueueStride = 64;  // words: counters lie in cache lines of their own

// Everything the adjoint of one pose needs about its receptor-ligand pair.
struct PairDesc {
    DProt rec, lig;
    DGrid inner, outer;
    DNL nl;
    DPar par;
    DBasis bin, bout;
    const float* dofs;   // n * dofStride floats
    const float* wts;    // n upstream weights, or nullptr (all 1)
    float* out;          // n * outStride floats
    unsigned dofStride, outStride, n, tabSlots;
    const unsigned* nDev;  // when set, the number of poses is read here at launch (<= n)
    const unsigned* order; // when set, a spatial permutation of the poses (XCD ranges)
    unsigned* queues;      // and, when set, zeroed counters of the ranges, kQueueStride apart
    // Grid part of the parameter gradient as records (when set): slot i's bead
    // k writes recKey/recPos[i * lig.n + k]; keys as PgKeys packs them, below
    // recKeys.invalid, that value for beads without a grid term.
    // Positions as {x, y, z, w} (recPos4), or {x, y, z} when the call has no
    // weights (recPos3; w = 1).
    unsigned* recKey;
    float4* recPos4;
    float3* recPos3;
    PgKeys recKeys;
    // when set, per pose {listed neighbours of the beads walked, pairs inside
    // the plateau}
    uint2* counts;
};

// Slot of workgroup b among nb in a non-persistent launch such that the
// workgroups of one XCD (dispatched round-robin: b % 8) take one contiguous
// range of slots: XCD x holds ceil((nb - x) / 8) workgroups, and its range
// starts after those of XCDs 0..x-1.  A bijection of [0, nb).
__device__ __forceinline__ unsigned xcd_slot(unsigned b, unsigned nb) {
    const unsigned x = b & 7u, q = nb >> 3, r = nb & 7u;
    return x * q + (x < r ? x : r) + (b >> 3);
}

// One unit of batched work: `count` consecutive poses of pair `pair` (in the
// pair's spatial order when it has one).
struct BatchTile {
    unsigned pair, first, count;
};

// Tile queues of a batched launch: one per XCD.
constexpr unsigned kBatchQueues = 8;

struct NoReaction {
    template <class Rec>
    __device__ void operator()(const Rec&, float, float, float) const {}
};

// Mode vectors of bead i (modes stored [c][m][n], coalesced over beads); MM
// is the compile-time capacity (>= the body's number of modes).
template <int MM>
struct BeadModes {
    float x[MM > 0 ? MM : 1], y[MM > 0 ? MM : 1], z[MM > 0 ? MM : 1];
};

template <int MM>
__device__ __forceinline__ void load_modes(const DProt& b, unsigned i, BeadModes<MM>& md) {
    const size_t nM = (size_t)b.M * b.n;
#pragma unroll
    for (unsigned m = 0; m < (unsigned)MM; ++m) {
        md.x[m] = m < b.M ? b.modes[(size_t)m * b.n + i] : 0.f;
        md.y[m] = m < b.M ? b.modes[nM + (size_t)m * b.n + i] : 0.f;
        md.z[m] = m < b.M ? b.modes[2 * nM + (size_t)m * b.n + i] : 0.f;
    }
}

// The row of bead i, f = {type bits, m0x, m0y, m0z, m1x, ...}, zero beyond the
// body's modes up to the capacity MM (4 * ceil((3 MM + 1) / 4) floats).
template <int MM>
__device__ __forceinline__ void load_row(const DProt& b, unsigned i, float* f) {
    constexpr unsigned Q = (3 * MM + 4) / 4;
    const float4* row = b.modesT + (size_t)i * b.rowT;
    float4 v[Q];
    if (b.rowT >= Q) {  // uniform; the loads issue together
#pragma unroll
        for (unsigned q = 0; q < Q; ++q) v[q] = row[q];
    } else {
#pragma unroll
        for (unsigned q = 0; q < Q; ++q) v[q] = q < b.rowT ? row[q] : make_float4(0.f, 0.f, 0.f, 0.f);
    }
#pragma unroll
    for (unsigned q = 0; q < Q; ++q) {
        f[4 * q] = v[q].x; f[4 * q + 1] = v[q].y; f[4 * q + 2] = v[q].z; f[4 * q + 3] = v[q].w;
    }
}

// A receptor bead as the list walks need it: position (deformed by the
// amplitudes amp, zero beyond the receptor's modes; the order of deform()),
// charge, type, and its row for the projections on the modes.
template <int MM>
struct RecBead {
    float x, y, z, q;
    unsigned type;
    unsigned index;  // with modes only
    float row[MM > 0 ? 4 * ((3 * MM + 4) / 4) : 1];

    __device__ __forceinline__ void load(const DProt& rec, unsigned j, const float* amp) {
        const float4 p = rec.pos[j];
        x = p.x; y = p.y; z = p.z; q = p.w;
        load_row<MM>(rec, j, row);
        type = __float_as_uint(row[0]);
#pragma unroll
        for (unsigned m = 0; m < (unsigned)MM; ++m) {
            x = x + amp[m] * row[3 * m + 1];
            y = y + amp[m] * row[3 * m + 2];
            z = z + amp[m] * row[3 * m + 3];
        }
    }
};

// The receptor beads of a list, every fourth entry from entry `at` on (clamped
// to the last one).  With modes the next entry's index is loaded one step
// ahead; without, the next bead itself and the index after it: five registers,
// 3 % of the rigid kernels.  (With modes the row ahead is 20 or 36 registers,
// and its spills cost more than the latency: 3 and 9 % slower.)
template <int MM>
struct RecStream {
    unsigned idx, type;
    float4 p;
    __device__ __forceinline__ RecStream(const DProt& rec, const uint32_t* lst, unsigned at, unsigned last) {
        idx = lst[min(at, last)];
        if constexpr (MM == 0) {
            p = rec.pos[idx];
            type = rec.type[idx];
            idx = lst[min(at + 4, last)];
        }
    }
    __device__ __forceinline__ void next(const DProt& rec, const uint32_t* lst, unsigned at,
                                         unsigned last, const float* amp, RecBead<MM>& rb) {
        const unsigned j = idx;
        if constexpr (MM == 0) {
            rb.x = p.x; rb.y = p.y; rb.z = p.z; rb.q = p.w;
            rb.type = type;
            p = rec.pos[j];
            type = rec.type[j];
            idx = lst[min(at + 8, last)];
        } else {
            idx = lst[min(at + 4, last)];
            rb.index = j;
            rb.load(rec, j, amp);
        }
    }
};

// The pair loop of NLPotForce for one ligand bead (model/neighborlist.h:66-158
// and the receptor reaction of model/neighborlist_modes.h:68-194), by the four
// lanes of a quad (s = lane in the quad) over the list d = {numEl, idx}
// (numEl > 0): each step takes four consecutive list entries, one per lane, and
// the four pairs' terms are then added to and subtracted from the bead's
// accumulators in list order on every lane, so every lane returns the
// reference's bits.  A pair outside the plateau, or past the
// list's end, adds zeros (an accumulator that starts at +0 never becomes -0,
// so that changes no bit).  reaction(rec, fx, fy, fz) receives each lane's
// pair's reaction force (zero for those).  Bound like the adjoint's adj_walk;
// 100,000 rigid poses (1000/300): 4.43 -> 3.42 ms against one lane per bead,
// 20,011 flexible ones (3000/800, 5 + 5 modes) 6.22 -> 5.08 ms.
template <int MM, class Reaction>
__device__ __forceinline__ float4 nl_walk_quad(const DNL& nl, const DPar& par, const PairTab& tab,
                                               const DProt& rec, const float* ampR,
                                               Reaction reaction, float px, float py, float pz,
                                               unsigned ligType, float ligCharge, uint2 d,
                                               unsigned s, unsigned& inside) {
    float fx = 0.f, fy = 0.f, fz = 0.f, e = 0.f;
    const unsigned lt1 = ligType - 1, last = d.x - 1;
    const uint32_t* lst = nl.list + d.y;
    RecStream<MM> recs(rec, lst, s, last);
    for (unsigned jj = 0; jj < d.x; jj += 4) {
        RecBead<MM> rb;
        recs.next(rec, lst, jj + s, last, ampR, rb);
        const float ddx = px - rb.x, ddy = py - rb.y, ddz = pz - rb.z;
        const float dr2 = ddx * ddx + ddy * ddy + ddz * ddz;
        const bool in = jj + s < d.x && dr2 <= nl.P2 && rb.type - 1u < par.T;
        inside += in ? 1u : 0u;
        const float ratio = in ? plateau_ratio_fast((unsigned)(int)(dr2 * 10000.f), nl.P2, nl.ratioC) : 0.f;
        const float dr2_inv = (float)(1.0 / (double)dr2);
        const float dx = ddx * dr2_inv, dy = ddy * dr2_inv, dz = ddz * dr2_inv;
        const att_pair_params p = tab[in ? par.T * (rb.type - 1) + lt1 : 0u];
        float vx, vy, vz, ve, wx, wy, wz, we;  // at r, at the plateau
        lj(dr2, dr2_inv, dx, dy, dz, p, par.shape, vx, vy, vz, ve);
        const float rdx = ratio * dx, rdy = ratio * dy, rdz = ratio * dz;
        lj(nl.P2, nl.P2_inv, rdx, rdy, rdz, p, par.shape, wx, wy, wz, we);
        if (!in) { vx = vy = vz = ve = 0.f; wx = wy = wz = we = 0.f; }
        float rfx = wx - vx, rfy = wy - vy, rfz = wz - vz;  // -v + w: (0 - v) + w exactly
        const float qlr = ligCharge * rb.q * par.ffelec;
        const bool charged = in && fabsf(qlr) > 0.001f;
        if (__any(charged)) {
            float cx, cy, cz, ce, ex, ey, ez, ee;
            coulomb(dr2_inv, dx, dy, dz, qlr, par.dielec, cx, cy, cz, ce);
            coulomb(nl.P2_inv, rdx, rdy, rdz, qlr, par.dielec, ex, ey, ez, ee);
            if (!charged) { cx = cy = cz = ce = 0.f; ex = ey = ez = ee = 0.f; }
            rfx = (rfx - cx) + ex; rfy = (rfy - cy) + ey; rfz = (rfz - cz) + ez;
            auto fold = [](float acc, float a, float b, float c, float g) __attribute__((always_inline)) {
                acc += quad_lane<0>(a); acc -= quad_lane<0>(b); acc += quad_lane<0>(c); acc -= quad_lane<0>(g);
                acc += quad_lane<1>(a); acc -= quad_lane<1>(b); acc += quad_lane<1>(c); acc -= quad_lane<1>(g);
                acc += quad_lane<2>(a); acc -= quad_lane<2>(b); acc += quad_lane<2>(c); acc -= quad_lane<2>(g);
                acc += quad_lane<3>(a); acc -= quad_lane<3>(b); acc += quad_lane<3>(c); acc -= quad_lane<3>(g);
                return acc;
            };
            fx = fold(fx, vx, wx, cx, ex);
            fy = fold(fy, vy, wy, cy, ey);
            fz = fold(fz, vz, wz, cz, ez);
            e = fold(e, ve, we, ce, ee);
        } else {
            auto fold = [](float acc, float a, float b) __attribute__((always_inline)) {
                acc += quad_lane<0>(a); acc -= quad_lane<0>(b);
                acc += quad_lane<1>(a); acc -= quad_lane<1>(b);
                acc += quad_lane<2>(a); acc -= quad_lane<2>(b);
                acc += quad_lane<3>(a); acc -= quad_lane<3>(b);
                return acc;
            };
            fx = fold(fx, vx, wx);
            fy = fold(fy, vy, wy);
            fz = fold(fz, vz, wz);
            e = fold(e, ve, we);
        }
        reaction(rb, rfx, rfy, rfz);
    }
    return make_float4(fx, fy, fz, e);
}

// Mode deformation x + sum_m a_m * mode_m, sequential over modes
// (model/transform.h:69-73).
template <int MM>
__device__ __forceinline__ V3 deform(const BeadModes<MM>& md, unsigned M, float x, float y,
                                     float z, const float* amp) {
    V3 p{x, y, z};
#pragma unroll
    for (unsigned m = 0; m < (unsigned)MM; ++m) {
        if (m < M) {
            const float a = amp[m];
            p.x = p.x + a * md.x[m];
            p.y = p.y + a * md.y[m];
            p.z = p.z + a * md.z[m];
        }
    }
    return p;
}

// The group (of nthr / 4) whose queue item this thread's quad takes in
// sub-round `sub`.
template <int WAVES>
__device__ __forceinline__ unsigned quad_group(unsigned tid, unsigned sub) {
    const unsigned wave = tid / kWave, quad = (tid & (kWave - 1)) >> 2;
    return (sub & 1u ? WAVES - 1u - wave : wave) * 16u + quad;
}

// A ligand bead's position from its row (one bead per quad: a few loads of one
// address per quad instead of 1 + 3 M), deformed as deform() does and moved by
// (R, t); amp is zero beyond the ligand's modes.
template <int MM>
__device__ __forceinline__ V3 place_from_row(const DProt& lig, unsigned i, const float* amp,
                                             const float* R, float tx, float ty, float tz, float4& x,
                                             unsigned& type) {
    x = lig.pos[i];
    V3 xt{x.x, x.y, x.z};
    if constexpr (MM > 0) {
        float row[4 * ((3 * MM + 4) / 4)];
        load_row<MM>(lig, i, row);
        type = __float_as_uint(row[0]);
#pragma unroll
        for (unsigned m = 0; m < (unsigned)MM; ++m)
            if (m < lig.M) {
                xt.x = xt.x + amp[m] * row[3 * m + 1];
                xt.y = xt.y + amp[m] * row[3 * m + 2];
                xt.z = xt.z + amp[m] * row[3 * m + 3];
            }
    } else {
        type = lig.type[i];
    }
    V3 p = matvec(R, xt.x, xt.y, xt.z);
    p.x = p.x + tx; p.y = p.y + ty; p.z = p.z + tz;
    return p;
}

// Accumulates -f . mode_m into g[m] (model/reduction_modes.h:49-55, 83-86).
template <int MM>
__device__ __forceinline__ void mode_dots(const BeadModes<MM>& md, unsigned M, float fx, float fy,
                                          float fz, float* g) {
#pragma unroll
    for (unsigned m = 0; m < (unsigned)MM; ++m)
        if (m < M) g[m] -= fx * md.x[m] + fy * md.y[m] + fz * md.z[m];
}

// Barrier over the lanes of one wave (LDS written by the wave is visible to it).
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The reference's per-pose reductions of the ligand's bead forces, in bead
// order, one quantity per lane (lanes 0..12 of a wave): reducePotForce's E
// and F (model/reduction.h:39-75) and reduceTorque's tensor sum of x_l * f_k
// over the undeformed coordinates (:80-104) in lane 4 + 3k + l.  Each call
// adds beads f[0..m) (float4 {fx, fy, fz, E}, LDS; zeros up to the next
// multiple of kReduceStep), the body's beads first.., to the lane's running
// sum.  Bound by the latency of a serial chain of adds: each lane reads its
// own component's row (ones where there is no coordinate factor) 16 beads per
// step, the next step's loads in flight.  With the modes' fold below (20,011
// flexible poses 3000/800, 5 + 5 modes) 5.08 -> 4.35 ms, a call of 100 poses 254 ->
// 190 us; 100,000 rigid poses (1000/300) 3.42 -> 3.18 ms, against eight beads
// per step without the next step's loads.
constexpr unsigned kReduceStep = 16;
__device__ __forceinline__ float reduce_beads_ref(float red, unsigned lane, const float4* f,
                                                  const DProt& lig, unsigned first, unsigned m) {
    if (lane >= 13u) return red;
    const unsigned fc = lane == 0 ? 3u : lane < 4u ? lane - 1u : (lane - 4u) / 3u;
    const unsigned xc = lane < 4u ? 3u : (lane - 4u) % 3u;
    const float* ff = reinterpret_cast<const float*>(f) + fc;
    const float4* xr = reinterpret_cast<const float4*>(lig.soa + (size_t)xc * lig.ns + first);
    constexpr unsigned Q = kReduceStep / 4;
    float4 x[Q];
    float v[kReduceStep];
    auto load = [&](unsigned k) __attribute__((always_inline)) {
#pragma unroll
        for (unsigned u = 0; u < Q; ++u) x[u] = xr[k / 4 + u];
#pragma unroll
        for (unsigned u = 0; u < kReduceStep; ++u) v[u] = ff[4 * (k + u)];
    };
    load(0);
    for (unsigned k = 0; k < m; k += kReduceStep) {
        float t[kReduceStep];
#pragma unroll
        for (unsigned u = 0; u < Q; ++u) {
            t[4 * u] = x[u].x * v[4 * u];  // 1 * f = f exactly
            t[4 * u + 1] = x[u].y * v[4 * u + 1];
            t[4 * u + 2] = x[u].z * v[4 * u + 2];
            t[4 * u + 3] = x[u].w * v[4 * u + 3];
        }
        if (k + kReduceStep < m) load(k + kReduceStep);
#pragma unroll
        for (unsigned u = 0; u < kReduceStep; ++u) red += t[u];
    }
    return red;
}

// Beads per super-chunk for n beads and at most smax (a multiple of 64) per
// super-chunk: the fewest super-chunks, of equal size rounded up to 64.
__host__ __device__ inline unsigned super_chunk(unsigned n, unsigned smax) {
    const unsigned parts = n ? (n + smax - 1) / smax : 1u;
    const unsigned per = (n + parts - 1) / parts;
    return (per + 63u) & ~63u;
}

// The epilogue of those reductions, by every lane of the wave that ran them:
// the 13 sums gathered, the force clamped (reducePotForce) and the torque
// tensor contracted with dR/d(angle) (reduceTorque, commons/TorqueMat.h:
// 27-37); out = {E, F[3], dE/dang[3]}.
__device__ __forceinline__ void finish_ref(float red, const float* t, float* out) {
    float v[13];
#pragma unroll
    for (int q = 0; q < 13; ++q) v[q] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(red), q));
    float Fx = v[1], Fy = v[2], Fz = v[3];
    force_clamp(Fx, Fy, Fz);
    float a3[3];
    torque_reduce(t[0], t[1], t[2], t[3], t[4], t[5], v + 4, a3);
    out[0] = v[0]; out[1] = Fx; out[2] = Fy; out[3] = Fz;
    out[4] = a3[0]; out[5] = a3[1]; out[6] = a3[2];
}

}  // namespace att
