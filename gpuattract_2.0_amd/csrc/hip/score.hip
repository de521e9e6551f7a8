// Scoring kernels for gfx950 and their launchers.
//
//  k_rigid  one 64-lane wavefront per pose, four poses per 256-thread workgroup.
//           Lanes stride over ligand beads (transform, grid interpolation,
//           neighbour-list cell), quads of lanes walk the beads' lists, and
//           the reference's bead-order reductions and a one-lane epilogue
//           (force clamp, torque matrix) write the 28-byte result.  Replaces
//           d_DOF2Pos, d_potForce, d_NLPotForce, d_reduce and h_finalReduce
//           (model/*.cu, model/reduction.h:159-207) with one launch and no
//           intermediate buffers.
//  k_modes  one workgroup per pose.  Phase A moves the deformed receptor into
//           the ligand frame and scores it on the ligand grid; phase B scores
//           the ligand on the receptor grid and walks the lists against the
//           receptor beads, deformed per pair from their mode rows, folding
//           the receptor reaction straight into the receptor mode gradients.
//           Semantics of service/CPUEnergyService6DModes.tpp:121-327.
#include <algorithm>

#include "device.h"
#include "internal.h"

namespace att {

// The LDS of one pose of k_rigid with WP waves per pose: a super-chunk's beads'
// force and energy, the class-ordered queue and its counters, pair counts.
template <int WP>
struct RigidLDS {
    static constexpr unsigned kChunks = WP > 4 ? 3 : kQueueChunks;  // per wave
    static constexpr unsigned kSuper = 64 * kChunks * WP;
    float4 f[kSuper];
    unsigned short q[kSuper];
    unsigned cc[queue_counters<Classes16>(kSuper)];
    unsigned cnt[WP][2];
};

// WP waves per pose: one (four poses per workgroup) or, for calls of few poses,
// a workgroup of four or eight.  Every per-bead sum and the bead-order
// reductions are the same in any of them: the same bits.
template <int WP>
__global__ __launch_bounds__(WP > 4 ? 64 * WP : 256) __attribute__((amdgpu_waves_per_eu(4))) void k_rigid(
    DProt rec, DProt lig, DGrid inner, DGrid outer, DNL nl, DPar par, const float* __restrict__ dofs,
    float* __restrict__ res, unsigned n, unsigned tabBytes, const unsigned* __restrict__ order,
    uint2* __restrict__ counts) {
    extern __shared__ __align__(16) att_pair_params s_tab[];
    using LDS = RigidLDS<WP>;
    const PairTab tab = stage_table(par, s_tab);
    __syncthreads();
    constexpr unsigned nthr = kWave * WP;
    const unsigned group = threadIdx.x / nthr, tid = threadIdx.x % nthr;  // group: pose of the workgroup
    const unsigned lane = tid & (kWave - 1), wave = tid / kWave;
    LDS& L = reinterpret_cast<LDS*>(reinterpret_cast<char*>(s_tab) + tabBytes)[group];
    float4* s_f = L.f;
    auto sync = [] {
        if constexpr (WP == 1) wave_sync(); else __syncthreads();
    };
    const unsigned wg = order ? xcd_slot(blockIdx.x, gridDim.x) : blockIdx.x;
    const unsigned slot = wg * (blockDim.x / nthr) + group;
    if (slot >= n) return;  // uniform per pose; with one wave per pose no workgroup barrier follows
    const unsigned pose = order ? order[slot] : slot;
    const float* d = dofs + 6 * (size_t)pose;
    const float tx = uniform(d[0]), ty = uniform(d[1]), tz = uniform(d[2]);
    float t[6];
    pose_trig(d[3], d[4], d[5], lane, t);
    float R[9];
    rotmat_from_trig(t[0], t[1], t[2], t[3], t[4], t[5], R);
#pragma unroll
    for (int k = 0; k < 9; ++k) R[k] = uniform(R[k]);
    auto place = [&](unsigned i, float4& x) {
        x = lig.pos[i];
        V3 p = matvec(R, x.x, x.y, x.z);
        p.x = p.x + tx; p.y = p.y + ty; p.z = p.z + tz;
        return p;
    };
    float red = 0.f;  // the reference's reduction held by this lane (reduce_beads_ref)
    unsigned listed = 0, inside = 0;  // this lane's pair counts (counts != nullptr)
    const unsigned span = super_chunk(lig.n, LDS::kSuper);
    for (unsigned sc = 0; sc < lig.n; sc += span) {
        const unsigned m = min(span, lig.n - sc);
        // P1: one bead per lane: rotate_translate, potForce, the list's cell.
        const unsigned padded = (m + kReduceStep - 1) & ~(kReduceStep - 1);
        if (m + tid < padded) s_f[m + tid] = make_float4(0.f, 0.f, 0.f, 0.f);
        unsigned classes = 0;
        for (unsigned k = tid, u = 0; k < m; k += nthr, ++u) {
            float4 x;
            const V3 p = place(sc + k, x);
            s_f[k] = pot_bead(inner, outer, p.x, p.y, p.z, lig.mtype[sc + k], x.w, nullptr);
            classes = pack_class<Classes16>(classes, u, nl_cell(nl, p.x, p.y, p.z, lig.type[sc + k]).x);
        }
        sync();
        // P2: beads with a list, longest lists first.
        const unsigned qn = class_queue<Classes16, WP, LDS::kChunks>(classes, m, L.q, L.cc, tid, sync);
        // P3: one bead per quad of lanes walks its list in the reference's
        // order (NLPotForce); its sums are added to the bead's grid values as
        // outLig[i] += fAcc.
        for (unsigned q0 = 0, round = 0; q0 < qn; q0 += nthr / 4, ++round) {
            const unsigned item = q0 + quad_group<WP>(tid, round);
            if (item < qn) {
                const unsigned k = L.q[item];
                float4 x;
                const V3 p = place(sc + k, x);
                const unsigned lt = lig.type[sc + k];
                const uint2 cell = nl_cell(nl, p.x, p.y, p.z, lt);
                const float4 a = nl_walk_quad<0>(nl, par, tab, rec, nullptr, NoReaction{}, p.x, p.y,
                                                 p.z, lt, x.w, cell, lane & 3u, inside);
                if ((lane & 3u) == 0) {
                    listed += cell.x;
                    float4 f = s_f[k];
                    f.x = f.x + a.x; f.y = f.y + a.y; f.z = f.z + a.z; f.w = f.w + a.w;
                    s_f[k] = f;
                }
            }
        }
        sync();
        // P4: reducePotForce and reduceTorque, in bead order.
        if (wave == 0) red = reduce_beads_ref(red, lane, s_f, lig, sc, m);
        sync();  // the super-chunk's arrays are reused
    }
    if (counts) {
        listed = wave_sum_u(listed);
        inside = wave_sum_u(inside);
        if (lane == 0) { L.cnt[wave][0] = listed; L.cnt[wave][1] = inside; }
        sync();
    }
    if (wave != 0) return;
    float o[7];
    finish_ref(red, t, o);
    if (lane == 0) {
        float* r = res + 7 * (size_t)pose;
#pragma unroll
        for (int q = 0; q < 7; ++q) r[q] = o[q];
        if (counts) {
            uint2 c = make_uint2(0u, 0u);
            for (int w = 0; w < WP; ++w) { c.x += L.cnt[w][0]; c.y += L.cnt[w][1]; }
            counts[pose] = c;
        }
    }
}

// reduceModeForce of the ligand (model/reduction_modes.h:28-57) over beads
// f[0..m) (LDS) of a super-chunk starting at bead sc, in bead order: red -=
// (R^T f) . mode, mode mm in lane mm of one wave.  The terms of 64 beads are
// formed one bead per lane, left in `tile`, and subtracted by the modes'
// lanes one after the other: only the subtractions are serial.
template <int MM>
struct ModeTile {
    static constexpr unsigned kRow = 68;  // 64 terms, padded: the modes' rows in different banks
    alignas(16) float t[(MM > 0 ? MM : 1) * kRow];
};
template <int MM>
__device__ __forceinline__ float reduce_modes_ref(float red, const float* RT, const float4* f,
                                                  const DProt& lig, ModeTile<MM>& tile,
                                                  unsigned lane, unsigned sc, unsigned m) {
    for (unsigned c = 0; c < m; c += kWave) {
        const unsigned k = c + lane;
        BeadModes<MM> md;
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (k < m) {
            v = f[k];
            load_modes(lig, sc + k, md);
        }
        const V3 fa = matvec(RT, v.x, v.y, v.z);
#pragma unroll
        for (unsigned mm = 0; mm < (unsigned)MM; ++mm)
            if (mm < lig.M)
                tile.t[mm * ModeTile<MM>::kRow + lane] =
                    k < m ? fa.x * md.x[mm] + fa.y * md.y[mm] + fa.z * md.z[mm] : 0.f;
        wave_sync();
        if (lane < lig.M) {
            const float4* row = reinterpret_cast<const float4*>(&tile.t[lane * ModeTile<MM>::kRow]);
#pragma unroll
            for (unsigned u = 0; u < kWave / 4; ++u) {
                const float4 q = row[u];
                red -= q.x; red -= q.y; red -= q.z; red -= q.w;
            }
        }
        wave_sync();
    }
    return red;
}

// One workgroup of W waves per pose (W = 1 below 384 ligand beads, else 4;
// att_set_modes_waves overrides it).
// Phase A: every receptor bead deformed and moved into the ligand frame
// (invertDOF, rotate_translate_deform), scored on the ligand grid, its force
// rotated back (rotate_forces) and projected on the receptor modes.  Phase B:
// the ligand in super-chunks of at most 256 * W beads, as k_rigid: grid term and list
// cell per bead (P1), the class-ordered queue (P2), one bead per quad of lanes walking
// its list in the reference's order against the deformed receptor (each
// receptor bead deformed again from its mode row, so receptors of any size
// need no LDS) with the reaction projected on the receptor modes (P3), and
// the reference's bead-order reductions (P4): E, F and the torque tensor in
// lanes 0..12 of wave 0, the ligand's reduceModeForce in lanes of the last
// wave.  Semantics of service/CPUEnergyService6DModes.tpp:121-327.
// Occupancy: at least 4 waves per SIMD, 3 with 10 modes (0-16 B of scratch per lane
// there; at 4 waves 10,000 poses 3000/800 2.93 -> 2.78 ms, 1000/300 1.13 -> 1.18, a
// call of 100 186 -> 194 us).
template <int MM, int W>
__global__ __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(MM >= 10 ? 3 : 4))) void k_modes(DProt rec, DProt lig, DGrid rInner, DGrid rOuter,
                                                  DNL nl, DGrid lInner, DGrid lOuter, DPar par,
                                                  const float* __restrict__ dofs,
                                                  float* __restrict__ res, unsigned n,
                                                  const unsigned* __restrict__ order,
                                                  uint2* __restrict__ counts) {
    constexpr unsigned kSuper = 256u * W;
    extern __shared__ __align__(16) att_pair_params s_tab[];
    __shared__ float4 s_f[kSuper];
    __shared__ uint2 s_n[kSuper];
    __shared__ unsigned short s_q[kSuper];
    __shared__ unsigned s_cc[queue_counters<Classes16>(kSuper)];
    __shared__ float s_red[W][ATT_MODES_MAX];
    __shared__ float s_gl[ATT_MODES_MAX];
    __shared__ ModeTile<MM> s_tile;
    __shared__ unsigned s_cnt[W][2];
    const PairTab tab = stage_table(par, s_tab);  // visible after phase B's first barrier
    if (blockIdx.x >= n) return;  // uniform per workgroup
    const unsigned pose = order ? order[xcd_slot(blockIdx.x, gridDim.x)] : blockIdx.x;
    const unsigned tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
    constexpr unsigned nthr = 64u * W;
    constexpr unsigned modeWave = W - 1;  // runs the ligand's reduceModeForce
    const float* d = dofs + 26 * (size_t)pose;
    const float tx = uniform(d[0]), ty = uniform(d[1]), tz = uniform(d[2]);
    constexpr int MA = MM > 0 ? MM : 1;
    float ampR[MA], ampL[MA];
#pragma unroll
    for (int m = 0; m < MA; ++m) {
        ampR[m] = m < (int)rec.M ? uniform(d[6 + m]) : 0.f;
        ampL[m] = m < (int)lig.M ? uniform(d[16 + m]) : 0.f;
    }
    float t[6];
    pose_trig(d[3], d[4], d[5], lane, t);
    float R[9], RT[9], Rinv[9];
    rotmat_from_trig(t[0], t[1], t[2], t[3], t[4], t[5], R);
#pragma unroll
    for (int k = 0; k < 9; ++k) R[k] = uniform(R[k]);
    RT[0] = R[0]; RT[1] = R[3]; RT[2] = R[6];
    RT[3] = R[1]; RT[4] = R[4]; RT[5] = R[7];
    RT[6] = R[2]; RT[7] = R[5]; RT[8] = R[8];
    // invertDOF (model/transform_modes.h:26-41): rotation R(-ang) (cos even,
    // sin odd), translation R^T (-pos).
    rotmat_from_trig(t[0], t[1], -t[2], -t[3], t[4], -t[5], Rinv);
#pragma unroll
    for (int k = 0; k < 9; ++k) Rinv[k] = uniform(Rinv[k]);
    V3 pinv = matvec(RT, -tx, -ty, -tz);
    pinv.x = uniform(pinv.x); pinv.y = uniform(pinv.y); pinv.z = uniform(pinv.z);

    float mR[MA];
#pragma unroll
    for (int m = 0; m < MA; ++m) mR[m] = 0.f;

    // Phase A: receptor beads, two lookups in flight per lane (pot_bead_flat).
#pragma unroll 2
    for (unsigned j = tid; j < rec.n; j += nthr) {
        const float4 x = rec.pos[j];
        BeadModes<MM> md;
        load_modes(rec, j, md);
        const V3 df = deform(md, rec.M, x.x, x.y, x.z, ampR);
        V3 p = matvec(Rinv, df.x, df.y, df.z);
        p.x = p.x + pinv.x; p.y = p.y + pinv.y; p.z = p.z + pinv.z;
        const float4 pot = pot_bead_flat(lInner, lOuter, p.x, p.y, p.z, rec.mtype[j], x.w);
        const V3 f = matvec(R, pot.x, pot.y, pot.z);  // rotate_forces (transform_modes.h:141-161)
        mode_dots(md, rec.M, f.x, f.y, f.z, mR);
    }

    // Phase B: ligand beads.
    const unsigned Mr = rec.M;
    auto reaction = [&](const RecBead<MM>& rb, float fx, float fy, float fz) {
#pragma unroll
        for (unsigned m = 0; m < (unsigned)MM; ++m)
            if (m < Mr) mR[m] -= fx * rb.row[3 * m + 1] + fy * rb.row[3 * m + 2] + fz * rb.row[3 * m + 3];
    };
    auto place = [&](unsigned i, float4& x) {
        x = lig.pos[i];
        BeadModes<MM> md;
        load_modes(lig, i, md);
        const V3 df = deform(md, lig.M, x.x, x.y, x.z, ampL);
        V3 p = matvec(R, df.x, df.y, df.z);
        p.x = p.x + tx; p.y = p.y + ty; p.z = p.z + tz;
        return p;
    };
    const unsigned nL = lig.n;
    auto place_row = [&](unsigned i, float4& x, unsigned& lt) {
        return place_from_row<MM>(lig, i, ampL, R, tx, ty, tz, x, lt);
    };
    float red = 0.f, redM = 0.f;  // wave 0: E, F, torque tensor; modeWave: ligand modes
    unsigned listed = 0, inside = 0;  // this lane's pair counts (counts != nullptr)
    const unsigned span = super_chunk(nL, kSuper);
    for (unsigned sc = 0; sc < nL; sc += span) {
        const unsigned m = min(span, nL - sc);
        // P1
        const unsigned padded = (m + kReduceStep - 1) & ~(kReduceStep - 1);
        if (m + tid < padded) s_f[m + tid] = make_float4(0.f, 0.f, 0.f, 0.f);
        unsigned classes = 0;
        for (unsigned k = tid, u = 0; k < m; k += nthr, ++u) {
            float4 x;
            const V3 p = place(sc + k, x);
            s_f[k] = pot_bead(rInner, rOuter, p.x, p.y, p.z, lig.mtype[sc + k], x.w, nullptr);
            const uint2 cell = nl_cell(nl, p.x, p.y, p.z, lig.type[sc + k]);
            s_n[k] = cell;
            classes = pack_class<Classes16>(classes, u, cell.x);
        }
        __syncthreads();
        // P2
        const unsigned qn = class_queue<Classes16, W, 4>(classes, m, s_q, s_cc, tid, [] { __syncthreads(); });
        // P3
        for (unsigned q0 = 0, round = 0; q0 < qn; q0 += nthr / 4, ++round) {
            const unsigned item = q0 + quad_group<W>(tid, round);
            if (item < qn) {
                const unsigned k = s_q[item];
                float4 x;
                unsigned lt;
                const V3 p = place_row(sc + k, x, lt);
                const float4 a = nl_walk_quad<MM>(nl, par, tab, rec, ampR, reaction, p.x, p.y, p.z,
                                                  lt, x.w, s_n[k], lane & 3u, inside);
                if ((lane & 3u) == 0) {
                    listed += s_n[k].x;
                    float4 f = s_f[k];
                    f.x = f.x + a.x; f.y = f.y + a.y; f.z = f.z + a.z; f.w = f.w + a.w;
                    s_f[k] = f;
                }
            }
        }
        __syncthreads();
        // P4: reducePotForce, reduceTorque and the ligand's reduceModeForce, in
        // bead order.
        if (wave == 0) red = reduce_beads_ref(red, lane, s_f, lig, sc, m);
        if (MM > 0 && wave == modeWave) redM = reduce_modes_ref<MM>(redM, RT, s_f, lig, s_tile, lane, sc, m);
        __syncthreads();  // the super-chunk's arrays are reused
    }

    // Receptor mode gradients: wave butterflies, then the waves in order.
#pragma unroll
    for (int m = 0; m < MM; ++m) mR[m] = wave_sum(mR[m]);
    if (lane == 0) {
#pragma unroll
        for (int m = 0; m < ATT_MODES_MAX; ++m) s_red[wave][m] = m < MM ? mR[m < MM ? m : 0] : 0.f;
    }
    if (wave == modeWave && lane < ATT_MODES_MAX) s_gl[lane] = redM;
    if (counts) {
        listed = wave_sum_u(listed);
        inside = wave_sum_u(inside);
        if (lane == 0) { s_cnt[wave][0] = listed; s_cnt[wave][1] = inside; }
    }
    __syncthreads();
    if (counts && threadIdx.x == 0) {
        uint2 c = make_uint2(0u, 0u);
        for (int w = 0; w < W; ++w) { c.x += s_cnt[w][0]; c.y += s_cnt[w][1]; }
        counts[pose] = c;
    }
    if (wave == 0) {
        float o[7];
        finish_ref(red, t, o);
        if (lane == 0) {
            float* r = res + 27 * (size_t)pose;
#pragma unroll
            for (int q = 0; q < 7; ++q) r[q] = o[q];
            for (unsigned m = 0; m < ATT_MODES_MAX; ++m) {
                float s = s_red[0][m];
                for (int w = 1; w < W; ++w) s += s_red[w][m];
                r[7 + m] = m < rec.M ? correct_mode(s, rec.modeForce[m]) : 0.f;
                r[17 + m] = m < lig.M ? correct_mode(s_gl[m], lig.modeForce[m]) : 0.f;
            }
        }
    }
}

// ---------------------------------------------------------------- diagnostics

// One wave; the beads' lists are walked as the scoring kernels walk them, one
// bead per quad of lanes, with the pair table in LDS where theirs is.
__global__ void k_debug_rigid(DProt rec, DProt lig, DGrid inner, DGrid outer, DNL nl, DPar par,
                              const float* dof, float* xyz, float* pot, int* cell,
                              unsigned* npairs) {
    extern __shared__ __align__(16) att_pair_params s_tab[];
    const PairTab tab = stage_table(par, s_tab);
    __syncthreads();
    const unsigned lane = threadIdx.x;
    float t[6];
    pose_trig(dof[3], dof[4], dof[5], lane, t);
    float R[9];
    rotmat_from_trig(t[0], t[1], t[2], t[3], t[4], t[5], R);
    const unsigned n = lig.n;
    for (unsigned i = lane >> 2; i < n; i += kWave / 4) {
        const float4 x = lig.pos[i];
        V3 p = matvec(R, x.x, x.y, x.z);
        p.x = p.x + dof[0]; p.y = p.y + dof[1]; p.z = p.z + dof[2];
        int c[9];
        for (int k = 0; k < 9; ++k) c[k] = -1;
        float4 pp = pot_bead(inner, outer, p.x, p.y, p.z, lig.mtype[i], x.w, c);
        const uint2 d = nl_cell(nl, p.x, p.y, p.z, lig.type[i], c + 6);
        float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
        unsigned np = 0;
        if (d.x)
            a = nl_walk_quad<0>(nl, par, tab, rec, nullptr, NoReaction{}, p.x, p.y, p.z, lig.type[i],
                                x.w, d, lane & 3u, np);
        if (c[6] >= 0) {  // inside the lists' box
            pp.x = pp.x + a.x; pp.y = pp.y + a.y; pp.z = pp.z + a.z; pp.w = pp.w + a.w;
        }
        np += __shfl_xor(np, 1);
        np += __shfl_xor(np, 2);
        if ((lane & 3u) != 0) continue;
        for (int k = 0; k < 9; ++k) cell[9 * i + k] = c[k];
        xyz[i] = p.x; xyz[n + i] = p.y; xyz[2 * n + i] = p.z;
        pot[i] = pp.x; pot[n + i] = pp.y; pot[2 * n + i] = pp.z; pot[3 * n + i] = pp.w;
        npairs[i] = np;
    }
}

// One wave; the neighbour-list phase runs on lanes 0..3 over the ligand beads in
// order so that receptor reaction forces accumulate in the CPU's order.
__global__ void k_debug_modes(DProt rec, DProt lig, DGrid rInner, DGrid rOuter, DNL nl,
                              DGrid lInner, DGrid lOuter, DPar par, const float* d, float* xyz,
                              float* pot, int* cell, unsigned* npairs, float* rpot, float* rxyz) {
    extern __shared__ __align__(16) att_pair_params s_tab[];
    const PairTab tab = stage_table(par, s_tab);
    const unsigned lane = threadIdx.x;
    float ampR[ATT_MODES_MAX], ampL[ATT_MODES_MAX];
    for (unsigned m = 0; m < ATT_MODES_MAX; ++m) {
        ampR[m] = m < rec.M ? d[6 + m] : 0.f;
        ampL[m] = m < lig.M ? d[16 + m] : 0.f;
    }
    float t[6];
    pose_trig(d[3], d[4], d[5], lane, t);
    float R[9], RT[9], Rinv[9];
    rotmat_from_trig(t[0], t[1], t[2], t[3], t[4], t[5], R);
    RT[0] = R[0]; RT[1] = R[3]; RT[2] = R[6];
    RT[3] = R[1]; RT[4] = R[4]; RT[5] = R[7];
    RT[6] = R[2]; RT[7] = R[5]; RT[8] = R[8];
    rotmat_from_trig(t[0], t[1], -t[2], -t[3], t[4], -t[5], Rinv);
    const V3 pinv = matvec(RT, -d[0], -d[1], -d[2]);
    const unsigned nr = rec.n, nL = lig.n;
    for (unsigned j = lane; j < nr; j += kWave) {
        const float4 x = rec.pos[j];
        BeadModes<ATT_MODES_MAX> md;
        load_modes(rec, j, md);
        const V3 df = deform(md, rec.M, x.x, x.y, x.z, d + 6);
        V3 p = matvec(Rinv, df.x, df.y, df.z);
        p.x = p.x + pinv.x; p.y = p.y + pinv.y; p.z = p.z + pinv.z;
        rxyz[j] = p.x; rxyz[nr + j] = p.y; rxyz[2 * nr + j] = p.z;
        // the lookup k_modes' phase A makes, so its per-bead values are under test
        const float4 pp = pot_bead_flat(lInner, lOuter, p.x, p.y, p.z, rec.mtype[j], x.w);
        const V3 f = matvec(R, pp.x, pp.y, pp.z);
        rpot[j] = f.x; rpot[nr + j] = f.y; rpot[2 * nr + j] = f.z;
    }
    for (unsigned i = lane; i < nL; i += kWave) {
        const float4 x = lig.pos[i];
        BeadModes<ATT_MODES_MAX> md;
        load_modes(lig, i, md);
        const V3 df = deform(md, lig.M, x.x, x.y, x.z, d + 16);
        V3 p = matvec(R, df.x, df.y, df.z);
        p.x = p.x + d[0]; p.y = p.y + d[1]; p.z = p.z + d[2];
        xyz[i] = p.x; xyz[nL + i] = p.y; xyz[2 * nL + i] = p.z;
        int* c = cell + 9 * i;
        for (int k = 0; k < 9; ++k) c[k] = -1;
        const float4 pp = pot_bead(rInner, rOuter, p.x, p.y, p.z, lig.mtype[i], x.w, c);
        pot[i] = pp.x; pot[nL + i] = pp.y; pot[2 * nL + i] = pp.z; pot[3 * nL + i] = pp.w;
    }
    __syncthreads();
    if (lane >= 4u) return;
    // A pair's lane adds its reaction; a list names a receptor bead once, and the
    // next ligand bead's pairs, on any lane, come after the fence.  Pairs that do
    // not count have none.
    auto reaction = [&](const RecBead<ATT_MODES_MAX>& rb, float fx, float fy, float fz) {
        if (fx == 0.f && fy == 0.f && fz == 0.f) return;
        const unsigned j = rb.index;
        rpot[j] += fx; rpot[nr + j] += fy; rpot[2 * nr + j] += fz;
    };
    for (unsigned i = 0; i < nL; ++i) {
        float4 x;
        unsigned lt;
        const V3 p = place_from_row<ATT_MODES_MAX>(lig, i, ampL, R, d[0], d[1], d[2], x, lt);
        int c[3] = {-1, -1, -1};
        const uint2 list = nl_cell(nl, p.x, p.y, p.z, lt, c);
        float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
        unsigned np = 0;
        if (list.x)
            a = nl_walk_quad<ATT_MODES_MAX>(nl, par, tab, rec, ampR, reaction, p.x, p.y, p.z, lt, x.w,
                                            list, lane, np);
        __threadfence_block();
        np += __shfl_xor(np, 1);
        np += __shfl_xor(np, 2);
        if (lane != 0) continue;
        for (int k = 0; k < 3; ++k) cell[9 * i + 6 + k] = c[k];
        if (c[0] >= 0) {  // inside the lists' box
            pot[i] += a.x; pot[nL + i] += a.y; pot[2 * nL + i] += a.z; pot[3 * nL + i] += a.w;
        }
        npairs[i] = np;
    }
}

__global__ void k_debug_rotmats(const float* ang, unsigned n, float* R) {
    const unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    // Per-lane evaluation (not the wave-cooperative path) of the same formula.
    float s0, c0, s1, c1, s2, c2;
    sincosf_libm(ang[3 * i + 1], &s0, &c0);  // ssi
    sincosf_libm(ang[3 * i + 0], &s1, &c1);  // phi
    sincosf_libm(ang[3 * i + 2], &s2, &c2);  // rot
    rotmat_from_trig(c0, c1, s0, s1, c2, s2, R + 9 * i);
}

__global__ void k_debug_sincosf(const float* x, unsigned n, float* sn, float* cs) {
    const unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) sincosf_libm(x[i], sn + i, cs + i);
}

__global__ void k_debug_plateau_ratio(float P2, double c, unsigned n, float* ratio) {
    const unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) ratio[i] = plateau_ratio_fast(i, P2, c);
}

// Expands a [grid][z][y][x] float4 grid into voxel octets and, with octE, their
// energy channel (see DGrid).
__global__ __launch_bounds__(256) void k_octets(const float4* __restrict__ g,
                                                float4* __restrict__ oct,
                                                float4* __restrict__ octE, unsigned nx,
                                                unsigned ny, unsigned nz, unsigned ngrids) {
    const size_t nvo = (size_t)(nx - 1) * (ny - 1) * (nz - 1);
    const size_t total = nvo * ngrids;
    for (size_t o = blockIdx.x * (size_t)blockDim.x + threadIdx.x; o < total;
         o += (size_t)gridDim.x * blockDim.x) {
        size_t r = o;
        const unsigned ix = r % (nx - 1); r /= (nx - 1);
        const unsigned iy = r % (ny - 1); r /= (ny - 1);
        const unsigned iz = r % (nz - 1); r /= (nz - 1);
        const size_t t = r;
        const size_t nxy = (size_t)nx * ny;
        const float4* b = g + t * nxy * nz + nxy * iz + (size_t)nx * iy + ix;
        float4* d = oct + 8 * o;
        d[0] = b[0];
        d[1] = b[1];
        d[2] = b[nx];
        d[3] = b[nxy];
        d[4] = b[nxy + 1];
        d[5] = b[nxy + nx];
        d[6] = b[nx + 1];
        d[7] = b[nxy + nx + 1];
        if (octE) {
            octE[2 * o] = make_float4(b[0].w, b[1].w, b[nx].w, b[nxy].w);
            octE[2 * o + 1] = make_float4(b[nxy + 1].w, b[nxy + nx].w, b[nx + 1].w, b[nxy + nx + 1].w);
        }
    }
}

__global__ __launch_bounds__(256) void k_copy(float4* __restrict__ dst,
                                              const float4* __restrict__ src, size_t n) {
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
         i += (size_t)gridDim.x * blockDim.x)
        dst[i] = src[i];
}

// ------------------------------------------------------------------ launchers

hipError_t launch_octets(const float4* grid, float4* oct, float4* octE, unsigned nx, unsigned ny,
                         unsigned nz, unsigned ngrids, hipStream_t s) {
    const size_t total = (size_t)(nx - 1) * (ny - 1) * (nz - 1) * ngrids;
    const size_t blocks = std::min<size_t>((total + 255) / 256, 256 * 256);
    hipLaunchKernelGGL(k_octets, dim3((unsigned)blocks), dim3(256), 0, s, grid, oct, octE, nx, ny,
                       nz, ngrids);
    return hipGetLastError();
}

hipError_t launch_copy(void* dst, const void* src, size_t n16, hipStream_t s) {
    if (n16 == 0) return hipSuccess;
    const size_t blocks = std::min<size_t>((n16 + 255) / 256, 256 * 64);
    hipLaunchKernelGGL(k_copy, dim3((unsigned)blocks), dim3(256), 0, s,
                       static_cast<float4*>(dst), static_cast<const float4*>(src), n16);
    return hipGetLastError();
}

// Calls launch(order, dofs, res, counts, m) for consecutive slices of a call's n
// poses.  A launch has fewer than 2^32 threads, and a larger one runs short
// without an error: calls of more poses (2^23 of four waves each) are several
// launches.
template <class Launch>
static void pose_slices(unsigned n, unsigned threadsPerPose, const unsigned* order, const float* dofs,
                        unsigned dofStride, float* res, unsigned resStride, uint2* counts, Launch launch) {
    const unsigned most = (1u << 31) / threadsPerPose;
    for (unsigned first = 0, m; first < n; first += m) {
        m = std::min(most, n - first);
        if (order)  // indices into the whole call's arrays
            launch(order + first, dofs, res, counts, m);
        else
            launch(order, dofs + (size_t)dofStride * first, res + (size_t)resStride * first,
                   counts ? counts + first : nullptr, m);
    }
}

hipError_t launch_rigid(const DProt& rec, const DProt& lig, const DGrid& inner, const DGrid& outer,
                        const DNL& nl, const DPar& par, const float* dofs, float* res, unsigned n,
                        const unsigned* order, uint2* counts, unsigned numCU, hipStream_t s) {
    if (n == 0) return hipSuccess;
    const unsigned slots = par.T <= kMaxTypesLDS ? par.T * par.T : 0;
    const unsigned tab = (unsigned)((sizeof(att_pair_params) * (size_t)slots + 15) & ~(size_t)15);
#define ATT_LAUNCH_RIGID(WP, POSES)                                                              \
    pose_slices(n, kWave * WP, order, dofs, 6, res, 7, counts,                                    \
                [&](const unsigned* o, const float* d, float* r, uint2* c, unsigned m) {          \
        hipLaunchKernelGGL(k_rigid<WP>, dim3((m + POSES - 1) / POSES), dim3(kWave * WP * POSES), \
                           tab + POSES * sizeof(RigidLDS<WP>), s, rec, lig, inner, outer, nl,    \
                           par, d, r, m, tab, o, c);                                             \
    })
    // Eight waves per pose while the CUs are not full (512 poses 1000/300: 40
    // us, 49 on four, 122 on one; 1024: 81, 62, 128), four while they are hardly
    // (2048: 110 on four, 142 on one; 4096: 208, 212, but 94 -> 120 for 300/80), and for
    // ligands that are more than one super-chunk of one wave (8192 poses 3000/800:
    // 955 -> 846).
    if (n <= 2 * numCU) ATT_LAUNCH_RIGID(8, 1);
    else if (n <= 8 * numCU || lig.n > RigidLDS<1>::kSuper) ATT_LAUNCH_RIGID(4, 1);
    else ATT_LAUNCH_RIGID(1, 4);
#undef ATT_LAUNCH_RIGID
    return hipGetLastError();
}

// Dynamic LDS of k_modes: the pair table (the super-chunk arrays are static).
size_t modes_lds_bytes(const DProt& rec, const DProt& lig, const DPar& par, unsigned* tabSlots) {
    (void)rec;
    (void)lig;
    const unsigned slots = par.T <= kMaxTypesLDS ? par.T * par.T : 0;
    if (tabSlots) *tabSlots = slots;
    return sizeof(att_pair_params) * (size_t)slots;
}

hipError_t launch_modes(const DProt& rec, const DProt& lig, const DGrid& rInner,
                        const DGrid& rOuter, const DNL& nl, const DGrid& lInner,
                        const DGrid& lOuter, const DPar& par, const float* dofs, float* res,
                        unsigned n, const unsigned* order, int waves, uint2* counts, hipStream_t s) {
    if (n == 0) return hipSuccess;
    const size_t lds = modes_lds_bytes(rec, lig, par, nullptr);
    const unsigned mm = rec.M > lig.M ? rec.M : lig.M;
#define ATT_LAUNCH_MODES(MMV, WV)                                                                 \
    pose_slices(n, kWave * WV, order, dofs, 26, res, 27, counts,                                  \
                [&](const unsigned* o, const float* d, float* r, uint2* c, unsigned m) {          \
        hipLaunchKernelGGL((k_modes<MMV, WV>), dim3(m), dim3(kWave * WV), lds, s, rec, lig,       \
                           rInner, rOuter, nl, lInner, lOuter, par, d, r, m, o, c);               \
    })
#define ATT_LAUNCH_MODES_W(MMV)                                                                  \
    switch (waves) {                                                                              \
    case 8: ATT_LAUNCH_MODES(MMV, 8); break;                                                      \
    case 4: ATT_LAUNCH_MODES(MMV, 4); break;                                                      \
    case 2: ATT_LAUNCH_MODES(MMV, 2); break;                                                      \
    default: ATT_LAUNCH_MODES(MMV, 1); break;                                                     \
    }
    if (mm == 0) ATT_LAUNCH_MODES_W(0)
    else if (mm <= 5) ATT_LAUNCH_MODES_W(5)
    else ATT_LAUNCH_MODES_W(ATT_MODES_MAX)
#undef ATT_LAUNCH_MODES_W
#undef ATT_LAUNCH_MODES
    return hipGetLastError();
}

hipError_t launch_debug_rigid(const DProt& rec, const DProt& lig, const DGrid& inner,
                              const DGrid& outer, const DNL& nl, const DPar& par,
                              const float* dof, float* xyz, float* pot, int* cell,
                              unsigned* npairs, hipStream_t s) {
    hipLaunchKernelGGL(k_debug_rigid, dim3(1), dim3(kWave), modes_lds_bytes(rec, lig, par, nullptr), s,
                       rec, lig, inner, outer, nl, par, dof, xyz, pot, cell, npairs);
    return hipGetLastError();
}

hipError_t launch_debug_modes(const DProt& rec, const DProt& lig, const DGrid& rInner,
                              const DGrid& rOuter, const DNL& nl, const DGrid& lInner,
                              const DGrid& lOuter, const DPar& par, const float* dof, float* xyz,
                              float* pot, int* cell, unsigned* npairs, float* rpot, float* rxyz,
                              hipStream_t s) {
    hipLaunchKernelGGL(k_debug_modes, dim3(1), dim3(kWave), modes_lds_bytes(rec, lig, par, nullptr), s,
                       rec, lig, rInner, rOuter, nl, lInner, lOuter, par, dof, xyz, pot, cell, npairs,
                       rpot, rxyz);
    return hipGetLastError();
}

hipError_t launch_debug_sincosf(const float* x, unsigned n, float* sn, float* cs, hipStream_t s) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_debug_sincosf, dim3((n + 255) / 256), dim3(256), 0, s, x, n, sn, cs);
    return hipGetLastError();
}

hipError_t launch_debug_plateau_ratio(float P2, unsigned n, float* ratio, hipStream_t s) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_debug_plateau_ratio, dim3((n + 255) / 256), dim3(256), 0, s, P2,
                       1.0 / (10000.0 * (double)P2), n, ratio);
    return hipGetLastError();
}

hipError_t launch_debug_rotmats(const float* ang, unsigned n, float* R, hipStream_t s) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_debug_rotmats, dim3((n + 255) / 256), dim3(256), 0, s, ang, n, R);
    return hipGetLastError();
}

}  // namespace att
