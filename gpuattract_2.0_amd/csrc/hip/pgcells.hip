// Cell pass of the parameter gradient (grid part).
//
// The grid energy of a bead of type t at p is sum_a ipon(a,t) (rc(a,t) S_a(p)
// - ac(a,t) S6_a(p)) with S_a, S6_a the trilinear interpolants of the basis
// grids, so dE/drc(a,t) summed over every bead of type t of every pose is
// ipon(a,t) sum_cells sum_corners D_t(cell, corner) S_a(corner) / vol, where
// D_t(cell, corner) sums w_pose * (corner weight) over the beads of type t in
// that cell.  k_adjoint writes one record per bead (key = cell and type, packed
// by PgKeys; {x, y, z, w}, or {x, y, z} when the call has no pose weights).
//
// Bucket pass (calls of many records, pg_keys): the records are sorted by bucket of
// cells only (stable radix sort: 16 key bits, two passes over the records
// instead of three over 24); one wave adds a bucket's corner weights into
// D[corner][type][cell] in LDS, then multiplies D of every touched cell,
// [types x corners], with the cell's basis, [corners x 2 T channels], on the
// matrix cores in FP32, accumulating over all of its cells.
//
// Run pass (few records, few types, or more types than D and the products fit):
// the records are sorted by the whole key, the corner weights of each run of
// equal keys within a group of 64 sorted records summed by a segmented scan
// across the wave, the run sums compacted (integer scan of the per-group run
// counts), and each run sum contracted with its cell's basis octets.
//
// Either way the basis grids are read about once per distinct cell instead of
// once per bead, and every step has a fixed order: calls repeat their bits.
#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>
#include <algorithm>
#include <type_traits>

#include "device.h"
#include "internal.h"

namespace att {

namespace {

// Summed corner weights of one (cell, type), corners in octet order
// 000 100 010 001 101 011 110 111.
struct CellW {
    float c[8];
};

// The geometry of one grid, as the adjoint's lookup uses it.
struct CellGeom {
    unsigned nx, ny;
    float lox, loy, loz, dVox;
};

__host__ __device__ inline CellGeom cell_geom(const DGrid& g) {
    return CellGeom{g.nx, g.ny, g.lox, g.loy, g.loz, g.dVox};
}

// A record's position and pose weight (1 for records without weights).
__device__ inline float4 record_pos(const float4* pos, size_t i) { return pos[i]; }
__device__ inline float4 record_pos(const float3* pos, size_t i) {
    const float3 p = pos[i];
    return make_float4(p.x, p.y, p.z, 1.f);
}

// Corner weights of a record {x, y, z, w} in cell `cell` (inner cells
// first), times its pose weight: the weights of grid_adj_one's trilinear
// interpolation (same cell, same differences).
__device__ inline CellW record_weights(const CellGeom& in, const CellGeom& out, unsigned cellsIn,
                                       unsigned cell, float4 p) {
    const bool inner = cell < cellsIn;
    const CellGeom& g = inner ? in : out;
    unsigned o = inner ? cell : cell - cellsIn;
    const unsigned ix = o % (g.nx - 1);
    o /= (g.nx - 1);
    const unsigned iy = o % (g.ny - 1), iz = o / (g.ny - 1);
    const float mnx = (float)(int)ix * g.dVox + g.lox;
    const float mny = (float)(int)iy * g.dVox + g.loy;
    const float mnz = (float)(int)iz * g.dVox + g.loz;
    const float ax = p.x - mnx, ay = p.y - mny, az = p.z - mnz;
    const float bx = (mnx + g.dVox) - p.x, by = (mny + g.dVox) - p.y, bz = (mnz + g.dVox) - p.z;
    CellW r;
    r.c[0] = bx * by * bz * p.w;
    r.c[1] = ax * by * bz * p.w;
    r.c[2] = bx * ay * bz * p.w;
    r.c[3] = bx * by * az * p.w;
    r.c[4] = ax * by * az * p.w;
    r.c[5] = bx * ay * az * p.w;
    r.c[6] = ax * ay * bz * p.w;
    r.c[7] = ax * ay * az * p.w;
    return r;
}

size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

__host__ __device__ inline size_t groups_of(size_t records) { return (records + 63) / 64; }

// The key bits the records are sorted by.
struct SortBits {
    unsigned begin, end;
};
SortBits sort_bits(const PgKeys& keys) {
    unsigned end = 0;
    while (end < 32 && (keys.invalid >> end) != 0) ++end;
    return SortBits{keys.cellBits ? keys.lowBits : 0u, end};
}

size_t temp_bytes(size_t records, const PgKeys& keys, bool weights) {
    const SortBits b = sort_bits(keys);
    size_t sortB = 0, scanB = 0;
    if (weights)
        (void)rocprim::radix_sort_pairs(nullptr, sortB, (unsigned*)nullptr, (unsigned*)nullptr,
                                        (float4*)nullptr, (float4*)nullptr, (unsigned)records, b.begin,
                                        b.end);
    else
        (void)rocprim::radix_sort_pairs(nullptr, sortB, (unsigned*)nullptr, (unsigned*)nullptr,
                                        (float3*)nullptr, (float3*)nullptr, (unsigned)records, b.begin,
                                        b.end);
    if (!keys.cellBits)
        (void)rocprim::exclusive_scan(nullptr, scanB, (const unsigned*)nullptr, (unsigned*)nullptr, 0u,
                                      groups_of(records), rocprim::plus<unsigned>());
    return align256(sortB > scanB ? sortB : scanB);
}

// LDS of one bucket: its sums, D[type][cell][corner], the cells of one type
// padded by one so that the types lie in different banks, and a flag per cell.
size_t bucket_lds(unsigned T, unsigned cellBits) {
    return sizeof(float) * 8 * T * ((1u << cellBits) + 1u) + sizeof(unsigned) * 64;
}

typedef float F4 __attribute__((ext_vector_type(4)));

// Sum over the 64 lanes of a wave, on lane 63 (DPP row shifts of 1, 2, 4 and 8
// lanes, then the row totals broadcast: a tree of six levels).
__device__ __forceinline__ float wave_total(float v) {
    auto from = [](float x, auto step) __attribute__((always_inline)) {
        constexpr int kStep = decltype(step)::value;
        constexpr int kRows = kStep == 0x142 ? 0xa : kStep == 0x143 ? 0xc : 0xf;
        return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), kStep, kRows, 0xf, false));
    };
    v += from(v, std::integral_constant<int, 0x111>{});
    v += from(v, std::integral_constant<int, 0x112>{});
    v += from(v, std::integral_constant<int, 0x114>{});
    v += from(v, std::integral_constant<int, 0x118>{});
    v += from(v, std::integral_constant<int, 0x142>{});
    v += from(v, std::integral_constant<int, 0x143>{});
    return v;
}

// From this many lanes of one cell and type on, their sum is formed first (k_pg_buckets).
constexpr int kCrowd = 16;

}  // namespace

// Runs of equal keys among the sorted records, per group of 64 (one wave,
// lane = record): a segmented inclusive scan of the corner weights across the
// lanes (sorted keys: lanes l - d and l hold the same key only if every lane
// between does), so the last lane of each run holds the run's sum.  COUNT
// writes each group's number of runs (keys below `invalid`); otherwise the
// runs go to cellKey/cellW from the group's offset, in lane order.
template <bool COUNT, class Pos>
__global__ __launch_bounds__(256) void k_pg_runs(const unsigned* __restrict__ key,
                                                 const Pos* __restrict__ pos, size_t records,
                                                 CellGeom in, CellGeom out, PgKeys keys,
                                                 unsigned* __restrict__ groupRuns,
                                                 const unsigned* __restrict__ groupOffset,
                                                 unsigned* __restrict__ cellKey,
                                                 CellW* __restrict__ cellW) {
    const unsigned lane = threadIdx.x & 63u;
    const size_t g = ((size_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    if (g >= groups_of(records)) return;  // uniform per wave
    const size_t i = g * 64 + lane;
    const unsigned k = i < records ? key[i] : 0xFFFFFFFFu;
    const bool live = k < keys.invalid;
    CellW d{};
    if (!COUNT && live) d = record_weights(in, out, keys.cellsIn, k >> keys.lowBits, record_pos(pos, i));
#pragma unroll
    for (unsigned off = 1; off < 64; off <<= 1) {
        const unsigned ko = __shfl_up(k, off);
        const bool add = lane >= off && ko == k;
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const float v = __shfl_up(d.c[c], off);
            if (!COUNT && add) d.c[c] = d.c[c] + v;
        }
    }
    const unsigned kn = __shfl_down(k, 1);
    const bool tail = live && (lane == 63 || kn != k);
    const unsigned long long b = __ballot(tail);
    if (COUNT) {
        if (lane == 0) groupRuns[g] = (unsigned)__popcll(b);
        return;
    }
    if (tail) {
        const unsigned r = groupOffset[g] + (unsigned)__popcll(b & ((1ull << lane) - 1ull));
        cellKey[r] = k;
        cellW[r] = d;
    }
}

// One wave per workgroup: workgroup b contracts runs [b*per, ...) (per =
// ceil(runs / blocks)), lane by lane, into its LDS row (lane order within each
// atomic, program order across them), then writes the row.
__global__ __launch_bounds__(64) void k_pgrad_cells(const unsigned* __restrict__ cellKey,
                                                    const CellW* __restrict__ cellW,
                                                    const unsigned* __restrict__ groupRuns,
                                                    const unsigned* __restrict__ groupOffset,
                                                    unsigned groups,
                                                    DGrid inner, DGrid outer, DBasis bin,
                                                    DBasis bout, const att_pair_params* __restrict__ tab,
                                                    unsigned T, PgKeys keys,
                                                    float* __restrict__ rows) {
    extern __shared__ float s_row[];
    const unsigned npg = 3 * T * T, lane = threadIdx.x;
    for (unsigned k = lane; k < npg; k += 64) s_row[k] = 0.f;
    __syncthreads();
    const unsigned n = groupOffset[groups - 1] + groupRuns[groups - 1];
    const unsigned per = (n + gridDim.x - 1) / gridDim.x;
    const unsigned lo = min(n, blockIdx.x * per), hi = min(n, lo + per);
    for (unsigned i = lo + lane; i < hi; i += 64) {
        const unsigned key = cellKey[i];
        if (key >= keys.invalid) continue;
        const unsigned t = key & ((1u << keys.lowBits) - 1u), cell = key >> keys.lowBits;
        const bool in = cell < keys.cellsIn;
        const unsigned o = in ? cell : cell - keys.cellsIn;
        const float4* __restrict__ row = (in ? bin.oct : bout.oct) + (size_t)o * (in ? bin.nb : bout.nb) * 2;
        const float vol_inv = in ? inner.vol_inv : outer.vol_inv;
        const CellW W = cellW[i];
        for (unsigned a = 0; a < T; ++a) {
            const float4 s0 = row[4 * a], s1 = row[4 * a + 1];  // S_a at the 8 corners
            const float4 u0 = row[4 * a + 2], u1 = row[4 * a + 3];  // S6_a
            const float S = (s0.x * W.c[0] + s0.y * W.c[1] + s0.z * W.c[2] + s0.w * W.c[3] +
                             s1.x * W.c[4] + s1.y * W.c[5] + s1.z * W.c[6] + s1.w * W.c[7]) * vol_inv;
            const float S6 = (u0.x * W.c[0] + u0.y * W.c[1] + u0.z * W.c[2] + u0.w * W.c[3] +
                              u1.x * W.c[4] + u1.y * W.c[5] + u1.z * W.c[6] + u1.w * W.c[7]) * vol_inv;
            const unsigned k = a * T + t;
            const float iv = (float)tab[k].ipon;
            atomicAdd(&s_row[3 * k], iv * S);
            atomicAdd(&s_row[3 * k + 1], -iv * S6);
        }
    }
    __syncthreads();
    for (unsigned k = lane; k < npg; k += 64) rows[(size_t)blockIdx.x * npg + k] = s_row[k];
}

// Bucket pass.  One wave per workgroup: workgroup b takes the records [b *
// per, (b + 1) * per) in order, 64 at a time, the next 64 in flight.  A bucket
// that ends inside them is contracted there: its part of the sums is complete.
// Matrix tiles of 16 types x 16 channels, MT x NT of them; the sum over the
// corners is the products' inner dimension, four at a time (lane group g = lane
// / 16 holds corners 2 g and 2 g + 1, one per product), and the accumulators run
// over every cell of the workgroup.  Bound by the instructions of the turns (a
// step's lanes of one cell and type add one after the other, four 16-byte LDS
// operations each) and their latency: 80 million records of 12 types 1.46 ms
// with 16 workgroups per CU, 1.71 with 12, 1.78 with 8; LDS float atomics in
// their place 3.7 (a wave's takes about 400 cycles).  16 also where the LDS holds
// fewer at a time (12 of 12 types, 7 of 20: smaller shares even the work out):
// calls of 20,000 poses 3000/800 3.29 ms, 3.37 with 12 per CU; 20 types 4.76, 5.06
// with 7.  The contraction, 2 MT NT products and one read of 64 T bytes of basis per
// cell, kFlight cells in flight, is 0.2 of it.  Scans and contraction of the run
// pass: 2.8 ms on the same records, and its third sort pass 0.7.
template <unsigned MT, class Pos>
__global__ __launch_bounds__(64) void k_pg_buckets(const unsigned* __restrict__ key,
                                                   const Pos* __restrict__ pos, size_t records,
                                                   CellGeom in, CellGeom out, float volIn, float volOut,
                                                   DBasis bin, DBasis bout,
                                                   const att_pair_params* __restrict__ tab, unsigned T,
                                                   PgKeys keys, float* __restrict__ rows) {
    constexpr unsigned NT = 2 * MT;
    constexpr unsigned kFlight = MT == 1 ? 4 : 2;
    extern __shared__ __align__(16) float s_d[];
    const unsigned lane = threadIdx.x, tm = lane & 15u, g = lane >> 4;
    const unsigned perType = 8 * ((1u << keys.cellBits) + 1u);
    unsigned* s_touched = reinterpret_cast<unsigned*>(s_d + T * perType);  // 64 cells at most
    for (unsigned k = lane; k < T * perType + 64; k += 64) s_d[k] = 0.f;
    wave_sync();
    F4 acc[MT][NT];
#pragma unroll
    for (unsigned m = 0; m < MT; ++m)
#pragma unroll
        for (unsigned c = 0; c < NT; ++c) acc[m][c] = F4{0.f, 0.f, 0.f, 0.f};
    float* out_row = rows + (size_t)blockIdx.x * 3 * T * T;
    for (unsigned e = lane; e < 3 * T * T; e += 64) out_row[e] = 0.f;
    __threadfence_block();
    // One cell of the contraction below with the types that are there only,
    // straight into the parameter row.
    auto by_type = [&](unsigned bucket, unsigned local) {
        const unsigned cell = (bucket << keys.cellBits) + local;
        const bool inner = cell < keys.cellsIn;
        const float* basis = reinterpret_cast<const float*>(inner ? bin.oct : bout.oct) +
                             (size_t)(inner ? cell : cell - keys.cellsIn) * 16 * T;
#pragma unroll 1
        for (unsigned e = lane; e < 2 * T * T; e += 64) {
            const unsigned t = e / (2 * T), ch = e % (2 * T), x = (ch >> 1) * T + t;
            const float* d = s_d + t * perType + 8 * local;
            bool any = false;
            float v = 0.f;
#pragma unroll 1
            for (unsigned c = 0; c < 8; ++c) {
                any |= d[c] != 0.f;
                v += d[c] * basis[8 * ch + c];
            }
            v *= inner ? volIn : volOut;
            const float iv = (float)tab[x].ipon;
            if (any) out_row[3 * x + (ch & 1u)] += ch & 1u ? -iv * v : iv * v;
        }
        wave_sync();
#pragma unroll 1
        for (unsigned k = lane; k < 8 * T; k += 64) s_d[(k >> 3) * perType + 8 * local + (k & 7u)] = 0.f;
        wave_sync();
    };
    // Contracts and clears the bucket's touched cells.
    auto contract = [&](unsigned bucket) __attribute__((always_inline)) {
        wave_sync();
        unsigned long long todo = __ballot(s_touched[lane] != 0u);
        s_touched[lane] = 0u;
        while (todo) {
            const unsigned long long before = todo;
            unsigned local[kFlight];
            float2 b[kFlight][NT];
            float vol[kFlight];
            unsigned cnt = 0;
            float finite = 0.f;  // NaN where a basis value is not finite
#pragma unroll
            for (unsigned f = 0; f < kFlight; ++f) {
                local[f] = 0;
                vol[f] = 0.f;
                if (todo) {  // uniform
                    local[f] = (unsigned)__builtin_ctzll(todo);
                    todo &= todo - 1;
                    ++cnt;
                }
                const unsigned cell = (bucket << keys.cellBits) + local[f];
                const bool inner = cell < keys.cellsIn;
                vol[f] = inner ? volIn : volOut;
                const float2* row = reinterpret_cast<const float2*>(inner ? bin.oct : bout.oct) +
                                    (size_t)(inner ? cell : cell - keys.cellsIn) * 8 * T;
#pragma unroll
                for (unsigned c = 0; c < NT; ++c) {
                    const unsigned ch = 16 * c + tm;
                    b[f][c] = f < cnt && ch < 2 * T ? row[4 * ch + g] : make_float2(0.f, 0.f);
                }
            }
#pragma unroll
            for (unsigned f = 0; f < kFlight; ++f)
#pragma unroll
                for (unsigned c = 0; c < NT; ++c) finite += 0.f * b[f][c].x + 0.f * b[f][c].y;
            if (__ballot(!(finite == 0.f))) {
                // Zero times such a value is no zero: only the types that are there take part.
                for (unsigned long long now = before ^ todo; now; now &= now - 1)
                    by_type(bucket, (unsigned)__builtin_ctzll(now));
                continue;
            }
#pragma unroll
            for (unsigned f = 0; f < kFlight; ++f) {
                if (f >= cnt) break;  // uniform
#pragma unroll
                for (unsigned m = 0; m < MT; ++m) {
                    const unsigned t = 16 * m + tm;
                    float a0 = 0.f, a1 = 0.f;
                    if (t < T) {
                        float2* d = reinterpret_cast<float2*>(s_d + t * perType + 8 * local[f] + 2 * g);
                        const float2 v = *d;
                        a0 = v.x * vol[f];
                        a1 = v.y * vol[f];
                        *d = make_float2(0.f, 0.f);
                    }
#pragma unroll
                    for (unsigned c = 0; c < NT; ++c) {
                        acc[m][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(a0, b[f][c].x, acc[m][c], 0, 0, 0);
                        acc[m][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(a1, b[f][c].y, acc[m][c], 0, 0, 0);
                    }
                }
            }
        }
        wave_sync();
    };
    const size_t per = ((records + gridDim.x - 1) / gridDim.x + 63) & ~(size_t)63;
    const size_t lo = min(records, blockIdx.x * per), hi = min(records, lo + per);
    constexpr unsigned kNone = 0xFFFFFFFFu;
    unsigned cur = kNone;
    unsigned k = lo + lane < hi ? key[lo + lane] : kNone;
    float4 p = lo + lane < hi ? record_pos(pos, lo + lane) : make_float4(0.f, 0.f, 0.f, 0.f);
    for (size_t i = lo; i < hi; i += 64) {
        const unsigned kc = k;
        const float4 pc = p;
        const size_t nx = i + 64 + lane;
        k = nx < hi ? key[nx] : kNone;
        if (nx < hi) p = record_pos(pos, nx);
        unsigned long long todo = __ballot(kc < keys.invalid);
        while (todo) {
            const unsigned first = (unsigned)__builtin_ctzll(todo);
            const unsigned bucket = (unsigned)__builtin_amdgcn_readlane((int)(kc >> keys.lowBits), (int)first);
            if (bucket != cur) {
                if (cur != kNone) contract(cur);
                cur = bucket;
            }
            const bool mine = kc < keys.invalid && kc >> keys.lowBits == bucket;
            const unsigned low = kc & ((1u << keys.lowBits) - 1u);
            const unsigned local = low & ((1u << keys.cellBits) - 1u), t = low >> keys.cellBits;
            // Lanes of one cell and type add in turn, in lane order.
            unsigned long long same = __ballot(mine);
            for (unsigned q = 0; q < keys.lowBits; ++q) {
                const unsigned long long ones = __ballot(low >> q & 1u);
                same &= low >> q & 1u ? ones : ~ones;
            }
            unsigned turn = mine ? (unsigned)__popcll(same & ((1ull << lane) - 1ull)) : 64u;
            const CellW w = record_weights(in, out, keys.cellsIn, mine ? (bucket << keys.cellBits) + local : 0u, pc);
            const unsigned at = mine ? t * perType + 8 * local : 0u;
            // A crowd of one cell and type is summed by a tree and added at once:
            // poses that lie together fill whole steps with few cells, and a turn
            // for every lane took 64 of them (30,000 equal poses of 300 beads 0.68
            // ms, 0.12 so).  A tree costs about as much as ten turns; 8 lanes as the line
            // were as fast, and 2 % slower for 4096 places.  The sum of a cell is
            // also at most a quarter as long a chain.
            unsigned long long crowd = 0;
            if (__ballot(mine && turn + 1u >= (unsigned)kCrowd)) crowd = __ballot(mine && __popcll(same) >= kCrowd);
            while (crowd) {  // uniform
                const int lead = __builtin_ctzll(crowd);
                const unsigned long long members =
                    (unsigned long long)(unsigned)__builtin_amdgcn_readlane((int)(same >> 32), lead) << 32 |
                    (unsigned)__builtin_amdgcn_readlane((int)same, lead);
                const bool member = members >> lane & 1u;
                float v[8];
#pragma unroll
                for (unsigned c = 0; c < 8; ++c) v[c] = wave_total(member ? w.c[c] : 0.f);
                const unsigned to = (unsigned)__builtin_amdgcn_readlane((int)at, lead);
                const unsigned cell = (unsigned)__builtin_amdgcn_readlane((int)local, lead);
                if (lane == 63) {
                    F4* d = reinterpret_cast<F4*>(s_d + to);
                    d[0] += F4{v[0], v[1], v[2], v[3]};
                    d[1] += F4{v[4], v[5], v[6], v[7]};
                    s_touched[cell] = 1u;
                }
                wave_sync();
                if (member) turn = 64u;
                crowd &= ~members;
            }
            F4* d = reinterpret_cast<F4*>(s_d + at);
            for (unsigned r = 0; __ballot(turn == r); ++r) {
                if (turn == r) {
                    const F4 lo4 = d[0] + F4{w.c[0], w.c[1], w.c[2], w.c[3]};
                    const F4 hi4 = d[1] + F4{w.c[4], w.c[5], w.c[6], w.c[7]};
                    d[0] = lo4;
                    d[1] = hi4;
                }
                wave_sync();
            }
            if (turn == 0u) s_touched[local] = 1u;
            todo &= ~__ballot(mine);
        }
    }
    if (cur != kNone) contract(cur);
    // acc[m][c][i] on lane l: type 16 m + 4 (l / 16) + i, channel 16 c + l % 16 (S_a, S6_a in turn)
    __threadfence_block();
#pragma unroll
    for (unsigned m = 0; m < MT; ++m)
#pragma unroll
        for (unsigned c = 0; c < NT; ++c)
#pragma unroll
            for (unsigned i = 0; i < 4; ++i) {
                const unsigned t = 16 * m + 4 * g + i, ch = 16 * c + tm;
                if (t < T && ch < 2 * T) {
                    const unsigned e = (ch >> 1) * T + t;
                    const float iv = (float)tab[e].ipon;
                    out_row[3 * e + (ch & 1u)] += ch & 1u ? -iv * acc[m][c][i] : iv * acc[m][c][i];
                }
            }
}

// The bucket pass works per cell (all types of a touched cell at once, and one
// wave reads its basis), the run pass per cell and type that is there.  Bucket
// pass from two records per cell and six types on, from 1.1 where the types fill
// a matrix tile (10 to 16).  us of a call on the bucket and on the run pass:
// 2.1-2.3 records per cell 455, 446 (8 types, 1000/300) and 1023, 1011 (3000/800),
// 1172, 1328 (32, 1500/1000); 1.1-1.2 679, 712 (12) and 863, 912 (16, 3000/800) but
// 1719, 1494 (32); 1.0 478, 434 (12, 1000/300); 0.3 381, 281 (20); 16 and 12
// records per cell 1560, 1615 and 3214, 3356 (6 types) but 1564, 1540 and 3142,
// 3120 (4).  Up to 32 types for the LDS of D.
bool pg_keys(size_t cellsIn, size_t cellsOut, unsigned T, size_t records, PgKeys* keys) {
    const size_t cells = cellsIn + cellsOut;
    unsigned typeBits = 0;
    while ((1u << typeBits) < T) ++typeBits;
    // Buckets of the fewest cells, 16 or more, for which 16 key bits number them
    // (a third pass of the sort costs a third of its time); 64 at most, for the LDS.
    unsigned cellBits = 0;
    if (T >= 6 && T <= 32 && records >= (T >= 10 && T <= 16 ? cells + cells / 10 : 2 * cells)) {
        cellBits = 4;
        while (cellBits < (T <= 16 ? 6u : 5u) && (cells >> cellBits) + 1 >= 65536) ++cellBits;
    }
    const size_t buckets = (cells + ((size_t)1 << cellBits) - 1) >> cellBits;
    const size_t invalid = buckets << (cellBits + typeBits);
    if (invalid >= 0xFFFFFFFFull) return false;
    *keys = PgKeys{(unsigned)cellsIn, cellBits, cellBits + typeBits, (unsigned)invalid};
    return true;
}

unsigned pg_cells_blocks(size_t records, const PgKeys& keys, unsigned numCU) {
    return keys.cellBits ? (unsigned)std::min<size_t>(16 * numCU, groups_of(records)) : 2048;
}

size_t pg_cells_bytes(size_t records, const PgKeys& keys, bool weights) {
    const size_t R = records, G = groups_of(records), pb = weights ? 16 : 12;
    const size_t runs = keys.cellBits ? 0 : align256(4 * R) + align256(sizeof(CellW) * R) + 2 * align256(4 * G);
    return 2 * align256(4 * R) + 2 * align256(pb * R) + runs + temp_bytes(records, keys, weights);
}

PgCellBufs pg_cells_layout(void* scratch, size_t records, const PgKeys& keys, bool weights) {
    const size_t R = records, pb = weights ? 16 : 12;
    char* p = static_cast<char*>(scratch);
    PgCellBufs B{};
    B.weights = weights;
    B.key = reinterpret_cast<unsigned*>(p); p += align256(4 * R);
    B.pos = p; p += align256(pb * R);
    B.keySorted = reinterpret_cast<unsigned*>(p); p += align256(4 * R);
    B.posSorted = p; p += align256(pb * R);
    if (!keys.cellBits) {
        B.cellKey = reinterpret_cast<unsigned*>(p); p += align256(4 * R);
        B.cellW = reinterpret_cast<float*>(p); p += align256(sizeof(CellW) * R);
        B.groupRuns = reinterpret_cast<unsigned*>(p); p += align256(4 * groups_of(R));
        B.groupOffset = reinterpret_cast<unsigned*>(p); p += align256(4 * groups_of(R));
    }
    B.temp = p;
    B.tempBytes = temp_bytes(records, keys, weights);
    return B;
}

namespace {
template <class Pos>
hipError_t pg_cells(const PairDesc& P, const PgCellBufs& B, size_t records, float* rows,
                    unsigned blocks, hipStream_t s) {
    const unsigned T = P.par.T;
    const SortBits bits = sort_bits(P.recKeys);
    size_t tb = B.tempBytes;
    Pos* pos = static_cast<Pos*>(B.pos);
    Pos* posSorted = static_cast<Pos*>(B.posSorted);
    hipError_t e = rocprim::radix_sort_pairs(B.temp, tb, B.key, B.keySorted, pos, posSorted,
                                             (unsigned)records, bits.begin, bits.end, s);
    if (e != hipSuccess) return e;
    const CellGeom in = cell_geom(P.inner), out = cell_geom(P.outer);
    if (P.recKeys.cellBits) {
        const size_t lds = bucket_lds(T, P.recKeys.cellBits);
        auto* kernel = T <= 16 ? k_pg_buckets<1, Pos> : k_pg_buckets<2, Pos>;
        hipLaunchKernelGGL(kernel, dim3(blocks), dim3(64), lds, s, B.keySorted, (const Pos*)posSorted,
                           records, in, out, P.inner.vol_inv, P.outer.vol_inv, P.bin, P.bout, P.par.tab, T,
                           P.recKeys, rows);
        return hipGetLastError();
    }
    const unsigned G = (unsigned)groups_of(records);
    const unsigned wgs = (G + 3) / 4;  // four groups (waves) per workgroup
    hipLaunchKernelGGL((k_pg_runs<true, Pos>), dim3(wgs), dim3(256), 0, s, B.keySorted,
                       (const Pos*)posSorted, records, in, out, P.recKeys, B.groupRuns, nullptr,
                       nullptr, nullptr);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    tb = B.tempBytes;
    e = rocprim::exclusive_scan(B.temp, tb, (const unsigned*)B.groupRuns, B.groupOffset, 0u, G,
                                rocprim::plus<unsigned>(), s);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((k_pg_runs<false, Pos>), dim3(wgs), dim3(256), 0, s, B.keySorted,
                       (const Pos*)posSorted, records, in, out, P.recKeys, B.groupRuns,
                       B.groupOffset, B.cellKey, reinterpret_cast<CellW*>(B.cellW));
    if ((e = hipGetLastError()) != hipSuccess) return e;
    const size_t lds = sizeof(float) * 3 * (size_t)T * T;
    hipLaunchKernelGGL(k_pgrad_cells, dim3(blocks), dim3(64), lds, s, B.cellKey,
                       reinterpret_cast<const CellW*>(B.cellW), B.groupRuns, B.groupOffset, G,
                       P.inner, P.outer, P.bin, P.bout, P.par.tab, T, P.recKeys, rows);
    return hipGetLastError();
}
}  // namespace

hipError_t launch_pg_cells(const PairDesc& P, const PgCellBufs& B, size_t records, float* rows,
                           unsigned blocks, hipStream_t s) {
    return B.weights ? pg_cells<float4>(P, B, records, rows, blocks, s)
                     : pg_cells<float3>(P, B, records, rows, blocks, s);
}

}  // namespace att
