// pairs_tile.h -- pair kernels on the FP64 matrix cores (replace the j-loops of
// PC/cpairs/npairs_3d_engine.pyx:103-182 and its siblings for the common bin
// layouts; the kernels of pairs_kernel.h take every other request).
//
// One wavefront takes a group of 64 lane points consecutive along the Hilbert
// curve, as four sub-groups of 16.  Stream points near the group's box are
// staged in LDS in coordinates relative to the box centre (the periodic shift
// folded in); staged points near a sub-group's own, smaller box are dealt to
// it in tiles of 16, and one v_mfma_f64_16x16x4 forms the 256 squared
// distances |a|^2 + |b|^2 - 2 a.b of a tile (planar ones for (rp, pi) bins).
//
// Exactness.  The matrix product's rounding is far below one unit of the high
// word of the distance (20 mantissa bits) except for very close pairs, so the
// bin follows from the high word alone unless it lies within one unit of an
// edge's or below the group's rounding floor; those pairs are evaluated again
// with the reference's arithmetic, (x1 - shift) - x2 and dx*dx + dy*dy + dz*dz
// in FP64, and binned with its "<=".  Every pair therefore lands in the bin
// the reference puts it in.
//
// What bounds it: instruction issue (1M clustered points, 20 edges to 50 Mpc/h:
// vector instructions 65 % and the matrix product 14 % of the issue slots, 13 of
// 16 waves alive on average).  The MFMA (65 cycles per 256 pairs, next to none of
// which other waves' VALU work fills: with 16 integer additions 112 to 119, 43 to
// 47 alone) replaces 8 FP64 instructions of 4.5 cycles
// per 64 pairs, the bin takes 6 instructions and two LDS accesses instead of 12
// and two, and sub-groups of 16 evaluate 2.4 pairs per pair in range where groups
// of 64 evaluated 4.4 (6.3e8 instead of 1.18e9 evaluations there).  Pair kernels
// against those of pairs_kernel.h: that count 1.04 -> 0.55 ms, 2M (rp, pi) 2.5 ->
// 1.65 ms, per-object rows of 1M 1.49 -> 1.04 ms, the 64-mock forward-mode pass
// 49 -> 35 ms, Jacobian rows of 1M 2.7 -> 1.9 ms.
#pragma once

#include "pairs_kernel.h"

namespace hp {

typedef double dbl4 __attribute__((ext_vector_type(4)));

#ifndef HP_TAN_COLS
#define HP_TAN_COLS 8
#endif
constexpr uint32_t kTanCols = HP_TAN_COLS;
#ifndef HP_TILE_WPS
#define HP_TILE_WPS 4
#endif
constexpr int kSub = 16;                   // lane points of a sub-group, stream points of a tile
// Staged stream points dealt at a time: 128, or 64 where the histogram leaves
// little LDS, so that more waves fit a CU (forward-mode pass of 64 mocks: 9.4 ->
// 12 waves per CU and 45.9 -> 42.6 ms; 1M marked (rp, pi) sums 1782 -> 1720 us;
// the 1M count, whose tiles fill less well with 64, loses 813 -> 860 us).
// Wide (rp, pi) counts (2M points, 656 cells: 12 -> 16 waves) take 64 (var 1), wp's
// few cells 128.
constexpr int deal_of(int mode, int var) {
    return (mode == kModeTan || mode == kModeWXYZ || mode == kModeObj || mode == kModeJac ||
            mode == kModeJack || (mode == kModeXYZ && var == 1))
               ? 64
               : 128;
}
// LDS layout of one wave ahead of its weights and histogram
template <int kDeal>
struct Stage {
static constexpr int kStage = kDeal + 64;         // staged points
static constexpr int kSlots = kStage + 1;         // and one that no pair bins
static constexpr int kIdOff = 4 * kSlots * 8;     // after x, y, z, squared norm: stream index and image of each
static constexpr int kListOff = kIdOff + (kSlots + 3) / 4 * 16;            // slots dealt to a sub-group, three tiles of padding
static constexpr int kMarkOff = kListOff + kDeal + 3 * kSub;    // 64: starts of stretches
static constexpr int kInfoOff = (kMarkOff + 64 + 15) / 16 * 16; // boxes of the sub-groups and the group, the cube window
static constexpr int kTileBytes = kInfoOff + 4 * 32 + 32 + 48;
};
constexpr int kImgShift = 26;              // a staged point's id: row of its mock, image above
constexpr uint32_t kRowMask = (1u << kImgShift) - 1u;
constexpr int kHere = 1 | (1 << 2) | (1 << 4);  // the unshifted image
constexpr double kFar = 1.0e300;           // squared norm of a point that no pair bins

struct TileArgs {
    PairLaunch L;
    TileSpec tr, tp;
    int tp_off;      // LDS byte offset of the pi table, a multiple of its size
    int lw_off;      // byte offset of the lane points' weights in a wave's LDS area
    int hist_off;    // ... of its histogram
    int cnt_off;     // ... of the count rows of a marked pass
    int ccol_sh;     // log2 of the columns of the (rp, pi) count cells
    int wave_bytes;
    int tab_bytes;
    int parts_sh;    // log2 of the work items per lane group (cubes dealt round-robin)
    int tail_sh;     // ... of the groups from `tail` on
    int64_t tail;
    int64_t items;
    int chunk_sh;    // log2 of the consecutive items one XCD takes
    uint32_t taken;  // items of each queue that the launch starts on (its waves' first ones)
    uint32_t* queue; // work queues, one per XCD: items taken beyond those; null: every wave has one item
};

typedef const __attribute__((address_space(4))) TileArgs kernarg_tile_args;  // as the kernel receives them
typedef const __attribute__((address_space(4))) MockGeom const_geom;         // scalar loads

// DPP moves: row rotations (all 16 lanes of a row), prefix steps over the wave
template <int CTRL, int ROWS>
__device__ __forceinline__ int dpp_or_zero(int v) {
    return __builtin_amdgcn_update_dpp(0, v, CTRL, ROWS, 0xf, false);
}
template <int CTRL>
__device__ __forceinline__ float dpp_ror(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xf, 0xf, false));
}
// minimum and maximum over each 16-lane row
__device__ __forceinline__ float row_min(float v) {
    v = fminf(v, dpp_ror<0x128>(v));
    v = fminf(v, dpp_ror<0x124>(v));
    v = fminf(v, dpp_ror<0x122>(v));
    return fminf(v, dpp_ror<0x121>(v));
}
__device__ __forceinline__ float row_max(float v) {
    v = fmaxf(v, dpp_ror<0x128>(v));
    v = fmaxf(v, dpp_ror<0x124>(v));
    v = fmaxf(v, dpp_ror<0x122>(v));
    return fmaxf(v, dpp_ror<0x121>(v));
}
// of the four rows' values (uniform)
__device__ __forceinline__ float lane_f(float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
__device__ __forceinline__ float rows_min(float v) {
    return fminf(fminf(lane_f(v, 0), lane_f(v, 16)), fminf(lane_f(v, 32), lane_f(v, 48)));
}
__device__ __forceinline__ float rows_max(float v) {
    return fmaxf(fmaxf(lane_f(v, 0), lane_f(v, 16)), fmaxf(lane_f(v, 32), lane_f(v, 48)));
}
__device__ __forceinline__ double unid(double v) {
    return __hiloint2double(uni(__double2hiint(v)), uni(__double2loint(v)));
}
// inclusive prefix sum and running maximum over the wave; values >= 0
__device__ __forceinline__ int wave_prefix(int v) {
    v += dpp_or_zero<0x111, 0xf>(v);
    v += dpp_or_zero<0x112, 0xf>(v);
    v += dpp_or_zero<0x114, 0xf>(v);
    v += dpp_or_zero<0x118, 0xf>(v);
    v += dpp_or_zero<0x142, 0xa>(v);
    v += dpp_or_zero<0x143, 0xc>(v);
    return v;
}
__device__ __forceinline__ int wave_scan_max(int v) {
    v = max(v, dpp_or_zero<0x111, 0xf>(v));
    v = max(v, dpp_or_zero<0x112, 0xf>(v));
    v = max(v, dpp_or_zero<0x114, 0xf>(v));
    v = max(v, dpp_or_zero<0x118, 0xf>(v));
    v = max(v, dpp_or_zero<0x142, 0xa>(v));
    v = max(v, dpp_or_zero<0x143, 0xc>(v));
    return v;
}
// lane I of the lane's row
template <int I>
__device__ __forceinline__ double row_bcast(double v) {
    return __hiloint2double(__builtin_amdgcn_mov_dpp(__double2hiint(v), 0x150 + I, 0xf, 0xf, false),
                            __builtin_amdgcn_mov_dpp(__double2loint(v), 0x150 + I, 0xf, 0xf, false));
}
// clamp to [lo, hi] in one instruction (lo <= hi)
__device__ __forceinline__ int med3i(int v, int lo, int hi) {
    int r;
    asm("v_med3_i32 %0, %1, %2, %3" : "=v"(r) : "v"(v), "v"(lo), "v"(hi));
    return r;
}
// an entry of a bucket table at a byte offset of the workgroup's LDS
__device__ __forceinline__ uint2 lds_entry(uint32_t off) {
    typedef __attribute__((address_space(3))) const unsigned long long lds_u64;
    const unsigned long long v = *(lds_u64*)(uintptr_t)off;
    return make_uint2((uint32_t)v, (uint32_t)(v >> 32));
}
// t = e - c; the address step: lo, or hi where e < c
__device__ __forceinline__ void edge_step(uint32_t e, uint32_t c, uint32_t lo, uint32_t hi, uint32_t& t, uint32_t& step) {
    asm("v_sub_co_u32_e32 %0, vcc, %2, %3\n\tv_cndmask_b32_e32 %1, %4, %5, vcc"
        : "=&v"(t), "=v"(step)
        : "v"(e), "v"(c), "v"(lo), "v"(hi)
        : "vcc");
}
// t = e - c, kout = k + (e < c): one subtraction with borrow, one addition with carry
__device__ __forceinline__ void sub_borrow(uint32_t e, uint32_t c, uint32_t k, uint32_t& t, uint32_t& kout) {
    asm("v_sub_co_u32_e32 %0, vcc, %2, %3\n\tv_addc_co_u32_e32 %1, vcc, 0, %4, vcc"
        : "=&v"(t), "=v"(kout)
        : "v"(e), "v"(c), "v"(k)
        : "vcc");
}
// additions at a byte offset of the workgroup's LDS
__device__ __forceinline__ void lds_add(uint32_t off, uint32_t v) {
    typedef __attribute__((address_space(3))) uint32_t lds_u32;
    __hip_atomic_fetch_add((lds_u32*)(uintptr_t)off, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void lds_add(uint32_t off, double v) {
    typedef __attribute__((address_space(3))) double lds_f64;
    __hip_atomic_fetch_add((lds_f64*)(uintptr_t)off, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// VAR: product marks compiled in (kModeWSum, kModeWXYZ: 1; 2, 3: other marks of
// two or one weights per point; 0: any); the swapped Jacobian pass (kModeJac: lanes are sample 2, the stream is
// sample 1).  ALSO: plain
// counts beside the sums.
template <int MODE, int VAR, int ALSO, int WAVES>
__global__ void __launch_bounds__(WAVES * 64, HP_TILE_WPS) k_tiles(const TileArgs A) {
    constexpr bool SWAP = (MODE == kModeJac) && VAR;
    constexpr bool PROD = (MODE == kModeWSum || MODE == kModeWXYZ) && VAR == 1;
    constexpr bool XY = (MODE == kModeXYZ || MODE == kModeWXYZ || MODE == kModeProj);
    // jackknife tables of an auto-count: per-lane-point rows, counts (VAR 0: unit
    // weights, u32) or sums of the pairs' products (VAR 1, FP64), added up by the
    // lane points' tags at the end.  (A point's weight times the sum of its
    // partners' would be one product per row, but is not a number where an infinite
    // weight meets a bin without pairs; the product per pair took 1546 against 1523
    // us a call at 1M points, 592 against 610 at 200k.)
    constexpr bool JK = (MODE == kModeJack);
    constexpr bool F64 = (MODE == kModeWSum || MODE == kModeWXYZ || MODE == kModeJac || MODE == kModeTan || (JK && VAR));
    constexpr bool TAN = (MODE == kModeTan);
    constexpr int kDeal = deal_of(MODE, VAR), kDealH = kDeal / 64;
    using ST = Stage<kDeal>;
    constexpr int kStage = ST::kStage, kSlots = ST::kSlots;
    constexpr int kPad = (F64 ? 3 : 2) * kSub;  // a list is read this far past its end
    extern __shared__ __align__(16) unsigned char lds[];
    const PairLaunch& L = A.L;
    const int lane = threadIdx.x & 63;
    const int wid = uni(threadIdx.x >> 6);
    const int K = L.br.nbins, Kp = XY ? L.bp.nbins : 1;
    const int nw = !F64                             ? 0
                   : TAN || VAR == 2                ? 2
                   : (MODE == kModeJac || JK)       ? 1
                   : (VAR == 1 || VAR == 3)         ? 1
                                                    : L.nw;
    const int wst = JK ? 2 : nw;  // doubles per weight row (jackknife: weight and tag)
    unsigned char* const wsm = lds + A.tab_bytes + wid * A.wave_bytes;
    // Bytes from a bin's histogram row to the next (and from a pi bin to the
    // next): the tables' entries hold the bin's offset, so that a pair's address
    // takes a select and an addition per table, and rows of pairs beyond the
    // last edge exist and are not read (adding under a mask costs more than
    // their space: per-object rows 1195 -> 1266 us).  Where many pairs would
    // meet on a few such cells (one histogram column), the bins' numbers are kept
    // instead and those pairs masked off ((rp, pi) counts 1905 -> 2090 us without).
    constexpr uint32_t TC = kTanCols, TR = 8u * TC;  // forward mode: columns of the W, dW and count rows
    constexpr bool CELL = MODE == kModeWXYZ || (MODE == kModeXYZ && VAR);
    const uint32_t rbytes = CELL ? 1u
                            : MODE == kModeXYZ ? (uint32_t)(Kp + 1) << (2 + A.ccol_sh)
                            : (MODE == kModeObj || (JK && !VAR)) ? 256u
                            : (MODE == kModeJac || JK) ? 512u
                            : TAN ? (ALSO ? 3u : 2u) * TR : 128u;
    const uint32_t pbytes = CELL ? 1u : (MODE == kModeXYZ ? 4u << A.ccol_sh : 0x10000u);
    {
        const uint2* gt = reinterpret_cast<const uint2*>(static_cast<const char*>(L.ws) + A.tr.off);
        uint2* st = reinterpret_cast<uint2*>(lds);
        for (int i = threadIdx.x; i <= (int)A.tr.mask; i += WAVES * 64)
            st[i] = make_uint2(gt[i].x, gt[i].y * rbytes);
        if (XY) {
            const uint2* gp = reinterpret_cast<const uint2*>(static_cast<const char*>(L.ws) + A.tp.off);
            uint2* sp = reinterpret_cast<uint2*>(lds + A.tp_off);
            for (int i = threadIdx.x; i <= (int)A.tp.mask; i += WAVES * 64)
                sp[i] = make_uint2(gp[i].x, gp[i].y * pbytes);
        }
    }
    double* const SX = reinterpret_cast<double*>(wsm);  // x[kSlots], y, z, n
    uint32_t* const ID = reinterpret_cast<uint32_t*>(wsm + ST::kIdOff);
    uint8_t* const list = wsm + ST::kListOff;
    uint8_t* const mark = wsm + ST::kMarkOff;
    float* const info = reinterpret_cast<float*>(wsm + ST::kInfoOff);  // per sub-group: low x, y, z, high x, y, z; the group's
    double* const LWT = reinterpret_cast<double*>(wsm + A.lw_off);  // lane points' weights: [nw][64]
    unsigned char* const hist = wsm + A.hist_off;
    __syncthreads();  // no block-level synchronisation below

    // Work items (lane groups or parts of them) in chunks of consecutive ones:
    // chunk c belongs to queue c % 8, and the waves of block b work on queue
    // b % 8 (blocks go to the XCDs round-robin, so an XCD's L2 sees one region;
    // the counter decides who takes an item, whichever XCD it runs on).  The
    // waves start on the first items and take the others one by one: with one
    // item per wave a workgroup's LDS stayed taken until the longest of its
    // waves was done, 12 of 16 waves alive on average (64-mock step 42.3 ->
    // 38.4 ms, (rp, pi) counts of 2M points 2220 -> 1900 us, 1M counts 810 ->
    // 745).  An addition or a look at a counter occupies its line for ~10 ns, so
    // a wave whose queue is empty ends: moving on to the others made every wave
    // look at eight lines (+75 us at 20k points); chunks of 64 items keep the
    // queues even instead (256: 1M counts 763 us).
    auto item_of = [&](int64_t t) __attribute__((always_inline)) -> int64_t {
        return ((((t >> A.chunk_sh) << 3) + (blockIdx.x & 7)) << A.chunk_sh) + (t & ((1 << A.chunk_sh) - 1));
    };
    auto take = [&]() __attribute__((always_inline)) -> int64_t {
        if (!A.queue) return -1;
        uint32_t c = 0u;
        if (lane == 0)
            c = __hip_atomic_fetch_add(A.queue + (blockIdx.x & 7) * kQueueWords, 1u, __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
        const int64_t it = item_of((int64_t)A.taken + (uint32_t)uni((int)c));
        return it < A.items ? it : -1;
    };
    int64_t item = item_of((int64_t)(blockIdx.x >> 3) * WAVES + wid);
    if (item >= A.items) item = take();
    const int lane0 = lane;
    for (; item >= 0; item = take()) {
        // (the empty asm keeps what follows from the lane inside the loop: kept in
        // registers from item to item, it would push the tiles' into scratch)
        int lane = lane0;
        kernarg_tile_args* args = (kernarg_tile_args*)__builtin_amdgcn_kernarg_segment_ptr();
        asm volatile("" : "+v"(lane), "+s"(args));
        kernarg_tile_args& A = *args;
        const __attribute__((address_space(4))) PairLaunch& L = A.L;
        for (int i = lane; i < (A.wave_bytes - A.hist_off) / 4; i += 64) reinterpret_cast<uint32_t*>(hist)[i] = 0u;
        int psh = A.parts_sh;
        int64_t g = item >> psh;
        int64_t it = item;
        if (g >= A.tail) {
            // the last groups go out in smaller items, which even out the end of the launch
            it -= A.tail << psh;
            psh = A.tail_sh;
            g = A.tail + (it >> psh);
        }
        const int parts = 1 << psh;
        const int part = uni((int)(it & (parts - 1)));

        constexpr int SD = SWAP ? 1 : 0;  // the lanes' side of the geometry, the stream's
        constexpr int SS = 1 - SD;
        const int m = L.group_mock ? uni(L.group_mock[g]) : 0;
        const_geom* const geom = (const_geom*)(L.geom + m);
        const int64_t gl = g - geom->group_off[SD];
        const int64_t p0 = geom->p_off[SD] + gl * kGroup;
        const int64_t left = geom->n[SD] - gl * kGroup;
        const int cnt = uni((int)(left < kGroup ? left : kGroup));
        const bool act = lane < cnt;
        const float r2xy = geom->r2xy;
        const float Rz = geom->search[2];
        const bool sym = L.sym != 0;
        const bool own = L.own != 0;  // one sample, every ordered pair from its first point: the group's own points come last

        // ---- the group's box, and the lane points relative to its centre
        float hx, hy, hz;     // half sizes, with the eps margin
        double cx, cy, cz;
        double Bf[4], NA[4];  // per sub-group: the tile's B operand and |a|^2
        int floor_hi;         // pairs below this high word are evaluated exactly
        int floor_pi = 0;     // ... (rp, pi): below this high word of dz^2
        bool low;             // ... which only matters where an edge is not above it
        {
            const float INF = __builtin_inff();
            const float eps = geom->eps;
            const double4 pr = reinterpret_cast<const double4*>(L.lane.x)[p0 + (act ? lane : 0)];
            const double px = pr.x, py = pr.y, pz = pr.z;
            // boxes of the sub-groups, one 16-lane row of the wave each
            float xl = row_min(act ? f32_down(px) : INF) - eps, xh = row_max(act ? f32_up(px) : -INF) + eps;
            float yl = row_min(act ? f32_down(py) : INF) - eps, yh = row_max(act ? f32_up(py) : -INF) + eps;
            float zl = row_min(act ? f32_down(pz) : INF) - eps, zh = row_max(act ? f32_up(pz) : -INF) + eps;
            const float bxlo = rows_min(xl), bylo = rows_min(yl), bzlo = rows_min(zl);
            const float bxhi = rows_max(xh), byhi = rows_max(yh), bzhi = rows_max(zh);
            const float fx = unif(0.5f * (bxlo + bxhi)), fy = unif(0.5f * (bylo + byhi)), fz = unif(0.5f * (bzlo + bzhi));
            cx = unid((double)fx);
            cy = unid((double)fy);
            cz = unid((double)fz);
            // half sizes of the box about its (rounded) centre; the eps margin covers the rounding
            hx = unif(0.5f * (bxhi - bxlo));
            hy = unif(0.5f * (byhi - bylo));
            hz = unif(0.5f * (bzhi - bzlo));
            const double ax = px - cx, ay = py - cy, az = pz - cz;
            const double na = !act ? kFar : (XY ? ax * ax + ay * ay : ax * ax + ay * ay + az * az);
            if ((lane & 15) == 0) {
                float* const f = info + (lane >> 4) * 8;
                f[0] = xl - fx; f[1] = yl - fy; f[2] = zl - fz; f[3] = xh - fx; f[4] = yh - fy; f[5] = zh - fz;
            }
            if (lane == 0) {
                float* const f = info + 32;
                f[0] = bxlo; f[1] = bylo; f[2] = bzlo; f[3] = bxhi; f[4] = byhi; f[5] = bzhi;
                // the window of cubes (the eps margin of the box covers the rounding here)
                const int nc = geom->ndiv[0];
                const int j0 = geom->pbc ? -nc : 0, j1 = geom->pbc ? 2 * nc - 1 : nc - 1;
                const float R = geom->search[0];
                const float ix = (float)geom->inv_cell[0], iy = (float)geom->inv_cell[1], iz = (float)geom->inv_cell[2];
                const int jx0 = max((int)floorf((bxlo - R) * ix), j0), jx1 = min((int)floorf((bxhi + R) * ix), j1);
                const int jy0 = max((int)floorf((bylo - R) * iy), j0), jy1 = min((int)floorf((byhi + R) * iy), j1);
                const int jz0 = max((int)floorf((bzlo - Rz) * iz), j0), jz1 = min((int)floorf((bzhi + Rz) * iz), j1);
                const int wy = jy1 - jy0 + 1, wz = jz1 - jz0 + 1;
                int* const w = reinterpret_cast<int*>(info) + 40;
                w[0] = jx0; w[1] = jy0; w[2] = jz0; w[3] = wy; w[4] = wz;
                w[5] = (jx1 >= jx0 && wy > 0 && wz > 0) ? (jx1 - jx0 + 1) * wy * wz : 0;
                f[14] = 1.0f / (float)wy;
                f[15] = 1.0f / (float)wz;
                f[16] = (float)geom->cell[0]; f[17] = (float)geom->cell[1]; f[18] = (float)geom->cell[2];
                // the slot that fills up a tile
                SX[kStage] = 0.0;
                SX[kSlots + kStage] = 0.0;
                SX[2 * kSlots + kStage] = 0.0;
                SX[3 * kSlots + kStage] = kFar;
                ID[kStage] = 0u;
            }
            if (F64) {
                const double* w = L.lane.w + (p0 + (act ? lane : 0)) * wst;
                for (int c = 0; c < nw; c++) LWT[c * 64 + lane] = w[c];
            }
            // B operand: lane l holds component l / 16 of point l % 16 of the sub-group
            SX[lane] = act ? -2.0 * ax : 0.0;
            SX[kSlots + lane] = act ? -2.0 * ay : 0.0;
            SX[2 * kSlots + lane] = (act && !XY) ? -2.0 * az : 0.0;
            SX[3 * kSlots + lane] = na;
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int s = 0; s < 4; s++) {
                const double v = SX[min(lane >> 4, 2) * kSlots + s * kSub + (lane & 15)];
                Bf[s] = (lane >> 4) == 3 ? 1.0 : v;
                NA[s] = SX[3 * kSlots + s * kSub + (lane & 15)];
            }
            __builtin_amdgcn_wave_barrier();
            if (XY) {
                // the lane points' z, read by the tiles
                reinterpret_cast<double*>(wsm + A.lw_off)[nw * 64 + lane] = az;
            }
            // Rounding of |a|^2 + |b|^2 - 2 a.b: below 2^-47 (|a|^2 + |b|^2), with
            // |a| <= h (half the box diagonal) and |b| <= h + R.  One unit of the
            // high word of d is at least 2^-21 d, so the rounding stays within a
            // unit for d >= 2^-26 S; the floor takes twice that.  The rounding of
            // the centre and of the periodic shift (2^-52 of the box) is covered
            // by the second term (dz^2 has only that one).
            const float h = sqrtf(hx * hx + hy * hy + (XY ? 0.f : hz * hz)) * 1.001f, hr = h + geom->search[0] * 1.001f;
            const double Lmax = fmax(fmax(geom->period[0], geom->period[1]), geom->period[2]);
            const double fl2 = Lmax * Lmax * 3.5527136788005009e-15;                          // 2^-48
            const double fl = (double)(h * h + hr * hr) * 2.9802322387695312e-08 + fl2;      // 2^-25
            floor_hi = uni(__double2hiint(fl) + 1);
            // (below every edge, all of them lie in the first bin)
            low = CELL || floor_hi + 2 >= (int)A.tr.first;
            if (XY) {
                floor_pi = uni(__double2hiint(fl2) + 1);
                low = low || floor_pi + 2 >= (int)A.tp.first;
            }
        }

        bool self_done = false;
        [[maybe_unused]] bool tied = false;  // Jacobian: the group's rows of corr are in use
        const uint32_t sbase = (uint32_t)uni((int)geom->p_off[SS]);
        const int tlo = (int)A.tr.lo, thi = (int)A.tr.hi;
        const uint32_t tsh = A.tr.sh3, tmask = A.tr.mask << 3;
        const int plo = (int)A.tp.lo, phi = (int)A.tp.hi;
        const uint32_t psh3 = A.tp.sh3, pmask = A.tp.mask << 3, ptab = (uint32_t)A.tp_off;
        const int lrow = ((lane & 3) << 2) | ((lane >> 2) & 3);   // list position of this lane's A row
        const int brow = ((lane >> 4) << 2) | (lane & 3);         // list position of the D row this lane's row broadcasts
        const double* const comp = SX + (lane >> 4) * kSlots;     // the component this lane holds of the A operand
        // histogram columns: u32 rows of 32 columns, f64 rows of 16 (no two lanes of
        // one LDS pass on one address); per lane point for object rows and Jacobians
        const uint32_t col4 = (uint32_t)(lane & 31) * 4u, col8 = (uint32_t)(lane & 15) * 8u;
        const uint32_t tcol8 = (uint32_t)(lane & (TC - 1)) * 8u, tcol4 = (uint32_t)(lane & (2 * TC - 1)) * 4u;
        const uint32_t ccol = (uint32_t)A.ccol_sh, ccl = (uint32_t)(lane & ((1 << A.ccol_sh) - 1));
        const uint32_t hbase = (uint32_t)(A.tab_bytes + wid * A.wave_bytes + A.hist_off);
        const uint32_t cbase = (uint32_t)(A.tab_bytes + wid * A.wave_bytes + A.cnt_off);
        uint64_t evals = 0;
        const double* const SWm = F64 ? L.strm.w + (int64_t)sbase * wst : nullptr;

        // Exact bin of the pair (lane point j of the group, staged slot): the first
        // edge not below the distance, scanning from edge k (and q along pi).  Rarely
        // taken: what it needs is loaded here, not kept in registers through the
        // kernel (the empty asm hides that it is the same).  rev: the pair's other
        // orientation, (x2 + shift) - x1.
        auto exact_bin = [&](int j, int slot, uint32_t k, uint32_t& kp, bool rev) __attribute__((always_inline)) -> uint32_t {
            kernarg_tile_args* ap = (kernarg_tile_args*)__builtin_amdgcn_kernarg_segment_ptr();
            const_geom* gp = geom;
            asm volatile("" : "+s"(ap), "+s"(gp));
            const double* ge = reinterpret_cast<const double*>(static_cast<const char*>(ap->L.ws) + ap->L.br.edges_off);
            const int64_t first = gp->p_off[SD] + gl * kGroup;
            const double* pl = ap->L.lane.x + (first + min(j, cnt - 1)) * 4;
            double px = pl[0], py = pl[1], pz = pl[2];
            const uint32_t id = ID[slot];
            const int img = (int)(id >> kImgShift);
            const double* r = ap->L.strm.x + (gp->p_off[SS] + (int64_t)(id & kRowMask)) * 4;
            const int tx = (img & 3) - 1, ty = ((img >> 2) & 3) - 1, tz = (img >> 4) - 1;
            double qx = r[0], qy = r[1], qz = r[2];
            // the image of the stream point lies at q + t L; the reference shifts the sample-1 point
            if ((!SWAP && !rev) || (SWAP && rev)) {
                if (tx) px = px - (double)tx * gp->period[0];
                if (ty) py = py - (double)ty * gp->period[1];
                if (tz) pz = pz - (double)tz * gp->period[2];
            } else {
                if (tx) qx = qx + (double)tx * gp->period[0];
                if (ty) qy = qy + (double)ty * gp->period[1];
                if (tz) qz = qz + (double)tz * gp->period[2];
            }
            const double dx = px - qx, dy = py - qy, dz = pz - qz;
            if (XY) {
                const double* gq = reinterpret_cast<const double*>(static_cast<const char*>(ap->L.ws) + ap->L.bp.edges_off);
                const double dz2 = dz * dz;
                uint32_t q = 0;
                while (gq[q] < dz2) ++q;
                kp = q;
                const double dxy = dx * dx + dy * dy;
                while (ge[k] < dxy) ++k;
            } else {
                const double dsq = dx * dx + dy * dy + dz * dz;
                while (ge[k] < dsq) ++k;
            }
            return k;
        };

        const uint32_t own0 = (uint32_t)(p0 - (int64_t)sbase);  // the group's first row, in one sample

        // ---- staged points: deal them to the sub-groups, evaluate the tiles
        // self: the slots hold the group's own points
        int qlen = 0;
        auto process = [&](bool self) __attribute__((always_inline)) {
            float fx[kDealH], fy[kDealH], fz[kDealH];
            uint64_t in[kDealH], plain[kDealH];
#pragma unroll
            for (int h = 0; h < kDealH; h++) {
                const int slot = h * 64 + lane;
                in[h] = (uint64_t)__ballot(slot < qlen);
                fx[h] = (float)SX[slot];
                fy[h] = (float)SX[kSlots + slot];
                fz[h] = (float)SX[2 * kSlots + slot];
                plain[h] = sym ? (uint64_t)__ballot((ID[slot] >> kImgShift) == (uint32_t)kHere) & in[h] : 0ull;
            }
            // symmetric counts: the shifted points (once), then the unshifted ones
            // (twice); other counts: every point once
            const bool two = sym && !self;
            for (int sc = two ? 0 : 4; sc < 8; sc++) {
                const int s = sc & 3;
                uint64_t mk[kDealH], any = 0;
#pragma unroll
                for (int h = 0; h < kDealH; h++) {
                    mk[h] = !two ? in[h] : (sc < 4 ? in[h] & ~plain[h] : plain[h]);
                    any |= mk[h];
                }
                if (any == 0) {
                    sc |= 3;  // none of this class
                    continue;
                }
                uint32_t inc = (two && sc >= 4) ? 2u : 1u;
                int n;
                if (self) {
                    n = sym ? min(qlen, (s + 1) * kSub) : qlen;  // the group's points (up to this sub-group)
                    list[lane] = (uint8_t)lane;
                    if (lane < kPad) list[64 + lane] = (uint8_t)kStage;
                } else {
                    // staged points near the sub-group's box
                    const float4 b0 = *reinterpret_cast<const float4*>(info + 8 * s);
                    const float2 b1 = *reinterpret_cast<const float2*>(info + 8 * s + 4);
                    n = 0;
#pragma unroll
                    for (int h = 0; h < kDealH; h++) {
                        const float gx = fmaxf(0.f, fmaxf(fx[h] - b0.w, b0.x - fx[h]));
                        const float gy = fmaxf(0.f, fmaxf(fy[h] - b1.x, b0.y - fy[h]));
                        const float gz = fmaxf(0.f, fmaxf(fz[h] - b1.y, b0.z - fz[h]));
                        const float gxy = __builtin_fmaf(gy, gy, gx * gx);
                        const bool near = XY ? (gxy <= r2xy && gz <= Rz) : (__builtin_fmaf(gz, gz, gxy) <= r2xy);
                        const uint64_t mm = (uint64_t)__ballot(near) & mk[h];
                        const uint32_t r = __builtin_amdgcn_mbcnt_hi((uint32_t)(mm >> 32),
                                                                     __builtin_amdgcn_mbcnt_lo((uint32_t)mm, (uint32_t)n));
                        if (__builtin_amdgcn_inverse_ballot_w64(mm)) list[r] = (uint8_t)(h * 64 + lane);
                        n += __builtin_popcountll(mm);
                    }
                    if (n == 0) continue;
                    if (lane < kPad) list[n + lane] = (uint8_t)kStage;
                    evals += (uint64_t)n * kSub;
                }
                __builtin_amdgcn_wave_barrier();
                const double bs = s == 0 ? Bf[0] : (s == 1 ? Bf[1] : (s == 2 ? Bf[2] : Bf[3]));
                const double ns = s == 0 ? NA[0] : (s == 1 ? NA[1] : (s == 2 ? NA[2] : NA[3]));
                const dbl4 cc = {ns, ns, ns, ns};
                // this sub-group's lane points: weights and z
                const int lj = s * kSub + (lane & 15);
                // the first bin's address for this lane, the second's, the one past the last edge
                const uint32_t adr0 = CELL ? 0u : hbase + (MODE == kModeXYZ ? ccl * 4u
                                               : (MODE == kModeObj || (JK && !VAR)) ? (uint32_t)lj * 4u
                                               : (MODE == kModeJac || JK) ? (uint32_t)lj * 8u
                                               : TAN ? tcol8 : (MODE == kModeWSum ? col8 : col4));
                const uint32_t adr1 = adr0 + rbytes, trash = adr0 + (uint32_t)K * rbytes;
                double lw[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
                if (F64) {
#pragma unroll
                    for (int c = 0; c < 5; c++)
                        if (c < nw) lw[c] = LWT[c * 64 + lj];
                }
                if (TAN && sym && !self && sc < 4) {
                    // symmetric sums are doubled at the end: a shifted pair counts from both sides
                    lw[0] *= 0.5;
                    lw[1] *= 0.5;
                }
                double za = 0.0;
                if (XY) za = LWT[nw * 64 + lj];
                // stream weights of the D row this lane's row broadcasts
                double wn[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
                auto load_weights = [&](uint32_t row) __attribute__((always_inline)) {
                    const double* w = SWm + (uint32_t)(row * (uint32_t)wst);
#pragma unroll
                    for (int c = 0; c < 5; c++)
                        if (c < nw) wn[c] = w[c];
                };
                // (loaded a tile ahead, their rows two and the slots three: the chain of
                // reads does not hold up a tile)
                uint32_t wrow = 0u;
                int wslot = 0;
                if (F64) {
                    load_weights(ID[list[brow]] & kRowMask);
                    wrow = ID[list[kSub + brow]] & kRowMask;
                    wslot = list[2 * kSub + brow];
                }
                // operands one tile ahead, their slots two
                double a = comp[list[lrow]];
                int slot2 = list[kSub + lrow];
                for (int t0 = 0; t0 < n; t0 += kSub) {
                    // rows: staged points list[t0 + 4 (lane / 16) + i]; columns: the sub-group's points
                    const double a1 = comp[slot2];
                    slot2 = list[t0 + 2 * kSub + lrow];
                    double zb = 0.0, wb[5];
                    if (XY) zb = SX[2 * kSlots + list[t0 + brow]];
                    if (F64) {
                        // this tile's stream weights were loaded a tile ago
#pragma unroll
                        for (int c = 0; c < 5; c++) wb[c] = wn[c];
                        load_weights(wrow);
                        wrow = ID[wslot] & kRowMask;
                        wslot = list[t0 + 3 * kSub + brow];
                    }
                    // (the next operands' reads go out before the product, which would otherwise
                    // hold them back: its result registers are reused at once)
                    __builtin_amdgcn_sched_barrier(0);
                    const dbl4 D = __builtin_amdgcn_mfma_f64_16x16x4f64(a, bs, cc, 0, 0, 0);
                    a = a1;
                    int hi[4], hp[4], c[4];
                    uint2 ent[4], enp[4];
                    uint32_t t[4], st[4], tp[4], sp[4], adr[4], pad[4];  // (addresses: row, pi part)
#pragma unroll
                    for (int i = 0; i < 4; i++) hi[i] = __double2hiint(D[i]);
                    bool diag = false;
                    if (self) {
                        inc = sym ? 2u : 1u;
                        diag = t0 == s * kSub;
                        if (diag) {
                            // inside a sub-group: ordered pairs, without a point and itself
                            inc = 1u;
#pragma unroll
                            for (int i = 0; i < 4; i++)
                                if ((lane >> 4) * 4 + i == (lane & 15)) hi[i] = 0x7e000000;
                        }
                    }
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        c[i] = med3i(hi[i], tlo, thi);
                        ent[i] = lds_entry(((uint32_t)c[i] >> tsh) & tmask);
                    }
                    if (XY) {
                        double dz[4];
                        dz[0] = row_bcast<0>(zb) - za;
                        dz[1] = row_bcast<1>(zb) - za;
                        dz[2] = row_bcast<2>(zb) - za;
                        dz[3] = row_bcast<3>(zb) - za;
#pragma unroll
                        for (int i = 0; i < 4; i++) {
                            hp[i] = __double2hiint(dz[i] * dz[i]);
                            const uint32_t off = (((uint32_t)med3i(hp[i], plo, phi) >> psh3) & pmask) | ptab;
                            enp[i] = lds_entry(off);
                        }
                    }
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        // (the clamped value: rounding may leave a square below zero)
                        if (CELL) {
                            sub_borrow(ent[i].x, (uint32_t)hi[i], ent[i].y, t[i], adr[i]);
                        } else {
                            edge_step(ent[i].x, (uint32_t)c[i], adr0, adr1, t[i], st[i]);
                            adr[i] = ent[i].y + st[i];
                        }
                    }
                    uint64_t odd = (uint64_t)__ballot(min(min(t[0], t[1]), min(t[2], t[3])) <= 2u);
                    if (XY) {
#pragma unroll
                        for (int i = 0; i < 4; i++) {
                            if (CELL) {
                                sub_borrow(enp[i].x, (uint32_t)hp[i], enp[i].y, tp[i], pad[i]);
                            } else {
                                edge_step(enp[i].x, (uint32_t)hp[i], 0u, pbytes, tp[i], sp[i]);
                                pad[i] = enp[i].y + sp[i];
                            }
                        }
                        odd |= (uint64_t)__ballot(min(min(tp[0], tp[1]), min(tp[2], tp[3])) <= 2u);
                    }
                    if (CELL || low) {
                        if (!CELL) asm volatile("");  // (a branch: most groups have no use for this)
                        odd |= (uint64_t)__ballot(min(min(hi[0], hi[1]), min(hi[2], hi[3])) < floor_hi);
                        if (XY) odd |= (uint64_t)__ballot(min(min(hp[0], hp[1]), min(hp[2], hp[3])) < floor_pi);
                    }
                    if (__builtin_expect(odd != 0, 0)) {
                        [[maybe_unused]] uint32_t ties = 0u;  // Jacobian: this lane's pairs whose other order has a bin of its own
#pragma unroll 1
                        for (int i = 0; i < 4; i++) {
                            const uint32_t ti = i == 0 ? t[0] : (i == 1 ? t[1] : (i == 2 ? t[2] : t[3]));
                            const int hv = i == 0 ? hi[0] : (i == 1 ? hi[1] : (i == 2 ? hi[2] : hi[3]));
                            const uint32_t eo = i == 0 ? ent[0].y : (i == 1 ? ent[1].y : (i == 2 ? ent[2].y : ent[3].y));
                            bool oi = ti <= 2u || (low && hv < floor_hi);
                            if (XY) {
                                const uint32_t pi = i == 0 ? tp[0] : (i == 1 ? tp[1] : (i == 2 ? tp[2] : tp[3]));
                                const int hq = i == 0 ? hp[0] : (i == 1 ? hp[1] : (i == 2 ? hp[2] : hp[3]));
                                oi = (oi || pi <= 2u || (low && hq < floor_pi)) && hv < 0x7e000000;
                            }
                            if (oi) {
                                const int slot = list[t0 + (lane >> 4) * 4 + i];
                                // (a bin's number from its offset, exactly: both are far below 2^22)
                                const uint32_t ek = (uint32_t)((float)eo / (float)rbytes + 0.5f);
                                const uint32_t kb = (low && hv < floor_hi) || ek == 0u ? 0u : ek - 1u;
                                uint32_t kq = 0u, kk = 0u;
                                // (a Jacobian's points meet themselves in the tiles, at
                                // distance 0: 64 exact evaluations per group otherwise)
                                const bool itself = MODE == kModeJac && L.lane.x == L.strm.x &&
                                                    ID[slot] == (own0 + (uint32_t)lj | ((uint32_t)kHere << kImgShift));
                                if (!itself) kk = exact_bin(lj, slot, kb, kq, false);
                                if (MODE == kModeJac && !SWAP && L.corr != nullptr && (ID[slot] >> kImgShift) != (uint32_t)kHere) {
                                    // Auto-count with one set of weights: the sample-2 rows take
                                    // the pair's other orientation, which across the periodic seam
                                    // may round into another bin (only these pairs can differ).
                                    uint32_t dummy = 0u;
                                    const uint32_t kr = exact_bin(s * kSub + (lane & 15), slot, kb, dummy, true);
                                    if (kr != kk && s * kSub + (lane & 15) < cnt) ties |= 1u << i;
                                }
                                if constexpr (JK) {
                                    // A pair of two tags gives half of its weight to each.  The rows
                                    // give all of an ordered pair's to its lane point's tag, which is
                                    // the same where the pair's other order lands in the same bin;
                                    // across the periodic seam it may not, and half moves over.
                                    const uint32_t id = ID[slot];
                                    uint32_t dummy = 0u;
                                    const uint32_t kr = exact_bin(lj, slot, kb, dummy, true);
                                    if (kr != kk && (id >> kImgShift) != (uint32_t)kHere && lj < cnt) {
                                        const double* wi = L.lane.w + (p0 + lj) * 2;
                                        const double v = 0.5 * wi[0] * L.strm.w[((int64_t)sbase + (int64_t)(id & kRowMask)) * 2];
                                        const int t = (int)wi[1];
                                        double* r = L.jacc + ((int64_t)m * (L.nsamp + 1) + t) * K;
                                        if (t >= 1 && t <= L.nsamp) {
                                            if (kk < (uint32_t)K)
                                                __hip_atomic_fetch_add(r + kk, -v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                                            if (kr < (uint32_t)K)
                                                __hip_atomic_fetch_add(r + kr, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                                        }
                                    }
                                }
#pragma unroll
                                for (int u = 0; u < 4; u++)
                                    if (i == u) {
                                        adr[u] = adr0 + kk * rbytes;
                                        if (XY) pad[u] = kq * pbytes;
                                    }
                            }
                        }
                        if constexpr (MODE == kModeJac && !SWAP) {
                            // Such a pair moves the partner's weight from one bin to the other
                            // in the lane point's own row of corr, rows2 = rows1 + corr.  This
                            // wave alone has these rows: it clears them at the group's first
                            // such pair, and most groups never touch them.
                            if ((uint64_t)__ballot(ties != 0u) != 0) {
                                double* const crow = L.corr + p0 * K;
                                if (!tied) {
                                    for (int e = lane; e < cnt * K; e += 64) crow[e] = 0.0;
                                    __threadfence();
                                    tied = true;
                                }
#pragma unroll 1
                                for (int i = 0; i < 4; i++) {
                                    if (!((ties >> i) & 1u)) continue;
                                    const int slot = list[t0 + (lane >> 4) * 4 + i];
                                    uint32_t dummy = 0u;
                                    const uint32_t kf = exact_bin(lj, slot, 0u, dummy, false);
                                    const uint32_t kr = exact_bin(lj, slot, 0u, dummy, true);
                                    const double w = SWm[ID[slot] & kRowMask];
                                    double* const r = crow + lj * K;
                                    if (kf < (uint32_t)K) __hip_atomic_fetch_add(r + kf, -w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                                    if (kr < (uint32_t)K) __hip_atomic_fetch_add(r + kr, w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                                }
                            }
                        }
                    }
                    // ---- accumulate
                    // generic marks: one choice of the function for the tile's four rows (a
                    // choice per row took more issue slots than the marks themselves)
                    double mv[4] = {0.0, 0.0, 0.0, 0.0};
                    if constexpr ((MODE == kModeWSum || MODE == kModeWXYZ) && !PROD) {
                        wfunc_switch(L.wfunc, [&](auto id) __attribute__((always_inline)) {
#pragma unroll
                            for (int i = 0; i < 4; i++) {
                                double bw[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
#pragma unroll
                                for (int c = 0; c < 5; c++)
                                    if (c < nw)
                                        bw[c] = i == 0 ? row_bcast<0>(wb[c])
                                                : (i == 1 ? row_bcast<1>(wb[c])
                                                          : (i == 2 ? row_bcast<2>(wb[c]) : row_bcast<3>(wb[c])));
                                mv[i] = wfunc_one<decltype(id)::value>(lw, bw);
                            }
                        });
                    }
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        // the row's stream weights (all lanes: a broadcast reads none that is masked off)
                        double sw[5];
                        if constexpr (F64) {
#pragma unroll
                            for (int c = 0; c < 5; c++)
                                sw[c] = c >= nw ? 0.0
                                                : (i == 0 ? row_bcast<0>(wb[c])
                                                          : (i == 1 ? row_bcast<1>(wb[c])
                                                                    : (i == 2 ? row_bcast<2>(wb[c]) : row_bcast<3>(wb[c]))));
                        }
                        if constexpr (MODE == kModeCount3D) {
                            lds_add(adr[i], inc);
                        } else if constexpr (MODE == kModeProj) {
                            lds_add(min(adr[i] + pad[i], trash), inc);  // beyond pi_max: the row past the last edge
                        } else if constexpr (MODE == kModeXYZ && !VAR) {
                            lds_add(adr[i] + pad[i], inc);
                        } else if constexpr (CELL) {
                            if (adr[i] < (uint32_t)K && pad[i] < (uint32_t)Kp) {
                                const uint32_t cell = __umul24(adr[i], (uint32_t)Kp) + pad[i];
                                if constexpr (MODE == kModeXYZ)
                                    lds_add((cell << (ccol + 2)) + (hbase + ccl * 4u), inc);
                                else
                                    lds_add(cell * 8u + hbase, PROD ? lw[0] * sw[0] : mv[i]);
                            }
                        } else if constexpr (MODE == kModeObj || (JK && !VAR)) {
                            lds_add(adr[i], 1u);
                        } else if constexpr (MODE == kModeJac || JK) {
                            lds_add(adr[i], JK ? lw[0] * sw[0] : sw[0]);
                            if (ALSO) lds_add(((adr[i] - adr0) >> 2) + cbase + col4, 1u);
                        } else if constexpr (MODE == kModeTan) {
                            // pair terms w_i w_j and t_i w_j + w_i t_j (t = dw/dtheta); the
                            // group's own pairs: ordered ones inside a sub-group count half
                            if (adr[i] < trash) {
                                double wj = sw[0], tj = sw[1];
                                if (diag) {
                                    wj *= 0.5;
                                    tj *= 0.5;
                                }
                                lds_add(adr[i], lw[0] * wj);
                                lds_add(adr[i] + TR, __builtin_fma(lw[0], tj, lw[1] * wj));
                                if (ALSO) lds_add(adr[i] + (2 * TR + tcol4 - tcol8), inc);
                            }
                        } else {
                            lds_add(adr[i], PROD ? lw[0] * sw[0] : mv[i]);
                            if (MODE == kModeWSum && ALSO) lds_add(adr[i] - adr0 + cbase + col4, 1u);
                        }
                    }
                }
                __builtin_amdgcn_wave_barrier();
            }
            // what was not dealt moves to the front
            const int rest = self ? 0 : max(qlen - kDeal, 0);
            if (rest > 0 && lane < rest) {
                const int f = kDeal + lane;
                const double x = SX[f], y = SX[kSlots + f], z = SX[2 * kSlots + f], nn = SX[3 * kSlots + f];
                const uint32_t id = ID[f];
                SX[lane] = x;
                SX[kSlots + lane] = y;
                SX[2 * kSlots + lane] = z;
                SX[3 * kSlots + lane] = nn;
                ID[lane] = id;
            }
            __builtin_amdgcn_wave_barrier();
            qlen = rest;
        };

        // ---- the cubes of the curve near the group.  A lane takes one cube of the
        // window and looks up the stretch of rows it holds; the stretches of 64 cubes
        // form one list of rows, which is walked 64 rows at a time: a scan over the
        // starts gives each lane its stretch.  Symmetric counts drop the rows before
        // the group's end here (unshifted cubes), a whole stretch at a time.
        const double4* const SR = reinterpret_cast<const double4*>(L.strm.x) + sbase;
        int cube0 = -64;                // the next 64 cubes of the window
        int cimg = 0;                   // the lane's cube: its image
        bool seam = false;              // some cube of the list is a periodic image
        int pre = 0, end = 0, run = 0;  // the lane's stretch: its place [pre, end) in the list, first row - pre
        int at = 0, total = 0;          // list position of the next rows, rows in the list
        // the next 64 rows: false when the group has no more.  The list is made
        // rarely: what that needs is loaded here.
        auto next = [&]() __attribute__((always_inline)) -> bool {
            at += 64;
            while (at >= total) {
                const_geom* gp = geom;
                asm volatile("" : "+s"(gp));
                const int cb = gp->cbits, nc = 1 << cb;  // cubes per dimension
                const int* const w = reinterpret_cast<const int*>(info) + 40;
                const int wy = w[3], wz = w[4], ncubes = uni(w[5]);
                cube0 += 64;
                if ((cube0 << psh) + part >= ncubes) return false;
                // cube ci of the window: z fastest (quotients from reciprocals: exact
                // for the few thousand cubes of a window, and one more test for more)
                const int ci = ((cube0 + lane) << psh) + part;
                int cxy = (int)((float)ci * info[47]);
                int jz = ci - cxy * wz;
                if (jz < 0) { jz += wz; cxy--; }
                if (jz >= wz) { jz -= wz; cxy++; }
                int jx = (int)((float)cxy * info[46]);
                int jy = cxy - jx * wy;
                if (jy < 0) { jy += wy; jx--; }
                if (jy >= wy) { jy -= wy; jx++; }
                jx += w[0];
                jy += w[1];
                jz += w[2];
                const float cxf = info[48], cyf = info[49], czf = info[50];
                const float gx = fmaxf(0.f, fmaxf((float)jx * cxf - info[35], info[32] - (float)(jx + 1) * cxf));
                const float gy = fmaxf(0.f, fmaxf((float)jy * cyf - info[36], info[33] - (float)(jy + 1) * cyf));
                const float gz = fmaxf(0.f, fmaxf((float)jz * czf - info[37], info[34] - (float)(jz + 1) * czf));
                at = 0;
                total = 0;
                const bool has = ci < ncubes && (XY ? gx * gx + gy * gy : gx * gx + gy * gy + gz * gz) <= r2xy;
                if ((uint64_t)__ballot(has) == 0) continue;
                // image: 0, 1, 2 for -L, 0, +L per dimension, two bits each
                const int ux = (jx >> cb) + 1, uy = (jy >> cb) + 1, uz = (jz >> cb) + 1;
                cimg = ux | (uy << 2) | (uz << 4);
                int len = 0;
                run = 0;
                if (has) {
                    const int cm = nc - 1;
                    const uint2 c = (L.strm.cubes + gp->cell_off)[(uint32_t)(((((jx & cm) << cb) + (jy & cm)) << cb) + (jz & cm))];
                    run = (int)c.x;
                    if (sym && cimg == kHere) run = max(run, (int)(gp->p_off[SD] + gl * kGroup + cnt));
                    len = max((int)c.y - run, 0);
                }
                seam = (uint64_t)__ballot(len > 0 && cimg != kHere) != 0;
                pre = wave_prefix(len);
                total = __builtin_amdgcn_readlane(pre, 63);
                end = len > 0 ? pre : -1;
                pre -= len;
                run -= pre + (int)sbase;
            }
            return true;
        };
        // this lane's row of the list (relative to the mock's first) and its image;
        // a row past the end repeats the last one
        auto fetch = [&](uint32_t& jj, int& img) __attribute__((always_inline)) {
            mark[lane] = 0;
            __builtin_amdgcn_wave_barrier();
            if (pre < at + 64 && end > at) mark[max(pre - at, 0)] = (uint8_t)lane;
            __builtin_amdgcn_wave_barrier();
            const int sg = wave_scan_max((int)mark[lane]) << 2;
            jj = (uint32_t)(min(at + lane, total - 1) + __builtin_amdgcn_ds_bpermute(sg, run));
            img = seam ? __builtin_amdgcn_ds_bpermute(sg, cimg) : kHere;
        };
        bool more = next();
        double4 row = make_double4(0.0, 0.0, 0.0, 0.0);
        uint32_t jn = 0;
        int imgn = kHere, nn = 0;  // the rows being loaded: indices, images, how many
        bool seamn = false;
        if (more) {
            fetch(jn, imgn);
            nn = total - at;
            seamn = seam;
            row = SR[jn];
        }
        for (;;) {
            bool self = false;
            if (more) {
                const double4 sr = row;
                const uint32_t jj = jn;
                const int img = imgn, nrow = nn;
                double x = sr.x - cx, y = sr.y - cy, z = sr.z - cz;
                if (seamn) {
                    const_geom* gp = geom;
                    asm volatile("" : "+s"(gp));
                    x = sr.x - __builtin_fma((double)(1 - (img & 3)), gp->period[0], cx);
                    y = sr.y - __builtin_fma((double)(1 - ((img >> 2) & 3)), gp->period[1], cy);
                    z = sr.z - __builtin_fma((double)(1 - (img >> 4)), gp->period[2], cz);
                }
                more = next();
                if (more) {
                    fetch(jn, imgn);
                    nn = total - at;
                    seamn = seam;
                    row = SR[jn];
                }
                const float gx = fmaxf(0.f, fabsf((float)x) - hx);
                const float gy = fmaxf(0.f, fabsf((float)y) - hy);
                const float gz = fmaxf(0.f, fabsf((float)z) - hz);
                const float gxy = __builtin_fmaf(gy, gy, gx * gx);
                // (the group's own rows wait for the end)
                const bool ok = lane < nrow && !(own && jj - own0 < (uint32_t)cnt && img == kHere) && (XY ? (gxy <= r2xy && gz <= Rz) : (__builtin_fmaf(gz, gz, gxy) <= r2xy));
                const uint64_t mk = (uint64_t)__ballot(ok);
                if (ok) {
                    const uint32_t slot = __builtin_amdgcn_mbcnt_hi(
                        (uint32_t)(mk >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mk, (uint32_t)qlen));
                    SX[slot] = x;
                    SX[kSlots + slot] = y;
                    SX[2 * kSlots + slot] = z;
                    SX[3 * kSlots + slot] = XY ? x * x + y * y : x * x + y * y + z * z;
                    ID[slot] = jj | ((uint32_t)img << kImgShift);
                }
                __builtin_amdgcn_wave_barrier();
                qlen += __builtin_popcountll(mk);
            } else if (qlen == 0) {
                if (!(sym || own) || part != 0 || self_done) break;
                // One sample, last: the group's own points.  Symmetric counts take each
                // unordered pair of different sub-groups twice and the ordered pairs
                // inside a sub-group once, other passes every ordered pair once; each
                // point with itself (distance 0: bin 0) is added here.
                const double4 pr = reinterpret_cast<const double4*>(L.lane.x)[p0 + (act ? lane : 0)];
                const double ax = pr.x - cx, ay = pr.y - cy, az = pr.z - cz;
                SX[lane] = act ? ax : 0.0;
                SX[kSlots + lane] = act ? ay : 0.0;
                SX[2 * kSlots + lane] = act ? az : 0.0;
                SX[3 * kSlots + lane] = !act ? kFar : (XY ? ax * ax + ay * ay : ax * ax + ay * ay + az * az);
                // (the lanes' rows are the stream's: one sample)
                ID[lane] = (uint32_t)(p0 + (act ? lane : 0) - (int64_t)sbase) | ((uint32_t)kHere << kImgShift);
                evals += (uint64_t)cnt * cnt;
                if constexpr (MODE == kModeTan) {
                    if (act) {
                        const double w = LWT[lane], t = LWT[64 + lane];
                        __hip_atomic_fetch_add(reinterpret_cast<double*>(hist + tcol8), 0.5 * (w * w), __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_WORKGROUP);
                        __hip_atomic_fetch_add(reinterpret_cast<double*>(hist + TR + tcol8), w * t, __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_WORKGROUP);
                    }
                    if (ALSO && lane == 0) *reinterpret_cast<uint32_t*>(hist + 2 * TR) += (uint32_t)cnt;
                } else if constexpr (MODE == kModeObj || (JK && !VAR)) {
                    if (act) reinterpret_cast<uint32_t*>(hist)[lane] += 1u;
                } else if constexpr (MODE == kModeJac || JK) {
                    if (act) reinterpret_cast<double*>(hist)[lane] += JK ? LWT[lane] * LWT[lane] : LWT[lane];
                } else if constexpr (MODE == kModeWSum || MODE == kModeWXYZ) {
                    if (act) {
                        double w[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
#pragma unroll
                        for (int c = 0; c < 5; c++)
                            if (c < nw) w[c] = LWT[c * 64 + lane];
                        const double v = PROD ? w[0] * w[0] : wfunc_eval(L.wfunc, w, w);
                        __hip_atomic_fetch_add(reinterpret_cast<double*>(hist + (MODE == kModeWSum ? col8 : 0u)), v,
                                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                    }
                } else {
                    if (lane == 0) *reinterpret_cast<uint32_t*>(hist) += (uint32_t)cnt;
                }
                if constexpr (ALSO && MODE != kModeTan) {
                    if (lane == 0) *reinterpret_cast<uint32_t*>(wsm + A.cnt_off) += (uint32_t)cnt;
                }
                __builtin_amdgcn_wave_barrier();
                qlen = cnt;
                self = true;
                self_done = true;
            }
            if (qlen >= kDeal || !more) process(self);
        }
        __builtin_amdgcn_wave_barrier();

        // ---- the group's results
        // columns are summed starting at a lane's own one (a bank per lane), counts
        // go to the mock's accumulators
        uint64_t* const cacc =
            L.pcount ? L.pcount + ((int64_t)m * L.crep + (int64_t)(gl % L.crep)) * ((MODE == kModeXYZ) ? K * Kp : K) : nullptr;
        if constexpr (MODE == kModeXYZ) {
            const uint32_t* h = reinterpret_cast<const uint32_t*>(hist);
            for (int k = lane; k < K * Kp; k += 64) {
                uint64_t tot = 0;
                const uint32_t cell = CELL ? (uint32_t)k : (uint32_t)k + (uint32_t)k / (uint32_t)Kp;  // (rows of Kp + 1)
                for (int c = 0; c < (1 << ccol); c++) tot += h[(cell << ccol) + ((c + lane) & ((1 << ccol) - 1))];
                if (tot) __hip_atomic_fetch_add(cacc + k, tot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        } else if constexpr (MODE == kModeCount3D || MODE == kModeProj || ALSO) {
            const uint32_t* h = reinterpret_cast<const uint32_t*>(wsm + A.cnt_off);
            constexpr int step = TAN ? 3 * (int)TR / 4 : 32, nc = TAN ? 2 * (int)TC : 32;
            for (int k = lane; k < K; k += 64) {
                uint64_t tot = 0;
                for (int c = 0; c < nc; c++) tot += h[k * step + ((c + lane) & (nc - 1))];
                if (tot) __hip_atomic_fetch_add(cacc + k, tot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
        if constexpr (MODE == kModeWXYZ) {
            const double* h = reinterpret_cast<const double*>(hist);
            double* dst = L.psum + ((g << psh) + part) * (int64_t)K * Kp;
            for (int k = lane; k < K * Kp; k += 64) dst[k] = h[k];
        }
        if constexpr (MODE == kModeWSum || MODE == kModeTan) {
            const double* h = reinterpret_cast<const double*>(hist);
            constexpr int nc = TAN ? (int)TC : 16;
            constexpr int step = TAN ? (ALSO ? 3 : 2) * (int)TC : 16;
            const double sc = (TAN && sym) ? 2.0 : 1.0;
            for (int k = lane; k < K; k += 64) {
                double v = 0.0, tv = 0.0;
                for (int c = 0; c < nc; c++) {
                    v += h[k * step + ((c + lane) & (nc - 1))];
                    if (TAN) tv += h[k * step + nc + ((c + lane) & (nc - 1))];
                }
                const int64_t at_ = ((g << psh) + part) * K + k;
                if (L.psum) L.psum[at_] = sc * v;
                if (TAN) L.ptan[at_] = sc * tv;
            }
        }
        if constexpr (JK) {
            // sums of the lane points' rows by tag, one distinct tag at a time: lane
            // k adds up bin k of the points that carry it.  (A group of very many
            // tags leaves the loop and adds point by point.)
            const int tag = act ? (int)L.lane.w[(p0 + lane) * 2 + 1] : 0;
            uint64_t todo = (uint64_t)__ballot(act && tag >= 1 && tag <= L.nsamp);
            auto value = [&](int k, int j) __attribute__((always_inline)) -> double {
                if (VAR) return reinterpret_cast<const double*>(hist)[k * 64 + j];
                return (double)reinterpret_cast<const uint32_t*>(hist)[k * 64 + j];
            };
            for (int round = 0; round < 8 && todo; round++) {
                const int t = __builtin_amdgcn_readlane(tag, __builtin_ctzll(todo));
                const uint64_t mine = (uint64_t)__ballot(tag == t) & todo;
                todo &= ~mine;
                double* r = L.jacc + ((int64_t)m * (L.nsamp + 1) + t) * K;
                for (int k0 = 0; k0 < K; k0 += 64) {
                    const int k = k0 + lane;
                    double sum = 0.0;
                    for (int c = 0; c < 64; c++) {
                        const int j = (c + lane) & 63;  // a bank per lane
                        if (((mine >> j) & 1) && k < K) sum += value(k, j);
                    }
                    if (k < K && sum != 0.0) __hip_atomic_fetch_add(r + k, sum, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
            }
            if (todo && ((todo >> lane) & 1)) {
                double* r = L.jacc + ((int64_t)m * (L.nsamp + 1) + tag) * K;
                for (int k = 0; k < K; k++) {
                    const double v = VAR ? reinterpret_cast<const double*>(hist)[k * 64 + lane]
                                         : (double)reinterpret_cast<const uint32_t*>(hist)[k * 64 + lane];
                    if (v != 0.0) __hip_atomic_fetch_add(r + k, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
            }
        }
        if constexpr (MODE == kModeObj || MODE == kModeJac) {
            if (act) {
                // the lane point's row at its input position
                const int64_t q = __double_as_longlong(L.lane.x[(p0 + lane) * 4 + 3]);
                if constexpr (MODE == kModeObj) {
                    int64_t* r = L.orows + q * K;
                    int64_t sum = 0;
                    for (int k = 0; k < K; k++) {
                        sum += (int64_t)reinterpret_cast<const uint32_t*>(hist)[k * 64 + lane];
                        r[k] = sum;
                    }
                } else if (L.rows) {
                    double* r = L.rows + q * K;
                    for (int k = 0; k < K; k++) r[k] = reinterpret_cast<const double*>(hist)[k * 64 + lane];
                }
            }
            if constexpr (MODE == kModeJac && !SWAP) {
                if (L.corr && lane == 0) {
                    L.cflag[g] = tied ? 1u : 0u;
                    if (tied && L.seam) atomicOr(L.seam, 4);
                }
                if (L.psum) {
                    const double w = act ? LWT[lane] : 0.0;
                    for (int k = 0; k < K; k++) {
                        const double tot = wave_sum_f64(act ? w * reinterpret_cast<const double*>(hist)[k * 64 + lane] : 0.0);
                        if (lane == 0) L.psum[g * K + k] = tot;
                    }
                }
            }
        }
        if (L.pevals && lane == 0)
            __hip_atomic_fetch_add(reinterpret_cast<unsigned long long*>(L.pevals + g), (unsigned long long)evals,
                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __builtin_amdgcn_wave_barrier();
    }
}

template <int MODE, int VAR, int ALSO, int WAVES>
static int launch_tiles_w(const TileArgs& A, int64_t blocks, int smem, hipStream_t s) {
    hipLaunchKernelGGL((k_tiles<MODE, VAR, ALSO, WAVES>), dim3((unsigned)blocks), dim3(WAVES * 64), (size_t)smem, s, A);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

template <int MODE, int VAR, int ALSO>
static int launch_tiles_v(const TileArgs& A, int waves, int64_t blocks, int smem, hipStream_t s) {
    if (blocks <= 0) return 0;
    if (waves == 8) return launch_tiles_w<MODE, VAR, ALSO, 8>(A, blocks, smem, s);
    if (waves == 4) return launch_tiles_w<MODE, VAR, ALSO, 4>(A, blocks, smem, s);
    if (waves == 2) return launch_tiles_w<MODE, VAR, ALSO, 2>(A, blocks, smem, s);
    return launch_tiles_w<MODE, VAR, ALSO, 1>(A, blocks, smem, s);
}

// One launch of mode MODE; each mode is instantiated in its own translation
// unit (pairs_tile_*.hip).
template <int MODE>
int launch_tiles_mode(const TileArgs& A, int waves, int64_t blocks, int smem, int also, int var, hipStream_t s) {
    if constexpr (MODE == kModeWSum) {
        if (var == 2)
            return also ? launch_tiles_v<MODE, 2, 1>(A, waves, blocks, smem, s)
                        : launch_tiles_v<MODE, 2, 0>(A, waves, blocks, smem, s);
        if (var == 3)
            return also ? launch_tiles_v<MODE, 3, 1>(A, waves, blocks, smem, s)
                        : launch_tiles_v<MODE, 3, 0>(A, waves, blocks, smem, s);
    }
    if constexpr (MODE == kModeWSum || MODE == kModeJac) {
        if (var)
            return also ? launch_tiles_v<MODE, 1, 1>(A, waves, blocks, smem, s)
                        : launch_tiles_v<MODE, 1, 0>(A, waves, blocks, smem, s);
        return also ? launch_tiles_v<MODE, 0, 1>(A, waves, blocks, smem, s)
                    : launch_tiles_v<MODE, 0, 0>(A, waves, blocks, smem, s);
    } else if constexpr (MODE == kModeWXYZ) {
        if (var == 2) return launch_tiles_v<MODE, 2, 0>(A, waves, blocks, smem, s);
        if (var == 3) return launch_tiles_v<MODE, 3, 0>(A, waves, blocks, smem, s);
        return var ? launch_tiles_v<MODE, 1, 0>(A, waves, blocks, smem, s)
                   : launch_tiles_v<MODE, 0, 0>(A, waves, blocks, smem, s);
    } else if constexpr (MODE == kModeXYZ || MODE == kModeJack) {
        return var ? launch_tiles_v<MODE, 1, 0>(A, waves, blocks, smem, s)
                   : launch_tiles_v<MODE, 0, 0>(A, waves, blocks, smem, s);
    } else if constexpr (MODE == kModeTan) {
        return also ? launch_tiles_v<MODE, 0, 1>(A, waves, blocks, smem, s)
                    : launch_tiles_v<MODE, 0, 0>(A, waves, blocks, smem, s);
    } else {
        return launch_tiles_v<MODE, 0, 0>(A, waves, blocks, smem, s);
    }
}

}  // namespace hp
