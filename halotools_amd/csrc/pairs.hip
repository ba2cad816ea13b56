// pairs.hip -- workgroup shape and LDS layout of the pair kernels, and the
// dispatch to the per-mode launchers.  The kernel itself is pairs_kernel.h.
#include <cstdlib>

#include "pairs_tile.h"

#ifndef HP_TILE_TAIL
#define HP_TILE_TAIL 8  // sixteenths of the resident waves whose groups go out in quarters at the end
#endif

namespace hp {

// instantiated in pairs_mode_*.hip
extern template int launch_mode<kModeCount3D>(const PairArgs&, int, int, int, int, hipStream_t);
extern template int launch_mode<kModeProj>(const PairArgs&, int, int, int, int, hipStream_t);
extern template int launch_mode<kModeXYZ>(const PairArgs&, int, int, int, int, hipStream_t);
extern template int launch_mode<kModeObj>(const PairArgs&, int, int, int, int, hipStream_t);
extern template int launch_mode<kModeWXYZ>(const PairArgs&, int, int, int, int, hipStream_t);
extern template int launch_mode<kModeJack>(const PairArgs&, int, int, int, int, hipStream_t);
extern template int launch_mode<kModeJackXY>(const PairArgs&, int, int, int, int, hipStream_t);
extern template int launch_mode<kModeWSum>(const PairArgs&, int, int, int, int, hipStream_t);
extern template int launch_mode<kModeJac>(const PairArgs&, int, int, int, int, hipStream_t);
extern template int launch_mode<kModeTan>(const PairArgs&, int, int, int, int, hipStream_t);

extern template int launch_tiles_mode<kModeCount3D>(const TileArgs&, int, int64_t, int, int, int, hipStream_t);
extern template int launch_tiles_mode<kModeProj>(const TileArgs&, int, int64_t, int, int, int, hipStream_t);
extern template int launch_tiles_mode<kModeXYZ>(const TileArgs&, int, int64_t, int, int, int, hipStream_t);
extern template int launch_tiles_mode<kModeWXYZ>(const TileArgs&, int, int64_t, int, int, int, hipStream_t);
extern template int launch_tiles_mode<kModeObj>(const TileArgs&, int, int64_t, int, int, int, hipStream_t);
extern template int launch_tiles_mode<kModeJack>(const TileArgs&, int, int64_t, int, int, int, hipStream_t);
extern template int launch_tiles_mode<kModeJac>(const TileArgs&, int, int64_t, int, int, int, hipStream_t);
extern template int launch_tiles_mode<kModeTan>(const TileArgs&, int, int64_t, int, int, int, hipStream_t);
extern template int launch_tiles_mode<kModeWSum>(const TileArgs&, int, int64_t, int, int, int, hipStream_t);

static int align16(int v) { return (v + 15) & ~15; }

// LDS layout of one wave's area for a launch that histograms kc radial / rp
// bins (plus the trash row); returns the bytes before the survivor ring.
static int wave_layout(const PairLaunch& L, int kc, int jslots, PairArgs& A) {
    const int Kp = L.bp.nbins;
    A.shared_count = 0;
    A.cnt_off = 0;
    A.jrow = 0;
    A.jr0_off = 0;
    switch (L.mode) {
        case kModeCount3D:
        case kModeProj:
            if (L.br.nbins > 64) { A.shared_count = 1; return (kc + 1) * 4; }
            return (kc + 1) * 32 * 4;  // rows shared by lanes l and l+32
        case kModeXYZ: return (kc + 1) * (Kp + 1) * 4;
        case kModeWXYZ: return kc * Kp * 8;  // only the cells pairs in range write
        case kModeJack:
        case kModeJackXY: {
            // row 0 plus one row per subsample tag the wave keeps in LDS
            A.jrow = (kc + 1) * (L.mode == kModeJackXY ? Kp + 1 : 1) * 8;
            int b = (jslots + 1) * A.jrow;
            if (L.mode == kModeJack) {
                // all-pairs rows in 16 lane columns for uniform-tag groups
                A.jr0_off = b;
                b += (kc + 1) * 16 * 8;
            }
            return b;
        }
        case kModeObj: return (kc + 1) * 64 * 4;
        case kModeJac:
            A.cnt_off = (kc + 1) * 64 * 8;
            return A.cnt_off + (L.also_count ? (kc + 1) * 64 * 4 : 0);
        case kModeWSum:  // rows shared by 4 lanes (16 columns), counts by 2 (32 columns)
            A.cnt_off = (kc + 1) * 16 * 8;
            return A.cnt_off + (L.also_count ? (kc + 1) * 32 * 4 : 0);
        case kModeTan:
            // per bin one block: W row, dW row (16 columns of 8 B each), then
            // the count row (32 columns of 4 B) when counts are wanted (the
            // kernel's kTanRow and kTanCnt)
            A.cnt_off = 256;
            return (kc + 1) * (L.also_count ? 384 : 256);
        default: return -1;
    }
}

// Jackknife: LDS rows for subsample tags, ~24 KB of table per wave.
static int jack_slots(const PairLaunch& L, int kc) {
    const int jrow = (kc + 1) * (L.mode == kModeJackXY ? L.bp.nbins + 1 : 1) * 8;
    return std::max(0, std::min(L.jslots, 24576 / jrow - 1));
}

static int num_compute_units() {
    static int n = 0;  // of the device, queried once
    if (n == 0) {
        int dev = 0, v = 0;
        if (hipGetDevice(&dev) == hipSuccess &&
            hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && v > 0)
            n = v;
        else
            n = 256;
    }
    return n;
}

// LDS layout of one wave of the matrix-core kernels: the stage, the weights of
// staged and lane points (and the lanes' z for (rp, pi) bins), the histogram.
static int tile_layout(int mode, int K, int Kp, int nw, int also, int var, bool many, TileArgs& A) {
    const bool xy = (mode == kModeXYZ || mode == kModeWXYZ || mode == kModeProj);
    A.lw_off = align16(deal_of(mode, var) == 64 ? Stage<64>::kTileBytes : Stage<128>::kTileBytes);
    A.ccol_sh = 0;
    A.hist_off = A.lw_off + nw * 512 + (xy ? 512 : 0);
    A.cnt_off = A.hist_off;
    int h = -1;
    switch (mode) {
        case kModeCount3D:
        case kModeProj: h = (K + 1) * 128; break;
        case kModeXYZ:
            // few cells (wp: one pi bin) in up to 32 columns, so that the lanes of
            // one LDS pass rarely meet on one cell; half the space where the launch
            // has more items than waves, which are then 16 a CU instead of 12 (wp
            // edges, 500k points: 750 -> 670 us; at 100k, two items a wave, 16 x 4
            // cells lose 219 -> 234)
            if (var) {
                while (A.ccol_sh < 5 && (K * Kp * 4 << (A.ccol_sh + 1)) <= 4096) A.ccol_sh++;
                h = K * Kp * 4 << A.ccol_sh;
            } else {
                while (A.ccol_sh < 5 && ((K + 1) * (Kp + 1) * 4 << (A.ccol_sh + 1)) <= (many ? 2048 : 4096)) A.ccol_sh++;
                h = (K + 1) * (Kp + 1) * 4 << A.ccol_sh;
            }
            break;
        case kModeWXYZ: h = K * Kp * 8; break;
        case kModeObj: h = (K + 1) * 256; break;
        case kModeJack: h = (K + 1) * (var ? 512 : 256); break;
        case kModeJac:
            h = (K + 1) * 512;
            if (also) { A.cnt_off = A.hist_off + h; h += (K + 1) * 128; }
            break;
        case kModeWSum:
            h = (K + 1) * 128;
            if (also) { A.cnt_off = A.hist_off + h; h += (K + 1) * 128; }
            break;
        case kModeTan:
            A.cnt_off = A.hist_off + 16 * (int)kTanCols;
            h = (K + 1) * (also ? 24 : 16) * (int)kTanCols;
            break;
        default: return -1;
    }
    A.wave_bytes = align16(A.hist_off + h);
    return A.wave_bytes;
}

// The kernel's VAR for a request (pairs_tile.h).
static int tile_var(int mode, int K, int Kp, int wfunc, int nw, int swap, int unit) {
    switch (mode) {
        case kModeXYZ: return K * Kp > 256 ? 1 : 0;  // cells in one column or two: their LDS bounds the waves
        case kModeWSum:
        // the number of weights compiled in where it is small: five rows of them cost
        // registers (sums of marks, id 2, of 400k points: 591 -> 406 us; (rp, pi) 1204 -> 787)
        case kModeWXYZ: return (wfunc == 1 && nw == 1) ? 1 : (nw == 2 ? 2 : (nw == 1 ? 3 : 0));
        case kModeJac: return swap;
        case kModeJack: return unit ? 0 : 1;
    }
    return 0;
}

int tile_wave_bytes(int mode, int K, int Kp, int nw, int also) {
    TileArgs A;
    if ((int64_t)K * std::max(Kp, 1) > 65536) return -1;
    return tile_layout(mode, K, Kp, nw, also, tile_var(mode, K, Kp, 0, nw, 0, 0), false, A);
}

// Matrix-core kernels: workgroup shape (the waves per workgroup that keep the
// most waves resident) and work items.
static int launch_tiles(const PairLaunch& L, int lds_per_block, hipStream_t s) {
    TileArgs A;
    A.L = L;
    A.tr = L.tr;
    A.tp = L.tp;
    const bool xy = (L.mode == kModeXYZ || L.mode == kModeWXYZ || L.mode == kModeProj);
    const int also = L.also_count ? 1 : 0;
    const int var = tile_var(L.mode, L.br.nbins, L.bp.nbins, L.wfunc, L.nw, L.swap, L.unit);
    const bool many = (L.ngroups << L.parts_sh) >= (int64_t)num_compute_units() * 32;
    if (tile_layout(L.mode, L.br.nbins, L.bp.nbins, L.nw, also, var, many, A) < 0) return -1;
    // tables of 2^n entries, the pi table at a multiple of its size
    A.tp_off = xy ? 8 * (int)std::max(L.tr.mask + 1, L.tp.mask + 1) : 0;
    A.tab_bytes = xy ? A.tp_off + 8 * ((int)L.tp.mask + 1) : 8 * ((int)L.tr.mask + 1);
    constexpr int kLdsPerCU = 160 * 1024, reg_waves = 4 * HP_TILE_WPS;
    // The shape with the most resident waves.  Four waves go one to each SIMD
    // and stay there; smaller workgroups spread unevenly (1M counts, 16 resident
    // waves of four: 740 us a call, 15 single ones: 820), so they have to gain a
    // ninth (per-object rows: 14 singles 1205, 12 in fours 1265; jackknife rows:
    // 13 singles 1635, 12 in fours 1605).  Of all modes at 1M and 200k points with
    // 20 radial or 16 x 41 bins, every shape forced, the choice is within 5 % of the
    // best one but for sums of two-weight marks (singles 1830, pairs 1685; 322, 300)
    // and 1M counts in one run (759, 706).
    int waves = 0, best = 0;
    double most = 0.0;
    for (const int w : {4, 8, 2, 1}) {
        if (L.waves > 0 && w != L.waves) continue;
        const int bytes = A.tab_bytes + w * A.wave_bytes;
        if (bytes > lds_per_block) continue;
        const int res = std::min(w * (kLdsPerCU / bytes), reg_waves);
        const double score = res * (w >= 4 ? 1.0 : (w == 2 ? 0.85 : 0.9));
        if (score > most) { most = score; best = res; waves = w; }
    }
    if (best == 0 && L.waves > 0) {
        PairLaunch M = L;
        M.waves = 0;  // the shape asked for does not fit: take the best one
        return launch_tiles(M, lds_per_block, s);
    }
    if (best == 0) return -2;
    A.parts_sh = L.parts_sh;
    A.tail_sh = L.parts_sh;
    A.tail = L.ngroups;
    const bool counts = (L.mode == kModeCount3D || L.mode == kModeProj || L.mode == kModeXYZ);
    if (counts && L.parts_sh < 2) {
        A.tail_sh = 2;
        A.tail = L.ngroups - std::min<int64_t>(L.ngroups, (int64_t)num_compute_units() * best * HP_TILE_TAIL / 16);
    }
    A.items = (A.tail << A.parts_sh) + ((L.ngroups - A.tail) << A.tail_sh);
    // chunks of at most 64 items, smaller where the launch has too few of them
    A.chunk_sh = 6;
    while (A.chunk_sh > 0 && (A.items >> (A.chunk_sh + 3)) < 4) A.chunk_sh--;
    const int64_t per_queue = ((A.items + (8 << A.chunk_sh) - 1) >> (A.chunk_sh + 3)) << A.chunk_sh;
    int64_t blocks = A.items > 0 ? 8 * ((per_queue + waves - 1) / waves) : 0;
    const int64_t resident = (int64_t)num_compute_units() * (best / waves) & ~(int64_t)7;
    A.queue = nullptr;
    A.taken = 0;
        // (the queues' lines cost more than they give where a wave has one or two items)
    if (L.queue && resident > 0 && blocks > 2 * resident) {
        blocks = resident;
        A.queue = L.queue;
        A.taken = (uint32_t)(blocks / 8 * waves);
    }
    const int smem = A.tab_bytes + waves * A.wave_bytes;
    switch (L.mode) {
        case kModeCount3D: return launch_tiles_mode<kModeCount3D>(A, waves, blocks, smem, also, var, s);
        case kModeProj: return launch_tiles_mode<kModeProj>(A, waves, blocks, smem, also, var, s);
        case kModeXYZ: return launch_tiles_mode<kModeXYZ>(A, waves, blocks, smem, also, var, s);
        case kModeWXYZ: return launch_tiles_mode<kModeWXYZ>(A, waves, blocks, smem, also, var, s);
        case kModeObj: return launch_tiles_mode<kModeObj>(A, waves, blocks, smem, also, var, s);
        case kModeJack: return launch_tiles_mode<kModeJack>(A, waves, blocks, smem, also, var, s);
        case kModeJac: return launch_tiles_mode<kModeJac>(A, waves, blocks, smem, also, var, s);
        case kModeTan: return launch_tiles_mode<kModeTan>(A, waves, blocks, smem, also, var, s);
        case kModeWSum: return launch_tiles_mode<kModeWSum>(A, waves, blocks, smem, also, var, s);
    }
    return -1;
}

int launch_pairs(const PairLaunch& L, hipStream_t s) {
    PairArgs A;
    A.L = L;
    const int Kr = L.br.nbins;
    if (L.br.nb > kTableMax || L.bp.nb > kTableMax) return -1;
    const bool xy = (L.mode == kModeXYZ || L.mode == kModeWXYZ || L.mode == kModeJackXY);
    A.tab_bytes = align16((int)sizeof(LdsEntry) * (L.br.nb + (xy ? L.bp.nb : 0)));
    // Workgroup shape: the number of waves per workgroup that keeps the most
    // waves resident per CU (160 KB of LDS; register-limited waves per CU as
    // the kernels' launch bounds hold them); on ties 4 waves, then 8 (4 was
    // never slower than 8 in measurements of every mode).
    constexpr int kLdsPerCU = 160 * 1024;
    static int lds_per_block = 0;  // the device's limit per workgroup (queried once)
    if (lds_per_block == 0) {
        int dev = 0, v = 0;
        if (hipGetDevice(&dev) == hipSuccess &&
            hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) == hipSuccess && v > 0)
            lds_per_block = std::min(v, kLdsPerCU);
        else
            lds_per_block = 64 * 1024;
    }
    const int kLdsPerBlock = lds_per_block;
    const int num_cus = num_compute_units();
    // the plan chose the kernels: their sorted copies differ
    if (L.tr.ok) return launch_tiles(L, kLdsPerBlock, s);
    // product marks (weight_func_id 1, one weight per point) have a compiled-in variant
    const int prod = (L.wfunc == 1 && L.nw == 1) ? 1 : 0;
    // waves per SIMD the kernels' registers allow (their launch bounds; the
    // per-lane-row Jacobian kernel is bounded by LDS long before registers)
    const int reg_waves =
        4 * (L.mode == kModeJac ? 6
                                : (((L.mode == kModeWSum || L.mode == kModeWXYZ) && prod) ? 5
                                   : ((L.mode == kModeWSum || L.mode == kModeTan || L.mode == kModeWXYZ ||
                                       L.mode == kModeJack || L.mode == kModeJackXY) ? 4
                                                                                     : (L.mode == kModeXYZ ? 5 : (L.mode == kModeObj ? 6 : HP_COUNT_WAVES)))));
    // shape for a launch of kc bins: sets A's layout, returns the waves per
    // workgroup (0 if nothing fits) and the resident waves per CU
    auto shape = [&](int kc, int* resident) -> int {
        const int wb = wave_layout(L, kc, jack_slots(L, kc), A);
        if (wb < 0) return 0;
        A.ring_off = align16(wb);
        A.wave_bytes = align16(A.ring_off + kRing * 4);
        int waves = 0, best = 0;
        for (const int w : {4, 8, 2, 1}) {
            if (L.waves > 0 && w != L.waves) continue;
            const int bytes = A.tab_bytes + w * A.wave_bytes;
            if (bytes > kLdsPerBlock) continue;
            const int res = std::min(w * (kLdsPerCU / bytes), reg_waves);
            if (res > best) { best = res; waves = w; }
        }
        *resident = best;
        return waves;
    };
    // Bins per launch: all of them when their histograms fit in LDS;
    // otherwise the largest share that keeps 4 waves per CU resident (fewer
    // if even one bin cannot), each launch histogramming its own range of
    // start bins over every pair (the pairs are evaluated once per launch).
    int res = 0;
    int kc = Kr;
    if (shape(Kr, &res) == 0) {
        int lo = 1, hi = Kr - 1, fit = 0;
        while (lo <= hi) {
            const int mid = (lo + hi) / 2;
            int r = 0;
            if (shape(mid, &r) != 0 && r >= std::min(4, reg_waves)) { fit = mid; lo = mid + 1; }
            else hi = mid - 1;
        }
        if (fit == 0) {
            lo = 1, hi = Kr - 1;
            while (lo <= hi) {
                const int mid = (lo + hi) / 2;
                int r = 0;
                if (shape(mid, &r) != 0) { fit = mid; lo = mid + 1; }
                else hi = mid - 1;
            }
        }
        if (fit == 0) return -2;
        kc = fit;
    }
    // launches over a range of the bins take the scanning lookup, which maps
    // start bins outside the range to the trash row
    const int multi = (L.br.multi || L.bp.multi || kc < Kr) ? 1 : 0;
    const int also = L.also_count ? 1 : 0;
    for (int k0 = 0; k0 < Kr; k0 += kc) {
        const int kn = std::min(kc, Kr - k0);
        const int waves = shape(kn, &res);
        if (waves == 0) return -2;
        A.L.jslots = jack_slots(L, kn);
        A.k0 = k0;
        A.kc = kn;
        A.smem = A.tab_bytes + waves * A.wave_bytes;
        A.L.pevals = k0 == 0 ? L.pevals : nullptr;  // every launch evaluates the same pairs
        A.grid = num_cus;  // persistent launches: times the workgroups one CU holds (launch_t)
        // below 2^32 by the largest batch of increments between two checks;
        // HALOPAIR_SHARED_FLUSH_AT lowers it (tests exercise the flush path)
        A.flush_at = 0xF0000000ull;
        if (const char* e = std::getenv("HALOPAIR_SHARED_FLUSH_AT")) {
            const unsigned long long v = std::strtoull(e, nullptr, 10);
            if (v > 0 && v < A.flush_at) A.flush_at = v;
        }
        int rc = -1;
        switch (L.mode) {
            case kModeCount3D: rc = launch_mode<kModeCount3D>(A, waves, multi, also, 0, s); break;
            case kModeProj: rc = launch_mode<kModeProj>(A, waves, multi, also, 0, s); break;
            case kModeXYZ: rc = launch_mode<kModeXYZ>(A, waves, multi, also, 0, s); break;
            case kModeObj: rc = launch_mode<kModeObj>(A, waves, multi, also, 0, s); break;
            case kModeWXYZ: rc = launch_mode<kModeWXYZ>(A, waves, multi, also, prod, s); break;
            case kModeJack: rc = launch_mode<kModeJack>(A, waves, multi, also, 0, s); break;
            case kModeJackXY: rc = launch_mode<kModeJackXY>(A, waves, multi, also, 0, s); break;
            case kModeWSum: rc = launch_mode<kModeWSum>(A, waves, multi, also, prod, s); break;
            case kModeJac: rc = launch_mode<kModeJac>(A, waves, multi, also, L.swap, s); break;
            case kModeTan: rc = launch_mode<kModeTan>(A, waves, multi, also, 0, s); break;
        }
        if (rc) return rc;
    }
    return 0;
}

}  // namespace hp
