// cellbuild.hip -- GPU cell-list build (replaces RectangularMesh,
// PC/rectangular_mesh.py:181-225, whose argsort + searchsorted bucket the
// points of each sample into a uniform grid).
//
// The build is a stable LSD counting sort of 32-bit cell keys (8-bit digits,
// tiles of 2048 or 8192 keys), so the order of points inside a cell is
// their input order and every downstream floating-point sum is run-to-run
// deterministic.  Two key flavours exist:
//   row-major  (ix*ny + iy)*nz + iz  -- stream side; the cells of one (ix, iy)
//              column are contiguous, so a column's z-range is one segment;
//   Hilbert    3-D Hilbert index    -- lane side; 64 consecutive points form a
//              spatially compact group (the curve has no jumps).
// Keys are local to a mock; the sort's tiles keep mocks apart, so one sort
// handles a whole batch of realisations with the key bits of one mock.
#include <cstdlib>
#include <cstring>

#include "hp_internal.h"

namespace hp {

// ----------------------------------------------------------------- utilities
struct ByteChunk {
    uint32_t* dst;
    uint32_t* clear;      // a word to set to zero, or null
    uint32_t nwords;
    uint32_t words[900];  // 3600 bytes of payload per launch (kernel arguments hold 4 KB)
};

__global__ void k_store_words(const ByteChunk c) {
    for (uint32_t i = threadIdx.x; i < c.nwords; i += blockDim.x) c.dst[i] = c.words[i];
    if (c.clear && threadIdx.x == 0) *c.clear = 0u;
}

int launch_store_bytes(void* dst, const void* src, size_t nbytes, uint32_t* clear, hipStream_t s) {
    // Carries a host blob into device memory through kernel arguments: no
    // memcpy API, so the upload is legal inside HIP-graph capture.
    const size_t nwords_total = (nbytes + 3) / 4;
    const uint8_t* bytes = static_cast<const uint8_t*>(src);
    for (size_t w0 = 0; w0 < nwords_total; w0 += 900) {
        ByteChunk c;
        const size_t nw = nwords_total - w0 < 900 ? nwords_total - w0 : 900;
        c.dst = static_cast<uint32_t*>(dst) + w0;
        c.nwords = static_cast<uint32_t>(nw);
        c.clear = w0 == 0 ? clear : nullptr;
        const size_t b0 = w0 * 4;
        const size_t nb = (b0 + nw * 4 <= nbytes) ? nw * 4 : nbytes - b0;
        std::memset(c.words, 0, sizeof(c.words));
        std::memcpy(c.words, bytes + b0, nb);
        hipLaunchKernelGGL(k_store_words, dim3(1), dim3(256), 0, s, c);
    }
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

__global__ void k_fill_u32(uint32_t* p, uint32_t v, int64_t n) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        p[i] = v;
}

int launch_fill_u32(uint32_t* p, uint32_t v, int64_t n, hipStream_t s) {
    if (n <= 0) return 0;
    int64_t blocks = (n + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    hipLaunchKernelGGL(k_fill_u32, dim3((unsigned)blocks), dim3(256), 0, s, p, v, n);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

__global__ void k_group_mock(const MockGeom* __restrict__ g, int nmocks, int side, int32_t* __restrict__ gm,
                             int64_t ngroups) {
    const int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (q >= ngroups) return;
    int lo = 0, hi = nmocks - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (g[mid].group_off[side] <= q) lo = mid; else hi = mid - 1;
    }
    gm[q] = lo;
}

int launch_group_mock(const MockGeom* g, int nmocks, int side, int32_t* gm, int64_t ngroups, hipStream_t s) {
    if (ngroups <= 0) return 0;
    hipLaunchKernelGGL(k_group_mock, dim3((unsigned)((ngroups + 255) / 256)), dim3(256), 0, s, g, nmocks, side,
                       gm, ngroups);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

// ----------------------------------------------------------------- cell keys
// Cell index of a coordinate: floor(v / cell), clamped into [0, n-1] so that
// v == period lands in the last cell (as PC/rectangular_mesh.py:19-22 does).
// The quotient is formed as v * (1 / cell): the pair kernels plan their
// windows with a safety margin, so the rounding of the quotient (a point
// within rounding of a cell face may land in the cell next to it) does not
// affect which pairs are counted.
__device__ __forceinline__ int cell_index(double v, double inv_cell, int n, bool& bad, double period, int pbc) {
    if (!(v == v) || v > 1.0e300 || v < -1.0e300) { bad = true; return 0; }
    if (pbc && (v < 0.0 || v > period)) bad = true;
    const double f = floor(v * inv_cell);
    if (!(f >= 0.0)) return 0;
    if (f >= (double)n) return n - 1;
    return (int)f;
}

// keys_row: when the same side is also sorted in row-major order, the
// Hilbert pass writes those keys too (one read of the coordinates for both).
// rows: the point's packed row (coordinates, and weights when they fit).
__global__ void k_keys(const MockGeom* __restrict__ geom, int nmocks, int side, int order,
                       const double* __restrict__ x, const double* __restrict__ y, const double* __restrict__ z,
                       int64_t n, uint32_t* __restrict__ keys, int32_t* __restrict__ status,
                       uint32_t* __restrict__ keys_row, const double* __restrict__ w, int nw, PackedRows rows,
                       int64_t xs) {
    const int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (p >= n) return;
    // the mock of the point: a wave's 64 consecutive points nearly always lie
    // in one mock, found by two wave-uniform searches (scalar loads); a wave
    // that straddles mocks searches per lane
    const int pf = __builtin_amdgcn_readfirstlane((int)p);
    const int64_t mf = mock_of_point(geom, nmocks, side, pf);
    const int64_t ml = mock_of_point(geom, nmocks, side, min((int64_t)pf + 63, n - 1));
    const int64_t m = (mf == ml) ? mf : mock_of_point(geom, nmocks, side, p);
    const MockGeom& G = geom[m];
    const double px = x[p * xs], py = y[p * xs], pz = z[p * xs];
    bool bad = false;
    const int ix = cell_index(px, G.inv_cell[0], G.ndiv[0], bad, G.period[0], G.pbc);
    const int iy = cell_index(py, G.inv_cell[1], G.ndiv[1], bad, G.period[1], G.pbc);
    const int iz = cell_index(pz, G.inv_cell[2], G.ndiv[2], bad, G.period[2], G.pbc);
    // keys are local to the mock: the sort keeps mocks apart by their tiles
    uint32_t key;
    const uint32_t rkey = (uint32_t)(((int64_t)ix * G.ndiv[1] + iy) * G.ndiv[2] + iz);
    if (order == kRowMajor) {
        key = rkey;
    } else {
        if (keys_row) keys_row[p] = rkey;
        // lane order: a power-of-two grid of 2^mbits cells per dimension, so the
        // Hilbert curve covers the box exactly (no passes through empty padding)
        const int hb = G.mbits;
        const int hn = 1 << hb;
        bool dummy = false;
        const int hx = cell_index(px, G.inv_hcell[0], hn, dummy, G.period[0], 0);
        const int hy = cell_index(py, G.inv_hcell[1], hn, dummy, G.period[1], 0);
        const int hz = cell_index(pz, G.inv_hcell[2], hn, dummy, G.period[2], 0);
        key = hilbert3((uint32_t)hx, (uint32_t)hy, (uint32_t)hz, hb);
    }
    keys[p] = key;
    if (rows.p) {
        // the row's fourth word: the Hilbert key (Hilbert order), which with the
        // point's index fixes its place in the stable Hilbert sort
        double* r = rows.p + p * rows.stride;
        const double slot = __hiloint2double(0, order == kRowMajor ? 0 : (int)key);
        reinterpret_cast<double4*>(r)[0] = make_double4(px, py, pz, slot);
        if (rows.nw > 0) {
            double4 wr = make_double4(0.0, 0.0, 0.0, 0.0);
            wr.x = w[p * nw];
            if (rows.nw > 1) wr.y = w[p * nw + 1];
            if (rows.nw > 2) wr.z = w[p * nw + 2];
            if (rows.nw > 3) wr.w = w[p * nw + 3];
            reinterpret_cast<double4*>(r)[1] = wr;
        }
    }
    if (bad && status) atomicOr(status, 1);
}

// ----------------------------------------------------- LSD counting sort
// Tiles of TILE keys: per-tile digit counts, an exclusive scan of each digit's
// counts over the tiles, then a scatter of every tile in digit order.  Large
// sorts take bigger tiles: the per-tile digit counts are read and written at
// 256 scattered words per tile, and a tile's keys leave in 256 runs, so 8192
// keys per tile (runs of ~32 keys, full cache lines) move a fraction of the
// bytes of 2048-key tiles (runs of ~8 keys) at tens of millions of points.
//
// Mocks are sorted side by side: the points of a mock are contiguous, its
// tiles never cross into the next mock (tile_first[m] = first tile of mock m,
// tile_first[nmocks] = tiles in all), and a mock's keys go to its own range of
// positions, so the keys only need the bits of the largest mock (one or two
// passes fewer than keys offset by mock for a batch of mocks).
struct TileSpan {
    int64_t start;  // first key of the tile
    int tn;         // keys in the tile
    int m;          // its mock
};

__device__ __forceinline__ TileSpan tile_span(const uint32_t* __restrict__ tile_first, const MockGeom* __restrict__ geom,
                                              int nmocks, int side, int t, int tile) {
    int lo = 0, hi = nmocks - 1;  // the last mock whose first tile is <= t (skips empty mocks)
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if ((int)tile_first[mid] <= t) lo = mid; else hi = mid - 1;
    }
    TileSpan r;
    r.m = lo;
    const int64_t k = (int64_t)(t - (int)tile_first[lo]) * tile;
    r.start = geom[lo].p_off[side] + k;
    r.tn = (int)min((int64_t)tile, geom[lo].n[side] - k);
    return r;
}

template <int TILE>
__global__ void __launch_bounds__(256) k_radix_hist(const uint32_t* __restrict__ keys, const MockGeom* __restrict__ geom,
                                                    const uint32_t* __restrict__ tile_first, int nmocks, int side,
                                                    int shift, uint32_t* __restrict__ tile_counts, int ntiles) {
    __shared__ uint32_t h[kRadixDigits];
    h[threadIdx.x] = 0;
    __syncthreads();
    const TileSpan ts = tile_span(tile_first, geom, nmocks, side, (int)blockIdx.x, TILE);
    if (ts.tn == TILE && (ts.start & 3) == 0) {
        // full, aligned tile: 16-byte loads
        const uint4* k4 = reinterpret_cast<const uint4*>(keys + ts.start);
        for (int i = threadIdx.x; i < TILE / 4; i += 256) {
            const uint4 k = k4[i];
            atomicAdd(&h[(k.x >> shift) & (kRadixDigits - 1)], 1u);
            atomicAdd(&h[(k.y >> shift) & (kRadixDigits - 1)], 1u);
            atomicAdd(&h[(k.z >> shift) & (kRadixDigits - 1)], 1u);
            atomicAdd(&h[(k.w >> shift) & (kRadixDigits - 1)], 1u);
        }
    } else {
        for (int i = threadIdx.x; i < ts.tn; i += 256)
            atomicAdd(&h[(keys[ts.start + i] >> shift) & (kRadixDigits - 1)], 1u);
    }
    __syncthreads();
    tile_counts[(int64_t)threadIdx.x * ntiles + blockIdx.x] = h[threadIdx.x];
}

// Exclusive scan of each digit's row of per-tile counts; row totals out.
__global__ void __launch_bounds__(256) k_radix_scan(uint32_t* __restrict__ tile_counts, int ntiles,
                                                    uint32_t* __restrict__ digit_totals) {
    __shared__ uint32_t part[256];
    uint32_t* row = tile_counts + (int64_t)blockIdx.x * ntiles;
    const int per = (ntiles + 255) / 256;
    const int b0 = threadIdx.x * per;
    const int b1 = min(b0 + per, ntiles);
    uint32_t sum = 0;
    for (int i = b0; i < b1; i++) sum += row[i];
    part[threadIdx.x] = sum;
    __syncthreads();
    // Hillis-Steele inclusive scan of 256 partial sums
    for (int off = 1; off < 256; off <<= 1) {
        uint32_t v = threadIdx.x >= off ? part[threadIdx.x - off] : 0;
        __syncthreads();
        part[threadIdx.x] += v;
        __syncthreads();
    }
    uint32_t run = threadIdx.x ? part[threadIdx.x - 1] : 0;
    for (int i = b0; i < b1; i++) {
        const uint32_t c = row[i];
        row[i] = run;
        run += c;
    }
    if (threadIdx.x == 255) digit_totals[blockIdx.x] = part[255];
}

// Inclusive Hillis-Steele scan of v over the first 256 threads of the block
// (every thread of the block calls it; threads >= 256 pass 0 and get 0).
template <int NT>
__device__ __forceinline__ uint32_t scan_digits(uint32_t* scan, uint32_t v) {
    const int d = threadIdx.x;
    if (d < kRadixDigits) scan[d] = v;
    __syncthreads();
    for (int off = 1; off < kRadixDigits; off <<= 1) {
        const uint32_t u = (d < kRadixDigits && d >= off) ? scan[d - off] : 0u;
        __syncthreads();
        if (d < kRadixDigits) scan[d] += u;
        __syncthreads();
    }
    return d < kRadixDigits ? scan[d] : 0u;
}

// One workgroup of WAVES wavefronts per tile of TILE keys.  Each wave ranks
// its TILE / WAVES keys stably (a lane's rank among lanes with the same digit
// comes from eight ballots; per-wave digit counters carry it across rounds),
// the tile is staged in LDS in digit order, and the staged keys go out in
// runs of equal digits, so consecutive threads write consecutive addresses.
// A mock's keys go to its own positions: position p_off[m] + (keys of the
// mock with smaller digits) + (keys of its earlier tiles with the same digit)
// + rank in the tile, all from the exclusive prefix G[d][t] of the digit
// counts over every tile.  The last row-major pass writes global cell ids
// (key + the mock's first cell) for the cell-start table.
template <int TILE, int WAVES>
__global__ void __launch_bounds__(WAVES * 64) k_radix_scatter(const uint32_t* __restrict__ kin,
                                                              const uint32_t* __restrict__ vin,
                                                              uint32_t* __restrict__ kout, uint32_t* __restrict__ vout,
                                                              const MockGeom* __restrict__ geom,
                                                              const uint32_t* __restrict__ tile_first, int nmocks,
                                                              int side, int shift, int add_cell_off,
                                                              const uint32_t* __restrict__ tile_counts,
                                                              const uint32_t* __restrict__ digit_totals, int ntiles) {
    constexpr int NT = WAVES * 64;
    constexpr int kPerWave = TILE / WAVES;
    constexpr int kRounds = kPerWave / 64;
    static_assert(NT >= kRadixDigits && kPerWave % 64 == 0, "tile shape");
    __shared__ uint32_t skey[TILE];
    __shared__ uint32_t sval[TILE];
    __shared__ uint32_t wcnt[WAVES][kRadixDigits];  // per-wave digit counts, then offsets
    __shared__ uint32_t toff[kRadixDigits];         // first staged position of each digit
    __shared__ uint32_t gbase[kRadixDigits];        // global position of the tile's first key per digit
    __shared__ uint32_t scan[kRadixDigits];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wv = tid >> 6;
    const int tile = blockIdx.x;
    const TileSpan ts = tile_span(tile_first, geom, nmocks, side, tile, TILE);
    const int64_t base = ts.start;
    const int tn = ts.tn;
    const uint32_t koff = add_cell_off ? (uint32_t)geom[ts.m].cell_off : 0u;

    for (int i = tid; i < WAVES * kRadixDigits; i += NT) (&wcnt[0][0])[i] = 0u;
    __syncthreads();

    // ---- stable ranks within each wave
    const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    uint32_t kk[kRounds], vv[kRounds], rk[kRounds];
#pragma unroll
    for (int r = 0; r < kRounds; r++) {
        const int li = wv * kPerWave + r * 64 + lane;  // position in the tile
        const bool valid = li < tn;
        const uint32_t key = valid ? kin[base + li] : 0u;
        const uint32_t val = valid ? (vin ? vin[base + li] : (uint32_t)(base + li)) : 0u;
        const uint32_t d = (key >> shift) & (kRadixDigits - 1);
        uint64_t peers = __ballot(valid);
#pragma unroll
        for (int bit = 0; bit < kRadixBits; bit++) {
            const bool on = (d >> bit) & 1u;
            const uint64_t bm = __ballot(on);
            peers &= on ? bm : ~bm;
        }
        const uint32_t before = (uint32_t)__popcll(peers & lt);
        const uint32_t cnt = valid ? wcnt[wv][d] : 0u;
        __builtin_amdgcn_wave_barrier();
        if (valid && before == 0) wcnt[wv][d] = cnt + (uint32_t)__popcll(peers);
        __builtin_amdgcn_wave_barrier();
        kk[r] = key;
        vv[r] = val;
        rk[r] = valid ? cnt + before : 0xffffffffu;
    }
    __syncthreads();

    // ---- digit offsets in the staged tile: digits in order, waves in order
    const int d = tid;  // the first 256 threads own one digit each
    uint32_t tot = 0;
    if (d < kRadixDigits)
        for (int w = 0; w < WAVES; w++) tot += wcnt[w][d];
    const uint32_t incl = scan_digits<NT>(scan, tot);
    if (d < kRadixDigits) {
        const uint32_t start = incl - tot;
        toff[d] = start;
        uint32_t run = start;
        for (int w = 0; w < WAVES; w++) {
            const uint32_t c = wcnt[w][d];
            wcnt[w][d] = run;
            run += c;
        }
    }
    // global base: the mock's first position, the mock's keys of smaller
    // digits (an exclusive scan of the mock's digit totals), then this digit's
    // keys of the mock's earlier tiles
    const int f0 = (int)tile_first[ts.m], f1 = (int)tile_first[ts.m + 1];
    uint32_t t = 0, g0 = 0;
    if (d < kRadixDigits) {
        const uint32_t* row = tile_counts + (int64_t)d * ntiles;
        g0 = row[f0];
        t = (f1 < ntiles ? row[f1] : digit_totals[d]) - g0;
    }
    __syncthreads();
    const uint32_t tincl = scan_digits<NT>(scan, t);
    if (d < kRadixDigits)
        gbase[d] = (uint32_t)geom[ts.m].p_off[side] + tincl - t + (tile_counts[(int64_t)d * ntiles + tile] - g0);
    __syncthreads();

    // ---- stage in digit order
#pragma unroll
    for (int r = 0; r < kRounds; r++) {
        if (rk[r] == 0xffffffffu) continue;
        const uint32_t dg = (kk[r] >> shift) & (kRadixDigits - 1);
        const uint32_t pos = wcnt[wv][dg] + rk[r];
        skey[pos] = kk[r];
        sval[pos] = vv[r];
    }
    __syncthreads();

    // ---- write out: runs of equal digits land on consecutive addresses
    for (int i = tid; i < tn; i += NT) {
        const uint32_t key = skey[i];
        const uint32_t dg = (key >> shift) & (kRadixDigits - 1);
        const uint32_t pos = gbase[dg] + (uint32_t)i - toff[dg];
        kout[pos] = key + koff;
        vout[pos] = sval[i];
    }
}

// Sorted copies in the new order: one 32-byte row per point (x, y, z and, with
// want_hkey, the point's Hilbert order key (Hilbert key << 32) | input index --
// the stable Hilbert sort orders the points of a mock by exactly this value --
// else zero), and the weight rows, read through each point's packed input row
// (x, y, z, the Hilbert key, and the weights when they fit in the row).
// With `keys` (the sorted global cell ids) the same pass writes the cell
// starts: cell_start[c] = first sorted position whose key >= c, for c in
// [0, total_cells]; thread q = n writes the trailing empty cells.
__global__ void k_gather(const uint32_t* __restrict__ perm, int64_t n, PackedRows rows, const double* __restrict__ w,
                         int nw, double* __restrict__ orow, double* __restrict__ ow, int want_hkey,
                         const uint32_t* __restrict__ keys, int64_t total_cells, uint32_t* __restrict__ cell_start) {
    const int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (q > n) return;
    if (keys) {
        const int64_t kcur = (q < n) ? (int64_t)keys[q] : total_cells;
        const int64_t kprev = (q > 0) ? (int64_t)keys[q - 1] : -1;
        for (int64_t c = kprev + 1; c <= kcur && c <= total_cells; c++) cell_start[c] = (uint32_t)q;
    }
    if (q == n) return;
    const int64_t p = perm[q];
    const double* r = rows.p + p * rows.stride;
    const double4 c = reinterpret_cast<const double4*>(r)[0];
    const uint64_t hk = want_hkey ? (((uint64_t)(uint32_t)__double2loint(c.w) << 32) | (uint64_t)(uint32_t)p) : 0ull;
    // bit copies (the order key is not a floating-point value)
    reinterpret_cast<ulonglong4*>(orow)[q] =
        make_ulonglong4((unsigned long long)__double_as_longlong(c.x), (unsigned long long)__double_as_longlong(c.y),
                        (unsigned long long)__double_as_longlong(c.z), (unsigned long long)hk);
    if (ow) {
        if (rows.nw > 0) {
            const double4 wr = reinterpret_cast<const double4*>(r)[1];
            ow[q * nw] = wr.x;
            if (nw > 1) ow[q * nw + 1] = wr.y;
            if (nw > 2) ow[q * nw + 2] = wr.z;
            if (nw > 3) ow[q * nw + 3] = wr.w;
        } else {
            for (int k = 0; k < nw; k++) ow[q * nw + k] = w[p * nw + k];
        }
    }
}

static inline int check(const char*) { return hipGetLastError() == hipSuccess ? 0 : -1; }

// Keys per counting-sort tile for a sort of n keys: 8192 from kSortLargeMin
// keys on (HALOPAIR_SORT_TILE=2048 or 8192 forces one size, for tests and
// measurements).
int sort_tile(int64_t n) {
    if (const char* e = std::getenv("HALOPAIR_SORT_TILE")) {
        const int v = std::atoi(e);
        if (v == kSortTile || v == kSortTileLarge) return v;
    }
    return n >= kSortLargeMin ? kSortTileLarge : kSortTile;
}

// The counting-sort passes of one order: keys from kin0 (or sb.keys[0]), the
// permutation into perm; returns the buffer that ends up with the sorted keys,
// or null on a bad tile shape.  counted: the first pass's digits are counted.
static uint32_t* sort_passes(const uint32_t* kin0, const MockGeom* geom, int nmocks, int side, int key_bits,
                             SortBufs sb, SortTiles st, uint32_t* perm, bool global_ids, hipStream_t s,
                             bool counted = false) {
    const int tile = st.tile, ntiles = st.ntiles;
    if ((tile != kSortTile && tile != kSortTileLarge) || ntiles <= 0) return nullptr;
    const int passes = key_bits <= 0 ? 1 : (key_bits + kRadixBits - 1) / kRadixBits;
    int cur = 0;
    for (int pass = 0; pass < passes; pass++) {
        const int shift = pass * kRadixBits;
        const uint32_t* kin = (pass == 0 && kin0) ? kin0 : sb.keys[cur];
        if (pass == 0 && counted) {
            // (k_curve_keys)
        } else if (tile == kSortTileLarge)
            hipLaunchKernelGGL(k_radix_hist<kSortTileLarge>, dim3(ntiles), dim3(256), 0, s, kin, geom, st.first,
                               nmocks, side, shift, sb.tile_counts, ntiles);
        else
            hipLaunchKernelGGL(k_radix_hist<kSortTile>, dim3(ntiles), dim3(256), 0, s, kin, geom, st.first, nmocks,
                               side, shift, sb.tile_counts, ntiles);
        hipLaunchKernelGGL(k_radix_scan, dim3(kRadixDigits), dim3(256), 0, s, sb.tile_counts, ntiles,
                           sb.digit_totals);
        // the last pass writes the permutation straight into perm, and (when
        // asked) the global cell ids for the cell-start table
        const bool last = pass == passes - 1;
        uint32_t* vdst = last ? perm : sb.vals[cur ^ 1];
        const uint32_t* vsrc = pass == 0 ? (const uint32_t*)nullptr : sb.vals[cur];
        const int add_off = (last && global_ids) ? 1 : 0;
        if (tile == kSortTileLarge)
            hipLaunchKernelGGL((k_radix_scatter<kSortTileLarge, 8>), dim3(ntiles), dim3(512), 0, s, kin, vsrc,
                               sb.keys[cur ^ 1], vdst, geom, st.first, nmocks, side, shift, add_off, sb.tile_counts,
                               sb.digit_totals, ntiles);
        else
            hipLaunchKernelGGL((k_radix_scatter<kSortTile, 4>), dim3(ntiles), dim3(256), 0, s, kin, vsrc,
                               sb.keys[cur ^ 1], vdst, geom, st.first, nmocks, side, shift, add_off, sb.tile_counts,
                               sb.digit_totals, ntiles);
        cur ^= 1;
    }
    return sb.keys[cur];
}

int build_sorted_side(const MockGeom* geom, int nmocks, int side, Order order, const double* x, const double* y,
                      const double* z, const double* w, int nw, int64_t n, int64_t total_cells, int key_bits,
                      SortBufs sb, SortTiles st, SortedSide out, int32_t* status, hipStream_t s, PackedRows rows,
                      bool want_hkey, uint32_t* keys_row_out, const uint32_t* keys_in, int64_t xs) {
    if (n <= 0) {
        if (order == kRowMajor) return launch_fill_u32(out.cell_start, 0u, total_cells + 1, s);
        return 0;
    }
    const unsigned nb = (unsigned)((n + 255) / 256);
    // keys_in: this order's keys were written by the other order's key pass
    if (!keys_in)
        hipLaunchKernelGGL(k_keys, dim3(nb), dim3(256), 0, s, geom, nmocks, side, (int)order, x, y, z, n, sb.keys[0],
                           status, order == kHilbert ? keys_row_out : (uint32_t*)nullptr, w, nw, rows, xs);
    const uint32_t* keys = sort_passes(keys_in, geom, nmocks, side, key_bits, sb, st, out.perm, order == kRowMajor, s);
    if (!keys) return -1;
    if (check("sort")) return -1;
    // The lane side (Hilbert order) is read once per group through the
    // permutation; only the stream side needs sorted copies.
    if (order == kRowMajor) {
        // the gather of the packed rows and the cell starts in one pass
        if (!rows.p) return -1;  // the row-major gather reads the packed rows
        hipLaunchKernelGGL(k_gather, dim3((unsigned)((n + 1 + 255) / 256)), dim3(256), 0, s, out.perm, n, rows, w,
                           nw, out.x, out.w, want_hkey ? 1 : 0, keys, total_cells, out.cell_start);
    }
    return check("gather");
}

// The curve-ordered rows of one side (see build_curve_side), and the rows of
// every cube that holds points: a cube of the 2^cbits grid is one stretch of the
// sorted keys, so the point at its start and the one at its end write its entry
// (the other entries were cleared).
__global__ void k_gather_curve(const uint32_t* __restrict__ perm, const uint32_t* __restrict__ keys, int64_t n,
                               const MockGeom* __restrict__ geom, int nmocks, int side, const double* __restrict__ x,
                               const double* __restrict__ y, const double* __restrict__ z, int64_t xs, PackedRows rows,
                               const double* __restrict__ w, int nw, double* __restrict__ orow,
                               double* __restrict__ ow, uint2* __restrict__ cubes) {
    const int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (q >= n) return;
    const int64_t p = perm[q];
    double px, py, pz;
    if (rows.p) {
        const double4 c = *reinterpret_cast<const double4*>(rows.p + p * rows.stride);
        px = c.x;
        py = c.y;
        pz = c.z;
    } else {
        px = x[p * xs];
        py = y[p * xs];
        pz = z[p * xs];
    }
    reinterpret_cast<double4*>(orow)[q] = make_double4(px, py, pz, __longlong_as_double((long long)p));
    if (ow)
        for (int k = 0; k < nw; k++) ow[q * nw + k] = w[p * nw + k];
    if (!cubes) return;
    const int qf = __builtin_amdgcn_readfirstlane((int)q);
    const int64_t mf = mock_of_point(geom, nmocks, side, qf);
    const int64_t ml = mock_of_point(geom, nmocks, side, min((int64_t)qf + 63, n - 1));
    const int64_t m = (mf == ml) ? mf : mock_of_point(geom, nmocks, side, q);
    const MockGeom& G = geom[m];
    const int sh = G.mbits - G.cbits;
    const uint32_t h = keys[q] >> (3 * sh);
    const int64_t q0 = G.p_off[side], q1 = q0 + G.n[side];
    const bool first = q == q0 || (keys[q - 1] >> (3 * sh)) != h;
    const bool last = q + 1 == q1 || (keys[q + 1] >> (3 * sh)) != h;
    if (!first && !last) return;
    bool bad = false;
    const int hn = 1 << G.mbits;
    const int cx = cell_index(px, G.inv_hcell[0], hn, bad, G.period[0], 0) >> sh;
    const int cy = cell_index(py, G.inv_hcell[1], hn, bad, G.period[1], 0) >> sh;
    const int cz = cell_index(pz, G.inv_hcell[2], hn, bad, G.period[2], 0) >> sh;
    uint2* c = cubes + G.cell_off + ((((int64_t)cx << G.cbits) + cy) << G.cbits) + cz;
    if (first) c->x = (uint32_t)q;
    if (last) c->y = (uint32_t)(q + 1);
}

// The Hilbert keys of one mock, the digit counts of the first pass and the
// clearing of what later kernels add into, in one launch: at 1M points the count
// and the two fills were 11 us and three launches of their own beside the keys'
// 16.  A workgroup takes one sort tile, two points a thread.
__global__ void __launch_bounds__(1024) k_curve_keys(const MockGeom* __restrict__ geom, const double* __restrict__ x,
                                                     const double* __restrict__ y, const double* __restrict__ z,
                                                     int64_t n, int64_t xs, uint32_t* __restrict__ keys,
                                                     int32_t* __restrict__ status, PackedRows rows,
                                                     uint32_t* __restrict__ tile_counts, uint32_t* __restrict__ cubes,
                                                     int64_t cube_words, uint32_t* __restrict__ clear,
                                                     int64_t clear_words) {
    __shared__ uint32_t h[kRadixDigits];
    const int64_t gt = blockIdx.x * (int64_t)1024 + threadIdx.x, gn = (int64_t)gridDim.x * 1024;
    for (int64_t i = gt; i < cube_words; i += gn) cubes[i] = 0u;
    for (int64_t i = gt; i < clear_words; i += gn) clear[i] = 0u;
    if (threadIdx.x < kRadixDigits) h[threadIdx.x] = 0u;
    __syncthreads();
    const MockGeom& G = geom[0];
    const int hb = G.mbits, hn = 1 << hb;
    bool bad = false;
#pragma unroll
    for (int r = 0; r < kSortTile / 1024; r++) {
        const int64_t p = blockIdx.x * (int64_t)kSortTile + r * 1024 + threadIdx.x;
        if (p >= n) break;
        const double px = x[p * xs], py = y[p * xs], pz = z[p * xs];
        cell_index(px, G.inv_cell[0], G.ndiv[0], bad, G.period[0], G.pbc);
        cell_index(py, G.inv_cell[1], G.ndiv[1], bad, G.period[1], G.pbc);
        cell_index(pz, G.inv_cell[2], G.ndiv[2], bad, G.period[2], G.pbc);
        bool dummy = false;
        const int hx = cell_index(px, G.inv_hcell[0], hn, dummy, G.period[0], 0);
        const int hy = cell_index(py, G.inv_hcell[1], hn, dummy, G.period[1], 0);
        const int hz = cell_index(pz, G.inv_hcell[2], hn, dummy, G.period[2], 0);
        const uint32_t key = hilbert3((uint32_t)hx, (uint32_t)hy, (uint32_t)hz, hb);
        keys[p] = key;
        atomicAdd(&h[key & (kRadixDigits - 1)], 1u);
        if (rows.p)
            *reinterpret_cast<double4*>(rows.p + p * rows.stride) = make_double4(px, py, pz, __hiloint2double(0, (int)key));
    }
    if (bad && status) atomicOr(status, 1);
    __syncthreads();
    if (threadIdx.x < kRadixDigits) tile_counts[(int64_t)threadIdx.x * gridDim.x + blockIdx.x] = h[threadIdx.x];
}

int build_curve_side(const MockGeom* geom, int nmocks, int side, const double* x, const double* y, const double* z,
                     const double* w, int nw, int64_t n, int64_t total_cells, int key_bits, SortBufs sb, SortTiles st,
                     SortedSide out, int32_t* status, hipStream_t s, PackedRows rows, int64_t xs, uint32_t* clear,
                     int64_t clear_words) {
    // (batches and the large tiles of tens of millions of points: the launches are nothing there)
    const bool fused = nmocks == 1 && st.tile == kSortTile && n > 0 && st.ntiles == (n + kSortTile - 1) / kSortTile;
    if (!fused && clear_words > 0 && launch_fill_u32(clear, 0u, clear_words, s)) return -1;
    if (!fused && out.cubes && launch_fill_u32(reinterpret_cast<uint32_t*>(out.cubes), 0u, 2 * total_cells, s)) return -1;
    if (n <= 0) return 0;
    const unsigned nb = (unsigned)((n + 255) / 256);
    if (fused)
        hipLaunchKernelGGL(k_curve_keys, dim3((unsigned)st.ntiles), dim3(1024), 0, s, geom, x, y, z, n, xs, sb.keys[0],
                           status, rows, sb.tile_counts, reinterpret_cast<uint32_t*>(out.cubes),
                           out.cubes ? 2 * total_cells : 0, clear, clear_words);
    else
        hipLaunchKernelGGL(k_keys, dim3(nb), dim3(256), 0, s, geom, nmocks, side, (int)kHilbert, x, y, z, n, sb.keys[0],
                           status, (uint32_t*)nullptr, (const double*)nullptr, 0, rows, xs);
    const uint32_t* keys = sort_passes(nullptr, geom, nmocks, side, key_bits, sb, st, out.perm, false, s, fused);
    if (!keys) return -1;
    hipLaunchKernelGGL(k_gather_curve, dim3(nb), dim3(256), 0, s, out.perm, keys, n, geom, nmocks, side, x, y, z, xs,
                       rows, w, nw, out.x, out.w, out.cubes);
    return check("curve");
}

// ------------------------------------------------------------ small builds
// A small request is bound by launches and their latency: three kernels build
// both sides (20k x 20k: 166 -> 64 us of kernels per call, of which the pair
// kernel is 25; the keys' workgroups have a thread per key, 10.4 -> 5.2 us against
// four keys a thread).  At most 128 tiles a side, so a workgroup adds up the digit
// counts of the tiles before its own itself (no scan launch), and the first
// pass counts the second pass's digits by atomics.
template <int TILE>
__global__ void __launch_bounds__(1024) k_small_keys(const SmallBuild B) {
    constexpr int NT = 1024;
    __shared__ uint32_t h[kSmallDigits];
    const SmallSide& S = B.s[blockIdx.y];
    const MockGeom& G = B.geom[0];
    const int tile = blockIdx.x, tiles = (S.n + TILE - 1) / TILE;
    // clear what later kernels add into: this side's cubes, the second pass's
    // counts, the caller's accumulators
    const int64_t gt = (int64_t)blockIdx.x * NT + threadIdx.x, gn = (int64_t)gridDim.x * NT;
    if (S.cubes)
        for (int64_t i = gt; i < B.total_cells; i += gn) S.cubes[i] = make_uint2(0x7fffffffu, 0u);
    for (int64_t i = gt; i < (int64_t)tiles * kSmallDigits; i += gn) S.counts[(int64_t)tiles * kSmallDigits + i] = 0u;
    if (blockIdx.y == 0)
        for (int64_t i = gt; i < B.clear_words; i += gn) B.clear[i] = 0u;
    if (tile >= tiles) return;
    for (int i = threadIdx.x; i < kSmallDigits; i += NT) h[i] = 0u;
    __syncthreads();
    const int hb = G.mbits, hn = 1 << hb;
    const int drop = max(3 * hb - 2 * kSmallBits, 0);  // a coarser curve beside a large sample's
    bool bad = false;
#pragma unroll
    for (int r = 0; r < TILE / NT; r++) {
        const int p = tile * TILE + r * NT + threadIdx.x;
        if (p >= S.n) break;
        const double v[3] = {S.x[p * S.xs], S.y[p * S.xs], S.z[p * S.xs]};
        uint32_t c[3];
        for (int d = 0; d < 3; d++) {
            bool dummy = false;
            if (!(v[d] == v[d]) || v[d] > 1.0e300 || v[d] < -1.0e300) bad = true;
            if (G.pbc && (v[d] < 0.0 || v[d] > G.period[d])) bad = true;
            c[d] = (uint32_t)cell_index(v[d], G.inv_hcell[d], hn, dummy, G.period[d], 0);
        }
        const uint32_t key = hilbert3(c[0], c[1], c[2], hb) >> drop;
        S.key0[p] = key;
        atomicAdd(&h[key & (kSmallDigits - 1)], 1u);
    }
    if (bad) atomicOr(B.status, 1);
    __syncthreads();
    for (int i = threadIdx.x; i < kSmallDigits; i += NT) S.counts[(int64_t)tile * kSmallDigits + i] = h[i];
}

// Exclusive sums over the workgroup's kSmallDigits threads.
__device__ __forceinline__ uint32_t small_scan(uint32_t v, uint32_t* tot) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    uint32_t inc = v;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t u = __shfl_up(inc, off);
        if (lane >= off) inc += u;
    }
    if (lane == 63) tot[wv] = inc;
    __syncthreads();
    uint32_t run = inc - v;
    for (int w = 0; w < kSmallDigits / 64; w++) run += w < wv ? tot[w] : 0u;
    return run;
}

// One stable pass over 9 bits; PASS 1 (the last) writes the points' rows and
// their cubes' first and last rows, from the tile staged in digit order: a
// tile's points of one cube follow each other there, and only its first and
// last one touch the cube's entry (two atomics for every point took most of the
// pass: 37 us at 60k + 240k points).
template <int PASS, int TILE>
__global__ void __launch_bounds__(kSmallDigits) k_small_scatter(const SmallBuild B) {
    constexpr int WAVES = kSmallDigits / 64, kRounds = TILE / WAVES / 64;
    __shared__ uint32_t wcnt[WAVES][kSmallDigits];
    __shared__ uint32_t tot[2][kSmallDigits / 64];
    __shared__ uint32_t skey[PASS ? TILE : 1], sval[PASS ? TILE : 1], sbase[PASS ? kSmallDigits : 1];
    const SmallSide& S = B.s[blockIdx.y];
    const int tile = blockIdx.x, tiles = (S.n + TILE - 1) / TILE;
    if (tile >= tiles) return;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int tn = min(TILE, S.n - tile * TILE);
    const uint32_t* kin = PASS ? S.key1 : S.key0;
    for (int w = 0; w < WAVES; w++) wcnt[w][tid] = 0u;
    // this digit's keys in earlier tiles, and in all
    const uint32_t* cnt = S.counts + (int64_t)PASS * tiles * kSmallDigits + tid;
    uint32_t before = 0, all = 0;
#pragma unroll 8
    for (int t = 0; t < tiles; t++) {
        const uint32_t c = cnt[(int64_t)t * kSmallDigits];
        before += t < tile ? c : 0u;
        all += c;
    }
    __syncthreads();
    const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    uint32_t kk[kRounds], rk[kRounds];
#pragma unroll
    for (int r = 0; r < kRounds; r++) {
        const int li = wv * (TILE / WAVES) + r * 64 + lane;
        const bool valid = li < tn;
        const uint32_t key = valid ? kin[tile * TILE + li] : 0u;
        const uint32_t d = key & (kSmallDigits - 1);
        uint64_t peers = __ballot(valid);
#pragma unroll
        for (int bit = 0; bit < kSmallBits; bit++) {
            const bool on = (d >> bit) & 1u;
            const uint64_t bm = __ballot(on);
            peers &= on ? bm : ~bm;
        }
        const uint32_t ahead = (uint32_t)__popcll(peers & lt);
        const uint32_t c = valid ? wcnt[wv][d] : 0u;
        __builtin_amdgcn_wave_barrier();
        if (valid && ahead == 0) wcnt[wv][d] = c + (uint32_t)__popcll(peers);
        __builtin_amdgcn_wave_barrier();
        kk[r] = key;
        rk[r] = c + ahead;
    }
    // the digit's first position, the tile's first one in it, then every wave's
    uint32_t run = small_scan(all, tot[0]) + before;
    uint32_t here = 0;
    for (int w = 0; w < WAVES; w++) here += wcnt[w][tid];
    if (PASS) {
        const uint32_t first = small_scan(here, tot[1]);
        sbase[tid] = run - first;  // from a staged place to its position
        run = first;
    }
    for (int w = 0; w < WAVES; w++) {
        const uint32_t c = wcnt[w][tid];
        wcnt[w][tid] = run;
        run += c;
    }
    __syncthreads();
    const MockGeom& G = B.geom[0];
#pragma unroll
    for (int r = 0; r < kRounds; r++) {
        const int li = wv * (TILE / WAVES) + r * 64 + lane;
        if (li >= tn) break;
        const uint32_t pos = wcnt[wv][kk[r] & (kSmallDigits - 1)] + rk[r];
        if (PASS == 0) {
            const uint32_t high = kk[r] >> kSmallBits;
            S.key1[pos] = high;
            S.val1[pos] = (uint32_t)(tile * TILE + li);
            atomicAdd(S.counts + ((int64_t)tiles + pos / TILE) * kSmallDigits + (high & (kSmallDigits - 1)), 1u);
        } else {
            skey[pos] = kk[r];
            sval[pos] = S.val1[tile * TILE + li];
        }
    }
    if (PASS == 0) return;
    __syncthreads();
    const int hn = 1 << G.mbits, sh = G.mbits - G.cbits;
    auto cube_of = [&](double x, double y, double z) {
        bool bad = false;
        const int cx = cell_index(x, G.inv_hcell[0], hn, bad, G.period[0], 0) >> sh;
        const int cy = cell_index(y, G.inv_hcell[1], hn, bad, G.period[1], 0) >> sh;
        const int cz = cell_index(z, G.inv_hcell[2], hn, bad, G.period[2], 0) >> sh;
        return (((cx << G.cbits) + cy) << G.cbits) + cz;
    };
#pragma unroll
    for (int r = 0; r < TILE / kSmallDigits; r++) {
        const int i = r * kSmallDigits + tid;
        const bool in = i < tn;
        const uint32_t pos = in ? sbase[skey[i] & (kSmallDigits - 1)] + (uint32_t)i : 0u;
        const int64_t p = in ? sval[i] : 0u;
        const double px = S.x[p * S.xs], py = S.y[p * S.xs], pz = S.z[p * S.xs];
        if (in) {
            reinterpret_cast<double4*>(S.row)[pos] = make_double4(px, py, pz, __longlong_as_double((long long)p));
            if (S.ow)
                for (int k = 0; k < B.nw; k++) S.ow[(int64_t)pos * B.nw + k] = S.w[p * B.nw + k];
        }
        if (S.cubes) {
            // (a wave's 64 staged points: their neighbours' cubes from the lanes beside them)
            const int c = in ? cube_of(px, py, pz) : -1;
            const int up = __shfl_up(c, 1), down = __shfl_down(c, 1);
            if (in) {
                if (lane == 0 || up != c) atomicMin(&S.cubes[c].x, pos);
                if (lane == 63 || down != c) atomicMax(&S.cubes[c].y, pos + 1u);
            }
        }
    }
}

int build_curve_small(const SmallBuild& b, int sides, hipStream_t s) {
    const int most = sides > 1 ? (b.s[0].n > b.s[1].n ? b.s[0].n : b.s[1].n) : b.s[0].n;
    const unsigned tiles = (unsigned)((most + b.tile - 1) / b.tile);
    // (at least a few workgroups for the clearing)
    const dim3 grid0(tiles < 16 ? 16 : tiles, sides), grid(tiles, sides);
    if (b.tile == 1024) {
        hipLaunchKernelGGL(k_small_keys<1024>, grid0, dim3(1024), 0, s, b);
        if (tiles == 0) return check("small");
        hipLaunchKernelGGL((k_small_scatter<0, 1024>), grid, dim3(kSmallDigits), 0, s, b);
        hipLaunchKernelGGL((k_small_scatter<1, 1024>), grid, dim3(kSmallDigits), 0, s, b);
    } else {
        hipLaunchKernelGGL(k_small_keys<2048>, grid0, dim3(1024), 0, s, b);
        if (tiles == 0) return check("small");
        hipLaunchKernelGGL((k_small_scatter<0, 2048>), grid, dim3(kSmallDigits), 0, s, b);
        hipLaunchKernelGGL((k_small_scatter<1, 2048>), grid, dim3(kSmallDigits), 0, s, b);
    }
    return check("small");
}

}  // namespace hp
