// reduce.hip -- fixed-order reductions of per-group partial histograms into
// the reference's cumulative outputs, and the backward contraction.
//
// The reference sums per-process count vectors with np.sum(..., axis=0)
// (PC/npairs_3d.py:142-146) and returns cumulative counts N(<= r_k) because its
// engines walk the bins from the top down (PC/cpairs/npairs_3d_engine.pyx:178-182).
// Here each group contributed the histogram of the *first* bin a pair falls in;
// an inclusive prefix sum over bins (2-D for xy_z) turns it into the same
// cumulative counts.  All sums run in a fixed order, so results are
// run-to-run bitwise reproducible, including the FP64 marked sums.
#include "hp_internal.h"

namespace hp {

constexpr int kChunk = 512;  // groups per stage-1 block

template <typename T>
__global__ void __launch_bounds__(256) k_reduce_s1(const T* __restrict__ partial, int nb, const MockGeom* __restrict__ geom,
                                                   int side, int nchunk_max, T* __restrict__ s1, int psh) {
    __shared__ T sh[256];
    const int m = blockIdx.y, c = blockIdx.x;
    // 2^psh partial rows per lane group
    const int64_t go = geom[m].group_off[side] << psh, ng = geom[m].ngroups[side] << psh;
    const int64_t r0 = (int64_t)c * kChunk;
    const int64_t r1 = r0 + kChunk < ng ? r0 + kChunk : ng;
    T* out = s1 + ((int64_t)m * nchunk_max + c) * nb;
    const int nbt = nb < 256 ? nb : 256;
    const int rstride = 256 / nbt;
    for (int b0 = 0; b0 < nb; b0 += nbt) {
        const int t = threadIdx.x;
        const int b = b0 + t % nbt;
        const int rr = t / nbt;
        T acc = 0;
        if (rr < rstride && b < nb) {
            for (int64_t r = r0 + rr; r < r1; r += rstride) acc += partial[(go + r) * nb + b];
        }
        sh[t] = acc;
        __syncthreads();
        if (t < nbt && b0 + t < nb) {
            T tot = 0;
            for (int q = 0; q < rstride; q++) tot += sh[q * nbt + t];
            out[b0 + t] = tot;
        }
        __syncthreads();
    }
}

// Stage 2: per mock, sum the chunk rows in order, then the inclusive prefix.
// dims: nr (and np for the 2-D xy_z histogram; np = 0 means 1-D).
template <typename T, typename TO>
__global__ void __launch_bounds__(256) k_reduce_s2(const T* __restrict__ s1, int nr, int np, const MockGeom* __restrict__ geom,
                                                   int side, int nchunk_max, TO* __restrict__ out, int psh) {
    const int m = blockIdx.x;
    const int nb = np > 0 ? nr * np : nr;
    const int64_t ng = geom[m].ngroups[side] << psh;
    const int nchunks = (int)((ng + kChunk - 1) / kChunk);
    TO* o = out + (int64_t)m * nb;
    for (int b = threadIdx.x; b < nb; b += blockDim.x) {
        T tot = 0;
        for (int c = 0; c < nchunks; c++) tot += s1[((int64_t)m * nchunk_max + c) * nb + b];
        o[b] = (TO)tot;
    }
    __threadfence_block();
    __syncthreads();
    if (np <= 0) {
        if (threadIdx.x == 0) {
            TO run = 0;
            for (int k = 0; k < nr; k++) { run += o[k]; o[k] = run; }
        }
    } else {
        for (int k = threadIdx.x; k < nr; k += blockDim.x) {
            TO run = 0;
            for (int q = 0; q < np; q++) { run += o[k * np + q]; o[k * np + q] = run; }
        }
        __threadfence_block();
        __syncthreads();
        for (int q = threadIdx.x; q < np; q += blockDim.x) {
            TO run = 0;
            for (int k = 0; k < nr; k++) { run += o[k * np + q]; o[k * np + q] = run; }
        }
    }
}

// One running sum c[0], c[step], ... in the order of its terms, eight reads at a
// time (one after the other, each waits for the write before it).
template <typename T>
__device__ __forceinline__ void run_sum(T* c, int n, int step) {
    T run = (T)0;
    for (int i0 = 0; i0 < n; i0 += 8) {
        T v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = i0 + u < n ? c[(i0 + u) * step] : (T)0;
#pragma unroll
        for (int u = 0; u < 8; u++) {
            if (i0 + u >= n) break;
            run += v[u];
            c[(i0 + u) * step] = run;
        }
    }
}

// Cumulative sums of [nr][np] cells in LDS (np <= 0: of nr cells); the whole
// workgroup calls it.
template <typename T>
__device__ __forceinline__ void prefix_cells(T* c, int nr, int np) {
    if (np <= 0) {
        if (threadIdx.x == 0) run_sum(c, nr, 1);
    } else {
        for (int k = threadIdx.x; k < nr; k += blockDim.x) run_sum(c + k * np, np, 1);
        __syncthreads();
        for (int q = threadIdx.x; q < np; q += blockDim.x) run_sum(c + q, nr, np);
    }
    __syncthreads();
}

// Counts: the pair kernel accumulates each mock's histogram directly (exact
// integer atomics); this turns it into the reference's cumulative counts, in LDS
// where the cells fit it.
constexpr int kPrefixThreads = 1024;  // two or three replica loads per thread instead of nine (7.2 -> 4 us)
__global__ void __launch_bounds__(kPrefixThreads) k_prefix_counts(const uint64_t* __restrict__ acc, int nr, int np, int crep,
                                                       int64_t* __restrict__ out) {
    __shared__ uint64_t sh[kPrefixThreads];
    __shared__ int64_t cells[kPrefixThreads];
    const int m = blockIdx.x;
    const int nb = np > 0 ? nr * np : nr;
    const bool fits = nb <= kPrefixThreads;
    const uint64_t* a = acc + (int64_t)m * crep * nb;
    int64_t* o = out + (int64_t)m * nb;
    // replica sums: threads split over (bin, replica stripe), then the stripes
    // are added in LDS (integer sums: exact in any order)
    const int nbt = nb < kPrefixThreads ? nb : kPrefixThreads;
    const int rstride = kPrefixThreads / nbt;
    for (int b0 = 0; b0 < nb; b0 += nbt) {
        const int t = threadIdx.x;
        const int b = b0 + t % nbt;
        const int rr = t / nbt;
        uint64_t acc_t = 0;
        if (rr < rstride && b < nb)
            for (int r = rr; r < crep; r += rstride) acc_t += a[(int64_t)r * nb + b];
        sh[t] = acc_t;
        __syncthreads();
        if (t < nbt && b0 + t < nb) {
            uint64_t tot = 0;
            for (int q = 0; q < rstride; q++) tot += sh[q * nbt + t];
            (fits ? cells : o)[b0 + t] = (int64_t)tot;
        }
        __syncthreads();
    }
    if (fits) {
        prefix_cells(cells, nr, np);
        for (int b = threadIdx.x; b < nb; b += blockDim.x) o[b] = cells[b];
        return;
    }
    __threadfence_block();
    __syncthreads();
    if (np <= 0) {
        if (threadIdx.x == 0) {
            int64_t run = 0;
            for (int k = 0; k < nr; k++) { run += o[k]; o[k] = run; }
        }
    } else {
        for (int k = threadIdx.x; k < nr; k += blockDim.x) {
            int64_t run = 0;
            for (int q = 0; q < np; q++) { run += o[k * np + q]; o[k * np + q] = run; }
        }
        __threadfence_block();
        __syncthreads();
        for (int q = threadIdx.x; q < np; q += blockDim.x) {
            int64_t run = 0;
            for (int k = 0; k < nr; k++) { run += o[k * np + q]; o[k * np + q] = run; }
        }
    }
}

int launch_prefix_counts(const uint64_t* acc, int nr, int np, int nmocks, int crep, int64_t* counts, hipStream_t s) {
    hipLaunchKernelGGL(k_prefix_counts, dim3(nmocks), dim3(kPrefixThreads), 0, s, acc, nr, np, crep, counts);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

// Plain per-mock totals (no prefix): used for the candidate-evaluation counter.
__global__ void __launch_bounds__(256) k_reduce_plain(const uint64_t* __restrict__ s1, const MockGeom* __restrict__ geom,
                                                      int side, int nchunk_max, int64_t* __restrict__ out) {
    const int m = blockIdx.x;
    const int64_t ng = geom[m].ngroups[side];
    const int nchunks = (int)((ng + kChunk - 1) / kChunk);
    if (threadIdx.x == 0) {
        uint64_t tot = 0;
        for (int c = 0; c < nchunks; c++) tot += s1[(int64_t)m * nchunk_max + c];
        out[m] = (int64_t)tot;
    }
}

static int64_t nchunk_of(int64_t max_groups) { return (max_groups + kChunk - 1) / kChunk; }

// Wide histograms (the (rp, pi) cells of marked xy_z, hundreds of cells per
// group): stage 1 takes chunks of kChunkW groups, one cell per thread, so a
// launch has (groups / 64) x (cells / 256) blocks instead of groups / 512;
// stage 2 sums a mock's chunk rows in four fixed stripes per cell, then the
// stripes in order; the 2-D prefix runs once per mock.
constexpr int kChunkW = 64;
constexpr int kWideCells = 64;  // histograms above this many cells take the wide path
static int64_t nchunk_w(int64_t max_groups) { return (max_groups + kChunkW - 1) / kChunkW; }

__global__ void __launch_bounds__(256) k_reduce_w1(const double* __restrict__ partial, int nb,
                                                   const MockGeom* __restrict__ geom, int side, int nchunk_max,
                                                   double* __restrict__ s1, int psh) {
    const int m = blockIdx.y, c = blockIdx.x;
    const int b = blockIdx.z * 256 + threadIdx.x;
    const int64_t go = geom[m].group_off[side] << psh, ng = geom[m].ngroups[side] << psh;
    const int64_t r0 = (int64_t)c * kChunkW;
    if (b >= nb || r0 >= ng) return;
    const int64_t r1 = r0 + kChunkW < ng ? r0 + kChunkW : ng;
    double acc = 0.0;
    for (int64_t r = r0; r < r1; r++) acc += partial[(go + r) * nb + b];
    s1[((int64_t)m * nchunk_max + c) * nb + b] = acc;
}

__global__ void __launch_bounds__(256) k_reduce_w2(const double* __restrict__ s1, int nb,
                                                   const MockGeom* __restrict__ geom, int side, int nchunk_max,
                                                   double* __restrict__ out, int psh) {
    __shared__ double sh[4][64];
    const int m = blockIdx.y;
    const int bl = threadIdx.x & 63, stripe = threadIdx.x >> 6;
    const int b = blockIdx.x * 64 + bl;
    const int64_t ng = geom[m].ngroups[side] << psh;
    const int nchunks = (int)((ng + kChunkW - 1) / kChunkW);
    double acc = 0.0;
    if (b < nb)
        for (int c = stripe; c < nchunks; c += 4) acc += s1[((int64_t)m * nchunk_max + c) * nb + b];
    sh[stripe][bl] = acc;
    __syncthreads();
    if (stripe == 0 && b < nb) out[(int64_t)m * nb + b] = ((sh[0][bl] + sh[1][bl]) + sh[2][bl]) + sh[3][bl];
}

// inclusive 2-D prefix of each mock's [nr][np] sums (over pi, then over rp), in
// LDS where the cells fit it (16 x 41 cells in global memory: 13.5 us)
constexpr int kPrefixCells = 4096;
__global__ void __launch_bounds__(256) k_prefix_2d(double* __restrict__ out, int nr, int np) {
    __shared__ double cells[kPrefixCells];
    double* o = out + (int64_t)blockIdx.x * nr * np;
    const int nb = nr * np;
    if (nb <= kPrefixCells) {
        for (int b = threadIdx.x; b < nb; b += blockDim.x) cells[b] = o[b];
        __syncthreads();
        prefix_cells(cells, nr, np);
        for (int b = threadIdx.x; b < nb; b += blockDim.x) o[b] = cells[b];
        return;
    }
    for (int k = threadIdx.x; k < nr; k += blockDim.x) {
        double run = 0.0;
        for (int q = 0; q < np; q++) { run += o[k * np + q]; o[k * np + q] = run; }
    }
    __threadfence_block();
    __syncthreads();
    for (int q = threadIdx.x; q < np; q += blockDim.x) {
        double run = 0.0;
        for (int k = 0; k < nr; k++) { run += o[k * np + q]; o[k * np + q] = run; }
    }
}

int64_t reduce_scratch_elems(int64_t max_groups_per_mock, int nmocks, int nb) {
    const int64_t g = max_groups_per_mock > 0 ? max_groups_per_mock : 1;
    const int64_t nc = nb > kWideCells ? nchunk_w(g) : nchunk_of(g);
    return nc * nmocks * (int64_t)nb;
}

// FP64 partial histograms [groups << parts_sh][nr] (2-D: [...][nr * np]) -> cumulative sums per mock
int launch_reduce_sums_s(const double* partial, int nr, int np, const MockGeom* geom, int nmocks, int side,
                         int64_t max_groups, int parts_sh, double* scratch, double* sums, hipStream_t s) {
    const int nb = np > 0 ? nr * np : nr;
    max_groups <<= parts_sh;
    if (np > 0 && nb > kWideCells) {
        const int nc = (int)(nchunk_w(max_groups) > 0 ? nchunk_w(max_groups) : 1);
        hipLaunchKernelGGL(k_reduce_w1, dim3(nc, nmocks, (nb + 255) / 256), dim3(256), 0, s, partial, nb, geom, side,
                           nc, scratch, parts_sh);
        hipLaunchKernelGGL(k_reduce_w2, dim3((nb + 63) / 64, nmocks), dim3(256), 0, s, scratch, nb, geom, side, nc,
                           sums, parts_sh);
        hipLaunchKernelGGL(k_prefix_2d, dim3(nmocks), dim3(256), 0, s, sums, nr, np);
        return hipGetLastError() == hipSuccess ? 0 : -1;
    }
    const int nc = (int)(nchunk_of(max_groups) > 0 ? nchunk_of(max_groups) : 1);
    hipLaunchKernelGGL(k_reduce_s1<double>, dim3(nc, nmocks), dim3(256), 0, s, partial, nb, geom, side, nc, scratch, parts_sh);
    hipLaunchKernelGGL((k_reduce_s2<double, double>), dim3(nmocks), dim3(256), 0, s, scratch, nr, np, geom, side, nc,
                       sums, parts_sh);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int launch_reduce_evals_s(const uint64_t* pevals, const MockGeom* geom, int nmocks, int side, int64_t max_groups,
                          uint64_t* scratch, int64_t* evals, hipStream_t s) {
    const int nc = (int)(nchunk_of(max_groups) > 0 ? nchunk_of(max_groups) : 1);
    hipLaunchKernelGGL(k_reduce_s1<uint64_t>, dim3(nc, nmocks), dim3(256), 0, s, pevals, 1, geom, side, nc, scratch,
                       0);
    hipLaunchKernelGGL(k_reduce_plain, dim3(nmocks), dim3(64), 0, s, scratch, geom, side, nc, evals);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

// ------------------------------------------------------------- backward
constexpr int kDotMocks = 240;
struct DotArgs {
    const double* rows;
    const double* g;
    double* grad;
    int nr;
    int nm;           // mocks in this launch
    int m0;           // first mock of this launch (row of g)
    int64_t off[kDotMocks + 1];
};

// grad[p] = sum_s rows[p][s] * g[mock(p)][s], the contraction of the per-point
// Jacobian rows with the suffix-summed upstream gradient, terms in bin order.
// Bound by the read of nr doubles per point: a workgroup of one wave reads 64
// rows as one contiguous stretch into LDS (rows an odd number of doubles apart,
// so that a column's 64 reads hit all banks), kDotCols columns at a time; with
// one lane per row reading its own row (160-byte steps) 1M rows of 20 took 136
// us, 1.2 TB/s.
constexpr int kDotCols = 32;

__global__ void __launch_bounds__(64) k_rows_dot(const DotArgs a) {
    extern __shared__ double stage[];
    const int lane = threadIdx.x;
    const int64_t p0 = a.off[0] + blockIdx.x * (int64_t)64, p = p0 + lane;
    const int64_t left = a.off[a.nm] - p0;
    const int nrow = left < 64 ? (int)left : 64;
    int lo = 0, hi = a.nm - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (a.off[mid] <= p) lo = mid; else hi = mid - 1;
    }
    const double* g = a.g + (int64_t)(a.m0 + lo) * a.nr;
    const double* rows = a.rows + p0 * a.nr;
    double acc = 0.0;
    for (int s0 = 0; s0 < a.nr; s0 += kDotCols) {
        const int nc = min(kDotCols, a.nr - s0), pitch = nc | 1;
        const int total = nrow * nc, dr = 64 / nc, dc = 64 - dr * nc;
        int r = lane / nc, c = lane - r * nc;
        if (s0) __syncthreads();
#pragma unroll 8
        for (int e = lane; e < total; e += 64) {
            stage[r * pitch + c] = rows[(int64_t)r * a.nr + s0 + c];
            r += dr;
            c += dc;
            if (c >= nc) {
                c -= nc;
                r++;
            }
        }
        __syncthreads();
        if (lane < nrow)
            for (int s = 0; s < nc; s++) acc += stage[lane * pitch + s] * g[s0 + s];
    }
    if (lane < nrow) a.grad[p] = acc;
}

int launch_rows_dot(const double* rows, int nr, const double* gsuffix, const int64_t* offsets, int nmocks,
                    double* grad, hipStream_t s) {
    for (int m0 = 0; m0 < nmocks; m0 += kDotMocks) {
        DotArgs a;
        a.rows = rows;
        a.g = gsuffix;
        a.grad = grad;
        a.nr = nr;
        a.nm = nmocks - m0 < kDotMocks ? nmocks - m0 : kDotMocks;
        a.m0 = m0;
        for (int i = 0; i <= a.nm; i++) a.off[i] = offsets[m0 + i];
        const int64_t n = a.off[a.nm] - a.off[0];
        if (n <= 0) continue;
        const size_t lds = (size_t)64 * ((nr < kDotCols ? nr : kDotCols) | 1) * 8;
        hipLaunchKernelGGL(k_rows_dot, dim3((unsigned)((n + 63) / 64)), dim3(64), lds, s, a);
    }
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

// ---------------------------------------------------------------- segment sums
// out[m] = sum of values[off[m] .. off[m+1]) for every mock m, in a fixed
// order: stage 1 sums chunks of kSegChunk values (one block each: strided
// per-thread sums, then a tree), stage 2 adds each mock's chunk sums in
// chunk order with one wavefront.  No atomics, so results are bitwise
// reproducible.
constexpr int kSegMocks = 120;
constexpr int kSegChunk = 4096;
struct SegArgs {
    const double* v;
    double* part;     // chunk sums of this launch
    double* out;
    int nm;           // mocks in this launch
    int m0;
    int64_t off[kSegMocks + 1];   // point offsets
    int64_t cc[kSegMocks + 1];    // cumulative chunk counts (cc[0] = 0)
};

__global__ void __launch_bounds__(256) k_seg_chunks(const SegArgs a) {
    __shared__ double t[256];
    const int64_t c = blockIdx.x;
    int lo = 0, hi = a.nm - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (a.cc[mid] <= c) lo = mid; else hi = mid - 1;
    }
    const int64_t b = a.off[lo] + (c - a.cc[lo]) * kSegChunk;
    const int64_t e = min(b + (int64_t)kSegChunk, a.off[lo + 1]);
    double acc = 0.0;
    for (int64_t i = b + threadIdx.x; i < e; i += 256) acc += a.v[i];
    t[threadIdx.x] = acc;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) t[threadIdx.x] += t[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) a.part[c] = t[0];
}

__global__ void __launch_bounds__(64) k_seg_mocks(const SegArgs a) {
    const int m = blockIdx.x;
    const int lane = threadIdx.x;
    double acc = 0.0;
    for (int64_t c = a.cc[m] + lane; c < a.cc[m + 1]; c += 64) acc += a.part[c];
    for (int w = 32; w > 0; w >>= 1) acc += __shfl_xor(acc, w, 64);
    if (lane == 0) a.out[a.m0 + m] = acc;
}

int64_t segment_sum_scratch(const int64_t* offsets, int nmocks) {
    int64_t need = 1;
    for (int m0 = 0; m0 < nmocks; m0 += kSegMocks) {
        const int nm = nmocks - m0 < kSegMocks ? nmocks - m0 : kSegMocks;
        int64_t chunks = 0;
        for (int i = 0; i < nm; i++) chunks += (offsets[m0 + i + 1] - offsets[m0 + i] + kSegChunk - 1) / kSegChunk;
        need = chunks > need ? chunks : need;
    }
    return need;
}

int launch_segment_sum(const double* v, const int64_t* offsets, int nmocks, double* out, double* scratch,
                       hipStream_t s) {
    for (int m0 = 0; m0 < nmocks; m0 += kSegMocks) {
        SegArgs a;
        a.v = v;
        a.part = scratch;
        a.out = out;
        a.nm = nmocks - m0 < kSegMocks ? nmocks - m0 : kSegMocks;
        a.m0 = m0;
        a.cc[0] = 0;
        for (int i = 0; i <= a.nm; i++) a.off[i] = offsets[m0 + i];
        for (int i = 0; i < a.nm; i++) a.cc[i + 1] = a.cc[i] + (a.off[i + 1] - a.off[i] + kSegChunk - 1) / kSegChunk;
        if (a.cc[a.nm] > 0)
            hipLaunchKernelGGL(k_seg_chunks, dim3((unsigned)a.cc[a.nm]), dim3(256), 0, s, a);
        hipLaunchKernelGGL(k_seg_mocks, dim3((unsigned)a.nm), dim3(64), 0, s, a);
    }
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

__global__ void k_add_rows(const double* __restrict__ a, const double* __restrict__ b, double* __restrict__ out,
                           int64_t n) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        out[i] = a[i] + b[i];
}

int launch_add_rows(const double* a, const double* b, double* out, int64_t n, hipStream_t s) {
    if (n <= 0) return 0;
    int64_t blocks = (n + 255) / 256;
    if (blocks > 8192) blocks = 8192;
    hipLaunchKernelGGL(k_add_rows, dim3((unsigned)blocks), dim3(256), 0, s, a, b, out, n);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

// The sample-2 rows of an auto-count with one set of weights from the matrix-core
// pass: a lane group's rows1, with its corrections where it wrote any (corr in
// the lanes' order; a lane row's fourth word is the point's input position).  A
// wave per group; bound by the rows' one read and write (1M x 20: 320 MB).
__global__ void __launch_bounds__(256) k_seam_rows(const MockGeom* __restrict__ geom, const int32_t* __restrict__ group_mock,
                                                   int64_t ngroups, const double* __restrict__ lane_rows, int nr,
                                                   const double* __restrict__ rows1, const double* __restrict__ corr,
                                                   const uint32_t* __restrict__ cflag, double* __restrict__ rows2) {
    const int64_t g = blockIdx.x * (int64_t)4 + (threadIdx.x >> 6);
    if (g >= ngroups) return;
    const MockGeom& G = geom[group_mock ? group_mock[g] : 0];
    const int64_t gl = g - G.group_off[0], p0 = G.p_off[0] + gl * kGroup, left = G.n[0] - gl * kGroup;
    const int total = (int)(left < kGroup ? left : kGroup) * nr;
    const bool tied = cflag[g] != 0u;
    for (int e = threadIdx.x & 63; e < total; e += 64) {
        const int r = e / nr;
        const int64_t q = __double_as_longlong(lane_rows[(p0 + r) * 4 + 3]) * nr + (e - r * nr);
        rows2[q] = tied ? rows1[q] + corr[p0 * nr + e] : rows1[q];
    }
}

int launch_seam_rows(const MockGeom* geom, const int32_t* group_mock, int64_t ngroups, const double* lane_rows, int nr,
                     const double* rows1, const double* corr, const uint32_t* cflag, double* rows2, hipStream_t s) {
    if (ngroups <= 0) return 0;
    hipLaunchKernelGGL(k_seam_rows, dim3((unsigned)((ngroups + 3) / 4)), dim3(256), 0, s, geom, group_mock, ngroups,
                       lane_rows, nr, rows1, corr, cflag, rows2);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

// ------------------------------------------------------------ jackknife
// (w, tag) rows for the pair kernel: the weight (1 when none is given) and the
// subsample tag as a double (exact below 2^53).  Tags outside [1, nsamp] set
// status bit 2; the pair kernel never indexes a table with them.
__global__ void k_pack_jack(const double* __restrict__ w, const int32_t* __restrict__ tags, int64_t n, int nsamp,
                            double* __restrict__ out, int32_t* __restrict__ status) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const int32_t t = tags[i];
        if ((t < 1 || t > nsamp) && status) atomicOr(status, 2);
        out[2 * i] = w ? w[i] : 1.0;
        out[2 * i + 1] = (double)t;
    }
}

int launch_pack_jack(const double* w, const int32_t* tags, int64_t n, int nsamp, double* out, int32_t* status,
                     hipStream_t s) {
    if (n <= 0) return 0;
    int64_t blocks = (n + 255) / 256;
    if (blocks > 8192) blocks = 8192;
    hipLaunchKernelGGL(k_pack_jack, dim3((unsigned)blocks), dim3(256), 0, s, w, tags, n, nsamp, out, status);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

// Row 0 of each mock's table (zero until here) as the sum of its subsample rows
// (every point carries one tag): 8 strided sums per bin, then those in order.  A
// workgroup takes kTotalTags rows, a chain of 64 loads, and adds its sum to row 0
// (65536 rows in one workgroup's chains of 8192: 2300 us a call, now 330).
constexpr int kTotalTags = 512;

__global__ void __launch_bounds__(256) k_jack_total(double* __restrict__ acc, int nr, int nsamp) {
    __shared__ double sh[8][32];
    const int chunks = (nsamp - 1) / kTotalTags + 1, m = blockIdx.x / chunks;
    double* t = acc + (int64_t)m * ((int64_t)nsamp + 1) * nr;
    const int b = blockIdx.y * 32 + (threadIdx.x & 31), g = threadIdx.x >> 5;
    const int s0 = (blockIdx.x - m * chunks) * kTotalTags, left = min(kTotalTags, nsamp - s0);
    double sum = 0.0;
    if (b < nr)
        for (int i = 1 + g; i <= left; i += 8) sum += t[((int64_t)s0 + i) * nr + b];
    sh[g][threadIdx.x & 31] = sum;
    __syncthreads();
    if (g == 0 && b < nr) {
        for (int i = 1; i < 8; i++) sum += sh[i][threadIdx.x];
        if (chunks == 1)
            t[b] = sum;
        else
            __hip_atomic_fetch_add(t + b, sum, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// Inclusive prefix of every (mock, subsample) table row: over bins (1-D) or
// over pi then rp (2-D, the order of k_reduce_s2).
__global__ void __launch_bounds__(256) k_jack_prefix(double* __restrict__ acc, int nr, int np) {
    double* o = acc + (int64_t)blockIdx.x * (np > 0 ? nr * np : nr);
    if (np <= 0) {
        if (threadIdx.x == 0) {
            double run = 0.0;
            for (int k = 0; k < nr; k++) { run += o[k]; o[k] = run; }
        }
        return;
    }
    for (int k = threadIdx.x; k < nr; k += blockDim.x) {
        double run = 0.0;
        for (int q = 0; q < np; q++) { run += o[k * np + q]; o[k * np + q] = run; }
    }
    __threadfence_block();
    __syncthreads();
    for (int q = threadIdx.x; q < np; q += blockDim.x) {
        double run = 0.0;
        for (int k = 0; k < nr; k++) { run += o[k * np + q]; o[k * np + q] = run; }
    }
}

// out[m][0] = all pairs; out[m][s] = all pairs - weight lost without subsample s.
__global__ void k_jack_out(const double* __restrict__ acc, int64_t nb, int nsamp, int64_t total,
                           double* __restrict__ out) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t b = i % nb;
        const int64_t row = i / nb;
        const int64_t sub = row % (nsamp + 1);
        const double h = acc[(row - sub) * nb + b];
        out[i] = sub == 0 ? h : h - acc[i];
    }
}

int launch_jack_finish(double* acc, int nr, int np, int nmocks, int nsamp, bool total, double* out, hipStream_t s) {
    if (total)
        hipLaunchKernelGGL(k_jack_total, dim3((unsigned)nmocks * (unsigned)((nsamp - 1) / kTotalTags + 1), (nr + 31) / 32),
                           dim3(256), 0, s, acc, nr, nsamp);
    const int64_t rows = (int64_t)nmocks * (nsamp + 1);
    const int64_t nb = np > 0 ? (int64_t)nr * np : nr;
    hipLaunchKernelGGL(k_jack_prefix, dim3((unsigned)rows), dim3(np > 0 ? 256 : 64), 0, s, acc, nr, np);
    const int64_t cells = rows * nb;
    int64_t blocks = (cells + 255) / 256;
    if (blocks > 8192) blocks = 8192;
    hipLaunchKernelGGL(k_jack_out, dim3((unsigned)blocks), dim3(256), 0, s, acc, nb, nsamp, cells, out);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

// ------------------------------------------------------- enclosing box
// The smallest and largest coordinate of two unperiodic samples, and both
// samples shifted by the smallest (PC/mesh_helpers.py:17-64): a pass over the
// points for the extremes of each workgroup's share and a pass that writes the
// shifted (x, y, z) rows.  Bound by its two launches up to ~1e6 points (60k +
// 240k points: 7 + 6 us, where a min, a max and a subtraction per column and
// sample were 33 kernels and 250 us a call).  A NaN stays (comparisons with it
// are false, so it is taken explicitly), as in the library's min and max.
constexpr int kBoxBlocks = 256;

struct BoxArgs {
    const double* c[2][3];
    int64_t st[2], n[2];
    double* rows[2];      // null: the second sample is the first
    double2* part;        // kBoxBlocks (smallest, largest)
    double* lohi;
};

__device__ __forceinline__ void box_take(double2& e, double v) {
    e.x = (v < e.x || v != v) ? v : e.x;
    e.y = (v > e.y || v != v) ? v : e.y;
}

// over the workgroup; every thread gets the result
__device__ __forceinline__ double2 box_reduce(double2 e, double2* t) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const double lo = __shfl_xor(e.x, off), hi = __shfl_xor(e.y, off);
        e.x = (lo < e.x || lo != lo) ? lo : e.x;
        e.y = (hi > e.y || hi != hi) ? hi : e.y;
    }
    const int nw = blockDim.x >> 6;
    if ((threadIdx.x & 63) == 0) t[threadIdx.x >> 6] = e;
    __syncthreads();
    e = t[0];
    for (int w = 1; w < nw; w++) {
        const double2 o = t[w];
        e.x = (o.x < e.x || o.x != o.x) ? o.x : e.x;
        e.y = (o.y > e.y || o.y != o.y) ? o.y : e.y;
    }
    return e;
}

__global__ void __launch_bounds__(1024) k_box_extremes(const BoxArgs a) {
    __shared__ double2 t[16];
    double2 e = make_double2(INFINITY, -INFINITY);
    const int64_t step = (int64_t)gridDim.x * blockDim.x;
    for (int sd = 0; sd < 2; sd++) {
        if (!a.rows[sd]) continue;
        for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < a.n[sd]; i += step) {
            const int64_t o = i * a.st[sd];
            const double x = a.c[sd][0][o], y = a.c[sd][1][o], z = a.c[sd][2][o];
            box_take(e, x);
            box_take(e, y);
            box_take(e, z);
        }
    }
    e = box_reduce(e, t);
    if (threadIdx.x == 0) a.part[blockIdx.x] = e;
}

__global__ void __launch_bounds__(kBoxBlocks) k_box_shift(const BoxArgs a, int parts) {
    __shared__ double2 t[kBoxBlocks / 64];
    double2 e = threadIdx.x < (unsigned)parts ? a.part[threadIdx.x] : make_double2(INFINITY, -INFINITY);
    e = box_reduce(e, t);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        a.lohi[0] = e.x;
        a.lohi[1] = e.y;
    }
    const int64_t step = (int64_t)gridDim.x * blockDim.x;
    for (int sd = 0; sd < 2; sd++) {
        if (!a.rows[sd]) continue;
        for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < a.n[sd]; i += step) {
            const int64_t o = i * a.st[sd];
            const double x = a.c[sd][0][o], y = a.c[sd][1][o], z = a.c[sd][2][o];
            a.rows[sd][3 * i] = x - e.x;
            a.rows[sd][3 * i + 1] = y - e.x;
            a.rows[sd][3 * i + 2] = z - e.x;
        }
    }
}

int launch_enclose(const double* const* c1, int64_t st1, int64_t n1, const double* const* c2, int64_t st2, int64_t n2,
                   double* rows1, double* rows2, double* lohi, double* scratch, hipStream_t s) {
    BoxArgs a;
    for (int d = 0; d < 3; d++) {
        a.c[0][d] = c1[d];
        a.c[1][d] = c2[d];
    }
    a.st[0] = st1;
    a.st[1] = st2;
    a.n[0] = n1;
    a.n[1] = n2;
    a.rows[0] = rows1;
    a.rows[1] = rows2;
    a.part = reinterpret_cast<double2*>(scratch);
    a.lohi = lohi;
    const int64_t most = rows2 && n2 > n1 ? n2 : n1;
    int64_t nb = (most + 1023) / 1024, nbs = (most + kBoxBlocks - 1) / kBoxBlocks;
    if (nb > kBoxBlocks) nb = kBoxBlocks;
    if (nbs > 2048) nbs = 2048;
    hipLaunchKernelGGL(k_box_extremes, dim3((unsigned)nb), dim3(1024), 0, s, a);
    hipLaunchKernelGGL(k_box_shift, dim3((unsigned)nbs), dim3(kBoxBlocks), 0, s, a, (int)nb);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int64_t enclose_scratch() { return 2 * kBoxBlocks; }

// ------------------------------------------------------- subsample tags
// Smallest and largest tag of one or two samples and how many of the tags 1 ..
// nsamp do not occur.  One pass (1M tags: 6 us) with a bitmap of the tags per
// workgroup, one workgroup that joins them, and one copy back, where a min, a
// max and a histogram of their own were 100 us of kernels and seven waits for
// the device (350 us a call).
constexpr int kTagBlocks = 256, kTagMax = 1 << 16;

struct TagArgs {
    const int64_t* t[2];
    int64_t n[2];
    int nsamp, words;     // 64-bit words of a bitmap
    int64_t* part;        // per side and workgroup: smallest, largest, bitmap
    int64_t* out;         // per side: smallest, largest, missing
};

__device__ __forceinline__ void tag_minmax(int64_t& lo, int64_t& hi, int64_t* t) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const int64_t l = __shfl_xor(lo, off), h = __shfl_xor(hi, off);
        lo = l < lo ? l : lo;
        hi = h > hi ? h : hi;
    }
    if ((threadIdx.x & 63) == 0) {
        t[2 * (threadIdx.x >> 6)] = lo;
        t[2 * (threadIdx.x >> 6) + 1] = hi;
    }
    __syncthreads();
    for (int w = 0; w < (int)(blockDim.x >> 6); w++) {
        lo = t[2 * w] < lo ? t[2 * w] : lo;
        hi = t[2 * w + 1] > hi ? t[2 * w + 1] : hi;
    }
}

__global__ void __launch_bounds__(1024) k_tag_parts(const TagArgs a) {
    extern __shared__ unsigned long long bits[];
    __shared__ int64_t t[32];
    const int sd = blockIdx.y;
    for (int w = threadIdx.x; w < a.words; w += blockDim.x) bits[w] = 0ull;
    __syncthreads();
    int64_t lo = INT64_MAX, hi = INT64_MIN;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < a.n[sd]; i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t v = a.t[sd][i];
        lo = v < lo ? v : lo;
        hi = v > hi ? v : hi;
        if (v >= 1 && v <= a.nsamp) {
            const unsigned long long bit = 1ull << ((v - 1) & 63);
            // (most tags are known after a few points: look first)
            if (!(*(volatile unsigned long long*)&bits[(v - 1) >> 6] & bit)) atomicOr(&bits[(v - 1) >> 6], bit);
        }
    }
    tag_minmax(lo, hi, t);
    int64_t* p = a.part + ((int64_t)sd * kTagBlocks + blockIdx.x) * (2 + a.words);
    if (threadIdx.x == 0) {
        p[0] = lo;
        p[1] = hi;
    }
    for (int w = threadIdx.x; w < a.words; w += blockDim.x) p[2 + w] = (int64_t)bits[w];
}

__global__ void __launch_bounds__(1024) k_tag_join(const TagArgs a, int blocks) {
    extern __shared__ unsigned long long bits[];
    __shared__ int64_t t[32];
    __shared__ int seen;
    const int sd = blockIdx.x;
    const int64_t* part = a.part + (int64_t)sd * kTagBlocks * (2 + a.words);
    if (threadIdx.x == 0) seen = 0;
    for (int w = threadIdx.x; w < a.words; w += 1024) bits[w] = 0ull;
    __syncthreads();
    int64_t lo = INT64_MAX, hi = INT64_MIN;
    for (int b = threadIdx.x; b < blocks; b += 1024) {
        const int64_t* p = part + (int64_t)b * (2 + a.words);
        lo = p[0] < lo ? p[0] : lo;
        hi = p[1] > hi ? p[1] : hi;
    }
    // (eight loads in flight: one by one in 256 threads, a call on 1M tags of 65536 took 424 us, now 109)
    const int cells = blocks * a.words;
    for (int i0 = threadIdx.x; i0 < cells; i0 += 8 * 1024) {
        unsigned long long v[8];
        int w[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const int i = i0 + u * 1024, b = i / a.words;
            w[u] = i - b * a.words;
            v[u] = i < cells ? (unsigned long long)part[(int64_t)b * (2 + a.words) + 2 + w[u]] : 0ull;
        }
#pragma unroll
        for (int u = 0; u < 8; u++)
            if (v[u]) atomicOr(&bits[w[u]], v[u]);
    }
    tag_minmax(lo, hi, t);  // (waits for the bitmap too)
    for (int w = threadIdx.x; w < a.words; w += 1024) atomicAdd(&seen, __popcll(bits[w]));
    __syncthreads();
    if (threadIdx.x == 0) {
        a.out[3 * sd] = lo;
        a.out[3 * sd + 1] = hi;
        a.out[3 * sd + 2] = a.nsamp - seen;
    }
}

int64_t tag_scratch(int nsamp) { return nsamp < 1 || nsamp > kTagMax ? -1 : 2 * kTagBlocks * (2 + (nsamp + 63) / 64); }

int launch_tag_stats(const int64_t* t1, int64_t n1, const int64_t* t2, int64_t n2, int nsamp, int64_t* out,
                     int64_t* scratch, hipStream_t s) {
    TagArgs a;
    a.t[0] = t1;
    a.t[1] = t2;
    a.n[0] = n1;
    a.n[1] = n2;
    a.nsamp = nsamp;
    a.words = (nsamp + 63) / 64;
    a.part = scratch;
    a.out = out;
    const int sides = t2 ? 2 : 1;
    const int64_t most = t2 && n2 > n1 ? n2 : n1;
    int64_t nb = (most + 1023) / 1024;
    if (nb > kTagBlocks) nb = kTagBlocks;
    const size_t lds = (size_t)a.words * 8;
    hipLaunchKernelGGL(k_tag_parts, dim3((unsigned)nb, sides), dim3(1024), lds, s, a);
    hipLaunchKernelGGL(k_tag_join, dim3(sides), dim3(1024), lds, s, a, (int)nb);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

// Zheng07 central occupation of each point and its derivative with respect to
// logMmin (empirical_models/occupation_models/zheng07_components.py:149-153):
// u = (log_mass - logMmin[mock]) / sigma, w = 0.5 * (1 + erf(u)),
// dw = -exp(-u * u) / (sqrt(pi) * sigma), written as (w, dw) rows: the weights
// and tangents of the batched forward-mode step, in one pass over the points
// (the divisions by the host constants are multiplications by their
// reciprocals, as torch evaluates a tensor divided by a Python float).
__global__ void k_zheng07_tangent(const double* __restrict__ logm, const int64_t* __restrict__ mock_id,
                                  const double* __restrict__ logMmin, double inv_sigma, double inv_dnorm, int64_t n,
                                  double2* __restrict__ wt) {
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double u = (logm[i] - logMmin[mock_id[i]]) * inv_sigma;
    const double w = 0.5 * (1.0 + erf(u));
    const double dw = -exp(-(u * u)) * inv_dnorm;
    wt[i] = make_double2(w, dw);
}

int launch_zheng07_tangent(const double* logm, const int64_t* mock_id, const double* logMmin, double sigma,
                           int64_t n, double* wt, hipStream_t s) {
    if (n <= 0) return 0;
    const double inv_sigma = 1.0 / sigma, inv_dnorm = 1.0 / (sqrt(M_PI) * sigma);
    hipLaunchKernelGGL(k_zheng07_tangent, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, logm, mock_id, logMmin,
                       inv_sigma, inv_dnorm, n, reinterpret_cast<double2*>(wt));
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace hp
