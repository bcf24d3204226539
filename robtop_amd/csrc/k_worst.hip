// Worst-case load search (modified power method) on the finest level: random
// start force, projection of a nodal field onto the admissible loads, and the
// unit normalisation / force-change reductions of each step.
//
// Load nodes are a compact list of slots; the projected force lives in a
// compact SoA array fs[3][nl] and is scattered into the full force vector,
// which is zero away from the load nodes.
#include "rt_internal.h"

namespace rt {

__device__ __forceinline__ double blk_sum_w(double v) {
    __shared__ double red[16];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    __syncthreads();
    if (lane == 0) red[wid] = v;
    __syncthreads();
    double t = 0;
    if (threadIdx.x == 0) {
        const int nw = (blockDim.x + 63) >> 6;
        for (int i = 0; i < nw; i++) t += red[i];
    }
    return t;
}

// splitmix64 finaliser: a counter-based generator, so the force does not
// depend on the launch shape
__device__ __forceinline__ uint64_t mix64(uint64_t z) {
    z += 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

// randForce (Grid.cu:2242-2245): components uniform in [-1, 1) on existing nodes
__global__ void __launch_bounds__(256) k_rand_force(int N, const uint8_t* __restrict__ vflag, uint64_t seed,
                                                    Vec3<double> F) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < N; i += gridDim.x * blockDim.x) {
        const bool act = vflag[i] & NF_ACTIVE;
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const uint64_t r = mix64(seed ^ mix64((uint64_t)i * 3 + c));
            const double u = (double)(r >> 11) * (1.0 / 9007199254740992.0);   // [0, 1)
            F.c[c][i] = act ? 2.0 * u - 1.0 : 0.0;
        }
    }
}
void launch_rand_force(const Geom& g, const uint8_t* vflag, uint64_t seed, Vec3<double> F, hipStream_t s) {
    hipLaunchKernelGGL(k_rand_force, dim3(1024), dim3(256), 0, s, g.N, vflag, seed, F);
    RT_HIP(hipGetLastError());
}

// fs = P x at the load nodes (projection.cu:165-231): the nodal value, or
// its normal component (f.n) n in the constrained-direction mode
// (projection.cpp:338-340); per-block partial sums of |fs|^2
__global__ void __launch_bounds__(256) k_pm_gather(int nl, const int* __restrict__ slots, Vec3<const double> X,
                                                   const double* __restrict__ nrm, double* __restrict__ fs,
                                                   double* __restrict__ partials) {
    double s = 0;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < nl; i += gridDim.x * blockDim.x) {
        const int v = slots[i];
        double f0 = X.c[0][v], f1 = X.c[1][v], f2 = X.c[2][v];
        if (nrm) {
            const double n0 = nrm[i], n1 = nrm[nl + i], n2 = nrm[2 * nl + i];
            const double d = f0 * n0 + f1 * n1 + f2 * n2;
            f0 = d * n0; f1 = d * n1; f2 = d * n2;
        }
        fs[i] = f0; fs[nl + i] = f1; fs[2 * nl + i] = f2;
        s += f0 * f0 + f1 * f1 + f2 * f2;
    }
    s = blk_sum_w(s);
    if (threadIdx.x == 0) partials[blockIdx.x] = s;
}
void launch_pm_gather(int nl, const int* slots, Vec3<const double> X, const double* nrm, double* fs,
                      double* partials, int nparts, hipStream_t s) {
    hipLaunchKernelGGL(k_pm_gather, dim3(nparts), dim3(256), 0, s, nl, slots, X, nrm, fs, partials);
    RT_HIP(hipGetLastError());
}

// F[slot] = scale * fs; partials[b] = sum |new - old|^2, partials[nparts + b] =
// sum |old|^2 (supportForceCh / supportForceNorm, Grid.cu:2255-2286); old <- new
__global__ void __launch_bounds__(256) k_pm_commit(int nl, const int* __restrict__ slots,
                                                   const double* __restrict__ fs, double scale, Vec3<double> F,
                                                   double* __restrict__ fold, double* __restrict__ partials) {
    double d = 0, o = 0;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < nl; i += gridDim.x * blockDim.x) {
        const int v = slots[i];
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const double nv = fs[c * nl + i] * scale, ov = fold[c * nl + i];
            F.c[c][v] = nv;
            d += (nv - ov) * (nv - ov);
            o += ov * ov;
            fold[c * nl + i] = nv;
        }
    }
    d = blk_sum_w(d);
    o = blk_sum_w(o);
    if (threadIdx.x == 0) { partials[blockIdx.x] = d; partials[gridDim.x + blockIdx.x] = o; }
}
void launch_pm_commit(int nl, const int* slots, const double* fs, double scale, Vec3<double> F, double* fold,
                      double* partials, int nparts, hipStream_t s) {
    hipLaunchKernelGGL(k_pm_commit, dim3(nparts), dim3(256), 0, s, nl, slots, fs, scale, F, fold, partials);
    RT_HIP(hipGetLastError());
}

// ---------------------------------------------------------------------------
// C = A^T B for tall A (m x na) and B (m x nb), column-major, both of a few
// columns: the block Lanczos projections. A GEMM of this shape has one output
// tile and runs its whole length of m in one workgroup (9.4 ms at m = 150,000,
// 8 x 8); here the rows are cut into chunks, each workgroup takes 4 x 4 columns
// of one chunk, and the chunks' partial sums are added in order.
// Bound: the reads, a column of A once per four columns of B and the other way
// round, from HBM the first time and from L2 after that.
// ---------------------------------------------------------------------------
namespace {
constexpr int kGramRows = 2048;     // rows of a chunk: eight per thread
constexpr int kGramTile = 4;
}  // namespace

__global__ void __launch_bounds__(256) k_gram(int m, int na, int nb, const double* __restrict__ A,
                                              const double* __restrict__ B, double* __restrict__ part) {
    __shared__ double red[4][kGramTile * kGramTile];
    const int ta = (na + kGramTile - 1) / kGramTile;
    const int i0 = (blockIdx.y % ta) * kGramTile, j0 = (blockIdx.y / ta) * kGramTile;
    // columns past the last one repeat it; their sums are dropped
    const double *a[kGramTile], *b[kGramTile];
#pragma unroll
    for (int k = 0; k < kGramTile; k++) {
        a[k] = A + (size_t)min(i0 + k, na - 1) * m;
        b[k] = B + (size_t)min(j0 + k, nb - 1) * m;
    }
    double acc[kGramTile][kGramTile] = {};
    const int r1 = min((int)(blockIdx.x + 1) * kGramRows, m);
    for (int r = blockIdx.x * kGramRows + threadIdx.x; r < r1; r += 256) {
        double x[kGramTile], y[kGramTile];
#pragma unroll
        for (int k = 0; k < kGramTile; k++) { x[k] = a[k][r]; y[k] = b[k][r]; }
#pragma unroll
        for (int i = 0; i < kGramTile; i++)
#pragma unroll
            for (int j = 0; j < kGramTile; j++) acc[i][j] += x[i] * y[j];
    }
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
    for (int i = 0; i < kGramTile; i++)
#pragma unroll
        for (int j = 0; j < kGramTile; j++) {
            double v = acc[i][j];
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
            if (lane == 0) red[w][kGramTile * j + i] = v;
        }
    __syncthreads();
    const int t = threadIdx.x;
    if (t < kGramTile * kGramTile)
        part[((size_t)blockIdx.y * gridDim.x + blockIdx.x) * kGramTile * kGramTile + t] =
            (red[0][t] + red[1][t]) + (red[2][t] + red[3][t]);
}

// one workgroup per tile: entry t % 16, chunks t / 16, t / 16 + 16, ...
__global__ void __launch_bounds__(256) k_gram_sum(int chunks, int na, int nb, const double* __restrict__ part,
                                                  double* __restrict__ C) {
    __shared__ double red[16][16];
    const int e = threadIdx.x & 15, q = threadIdx.x >> 4;
    const double* p = part + (size_t)blockIdx.x * chunks * 16;
    double v = 0;
    for (int c = q; c < chunks; c += 16) v += p[(size_t)c * 16 + e];
    red[q][e] = v;
    __syncthreads();
    if (q) return;
    double t = 0;
#pragma unroll
    for (int k = 0; k < 16; k++) t += red[k][e];
    const int ta = (na + kGramTile - 1) / kGramTile;
    const int i = (blockIdx.x % ta) * kGramTile + e % kGramTile, j = (blockIdx.x / ta) * kGramTile + e / kGramTile;
    if (i < na && j < nb) C[(size_t)j * na + i] = t;
}

static int gram_tiles(int na, int nb) {
    return ((na + kGramTile - 1) / kGramTile) * ((nb + kGramTile - 1) / kGramTile);
}
static int gram_chunks(int m) { return (m + kGramRows - 1) / kGramRows; }
size_t gram_work(int m, int na, int nb) {
    return (size_t)gram_tiles(na, nb) * gram_chunks(m) * kGramTile * kGramTile;
}
void launch_gram(int m, int na, int nb, const double* A, const double* B, double* C, double* work, hipStream_t s) {
    if (m < 1 || na < 1 || nb < 1) throw std::invalid_argument("launch_gram: empty operand");
    const int tiles = gram_tiles(na, nb), chunks = gram_chunks(m);
    hipLaunchKernelGGL(k_gram, dim3(chunks, tiles), dim3(256), 0, s, m, na, nb, A, B, work);
    hipLaunchKernelGGL(k_gram_sum, dim3(tiles), dim3(256), 0, s, chunks, na, nb, (const double*)work, C);
    RT_HIP(hipGetLastError());
}

}  // namespace rt
