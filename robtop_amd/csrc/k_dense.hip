// Explicit inverse of the small dense SPD systems (the coarsest level, and the
// level above it in the preconditioner's cycle) by blocked Gauss-Jordan sweeps
// on the FP64 matrix cores.
//
// Sweeping the 64-wide pivot block k of a symmetric A (its lower tiles are
// stored) replaces
//     A_kk by -D,  A_ik by W_i = A_ik D,  A_ij by A_ij - W_i A_jk^T,
// with D = A_kk^-1; once every block has been swept the matrix is -A^-1. The
// Schur complements are those of a Cholesky factorisation in the same order,
// so a system that is not positive definite shows as a non-positive pivot.
//
// What bounds it is the chain of pivot blocks, each a launch, not the matrix
// cores: hence
//   - blocks that do not couple are swept by the same launch. The unknowns are
//     numbered with the level's longest axis slowest, so A is banded; nested
//     dissection of the band into up to kGjMax segments sweeps the segments
//     side by side, then the separators between them (direct_plan);
//   - a block is combined only with the tile rows that it couples to by then
//     (one contiguous range per block), the others are skipped;
//   - the launch also writes the next blocks' columns, transposed, into PTn
//     (the next launch reads them while it overwrites the tiles), and inverts
//     the next blocks' diagonal tiles in workgroups of their own, so the
//     serial 64-pivot inversion overlaps the other tiles' products.
// Measured: 4,131 unknowns (17 x 9 x 9 nodes: 26 launches for 65 blocks) 1.33
// ms, 675 unknowns 0.32 ms; rocSOLVER's dpotrf and dpotri took 18 ms for the
// two together, as much as the rest of a SIMP step at 64 x 32 x 32 elements.
// Larger ones, where rt_set_coarse_direct_dofs admits them: 10,125 unknowns (112^3
// elements) 9 ms against 83, 22,356 (36 rods) 64 ms against 481.
// A workgroup owns one tile row I and up to kGjCols tiles of it: W_I is formed
// once (as much work as one tile), each wave 16 rows of it, and goes to MFMA
// operand order through LDS.
#include "rt_internal.h"

#include <algorithm>

namespace rt {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef double d2 __attribute__((ext_vector_type(2)));

namespace {
constexpr int GB = 64;          // pivot block
constexpr int kGjCols = 4;      // tiles per workgroup
constexpr int WP = 17;          // LDS row of a wave's 16-row W (padded)
constexpr int TP = GB + 8;      // LDS row of a staged tile (padded; two workgroups fit a CU)
}  // namespace

// v_mfma_f64_16x16x4_f64: lane l holds A[l % 16][l / 16], B[l / 16][l % 16],
// and D[4 r + l / 16][l % 16] in register r
__device__ __forceinline__ d4 mfma64(double a, double b, d4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// 1 / x to about an ulp: the hardware estimate and two Newton steps (the IEEE
// division sequence would sit on the pivot chain)
__device__ __forceinline__ double gj_rcp(double x) {
    double r = __builtin_amdgcn_rcp(x);
    r = __builtin_fma(__builtin_fma(-x, r, 1.0), r, r);
    return __builtin_fma(__builtin_fma(-x, r, 1.0), r, r);
}

// D = S^-1 of the 64 x 64 SPD tile in LDS, two pivots (a 2 x 2 block) at a
// time with one barrier each. Thread (ti, tj) holds the 4 x 4 block of rows
// 4 ti.. and columns 4 tj.. in registers; by symmetry the pivot rows are the
// pivot columns, which their 16 threads put into LDS. 4 x 4 blocks, since the
// LDS reads of the pivot columns are what a step takes: 8 values a thread and
// column against 17 with a thread per row.
// A pivot block's determinant is formed times a power of two (exact; lane l of a
// wave keeps that of pivots 2 l, 2 l + 1, from the tile's diagonal before the
// sweeps), so that it is in range for every stiffness whose inverse is.
__device__ __forceinline__ void gj_invert(const double (*S)[GB + 1], double (*col)[2][GB], double* __restrict__ D,
                                          int* __restrict__ info) {
    const int ti = threadIdx.x >> 4, tj = threadIdx.x & 15;
    double a[4][4];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) a[i][j] = S[4 * ti + i][4 * tj + j];
    const int dg = 2 * (threadIdx.x & 31);
    const int sc_hi = (1023 - min(max(__builtin_amdgcn_frexp_exp(S[dg][dg]), -1000), 1000)) << 20;
    bool bad = false;
    for (int tp = 0; tp < 16; tp++) {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int p = 4 * tp + 2 * h;
            double(*c)[GB] = col[h];
            if (tj == tp) {
#pragma unroll
                for (int i = 0; i < 4; i++) { c[0][4 * ti + i] = a[i][2 * h]; c[1][4 * ti + i] = a[i][2 * h + 1]; }
            }
            __syncthreads();
            const double d00 = c[0][p], d01 = c[1][p], d11 = c[1][p + 1];
            const double sc = __hiloint2double(__builtin_amdgcn_readlane(sc_hi, 2 * tp + h), 0);
            const double s00 = d00 * sc, s01 = d01 * sc, s11 = d11 * sc;
            double r0[4], r1[4], k0[4], k1[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                r0[i] = c[0][4 * ti + i]; r1[i] = c[1][4 * ti + i];
                k0[i] = c[0][4 * tj + i]; k1[i] = c[1][4 * tj + i];
            }
            const double det = s00 * d11 - s01 * d01;                    // times sc, as the others
            bad = bad || !(d00 > 0) || !(det > 0);
            const double rd = gj_rcp(det), e00 = s11 * rd, e01 = -s01 * rd, e11 = s00 * rd;
            double x0[4], x1[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {                                // W
                x0[i] = r0[i] * e00 + r1[i] * e01;
                x1[i] = r0[i] * e01 + r1[i] * e11;
            }
            if (ti == tp) {                                              // the pivot rows: W^T and -D
                x0[2 * h] = -e00; x1[2 * h] = -e01;
                x0[2 * h + 1] = -e01; x1[2 * h + 1] = -e11;
#pragma unroll
                for (int j = 0; j < 4; j++) a[2 * h][j] = a[2 * h + 1][j] = 0;
            }
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int j = 0; j < 4; j++) a[i][j] = (a[i][j] - x0[i] * k0[j]) - x1[i] * k1[j];
            if (tj == tp) {
#pragma unroll
                for (int i = 0; i < 4; i++) { a[i][2 * h] = x0[i]; a[i][2 * h + 1] = x1[i]; }
            }
        }
    }
    if (bad) *info = 1;
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) D[(4 * ti + i) * GB + 4 * tj + j] = -a[i][j];
}

struct GjStep {
    double* A;                   // ld x ld, lower tiles
    int ld, nc, nn;              // row stride, blocks swept now, blocks of the next launch
    GjPivot cur[kGjMax], nxt[kGjMax];
    const double *PT, *D;        // per block: its column transposed [64][ld], inverse of its tile [64][64]
    double *PTn, *Dn;            // the same of the next blocks
    int* info;
};

// a 64 x 64 tile on its way to LDS: eight 16-byte loads per thread, all in flight
struct GjTile {
    d2 v[8];
    __device__ __forceinline__ void load(const double* p, int ld) {
        const unsigned o = (threadIdx.x >> 5) * ld + 2 * (threadIdx.x & 31);
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] = *reinterpret_cast<const d2*>(p + (size_t)(8 * i) * ld + o);
    }
    __device__ __forceinline__ void store(double (*T)[TP]) const {
        const int c = 2 * (threadIdx.x & 31), r = threadIdx.x >> 5;
#pragma unroll
        for (int i = 0; i < 8; i++) *reinterpret_cast<d2*>(&T[r + 8 * i][c]) = v[i];
    }
};

__global__ void __launch_bounds__(256, 2) k_gj_step(GjStep s, int nwork) {
    __shared__ union {
        double T[GB][TP];            // D, then W, then (workgroups of next blocks) the tile to invert
        double w[4][GB * WP];
        double S[GB][GB + 1];
    } sh;
    __shared__ double P[GB][TP];     // the current tile's P_J^T
    __shared__ double col[2][2][GB];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, q = lane >> 4;
    const int ld = s.ld, nb = ld / GB;
    // lane offsets from wave-uniform addresses: an operand's (row q, column
    // l16) of a matrix of stride ld or 64, and the transposed (row l16, column q)
    const unsigned oq = q * ld + l16, oq64 = q * GB + l16, ot = l16 * ld + q;
    const size_t pts = (size_t)GB * ld;      // panel stride
    const bool diag = (int)blockIdx.x < s.nn;
    int I, J0, J1;
    if (diag) {
        I = 0;
#pragma unroll
        for (int c = 0; c < kGjMax; c++)
            if ((int)blockIdx.x == c) I = s.nxt[c].k;
        J0 = I;
        J1 = I + 1;
    } else {
        // rows 4 g .. 4 g + 3 have g + 1 groups of tiles each; the longest rows first
        const int t = nwork - 1 - ((int)blockIdx.x - s.nn);
        int g = (int)((sqrtf(2.f * (float)t + 1.f) - 1.f) * 0.5f);
        while (2 * (g + 1) * (g + 2) <= t) g++;
        while (2 * g * (g + 1) > t) g--;
        const int rem = t - 2 * g * (g + 1);
        I = 4 * g + rem / (g + 1);
        if (I >= nb) return;
        J0 = kGjCols * (rem % (g + 1));
        J1 = min(J0 + kGjCols, I + 1);
    }
    // the blocks swept now that row I couples to: at most two (gj_region)
    int c0 = -1, c1 = -1, l0 = 0, l1 = 0, k0 = -1, k1 = -1;
#pragma unroll
    for (int c = 0; c < kGjMax; c++)
        if (c < s.nc && I >= s.cur[c].lo && I < s.cur[c].hi && J1 > s.cur[c].lo) {
            if (c0 < 0) {
                c0 = c; l0 = s.cur[c].lo; k0 = s.cur[c].k;
            } else {
                c1 = c; l1 = s.cur[c].lo; k1 = s.cur[c].k;
            }
        }
    // the next block whose column holds a tile of this row: of row I (nI, its
    // columns [nlo, nhi)), and of column nk
    int nI = -1, nlo = 0, nhi = 0, nJ = -1, nk = -1;
#pragma unroll
    for (int c = 0; c < kGjMax; c++) {
        if (c < s.nn && s.nxt[c].k == I) {
            nI = c; nlo = s.nxt[c].lo; nhi = s.nxt[c].hi;
        }
        if (c < s.nn && s.nxt[c].k >= J0 && s.nxt[c].k < J1 && I >= s.nxt[c].lo && I < s.nxt[c].hi) {
            nJ = c; nk = s.nxt[c].k;
        }
    }
    if (c0 < 0 && nI < 0 && nJ < 0) return;
    const size_t arow = (size_t)I * GB + 16 * w;   // first row of this wave
    // one pass per swept block (a row of two blocks' ranges takes both, one
    // after the other, through its tiles); without any, only the columns of
    // the next blocks are copied
    for (int m = 0; m < (c1 >= 0 ? 2 : 1); m++) {
        const int c = m ? c1 : c0, k = m ? k1 : k0, lo = m ? l1 : l0;
        const double* PT = s.PT + (c >= 0 ? c : 0) * pts;
        const bool prow = c >= 0 && I == k;      // the block's own row: W_J^T = D P_J^T
        int J = J0;
        GjTile nextP;
        auto product_at = [&](int j) __attribute__((always_inline)) { return c >= 0 && j >= lo && j < J1 && j != k; };
        if (product_at(J)) nextP.load(PT + (size_t)J * GB, ld);
        double wv[16];
        if (c >= 0) {
            const double* D = s.D + (size_t)c * GB * GB;
            if (prow) {
#pragma unroll
                for (int t = 0; t < 16; t++) wv[t] = (D + 4 * t * GB + 16 * w)[oq64];
            } else {
                GjTile td;
                td.load(D, GB);
                double a[16];
#pragma unroll
                for (int t = 0; t < 16; t++) a[t] = (PT + (size_t)(4 * t) * ld + arow)[oq];
                __syncthreads();                 // the W of an earlier pass has been read
                td.store(sh.T);
                __syncthreads();
                d4 acc[4];
#pragma unroll
                for (int f = 0; f < 4; f++) acc[f] = d4{0, 0, 0, 0};
#pragma unroll
                for (int t = 0; t < 16; t++) {
#pragma unroll
                    for (int f = 0; f < 4; f++) acc[f] = mfma64(a[t], sh.T[4 * t + q][16 * f + l16], acc[f]);
                    if (t % 4 == 3) __builtin_amdgcn_sched_barrier(0);   // (bounds the operands in registers)
                }
                __syncthreads();                 // D has been read
#pragma unroll
                for (int f = 0; f < 4; f++)
#pragma unroll
                    for (int r = 0; r < 4; r++) sh.w[w][(16 * f + l16) * WP + 4 * r + q] = acc[f][r];
                __syncthreads();
#pragma unroll
                for (int t = 0; t < 16; t++) wv[t] = sh.w[w][(4 * t + q) * WP + l16];
            }
        }
        const double sign = prow ? 1.0 : -1.0;
        for (; J < J1; J++) {
            const bool on = c >= 0 && J >= lo;                      // J <= I < hi
            const bool last = m == 1 || c1 < 0 || J < l1;           // no later pass changes this tile
            // columns of the next blocks that this tile belongs to
            const bool pI = last && nI >= 0 && J >= nlo && J < nhi, pJ = last && nJ >= 0 && J == nk;
            if (!on && (m == 1 || (!pI && !pJ))) {
                if (product_at(J + 1)) nextP.load(PT + (size_t)(J + 1) * GB, ld);
                continue;
            }
            const bool own = !diag && I == J && nI >= 0;            // a next block's diagonal tile: its own workgroup's
            double* At = s.A + arow * ld + (size_t)J * GB;          // 16 rows x 64 columns of the tile
            double* PIn = pI ? s.PTn + nI * pts : nullptr;
            double* PJn = pJ ? s.PTn + nJ * pts : nullptr;
            // a tile in the block's column (I > k: W_I) or its diagonal (-D)
            if (on && J == k) {
#pragma unroll
                for (int t = 0; t < 16; t++) {
                    const double v = I == J ? -wv[t] : wv[t];
                    (At + 4 * t)[ot] = v;
                    if (PIn) (PIn + (size_t)(16 * w) * ld + (size_t)J * GB + 4 * t)[ot] = v;
                }
                if (product_at(J + 1)) nextP.load(PT + (size_t)(J + 1) * GB, ld);
                continue;
            }
            d4 acc[4];
#pragma unroll
            for (int f = 0; f < 4; f++)
#pragma unroll
                for (int r = 0; r < 4; r++) acc[f][r] = on && prow ? 0.0 : (At + (size_t)(4 * r) * ld + 16 * f)[oq];
            if (on) {
                __syncthreads();                 // the previous P_J has been read
                nextP.store(P);
                if (product_at(J + 1)) nextP.load(PT + (size_t)(J + 1) * GB, ld);
                __syncthreads();
#pragma unroll
                for (int t = 0; t < 16; t++) {
                    const double a = sign * wv[t];
#pragma unroll
                    for (int f = 0; f < 4; f++) acc[f] = mfma64(a, P[4 * t + q][16 * f + l16], acc[f]);
                    if (t % 4 == 3) __builtin_amdgcn_sched_barrier(0);
                }
            } else if (product_at(J + 1)) {
                nextP.load(PT + (size_t)(J + 1) * GB, ld);
            }
            if (own) continue;
            if (diag && last) {
                __syncthreads();                 // sh.w has been read
#pragma unroll
                for (int f = 0; f < 4; f++)
#pragma unroll
                    for (int r = 0; r < 4; r++) sh.S[16 * w + 4 * r + q][16 * f + l16] = acc[f][r];
                __syncthreads();
                gj_invert(sh.S, col, s.Dn + (size_t)blockIdx.x * GB * GB, s.info);
                return;
            }
#pragma unroll
            for (int f = 0; f < 4; f++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const double v = acc[f][r];
                    if (on) (At + (size_t)(4 * r) * ld + 16 * f)[oq] = v;
                    if (PJn) (PJn + (size_t)(16 * f) * ld + arow + 4 * r)[ot] = v;
                    if (PIn) (PIn + (size_t)(16 * w + 4 * r) * ld + (size_t)J * GB + 16 * f)[oq] = v;
                }
        }
    }
}

// A = -A in both triangles from the lower tiles: one workgroup per tile pair
__global__ void __launch_bounds__(256) k_gj_finish(double* __restrict__ A, int ld) {
    __shared__ double S[GB][GB + 1];
    const int I = blockIdx.y, J = blockIdx.x;
    if (J > I) return;
    const int c = threadIdx.x & 63, r0 = threadIdx.x >> 6;
    double* lo = A + (size_t)I * GB * ld + (size_t)J * GB;
    double* up = A + (size_t)J * GB * ld + (size_t)I * GB;
#pragma unroll 4
    for (int r = r0; r < GB; r += 4) S[r][c] = -lo[(size_t)r * ld + c];
    __syncthreads();
#pragma unroll 4
    for (int r = r0; r < GB; r += 4) {
        lo[(size_t)r * ld + c] = I == J && c > r ? S[c][r] : S[r][c];
        if (I != J) up[(size_t)r * ld + c] = S[c][r];
    }
}

// the sweeps of blocks [a, b), whose couplings end within [lo, hi): the two
// sides of a separator in the middle step by step together, then the separator
static void gj_region(const std::vector<int>& reach, int a, int b, int lo, int hi, int parts, GjPlan& out) {
    const int mid = (a + b) / 2;
    int e = mid;                              // the separator [mid, e) ends the reach of every block before mid
    for (int k = lo; k < mid; k++) e = std::max(e, reach[k]);
    // worth it when the chain gets shorter: half the blocks, with the separator after them
    if (parts < 2 || mid <= a || e >= b || std::max(mid - a, b - e) + (e - mid) >= b - a) {
        int far = 0;
        for (int k = a; k < b; k++) {
            far = std::max({far, reach[k], std::min(k + 2, hi)});
            out.push_back({GjPivot{k, lo, std::min(far, hi)}});
        }
        return;
    }
    GjPlan l, r;
    gj_region(reach, a, mid, lo, e, parts / 2, l);
    gj_region(reach, e, b, mid, hi, parts / 2, r);
    for (size_t i = 0; i < std::max(l.size(), r.size()); i++) {
        std::vector<GjPivot> step;
        if (i < l.size()) step = l[i];
        if (i < r.size()) step.insert(step.end(), r[i].begin(), r[i].end());
        out.push_back(step);
    }
    for (int k = mid; k < e; k++) out.push_back({GjPivot{k, lo, hi}});
}

// reach[k]: end of the tile rows that block k couples to in A
GjPlan spd_inverse_plan(const std::vector<int>& reach) {
    GjPlan out;
    const int nb = (int)reach.size();
    gj_region(reach, 0, nb, 0, nb, kGjMax, out);
    return out;
}

size_t spd_inverse_work(int n) { return (size_t)2 * kGjMax * (GB * (size_t)dense_ld(n) + GB * GB); }

// In place: A (dense_ld(n) square, row-major, the unknowns past n decoupled
// with a unit diagonal) becomes its inverse. work: spd_inverse_work(n)
// doubles. *info (device) is set to 1 when a pivot is not positive, else 0.
void launch_spd_inverse(double* A, int n, const GjPlan& plan, double* work, int* info, hipStream_t s) {
    const int ld = dense_ld(n), nb = ld / GB;
    double* PT[2] = {work, work + (size_t)kGjMax * GB * ld};
    double* D[2] = {work + (size_t)2 * kGjMax * GB * ld, work + (size_t)2 * kGjMax * GB * ld + kGjMax * GB * GB};
    const int g = (nb + 3) / 4, nwork = 2 * g * (g + 1);
    launch_fill<uint8_t>(reinterpret_cast<uint8_t*>(info), 0, sizeof(int), s);
    for (int t = -1; t < (int)plan.size(); t++) {
        GjStep st{};
        st.A = A; st.ld = ld;
        if (t >= 0) {
            st.nc = (int)plan[t].size();
            std::copy(plan[t].begin(), plan[t].end(), st.cur);
        }
        if (t + 1 < (int)plan.size()) {
            st.nn = (int)plan[t + 1].size();
            std::copy(plan[t + 1].begin(), plan[t + 1].end(), st.nxt);
        }
        const int c = t & 1, m = c ^ 1;
        st.PT = PT[c]; st.D = D[c]; st.PTn = PT[m]; st.Dn = D[m];
        st.info = info;
        hipLaunchKernelGGL(k_gj_step, dim3((unsigned)(st.nn + nwork)), dim3(256), 0, s, st, nwork);
    }
    hipLaunchKernelGGL(k_gj_finish, dim3(nb, nb), dim3(256), 0, s, A, ld);
    RT_HIP(hipGetLastError());
}

}  // namespace rt
