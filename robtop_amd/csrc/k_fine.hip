// Finest-level nodal Gauss-Seidel on the octant layout (see rt_internal.h).
//
// For a node v the reference forms, element by element (Grid.cu:922-1066),
//     KeU_v = sum_{e ni v} rho_e^p * sum_{j in e, j != v} KE[v_loc(e)][j_loc(e)] u_j
//     S_v   = sum_{e ni v} rho_e^p * KE[v_loc(e)][v_loc(e)]
// where the element incident at w = (w%2-1, w/2%2-1, w/4-1) holds v as local
// vertex 7-w; support ("fixed") neighbours contribute nothing, a fixed node
// gets S = n_e I and KeU = 0; then x, y, z are relaxed in turn.
//
// One thread per node of the colour being relaxed; the colour is a template
// parameter, so each of the 27 neighbour slots and 8 element slots is the
// thread's base index plus a wave-uniform offset. Loads are raw buffer loads
// with that offset in a scalar register (no per-load address arithmetic). The
// loop runs over neighbours and accumulates into 8 per-element partials, so a
// neighbour's displacement is live only while it is used. KE enters as 10
// signed scalar constants (ke_pattern.h): every FMA takes its coefficient from
// an SGPR with a sign modifier.
#include "rt_internal.h"
#include "ke_pattern.h"

#include <algorithm>
#include <cmath>
#include <type_traits>
#include <utility>

namespace rt {

// the smoother addresses u, rho^p and the flags through buffer resources whose
// byte ranges are 32-bit: a level whose vectors pass 2 GiB is refused instead of
// being read as zeros past the limit
template <typename T>
static void check_buffer_range(const Geom& g) {
    if ((long long)g.N * (long long)sizeof(T) >= (1ll << 31))
        throw std::invalid_argument(std::string("finest level of ") + std::to_string(g.N) +
                                    " slots is too large for 32-bit buffer offsets in this precision's smoother" +
                                    (sizeof(T) == 8 ? " (FP32 cycles reach twice the size)" : ""));
}


template <typename T> struct KeC { T c[RT_KE_NVAL]; };

static double g_kec[RT_KE_NVAL];

// the 10 distinct magnitudes of KE, read off the table (validated entry by entry)
void set_ke_constants(const double* ke576, hipStream_t) {
    bool seen[RT_KE_NVAL] = {false};
    for (int i = 0; i < 576; i++) {
        const int c = rt_ke_code[i];
        if (c && !seen[std::abs(c) - 1]) { g_kec[std::abs(c) - 1] = c > 0 ? ke576[i] : -ke576[i]; seen[std::abs(c) - 1] = true; }
    }
    double scale = 0;
    for (int i = 0; i < 576; i++) scale = std::max(scale, std::fabs(ke576[i]));
    for (int i = 0; i < 576; i++) {
        const int c = rt_ke_code[i];
        const double v = c == 0 ? 0.0 : (c > 0 ? g_kec[c - 1] : -g_kec[-c - 1]);
        if (std::fabs(v - ke576[i]) > 1e-12 * scale)
            throw std::runtime_error("element matrix does not follow the isotropic hexahedron pattern");
    }
}

template <typename T>
static KeC<T> kec() {
    KeC<T> k;
    for (int i = 0; i < RT_KE_NVAL; i++) k.c[i] = (T)g_kec[i];
    return k;
}

// offset (in slots, shifted to be >= 0) of the point at (DX,DY,DZ) in {-1,0,1}^3
// from a colour-C node whose half-index base is b: slot = (b - hxy - hx - 1) + off
template <int C, int DX, int DY, int DZ>
__device__ __forceinline__ int rel_off(const Geom& g) {
    constexpr int cx = C & 1, cy = (C >> 1) & 1, cz = C >> 2;
    constexpr int col = C ^ ((DX & 1) | ((DY & 1) << 1) | ((DZ & 1) << 2));
    constexpr int ox = (cx + DX) >> 1, oy = (cy + DY) >> 1, oz = (cz + DZ) >> 1;
    return col * g.cs + ((oz + 1) * g.h[1] + (oy + 1)) * g.h[0] + (ox + 1);
}

constexpr int ke_code_at(int i) { return rt_ke_code[i]; }

template <int CODE, typename T>
__device__ __forceinline__ T kc(const KeC<T>& K) {
    static_assert(CODE != 0, "isotropic KE has no zero entry");
    if constexpr (CODE > 0) return K.c[CODE - 1];
    else return -K.c[-CODE - 1];
}

// acc[W] += KE[vi rows][vj cols] u_nb for neighbour NB (position NB%3, NB/3%3,
// NB/9 in the 3x3x3 block around the node) if it is vertex vj != vi of element W
template <typename T, int NB, int W>
__device__ __forceinline__ void nb_elem(T (&acc)[8][3], const KeC<T>& K, T u0, T u1, T u2) {
    constexpr int px = NB % 3, py = NB / 3 % 3, pz = NB / 9;
    constexpr int jx = px - (W & 1), jy = py - ((W >> 1) & 1), jz = pz - (W >> 2);
    if constexpr (jx >= 0 && jx <= 1 && jy >= 0 && jy <= 1 && jz >= 0 && jz <= 1) {
        constexpr int vj = jx + 2 * jy + 4 * jz, vi = 7 - W;
        if constexpr (vj != vi) {
            acc[W][0] += kc<ke_code_at((3 * vi + 0) * 24 + 3 * vj + 0)>(K) * u0;
            acc[W][0] += kc<ke_code_at((3 * vi + 0) * 24 + 3 * vj + 1)>(K) * u1;
            acc[W][0] += kc<ke_code_at((3 * vi + 0) * 24 + 3 * vj + 2)>(K) * u2;
            acc[W][1] += kc<ke_code_at((3 * vi + 1) * 24 + 3 * vj + 0)>(K) * u0;
            acc[W][1] += kc<ke_code_at((3 * vi + 1) * 24 + 3 * vj + 1)>(K) * u1;
            acc[W][1] += kc<ke_code_at((3 * vi + 1) * 24 + 3 * vj + 2)>(K) * u2;
            acc[W][2] += kc<ke_code_at((3 * vi + 2) * 24 + 3 * vj + 0)>(K) * u0;
            acc[W][2] += kc<ke_code_at((3 * vi + 2) * 24 + 3 * vj + 1)>(K) * u1;
            acc[W][2] += kc<ke_code_at((3 * vi + 2) * 24 + 3 * vj + 2)>(K) * u2;
        }
    }
}

template <typename T, int NB, int... Ws>
__device__ __forceinline__ void nb_elems(T (&acc)[8][3], const KeC<T>& K, T u0, T u1, T u2,
                                         std::integer_sequence<int, Ws...>) {
    (nb_elem<T, NB, Ws>(acc, K, u0, u1, u2), ...);
}

struct GsBufs {
    __amdgpu_buffer_rsrc_t u0, u1, u2, rho, flag;
};

// colour of the neighbour at (DX, DY, DZ) of a colour-C node
template <int C, int DX, int DY, int DZ>
constexpr int nb_colour() { return C ^ ((DX & 1) | ((DY & 1) << 1) | ((DZ & 1) << 2)); }

// Z0 ("zero start"): the sweep is the first of a forward cycle from u = 0, so
// a neighbour whose colour comes later in the order 0..7 still holds 0 and is
// neither loaded nor multiplied (adding KE * 0 leaves the sums unchanged).
template <typename T, int C, bool CHECK_FIX, int NB, bool Z0 = false>
__device__ __forceinline__ void nb_step(const Geom& g, int vb, const KeC<T>& K, const GsBufs& B, T (&acc)[8][3]) {
    if constexpr (NB != 13 && !(Z0 && nb_colour<C, NB % 3 - 1, NB / 3 % 3 - 1, NB / 9 - 1>() > C)) {
        const int so = rel_off<C, NB % 3 - 1, NB / 3 % 3 - 1, NB / 9 - 1>(g);
        const int vo = vb * (int)sizeof(T), sob = so * (int)sizeof(T);
        T u0 = bload<T>(B.u0, vo, sob);
        T u1 = bload<T>(B.u1, vo, sob);
        T u2 = bload<T>(B.u2, vo, sob);
        if constexpr (CHECK_FIX) {
            if (bload_u8(B.flag, vb, so) & NF_FIXED) { u0 = T(0); u1 = T(0); u2 = T(0); }
        }
        nb_elems<T, NB>(acc, K, u0, u1, u2, std::make_integer_sequence<int, 8>{});
    }
}

// two consecutive values of one stream with one load (dword-aligned 8- or 16-byte
// buffer load)
template <typename T> struct Two { T lo, hi; };
template <typename T> __device__ __forceinline__ Two<T> bload2(__amdgpu_buffer_rsrc_t r, int voff, int soff);
template <>
__device__ __forceinline__ Two<float> bload2<float>(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
    return __builtin_bit_cast(Two<float>, __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0));
}
template <>
__device__ __forceinline__ Two<double> bload2<double>(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
    return __builtin_bit_cast(Two<double>, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
}

// The x-neighbours (dx = -1, +1) of a row (dy, dz) have the opposite x parity,
// so both sit in one colour block at consecutive slots (offset of dx = -1, then
// + 1): one two-wide load fetches both. The dx = 0 neighbour is a single load.
template <typename T, int C, bool CHECK_FIX, int ROW, bool Z0 = false>
__device__ __forceinline__ void nb_row(const Geom& g, int vb, const KeC<T>& K, const GsBufs& B, T (&acc)[8][3]) {
    constexpr int DY = ROW % 3 - 1, DZ = ROW / 3 - 1;
    constexpr int NBM = 9 * (DZ + 1) + 3 * (DY + 1);   // dx = -1; dx = 0, +1 follow
    const int vo = vb * (int)sizeof(T);
    if constexpr (!(Z0 && nb_colour<C, -1, DY, DZ>() > C)) {
        const int so = rel_off<C, -1, DY, DZ>(g), sob = so * (int)sizeof(T);
        const Two<T> a = bload2<T>(B.u0, vo, sob), b = bload2<T>(B.u1, vo, sob), c = bload2<T>(B.u2, vo, sob);
        T l0 = a.lo, l1 = b.lo, l2 = c.lo, r0 = a.hi, r1 = b.hi, r2 = c.hi;
        if constexpr (CHECK_FIX) {
            if (bload_u8(B.flag, vb, so) & NF_FIXED) { l0 = T(0); l1 = T(0); l2 = T(0); }
            if (bload_u8(B.flag, vb, so + 1) & NF_FIXED) { r0 = T(0); r1 = T(0); r2 = T(0); }
        }
        nb_elems<T, NBM>(acc, K, l0, l1, l2, std::make_integer_sequence<int, 8>{});
        nb_elems<T, NBM + 2>(acc, K, r0, r1, r2, std::make_integer_sequence<int, 8>{});
    }
    nb_step<T, C, CHECK_FIX, NBM + 1, Z0>(g, vb, K, B, acc);   // skips the node itself
}

// the neighbour rows in the order of every smoother kernel here: the node's
// own row last, since the row kernel has its second node's neighbours there
// only once the first ones are relaxed
typedef std::integer_sequence<int, 0, 1, 2, 3, 5, 6, 7, 8, 4> RowOrder;

template <typename T, int C, bool CHECK_FIX, bool Z0, int... ROWs>
__device__ __forceinline__ void nb_all(const Geom& g, int vb, const KeC<T>& K, const GsBufs& B, T (&acc)[8][3],
                                       std::integer_sequence<int, ROWs...>) {
    (nb_row<T, C, CHECK_FIX, ROWs, Z0>(g, vb, K, B, acc), ...);
}

template <typename T, int C, int W>
__device__ __forceinline__ void elem_step(const Geom& g, int vb, const KeC<T>& K, const GsBufs& B,
                                          const T (&acc)[8][3], T KU[3], T S[9]) {
    constexpr int vi = 7 - W;
    const int so = rel_off<C, (W & 1) - 1, ((W >> 1) & 1) - 1, (W >> 2) - 1>(g);
    const T pen = (T)bload<float>(B.rho, vb * 4, so * 4);
    KU[0] += pen * acc[W][0];
    KU[1] += pen * acc[W][1];
    KU[2] += pen * acc[W][2];
    S[0] += pen * kc<ke_code_at((3 * vi + 0) * 24 + 3 * vi + 0)>(K);
    S[1] += pen * kc<ke_code_at((3 * vi + 0) * 24 + 3 * vi + 1)>(K);
    S[2] += pen * kc<ke_code_at((3 * vi + 0) * 24 + 3 * vi + 2)>(K);
    S[3] += pen * kc<ke_code_at((3 * vi + 1) * 24 + 3 * vi + 0)>(K);
    S[4] += pen * kc<ke_code_at((3 * vi + 1) * 24 + 3 * vi + 1)>(K);
    S[5] += pen * kc<ke_code_at((3 * vi + 1) * 24 + 3 * vi + 2)>(K);
    S[6] += pen * kc<ke_code_at((3 * vi + 2) * 24 + 3 * vi + 0)>(K);
    S[7] += pen * kc<ke_code_at((3 * vi + 2) * 24 + 3 * vi + 1)>(K);
    S[8] += pen * kc<ke_code_at((3 * vi + 2) * 24 + 3 * vi + 2)>(K);
}

template <typename T, int C, int... Ws>
__device__ __forceinline__ void elem_all(const Geom& g, int vb, const KeC<T>& K, const GsBufs& B, const T (&acc)[8][3],
                                         T KU[3], T S[9], std::integer_sequence<int, Ws...>) {
    (elem_step<T, C, Ws>(g, vb, K, B, acc, KU, S), ...);
}

template <typename T, int C, bool CHECK_FIX, bool Z0 = false>
__device__ __forceinline__ void gs_node(const Geom& g, int base, const KeC<T>& K, const GsBufs& B, T KU[3], T S[9]) {
    const int vb = base - g.h[0] * g.h[1] - g.h[0] - 1;
    T acc[8][3];
#pragma unroll
    for (int w = 0; w < 8; w++) acc[w][0] = acc[w][1] = acc[w][2] = T(0);
    nb_all<T, C, CHECK_FIX, Z0>(g, vb, K, B, acc, RowOrder{});
    KU[0] = KU[1] = KU[2] = T(0);
#pragma unroll
    for (int i = 0; i < 9; i++) S[i] = T(0);
    elem_all<T, C>(g, vb, K, B, acc, KU, S, std::make_integer_sequence<int, 8>{});
}

// the three divisions of a node update; FP32 optionally by the hardware
// reciprocal (1 ulp) times the numerator instead of the IEEE division sequence
#ifndef RT_GS_FAST_DIV
#define RT_GS_FAST_DIV 0
#endif
template <typename T> __device__ __forceinline__ T gs_div(T a, T b) { return a / b; }
template <> __device__ __forceinline__ float gs_div<float>(float a, float b) {
    return RT_GS_FAST_DIV ? a * __builtin_amdgcn_rcpf(b) : a / b;
}

// GS update of the colour-C node with half-index base (Grid.cu:1007-1062)
// ZS ("zero supports"): the caller guarantees u = 0 at every support node for
// the whole sweep (f = 0 there, so the relaxation keeps it 0, and the
// prolongation skips supports), so a neighbour never needs its flag checked.
// Z0: the node's own old value is 0 as well, and an inactive node, which the
// sweep otherwise leaves alone, gets the 0 that a cleared vector would hold.
// fu: f . u_new of the node is added to it (the last sweep of a cycle, whose
// values are final: the preconditioned residual's r . z without another pass).
template <typename T, int C, bool ZS, bool Z0 = false>
__device__ __forceinline__ void gs_update(const Geom& g, int base, Vec3<T> U, Vec3<const T> F,
                                          const uint8_t* __restrict__ vflag, const KeC<T>& K, const GsBufs& B,
                                          bool reverse, double* fu = nullptr) {
    const int v = C * g.cs + base;
    const uint8_t fl = vflag[v];
    if (!(fl & NF_ACTIVE)) {
        if constexpr (Z0) { U.c[0][v] = T(0); U.c[1][v] = T(0); U.c[2][v] = T(0); }
        return;
    }
    const T f[3] = {F.c[0][v], F.c[1][v], F.c[2][v]};
    if (fl & NF_FIXED) {
        // S = n_e I, KeU = 0 (Grid.cu:1007-1014)
        const T ne = (T)(fl >> 4);
        const T u0 = f[0] / ne, u1 = f[1] / ne, u2 = f[2] / ne;
        U.c[0][v] = u0; U.c[1][v] = u1; U.c[2][v] = u2;
        if (fu) *fu += ((double)f[0] * (double)u0 + (double)f[1] * (double)u1) + (double)f[2] * (double)u2;
        return;
    }
    T KU[3], S[9];
    if (!ZS && (fl & NF_NEARFIX)) gs_node<T, C, true, Z0>(g, base, K, B, KU, S);
    else gs_node<T, C, false, Z0>(g, base, K, B, KU, S);
    T u[3];
    if constexpr (Z0) {
        u[0] = u[1] = u[2] = T(0);
    } else {
        u[0] = U.c[0][v]; u[1] = U.c[1][v]; u[2] = U.c[2][v];
    }
    // component-wise Gauss-Seidel with the 3x3 self block (Grid.cu:1056-1062)
    if (!reverse) {
        u[0] = gs_div<T>(f[0] - S[1] * u[1] - S[2] * u[2] - KU[0], S[0]);
        u[1] = gs_div<T>(f[1] - S[3] * u[0] - S[5] * u[2] - KU[1], S[4]);
        u[2] = gs_div<T>(f[2] - S[6] * u[0] - S[7] * u[1] - KU[2], S[8]);
    } else {
        u[2] = gs_div<T>(f[2] - S[6] * u[0] - S[7] * u[1] - KU[2], S[8]);
        u[1] = gs_div<T>(f[1] - S[3] * u[0] - S[5] * u[2] - KU[1], S[4]);
        u[0] = gs_div<T>(f[0] - S[1] * u[1] - S[2] * u[2] - KU[0], S[0]);
    }
    U.c[0][v] = u[0]; U.c[1][v] = u[1]; U.c[2][v] = u[2];
    if (fu) *fu += ((double)f[0] * (double)u[0] + (double)f[1] * (double)u[1]) + (double)f[2] * (double)u[2];
}

// Colours C and C^1 (same y, z parity, opposite x parity) couple only through
// the x-neighbours in the same row, so one workgroup owns a whole row
// (y, z) and relaxes its even-x nodes, then (after a barrier, which makes the
// new values visible to the block) its odd-x nodes; REV swaps the two.
// Every other neighbour belongs to a row of another colour pair and is
// read-only during the launch. Four launches make a sweep, in the reference's
// colour order 0..7 (or 7..0).
template <typename T, int C, bool ZS, bool Z0 = false>
__device__ __forceinline__ void gs_row_phase(const Geom& g, int j, int k, Vec3<T> U, Vec3<const T> F,
                                             const uint8_t* __restrict__ vflag, const KeC<T>& K, const GsBufs& B,
                                             bool reverse, double* fu = nullptr) {
    const int nhx = (g.n[0] - (C & 1) + 1) >> 1;
    const int rowbase = ((k + 1) * g.h[1] + (j + 1)) * g.h[0] + 1;
    for (int i = threadIdx.x; i < nhx; i += blockDim.x)
        gs_update<T, C, ZS, Z0>(g, rowbase + i, U, F, vflag, K, B, reverse, fu);
}

// sum of a double over the workgroup, valid in thread 0
__device__ __forceinline__ double gs_blk_sum(double v) {
    __shared__ double red[16];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    if (lane == 0) red[wid] = v;
    __syncthreads();
    double t = 0;
    if (threadIdx.x == 0)
        for (int i = 0; i < (int)((blockDim.x + 63) >> 6); i++) t += red[i];
    return t;
}

// optional occupancy target (waves per SIMD) for the smoother, a build-time knob
#if defined(RT_GS_WAVES_PER_EU) && RT_GS_WAVES_PER_EU > 0
#define RT_GS_ATTR __attribute__((amdgpu_waves_per_eu(RT_GS_WAVES_PER_EU)))
#else
#define RT_GS_ATTR
#endif

// DOT: partial sums of f . u_new over each workgroup's rows, one per workgroup
// in fu_part[blockIdx.x]
template <typename T, int CY, int CZ, bool REV, bool ZS, bool Z0 = false, bool DOT = false>
__global__ void __launch_bounds__(256) RT_GS_ATTR k_fine_gs_pair(Geom g, Vec3<T> U, Vec3<const T> F,
                                                      const float* __restrict__ rhop,
                                                      const uint8_t* __restrict__ vflag, KeC<T> K, int nrows, int bs,
                                                      double* __restrict__ fu_part = nullptr) {
    static_assert(!(Z0 && REV), "a zero-start sweep runs forward");
    at_batch(U, blockIdx.y, bs);
    at_batch(F, blockIdx.y, bs);
    double fu = 0;
    double* fup = DOT ? &fu : nullptr;
    const int nhy = (g.n[1] - CY + 1) >> 1;
    const int row = xcd_row(blockIdx.x, nrows);
    const int nbytes = g.N * (int)sizeof(T);
    const GsBufs B = {rsrc(U.c[0], nbytes), rsrc(U.c[1], nbytes), rsrc(U.c[2], nbytes), rsrc(rhop, g.N * 4),
                      rsrc(vflag, g.N)};
    constexpr int CA = (REV ? 1 : 0) | (CY << 1) | (CZ << 2);
    const int j = row % nhy, k = row / nhy;
    gs_row_phase<T, CA, ZS, Z0>(g, j, k, U, F, vflag, K, B, REV, fup);
    __syncthreads();
    gs_row_phase<T, CA ^ 1, ZS, Z0>(g, j, k, U, F, vflag, K, B, REV, fup);
    if constexpr (DOT) {
        const double t = gs_blk_sum(fu);
        if (threadIdx.x == 0) fu_part[blockIdx.x] = t;
    }
}

// ---------------------------------------------------------------------------
// The row kernel: k_fine_gs_pair's launch with both x parities of a thread's
// place in the row at once. A thread holds the nodes x = 2 i and 2 i + 1: of
// every other row they need the same four values per component, E(2i), E(2i+2)
// and O(2i-1), O(2i+1) (consecutive slots: two two-wide loads), and of the
// elements three values for four. All of that is read-only during the launch,
// so it is loaded and multiplied once, before the first parity is relaxed;
// only the own row's new values have to cross the barrier, through LDS.
//
// Against a pass per parity it issues 2 loads where that issued 4, reads the
// neighbour rows from the caches once instead of twice, and waits for memory
// once. Same arithmetic per node and the same order, so the same bits.
//
// Bound: VALU issue (at 511 x 256 x 256 elements 0.60 of a sweep's 0.79 ms, 0.48 of
// it the 555 FMA a node) with the latency of the row loads, which 4 waves per SIMD
// hide in part; the pass per parity was bound by its traffic beyond L2, 1.59 GB a
// launch against 0.82 now. Measured, ms per FP32 sweep: 511 x 256 x 256 1.03 -> 0.79, 256 x
// 128 x 128 0.156 -> 0.130, 128 x 64 x 64 0.041 -> 0.037; FP64 1.66 -> 1.20,
// 0.195 -> 0.178, 0.049 -> 0.045. A spilled register or a fifth wave of one
// lane (see row_shape) costs all of that: 5 waves per SIMD with 7 spilled
// registers 1.23, a workgroup of 257 threads 0.96.
// ---------------------------------------------------------------------------
// a point that no load and no term of the sums moves across (the sums pass
// through it; it emits nothing)
template <typename T>
__device__ __forceinline__ void row_fence(T (&aE)[8][3], T (&aO)[8][3]) {
#pragma unroll
    for (int w = 0; w < 8; w++)
        asm volatile("" : "+v"(aE[w][0]), "+v"(aE[w][1]), "+v"(aE[w][2]), "+v"(aO[w][0]), "+v"(aO[w][1]), "+v"(aO[w][2])
                     : : "memory");
}

template <typename T> struct RowVals {
    Two<T> e[3], o[3];
    uint8_t fl[4];          // CHECK_FIX: flags of e.lo, e.hi, o.lo, o.hi
};

// whether the rows (DY, DZ) still hold 0 in a zero-start sweep (both colours of
// a row come later than both of the pair, or neither)
template <int CE, int ROW, bool Z0>
constexpr bool row_used() { return !(Z0 && nb_colour<CE, 0, ROW % 3 - 1, ROW / 3 - 1>() > CE); }

template <typename T, int CE, bool CHECK_FIX, int ROW, bool Z0>
__device__ __forceinline__ void row_load(const Geom& g, int vb, const GsBufs& B, RowVals<T>& v) {
    if constexpr (row_used<CE, ROW, Z0>()) {
        constexpr int DY = ROW % 3 - 1, DZ = ROW / 3 - 1;
        const int vo = vb * (int)sizeof(T);
        const int se = rel_off<CE, 0, DY, DZ>(g), so = rel_off<CE, -1, DY, DZ>(g);
        const __amdgpu_buffer_rsrc_t u[3] = {B.u0, B.u1, B.u2};
#pragma unroll
        for (int c = 0; c < 3; c++) {
            v.e[c] = bload2<T>(u[c], vo, se * (int)sizeof(T));
            v.o[c] = bload2<T>(u[c], vo, so * (int)sizeof(T));
        }
        if constexpr (CHECK_FIX) {
            v.fl[0] = bload_u8(B.flag, vb, se); v.fl[1] = bload_u8(B.flag, vb, se + 1);
            v.fl[2] = bload_u8(B.flag, vb, so); v.fl[3] = bload_u8(B.flag, vb, so + 1);
        }
    }
}

template <typename T, int CE, bool CHECK_FIX, int ROW, bool Z0>
__device__ __forceinline__ void row_use(const KeC<T>& K, RowVals<T>& v, T (&aE)[8][3], T (&aO)[8][3]) {
    if constexpr (row_used<CE, ROW, Z0>()) {
        constexpr int NBM = 9 * (ROW / 3) + 3 * (ROW % 3);   // dx = -1; dx = 0, +1 follow
        if constexpr (CHECK_FIX) {
#pragma unroll
            for (int c = 0; c < 3; c++) {
                if (v.fl[0] & NF_FIXED) v.e[c].lo = T(0);
                if (v.fl[1] & NF_FIXED) v.e[c].hi = T(0);
                if (v.fl[2] & NF_FIXED) v.o[c].lo = T(0);
                if (v.fl[3] & NF_FIXED) v.o[c].hi = T(0);
            }
        }
        const auto ws = std::make_integer_sequence<int, 8>{};
        nb_elems<T, NBM>(aE, K, v.o[0].lo, v.o[1].lo, v.o[2].lo, ws);
        nb_elems<T, NBM + 2>(aE, K, v.o[0].hi, v.o[1].hi, v.o[2].hi, ws);
        nb_elems<T, NBM + 1>(aE, K, v.e[0].lo, v.e[1].lo, v.e[2].lo, ws);
        nb_elems<T, NBM>(aO, K, v.e[0].lo, v.e[1].lo, v.e[2].lo, ws);
        nb_elems<T, NBM + 2>(aO, K, v.e[0].hi, v.e[1].hi, v.e[2].hi, ws);
        nb_elems<T, NBM + 1>(aO, K, v.o[0].hi, v.o[1].hi, v.o[2].hi, ws);
    }
}

// the eight rows besides the own one, in RowOrder: the values of a row are
// loaded kRowAhead rows before they are multiplied (the fences keep it at
// that: the compiler would otherwise start all of them at once and spill), and
// `last` issues the loads that the node updates need before the last row
template <typename T> constexpr int kRowAhead = sizeof(T) == 4 ? 1 : 2;
constexpr int row_at(int i) { return i < 4 ? i : i + 1; }

template <typename T, int CE, bool CHECK_FIX, bool Z0, int I, typename L>
__device__ __forceinline__ void pair_rows(const Geom& g, int vb, const KeC<T>& K, const GsBufs& B,
                                          RowVals<T> (&v)[kRowAhead<T> + 1], T (&aE)[8][3], T (&aO)[8][3], L&& last) {
    if constexpr (I + kRowAhead<T> < 8)
        row_load<T, CE, CHECK_FIX, row_at(I + kRowAhead<T>), Z0>(g, vb, B, v[(I + kRowAhead<T>) % (kRowAhead<T> + 1)]);
    if constexpr (I == 7) last();
    row_fence(aE, aO);
    row_use<T, CE, CHECK_FIX, row_at(I), Z0>(K, v[I % (kRowAhead<T> + 1)], aE, aO);
    if constexpr (I < 7) {
        row_fence(aE, aO);
        pair_rows<T, CE, CHECK_FIX, Z0, I + 1>(g, vb, K, B, v, aE, aO, last);
    }
}

// the old values of the own row's neighbours of the parity relaxed first (REV:
// the odd node), added to its sums
template <typename T, int CE, bool CHECK_FIX, bool REV>
__device__ __forceinline__ void own_load(const Geom& g, int vb, const GsBufs& B, RowVals<T>& v) {
    const int vo = vb * (int)sizeof(T);
    const int s = REV ? rel_off<CE, 0, 0, 0>(g) : rel_off<CE, -1, 0, 0>(g), sb = s * (int)sizeof(T);
    v.e[0] = bload2<T>(B.u0, vo, sb);
    v.e[1] = bload2<T>(B.u1, vo, sb);
    v.e[2] = bload2<T>(B.u2, vo, sb);
    if constexpr (CHECK_FIX) {
        v.fl[0] = bload_u8(B.flag, vb, s); v.fl[1] = bload_u8(B.flag, vb, s + 1);
    }
}
template <typename T, bool CHECK_FIX>
__device__ __forceinline__ void own_use(const KeC<T>& K, RowVals<T>& v, T (&a)[8][3]) {
    if constexpr (CHECK_FIX) {
#pragma unroll
        for (int c = 0; c < 3; c++) {
            if (v.fl[0] & NF_FIXED) v.e[c].lo = T(0);
            if (v.fl[1] & NF_FIXED) v.e[c].hi = T(0);
        }
    }
    nb_elems<T, 12>(a, K, v.e[0].lo, v.e[1].lo, v.e[2].lo, std::make_integer_sequence<int, 8>{});
    nb_elems<T, 14>(a, K, v.e[0].hi, v.e[1].hi, v.e[2].hi, std::make_integer_sequence<int, 8>{});
}

template <typename T, int W>
__device__ __forceinline__ void pair_elem(const KeC<T>& K, T pen, const T (&acc)[8][3], T (&KU)[3], T (&S)[9]) {
    constexpr int vi = 7 - W;
    KU[0] += pen * acc[W][0];
    KU[1] += pen * acc[W][1];
    KU[2] += pen * acc[W][2];
    S[0] += pen * kc<ke_code_at((3 * vi + 0) * 24 + 3 * vi + 0)>(K);
    S[1] += pen * kc<ke_code_at((3 * vi + 0) * 24 + 3 * vi + 1)>(K);
    S[2] += pen * kc<ke_code_at((3 * vi + 0) * 24 + 3 * vi + 2)>(K);
    S[3] += pen * kc<ke_code_at((3 * vi + 1) * 24 + 3 * vi + 0)>(K);
    S[4] += pen * kc<ke_code_at((3 * vi + 1) * 24 + 3 * vi + 1)>(K);
    S[5] += pen * kc<ke_code_at((3 * vi + 1) * 24 + 3 * vi + 2)>(K);
    S[6] += pen * kc<ke_code_at((3 * vi + 2) * 24 + 3 * vi + 0)>(K);
    S[7] += pen * kc<ke_code_at((3 * vi + 2) * 24 + 3 * vi + 1)>(K);
    S[8] += pen * kc<ke_code_at((3 * vi + 2) * 24 + 3 * vi + 2)>(K);
}
template <typename T, int... Ws>
__device__ __forceinline__ void pair_elems(const KeC<T>& K, const float (&pen)[8], const T (&acc)[8][3], T (&KU)[3],
                                           T (&S)[9], std::integer_sequence<int, Ws...>) {
    (pair_elem<T, Ws>(K, (T)pen[Ws], acc, KU, S), ...);
}

// the update of gs_update from the sums; u: the node's old value in, its new one out
template <typename T, bool REV>
__device__ __forceinline__ void pair_relax(uint8_t fl, const T (&f)[3], const KeC<T>& K, const float (&pen)[8],
                                           const T (&acc)[8][3], T (&u)[3]) {
    if (fl & NF_FIXED) {
        const T ne = (T)(fl >> 4);
        u[0] = f[0] / ne; u[1] = f[1] / ne; u[2] = f[2] / ne;
        return;
    }
    T KU[3] = {T(0), T(0), T(0)}, S[9];
#pragma unroll
    for (int i = 0; i < 9; i++) S[i] = T(0);
    pair_elems<T>(K, pen, acc, KU, S, std::make_integer_sequence<int, 8>{});
    if (!REV) {
        u[0] = gs_div<T>(f[0] - S[1] * u[1] - S[2] * u[2] - KU[0], S[0]);
        u[1] = gs_div<T>(f[1] - S[3] * u[0] - S[5] * u[2] - KU[1], S[4]);
        u[2] = gs_div<T>(f[2] - S[6] * u[0] - S[7] * u[1] - KU[2], S[8]);
    } else {
        u[2] = gs_div<T>(f[2] - S[6] * u[0] - S[7] * u[1] - KU[2], S[8]);
        u[1] = gs_div<T>(f[1] - S[3] * u[0] - S[5] * u[2] - KU[1], S[4]);
        u[0] = gs_div<T>(f[0] - S[1] * u[1] - S[2] * u[2] - KU[0], S[0]);
    }
}

// threads of the row kernel's largest workgroup, and the waves per SIMD that
// its registers (a pair has 48 sums) are kept down to
constexpr int kRowThreads = 512;
template <typename T> constexpr int kRowWaves = sizeof(T) == 4 ? 4 : 2;

template <typename T, int CY, int CZ, bool REV, bool ZS, bool Z0 = false, bool DOT = false>
__global__ void __launch_bounds__(kRowThreads) __attribute__((amdgpu_waves_per_eu(kRowWaves<T>)))
k_fine_gs_row(Geom g, Vec3<T> U, Vec3<const T> F, const float* __restrict__ rhop, const uint8_t* __restrict__ vflag,
              KeC<T> K, int nrows, int rpw, int npr, int bs, double* __restrict__ fu_part) {
    static_assert(!(Z0 && REV), "a zero-start sweep runs forward");
    at_batch(U, blockIdx.y, bs);
    at_batch(F, blockIdx.y, bs);
    constexpr int CE = (CY << 1) | (CZ << 2);
    __shared__ T sh[3][kRowThreads];         // new values of the parity relaxed first
    const int nhy = (g.n[1] - CY + 1) >> 1;
    // thread t: pair i of the workgroup's row r; the last pair's thread also
    // relaxes the row's last even node where that has no thread (row_shape)
    const int t = threadIdx.x, r = t / npr, i = t - r * npr;
    const int row = xcd_row(blockIdx.x, gridDim.x) * rpw + r;
    const bool in = r < rpw && row < nrows;
    const int j = in ? row % nhy : 0, k = in ? row / nhy : 0;
    const int nbytes = g.N * (int)sizeof(T);
    const GsBufs B = {rsrc(U.c[0], nbytes), rsrc(U.c[1], nbytes), rsrc(U.c[2], nbytes), rsrc(rhop, g.N * 4),
                      rsrc(vflag, g.N)};
    const int base = ((k + 1) * g.h[1] + (j + 1)) * g.h[0] + 1 + i;
    const int vb = base - g.h[0] * g.h[1] - g.h[0] - 1;
    const int vE = CE * g.cs + base, vO = vE + g.cs;
    const bool inO = in && 2 * i + 1 < g.n[0], extra = in && i == npr - 1 && 2 * npr < g.n[0];
    const uint8_t flE = in ? vflag[vE] : 0, flO = inO ? vflag[vO] : 0;
    T aE[8][3], aO[8][3], fE[3], fO[3], uE[3], uO[3];
    float pE[8], pO[8];
    double fu = 0;
    auto store = [&](int v, const T (&f)[3], const T (&u)[3]) __attribute__((always_inline)) {
        U.c[0][v] = u[0]; U.c[1][v] = u[1]; U.c[2][v] = u[2];
        if constexpr (DOT) fu += ((double)f[0] * (double)u[0] + (double)f[1] * (double)u[1]) + (double)f[2] * (double)u[2];
    };
    T first[3] = {T(0), T(0), T(0)}, beyond[3] = {T(0), T(0), T(0)};
    if (!REV && extra) {
        gs_update<T, CE, ZS, Z0>(g, base + 1, U, F, vflag, K, B, REV, DOT ? &fu : nullptr);
        if (ZS || !(vflag[vE + 1] & NF_FIXED)) {
            beyond[0] = U.c[0][vE + 1]; beyond[1] = U.c[1][vE + 1]; beyond[2] = U.c[2][vE + 1];
        }
    }
    // the first rows are on their way before the flags are looked at
    RowVals<T> v[kRowAhead<T> + 1];
    auto load_first = [&](auto check) __attribute__((always_inline)) {
        constexpr bool CHECK = decltype(check)::value;
        row_load<T, CE, CHECK, 0, Z0>(g, vb, B, v[0]);
        if constexpr (kRowAhead<T> > 1) row_load<T, CE, CHECK, 1, Z0>(g, vb, B, v[1]);
    };
    if (in) load_first(std::false_type{});
    asm volatile("" ::: "memory");
    const bool actE = flE & NF_ACTIVE, actO = flO & NF_ACTIVE;
    if (actE || actO) {
        // rho^p: the even node's elements are O(i), E(i + 1), the odd one's E(i + 1), O(i + 1)
        auto pens = [&](auto r) __attribute__((always_inline)) {
            constexpr int EY = (decltype(r)::value & 1) - 1, EZ = (decltype(r)::value >> 1) - 1;
            constexpr int w = 2 * (EY + 1) + 4 * (EZ + 1);
            const Two<float> o = bload2<float>(B.rho, vb * 4, rel_off<CE, -1, EY, EZ>(g) * 4);
            const float e = bload<float>(B.rho, vb * 4, rel_off<CE, 0, EY, EZ>(g) * 4);
            pE[w] = o.lo; pE[w + 1] = e; pO[w] = e; pO[w + 1] = o.hi;
        };
        auto node_values = [&]() __attribute__((always_inline)) {
            pens(std::integral_constant<int, 0>{});
            pens(std::integral_constant<int, 1>{});
            pens(std::integral_constant<int, 2>{});
            pens(std::integral_constant<int, 3>{});
#pragma unroll
            for (int c = 0; c < 3; c++) {
                fE[c] = F.c[c][vE]; fO[c] = F.c[c][vO];
                uE[c] = Z0 ? T(0) : U.c[c][vE]; uO[c] = Z0 ? T(0) : U.c[c][vO];
            }
        };
        auto sums = [&](auto check) __attribute__((always_inline)) {
            constexpr bool CHECK = decltype(check)::value;
            RowVals<T> own;
            if constexpr (CHECK) load_first(check);
#pragma unroll
            for (int w = 0; w < 8; w++)
#pragma unroll
                for (int c = 0; c < 3; c++) aE[w][c] = aO[w][c] = T(0);
            pair_rows<T, CE, CHECK, Z0, 0>(g, vb, K, B, v, aE, aO, [&]() __attribute__((always_inline)) {
                if constexpr (!Z0) own_load<T, CE, CHECK, REV>(g, vb, B, own);
                node_values();
            });
            if constexpr (!Z0) own_use<T, CHECK>(K, own, REV ? aO : aE);
        };
        if (!ZS && ((flE | flO) & NF_NEARFIX)) sums(std::true_type{});
        else sums(std::false_type{});
        if constexpr (REV) {
            pair_relax<T, REV>(flO, fO, K, pO, aO, uO);
            if (actO) store(vO, fO, uO);
        } else {
            pair_relax<T, REV>(flE, fE, K, pE, aE, uE);
            if (actE) store(vE, fE, uE);
        }
        // a support counts as 0 for its neighbours
        const uint8_t fl = REV ? flO : flE;
        const bool live = (fl & NF_ACTIVE) && (ZS || !(fl & NF_FIXED));
#pragma unroll
        for (int c = 0; c < 3; c++) first[c] = live ? (REV ? uO[c] : uE[c]) : T(0);
    }
#pragma unroll
    for (int c = 0; c < 3; c++) sh[c][t] = first[c];
    __syncthreads();
    if (REV ? actE : actO) {
        T (&a)[8][3] = REV ? aE : aO;
        // the neighbour pair's value; past the row's ends the extra node's, or the ghost slots' 0
        const bool end = REV ? i == 0 : i == npr - 1;
        const int to = end ? t : REV ? t - 1 : t + 1;
        const T other[3] = {end ? beyond[0] : sh[0][to], end ? beyond[1] : sh[1][to], end ? beyond[2] : sh[2][to]};
        const T l[3] = {REV ? other[0] : first[0], REV ? other[1] : first[1], REV ? other[2] : first[2]};
        const T rr[3] = {REV ? first[0] : other[0], REV ? first[1] : other[1], REV ? first[2] : other[2]};
        nb_elems<T, 12>(a, K, l[0], l[1], l[2], std::make_integer_sequence<int, 8>{});
        nb_elems<T, 14>(a, K, rr[0], rr[1], rr[2], std::make_integer_sequence<int, 8>{});
        if constexpr (REV) {
            pair_relax<T, REV>(flE, fE, K, pE, aE, uE);
            store(vE, fE, uE);
        } else {
            pair_relax<T, REV>(flO, fO, K, pO, aO, uO);
            store(vO, fO, uO);
        }
    }
    if (REV && extra) gs_update<T, CE, ZS, Z0>(g, base + 1, U, F, vflag, K, B, REV, DOT ? &fu : nullptr);
    if constexpr (Z0) {   // what a cleared vector would hold
        if (!actE && in) { U.c[0][vE] = T(0); U.c[1][vE] = T(0); U.c[2][vE] = T(0); }
        if (!actO && inO) { U.c[0][vO] = T(0); U.c[1][vO] = T(0); U.c[2][vO] = T(0); }
    }
    if constexpr (DOT) {
        const double t = gs_blk_sum(fu);
        if (threadIdx.x == 0) fu_part[blockIdx.x] = t;
    }
}

// ---------------------------------------------------------------------------
// Tiled sweep: two launches per sweep instead of four, reading the old values
// from Uin and writing the new ones to Uout (a second buffer).
//
// In the reference's colour order all colours of the z-parity class relaxed
// first (z even forward, z odd in reverse) come before any colour of the other
// class, and planes of one class never neighbour each other. So a launch
// relaxes the four colours of one class, plane by plane, and a workgroup owns a
// tile of TR whole rows (all x) of one plane. Inside the tile the four colours
// follow the sweep order with a barrier between them; a neighbour in the same
// plane is new (read from Uout, written earlier by this workgroup) if its
// colour comes earlier, old (read from Uin) otherwise; a neighbour in the other
// z class is old in the first launch and new (Uout, written by the first
// launch) in the second. The second pair of colours of the plane (the "lag"
// rows, y parity relaxed last) needs the new values of the first pair on the
// rows on either side, so the first pair is also relaxed on the one row of the
// next tile it needs (below the tile in reverse order, above it forward). That
// row is computed from the same values and with the same arithmetic as its
// owner computes it, so both write identical bits. Uin is never written, so
// the result does not depend on the order in which workgroups run, and each
// node gets exactly the value of the colour-pair sweep above.
// ---------------------------------------------------------------------------
struct GsBufs2 {
    __amdgpu_buffer_rsrc_t in0, in1, in2, out0, out1, out2, rho, flag;
};

// whether the neighbour at (DX, DY, DZ) of a colour-C node already holds its
// new value when the node is relaxed (FIRST: this launch relaxes the first z
// class of the sweep; REV: reverse colour order)
template <int C, int DX, int DY, int DZ, bool FIRST, bool REV>
constexpr bool nb_is_new() {
    if constexpr (DZ != 0) {
        return !FIRST;
    } else {
        constexpr int cn = C ^ ((DX & 1) | ((DY & 1) << 1));
        constexpr int o = ((C >> 1) & 1) * 2 + (C & 1), on = ((cn >> 1) & 1) * 2 + (cn & 1);
        return REV ? (on > o) : (on < o);
    }
}

template <typename T, int C, bool CHECK_FIX, int NB, bool FIRST, bool REV>
__device__ __forceinline__ void nb_step2(const Geom& g, int vb, const KeC<T>& K, const GsBufs2& B, T (&acc)[8][3]) {
    if constexpr (NB != 13) {
        constexpr int DX = NB % 3 - 1, DY = NB / 3 % 3 - 1, DZ = NB / 9 - 1;
        constexpr bool NW = nb_is_new<C, DX, DY, DZ, FIRST, REV>();
        const int so = rel_off<C, DX, DY, DZ>(g);
        const int vo = vb * (int)sizeof(T), sob = so * (int)sizeof(T);
        T u0 = bload<T>(NW ? B.out0 : B.in0, vo, sob);
        T u1 = bload<T>(NW ? B.out1 : B.in1, vo, sob);
        T u2 = bload<T>(NW ? B.out2 : B.in2, vo, sob);
        if constexpr (CHECK_FIX) {
            if (bload_u8(B.flag, vb, so) & NF_FIXED) { u0 = T(0); u1 = T(0); u2 = T(0); }
        }
        nb_elems<T, NB>(acc, K, u0, u1, u2, std::make_integer_sequence<int, 8>{});
    }
}

template <typename T, int C, bool CHECK_FIX, int ROW, bool FIRST, bool REV>
__device__ __forceinline__ void nb_row2(const Geom& g, int vb, const KeC<T>& K, const GsBufs2& B, T (&acc)[8][3]) {
    constexpr int DY = ROW % 3 - 1, DZ = ROW / 3 - 1;
    constexpr int NBM = 9 * (DZ + 1) + 3 * (DY + 1);
    constexpr bool NW = nb_is_new<C, -1, DY, DZ, FIRST, REV>();   // dx = -1 and +1 share a colour
    const int vo = vb * (int)sizeof(T);
    {
        const int so = rel_off<C, -1, DY, DZ>(g), sob = so * (int)sizeof(T);
        const Two<T> a = bload2<T>(NW ? B.out0 : B.in0, vo, sob), b = bload2<T>(NW ? B.out1 : B.in1, vo, sob),
                     c = bload2<T>(NW ? B.out2 : B.in2, vo, sob);
        T l0 = a.lo, l1 = b.lo, l2 = c.lo, r0 = a.hi, r1 = b.hi, r2 = c.hi;
        if constexpr (CHECK_FIX) {
            if (bload_u8(B.flag, vb, so) & NF_FIXED) { l0 = T(0); l1 = T(0); l2 = T(0); }
            if (bload_u8(B.flag, vb, so + 1) & NF_FIXED) { r0 = T(0); r1 = T(0); r2 = T(0); }
        }
        nb_elems<T, NBM>(acc, K, l0, l1, l2, std::make_integer_sequence<int, 8>{});
        nb_elems<T, NBM + 2>(acc, K, r0, r1, r2, std::make_integer_sequence<int, 8>{});
    }
    nb_step2<T, C, CHECK_FIX, NBM + 1, FIRST, REV>(g, vb, K, B, acc);
}

template <typename T, int C, bool CHECK_FIX, bool FIRST, bool REV, int... ROWs>
__device__ __forceinline__ void nb_all2(const Geom& g, int vb, const KeC<T>& K, const GsBufs2& B, T (&acc)[8][3],
                                        std::integer_sequence<int, ROWs...>) {
    (nb_row2<T, C, CHECK_FIX, ROWs, FIRST, REV>(g, vb, K, B, acc), ...);
}

template <typename T, int C, bool CHECK_FIX, bool FIRST, bool REV>
__device__ __forceinline__ void gs_node2(const Geom& g, int base, const KeC<T>& K, const GsBufs2& B, T KU[3],
                                         T S[9]) {
    const int vb = base - g.h[0] * g.h[1] - g.h[0] - 1;
    T acc[8][3];
#pragma unroll
    for (int w = 0; w < 8; w++) acc[w][0] = acc[w][1] = acc[w][2] = T(0);
    nb_all2<T, C, CHECK_FIX, FIRST, REV>(g, vb, K, B, acc, RowOrder{});
    KU[0] = KU[1] = KU[2] = T(0);
#pragma unroll
    for (int i = 0; i < 9; i++) S[i] = T(0);
    const GsBufs Be = {B.in0, B.in1, B.in2, B.rho, B.flag};
    elem_all<T, C>(g, vb, K, Be, acc, KU, S, std::make_integer_sequence<int, 8>{});
}

// the GS update of gs_update, old values from Uin, the result to Uout
template <typename T, int C, bool ZS, bool FIRST, bool REV>
__device__ __forceinline__ void gs_update2(const Geom& g, int base, Vec3<const T> Uin, Vec3<T> Uout, Vec3<const T> F,
                                           const uint8_t* __restrict__ vflag, const KeC<T>& K, const GsBufs2& B) {
    const int v = C * g.cs + base;
    const uint8_t fl = vflag[v];
    if (!(fl & NF_ACTIVE)) return;
    const T f[3] = {F.c[0][v], F.c[1][v], F.c[2][v]};
    if (fl & NF_FIXED) {
        const T ne = (T)(fl >> 4);
        Uout.c[0][v] = f[0] / ne; Uout.c[1][v] = f[1] / ne; Uout.c[2][v] = f[2] / ne;
        return;
    }
    T KU[3], S[9];
    if (!ZS && (fl & NF_NEARFIX)) gs_node2<T, C, true, FIRST, REV>(g, base, K, B, KU, S);
    else gs_node2<T, C, false, FIRST, REV>(g, base, K, B, KU, S);
    T u[3] = {Uin.c[0][v], Uin.c[1][v], Uin.c[2][v]};
    if (!REV) {
        u[0] = gs_div<T>(f[0] - S[1] * u[1] - S[2] * u[2] - KU[0], S[0]);
        u[1] = gs_div<T>(f[1] - S[3] * u[0] - S[5] * u[2] - KU[1], S[4]);
        u[2] = gs_div<T>(f[2] - S[6] * u[0] - S[7] * u[1] - KU[2], S[8]);
    } else {
        u[2] = gs_div<T>(f[2] - S[6] * u[0] - S[7] * u[1] - KU[2], S[8]);
        u[1] = gs_div<T>(f[1] - S[3] * u[0] - S[5] * u[2] - KU[1], S[4]);
        u[0] = gs_div<T>(f[0] - S[1] * u[1] - S[2] * u[2] - KU[0], S[0]);
    }
    Uout.c[0][v] = u[0]; Uout.c[1][v] = u[1]; Uout.c[2][v] = u[2];
}

// colour-C nodes of the rows y in [ya, yb) (clipped to the box) of plane
// half-index k, spread over the workgroup
template <typename T, int C, bool ZS, bool FIRST, bool REV>
__device__ __forceinline__ void tile_phase(const Geom& g, int k, int ya, int yb, Vec3<const T> Uin, Vec3<T> Uout,
                                           Vec3<const T> F, const uint8_t* __restrict__ vflag, const KeC<T>& K,
                                           const GsBufs2& B) {
    constexpr int cx = C & 1, cy = (C >> 1) & 1;
    const int nhx = (g.n[0] - cx + 1) >> 1, nhy = (g.n[1] - cy + 1) >> 1;
    const int jlo = max(0, (ya - cy + 1) >> 1), jhi = min(nhy, (yb - cy + 1) >> 1);
    const int cnt = (jhi - jlo) * nhx;
    for (int t = threadIdx.x; t < cnt; t += blockDim.x) {
        const int j = jlo + t / nhx, i = t % nhx;
        gs_update2<T, C, ZS, FIRST, REV>(g, ((k + 1) * g.h[1] + (j + 1)) * g.h[0] + (i + 1), Uin, Uout, F, vflag, K,
                                         B);
    }
}

// rows per tile. Measured at 511 x 256 x 256 elements (ms per sweep, against
// 1.06 for the colour-pair launches): 4 rows 1.41, 8 rows 1.38, 16 rows 1.44,
// 32 rows 1.56; tiles ordered y-fastest instead of plane-fastest 1.50. Fewer,
// longer-lived workgroups with three barriers each hide memory latency worse
// than the colour-pair launches' one row per workgroup, although they move
// less data, so this sweep is not the default.
#ifndef RT_GS_TILE_ROWS
#define RT_GS_TILE_ROWS 8
#endif

template <typename T, int CZ, bool REV, bool ZS>
__global__ void __launch_bounds__(256) k_fine_gs_tile(Geom g, Vec3<const T> Uin, Vec3<T> Uout, Vec3<const T> F,
                                                      const float* __restrict__ rhop,
                                                      const uint8_t* __restrict__ vflag, KeC<T> K, int nplanes) {
    constexpr bool FIRST = CZ == (REV ? 1 : 0);
    constexpr int TR = RT_GS_TILE_ROWS;
    static_assert(TR % 2 == 0, "tiles start on even rows");
    // planes fastest, so that the tiles sharing the other class's planes in
    // between run close together on one XCD
    const int b = xcd_row(blockIdx.x, gridDim.x);
    const int k = b % nplanes, ty = b / nplanes;
    const int ny = g.n[1];
    const int y0 = ty * TR, y1 = min(y0 + TR, ny);
    const int nbytes = g.N * (int)sizeof(T);
    const GsBufs2 B = {rsrc(Uin.c[0], nbytes),  rsrc(Uin.c[1], nbytes),  rsrc(Uin.c[2], nbytes),
                       rsrc(Uout.c[0], nbytes), rsrc(Uout.c[1], nbytes), rsrc(Uout.c[2], nbytes),
                       rsrc(rhop, g.N * 4),     rsrc(vflag, g.N)};
    // lead rows (the y parity relaxed first) with the one extra row the lag rows need
    const int la = REV ? y0 - 1 : y0, lb = REV ? y1 : y1 + 1;
    constexpr int Z = CZ << 2;
    if constexpr (!REV) {
        tile_phase<T, Z | 0, ZS, FIRST, REV>(g, k, la, lb, Uin, Uout, F, vflag, K, B);
        __syncthreads();
        tile_phase<T, Z | 1, ZS, FIRST, REV>(g, k, la, lb, Uin, Uout, F, vflag, K, B);
        __syncthreads();
        tile_phase<T, Z | 2, ZS, FIRST, REV>(g, k, y0, y1, Uin, Uout, F, vflag, K, B);
        __syncthreads();
        tile_phase<T, Z | 3, ZS, FIRST, REV>(g, k, y0, y1, Uin, Uout, F, vflag, K, B);
    } else {
        tile_phase<T, Z | 3, ZS, FIRST, REV>(g, k, la, lb, Uin, Uout, F, vflag, K, B);
        __syncthreads();
        tile_phase<T, Z | 2, ZS, FIRST, REV>(g, k, la, lb, Uin, Uout, F, vflag, K, B);
        __syncthreads();
        tile_phase<T, Z | 1, ZS, FIRST, REV>(g, k, y0, y1, Uin, Uout, F, vflag, K, B);
        __syncthreads();
        tile_phase<T, Z | 0, ZS, FIRST, REV>(g, k, y0, y1, Uin, Uout, F, vflag, K, B);
    }
}

// one full sweep (colours 0..7, or 7..0 when reverse) from Uin to Uout
template <typename T>
void launch_fine_gs_sweep2(const Geom& g, Vec3<const T> Uin, Vec3<T> Uout, Vec3<const T> F, const float* rhop,
                           const uint8_t* vflag, bool reverse, bool zero_support, hipStream_t s) {
    check_buffer_range<T>(g);
    const KeC<T> K = kec<T>();
    const int ntile = (g.n[1] + RT_GS_TILE_ROWS - 1) / RT_GS_TILE_ROWS;
    for (int pass = 0; pass < 2; pass++) {
        const int cz = reverse ? 1 - pass : pass;
        const int nplanes = (g.n[2] - cz + 1) >> 1;
        if (nplanes <= 0) continue;
        dim3 grid((unsigned)(nplanes * ntile));
        switch (cz * 4 + (reverse ? 2 : 0) + (zero_support ? 1 : 0)) {
#define RT_CASE(c, r, z) case c * 4 + r * 2 + z: hipLaunchKernelGGL((k_fine_gs_tile<T, c, (r) != 0, (z) != 0>), grid, dim3(256), 0, s, g, Uin, Uout, F, rhop, vflag, K, nplanes); break;
            RT_CASE(0, 0, 0) RT_CASE(0, 0, 1) RT_CASE(0, 1, 0) RT_CASE(0, 1, 1)
            RT_CASE(1, 0, 0) RT_CASE(1, 0, 1) RT_CASE(1, 1, 0) RT_CASE(1, 1, 1)
#undef RT_CASE
        }
        RT_HIP(hipGetLastError());
    }
}

template void launch_fine_gs_sweep2<float>(const Geom&, Vec3<const float>, Vec3<float>, Vec3<const float>,
                                           const float*, const uint8_t*, bool, bool, hipStream_t);
template void launch_fine_gs_sweep2<double>(const Geom&, Vec3<const double>, Vec3<double>, Vec3<const double>,
                                            const float*, const uint8_t*, bool, bool, hipStream_t);

// the row kernel's workgroup for a launch of `rows` rows (of all its vectors): rpw
// whole rows of npr pairs in nt threads, or rpw = 0 where the pair kernel takes the
// launch: rows too long for a workgroup, and FP64 rows of five waves, which leave
// three of a CU's eight wave slots empty (520 x 72 x 72 elements: 228 us a sweep, 192
// by the pair kernel, 544 x 80 x 80 242 and 212; with nearly full lanes the two are
// close: 600 x 64 x 64 141 and 142, 600 x 128 x 128 525 and 551).
// Boxes are a multiple of the coarsest spacing plus one node long, so a row's pairs
// often pass a multiple of 64 by one. The last pair's thread then takes the even
// node left over as well where that puts more workgroups on a CU (row_fit): after
// two, four or eight whole waves, and one or (FP32) three (512 x 96 x 96 elements:
// 125 us a sweep, 164 with a wave of one lane; FP64 195 and 272). Where it does not,
// it only lengthens the chain: 640 x 96 x 96 219 against 182 us, FP64 393 and 301, and
// FP64 at 384 x 128 x 128 315 and 285; the same in launches that do not fill the
// chip (128 x 64 x 64: 42.7 against 36.5 us). Other lengths put several rows into a
// workgroup if that fills its lanes better and enough workgroups remain.
struct RowShape { int rpw, nt, npr; };
// workgroups of w waves that a CU holds: up to four waves of one share the wave
// slots freely, more are placed evenly over the four SIMDs
template <typename T> static int row_fit(int w) { return 4 * kRowWaves<T> / (w <= 4 ? w : (w + 3) / 4 * 4); }
template <typename T>
static RowShape row_shape(const Geom& g, long long rows) {
    const int nxe = (g.n[0] + 1) / 2, w = nxe / 64;
    if (w > 0 && nxe % 64 == 1 && nxe - 1 <= kRowThreads && row_fit<T>(w) > row_fit<T>(w + 1) && rows * (w + 1) > 4096)
        return RowShape{1, nxe - 1, nxe - 1};
    RowShape best{0, 0, nxe};
    double eff = 0;
    for (int rpw = 1; rpw <= 8 && rpw * nxe <= kRowThreads; rpw++) {
        if (rpw > 1 && rows / rpw < 1024) break;
        const int nt = (rpw * nxe + 63) / 64 * 64;
        if (sizeof(T) == 8 && nt == 5 * 64) continue;
        const double e = (double)(rpw * nxe) / nt;
        if (e > eff * 1.05) {
            eff = e;
            best.rpw = rpw;
            best.nt = nt;
        }
    }
    return best;
}

// pair p = 0..3 relaxes colours (2p, 2p+1), or (2p+1, 2p) when reverse
// zero_start: the first forward sweep from u = 0 (with zero supports); U may
// hold anything on entry, and every slot the sweep visits is written
// workgroups of one colour-pair launch (the partials a fu launch writes)
int fine_gs_pair_blocks(const Geom& g, int pair) {
    const int cy = pair & 1, cz = pair >> 1;
    const long long rows = (long long)((g.n[1] - cy + 1) >> 1) * ((g.n[2] - cz + 1) >> 1);
    if (rows <= 0) return 0;
    const RowShape w = row_shape<float>(g, rows);
    return (int)(w.rpw ? (rows + w.rpw - 1) / w.rpw : rows);
}

template <typename T>
void launch_fine_gs(const Geom& g, Vec3<T> U, Vec3<const T> F, const float* rhop, const uint8_t* vflag, int pair,
                    bool reverse, bool zero_support, hipStream_t s, bool zero_start, double* fu_part, int nb) {
    check_buffer_range<T>(g);
    const int cy = pair & 1, cz = pair >> 1;
    const long long rows = (long long)((g.n[1] - cy + 1) >> 1) * ((g.n[2] - cz + 1) >> 1);
    if (rows <= 0) return;
    if (fu_part && (!reverse || !zero_support || zero_start || nb != 1))
        throw std::logic_error("f.u partials come from a reverse sweep with zero supports");
    if (zero_start && (reverse || !zero_support))
        throw std::logic_error("a zero-start sweep is forward with zero supports");
    const KeC<T> K = kec<T>();
    const RowShape w = row_shape<T>(g, rows * nb);
    const bool row = w.rpw > 0;
    const dim3 grid(row ? (unsigned)((rows + w.rpw - 1) / w.rpw) : (unsigned)rows, nb), block(row ? w.nt : 256);
    const int bs = 3 * g.N;
#define RT_LAUNCH(p, ...)                                                                                            \
    if (row)                                                                                                         \
        hipLaunchKernelGGL((k_fine_gs_row<T, ((p) & 1), ((p) >> 1), __VA_ARGS__>), grid, block, 0, s, g, U, F, rhop, \
                           vflag, K, (int)rows, w.rpw, w.npr, bs, fu_part);                                          \
    else                                                                                                             \
        hipLaunchKernelGGL((k_fine_gs_pair<T, ((p) & 1), ((p) >> 1), __VA_ARGS__>), grid, block, 0, s, g, U, F, rhop, \
                           vflag, K, (int)rows, bs, fu_part);                                                        \
    break;
    switch (pair * 8 + (fu_part ? 4 : zero_start ? 5 : (reverse ? 2 : 0) + (zero_support ? 1 : 0))) {
#define RT_CASE(p)                                          \
    case p * 8 + 0: RT_LAUNCH(p, false, false)              \
    case p * 8 + 1: RT_LAUNCH(p, false, true)               \
    case p * 8 + 2: RT_LAUNCH(p, true, false)               \
    case p * 8 + 3: RT_LAUNCH(p, true, true)                \
    case p * 8 + 4: RT_LAUNCH(p, true, true, false, true)   \
    case p * 8 + 5: RT_LAUNCH(p, false, true, true)
        RT_CASE(0) RT_CASE(1) RT_CASE(2) RT_CASE(3)
#undef RT_CASE
#undef RT_LAUNCH
    }
    RT_HIP(hipGetLastError());
}

template void launch_fine_gs<float>(const Geom&, Vec3<float>, Vec3<const float>, const float*, const uint8_t*, int,
                                    bool, bool, hipStream_t, bool, double*, int);
template void launch_fine_gs<double>(const Geom&, Vec3<double>, Vec3<const double>, const float*, const uint8_t*, int,
                                     bool, bool, hipStream_t, bool, double*, int);

}  // namespace rt
