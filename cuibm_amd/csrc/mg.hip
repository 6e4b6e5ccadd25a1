// Tensor multigrid on the device (mg.hpp): one launch down and one up per smoothed level,
// four launches of matrix-core products on the directly solved one.
//
// Smoothed levels. Bound by launch and load latency (a 1024 x 1024 level moves 15 MB down and
// 23 MB up in FP32, every other level less than half of that), not by arithmetic. A wavefront
// owns a strip of columns (one per lane, the couplings of its column in registers) and R rows,
// loads its rows of b with the halo that three sweeps and a residual need, all at once, and
// computes every sweep row by row in registers; east and west neighbours come from the next
// lanes (DPP), north and south ones from the rows before. No LDS tile, no barrier, no D^-1 in
// memory: the diagonal is the sum of four couplings already at hand, its reciprocal one
// instruction (and a Newton step in FP64). Neither the residual nor an unrestricted or
// uninterpolated vector is ever written.
//
// Direct level. Four products with 1-D eigenvector matrices as 16 x 16 tiles of
// v_mfma_*_16x16x4: all operands are rows along the contraction (four consecutive values per
// lane and load), so the first two products write their results transposed.
#include <hip/hip_ext.h>

#include <algorithm>
#include <cmath>

#include "batch.hpp"
#include "mg.hpp"

namespace cuibm {

namespace {

constexpr int WV = 4;                      // wavefronts per block
constexpr int DOWN_W = 57, UP_W = 58;      // columns a wavefront owns: 64 less the halo lanes

__device__ __forceinline__ float fma_(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double fma_(double a, double b, double c) { return __builtin_fma(a, b, c); }
// reciprocal of a diagonal: a relaxation weight, any fixed value near 1/d makes the sweep the
// same linear map at every apply
__device__ __forceinline__ float recip(float d) { return __builtin_amdgcn_rcpf(d); }
__device__ __forceinline__ double recip(double d) {
    const double r = __builtin_amdgcn_rcp(d);
    return fma_(fma_(-d, r, 1.0), r, r);
}
// the previous and the next lane's value (0 beyond the wavefront)
template <int CTRL>
__device__ __forceinline__ int dpp(int v) { return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xf, 0xf, true); }
__device__ __forceinline__ float lane_prev(float v) { return __int_as_float(dpp<0x138>(__float_as_int(v))); }
__device__ __forceinline__ float lane_next(float v) { return __int_as_float(dpp<0x130>(__float_as_int(v))); }
template <int CTRL>
__device__ __forceinline__ double dpp64(double v) {
    return __hiloint2double(dpp<CTRL>(__double2hiint(v)), dpp<CTRL>(__double2loint(v)));
}
__device__ __forceinline__ double lane_prev(double v) { return dpp64<0x138>(v); }
__device__ __forceinline__ double lane_next(double v) { return dpp64<0x130>(v); }

__device__ __forceinline__ double wave_total(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}
// the constant mode of the input, the same in every wavefront that forms it
__device__ __forceinline__ double pin_constant(const MgPins &P) {
    double t = 0;
    for (int k = threadIdx.x & 63; k < P.npart; k += 64) t += P.part[k];
    return wave_total(t) * P.inv_wa;
}

// blocks in XCD-contiguous bands (stencil.hpp)
__device__ __forceinline__ int band(int count) {
    const int per = (count + 7) / 8;
    return (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
}

__device__ __forceinline__ int wave_id() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); }

// (A x) of one cell from its diagonal, couplings and neighbours
template <class T>
__device__ __forceinline__ T row5(T d, T e, T w, T n, T s, T x, T xe, T xw, T xn, T xs) {
    return fma_(-n, xn, fma_(-s, xs, fma_(-e, xe, fma_(-w, xw, d * x))));
}

// Pre-smoothing from zero, residual and restriction of R rows of one strip. Rows k = 0 .. R+6
// are J0 - 3 + k: sweep 1 needs b alone, each further sweep and the residual one row and one
// column more on either side; the extra row and column at the end complete an aggregate that
// starts on the last owned one.
template <class T, bool FINE, int R>
__device__ __forceinline__ void down_tile(const MgTask<T> &K, const double *__restrict__ b0, int tile) {
    constexpr int N = R + 7;
    const MgLevelDev<T> &L = K.L;
    const double stopv = K.stop ? *K.stop : 0.0;
    const int nx = L.nx, ny = L.ny, strips = (nx + DOWN_W - 1) / DOWN_W;
    const int J0 = tile / strips * R, lane = threadIdx.x & 63;
    const int I = tile % strips * DOWN_W - 3 + lane, Ic = min(max(I, 0), nx - 1);
    if (J0 >= ny) return;  // uniform per wavefront; there is no barrier
    const bool in = I == Ic;
    const double *bf = FINE ? b0 + K.off : nullptr;
    T b[N];
    if (FINE) {
        double raw[N];
#pragma unroll
        for (int k = 0; k < N; k++) raw[k] = bf[(size_t)min(max(J0 - 3 + k, 0), ny - 1) * L.ld + Ic];
        const int cI = K.pins.centre % nx, cJ = K.pins.centre / nx;
        auto near = [&](int pI, int pJ) {
            return pI >= I - lane && pI < I - lane + 64 && pJ >= J0 - 3 && pJ < J0 - 3 + N;
        };
        if (near(0, 0) || (K.pins.centre > 0 && near(cI, cJ))) {
            const double c = pin_constant(K.pins);
            if (tile == 0 && lane == 0) K.pins.c[0] = c;  // for the way up
#pragma unroll
            for (int k = 0; k < N; k++) {
                if (I == 0 && J0 - 3 + k == 0) raw[k] -= c * K.pins.a0;
                if (K.pins.centre > 0 && I == cI && J0 - 3 + k == cJ) raw[k] -= c * K.pins.ac;
            }
        }
#pragma unroll
        for (int k = 0; k < N; k++) b[k] = (T)raw[k];
    } else {
#pragma unroll
        for (int k = 0; k < N; k++) b[k] = K.b[(size_t)min(max(J0 - 3 + k, 0), ny - 1) * L.ld + Ic];
    }
    const T ce = L.cE[Ic], cw = L.cW[Ic], rx = L.rx[Ic];
    const int ax = L.ax[Ic];
    const bool pair = in && I + 1 < nx && L.ax[min(Ic + 1, nx - 1)] == ax;
    const bool first = !(I > 0 && L.ax[max(Ic - 1, 0)] == ax);
    if (stopv != 0.0) return;
    T x1[N], x2[N], x3[N], dg[N], dv[N], cn[N], cs[N], v[N];
#pragma unroll
    for (int k = 0; k < N; k++) {
        const int j = J0 - 3 + k, jc = min(max(j, 0), ny - 1);
        const bool ok = in && j == jc;
        cn[k] = L.cN[jc];
        cs[k] = L.cS[jc];
        dg[k] = (ce + cw) + (cn[k] + cs[k]);
        dv[k] = ok ? recip(dg[k]) : T(0);
        b[k] = ok ? b[k] : T(0);
        x1[k] = K.w[0] * dv[k] * b[k];
        if (k >= 2) {
            const int m = k - 1;
            const T s = row5(dg[m], ce, cw, cn[m], cs[m], x1[m], lane_next(x1[m]), lane_prev(x1[m]), x1[m + 1], x1[m - 1]);
            x2[m] = fma_(K.w[1] * dv[m], b[m] - s, x1[m]);
        }
        if (k >= 4) {
            const int m = k - 2;
            const T s = row5(dg[m], ce, cw, cn[m], cs[m], x2[m], lane_next(x2[m]), lane_prev(x2[m]), x2[m + 1], x2[m - 1]);
            x3[m] = fma_(K.w[2] * dv[m], b[m] - s, x2[m]);
        }
        if (k >= 6) {
            const int m = k - 3;
            const T s = row5(dg[m], ce, cw, cn[m], cs[m], x3[m], lane_next(x3[m]), lane_prev(x3[m]), x3[m + 1], x3[m - 1]);
            const T r = (b[m] - s) * rx, rn = lane_next(r);  // every lane active: not inside the choice
            v[m] = r + (pair ? rn : T(0));
        }
    }
    const bool own = in && lane >= 3 && lane < 3 + DOWN_W;
#pragma unroll
    for (int m = 3; m < R + 3; m++) {
        const int j = J0 - 3 + m;
        if (j >= ny) break;  // uniform
        if (own) K.x3[(size_t)j * L.ld + I] = x3[m];
        const int ay = L.ay[j];
        if (j > 0 && L.ay[j - 1] == ay) continue;  // uniform: the aggregate starts a row earlier
        T t = v[m] * L.ry[j];
        if (j + 1 < ny && L.ay[j + 1] == ay) t = fma_(v[m + 1], L.ry[j + 1], t);
        if (own && first) K.rc[(size_t)ay * L.ldc + ax] = t;
    }
}

// Prolongation and post-smoothing of R rows of one strip: x = x3 + P e on a halo of three,
// three sweeps. The x interpolation of the coarse rows the strip touches is done once per
// coarse row and kept in LDS, each lane its own column (so no barrier); ex holds R + 8 rows.
template <class T, bool FINE, int R>
__device__ __forceinline__ void up_tile(const MgTask<T> &K, const double *__restrict__ b0, double *__restrict__ z0,
                                        T (*ex)[64], int tile) {
    constexpr int N = R + 6;
    const MgLevelDev<T> &L = K.L;
    const double stopv = K.stop ? *K.stop : 0.0;
    const int nx = L.nx, ny = L.ny, strips = (nx + UP_W - 1) / UP_W;
    const int J0 = tile / strips * R, lane = threadIdx.x & 63;
    const int I = tile % strips * UP_W - 3 + lane, Ic = min(max(I, 0), nx - 1);
    if (J0 >= ny) return;  // uniform per wavefront; there is no barrier
    const bool in = I == Ic;
    T x0[N], b[N];
#pragma unroll
    for (int k = 0; k < N; k++) x0[k] = K.x3[(size_t)min(max(J0 - 3 + k, 0), ny - 1) * L.ld + Ic];
    double c = 0;
    if (FINE) {
        const double *bf = b0 + K.off;
        double raw[N];
#pragma unroll
        for (int k = 1; k < N - 1; k++) raw[k] = bf[(size_t)min(max(J0 - 3 + k, 0), ny - 1) * L.ld + Ic];
        c = K.pins.c[0];
        const int cI = K.pins.centre % nx, cJ = K.pins.centre / nx;
#pragma unroll
        for (int k = 1; k < N - 1; k++) {
            if (I == 0 && J0 - 3 + k == 0) raw[k] -= c * K.pins.a0;
            if (K.pins.centre > 0 && I == cI && J0 - 3 + k == cJ) raw[k] -= c * K.pins.ac;
            b[k] = (T)raw[k];
        }
    } else {
#pragma unroll
        for (int k = 1; k < N - 1; k++) b[k] = K.b[(size_t)min(max(J0 - 3 + k, 0), ny - 1) * L.ld + Ic];
    }
    // coarse rows c0 .. c1 of this strip
    const int jlo = max(J0 - 3, 0), jhi = min(J0 + R + 2, ny - 1);
    const int c0 = max(L.ay[jlo] - 1, 0), c1 = min(L.ay[jhi] + 1, L.ay[ny - 1]);
    {
        const int a = L.ax[Ic], o = L.ox[Ic];
        const T t = L.tx[Ic];
        T va[R + 8], vo[R + 8];
#pragma unroll
        for (int r = 0; r < R + 8; r++) {
            const T *row = K.e + (size_t)min(c0 + r, c1) * L.ldc;
            va[r] = row[a];
            vo[r] = row[o];
        }
#pragma unroll
        for (int r = 0; r < R + 8; r++) ex[r][lane] = fma_(t, vo[r] - va[r], va[r]);
    }
    const T ce = L.cE[Ic], cw = L.cW[Ic];
    if (stopv != 0.0) return;
    T y1[N], y2[N], y3[N], dg[N], dv[N], cn[N], cs[N];
#pragma unroll
    for (int k = 0; k < N; k++) {
        const int j = J0 - 3 + k, jc = min(max(j, 0), ny - 1);
        const bool ok = in && j == jc;
        cn[k] = L.cN[jc];
        cs[k] = L.cS[jc];
        dg[k] = (ce + cw) + (cn[k] + cs[k]);
        dv[k] = ok ? recip(dg[k]) : T(0);
        const T ea = ex[L.ay[jc] - c0][lane], eo = ex[L.oy[jc] - c0][lane];
        x0[k] = ok ? x0[k] + fma_(L.ty[jc], eo - ea, ea) : T(0);
        if (k >= 2) {
            const int m = k - 1;
            const T s = row5(dg[m], ce, cw, cn[m], cs[m], x0[m], lane_next(x0[m]), lane_prev(x0[m]), x0[m + 1], x0[m - 1]);
            y1[m] = fma_(K.w[2] * dv[m], b[m] - s, x0[m]);
        }
        if (k >= 4) {
            const int m = k - 2;
            const T s = row5(dg[m], ce, cw, cn[m], cs[m], y1[m], lane_next(y1[m]), lane_prev(y1[m]), y1[m + 1], y1[m - 1]);
            y2[m] = fma_(K.w[1] * dv[m], b[m] - s, y1[m]);
        }
        if (k >= 6) {
            const int m = k - 3;
            const T s = row5(dg[m], ce, cw, cn[m], cs[m], y2[m], lane_next(y2[m]), lane_prev(y2[m]), y2[m + 1], y2[m - 1]);
            y3[m] = fma_(K.w[0] * dv[m], b[m] - s, y2[m]);
        }
    }
    const bool own = in && lane >= 3 && lane < 3 + UP_W;
#pragma unroll
    for (int m = 3; m < R + 3; m++) {
        const int j = J0 - 3 + m;
        if (j >= ny) break;  // uniform
        if (!own) continue;
        if (FINE) z0[K.off + (size_t)j * L.ld + I] = (double)y3[m] + c;
        else K.x[(size_t)j * L.ld + I] = y3[m];
    }
}

template <class T, bool FINE, int R>
__global__ void __launch_bounds__(64 * WV) k_mg_down(MgTask<T> K, const double *__restrict__ b0, int nblk) {
    const int blk = band(nblk);
    if (blk < nblk) down_tile<T, FINE, R>(K, b0, blk * WV + wave_id());
}
template <class T, bool FINE, int R>
__global__ void __launch_bounds__(64 * WV) k_mg_up(MgTask<T> K, const double *__restrict__ b0, double *__restrict__ z0,
                                                   int nblk) {
    __shared__ T ex[WV][R + 8][64];
    const int blk = band(nblk), w = wave_id();
    if (blk < nblk) up_tile<T, FINE, R>(K, b0, z0, ex[w], blk * WV + w);
}
// the same over a batch of cases (blocks in dispatch order, as the batch's other kernels)
template <class T, bool FINE, int R>
__global__ void __launch_bounds__(64 * WV) k_b_mg_down(const MgTask<T> *__restrict__ tab, BMapDev m,
                                                       const double *__restrict__ b0) {
    down_tile<T, FINE, R>(tab[m.cs[blockIdx.x]], b0, m.loc[blockIdx.x] * WV + wave_id());
}
template <class T, bool FINE, int R>
__global__ void __launch_bounds__(64 * WV) k_b_mg_up(const MgTask<T> *__restrict__ tab, BMapDev m,
                                                     const double *__restrict__ b0, double *__restrict__ z0) {
    __shared__ T ex[WV][R + 8][64];
    const int w = wave_id();
    up_tile<T, FINE, R>(tab[m.cs[blockIdx.x]], b0, z0, ex[w], m.loc[blockIdx.x] * WV + w);
}

// ---- direct level ----

typedef double v4d __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
template <class T>
struct Mma;
template <>
struct Mma<double> {
    typedef v4d V;
    static __device__ __forceinline__ V mul(double a, double b, V c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int g, int r) { return g + 4 * r; }  // of result element r
};
template <>
struct Mma<float> {
    typedef v4f V;
    static __device__ __forceinline__ V mul(float a, float b, V c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int g, int r) { return 4 * g + r; }
};

template <class T>
__device__ __forceinline__ typename Mma<T>::V load_v4(const T *p) {
    return *reinterpret_cast<const typename Mma<T>::V *>(p);
}

// C[m][n] = sum_k A[m][k] B[n][k] of a 16 x 16 tile over k < n16 (a multiple of 16), by a
// block of WV wavefronts that share the contraction: a level of 192 cells has 144 tiles, too
// few wavefronts for the chip, and a tile's chain of loads and products over the whole
// contraction was most of a launch (one wavefront per tile: 29 us for the four products of a
// 185^2 level in FP32 against 12). Lane
// (l & 15, g = l >> 4) gives la(k) and lb(k), the values k .. k + 3 of its row of A and of B,
// for k = 16 t + 4 g. (An instruction contracts 4 values of k, one per g; which four is free as
// long as A and B agree.) Returns element (m, n) of the block's thread: m = thread / 16 and
// n = thread % 16, or the other way round with `by_column`. Ends with every wavefront past its
// last read of `part` by the caller's own accesses only: one use per launch.
template <class T, class LA, class LB>
__device__ __forceinline__ T nt_tile(int n16, T (*part)[16][17], bool by_column, LA la, LB lb) {
    typedef typename Mma<T>::V V;
    const int w = wave_id(), l = threadIdx.x & 15, g = (threadIdx.x & 63) >> 4;
    V c0 = {0, 0, 0, 0}, c1 = {0, 0, 0, 0};
#pragma unroll 5
    for (int k = 16 * w + 4 * g; k < n16; k += 16 * WV) {
        const V a = la(k), b = lb(k);
        c0 = Mma<T>::mul(a[0], b[0], c0);
        c1 = Mma<T>::mul(a[1], b[1], c1);
        c0 = Mma<T>::mul(a[2], b[2], c0);
        c1 = Mma<T>::mul(a[3], b[3], c1);
    }
#pragma unroll
    for (int r = 0; r < 4; r++) part[w][Mma<T>::row(g, r)][l] = c0[r] + c1[r];
    __syncthreads();
    const int hi = threadIdx.x >> 4, lo = threadIdx.x & 15;
    const int m = by_column ? lo : hi, n = by_column ? hi : lo;
    return (part[0][m][n] + part[1][m][n]) + (part[2][m][n] + part[3][m][n]);
}

// One of the four products of a direct solve, a block per tile:
//   0: t1[i][J] = sum_I Fx[i][I] b[J][I]
//   1: t2[i][j] = (sum_J Fy[j][J] t1[i][J]) / (ly_j + lx_i)    (0 for the constant)
//   2: t3[J][i] = sum_j By[J][j] t2[i][j]                      (t3 over t1)
//   3: x[J][I]  = sum_i t3[J][i] Bx[I][i]
// On the finest level, 0 reads the Krylov vector less c a and 3 writes the solution of the pinned
// operator: with one pin x(0) = c, with two the consistent pair (mg.hpp: MgPins).
template <class T, bool FINE, int STAGE>
__device__ __forceinline__ void fdm_stage(const FdmTask<T> &K, const double *__restrict__ b0, double *__restrict__ z0,
                                          T (*part)[16][17], int tile) {
    const FdmDev<T> &F = K.F;
    const double stopv = K.stop ? *K.stop : 0.0;
    const int nt = F.px / 16, R = tile / nt * 16, C = tile % nt * 16;  // rows (of the y axis) and columns
    if (R >= F.py) return;  // uniform per block, before the barrier
    const int l = threadIdx.x & 15, hi = threadIdx.x >> 4, lo = threadIdx.x & 15;
    if (STAGE == 0) {
        double c = 0;
        const int cI = K.pins.centre % F.nx, cJ = K.pins.centre / F.nx;
        const bool p0 = FINE && R == 0, p1 = FINE && K.pins.centre > 0 && cJ / 16 * 16 == R;
        if (p0 || p1) {
            c = pin_constant(K.pins);
            if (tile == 0 && threadIdx.x == 0) K.pins.c[0] = c;  // for the last stage
        }
        if (stopv != 0.0) return;
        const T *f = F.Fx + (size_t)(C + l) * F.px, *br = FINE ? nullptr : K.b + (size_t)(R + l) * F.px;
        const double *bf = FINE ? b0 + K.off + (size_t)min(R + l, F.ny - 1) * F.nx : nullptr;
        const T t = nt_tile<T>(
            F.px, part, true,
            [&](int k) {
                typename Mma<T>::V a;
                if (!FINE) return load_v4<T>(br + k);
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    double v = bf[min(k + q, F.nx - 1)];
                    if (R + l >= F.ny || k + q >= F.nx) v = 0.0;
                    if (p0 && R + l == 0 && k + q == 0) v -= c * K.pins.a0;
                    if (p1 && R + l == cJ && k + q == cI) v -= c * K.pins.ac;
                    a[q] = (T)v;
                }
                return a;
            },
            [&](int k) { return load_v4<T>(f + k); });
        F.t1[(size_t)(C + hi) * F.py + R + lo] = t;
    } else if (STAGE == 1) {
        if (stopv != 0.0) return;
        const T *f = F.Fy + (size_t)(R + l) * F.py, *t1 = F.t1 + (size_t)(C + l) * F.py;
        const T t = nt_tile<T>(F.py, part, true, [&](int k) { return load_v4<T>(f + k); }, [&](int k) { return load_v4<T>(t1 + k); });
        const bool zero = R + lo == F.zy && C + hi == F.zx;  // the constant: pseudo-inverse
        F.t2[(size_t)(C + hi) * F.py + R + lo] = zero ? T(0) : t / (F.ly[R + lo] + F.lx[C + hi]);
    } else if (STAGE == 2) {
        if (stopv != 0.0) return;
        const T *f = F.By + (size_t)(R + l) * F.py, *t2 = F.t2 + (size_t)(C + l) * F.py;
        const T t = nt_tile<T>(F.py, part, false, [&](int k) { return load_v4<T>(f + k); }, [&](int k) { return load_v4<T>(t2 + k); });
        F.t1[(size_t)(R + hi) * F.px + C + lo] = t;
    } else {
        if (stopv != 0.0) return;
        double shift = 0, q0 = 0;
        if (FINE) {
            const double c = K.pins.c[0];
            auto at = [&](int pJ, int pI) {
                double t = 0;
                for (int k = threadIdx.x & 63; k < F.px; k += 64)
                    t += (double)F.t1[(size_t)pJ * F.px + k] * (double)F.Bx[(size_t)pI * F.px + k];
                return wave_total(t);
            };
            const double g0 = at(0, 0);
            if (K.pins.H) {
                q0 = (g0 - at(K.pins.centre / F.nx, K.pins.centre % F.nx)) * K.pins.hq;
                shift = c + q0 - g0 + q0 * K.pins.H[0];
            } else {
                shift = c - g0;
            }
        }
        const T *a = F.t1 + (size_t)(R + l) * F.px, *b = F.Bx + (size_t)(C + l) * F.px;
        const T t = nt_tile<T>(F.px, part, false, [&](int k) { return load_v4<T>(a + k); }, [&](int k) { return load_v4<T>(b + k); });
        if (R + hi >= F.ny || C + lo >= F.nx) return;
        if (FINE) {
            const size_t ip = (size_t)(R + hi) * F.nx + C + lo;
            z0[K.off + ip] = (double)t + shift - (K.pins.H ? q0 * K.pins.H[ip] : 0.0);
        } else {
            K.x[(size_t)(R + hi) * F.px + C + lo] = t;
        }
    }
}

template <class T, bool FINE, int STAGE>
__global__ void __launch_bounds__(64 * WV) k_fdm(FdmTask<T> K, const double *__restrict__ b0, double *__restrict__ z0) {
    __shared__ T part[WV][16][17];
    fdm_stage<T, FINE, STAGE>(K, b0, z0, part, blockIdx.x);
}
template <class T, bool FINE, int STAGE>
__global__ void __launch_bounds__(64 * WV) k_b_fdm(const FdmTask<T> *__restrict__ tab, BMapDev m,
                                                   const double *__restrict__ b0, double *__restrict__ z0) {
    __shared__ T part[WV][16][17];
    fdm_stage<T, FINE, STAGE>(tab[m.cs[blockIdx.x]], b0, z0, part, m.loc[blockIdx.x]);
}

// Rows per wavefront: 8 rows keep the halo's share at 7 rows in 15; where that leaves under
// MG_SHORT wavefronts (two per SIMD of the 1024), 4 rows shorten each wavefront's chain instead.
// A cycle with 8 rows everywhere, 4 everywhere, and this rule: 336^2 (FP32) 44.2, 38.4, 38.3 us;
// 498^2 (FP64) 72.3, 62.8, 63.1; 1024^2 (FP32) 85.9, 77.1, 78.5, where only the finest
// level has 8 (about even).
constexpr int MG_SHORT = 2048;
int strips(int nx, int w) { return (nx + w - 1) / w; }
bool short_rows(int nx, int ny) { return (long)strips(nx, DOWN_W) * ((ny + 7) / 8) < MG_SHORT; }
long mg_tiles(int nx, int ny, int w, int R) { return (long)strips(nx, w) * ((ny + R - 1) / R); }

unsigned grid8(int blocks) { return (unsigned)((blocks + 7) / 8 * 8); }

}  // namespace

template <class T>
struct TensorMg::Levels {
    struct Lvl {
        DArray<T> coef;
        DArray<int> map;
        DArray<T> b, x3, x;
        MgTask<T> task{};
        int R = 8;
    };
    std::vector<Lvl> lv;  // the smoothed levels
    DArray<T> fdm, scratch, fb, fx;
    DArray<double> H, part, c;
    FdmTask<T> direct{};
    bool fine_direct = false;

    // `sign`: of the cell areas that weight the partial sums (h has the magnitudes)
    void build(const std::vector<MgHostLevel> &h, double dt, int centre, bool round32, double sign, hipStream_t s) {
        const size_t n = h.size() - 1;  // smoothed levels
        fine_direct = n == 0;
        const int nx = (int)h[0].dx.size(), ny = (int)h[0].dy.size();
        auto val = [&](double v) { return round32 ? (T)(float)v : (T)v; };
        // pins
        std::vector<double> e0, w0, n0, s0;
        axis_couplings(h[0].dx, dt, e0, w0);
        axis_couplings(h[0].dy, dt, n0, s0);
        MgPins P;
        P.centre = centre;
        auto diag = [&](int ip) { return e0[ip % nx] + w0[ip % nx] + n0[ip / nx] + s0[ip / nx]; };
        auto area = [&](int ip) { return h[0].dx[ip % nx] * h[0].dy[ip / nx]; };
        P.a0 = diag(0);
        double wa = area(0) * P.a0;
        if (centre > 0) {
            P.ac = diag(centre);
            wa += area(centre) * P.ac;
        }
        if (!(wa > 0)) throw Error("the Poisson operator has no pinned cell to deflate", ERR_ARGUMENT);
        P.inv_wa = sign / wa;
        part.alloc(RED_GRID);
        c.alloc(1);
        launch_fill(c.p(), 0.0, 1, s);
        P.part = part.p();
        P.npart = red_parts((long)nx * ny);
        P.c = c.p();
        // Chebyshev weights of three sweeps on [lmax / 10, lmax], lmax = 2 >= the largest
        // eigenvalue of D^-1 A. Iterations on the 336^2, 498^2 and 1024^2 cylinders at their
        // tolerances: 2, 4, 3 for 6 to 10; 3, 5, 3 at 14; 4, 6, 4 at 22
        T w[3];
        for (int k = 0; k < 3; k++) {
            const double a = 2.0 / 10.0, th = 0.5 * (2.0 + a), de = 0.5 * (2.0 - a);
            w[k] = val(1.0 / (th + de * std::cos(M_PI * (2 * k + 1) / 6.0)));
        }
        // the direct level
        const MgHostLevel &D = h.back();
        const AxisModes mx = axis_modes(D.dx, dt), my = D.dy == D.dx ? mx : axis_modes(D.dy, dt);
        {
            std::vector<T> all;
            size_t at[6];
            const std::vector<double> *src[6] = {&mx.F, &my.F, &mx.B, &my.B, &mx.lam, &my.lam};
            for (int k = 0; k < 6; k++) {
                at[k] = all.size();
                for (double v : *src[k]) all.push_back(val(v));
                all.resize((all.size() + 63) / 64 * 64, T(0));  // 256-byte rows for the vector loads
            }
            fdm.upload(all, s);
            CUIBM_HIP(hipStreamSynchronize(s));
            FdmDev<T> &F = direct.F;
            F.nx = mx.n;
            F.ny = my.n;
            F.px = mx.pad;
            F.py = my.pad;
            const T **dst[6] = {&F.Fx, &F.Fy, &F.Bx, &F.By, &F.lx, &F.ly};
            for (int k = 0; k < 6; k++) *dst[k] = fdm.p() + at[k];
            F.zx = mx.zero;
            F.zy = my.zero;
            const size_t np = (size_t)mx.pad * my.pad;
            scratch.alloc(2 * np);
            F.t1 = scratch.p();
            F.t2 = scratch.p() + np;
            if (!fine_direct) {  // the padding stays zero
                for (DArray<T> *a : {&fb, &fx}) {
                    a->alloc(np);
                    std::vector<T> z(np, T(0));
                    a->upload(z, s);
                    CUIBM_HIP(hipStreamSynchronize(s));
                }
                direct.b = fb.p();
                direct.x = fx.p();
            } else {
                direct.b = nullptr;
                direct.x = nullptr;
                if (centre > 0) {
                    const std::vector<double> Hv = two_pins(mx, my, P, nx, area(0) * P.a0 / area(centre));
                    H.upload(Hv, s);
                    CUIBM_HIP(hipStreamSynchronize(s));
                    P.H = H.p();
                    P.hq = 1.0 / (1.0 + area(0) * P.a0 / (area(centre) * P.ac) + Hv[0] - Hv[centre]);
                }
                direct.pins = P;
            }
        }
        lv.resize(n);
        for (size_t l = 0; l < n; l++) {
            const MgHostLevel &G = h[l], &C = h[l + 1];
            Lvl &L = lv[l];
            const int lx = (int)G.dx.size(), ly = (int)G.dy.size();
            std::vector<double> cE, cW, cN, cS, rx(lx), ry(ly);
            axis_couplings(G.dx, dt, cE, cW);
            axis_couplings(G.dy, dt, cN, cS);
            for (int i = 0; i < lx; i++) rx[i] = G.dx[i] / C.dx[G.ax[i]];
            for (int j = 0; j < ly; j++) ry[j] = G.dy[j] / C.dy[G.ay[j]];
            std::vector<T> co;
            size_t at[8];
            const std::vector<double> *src[8] = {&cE, &cW, &rx, &G.tx, &cN, &cS, &ry, &G.ty};
            for (int k = 0; k < 8; k++) {
                at[k] = co.size();
                for (double v : *src[k]) co.push_back(val(v));
            }
            L.coef.upload(co, s);
            std::vector<int> mp;
            size_t am[4];
            const std::vector<int> *sm[4] = {&G.ax, &G.ox, &G.ay, &G.oy};
            for (int k = 0; k < 4; k++) {
                am[k] = mp.size();
                mp.insert(mp.end(), sm[k]->begin(), sm[k]->end());
            }
            L.map.upload(mp, s);
            CUIBM_HIP(hipStreamSynchronize(s));
            MgLevelDev<T> &V = L.task.L;
            V.nx = lx;
            V.ny = ly;
            V.ld = lx;
            V.ldc = l + 1 == n ? mx.pad : (int)C.dx.size();
            const T **dst[8] = {&V.cE, &V.cW, &V.rx, &V.tx, &V.cN, &V.cS, &V.ry, &V.ty};
            for (int k = 0; k < 8; k++) *dst[k] = L.coef.p() + at[k];
            const int **dm[4] = {&V.ax, &V.ox, &V.ay, &V.oy};
            for (int k = 0; k < 4; k++) *dm[k] = L.map.p() + am[k];
            const size_t cells = (size_t)lx * ly;
            L.x3.alloc(cells);
            if (l > 0) {
                L.b.alloc(cells);
                L.x.alloc(cells);
            }
            for (int k = 0; k < 3; k++) L.task.w[k] = w[k];
            L.task.pins = P;
            L.R = short_rows(lx, ly) ? 4 : 8;
        }
        for (size_t l = 0; l < n; l++) {
            MgTask<T> &K = lv[l].task;
            K.b = lv[l].b.p();
            K.x3 = lv[l].x3.p();
            K.x = lv[l].x.p();
            K.rc = l + 1 == n ? fb.p() : lv[l + 1].b.p();
            K.e = l + 1 == n ? fx.p() : lv[l + 1].x.p();
        }
        CUIBM_HIP(hipStreamSynchronize(s));
    }

    // H = A0^+ (a0 e_0 - beta e_centre)
    static std::vector<double> two_pins(const AxisModes &mx, const AxisModes &my, const MgPins &P, int nx, double beta) {
        const int n = mx.n, m = my.n, cI = P.centre % nx, cJ = P.centre / nx;
        std::vector<double> t((size_t)m * n), u((size_t)m * n, 0.0), H((size_t)m * n, 0.0);
        for (int j = 0; j < m; j++)
            for (int i = 0; i < n; i++) {
                const double v = P.a0 * my.F[(size_t)j * my.pad] * mx.F[(size_t)i * mx.pad] -
                                 beta * my.F[(size_t)j * my.pad + cJ] * mx.F[(size_t)i * mx.pad + cI];
                t[(size_t)j * n + i] = j == my.zero && i == mx.zero ? 0.0 : v / (my.lam[j] + mx.lam[i]);
            }
        for (int J = 0; J < m; J++)
            for (int j = 0; j < m; j++) {
                const double f = my.B[(size_t)J * my.pad + j];
                for (int i = 0; i < n; i++) u[(size_t)J * n + i] += f * t[(size_t)j * n + i];
            }
        std::vector<double> bt((size_t)n * n);  // Bx transposed: unit-stride sums
        for (int I = 0; I < n; I++)
            for (int i = 0; i < n; i++) bt[(size_t)i * n + I] = mx.B[(size_t)I * mx.pad + i];
        for (int J = 0; J < m; J++)
            for (int i = 0; i < n; i++) {
                const double f = u[(size_t)J * n + i];
                for (int I = 0; I < n; I++) H[(size_t)J * n + I] += f * bt[(size_t)i * n + I];
            }
        return H;
    }

    void set_stop(const double *stop) {
        for (Lvl &L : lv) L.task.stop = stop;
        direct.stop = stop;
    }

    int blocks(size_t l, bool down) const {
        const MgLevelDev<T> &L = lv[l].task.L;
        return (int)((mg_tiles(L.nx, L.ny, down ? DOWN_W : UP_W, lv[l].R) + WV - 1) / WV);
    }
    void down(size_t l, const double *b, hipStream_t s, KernelProbe *probe) {
        const int nb = blocks(l, true);
        const dim3 g(grid8(nb)), t(64 * WV);
        const MgTask<T> &K = lv[l].task;
        auto go = [&](auto k) {
            if (probe && probe->enabled()) {
                hipEvent_t e0, e1;
                probe->pair(e0, e1);
                hipExtLaunchKernelGGL(k, g, t, 0, s, e0, e1, 0, K, b, nb);
            } else {
                hipLaunchKernelGGL(k, g, t, 0, s, K, b, nb);
            }
        };
        if (l == 0) lv[l].R == 8 ? go(k_mg_down<T, true, 8>) : go(k_mg_down<T, true, 4>);
        else lv[l].R == 8 ? go(k_mg_down<T, false, 8>) : go(k_mg_down<T, false, 4>);
        CUIBM_LAUNCH_CHECK();
    }
    void up(size_t l, const double *b, double *z, hipStream_t s) {
        const int nb = blocks(l, false);
        const dim3 g(grid8(nb)), t(64 * WV);
        const MgTask<T> &K = lv[l].task;
        auto go = [&](auto k) { hipLaunchKernelGGL(k, g, t, 0, s, K, b, z, nb); };
        if (l == 0) lv[l].R == 8 ? go(k_mg_up<T, true, 8>) : go(k_mg_up<T, true, 4>);
        else lv[l].R == 8 ? go(k_mg_up<T, false, 8>) : go(k_mg_up<T, false, 4>);
        CUIBM_LAUNCH_CHECK();
    }
    template <int STAGE>
    void product(const double *b, double *z, hipStream_t s, KernelProbe *probe = nullptr) {
        const dim3 g((unsigned)(direct.F.px / 16 * (direct.F.py / 16))), t(64 * WV);
        auto go = [&](auto k) {
            if (probe && probe->enabled()) {
                hipEvent_t e0, e1;
                probe->pair(e0, e1);
                hipExtLaunchKernelGGL(k, g, t, 0, s, e0, e1, 0, direct, b, z);
            } else {
                hipLaunchKernelGGL(k, g, t, 0, s, direct, b, z);
            }
        };
        // stages 1 and 2 never see the Krylov vectors, and FP32 levels are never the finest
        constexpr bool ends = (STAGE == 0 || STAGE == 3) && std::is_same<T, double>::value;
        if constexpr (ends) fine_direct ? go(k_fdm<T, true, STAGE>) : go(k_fdm<T, false, STAGE>);
        else go(k_fdm<T, false, STAGE>);
        CUIBM_LAUNCH_CHECK();
    }
    // one cycle from zero; the partial sums of w b are in `part`
    void apply(const double *b, double *z, hipStream_t s, KernelProbe *probe) {
        for (size_t l = 0; l < lv.size(); l++) down(l, b, s, l == 0 ? probe : nullptr);
        product<0>(b, z, s, fine_direct ? probe : nullptr);
        product<1>(b, z, s);
        product<2>(b, z, s);
        product<3>(b, z, s);
        for (size_t l = lv.size(); l-- > 0;) up(l, b, z, s);
    }
};

TensorMg::TensorMg(const std::vector<double> &dx, const std::vector<double> &dy, double dt, int centre, int precision,
                   int coarse_max, const double *dx_dev, const double *dy_dev, hipStream_t s) {
    // a small grid is solved directly, in FP64 whatever the precision of the levels would be
    const bool direct = coarse_max <= 0 && std::max(dx.size(), dy.size()) <= (size_t)MG_DIRECT_MAX;
    // an axis that runs downwards has negative widths; the operator holds products of two
    auto magnitudes = [](std::vector<double> w) {
        for (double &v : w) v = std::fabs(v);
        return w;
    };
    const double sign = (dx[0] < 0) == (dy[0] < 0) ? 1.0 : -1.0;
    const std::vector<MgHostLevel> h = mg_levels(magnitudes(dx), magnitudes(dy), direct ? MG_DIRECT_MAX : MG_FDM_MAX, coarse_max);
    for (const MgHostLevel &L : h) sizes_.emplace_back((int)L.dx.size(), (int)L.dy.size());
    if (precision == 32 && h.size() > 1) {
        f_.reset(new Levels<float>);
        f_->build(h, dt, centre, false, sign, s);
    } else {
        d_.reset(new Levels<double>);
        d_->build(h, dt, centre, precision == 3264 && h.size() > 1, sign, s);
    }
    w_.nx = (int)dx.size();
    w_.wx = dx_dev;
    w_.wy = dy_dev;
    w_.part = f_ ? f_->part.p() : d_->part.p();
    wdot_ = P5Dev{};
    wdot_.nx = (int)dx.size();
    wdot_.ny = (int)dy.size();
    wdot_.dx = dx_dev;
    wdot_.dy = dy_dev;
}

TensorMg::~TensorMg() = default;

void TensorMg::set_stop(const double *stop) {
    wdot_.stop = stop;
    if (f_) f_->set_stop(stop);
    else d_->set_stop(stop);
}

void TensorMg::apply(const double *r, double *z, hipStream_t s, bool weighted) {
    if (!weighted) launch_p5_wdot(wdot_, r, w_.part, s);
    if (f_) f_->apply(r, z, s, &probe_);
    else d_->apply(r, z, s, &probe_);
}

void TensorMg::fine_first(const double *b, hipStream_t s) {
    auto go = [&](auto &L) { L.fine_direct ? L.template product<0>(b, nullptr, s) : L.down(0, b, s, nullptr); };
    if (f_) go(*f_);
    else go(*d_);
}

void TensorMg::fine_last(const double *b, double *z, hipStream_t s) {
    auto go = [&](auto &L) { L.fine_direct ? L.template product<3>(b, z, s) : L.up(0, b, z, s); };
    if (f_) go(*f_);
    else go(*d_);
}

std::vector<double> TensorMg::launch_bytes() const {
    const double sv = f_ ? 4.0 : 8.0;
    std::vector<double> out;
    const size_t n = sizes_.size() - 1;
    auto cells = [&](size_t l) { return (double)sizes_[l].first * sizes_[l].second; };
    auto edge = [&](size_t l) { return (double)(sizes_[l].first + sizes_[l].second); };
    // couplings, restriction and interpolation weights, aggregates
    auto oned = [&](size_t l) { return edge(l) * (4 * sv + 8); };
    for (size_t l = 0; l < n; l++)  // b in; smoothed iterate and coarse right-hand side out
        out.push_back(cells(l) * ((l == 0 ? 8 : sv) + sv) + cells(l + 1) * sv + oned(l));
    const double nc = cells(n), px = sizes_[n].first, py = sizes_[n].second;
    const double io = n == 0 ? 8.0 : sv;
    out.push_back(nc * (io + sv) + px * px * sv);
    out.push_back(2 * nc * sv + py * py * sv);
    out.push_back(2 * nc * sv + py * py * sv);
    out.push_back(nc * (io + sv) + px * px * sv);
    for (size_t l = n; l-- > 0;)  // smoothed iterate, correction and b in; result out
        out.push_back(cells(l) * (sv + 2 * (l == 0 ? 8 : sv)) + cells(l + 1) * sv + oned(l));
    return out;
}

// ---- lockstep batches: the cycles of many cases as one preconditioner ----
// Level l of every case that smooths on it is one launch (task table and block map per level),
// and so is each of the four products of all directly solved levels.

struct BatchMg::Impl {
    template <class T>
    struct Set {  // the cases with levels of type T
        struct Lvl {
            BMap down[2], up[2];  // cases with 8 and with 4 rows per wavefront
            std::vector<long> nd[2], nu[2];
            std::vector<MgTask<T>> host[2];
            DArray<MgTask<T>> tabR[2];
        };
        std::vector<Lvl> lv;
        std::vector<FdmTask<T>> host[2];  // [1]: finest level
        DArray<FdmTask<T>> tab[2];
        BMap tiles[2];
        std::vector<long> nt[2];

        void add(const TensorMg::Levels<T> &C, long off, const double *stop, double *c, const double *part, int npart) {
            auto pins = [&](MgPins P) {
                P.part = part;
                P.npart = npart;
                P.c = c;
                return P;
            };
            for (size_t l = 0; l < C.lv.size(); l++) {
                if (lv.size() <= l) lv.resize(l + 1);
                const int r = C.lv[l].R == 8 ? 0 : 1;
                MgTask<T> K = C.lv[l].task;
                K.off = off;
                K.stop = stop;
                K.pins = pins(K.pins);
                lv[l].host[r].push_back(K);
                lv[l].nd[r].push_back(mg_tiles(K.L.nx, K.L.ny, DOWN_W, C.lv[l].R));
                lv[l].nu[r].push_back(mg_tiles(K.L.nx, K.L.ny, UP_W, C.lv[l].R));
            }
            const int f = C.fine_direct ? 1 : 0;
            FdmTask<T> K = C.direct;
            K.off = off;
            K.stop = stop;
            K.pins = pins(K.pins);
            host[f].push_back(K);
            nt[f].push_back((long)(K.F.px / 16) * (K.F.py / 16));
        }
        void finish(hipStream_t s) {
            for (Lvl &L : lv)
                for (int r = 0; r < 2; r++) {
                    if (L.host[r].empty()) continue;
                    L.tabR[r].upload(L.host[r], s);
                    L.down[r].build(L.nd[r], WV, s);
                    L.up[r].build(L.nu[r], WV, s);
                }
            for (int f = 0; f < 2; f++) {
                if (host[f].empty()) continue;
                tab[f].upload(host[f], s);
                tiles[f].build(nt[f], 1, s);
            }
            CUIBM_HIP(hipStreamSynchronize(s));
        }
        void apply(const double *b, double *z, hipStream_t s) {
            const dim3 t(64 * WV);
            for (size_t l = 0; l < lv.size(); l++)
                for (int r = 0; r < 2; r++) {
                    if (lv[l].host[r].empty()) continue;
                    const BMapDev m = lv[l].down[r].dev();
                    auto go = [&](auto k) { hipLaunchKernelGGL(k, dim3(m.nblk), t, 0, s, lv[l].tabR[r].p(), m, b); };
                    if (l == 0) r == 0 ? go(k_b_mg_down<T, true, 8>) : go(k_b_mg_down<T, true, 4>);
                    else r == 0 ? go(k_b_mg_down<T, false, 8>) : go(k_b_mg_down<T, false, 4>);
                    CUIBM_LAUNCH_CHECK();
                }
            for (int f = 0; f < 2; f++) {
                if (host[f].empty()) continue;
                const BMapDev m = tiles[f].dev();
                auto go = [&](auto k) {
                    hipLaunchKernelGGL(k, dim3(m.nblk), t, 0, s, tab[f].p(), m, b, z);
                    CUIBM_LAUNCH_CHECK();
                };
                constexpr bool fine = std::is_same<T, double>::value;  // FP32 levels are never the finest
                f ? go(k_b_fdm<T, fine, 0>) : go(k_b_fdm<T, false, 0>);
                go(k_b_fdm<T, false, 1>);
                go(k_b_fdm<T, false, 2>);
                f ? go(k_b_fdm<T, fine, 3>) : go(k_b_fdm<T, false, 3>);
            }
            for (size_t l = lv.size(); l-- > 0;)
                for (int r = 0; r < 2; r++) {
                    if (lv[l].host[r].empty()) continue;
                    const BMapDev m = lv[l].up[r].dev();
                    auto go = [&](auto k) { hipLaunchKernelGGL(k, dim3(m.nblk), t, 0, s, lv[l].tabR[r].p(), m, b, z); };
                    if (l == 0) r == 0 ? go(k_b_mg_up<T, true, 8>) : go(k_b_mg_up<T, true, 4>);
                    else r == 0 ? go(k_b_mg_up<T, false, 8>) : go(k_b_mg_up<T, false, 4>);
                    CUIBM_LAUNCH_CHECK();
                }
        }
    };
    Set<double> d;
    Set<float> f;
    int levels = 0;
    DArray<double> part, c;
};

BatchMg::BatchMg(const std::vector<TensorMg *> &mg, const std::vector<long> &offP, const std::vector<BCase> &tab_host,
                 const std::vector<int> &nblk, hipStream_t s)
    : im_(new Impl) {
    if (mg.empty()) throw Error("batched V-cycle without cases", ERR_ARGUMENT);
    Impl &B = *im_;
    B.c.alloc(mg.size());
    launch_fill(B.c.p(), 0.0, (long)mg.size(), s);
    size_t total = 0, first = 0;
    for (int n : nblk) total += n;
    B.part.alloc(std::max<size_t>(total, 1));
    for (size_t k = 0; k < mg.size(); k++) {
        const size_t part = first;
        first += nblk[k];
        if (!mg[k]) continue;
        const TensorMg &M = *mg[k];
        const double *stop = tab_host[k].scP + SC_STOP;
        auto take = [&](auto &set, const auto &L) {
            set.add(L, offP[k], stop, B.c.p() + k, B.part.p() + part, nblk[k]);
        };
        if (M.f_) take(B.f, *M.f_);
        else take(B.d, *M.d_);
        B.levels = std::max(B.levels, (int)M.sizes().size());
    }
    B.d.finish(s);
    B.f.finish(s);
}

double *BatchMg::weights_part() const { return im_->part.p(); }

BatchMg::~BatchMg() = default;

void BatchMg::apply(const double *r, double *z, hipStream_t s) {
    Impl &B = *im_;
    B.d.apply(r, z, s);
    B.f.apply(r, z, s);
}

int BatchMg::levels() const { return im_->levels; }

}  // namespace cuibm
