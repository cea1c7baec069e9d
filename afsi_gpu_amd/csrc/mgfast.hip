// Fused V-cycle for gfx950: few launches per cycle, one HBM pass per sweep.
//
// * rb_sweep_kernel: one full red-black Gauss-Seidel sweep per launch. A
//   workgroup stages its 8x8x32 tile plus a 2-cell halo of p in LDS,
//   updates the red cells of the tile and its 1-cell ring in LDS, then the
//   black cells of the tile, and writes the tile (out of place: p_in is
//   never written, so every tile reads start-of-sweep values). Update
//   p = (rhs + sum_nb w_a p_nb) / sum w_a, w_a = 1/h_a^2, over the existing
//   neighbours, which equals p + (rhs - A p)/diag.
// * Mean removal. The reference subtracts the mean of p after each
//   smoothing stage and of every restricted residual (mac/multigrid.py:
//   107-123). The V-cycle commutes with adding a constant (A 1 = 0, both
//   smoothers and the prolongation reproduce constants, and the coarse
//   inverse of a zero-mean residual has zero mean), so on the fine levels
//   those subtractions change nothing but rounding; this driver performs
//   them inside the LDS coarse kernel only; the caller removes the mean of
//   the level-0 iterate once, after the last cycle. No kernel needs a
//   grid-wide reduction, fence or atomic.
// * coarse_cycle_kernel: one 1024-thread workgroup runs the complete
//   V-cycle of every level with <= COARSE_MAX cells (smoothing, restriction,
//   means, the dense coarse solve, prolongation) out of LDS.
// * Tiles are mapped XCD-aware: consecutive workgroup ids are dealt
//   round-robin to the 8 XCDs, so each XCD is given one contiguous run of
//   tiles and the halos it re-reads stay in its own L2.
#include "mgcommon.hpp"
#include <algorithm>
#include <mutex>
#include <vector>

namespace afsi {

template <class T>
int launch_fill(T* x, int64_t count, T value, hipStream_t s);
int launch_reduce_final(const double* partials, int64_t nparts, double* result, hipStream_t s);

constexpr int COARSE_THREADS = 1024;
constexpr int64_t COARSE_MAX = 4096;  // cells of the finest level solved in LDS
constexpr int COARSE_TOTAL = 4800;    // cells of all LDS levels

struct Dim32 {
    int n0, n1, n2;
};

template <class T>
struct W3 {
    T w[3];          // 1/h^2
    T relax = T(1);  // red-black over-relaxation weight (1: Gauss-Seidel)
};

// Red-black update of a cell from its Gauss-Seidel value gs: gs itself, or
// old + relax * (gs - old) when over-relaxed (relax is uniform per launch).
template <class T>
__device__ inline T rb_relax(const W3<T>& k, T old, T gs) {
    return k.relax == T(1) ? gs : fma_of(k.relax, gs - old, old);
}

__device__ inline int wrap32(int g, int n) {
    while (g < 0) g += n;
    while (g >= n) g -= n;
    return g;
}

__device__ inline int64_t xcd_tile(int64_t b, int64_t ntiles) {
    if (ntiles % 8) return b;
    return (b % 8) * (ntiles / 8) + b / 8;
}

// Gauss-Seidel / Jacobi pieces on an array with strides (sx, sy, 1).
// s = sum_nb w_a p_nb and d = sum w_a over the neighbours that exist.
template <class T, bool P>
__device__ inline void neighbour_sums(const T* __restrict__ a, int li, int sx, int sy, int gx,
                                      int gy, int gz, const Dim32& d, const W3<T>& k, T& s, T& dg) {
    s = T(0);
    dg = T(0);
    if (P || gx + 1 < d.n0) { s += k.w[0] * a[li + sx]; dg += k.w[0]; }
    if (P || gx > 0) { s += k.w[0] * a[li - sx]; dg += k.w[0]; }
    if (P || gy + 1 < d.n1) { s += k.w[1] * a[li + sy]; dg += k.w[1]; }
    if (P || gy > 0) { s += k.w[1] * a[li - sy]; dg += k.w[1]; }
    if (P || gz + 1 < d.n2) { s += k.w[2] * a[li + 1]; dg += k.w[2]; }
    if (P || gz > 0) { s += k.w[2] * a[li - 1]; dg += k.w[2]; }
}

// A p = sum_nb w_a (p - p_nb) over existing neighbours (difference form:
// neighbour differences of a smooth field are nearly exact, so the residual
// keeps its accuracy when p carries a constant offset).
template <class T, bool P>
__device__ inline T apply_diff(const T* __restrict__ a, int li, int sx, int sy,
                               int gx, int gy, int gz, const Dim32& d, const W3<T>& k) {
    const T c = a[li];
    T r = T(0);
    if (P) {
        r += k.w[0] * (c - a[li + (gx + 1 < d.n0 ? sx : -(d.n0 - 1) * sx)]);
        r += k.w[0] * (c - a[li + (gx > 0 ? -sx : (d.n0 - 1) * sx)]);
        r += k.w[1] * (c - a[li + (gy + 1 < d.n1 ? sy : -(d.n1 - 1) * sy)]);
        r += k.w[1] * (c - a[li + (gy > 0 ? -sy : (d.n1 - 1) * sy)]);
        r += k.w[2] * (c - a[li + (gz + 1 < d.n2 ? 1 : -(d.n2 - 1))]);
        r += k.w[2] * (c - a[li + (gz > 0 ? -1 : (d.n2 - 1))]);
    } else {
        if (gx + 1 < d.n0) r += k.w[0] * (c - a[li + sx]);
        if (gx > 0) r += k.w[0] * (c - a[li - sx]);
        if (gy + 1 < d.n1) r += k.w[1] * (c - a[li + sy]);
        if (gy > 0) r += k.w[1] * (c - a[li - sy]);
        if (gz + 1 < d.n2) r += k.w[2] * (c - a[li + 1]);
        if (gz > 0) r += k.w[2] * (c - a[li - 1]);
    }
    return r;
}

// ---------------------------------------------------------------------------
// fine levels

// Tile TX x TY x TZ cells, NT threads. All global loads of a thread (its
// share of the p box and the rhs of its red-ring and black-tile cells) are
// issued into registers before the first LDS write, so their latencies
// overlap instead of serialising one loop iteration at a time.
template <class T, bool P, int TX, int TY, int TZ, int NT>
__global__ void __launch_bounds__(NT) rb_sweep_kernel(const T* __restrict__ pin,
                                                      const T* __restrict__ rhs,
                                                      T* __restrict__ pout, Dim32 d, W3<T> k,
                                                      int zero_in, int ntx, int nty, int ntz) {
    constexpr int BX = TX + 4, BY = TY + 4, BZ = TZ + 4, BOX = BX * BY * BZ;
    constexpr int RX = TX + 2, RY = TY + 2, RZ = TZ + 2, RING = RX * RY * RZ;
    constexpr int TILE = TX * TY * TZ;
    constexpr int NB = (BOX + NT - 1) / NT, NR = (RING + NT - 1) / NT, NL = (TILE + NT - 1) / NT;
    __shared__ T box[BOX];
    const int tile = int(xcd_tile(blockIdx.x, int64_t(ntx) * nty * ntz));
    const int tz = tile % ntz, ty = (tile / ntz) % nty, tx = tile / (ntz * nty);
    const int x0 = tx * TX - 2, y0 = ty * TY - 2, z0 = tz * TZ - 2;
    const int sxg = d.n1 * d.n2;
    const int t = threadIdx.x;
    T pv[NB], rr[NR], rt[NL];
#pragma unroll
    for (int j = 0; j < NB; ++j) {
        const int e = t + j * NT;
        pv[j] = T(0);
        if (e < BOX && !zero_in) {
            const int lz = e % BZ, ly = (e / BZ) % BY, lx = e / (BZ * BY);
            int gx = x0 + lx, gy = y0 + ly, gz = z0 + lz;
            if (P) {
                gx = wrap32(gx, d.n0); gy = wrap32(gy, d.n1); gz = wrap32(gz, d.n2);
                pv[j] = pin[gx * sxg + gy * d.n2 + gz];
            } else if (gx >= 0 && gx < d.n0 && gy >= 0 && gy < d.n1 && gz >= 0 && gz < d.n2) {
                pv[j] = pin[gx * sxg + gy * d.n2 + gz];
            }
        }
    }
#pragma unroll
    for (int j = 0; j < NR; ++j) {
        const int e = t + j * NT;
        rr[j] = T(0);
        if (e < RING) {
            const int lz = e % RZ + 1, ly = (e / RZ) % RY + 1, lx = e / (RZ * RY) + 1;
            int gx = x0 + lx, gy = y0 + ly, gz = z0 + lz;
            bool in = true;
            if (P) { gx = wrap32(gx, d.n0); gy = wrap32(gy, d.n1); gz = wrap32(gz, d.n2); }
            else in = gx >= 0 && gx < d.n0 && gy >= 0 && gy < d.n1 && gz >= 0 && gz < d.n2;
            if (in && !((gx + gy + gz) & 1)) rr[j] = rhs[gx * sxg + gy * d.n2 + gz];
        }
    }
#pragma unroll
    for (int j = 0; j < NL; ++j) {
        const int e = t + j * NT;
        rt[j] = T(0);
        if (e < TILE) {
            const int lz = e % TZ + 2, ly = (e / TZ) % TY + 2, lx = e / (TZ * TY) + 2;
            const int gx = x0 + lx, gy = y0 + ly, gz = z0 + lz;
            if (gx < d.n0 && gy < d.n1 && gz < d.n2 && ((gx + gy + gz) & 1))
                rt[j] = rhs[gx * sxg + gy * d.n2 + gz];
        }
    }
#pragma unroll
    for (int j = 0; j < NB; ++j) {
        const int e = t + j * NT;
        if (e < BOX) box[e] = pv[j];
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < NR; ++j) {
        const int e = t + j * NT;
        if (e >= RING) continue;
        const int lz = e % RZ + 1, ly = (e / RZ) % RY + 1, lx = e / (RZ * RY) + 1;
        int gx = x0 + lx, gy = y0 + ly, gz = z0 + lz;
        if (P) {
            gx = wrap32(gx, d.n0); gy = wrap32(gy, d.n1); gz = wrap32(gz, d.n2);
        } else if (gx < 0 || gx >= d.n0 || gy < 0 || gy >= d.n1 || gz < 0 || gz >= d.n2) {
            continue;
        }
        if ((gx + gy + gz) & 1) continue;  // red = even parity
        const int li = (lx * BY + ly) * BZ + lz;
        T sum, dg;
        neighbour_sums<T, P>(box, li, BY * BZ, BZ, gx, gy, gz, d, k, sum, dg);
        box[li] = rb_relax(k, box[li], (rr[j] + sum) / dg);
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < NL; ++j) {
        const int e = t + j * NT;
        if (e >= TILE) continue;
        const int lz = e % TZ + 2, ly = (e / TZ) % TY + 2, lx = e / (TZ * TY) + 2;
        const int gx = x0 + lx, gy = y0 + ly, gz = z0 + lz;
        if (gx >= d.n0 || gy >= d.n1 || gz >= d.n2) continue;
        const int li = (lx * BY + ly) * BZ + lz;
        T v = box[li];
        if ((gx + gy + gz) & 1) {
            T sum, dg;
            neighbour_sums<T, P>(box, li, BY * BZ, BZ, gx, gy, gz, d, k, sum, dg);
            v = rb_relax(k, v, (rt[j] + sum) / dg);
        }
        pout[gx * sxg + gy * d.n2 + gz] = v;
    }
}

// weighted Jacobi: out = p + omega*(rhs - A p)/diag
template <class T, bool P>
__global__ void __launch_bounds__(256) jacobi_fast_kernel(const T* __restrict__ pin,
                                                          const T* __restrict__ rhs,
                                                          T* __restrict__ pout, Dim32 d, W3<T> k,
                                                          T omega, int zero_in) {
    const int sxg = d.n1 * d.n2;
    const int total = sxg * d.n0;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < total; i += gridDim.x * blockDim.x) {
        const int x = i / sxg;
        const int r = i - x * sxg;
        const int y = r / d.n2, z = r - y * d.n2;
        const T dg = (P || x + 1 < d.n0 ? k.w[0] : T(0)) + (P || x > 0 ? k.w[0] : T(0)) +
                     (P || y + 1 < d.n1 ? k.w[1] : T(0)) + (P || y > 0 ? k.w[1] : T(0)) +
                     (P || z + 1 < d.n2 ? k.w[2] : T(0)) + (P || z > 0 ? k.w[2] : T(0));
        const T c = zero_in ? T(0) : pin[i];
        const T a = zero_in ? T(0) : apply_diff<T, P>(pin, i, sxg, d.n2, x, y, z, d, k);
        pout[i] = c + omega * (rhs[i] - a) / dg;
    }
}

// coarse = avg8(rhs - A p)
template <class T, bool P>
__global__ void __launch_bounds__(256) restrict_fast_kernel(const T* __restrict__ p,
                                                            const T* __restrict__ rhs,
                                                            T* __restrict__ coarse, Dim32 d,
                                                            W3<T> k) {
    const int c1 = d.n1 / 2, c2 = d.n2 / 2;
    const int cs = c1 * c2;
    const int total = cs * (d.n0 / 2);
    const int sxg = d.n1 * d.n2;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < total; i += gridDim.x * blockDim.x) {
        const int x = i / cs;
        const int r = i - x * cs;
        const int y = r / c2, z = r - y * c2;
        T v = T(0);
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int cc = 0; cc < 2; ++cc) {
                    const int fx = 2 * x + a, fy = 2 * y + b, fz = 2 * z + cc;
                    const int j = fx * sxg + fy * d.n2 + fz;
                    v += rhs[j] - apply_diff<T, P>(p, j, sxg, d.n2, fx, fy, fz, d, k);
                }
        coarse[i] = v * T(0.125);
    }
}

template <class T, bool P>
__device__ inline T prolong32(const T* __restrict__ coarse, int x, int y, int z, int C0, int C1,
                              int C2) {
    const int ax = x / 2 - 1 + x % 2, ay = y / 2 - 1 + y % 2, az = z / 2 - 1 + z % 2;
    int x0, x1, y0, y1, z0, z1;
    if (P) {  // -1 <= ax and ax + 1 <= C0: one conditional wrap each
        x0 = ax < 0 ? ax + C0 : ax; x1 = ax + 1 >= C0 ? ax + 1 - C0 : ax + 1;
        y0 = ay < 0 ? ay + C1 : ay; y1 = ay + 1 >= C1 ? ay + 1 - C1 : ay + 1;
        z0 = az < 0 ? az + C2 : az; z1 = az + 1 >= C2 ? az + 1 - C2 : az + 1;
    } else {
        x0 = ax > 0 ? ax : 0; x1 = ax + 1 < C0 - 1 ? ax + 1 : C0 - 1;
        y0 = ay > 0 ? ay : 0; y1 = ay + 1 < C1 - 1 ? ay + 1 : C1 - 1;
        z0 = az > 0 ? az : 0; z1 = az + 1 < C2 - 1 ? az + 1 : C2 - 1;
    }
    const T wx = (x % 2 == 0) ? T(0.75) : T(0.25);
    const T wy = (y % 2 == 0) ? T(0.75) : T(0.25);
    const T wz = (z % 2 == 0) ? T(0.75) : T(0.25);
    const int s1 = C2, s0 = C1 * C2;
    const T* b00 = coarse + x0 * s0 + y0 * s1;
    const T* b01 = coarse + x0 * s0 + y1 * s1;
    const T* b10 = coarse + x1 * s0 + y0 * s1;
    const T* b11 = coarse + x1 * s0 + y1 * s1;
    const T c00 = b00[z0] * (T(1) - wz) + b00[z1] * wz;
    const T c01 = b01[z0] * (T(1) - wz) + b01[z1] * wz;
    const T c10 = b10[z0] * (T(1) - wz) + b10[z1] * wz;
    const T c11 = b11[z0] * (T(1) - wz) + b11[z1] * wz;
    return (c00 * (T(1) - wy) + c01 * wy) * (T(1) - wx) + (c10 * (T(1) - wy) + c11 * wy) * wx;
}

template <class T, bool P>
__global__ void __launch_bounds__(256) prolong_fast_kernel(const T* __restrict__ coarse,
                                                           T* __restrict__ fine, Dim32 d) {
    const int sxg = d.n1 * d.n2;
    const int total = sxg * d.n0;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < total; i += gridDim.x * blockDim.x) {
        const int x = i / sxg;
        const int r = i - x * sxg;
        const int y = r / d.n2, z = r - y * d.n2;
        fine[i] = fine[i] + prolong32<T, P>(coarse, x, y, z, d.n0 / 2, d.n1 / 2, d.n2 / 2);
    }
}

// per-workgroup [sum r, sum r^2, sum |r|, non-finite] of r = rhs - A p
template <class T, bool P>
__global__ void __launch_bounds__(256) residual_partials_kernel(const T* __restrict__ p,
                                                                const T* __restrict__ rhs, Dim32 d,
                                                                W3<T> k, double* __restrict__ partials) {
    __shared__ double sh[4][256 / WAVE];
    const int sxg = d.n1 * d.n2;
    const int total = sxg * d.n0;
    double v[4] = {0.0, 0.0, 0.0, 0.0};
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < total; i += gridDim.x * blockDim.x) {
        const int x = i / sxg;
        const int rr = i - x * sxg;
        const int y = rr / d.n2, z = rr - y * d.n2;
        const double r = double(rhs[i] - apply_diff<T, P>(p, i, sxg, d.n2, x, y, z, d, k));
        if (isfinite(r)) {
            v[0] += r;
            v[1] += r * r;
            v[2] += fabs(r);
        } else {
            v[3] += 1.0;
        }
    }
    const int wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
    for (int q = 0; q < 4; ++q) {
        double t = v[q];
#pragma unroll
        for (int dd = 32; dd >= 1; dd >>= 1) t += __shfl_xor(t, dd, WAVE);
        if (lane == 0) sh[q][wave] = t;
    }
    __syncthreads();
    if (threadIdx.x < 4) {
        double t = 0.0;
        for (int w = 0; w < 256 / WAVE; ++w) t += sh[threadIdx.x][w];
        partials[4 * blockIdx.x + threadIdx.x] = t;
    }
}

// ---------------------------------------------------------------------------
// Row kernels (levels with an even z extent <= ZROW): one wavefront per
// (x, y) row, lanes along z. Row decode, wrap and boundary tests are
// wave-uniform, lanes map to z (or to the red / black cells of a row by
// parity), so no per-element integer division remains.

constexpr int ZROW = 128;

__device__ inline int face_class(int g, int n) { return g == 0 ? 0 : (g == n - 1 ? 2 : 1); }

// Diagonal of the Neumann operator by boundary class (0 low, 1 interior,
// 2 high) per axis; entry t of a 27-table.
template <class T>
__device__ inline T diag_entry(int t, const W3<T>& k) {
    const int cls[3] = {t / 9, (t / 3) % 3, t % 3};
    T dg = T(0);
    for (int a = 0; a < 3; ++a) dg += k.w[a] * T(cls[a] == 1 ? 2 : 1);
    return dg;
}
template <class T>
__device__ inline T inv_diag_entry(int t, const W3<T>& k) { return T(1) / diag_entry<T>(t, k); }

// A reciprocal and what its rounding left out: t * hi + t * lo rounds like t / diag.
template <class T>
struct Recip {
    T hi, lo;
};
template <class T>
__device__ inline Recip<T> recip(T diag) {
    const T r = T(1) / diag;
    return {r, fma_of(-diag, r, T(1)) * r};
}

template <class T, bool P>
__device__ inline int wrap_or(int g, int n, bool& in) {
    if (P) return wrap32(g, n);
    in = in && g >= 0 && g < n;
    return g;
}

#include "mgtile.hpp"

// One red-black Gauss-Seidel sweep of TX x TY columns of rows spanning all
// of z. LDS holds the (TX+4) x (TY+4) rows of p of one tile; red is updated
// on the tile and its 1-row ring, then black on the tile. Lane r < ROWS
// writes the record of box row r (wrapped global offset, coordinates,
// in-domain flag) to LDS, so per-row bookkeeping is done once per row.
// The kernel is persistent: workgroup b sweeps tiles b, b + G, ... (XCD-
// aware: each XCD owns a contiguous run of tiles, so halo re-reads stay in
// its L2) and software-pipelined: once tile j is staged in LDS, the global
// loads of tile j+1 are issued before the red and black phases of tile j,
// so HBM traffic overlaps compute. G = ntiles gives one tile per workgroup.
struct RowRec {
    int off, gx, gy, in;
};

// Tiles first, first + slots, ... (count of them) of one level.
template <class T, bool P, int TX, int TY, int N2>
__device__ __forceinline__ void rb_rows_tiles(const T* __restrict__ pin, const T* __restrict__ rhs,
                                              T* __restrict__ pout, const Dim32 d, const W3<T> k,
                                              int zero_in, int ntx, int nty, int first, int count,
                                              int slots) {
    constexpr int NW = 4;
    constexpr int BYr = TY + 4, ROWS = (TX + 4) * BYr;
    constexpr int RYr = TY + 2, RING = (TX + 2) * RYr;
    constexpr int TILE = TX * TY;
    constexpr int LR = (ROWS + NW - 1) / NW, RR = (RING + NW - 1) / NW, TR = (TILE + NW - 1) / NW;
    static_assert(ROWS <= 256, "one thread per box row");
    extern __shared__ unsigned char raw[];
    T* box = reinterpret_cast<T*>(raw);
    __shared__ T tab[27];
    __shared__ RowRec rec[2][ROWS];
    // N2 > 0: the z extent is N2 and the x/y extents are multiples of TX/TY
    // (compile-time lane tests and tile bounds); N2 = 0: any extents.
    constexpr bool EXACT = N2 > 0;
    const int n2 = N2 > 0 ? N2 : d.n2, h2 = n2 >> 1;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (wave >= NW) __builtin_unreachable();  // 256 threads = NW wavefronts
    const int sxg = d.n1 * n2;
    auto build = [&](int buf, int tile) {
        if (threadIdx.x < ROWS) {
            const int r = threadIdx.x;
            int gx = (tile / nty) * TX - 2 + r / BYr, gy = (tile % nty) * TY - 2 + r % BYr;
            int in = 1;
            if (P) {
                gx = gx < 0 ? gx + d.n0 : (gx >= d.n0 ? gx - d.n0 : gx);
                gy = gy < 0 ? gy + d.n1 : (gy >= d.n1 ? gy - d.n1 : gy);
            } else {
                in = gx >= 0 && gx < d.n0 && gy >= 0 && gy < d.n1;
            }
            rec[buf][r] = RowRec{in ? gx * sxg + gy * n2 : 0, gx, gy, in};
        }
    };
    auto load_rec = [&](int buf, int r) {
        RowRec q = rec[buf][r];
        q.off = __builtin_amdgcn_readfirstlane(q.off);
        q.gx = __builtin_amdgcn_readfirstlane(q.gx);
        q.gy = __builtin_amdgcn_readfirstlane(q.gy);
        q.in = __builtin_amdgcn_readfirstlane(q.in);
        return q;
    };
    T pv[LR][2], rr[RR], rt[TR];
    // global loads of one tile into registers (records in rec[buf])
    auto fetch = [&](int buf, int tile) {
        const int x0 = (tile / nty) * TX - 2, y0 = (tile % nty) * TY - 2;
#pragma unroll
        for (int q = 0; q < LR; ++q) pv[q][0] = pv[q][1] = T(0);
        if (!zero_in) {
#pragma unroll
            for (int q = 0; q < LR; ++q) {
                const int r = wave + q * NW;
                if (r < ROWS) {
                    const RowRec rc = load_rec(buf, r);
                    if (P || rc.in) {
                        const T* src = pin + rc.off;
                        if (lane < n2) pv[q][0] = src[lane];
                        if (lane + 64 < n2) pv[q][1] = src[lane + 64];
                    }
                }
            }
        }
#pragma unroll
        for (int q = 0; q < RR; ++q) {
            const int rw = wave + q * NW;
            rr[q] = T(0);
            if (rw < RING && lane < h2) {
                const RowRec rc = load_rec(buf, (1 + rw / RYr) * BYr + 1 + rw % RYr);
                if (P || rc.in) rr[q] = rhs[rc.off + 2 * lane + ((rc.gx + rc.gy) & 1)];
            }
        }
#pragma unroll
        for (int q = 0; q < TR; ++q) {
            const int tw = wave + q * NW;
            rt[q] = T(0);
            if (tw < TILE && lane < h2) {
                const RowRec rc = load_rec(buf, (2 + tw / TY) * BYr + 2 + tw % TY);
                if (EXACT || (x0 + 2 + tw / TY < d.n0 && y0 + 2 + tw % TY < d.n1))
                    rt[q] = rhs[rc.off + 2 * lane + ((rc.gx + rc.gy + 1) & 1)];
            }
        }
    };
    build(0, first);
    if (!P && threadIdx.x < 27) tab[threadIdx.x] = inv_diag_entry<T>(threadIdx.x, k);
    __syncthreads();
    fetch(0, first);
    const Recip<T> inv_p = recip(T(2) * (k.w[0] + k.w[1] + k.w[2]));
    auto update = [&](const T* row, int r, int gx, int gy, int z, T b) -> T {
        // a missing neighbour adds zero
        const T zs = (P || z + 1 < n2 ? row[P && z + 1 == n2 ? 0 : z + 1] : T(0)) +
                     (P || z > 0 ? row[P && z == 0 ? n2 - 1 : z - 1] : T(0));
        const T ys = (P || gy + 1 < d.n1 ? box[(r + 1) * n2 + z] : T(0)) + (P || gy > 0 ? box[(r - 1) * n2 + z] : T(0));
        const T xs = (P || gx + 1 < d.n0 ? box[(r + BYr) * n2 + z] : T(0)) +
                     (P || gx > 0 ? box[(r - BYr) * n2 + z] : T(0));
        const Recip<T> inv = P ? inv_p : Recip<T>{tab[face_class(gx, d.n0) * 9 + face_class(gy, d.n1) * 3 + face_class(z, n2)], T(0)};
        return rb_relax(k, row[z], gs_value<T>(k, b, zs, ys, xs, inv));
    };
    for (int j = 0; j < count; ++j) {
        const int cur = j & 1;
        const int tile = first + j * slots;
        const int x0 = (tile / nty) * TX - 2, y0 = (tile % nty) * TY - 2;
#pragma unroll
        for (int q = 0; q < LR; ++q) {
            const int r = wave + q * NW;
            if (r < ROWS) {
                if (lane < n2) box[r * n2 + lane] = pv[q][0];
                if (lane + 64 < n2) box[r * n2 + lane + 64] = pv[q][1];
            }
        }
        T rrc[RR], rtc[TR];
#pragma unroll
        for (int q = 0; q < RR; ++q) rrc[q] = rr[q];
#pragma unroll
        for (int q = 0; q < TR; ++q) rtc[q] = rt[q];
        const bool more = j + 1 < count;
        if (more) build(cur ^ 1, tile + slots);
        __syncthreads();
        if (more) fetch(cur ^ 1, tile + slots);
#pragma unroll
        for (int q = 0; q < RR; ++q) {
            const int rw = wave + q * NW;
            if (rw >= RING || lane >= h2) continue;
            const int r = (1 + rw / RYr) * BYr + 1 + rw % RYr;
            const RowRec rc = load_rec(cur, r);
            if (!P && !rc.in) continue;
            T* row = box + r * n2;
            const int z = 2 * lane + ((rc.gx + rc.gy) & 1);
            row[z] = update(row, r, rc.gx, rc.gy, z, rrc[q]);
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < TR; ++q) {
            const int tw = wave + q * NW;
            if (tw >= TILE || lane >= h2) continue;
            if (!EXACT && (x0 + 2 + tw / TY >= d.n0 || y0 + 2 + tw % TY >= d.n1)) continue;
            const int r = (2 + tw / TY) * BYr + 2 + tw % TY;
            const RowRec rc = load_rec(cur, r);
            const T* row = box + r * n2;
            const int zb = 2 * lane + ((rc.gx + rc.gy + 1) & 1), zr = 2 * lane + ((rc.gx + rc.gy) & 1);
            T* dst = pout + rc.off;
            dst[zb] = update(row, r, rc.gx, rc.gy, zb, rtc[q]);
            dst[zr] = row[zr];
        }
        __syncthreads();
    }
}

template <class T, bool P, int TX, int TY, int N2>
__global__ void __launch_bounds__(256) rb_rows_kernel(const T* __restrict__ pin,
                                                      const T* __restrict__ rhs,
                                                      T* __restrict__ pout, Dim32 d, W3<T> k,
                                                      int zero_in, int ntx, int nty) {
    // tile sequence of this workgroup
    const int ntiles = ntx * nty;
    const bool by_xcd = (gridDim.x % 8 == 0) && (ntiles % 8 == 0);
    const int per = by_xcd ? ntiles / 8 : ntiles;
    const int slots = by_xcd ? int(gridDim.x) / 8 : int(gridDim.x);
    const int slot = by_xcd ? int(blockIdx.x) / 8 : int(blockIdx.x);
    const int first = (by_xcd ? int(blockIdx.x % 8) * per : 0) + slot;
    const int count = slot < per ? (per - slot + slots - 1) / slots : 0;
    if (count == 0) return;  // uniform over the workgroup
    rb_rows_tiles<T, P, TX, TY, N2>(pin, rhs, pout, d, k, zero_in, ntx, nty, first, count, slots);
}

// Pointers to a row and its four x/y neighbour rows (null where a Neumann
// neighbour does not exist).
template <class T, bool P>
struct Rows5 {
    const T *c, *xm, *xp, *ym, *yp;
};

template <class T, bool P>
__device__ inline Rows5<T, P> rows5(const T* base, int x, int y, const Dim32& d) {
    const int sx = d.n1 * d.n2, sy = d.n2;
    Rows5<T, P> r;
    r.c = base + x * sx + y * sy;
    if (P) {
        r.xm = base + (x > 0 ? x - 1 : d.n0 - 1) * sx + y * sy;
        r.xp = base + (x + 1 < d.n0 ? x + 1 : 0) * sx + y * sy;
        r.ym = base + x * sx + (y > 0 ? y - 1 : d.n1 - 1) * sy;
        r.yp = base + x * sx + (y + 1 < d.n1 ? y + 1 : 0) * sy;
    } else {
        r.xm = x > 0 ? r.c - sx : nullptr;
        r.xp = x + 1 < d.n0 ? r.c + sx : nullptr;
        r.ym = y > 0 ? r.c - sy : nullptr;
        r.yp = y + 1 < d.n1 ? r.c + sy : nullptr;
    }
    return r;
}

// (A p)_z on a row, difference form.
template <class T, bool P>
__device__ inline T apply_row(const Rows5<T, P>& r, int z, int n2, const W3<T>& k) {
    const T c = r.c[z];
    T a = T(0);
    if (P) {
        a += k.w[0] * (c - r.xp[z]);
        a += k.w[0] * (c - r.xm[z]);
        a += k.w[1] * (c - r.yp[z]);
        a += k.w[1] * (c - r.ym[z]);
        a += k.w[2] * (c - r.c[z + 1 < n2 ? z + 1 : 0]);
        a += k.w[2] * (c - r.c[z > 0 ? z - 1 : n2 - 1]);
    } else {
        if (r.xp) a += k.w[0] * (c - r.xp[z]);
        if (r.xm) a += k.w[0] * (c - r.xm[z]);
        if (r.yp) a += k.w[1] * (c - r.yp[z]);
        if (r.ym) a += k.w[1] * (c - r.ym[z]);
        if (z + 1 < n2) a += k.w[2] * (c - r.c[z + 1]);
        if (z > 0) a += k.w[2] * (c - r.c[z - 1]);
    }
    return a;
}

// coarse = avg8(rhs - A p); one wavefront per coarse row.
template <class T, bool P>
__device__ __forceinline__ void restrict_row(const T* __restrict__ p, const T* __restrict__ rhs,
                                             T* __restrict__ coarse, const Dim32 d, const W3<T> k,
                                             int row) {
    const int lane = threadIdx.x & 63;
    const int C0 = d.n0 / 2, C1 = d.n1 / 2, C2 = d.n2 / 2;
    if (row >= C0 * C1) return;
    const int cx = row / C1, cy = row - cx * C1;
    Rows5<T, P> pr[2][2];
    const T* rr[2][2];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            pr[a][b] = rows5<T, P>(p, 2 * cx + a, 2 * cy + b, d);
            rr[a][b] = rhs + (2 * cx + a) * d.n1 * d.n2 + (2 * cy + b) * d.n2;
        }
    T* out = coarse + (cx * C1 + cy) * C2;
    for (int cz = lane; cz < C2; cz += 64) {
        T v = T(0);
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    const int z = 2 * cz + c;
                    v += rr[a][b][z] - apply_row<T, P>(pr[a][b], z, d.n2, k);
                }
        out[cz] = v * T(0.125);
    }
}

template <class T, bool P>
__global__ void __launch_bounds__(256) restrict_rows_kernel(const T* __restrict__ p,
                                                            const T* __restrict__ rhs,
                                                            T* __restrict__ coarse, Dim32 d,
                                                            W3<T> k) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform
    restrict_row<T, P>(p, rhs, coarse, d, k, int(blockIdx.x) * 4 + wave);
}

// fine += trilinear(coarse) for a 2x2 group of fine rows: fine rows 2k+1 and
// 2k+2 of an axis interpolate between the same coarse rows k and k+1 (only
// their weights differ), so one wave reads the four coarse rows once and
// updates up to four fine rows. Group (kx, ky), kx in [-1, C0), ky in
// [-1, C1).
template <class T, bool P>
__global__ void __launch_bounds__(256) prolong_groups_kernel(const T* __restrict__ coarse,
                                                             T* __restrict__ fine, Dim32 d) {
    const int g = int(blockIdx.x) * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const int C0 = d.n0 / 2, C1 = d.n1 / 2, C2 = d.n2 / 2;
    if (g >= (C0 + 1) * (C1 + 1)) return;
    const int ax = g / (C1 + 1) - 1, ay = g - (ax + 1) * (C1 + 1) - 1;
    int x0, x1, y0, y1;
    if (P) {  // -1 <= ax and ax + 1 <= C0
        x0 = ax < 0 ? ax + C0 : ax; x1 = ax + 1 >= C0 ? ax + 1 - C0 : ax + 1;
        y0 = ay < 0 ? ay + C1 : ay; y1 = ay + 1 >= C1 ? ay + 1 - C1 : ay + 1;
    } else {
        x0 = ax > 0 ? ax : 0; x1 = ax + 1 < C0 - 1 ? ax + 1 : C0 - 1;
        y0 = ay > 0 ? ay : 0; y1 = ay + 1 < C1 - 1 ? ay + 1 : C1 - 1;
    }
    const T* c00 = coarse + (x0 * C1 + y0) * C2;
    const T* c01 = coarse + (x0 * C1 + y1) * C2;
    const T* c10 = coarse + (x1 * C1 + y0) * C2;
    const T* c11 = coarse + (x1 * C1 + y1) * C2;
    const int fx[2] = {2 * ax + 1, 2 * ax + 2}, fy[2] = {2 * ay + 1, 2 * ay + 2};
    // fine rows of the group (wave-uniform; null where outside the level)
    T* rows[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
            rows[i][j] = fx[i] >= 0 && fx[i] < d.n0 && fy[j] >= 0 && fy[j] < d.n1
                             ? fine + (fx[i] * d.n1 + fy[j]) * d.n2 : nullptr;
    // Two z per lane per pass (z and z + 64): every load of a pass is issued
    // before its stores, so a 128-wide row takes one memory round trip.
    for (int zs = 0; zs < d.n2; zs += 128) {
        T v[2][4], f[2][2][2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int z = zs + lane + 64 * h;
            if (z >= d.n2) continue;
            const int az = z / 2 - 1 + (z & 1);
            int z0, z1;
            if (P) { z0 = az < 0 ? az + C2 : az; z1 = az + 1 >= C2 ? az + 1 - C2 : az + 1; }
            else { z0 = az > 0 ? az : 0; z1 = az + 1 < C2 - 1 ? az + 1 : C2 - 1; }
            const T wz = (z & 1) ? T(0.25) : T(0.75);
            v[h][0] = c00[z0] * (T(1) - wz) + c00[z1] * wz;
            v[h][1] = c01[z0] * (T(1) - wz) + c01[z1] * wz;
            v[h][2] = c10[z0] * (T(1) - wz) + c10[z1] * wz;
            v[h][3] = c11[z0] * (T(1) - wz) + c11[z1] * wz;
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    if (rows[i][j]) f[h][i][j] = rows[i][j][z];
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int z = zs + lane + 64 * h;
            if (z >= d.n2) continue;
            const T v00 = v[h][0], v01 = v[h][1], v10 = v[h][2], v11 = v[h][3];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const T wx = (fx[i] & 1) ? T(0.25) : T(0.75);
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    if (!rows[i][j]) continue;
                    const T wy = (fy[j] & 1) ? T(0.25) : T(0.75);
                    rows[i][j][z] = f[h][i][j] +
                                    ((v00 * (T(1) - wy) + v01 * wy) * (T(1) - wx) + (v10 * (T(1) - wy) + v11 * wy) * wx);
                }
            }
        }
    }
}

// per-workgroup [sum r, sum r^2, sum |r|, non-finite] of r = rhs - A p,
// one wavefront per row, grid-stride over rows.
template <class T, bool P>
__global__ void __launch_bounds__(256) residual_rows_kernel(const T* __restrict__ p,
                                                            const T* __restrict__ rhs, Dim32 d,
                                                            W3<T> k, double* __restrict__ partials) {
    __shared__ double sh[4][4];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform
    double v[4] = {0.0, 0.0, 0.0, 0.0};
    for (int row = blockIdx.x * 4 + wave; row < d.n0 * d.n1; row += gridDim.x * 4) {
        const int x = row / d.n1, y = row - x * d.n1;
        const Rows5<T, P> pr = rows5<T, P>(p, x, y, d);
        const T* rr = rhs + x * d.n1 * d.n2 + y * d.n2;
        for (int z = lane; z < d.n2; z += 64) {
            const double r = double(rr[z] - apply_row<T, P>(pr, z, d.n2, k));
            if (isfinite(r)) {
                v[0] += r;
                v[1] += r * r;
                v[2] += fabs(r);
            } else {
                v[3] += 1.0;
            }
        }
    }
    for (int q = 0; q < 4; ++q) {
        double t = v[q];
#pragma unroll
        for (int dd = 32; dd >= 1; dd >>= 1) t += __shfl_xor(t, dd, WAVE);
        if (lane == 0) sh[q][wave] = t;
    }
    __syncthreads();
    if (threadIdx.x < 4) {
        double t = 0.0;
        for (int w = 0; w < 4; ++w) t += sh[threadIdx.x][w];
        partials[4 * blockIdx.x + threadIdx.x] = t;
    }
}

// ---------------------------------------------------------------------------
// FP64 iterative refinement around FP32 V-cycles: r = b - A x in FP64 with
// the FP32 copy of r written for the inner solve and [sum, sum r^2,
// sum |r|, non-finite] partials per workgroup; and x += e.

template <bool P>
__global__ void __launch_bounds__(256) refine_residual_kernel(const double* __restrict__ x,
                                                              const double* __restrict__ b,
                                                              float* __restrict__ r32, Dim32 d,
                                                              W3<double> k,
                                                              double* __restrict__ partials) {
    __shared__ double sh[4][4];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    double v[4] = {0.0, 0.0, 0.0, 0.0};
    for (int row = blockIdx.x * 4 + wave; row < d.n0 * d.n1; row += gridDim.x * 4) {
        const int xx = row / d.n1, yy = row - xx * d.n1;
        const Rows5<double, P> pr = rows5<double, P>(x, xx, yy, d);
        const int off = row * d.n2;
        for (int z = lane; z < d.n2; z += 64) {
            const double r = b[off + z] - apply_row<double, P>(pr, z, d.n2, k);
            r32[off + z] = float(r);
            if (isfinite(r)) {
                v[0] += r;
                v[1] += r * r;
                v[2] += fabs(r);
            } else {
                v[3] += 1.0;
            }
        }
    }
    for (int q = 0; q < 4; ++q) {
        double t = v[q];
#pragma unroll
        for (int dd = 32; dd >= 1; dd >>= 1) t += __shfl_xor(t, dd, WAVE);
        if (lane == 0) sh[q][wave] = t;
    }
    __syncthreads();
    if (threadIdx.x < 4) {
        double t = 0.0;
        for (int w = 0; w < 4; ++w) t += sh[threadIdx.x][w];
        partials[4 * blockIdx.x + threadIdx.x] = t;
    }
}

// One refinement step in one pass: x_out = x + e (FP64 + FP32 correction)
// and r = b - A x_out in FP64, with the neighbours' x + e formed on the fly
// from the same expression that writes them, so the result is identical to
// an update pass followed by a residual pass. Reduce: also the residual's
// block partials [sum, sum of squares, sum |.|, non-finite].
template <bool P, bool Reduce>
__global__ void __launch_bounds__(256) refine_step_kernel(const double* __restrict__ x,
                                                          const float* __restrict__ e,
                                                          const double* __restrict__ b,
                                                          double* __restrict__ xo,
                                                          float* __restrict__ r32, Dim32 d,
                                                          W3<double> k,
                                                          double* __restrict__ partials) {
    __shared__ double sh[4][4];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    double v[4] = {0.0, 0.0, 0.0, 0.0};
    for (int row = blockIdx.x * 4 + wave; row < d.n0 * d.n1; row += gridDim.x * 4) {
        const int xx = row / d.n1, yy = row - xx * d.n1;
        const Rows5<double, P> px = rows5<double, P>(x, xx, yy, d);
        const Rows5<float, P> pe = rows5<float, P>(e, xx, yy, d);
        const int off = row * d.n2;
        for (int z = lane; z < d.n2; z += 64) {
            const double c = px.c[z] + double(pe.c[z]);
            double a = 0.0;
            if (P) {
                a += k.w[0] * (c - (px.xp[z] + double(pe.xp[z])));
                a += k.w[0] * (c - (px.xm[z] + double(pe.xm[z])));
                a += k.w[1] * (c - (px.yp[z] + double(pe.yp[z])));
                a += k.w[1] * (c - (px.ym[z] + double(pe.ym[z])));
                const int zp = z + 1 < d.n2 ? z + 1 : 0, zm = z > 0 ? z - 1 : d.n2 - 1;
                a += k.w[2] * (c - (px.c[zp] + double(pe.c[zp])));
                a += k.w[2] * (c - (px.c[zm] + double(pe.c[zm])));
            } else {
                if (px.xp) a += k.w[0] * (c - (px.xp[z] + double(pe.xp[z])));
                if (px.xm) a += k.w[0] * (c - (px.xm[z] + double(pe.xm[z])));
                if (px.yp) a += k.w[1] * (c - (px.yp[z] + double(pe.yp[z])));
                if (px.ym) a += k.w[1] * (c - (px.ym[z] + double(pe.ym[z])));
                if (z + 1 < d.n2) a += k.w[2] * (c - (px.c[z + 1] + double(pe.c[z + 1])));
                if (z > 0) a += k.w[2] * (c - (px.c[z - 1] + double(pe.c[z - 1])));
            }
            const double r = b[off + z] - a;
            xo[off + z] = c;
            r32[off + z] = float(r);
            if (Reduce) {
                if (isfinite(r)) {
                    v[0] += r;
                    v[1] += r * r;
                    v[2] += fabs(r);
                } else {
                    v[3] += 1.0;
                }
            }
        }
    }
    if (!Reduce) return;
    for (int q = 0; q < 4; ++q) {
        double t = v[q];
#pragma unroll
        for (int dd = 32; dd >= 1; dd >>= 1) t += __shfl_xor(t, dd, WAVE);
        if (lane == 0) sh[q][wave] = t;
    }
    __syncthreads();
    if (threadIdx.x < 4) {
        double t = 0.0;
        for (int w = 0; w < 4; ++w) t += sh[threadIdx.x][w];
        partials[4 * blockIdx.x + threadIdx.x] = t;
    }
}

__global__ void refine_update_kernel(double* __restrict__ x, const float* __restrict__ e,
                                     int64_t count) {
    for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < count;
         i += int64_t(gridDim.x) * blockDim.x)
        x[i] = x[i] + double(e[i]);
}

// ---------------------------------------------------------------------------
// single-workgroup V-cycle over the coarse levels, all arrays in LDS. Like
// the fine levels it removes no means: the operator annihilates constants,
// smoothing and prolongation carry a constant unchanged, restricted
// residuals of a zero-mean right-hand side have zero mean, and the coarsest
// inv(A + 11^T/n) solve returns the mean of its right-hand side, so the
// reference's mean subtractions change only rounding; the caller removes
// the level-0 mean once after the last cycle.

#include "mgcoarse.hpp"

template <class T, bool P>
__global__ void __launch_bounds__(COARSE_THREADS) coarse_cycle_kernel(CoarseArgs<T> a) {
    coarse_cycle_body<T, P>(a);
}

// ---------------------------------------------------------------------------
// batched kernels: entry i of a launch's descriptor array covers workgroups
// [begin_i, begin_{i+1}); workgroup b finds its entry by binary search over
// the (few) entries with wave-uniform scalar loads.

template <class D>
__device__ inline int find_entry(const D* __restrict__ desc, int n, int b) {
    int lo = 0, hi = n;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (desc[mid].begin <= b) lo = mid;
        else hi = mid;
    }
    return __builtin_amdgcn_readfirstlane(lo);
}

struct StageDesc {
    StageArgs<float> a;
    const int32_t* active;
    int begin;
};

struct RefDesc {
    const double* x;
    const float* e;
    const double* b;
    double* xo;
    float* r32;
    const int32_t* active;
    Dim32 d;
    W3<double> k;
    int begin;
};

struct VecDesc {
    double* x;
    int n;
    int begin;
};

constexpr int VEC_CHUNK = 4096;  // elements per workgroup in batched vector passes

// The stage of every instance that has the level, tiles in the order of the
// instances (not dealt to the XCDs in runs as in stage_kernel).
template <bool P, int TX, int NPH, bool RESTRICT>
__global__ void __launch_bounds__((Tile3<float, TX, 8, NPH, RESTRICT>::NT)) stage_batch_kernel(
    const StageDesc* __restrict__ desc, int n) {
    extern __shared__ unsigned char raw[];
    const int b = blockIdx.x;
    const StageDesc& s = desc[find_entry(desc, n, b)];
    if (s.active[0] == 0) return;  // uniform over the workgroup
    stage_tile<float, P, true, TX, 8, NPH, RESTRICT>(s.a, b - s.begin, reinterpret_cast<float*>(raw));
}

template <class T, bool P>
__global__ void __launch_bounds__(COARSE_THREADS) coarse_batch_kernel(const CoarseArgs<T>* __restrict__ args) {
    const CoarseArgs<T>& a = args[blockIdx.x];
    if (a.active && a.active[0] == 0) return;
    coarse_cycle_body<T, P>(a);
}

__device__ inline void block_stats(double v[4], double* __restrict__ out) {
    __shared__ double sh[4][4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int q = 0; q < 4; ++q) {
        double t = v[q];
#pragma unroll
        for (int dd = 32; dd >= 1; dd >>= 1) t += __shfl_xor(t, dd, WAVE);
        if (lane == 0) sh[q][wave] = t;
    }
    __syncthreads();
    if (threadIdx.x < 4) {
        double t = 0.0;
        for (int w = 0; w < 4; ++w) t += sh[threadIdx.x][w];
        out[threadIdx.x] = t;
    }
}

__device__ inline void add_stats(double v[4], double r) {
    if (isfinite(r)) {
        v[0] += r;
        v[1] += r * r;
        v[2] += fabs(r);
    } else {
        v[3] += 1.0;
    }
}

// Step: x_out = x + e and r = b - A x_out (one wavefront per row);
// otherwise r = b - A x. Inactive instances copy x to x_out (Step).
template <bool P, bool Step, bool Reduce>
__global__ void __launch_bounds__(256) refine_batch_kernel(const RefDesc* __restrict__ desc, int n,
                                                           double* __restrict__ partials) {
    const int b = blockIdx.x;
    const RefDesc& s = desc[find_entry(desc, n, b)];
    const bool live = !(s.active && s.active[0] == 0);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const Dim32 d = s.d;
    const W3<double> k = s.k;
    const int row = (b - s.begin) * 4 + wave;
    double v[4] = {0.0, 0.0, 0.0, 0.0};
    if (row < d.n0 * d.n1) {
        const int off = row * d.n2;
        if (!live) {
            if (Step)
                for (int z = lane; z < d.n2; z += 64) s.xo[off + z] = s.x[off + z];
        } else {
            const int xx = row / d.n1, yy = row - xx * d.n1;
            const Rows5<double, P> px = rows5<double, P>(s.x, xx, yy, d);
            const Rows5<float, P> pe = rows5<float, P>(s.e, xx, yy, d);
            auto val = [&](const double* xr, const float* er, int z) -> double {
                return Step ? xr[z] + double(er[z]) : xr[z];
            };
            for (int z = lane; z < d.n2; z += 64) {
                const double c = val(px.c, pe.c, z);
                double a = 0.0;
                if (P) {
                    a += k.w[0] * (c - val(px.xp, pe.xp, z));
                    a += k.w[0] * (c - val(px.xm, pe.xm, z));
                    a += k.w[1] * (c - val(px.yp, pe.yp, z));
                    a += k.w[1] * (c - val(px.ym, pe.ym, z));
                    const int zp = z + 1 < d.n2 ? z + 1 : 0, zm = z > 0 ? z - 1 : d.n2 - 1;
                    a += k.w[2] * (c - val(px.c, pe.c, zp));
                    a += k.w[2] * (c - val(px.c, pe.c, zm));
                } else {
                    if (px.xp) a += k.w[0] * (c - val(px.xp, pe.xp, z));
                    if (px.xm) a += k.w[0] * (c - val(px.xm, pe.xm, z));
                    if (px.yp) a += k.w[1] * (c - val(px.yp, pe.yp, z));
                    if (px.ym) a += k.w[1] * (c - val(px.ym, pe.ym, z));
                    if (z + 1 < d.n2) a += k.w[2] * (c - val(px.c, pe.c, z + 1));
                    if (z > 0) a += k.w[2] * (c - val(px.c, pe.c, z - 1));
                }
                const double r = s.b[off + z] - a;
                if (Step) s.xo[off + z] = c;
                s.r32[off + z] = float(r);
                if (Reduce) add_stats(v, r);
            }
        }
    }
    if (Reduce) block_stats(v, partials + 4 * b);
}

// Per instance: sum its workgroups' partials in a fixed order, store the
// stats at results[16 i + slot]; slot 0 (the residual) also updates
// active[i] (0 once the residual meets tol[i] or is non-finite). Frozen
// (inactive) instances are left untouched.
template <class D>
__global__ void __launch_bounds__(64) batch_reduce_kernel(const D* __restrict__ desc, int n,
                                                          int total_blocks,
                                                          const double* __restrict__ partials,
                                                          double* __restrict__ results, int slot,
                                                          const double* __restrict__ tol,
                                                          int32_t* __restrict__ active) {
    const int i = blockIdx.x;
    if (slot == 0 && active[i] == 0) return;
    const int beg = desc[i].begin, end = i + 1 < n ? desc[i + 1].begin : total_blocks;
    double v[4] = {0.0, 0.0, 0.0, 0.0};
    for (int b = beg + int(threadIdx.x); b < end; b += 64)
        for (int q = 0; q < 4; ++q) v[q] += partials[4 * b + q];
    for (int q = 0; q < 4; ++q) {
#pragma unroll
        for (int dd = 32; dd >= 1; dd >>= 1) v[q] += __shfl_xor(v[q], dd, WAVE);
    }
    if (threadIdx.x == 0) {
        for (int q = 0; q < 4; ++q) results[16 * i + slot + q] = v[q];
        if (slot == 0 && (v[3] > 0.0 || !(sqrt(v[1]) > tol[i]))) active[i] = 0;
    }
}

__global__ void __launch_bounds__(256) vec_partials_kernel(const VecDesc* __restrict__ desc, int n,
                                                           double* __restrict__ partials) {
    const int b = blockIdx.x;
    const VecDesc& s = desc[find_entry(desc, n, b)];
    const int lo = (b - s.begin) * VEC_CHUNK, hi = min(s.n, lo + VEC_CHUNK);
    double v[4] = {0.0, 0.0, 0.0, 0.0};
    for (int j = lo + int(threadIdx.x); j < hi; j += 256) add_stats(v, s.x[j]);
    block_stats(v, partials + 4 * b);
}

__global__ void __launch_bounds__(256) vec_sub_mean_kernel(const VecDesc* __restrict__ desc, int n,
                                                           const double* __restrict__ results,
                                                           int slot) {
    const int b = blockIdx.x;
    const int i = find_entry(desc, n, b);
    const VecDesc& s = desc[i];
    const double m = results[16 * i + slot] / double(s.n);
    const int lo = (b - s.begin) * VEC_CHUNK, hi = min(s.n, lo + VEC_CHUNK);
    for (int j = lo + int(threadIdx.x); j < hi; j += 256) s.x[j] = s.x[j] - m;
}

__global__ void batch_begin_kernel(int n, const double* __restrict__ results, double* __restrict__ tol,
                                   int32_t* __restrict__ active, double rtol, double atol) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    // b statistics after the mean removal sit in slot 8
    tol[i] = fmax(atol, rtol * sqrt(results[16 * i + 8 + 1]));
    active[i] = 1;
}


// ---------------------------------------------------------------------------
// host driver

// Dynamic LDS a kernel may request: the device's per-workgroup LDS minus the
// kernel's static LDS. The first call per (kernel, device) raises the
// kernel's dynamic-LDS attribute to that amount; `need` is checked against it.
int dynamic_lds(const void* fn, size_t need) {
    struct Entry { const void* fn; int dev; size_t avail; };
    static std::mutex lock;
    static Entry cache[64];
    static int used = 0;
    int dev = 0;
    AFSI_HIP(hipGetDevice(&dev));
    size_t avail = 0;
    bool found = false;
    {
        std::lock_guard<std::mutex> g(lock);
        for (int i = 0; i < used && !found; ++i)
            if (cache[i].fn == fn && cache[i].dev == dev) { avail = cache[i].avail; found = true; }
    }
    if (!found) {
        int per_block = 0, optin = 0;
        AFSI_HIP(hipDeviceGetAttribute(&per_block, hipDeviceAttributeMaxSharedMemoryPerBlock, dev));
        AFSI_HIP(hipDeviceGetAttribute(&optin, hipDeviceAttributeSharedMemPerBlockOptin, dev));
        const size_t limit = size_t(per_block > optin ? per_block : optin);
        hipFuncAttributes attr{};
        AFSI_HIP(hipFuncGetAttributes(&attr, fn));
        avail = limit > attr.sharedSizeBytes ? limit - attr.sharedSizeBytes : 0;
        AFSI_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, int(avail)));
        std::lock_guard<std::mutex> g(lock);
        if (used < 64) cache[used++] = Entry{fn, dev, avail};
    }
    if (need > avail) {
        set_error("kernel needs %zu bytes of dynamic LDS; the device allows %zu", need, avail);
        return E_LIMIT;
    }
    return OK;
}

template <class T>
struct FastRunner {
    const afsi_mg3d_plan& pl;
    hipStream_t s;
    int coarse_first;  // first level solved in LDS

    T* P(int l) const { return static_cast<T*>(pl.p[l]); }
    T* R(int l) const { return static_cast<T*>(pl.rhs[l]); }
    T* W(int l) const { return static_cast<T*>(pl.tmp[l]); }
    Dim32 D(int l) const { return Dim32{int(pl.n[l][0]), int(pl.n[l][1]), int(pl.n[l][2])}; }
    int64_t cells(int l) const { return pl.n[l][0] * pl.n[l][1] * pl.n[l][2]; }
    W3<T> K(int l) const {
        W3<T> k;
        for (int a = 0; a < 3; ++a) k.w[a] = T(pl.inv_h2[l][a]);
        k.relax = T(pl.relax > 0.0 ? pl.relax : 1.0);
        return k;
    }

    bool rows_ok(int l) const { return pl.n[l][2] <= ZROW && pl.n[l][2] % 2 == 0; }

    template <int TXr, int TYr, int N2>
    int rb_rows_n(int l, const T* in, T* out, bool zero_in) const {
        const Dim32 d = D(l);
        const int ntx = int(cdiv(d.n0, TXr)), nty = int(cdiv(d.n1, TYr));
        const int ntiles = ntx * nty;
        const size_t bytes = size_t((TXr + 4) * (TYr + 4)) * d.n2 * sizeof(T);
        const void* fn = pl.periodic ? reinterpret_cast<const void*>(rb_rows_kernel<T, true, TXr, TYr, N2>)
                                     : reinterpret_cast<const void*>(rb_rows_kernel<T, false, TXr, TYr, N2>);
        if (int r = dynamic_lds(fn, bytes)) return r;
        int g = pl.sweep_blocks[l] > 0 ? pl.sweep_blocks[l] : ntiles;
        if (g > ntiles) g = ntiles;
        if (pl.periodic)
            rb_rows_kernel<T, true, TXr, TYr, N2><<<unsigned(g), 256, bytes, s>>>(in, R(l), out, d, K(l), zero_in, ntx, nty);
        else
            rb_rows_kernel<T, false, TXr, TYr, N2><<<unsigned(g), 256, bytes, s>>>(in, R(l), out, d, K(l), zero_in, ntx, nty);
        AFSI_LAUNCH_CHECK();
        return OK;
    }

    // z extent as a compile-time constant where the level tiles exactly
    template <int TXr, int TYr>
    int rb_rows(int l, const T* in, T* out, bool zero_in) const {
        const Dim32 d = D(l);
        if (d.n0 % TXr == 0 && d.n1 % TYr == 0) {
            if (d.n2 == 128) return rb_rows_n<TXr, TYr, 128>(l, in, out, zero_in);
            if (d.n2 == 64) return rb_rows_n<TXr, TYr, 64>(l, in, out, zero_in);
            if (d.n2 == 32) return rb_rows_n<TXr, TYr, 32>(l, in, out, zero_in);
        }
        return rb_rows_n<TXr, TYr, 0>(l, in, out, zero_in);
    }

    int sweep(int l, const T* in, T* out, bool zero_in) const {
        const Dim32 d = D(l);
        const W3<T> k = K(l);
        if (pl.smoother == 1 && rows_ok(l)) {
            int tile = pl.sweep_tile[l];
            if (tile != 2 && tile != 4 && tile != 8 && tile != 84)
                tile = cdiv(d.n0, 4) * cdiv(d.n1, 4) >= 1024 ? 4 : 2;
            if (tile == 8) return rb_rows<8, 8>(l, in, out, zero_in);
            if (tile == 84) return rb_rows<8, 4>(l, in, out, zero_in);
            if (tile == 4) return rb_rows<4, 4>(l, in, out, zero_in);
            return rb_rows<2, 2>(l, in, out, zero_in);
        }
        if (pl.smoother == 1) {
            // 8x8x32 tiles on large levels, 4x4x32 where that leaves < 512 tiles
            const bool big = cdiv(d.n0, 8) * cdiv(d.n1, 8) * cdiv(d.n2, 32) >= 512;
            const int tx = big ? 8 : 4, ty = big ? 8 : 4, tz = 32;
            const int ntx = int(cdiv(d.n0, tx)), nty = int(cdiv(d.n1, ty)), ntz = int(cdiv(d.n2, tz));
            const unsigned g = unsigned(ntx * nty * ntz);
            if (big) {
                if (pl.periodic)
                    rb_sweep_kernel<T, true, 8, 8, 32, 512><<<g, 512, 0, s>>>(in, R(l), out, d, k, zero_in, ntx, nty, ntz);
                else
                    rb_sweep_kernel<T, false, 8, 8, 32, 512><<<g, 512, 0, s>>>(in, R(l), out, d, k, zero_in, ntx, nty, ntz);
            } else {
                if (pl.periodic)
                    rb_sweep_kernel<T, true, 4, 4, 32, 256><<<g, 256, 0, s>>>(in, R(l), out, d, k, zero_in, ntx, nty, ntz);
                else
                    rb_sweep_kernel<T, false, 4, 4, 32, 256><<<g, 256, 0, s>>>(in, R(l), out, d, k, zero_in, ntx, nty, ntz);
            }
        } else {
            const unsigned g = grid_for(cells(l), 256, 16384);
            if (pl.periodic)
                jacobi_fast_kernel<T, true><<<g, 256, 0, s>>>(in, R(l), out, d, k, T(pl.omega), zero_in);
            else
                jacobi_fast_kernel<T, false><<<g, 256, 0, s>>>(in, R(l), out, d, k, T(pl.omega), zero_in);
        }
        AFSI_LAUNCH_CHECK();
        return OK;
    }

    // nu sweeps ping-ponging between p and tmp; `cur` tracks the result.
    int smooth(int l, T*& cur, bool zero_first) const {
        for (int it = 0; it < pl.nu; ++it) {
            T* out = (cur == P(l)) ? W(l) : P(l);
            if (int r = sweep(l, cur, out, it == 0 && zero_first)) return r;
            cur = out;
        }
        return OK;
    }

    int coarse(int first, const T* p_in, T* p_out) const {
        CoarseArgs<T> a;
        const size_t bytes = size_t(coarse_args<T>(pl, first, a)) * sizeof(T);
        a.p_in = p_in;
        a.p_out = p_out;
        if (int r = dynamic_lds(pl.periodic ? reinterpret_cast<const void*>(coarse_cycle_kernel<T, true>)
                                            : reinterpret_cast<const void*>(coarse_cycle_kernel<T, false>),
                                bytes))
            return r;
        if (pl.periodic) coarse_cycle_kernel<T, true><<<1, COARSE_THREADS, bytes, s>>>(a);
        else coarse_cycle_kernel<T, false><<<1, COARSE_THREADS, bytes, s>>>(a);
        AFSI_LAUNCH_CHECK();
        return OK;
    }

    // Whether level l's smoothing stages run as stage launches.
    bool staged(int l) const {
        if (pl.n[l][1] * pl.n[l][2] >= (int64_t(1) << 28)) return false;  // 32-bit byte offsets in a plane
        if (l >= coarse_first || pl.fuse_cells < 0 || (pl.fuse_cells > 0 && cells(l) > int64_t(pl.fuse_cells))) return false;
        const void* ptrs[4] = {pl.p[l], pl.tmp[l], pl.rhs[l], pl.p[l + 1]};
        for (const void* q : ptrs)
            if (reinterpret_cast<uintptr_t>(q) % 16) return false;
        return true;
    }

    template <bool Per, bool GS, int TX, int TY, int NPH, bool RESTRICT>
    int stage_n(const StageArgs<T>& a) const {
        using G = Tile3<T, TX, TY, NPH, RESTRICT>;
        if (int r = dynamic_lds(reinterpret_cast<const void*>(stage_kernel<T, Per, GS, TX, TY, NPH, RESTRICT>), G::LDS)) return r;
        const int tiles = stage_tiles(a.d, TX, TY);
        stage_kernel<T, Per, GS, TX, TY, NPH, RESTRICT><<<unsigned(tiles), G::NT, G::LDS, s>>>(a, tiles);
        AFSI_LAUNCH_CHECK();
        return OK;
    }

    template <int TX, int TY, int NPH, bool GS>
    int stage_tx(const StageArgs<T>& a) const {
        if (pl.periodic) return a.restricted ? stage_n<true, GS, TX, TY, NPH, true>(a) : stage_n<true, GS, TX, TY, NPH, false>(a);
        return a.restricted ? stage_n<false, GS, TX, TY, NPH, true>(a) : stage_n<false, GS, TX, TY, NPH, false>(a);
    }

    // Phases per launch and tile of a level. Two phases keep the halo small
    // where the level fills the chip several times over (redundant cells are
    // then the cost); smaller levels are bound by launches and by the length of
    // one workgroup's instruction stream, so they take four phases and, up to
    // 256 (down) or below 256 (up) 8x8 tiles, the shorter 4x8 tile. Measured
    // per V-cycle in us with level 0 in two phases / four on 4x8 / four on 8x8,
    // V(2,2) red-black or V(4,4) Jacobi:
    //             periodic RB FP64   periodic RB FP32   closed Jacobi FP64
    //   48^3      56.3 47.4 53.8     49.4 41.7 45.0     76.9 67.1 76.0
    //   64^3      60.8 58.3 59.0     53.0 50.4 50.1     82.2 81.8 81.7
    //   80^3      92.1 80.2 85.3     73.5 62.9 67.3     126 118 132
    //   96^3      93.9 98.6 96.3     74.2 73.7 72.2     141 155 179
    //   112^3     178 159 168        138 121 122        241 239 285
    //   128^3     136 158 144        102 112 103        221 265 299
    // Over both boundary types, smoothers and precisions from 32^3 to 160^3 the
    // rule is within 8% of the best of the three except where extents are no
    // multiples of the tile (112^3 red-black: 4% to 17% behind 4x8) and for
    // closed FP64 Jacobi from 80^3 to 112x96x96, whose 8x8 four-phase form
    // runs out of registers (12% to 26% behind the best).
    static constexpr int64_t WIDE_TILES = 1024;
    bool wide(int l) const { return stage_tiles(D(l), 8, 8) >= WIDE_TILES; }

    template <bool GS>
    int stage_launch(const StageArgs<T>& a, bool wide_level, bool up) const {
        if (wide_level) return stage_tx<8, 8, 2, GS>(a);
        const int tiles = stage_tiles(a.d, 8, 8);
        return (up ? tiles < 256 : tiles <= 256) ? stage_tx<4, 8, 4, GS>(a) : stage_tx<8, 8, 4, GS>(a);
    }

    // One smoothing stage of level l (restriction or prolongation included)
    // as launches of a few phases; p and tmp alternate.
    int stage(int l, T*& cur, bool up, const T* coarse, bool zero) const {
        const bool two = wide(l);
        const int per = two ? 2 : 4;
        const int phases = pl.smoother == 1 ? 2 * pl.nu : pl.nu, chunks = (phases + per - 1) / per;
        for (int c = 0; c < chunks; ++c) {
            StageArgs<T> a{};
            a.in = cur;
            a.rhs = R(l);
            a.out = cur == P(l) ? W(l) : P(l);
            a.coarse = up && c == 0 ? coarse : nullptr;
            a.restricted = !up && c == chunks - 1 ? R(l + 1) : nullptr;
            a.d = D(l);
            a.k = K(l);
            a.omega = T(pl.omega);
            a.count = std::min(per, phases - c * per);
            a.zero = zero && c == 0;
            const int r = pl.smoother == 1 ? stage_launch<true>(a, two, up) : stage_launch<false>(a, two, up);
            if (r) return r;
            cur = a.out;
        }
        return OK;
    }

    int cycle(int l, T*& cur, bool zero_initial = false) const {
        if (l == coarse_first) return coarse(l, (l == 0 && !zero_initial) ? cur : nullptr, cur);
        if (staged(l)) {  // as many launches up as down: the iterate ends in cur's first buffer
            if (int r = stage(l, cur, false, nullptr, l > 0 || zero_initial)) return r;
            T* cc = P(l + 1);
            if (int r = cycle(l + 1, cc)) return r;
            return stage(l, cur, true, cc, false);
        }
        // coarse iterates (and a zero initial level-0 iterate) start at zero
        if (int r = smooth(l, cur, l > 0 || zero_initial)) return r;
        const Dim32 d = D(l);
        const W3<T> k = K(l);
        if (rows_ok(l)) {
            const unsigned g = unsigned(cdiv(int64_t(d.n0 / 2) * (d.n1 / 2), 4));
            if (pl.periodic) restrict_rows_kernel<T, true><<<g, 256, 0, s>>>(cur, R(l), R(l + 1), d, k);
            else restrict_rows_kernel<T, false><<<g, 256, 0, s>>>(cur, R(l), R(l + 1), d, k);
        } else {
            const unsigned g = grid_for(cells(l + 1), 256, 16384);
            if (pl.periodic) restrict_fast_kernel<T, true><<<g, 256, 0, s>>>(cur, R(l), R(l + 1), d, k);
            else restrict_fast_kernel<T, false><<<g, 256, 0, s>>>(cur, R(l), R(l + 1), d, k);
        }
        AFSI_LAUNCH_CHECK();
        T* cc = P(l + 1);
        if (int r = cycle(l + 1, cc)) return r;
        if (rows_ok(l)) {
            const unsigned gf = unsigned(cdiv(int64_t(d.n0 / 2 + 1) * (d.n1 / 2 + 1), 4));
            if (pl.periodic) prolong_groups_kernel<T, true><<<gf, 256, 0, s>>>(cc, cur, d);
            else prolong_groups_kernel<T, false><<<gf, 256, 0, s>>>(cc, cur, d);
        } else {
            const unsigned gf = grid_for(cells(l), 256, 16384);
            if (pl.periodic) prolong_fast_kernel<T, true><<<gf, 256, 0, s>>>(cc, cur, d);
            else prolong_fast_kernel<T, false><<<gf, 256, 0, s>>>(cc, cur, d);
        }
        AFSI_LAUNCH_CHECK();
        return smooth(l, cur, false);
    }
};

// First level solved by the LDS kernel: at most COARSE_MAX cells, every
// extent <= 64, and at most COARSE_TOTAL cells on all of its levels.
static int choose_coarse(const afsi_mg3d_plan& pl) {
    for (int l = 0; l < pl.levels; ++l) {
        int64_t total = 0;
        bool ok = pl.n[l][0] * pl.n[l][1] * pl.n[l][2] <= COARSE_MAX;
        for (int j = l; j < pl.levels && ok; ++j) {
            ok = pl.n[j][0] <= 64 && pl.n[j][1] <= 64 && pl.n[j][2] <= 64;
            total += pl.n[j][0] * pl.n[j][1] * pl.n[j][2];
        }
        if (ok && total <= COARSE_TOTAL) return l;
    }
    return -1;
}

template <class T>
static int fast_check(const afsi_mg3d_plan* pl) {
    AFSI_REQUIRE(pl && pl->levels >= 1 && pl->levels <= AFSI_MG_MAX_LEVELS, "invalid multigrid plan");
    AFSI_REQUIRE(pl->nu >= 1 && (pl->smoother == 0 || pl->smoother == 1), "invalid smoother");
    AFSI_REQUIRE(pl->reduce_partials && pl->reduce_result, "missing reduction scratch");
    for (int l = 0; l < pl->levels; ++l) {
        AFSI_REQUIRE(pl->n[l][0] > 0 && pl->n[l][1] > 0 && pl->n[l][2] > 0 && pl->p[l] && pl->rhs[l],
                     "invalid level %d", l);
        AFSI_REQUIRE(pl->n[l][0] * pl->n[l][1] * pl->n[l][2] < (int64_t(1) << 31),
                     "level %d exceeds 2^31 cells", l);
        AFSI_REQUIRE(pl->tmp[l], "missing smoothing buffer at level %d", l);
        if (l + 1 < pl->levels)
            for (int a = 0; a < 3; ++a)
                AFSI_REQUIRE(pl->n[l][a] == 2 * pl->n[l + 1][a], "levels %d/%d are not 2:1", l, l + 1);
    }
    const int last = pl->levels - 1;
    AFSI_REQUIRE(pl->coarse_inverse &&
                     pl->coarse_cells == pl->n[last][0] * pl->n[last][1] * pl->n[last][2],
                 "coarse inverse does not match the coarsest level");
    AFSI_REQUIRE(pl->coarse_cells <= 512, "coarsest level exceeds 512 cells");
    AFSI_REQUIRE(choose_coarse(*pl) >= 0,
                 "fused driver needs coarse levels with extents <= 64 (use the unfused driver)");
    return OK;
}

template <class T>
static int fast_cycles(const afsi_mg3d_plan* pl, int32_t cycles, void* stream) {
    if (int r = fast_check<T>(pl)) return r;
    AFSI_REQUIRE(cycles >= 0, "negative cycle count");
    const FastRunner<T> run{*pl, hipStream_t(stream), choose_coarse(*pl)};
    for (int c = 0; c < cycles; ++c) {
        T* cur = run.P(0);
        if (int r = run.cycle(0, cur, c == 0 && pl->zero_initial)) return r;
        AFSI_REQUIRE(cur == run.P(0), "level-0 iterate left the canonical buffer");
    }
    return OK;
}

template <class T>
static int fast_residual(const afsi_mg3d_plan* pl, void* stream) {
    if (int r = fast_check<T>(pl)) return r;
    const FastRunner<T> run{*pl, hipStream_t(stream), choose_coarse(*pl)};
    const hipStream_t s = hipStream_t(stream);
    const int64_t nb = grid_for(run.cells(0), 256, pl->partials_capacity / 4);
    AFSI_REQUIRE(4 * nb <= pl->partials_capacity, "reduction scratch too small");
    if (run.rows_ok(0)) {
        const int64_t rows = pl->n[0][0] * pl->n[0][1];
        int64_t nr = cdiv(rows, 4);
        if (nr > pl->partials_capacity / 4) nr = pl->partials_capacity / 4;
        if (pl->periodic)
            residual_rows_kernel<T, true><<<unsigned(nr), 256, 0, s>>>(run.P(0), run.R(0), run.D(0), run.K(0),
                                                                      pl->reduce_partials);
        else
            residual_rows_kernel<T, false><<<unsigned(nr), 256, 0, s>>>(run.P(0), run.R(0), run.D(0), run.K(0),
                                                                       pl->reduce_partials);
        AFSI_LAUNCH_CHECK();
        return launch_reduce_final(pl->reduce_partials, nr, pl->reduce_result, s);
    }
    if (pl->periodic)
        residual_partials_kernel<T, true><<<unsigned(nb), 256, 0, s>>>(run.P(0), run.R(0), run.D(0), run.K(0),
                                                                      pl->reduce_partials);
    else
        residual_partials_kernel<T, false><<<unsigned(nb), 256, 0, s>>>(run.P(0), run.R(0), run.D(0), run.K(0),
                                                                       pl->reduce_partials);
    AFSI_LAUNCH_CHECK();
    return launch_reduce_final(pl->reduce_partials, nb, pl->reduce_result, s);
}

// ---------------------------------------------------------------------------
// batched mixed-precision solve (host side)

struct BatchLayout {
    int n = 0, levels = 0, nu = 0, periodic = 0;
    int cf[1024];                      // first LDS-solved level per instance
    std::vector<int> members[AFSI_MG_MAX_LEVELS];
    // smoothing stages of a level: `chunks` launches down (desc 0..chunks-1),
    // as many up, and the first down launch of a later inner cycle (last desc)
    size_t stage_off[AFSI_MG_MAX_LEVELS];
    int tile_x[AFSI_MG_MAX_LEVELS], phases[AFSI_MG_MAX_LEVELS], chunks[AFSI_MG_MAX_LEVELS];
    int stage_blocks[AFSI_MG_MAX_LEVELS];
    size_t coarse_off[2] = {0, 0}, coarse_lds = 0;  // first cycle of an iteration (zero start); later ones
    size_t ref_off[4] = {0, 0, 0, 0};  // residual of x[0]; step from x[0]; step from x[1]; residual of x[1]
    int ref_blocks = 0;
    size_t vec_off[3] = {0, 0, 0};     // b, x[0], x[1]
    int vec_blocks[3] = {0, 0, 0};
    size_t total = 0;
    int64_t partials = 0;              // doubles
};

static size_t align64(size_t b) { return (b + 63) & ~size_t(63); }

static int batch_layout(const afsi_mgb_batch* bt, BatchLayout& L) {
    AFSI_REQUIRE(bt && bt->items && bt->count >= 1 && bt->count <= 1024, "invalid batch (1..1024 instances)");
    L.n = bt->count;
    L.periodic = bt->items[0].plan.periodic;
    L.nu = bt->items[0].plan.nu;
    for (int i = 0; i < L.n; ++i) {
        const afsi_mgb_item& it = bt->items[i];
        const afsi_mg3d_plan& pl = it.plan;
        if (int r = fast_check<float>(&pl)) return r;
        AFSI_REQUIRE(pl.periodic == L.periodic, "instances of one batch share the boundary type");
        AFSI_REQUIRE(pl.smoother == 1 && pl.nu == L.nu, "batched instances use red-black GS with one nu");
        AFSI_REQUIRE(it.x[0] && it.x[1] && it.b && it.x[0] != it.x[1], "invalid FP64 iterate buffers");
        L.cf[i] = choose_coarse(pl);
        for (int l = 0; l < L.cf[i]; ++l)
            AFSI_REQUIRE(pl.n[l][2] <= ZROW && pl.n[l][2] % 2 == 0 && pl.n[l][0] % 2 == 0 &&
                             pl.n[l][1] % 2 == 0,
                         "instance %d level %d: batched solves need even extents and z <= %d", i, l, ZROW);
        AFSI_REQUIRE(pl.n[0][0] * pl.n[0][1] * pl.n[0][2] < (int64_t(1) << 31), "instance too large");
        if (L.cf[i] > L.levels) L.levels = L.cf[i];
    }
    size_t off = 0;
    int64_t partials = 0;
    for (int l = 0; l < L.levels; ++l) {
        L.members[l].clear();
        int64_t tiles = 0;
        for (int i = 0; i < L.n; ++i) {
            if (l >= L.cf[i]) continue;
            L.members[l].push_back(i);
            const int64_t* nn = bt->items[i].plan.n[l];
            tiles += stage_tiles(Dim32{int(nn[0]), int(nn[1]), int(nn[2])}, 8, 8);
        }
        // the rule of FastRunner::wide and stage_launch over the whole level, one
        // tile for both directions
        L.phases[l] = tiles >= FastRunner<float>::WIDE_TILES ? 2 : 4;
        L.tile_x[l] = tiles < 256 ? 4 : 8;
        L.chunks[l] = (2 * L.nu + L.phases[l] - 1) / L.phases[l];
        int64_t blocks = 0;
        for (int i : L.members[l]) {
            const int64_t* nn = bt->items[i].plan.n[l];
            blocks += stage_tiles(Dim32{int(nn[0]), int(nn[1]), int(nn[2])}, L.tile_x[l], 8);
        }
        AFSI_REQUIRE(blocks < (int64_t(1) << 30), "batch level too large");
        L.stage_blocks[l] = int(blocks);
        L.stage_off[l] = off;
        off = align64(off + L.members[l].size() * size_t(2 * L.chunks[l] + 1) * sizeof(StageDesc));
    }
    for (int c = 0; c < 2; ++c) {
        L.coarse_off[c] = off;
        off = align64(off + size_t(L.n) * sizeof(CoarseArgs<float>));
    }
    L.coarse_lds = 0;
    L.ref_blocks = 0;
    for (int i = 0; i < L.n; ++i) {
        const afsi_mg3d_plan& pl = bt->items[i].plan;
        CoarseArgs<float> a;
        const size_t bytes = size_t(coarse_args<float>(pl, L.cf[i], a)) * sizeof(float);
        if (bytes > L.coarse_lds) L.coarse_lds = bytes;
        L.ref_blocks += int(cdiv(pl.n[0][0] * pl.n[0][1], 4));
    }
    for (int v = 0; v < 4; ++v) {
        L.ref_off[v] = off;
        off = align64(off + size_t(L.n) * sizeof(RefDesc));
    }
    for (int v = 0; v < 3; ++v) {
        L.vec_off[v] = off;
        off = align64(off + size_t(L.n) * sizeof(VecDesc));
        int nb = 0;
        for (int i = 0; i < L.n; ++i) {
            const int64_t* nn = bt->items[i].plan.n[0];
            nb += int(cdiv(nn[0] * nn[1] * nn[2], VEC_CHUNK));
        }
        L.vec_blocks[v] = nb;
    }
    L.total = off;
    partials = std::max<int64_t>(L.ref_blocks, L.vec_blocks[0]);
    L.partials = 4 * partials;
    return OK;
}

template <class D>
static D* at(void* ws, size_t off) {
    return reinterpret_cast<D*>(static_cast<char*>(ws) + off);
}

static int batch_prepare(const afsi_mgb_batch* bt, hipStream_t s) {
    BatchLayout L;
    if (int r = batch_layout(bt, L)) return r;
    AFSI_REQUIRE(bt->workspace && bt->workspace_bytes >= L.total, "batch workspace too small");
    AFSI_REQUIRE(bt->active && bt->tol && bt->results && bt->partials, "missing batch state buffers");
    std::vector<char> host(L.total, 0);
    void* hw = host.data();
    for (int l = 0; l < L.levels; ++l) {
        int begin = 0;
        const size_t m = L.members[l].size();
        StageDesc* descs = at<StageDesc>(hw, L.stage_off[l]);
        for (size_t j = 0; j < m; ++j) {
            const int i = L.members[l][j];
            const afsi_mg3d_plan& pl = bt->items[i].plan;
            float* buffers[2] = {static_cast<float*>(pl.p[l]), static_cast<float*>(pl.tmp[l])};
            StageArgs<float> a{};
            a.rhs = static_cast<const float*>(pl.rhs[l]);
            a.d = Dim32{int(pl.n[l][0]), int(pl.n[l][1]), int(pl.n[l][2])};
            for (int q = 0; q < 3; ++q) a.k.w[q] = float(pl.inv_h2[l][q]);
            a.k.relax = float(pl.relax > 0.0 ? pl.relax : 1.0);
            for (int c = 0; c < 2 * L.chunks[l]; ++c) {
                const bool up = c >= L.chunks[l];
                const int k = up ? c - L.chunks[l] : c;
                a.in = buffers[c & 1];
                a.out = buffers[1 - (c & 1)];
                a.coarse = up && k == 0 ? static_cast<const float*>(pl.p[l + 1]) : nullptr;
                a.restricted = !up && k == L.chunks[l] - 1 ? static_cast<float*>(pl.rhs[l + 1]) : nullptr;
                a.count = std::min(L.phases[l], 2 * L.nu - k * L.phases[l]);
                a.zero = c == 0;  // a cycle starts from zero
                descs[size_t(c) * m + j] = StageDesc{a, bt->active + i, begin};
                if (c == 0) {  // except on level 0 of a later cycle of one refinement iteration
                    a.zero = 0;
                    descs[size_t(2 * L.chunks[l]) * m + j] = StageDesc{a, bt->active + i, begin};
                }
            }
            begin += stage_tiles(a.d, L.tile_x[l], 8);
        }
    }
    int rbeg = 0, vbeg = 0;
    for (int i = 0; i < L.n; ++i) {
        const afsi_mgb_item& it = bt->items[i];
        const afsi_mg3d_plan& pl = it.plan;
        CoarseArgs<float> a;
        const int first = L.cf[i];
        coarse_args<float>(pl, first, a);
        a.p_in = nullptr;  // zero initial guess on every level
        a.active = bt->active + i;
        at<CoarseArgs<float>>(hw, L.coarse_off[0])[i] = a;
        // a later cycle of one refinement iteration continues from the
        // correction so far when the coarse kernel holds level 0 (it loads
        // p_in before it writes p_out, so the two may alias)
        if (first == 0) a.p_in = a.p_out;
        at<CoarseArgs<float>>(hw, L.coarse_off[1])[i] = a;
        const Dim32 d0{int(pl.n[0][0]), int(pl.n[0][1]), int(pl.n[0][2])};
        W3<double> k0;
        for (int q = 0; q < 3; ++q) k0.w[q] = pl.inv_h2[0][q];
        const float* e = static_cast<const float*>(pl.p[0]);
        float* r32 = static_cast<float*>(pl.rhs[0]);
        const int32_t* act = bt->active + i;
        at<RefDesc>(hw, L.ref_off[0])[i] = RefDesc{it.x[0], e, it.b, it.x[0], r32, nullptr, d0, k0, rbeg};
        at<RefDesc>(hw, L.ref_off[1])[i] = RefDesc{it.x[0], e, it.b, it.x[1], r32, act, d0, k0, rbeg};
        at<RefDesc>(hw, L.ref_off[2])[i] = RefDesc{it.x[1], e, it.b, it.x[0], r32, act, d0, k0, rbeg};
        at<RefDesc>(hw, L.ref_off[3])[i] = RefDesc{it.x[1], e, it.b, it.x[1], r32, nullptr, d0, k0, rbeg};
        rbeg += int(cdiv(int64_t(d0.n0) * d0.n1, 4));
        const int cells = d0.n0 * d0.n1 * d0.n2;
        at<VecDesc>(hw, L.vec_off[0])[i] = VecDesc{it.b, cells, vbeg};
        at<VecDesc>(hw, L.vec_off[1])[i] = VecDesc{it.x[0], cells, vbeg};
        at<VecDesc>(hw, L.vec_off[2])[i] = VecDesc{it.x[1], cells, vbeg};
        vbeg += int(cdiv(cells, VEC_CHUNK));
    }
    AFSI_HIP(hipMemcpyAsync(bt->workspace, host.data(), L.total, hipMemcpyHostToDevice, s));
    AFSI_HIP(hipStreamSynchronize(s));
    return OK;
}

template <bool P, int TX, int NPH, bool RESTRICT>
static int batch_stage_n(const StageDesc* desc, int m, int blocks, hipStream_t s) {
    using G = Tile3<float, TX, 8, NPH, RESTRICT>;
    if (int r = dynamic_lds(reinterpret_cast<const void*>(stage_batch_kernel<P, TX, NPH, RESTRICT>), G::LDS)) return r;
    stage_batch_kernel<P, TX, NPH, RESTRICT><<<unsigned(blocks), G::NT, G::LDS, s>>>(desc, m);
    AFSI_LAUNCH_CHECK();
    return OK;
}

template <bool P>
static int batch_stage(const BatchLayout& L, int l, const StageDesc* desc, bool restricts, hipStream_t s) {
    const int m = int(L.members[l].size()), blocks = L.stage_blocks[l];
    if (L.phases[l] == 2)
        return restricts ? batch_stage_n<P, 8, 2, true>(desc, m, blocks, s) : batch_stage_n<P, 8, 2, false>(desc, m, blocks, s);
    if (L.tile_x[l] == 4)
        return restricts ? batch_stage_n<P, 4, 4, true>(desc, m, blocks, s) : batch_stage_n<P, 4, 4, false>(desc, m, blocks, s);
    return restricts ? batch_stage_n<P, 8, 4, true>(desc, m, blocks, s) : batch_stage_n<P, 8, 4, false>(desc, m, blocks, s);
}

template <bool P>
static int batch_vcycle(const afsi_mgb_batch* bt, const BatchLayout& L, hipStream_t s, bool first = true) {
    void* ws = bt->workspace;
    const auto desc = [&](int l, int c) { return at<StageDesc>(ws, L.stage_off[l]) + size_t(c) * L.members[l].size(); };
    for (int l = 0; l < L.levels; ++l)
        for (int c = 0; c < L.chunks[l]; ++c) {
            const bool later = c == 0 && l == 0 && !first;
            if (int r = batch_stage<P>(L, l, desc(l, later ? 2 * L.chunks[l] : c), c == L.chunks[l] - 1, s)) return r;
        }
    const void* coarse_fn = reinterpret_cast<const void*>(coarse_batch_kernel<float, P>);
    if (int r = dynamic_lds(coarse_fn, L.coarse_lds)) return r;
    coarse_batch_kernel<float, P><<<unsigned(L.n), COARSE_THREADS, L.coarse_lds, s>>>(
        at<CoarseArgs<float>>(ws, L.coarse_off[first ? 0 : 1]));
    AFSI_LAUNCH_CHECK();
    for (int l = L.levels - 1; l >= 0; --l)
        for (int c = 0; c < L.chunks[l]; ++c)
            if (int r = batch_stage<P>(L, l, desc(l, L.chunks[l] + c), false, s)) return r;
    return OK;
}

template <bool P>
static int batch_refine(const afsi_mgb_batch* bt, const BatchLayout& L, int which, bool reduce,
                        hipStream_t s) {
    const RefDesc* desc = at<RefDesc>(bt->workspace, L.ref_off[which]);
    const unsigned g = unsigned(L.ref_blocks);
    const bool residual_only = which == 0 || which == 3;
    if (residual_only) refine_batch_kernel<P, false, true><<<g, 256, 0, s>>>(desc, L.n, bt->partials);
    else if (reduce) refine_batch_kernel<P, true, true><<<g, 256, 0, s>>>(desc, L.n, bt->partials);
    else refine_batch_kernel<P, true, false><<<g, 256, 0, s>>>(desc, L.n, bt->partials);
    AFSI_LAUNCH_CHECK();
    if (residual_only || reduce) {
        batch_reduce_kernel<RefDesc><<<unsigned(L.n), 64, 0, s>>>(desc, L.n, L.ref_blocks, bt->partials,
                                                                  bt->results, 0, bt->tol, bt->active);
        AFSI_LAUNCH_CHECK();
    }
    return OK;
}

// stats of vector v into results slot, optionally followed by mean removal
static int batch_vec(const afsi_mgb_batch* bt, const BatchLayout& L, int v, int slot, bool sub,
                     hipStream_t s) {
    const VecDesc* desc = at<VecDesc>(bt->workspace, L.vec_off[v]);
    vec_partials_kernel<<<unsigned(L.vec_blocks[v]), 256, 0, s>>>(desc, L.n, bt->partials);
    batch_reduce_kernel<VecDesc><<<unsigned(L.n), 64, 0, s>>>(desc, L.n, L.vec_blocks[v], bt->partials,
                                                              bt->results, slot, bt->tol, bt->active);
    if (sub) vec_sub_mean_kernel<<<unsigned(L.vec_blocks[v]), 256, 0, s>>>(desc, L.n, bt->results, slot);
    AFSI_LAUNCH_CHECK();
    return OK;
}

static int batch_check_ws(const afsi_mgb_batch* bt, BatchLayout& L) {
    if (int r = batch_layout(bt, L)) return r;
    AFSI_REQUIRE(bt->workspace && bt->workspace_bytes >= L.total, "batch workspace too small");
    AFSI_REQUIRE(bt->active && bt->tol && bt->results && bt->partials, "missing batch state buffers");
    return OK;
}

}  // namespace afsi

extern "C" {
int64_t afsi_mg3d_partials_doubles(const int64_t n[3]) {
    if (!n || n[0] <= 0 || n[1] <= 0 || n[2] <= 0) return -1;
    int64_t blocks = afsi::cdiv(n[0] * n[1] * n[2], 256);
    if (blocks > 4096) blocks = 4096;
    return 4 * blocks;
}
int afsi_refine_residual_3d(const double* x, const double* b, float* r32, const int64_t n[3],
                            const double inv_h2[3], int periodic, double* partials,
                            int64_t partials_capacity, double* result, void* stream) {
    using namespace afsi;
    AFSI_REQUIRE(n && inv_h2 && x && b && r32 && partials && result, "invalid refinement arguments");
    AFSI_REQUIRE(n[0] > 0 && n[1] > 0 && n[2] > 0 && n[0] * n[1] * n[2] < (int64_t(1) << 31),
                 "invalid grid");
    const Dim32 d{int(n[0]), int(n[1]), int(n[2])};
    W3<double> k;
    for (int a = 0; a < 3; ++a) k.w[a] = inv_h2[a];
    int64_t nb = cdiv(n[0] * n[1], 4);
    if (nb > partials_capacity / 4) nb = partials_capacity / 4;
    AFSI_REQUIRE(nb >= 1, "reduction scratch too small");
    const hipStream_t s = hipStream_t(stream);
    if (periodic) refine_residual_kernel<true><<<unsigned(nb), 256, 0, s>>>(x, b, r32, d, k, partials);
    else refine_residual_kernel<false><<<unsigned(nb), 256, 0, s>>>(x, b, r32, d, k, partials);
    AFSI_LAUNCH_CHECK();
    return launch_reduce_final(partials, nb, result, s);
}
int afsi_refine_step_3d(const double* x, const float* e, const double* b, double* x_out,
                        float* r32, const int64_t n[3], const double inv_h2[3], int periodic,
                        double* partials, int64_t partials_capacity, double* result, void* stream) {
    using namespace afsi;
    AFSI_REQUIRE(n && inv_h2 && x && e && b && x_out && r32, "invalid refinement arguments");
    AFSI_REQUIRE(x != x_out, "the refinement step needs distinct input and output iterates");
    AFSI_REQUIRE(n[0] > 0 && n[1] > 0 && n[2] > 0 && n[0] * n[1] * n[2] < (int64_t(1) << 31),
                 "invalid grid");
    const Dim32 d{int(n[0]), int(n[1]), int(n[2])};
    W3<double> k;
    for (int a = 0; a < 3; ++a) k.w[a] = inv_h2[a];
    const hipStream_t s = hipStream_t(stream);
    int64_t nb = cdiv(n[0] * n[1], 4);
    if (result) {
        AFSI_REQUIRE(partials, "missing reduction scratch");
        if (nb > partials_capacity / 4) nb = partials_capacity / 4;
        AFSI_REQUIRE(nb >= 1, "reduction scratch too small");
        if (periodic) refine_step_kernel<true, true><<<unsigned(nb), 256, 0, s>>>(x, e, b, x_out, r32, d, k, partials);
        else refine_step_kernel<false, true><<<unsigned(nb), 256, 0, s>>>(x, e, b, x_out, r32, d, k, partials);
        AFSI_LAUNCH_CHECK();
        return launch_reduce_final(partials, nb, result, s);
    }
    if (nb > 16384) nb = 16384;
    if (periodic) refine_step_kernel<true, false><<<unsigned(nb), 256, 0, s>>>(x, e, b, x_out, r32, d, k, nullptr);
    else refine_step_kernel<false, false><<<unsigned(nb), 256, 0, s>>>(x, e, b, x_out, r32, d, k, nullptr);
    AFSI_LAUNCH_CHECK();
    return OK;
}
int afsi_refine_update(double* x, const float* e, int64_t count, void* stream) {
    using namespace afsi;
    AFSI_REQUIRE(count >= 0 && (count == 0 || (x && e)), "invalid refinement update");
    if (count == 0) return OK;
    refine_update_kernel<<<grid_for(count, 256, 16384), 256, 0, hipStream_t(stream)>>>(x, e, count);
    AFSI_LAUNCH_CHECK();
    return OK;
}
size_t afsi_mgb_workspace_bytes(const afsi_mgb_batch* batch) {
    afsi::BatchLayout L;
    return afsi::batch_layout(batch, L) == afsi::OK ? L.total : 0;
}
int64_t afsi_mgb_partials_doubles(const afsi_mgb_batch* batch) {
    afsi::BatchLayout L;
    return afsi::batch_layout(batch, L) == afsi::OK ? L.partials : -1;
}
int afsi_mgb_prepare(const afsi_mgb_batch* batch, void* stream) {
    return afsi::batch_prepare(batch, hipStream_t(stream));
}
int afsi_mgb_begin_at(const afsi_mgb_batch* batch, int32_t start, double rtol, double atol, void* stream) {
    using namespace afsi;
    BatchLayout L;
    if (int r = batch_check_ws(batch, L)) return r;
    AFSI_REQUIRE(start == 0 || start == 1, "invalid iterate index");
    const hipStream_t s = hipStream_t(stream);
    if (int r = batch_vec(batch, L, 0, 4, true, s)) return r;          // b: stats, mean removal
    if (int r = batch_vec(batch, L, 1 + start, 12, true, s)) return r;  // x[start]: stats, mean removal
    if (int r = batch_vec(batch, L, 0, 8, false, s)) return r;         // ||b|| after the removal
    batch_begin_kernel<<<unsigned(cdiv(L.n, 256)), 256, 0, s>>>(L.n, batch->results, batch->tol,
                                                               batch->active, rtol, atol);
    AFSI_LAUNCH_CHECK();
    const int which = start == 0 ? 0 : 3;  // residual of x[start]
    return L.periodic ? batch_refine<true>(batch, L, which, true, s) : batch_refine<false>(batch, L, which, true, s);
}
int afsi_mgb_begin(const afsi_mgb_batch* batch, double rtol, double atol, void* stream) {
    return afsi_mgb_begin_at(batch, 0, rtol, atol, stream);
}
int afsi_mgb_iterate(const afsi_mgb_batch* batch, int32_t start, int32_t count, void* stream) {
    using namespace afsi;
    BatchLayout L;
    if (int r = batch_check_ws(batch, L)) return r;
    AFSI_REQUIRE((start == 0 || start == 1) && count >= 1, "invalid batch iteration range");
    const hipStream_t s = hipStream_t(stream);
    const int inner = batch->inner_cycles > 0 ? batch->inner_cycles : 1;
    for (int it = 0; it < count; ++it) {
        const int from = (start + it) % 2;
        const bool last = it == count - 1;
        for (int c = 0; c < inner; ++c) {
            const int r = L.periodic ? batch_vcycle<true>(batch, L, s, c == 0) : batch_vcycle<false>(batch, L, s, c == 0);
            if (r) return r;
        }
        if (L.periodic) {
            if (int r = batch_refine<true>(batch, L, 1 + from, last, s)) return r;
        } else {
            if (int r = batch_refine<false>(batch, L, 1 + from, last, s)) return r;
        }
    }
    return OK;
}
int afsi_mgb_finish(const afsi_mgb_batch* batch, int32_t cur, void* stream) {
    using namespace afsi;
    BatchLayout L;
    if (int r = batch_check_ws(batch, L)) return r;
    AFSI_REQUIRE(cur == 0 || cur == 1, "invalid iterate index");
    return batch_vec(batch, L, 1 + cur, 12, true, hipStream_t(stream));
}
int afsi_mg3d_sweep_f64(const afsi_mg3d_plan* plan, int32_t level, void* stream) {
    using namespace afsi;
    if (int r = fast_check<double>(plan)) return r;
    AFSI_REQUIRE(level >= 0 && level < plan->levels, "invalid level");
    const FastRunner<double> run{*plan, hipStream_t(stream), choose_coarse(*plan)};
    return run.sweep(level, run.P(level), run.W(level), false);
}
int afsi_mg3d_sweep_f32(const afsi_mg3d_plan* plan, int32_t level, void* stream) {
    using namespace afsi;
    if (int r = fast_check<float>(plan)) return r;
    AFSI_REQUIRE(level >= 0 && level < plan->levels, "invalid level");
    const FastRunner<float> run{*plan, hipStream_t(stream), choose_coarse(*plan)};
    return run.sweep(level, run.P(level), run.W(level), false);
}
int afsi_mg3d_supported(const afsi_mg3d_plan* plan) {
    return afsi::fast_check<double>(plan) == afsi::OK ? 1 : 0;
}
int afsi_mg3d_cycles_f64(const afsi_mg3d_plan* plan, int32_t cycles, void* stream) {
    return afsi::fast_cycles<double>(plan, cycles, stream);
}
int afsi_mg3d_cycles_f32(const afsi_mg3d_plan* plan, int32_t cycles, void* stream) {
    return afsi::fast_cycles<float>(plan, cycles, stream);
}
int afsi_mg3d_residual_f64(const afsi_mg3d_plan* plan, void* stream) {
    return afsi::fast_residual<double>(plan, stream);
}
int afsi_mg3d_residual_f32(const afsi_mg3d_plan* plan, void* stream) {
    return afsi::fast_residual<float>(plan, stream);
}
}  // extern "C"
