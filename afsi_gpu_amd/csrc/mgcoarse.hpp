// The lower levels of a 3D V-cycle in one workgroup (included by mgfast.hip,
// namespace afsi): every array in LDS, one 1024-thread workgroup per instance.
//
// One compute unit issues all of it, so instructions and LDS round trips
// are the time. A thread keeps its z pairs of a level (at most two) in
// registers over a smoothing stage: both values, right-hand sides and 1/diag
// and the LDS places of the neighbours, decoded once per stage. Red and
// black cells of a level are separate arrays indexed by pair, so lanes read
// consecutive words and a cell's neighbours are all in the other colour's
// array (the pair's own neighbour is a register). A missing neighbour is a
// word of zeros behind the array (red-black) or the cell itself (Jacobi, whose
// update is in difference form). Kernel time of the 16^3 cycle with its 8^3
// and 4^3 levels: FP32 periodic red-black 21.0 -> 16.6 us, FP64 23.7 -> 17.9,
// FP64 closed Jacobi V(4,4) 43 -> 24.7 (packed cell lists decoded per
// update, colours interleaved in one array). Half to two thirds of the cycles
// of its four SIMDs issue VALU instructions (0.55 of the Jacobi, 0.65 of the
// FP32 kernel); the rest are barriers and LDS round trips.

constexpr int COARSE_PAIRS = int(COARSE_MAX / 2 / COARSE_THREADS);  // z pairs per thread
static_assert(COARSE_PAIRS * 2 * COARSE_THREADS == COARSE_MAX, "whole pairs per thread");

template <class T>
struct CoarseArgs {
    int32_t levels;  // number of levels handled (>= 1)
    int32_t smoother, nu;
    T omega;
    Dim32 d[AFSI_MG_MAX_LEVELS];
    W3<T> k[AFSI_MG_MAX_LEVELS];
    int32_t off_p[AFSI_MG_MAX_LEVELS], off_r[AFSI_MG_MAX_LEVELS];
    const T* rhs_in;   // first handled level's rhs (global)
    const T* p_in;     // its initial iterate, or null (zero)
    T* p_out;          // result of the first handled level
    const T* coarse_inverse;
    int32_t coarse_cells;
    const int32_t* active;  // batched launches: skip when *active == 0 (null: always run)
};

// Levels first.. of a plan as arguments; returns the LDS values they need: p
// as two colours of n / 2 + 1 words and rhs as two of n / 2 (the coarsest
// level: n words each, in cell order).
template <class T>
int coarse_args(const afsi_mg3d_plan& pl, int first, CoarseArgs<T>& a) {
    a = CoarseArgs<T>{};
    a.levels = pl.levels - first;
    a.smoother = pl.smoother;
    a.nu = pl.nu;
    a.omega = T(pl.omega);
    int32_t off = 0;
    for (int j = 0; j < a.levels; ++j) {
        const int l = first + j;
        a.d[j] = Dim32{int(pl.n[l][0]), int(pl.n[l][1]), int(pl.n[l][2])};
        for (int q = 0; q < 3; ++q) a.k[j].w[q] = T(pl.inv_h2[l][q]);
        a.k[j].relax = T(pl.relax > 0.0 ? pl.relax : 1.0);
        const int32_t n = a.d[j].n0 * a.d[j].n1 * a.d[j].n2;
        a.off_p[j] = off;
        off += n + (j + 1 < a.levels ? 2 : 0);
        a.off_r[j] = off;
        off += n;
    }
    a.rhs_in = static_cast<const T*>(pl.rhs[first]);
    a.p_out = static_cast<T*>(pl.p[first]);
    a.coarse_inverse = static_cast<const T*>(pl.coarse_inverse);
    a.coarse_cells = int32_t(pl.coarse_cells);
    return off;
}

// floor(e / d) for 0 <= e < 2^13, d >= 1 (the float quotient of e + 1/2 is
// at least 1/(2d) from an integer, far more than its rounding).
__device__ inline int small_div(int e, float inverse) { return int((float(e) + 0.5f) * inverse); }

// Sum over the 16 lanes of a row, in every lane (row rotations, no LDS).
template <int ROR>
__device__ __forceinline__ float row_rotate(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x120 + ROR, 0xf, 0xf, false));
}
template <int ROR>
__device__ __forceinline__ double row_rotate(double v) {
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = uint32_t(__builtin_amdgcn_update_dpp(0, int(uint32_t(b)), 0x120 + ROR, 0xf, 0xf, false));
    const uint32_t hi = uint32_t(__builtin_amdgcn_update_dpp(0, int(uint32_t(b >> 32)), 0x120 + ROR, 0xf, 0xf, false));
    return __builtin_bit_cast(double, (uint64_t(hi) << 32) | lo);
}
template <class T>
__device__ __forceinline__ T row_sum16(T v) {
    v += row_rotate<8>(v);
    v += row_rotate<4>(v);
    v += row_rotate<2>(v);
    v += row_rotate<1>(v);
    return v;
}

// Value of coarse cell (x, y, z) in LDS: colours by pair, or cell order on
// the coarsest level.
template <class T>
__device__ __forceinline__ T coarse_cell(const T* p, const Dim32& d, bool plain, int row, int parity, int z) {
    if (plain) return p[row * d.n2 + z];
    return p[((parity + z) & 1) * (d.n0 * d.n1 * d.n2 / 2 + 1) + row * (d.n2 / 2) + (z >> 1)];
}

// One smoothing stage of level l: down (from the first level's initial
// iterate or zero) or up (from the pre-smoothed iterate plus the
// prolongation of level l + 1).
template <class T, bool P>
__device__ __forceinline__ void coarse_stage(const CoarseArgs<T>& a, int l, bool up, T* lds, const T* tab) {
    const Dim32 d = a.d[l];
    const W3<T> k = a.k[l];
    const int hz = d.n2 / 2, np = d.n0 * d.n1 * hz, cs = np + 1, tid = int(threadIdx.x);
    const float inv_hz = 1.0f / float(hz), inv_n1 = 1.0f / float(d.n1);
    T* red = lds + a.off_p[l];
    T* rr = lds + a.off_r[l];
    T p[COARSE_PAIRS][2], r[COARSE_PAIRS][2], inv[COARSE_PAIRS][2];
    int xp[COARSE_PAIRS], xm[COARSE_PAIRS], yp[COARSE_PAIRS], ym[COARSE_PAIRS], zo[COARSE_PAIRS][2];
    const T inv_p = T(1) / (T(2) * (k.w[0] + k.w[1] + k.w[2]));
    if (tid < 2) red[tid * cs + np] = T(0);
#pragma unroll
    for (int q = 0; q < COARSE_PAIRS; ++q) {
        const int e = tid + q * COARSE_THREADS;
        if (e >= np) continue;
        const int row = small_div(e, inv_hz), zp = e - row * hz;
        const int x = small_div(row, inv_n1), y = row - x * d.n1;
        const int sx = d.n1 * hz, lead = (x + y) & 1;  // red is the pair's cell `lead`
        xp[q] = x + 1 < d.n0 ? e + sx : (P ? e - (d.n0 - 1) * sx : np);
        xm[q] = x > 0 ? e - sx : (P ? e + (d.n0 - 1) * sx : np);
        yp[q] = y + 1 < d.n1 ? e + hz : (P ? e - (d.n1 - 1) * hz : np);
        ym[q] = y > 0 ? e - hz : (P ? e + (d.n1 - 1) * hz : np);
        const int above = zp + 1 < hz ? e + 1 : (P ? e - (hz - 1) : np), below = zp > 0 ? e - 1 : (P ? e + (hz - 1) : np);
        zo[q][0] = lead ? above : below;
        zo[q][1] = lead ? below : above;
        if (P) {
            inv[q][0] = inv[q][1] = inv_p;
        } else {
            const T* t = tab + face_class(x, d.n0) * 9 + face_class(y, d.n1) * 3;
            inv[q][0] = t[face_class(2 * zp + lead, d.n2)];
            inv[q][1] = t[face_class(2 * zp + 1 - lead, d.n2)];
        }
        T c0 = T(0), c1 = T(0);  // the pair's cells in z order
        if (!up && l == 0) {
            const T r0 = a.rhs_in[2 * e], r1 = a.rhs_in[2 * e + 1];
            if (a.p_in) {
                c0 = a.p_in[2 * e];
                c1 = a.p_in[2 * e + 1];
            }
            r[q][0] = lead ? r1 : r0;
            r[q][1] = lead ? r0 : r1;
            rr[e] = r[q][0];
            rr[np + e] = r[q][1];
        } else {
            r[q][0] = rr[e];
            r[q][1] = rr[np + e];
        }
        if (up) {
            const Dim32 c = a.d[l + 1];
            const bool plain = l + 2 == a.levels;
            const T* pc = lds + a.off_p[l + 1];
            const int ax = x / 2 - 1 + (x & 1), ay = y / 2 - 1 + (y & 1);
            const auto near = [](int i, int n) { return P ? (i < 0 ? i + n : (i >= n ? i - n : i)) : (i < 0 ? 0 : (i >= n ? n - 1 : i)); };
            const T wx = (x & 1) ? T(0.25) : T(0.75), wy = (y & 1) ? T(0.25) : T(0.75), lo = T(0.25), hi = T(0.75);
            const int za = near(zp - 1, c.n2), zc = near(zp + 1, c.n2);
            T v0[2], v1[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                T w0[2], w1[2];
                const int cx = near(ax + i, c.n0);
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const int cy = near(ay + j, c.n1), crow = cx * c.n1 + cy, par = cx + cy;
                    const T below_v = coarse_cell(pc, c, plain, crow, par, za), mid = coarse_cell(pc, c, plain, crow, par, zp),
                            above_v = coarse_cell(pc, c, plain, crow, par, zc);
                    w0[j] = below_v * lo + mid * hi;
                    w1[j] = mid * hi + above_v * lo;
                }
                v0[i] = w0[0] * (T(1) - wy) + w0[1] * wy;
                v1[i] = w1[0] * (T(1) - wy) + w1[1] * wy;
            }
            c0 = v0[0] * (T(1) - wx) + v0[1] * wx;
            c1 = v1[0] * (T(1) - wx) + v1[1] * wx;
        }
        p[q][0] = lead ? c1 : c0;
        p[q][1] = lead ? c0 : c1;
        if (up) {
            p[q][0] += red[e];
            p[q][1] += red[cs + e];
        }
        red[e] = p[q][0];
        red[cs + e] = p[q][1];
    }
    __syncthreads();
    const auto value = [&](int q, int colour) -> T {
        const T* o = red + (1 - colour) * cs;
        return gs_sum<T>(k, r[q][colour], p[q][1 - colour] + o[zo[q][colour]], o[yp[q]] + o[ym[q]], o[xp[q]] + o[xm[q]]) *
               inv[q][colour];
    };
    if (a.smoother == 1) {
        for (int it = 0; it < a.nu; ++it) {
#pragma unroll
            for (int colour = 0; colour < 2; ++colour) {
#pragma unroll
                for (int q = 0; q < COARSE_PAIRS; ++q) {
                    if (tid + q * COARSE_THREADS >= np) continue;
                    p[q][colour] = rb_relax(k, p[q][colour], value(q, colour));
                    red[colour * cs + tid + q * COARSE_THREADS] = p[q][colour];
                }
                __syncthreads();
            }
        }
    } else {
        // difference form, p + omega (b - sum w (p - nb)) / diag, as on the
        // tiled levels; a missing neighbour's place is the cell's own
        int nb[COARSE_PAIRS][2][5];
#pragma unroll
        for (int q = 0; q < COARSE_PAIRS; ++q) {
            const int e = tid + q * COARSE_THREADS;
            if (e >= np) continue;
#pragma unroll
            for (int colour = 0; colour < 2; ++colour) {
                const int from[5] = {xp[q], xm[q], yp[q], ym[q], zo[q][colour]};
#pragma unroll
                for (int i = 0; i < 5; ++i) nb[q][colour][i] = !P && from[i] == np ? e + (colour ? cs : -cs) : from[i];
                inv[q][colour] *= a.omega;
            }
        }
        for (int it = 0; it < a.nu; ++it) {
            T w[COARSE_PAIRS][2];
#pragma unroll
            for (int q = 0; q < COARSE_PAIRS; ++q) {
                if (tid + q * COARSE_THREADS >= np) continue;
#pragma unroll
                for (int colour = 0; colour < 2; ++colour) {
                    const T* o = red + (1 - colour) * cs;
                    const int* at = nb[q][colour];
                    const T c = p[q][colour], zs = (p[q][1 - colour] - c) + (o[at[4]] - c);
                    const T ys = (o[at[2]] - c) + (o[at[3]] - c), xs = (o[at[0]] - c) + (o[at[1]] - c);
                    const T d = fma_of(k.w[0], xs, fma_of(k.w[1], ys, fma_of(k.w[2], zs, r[q][colour])));
                    w[q][colour] = fma_of(inv[q][colour], d, c);
                }
            }
            __syncthreads();
#pragma unroll
            for (int q = 0; q < COARSE_PAIRS; ++q) {
                if (tid + q * COARSE_THREADS >= np) continue;
#pragma unroll
                for (int colour = 0; colour < 2; ++colour) {
                    p[q][colour] = w[q][colour];
                    red[colour * cs + tid + q * COARSE_THREADS] = p[q][colour];
                }
            }
            __syncthreads();
        }
    }
    if (up && l == 0) {
#pragma unroll
        for (int q = 0; q < COARSE_PAIRS; ++q) {
            const int e = tid + q * COARSE_THREADS;
            if (e >= np) continue;
            const int row = small_div(e, inv_hz), x = small_div(row, inv_n1), lead = (x + row - x * d.n1) & 1;
            a.p_out[2 * e] = lead ? p[q][1] : p[q][0];
            a.p_out[2 * e + 1] = lead ? p[q][0] : p[q][1];
        }
    }
}

// Residual of level l restricted to level l + 1's right-hand side: one
// thread per coarse cell, whose eight children's colours are the parities of
// their places.
template <class T, bool P>
__device__ __forceinline__ void coarse_restrict(const CoarseArgs<T>& a, int l, T* lds) {
    const Dim32 d = a.d[l], c = a.d[l + 1];
    const W3<T> k = a.k[l];
    const int hz = c.n2, np = d.n0 * d.n1 * hz, cs = np + 1, sx = d.n1 * hz, nc = c.n0 * c.n1 * c.n2;
    const bool plain = l + 2 == a.levels;
    const T* red = lds + a.off_p[l];
    const T* rr = lds + a.off_r[l];
    T* out = lds + a.off_r[l + 1];
    const float inv_c2 = 1.0f / float(c.n2), inv_c1 = 1.0f / float(c.n1);
    for (int e = threadIdx.x; e < nc; e += COARSE_THREADS) {
        const int row = small_div(e, inv_c2), z = e - row * c.n2, x = small_div(row, inv_c1), y = row - x * c.n1;
        const int base = 2 * x * sx + 2 * y * hz + z;  // pair of the children (0, 0, .)
        // pair offsets of the neighbours outside the block
        const int xm = x > 0 ? -sx : (d.n0 - 1) * sx, xp = x + 1 < c.n0 ? sx : -(d.n0 - 1) * sx;
        const int ym = y > 0 ? -hz : (d.n1 - 1) * hz, yp = y + 1 < c.n1 ? hz : -(d.n1 - 1) * hz;
        const int zm = z > 0 ? -1 : hz - 1, zp = z + 1 < c.n2 ? 1 : -(hz - 1);
        T v = T(0);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int ax = i >> 2, ay = (i >> 1) & 1, az = i & 1, colour = (ax + ay + az) & 1;
            const int at = base + ax * sx + ay * hz;
            const T* o = red + (1 - colour) * cs + at;
            const T w = red[colour * cs + at];
            T ap = T(0);
            if (P || ax == 0 || x + 1 < c.n0) ap += k.w[0] * (w - o[ax ? xp : sx]);
            if (P || ax == 1 || x > 0) ap += k.w[0] * (w - o[ax ? -sx : xm]);
            if (P || ay == 0 || y + 1 < c.n1) ap += k.w[1] * (w - o[ay ? yp : hz]);
            if (P || ay == 1 || y > 0) ap += k.w[1] * (w - o[ay ? -hz : ym]);
            if (P || az == 0 || z + 1 < c.n2) ap += k.w[2] * (w - o[az ? zp : 0]);
            if (P || az == 1 || z > 0) ap += k.w[2] * (w - o[az ? 0 : zm]);
            v += rr[colour * np + at] - ap;
        }
        v *= T(0.125);
        if (plain) out[e] = v;
        else out[((x + y + z) & 1) * (nc / 2) + row * (c.n2 / 2) + (z >> 1)] = v;
    }
}

template <class T, bool P>
__device__ __forceinline__ void coarse_cycle_body(const CoarseArgs<T>& a) {
    extern __shared__ unsigned char smem_raw[];
    T* lds = reinterpret_cast<T*>(smem_raw);
    __shared__ T tabs[AFSI_MG_MAX_LEVELS][27];
    const int last = a.levels - 1, tid = int(threadIdx.x), m = a.coarse_cells;
    // 16 lanes per row of the coarse product; rows of a small inverse are
    // loaded before the cycle and held
    constexpr int SEG = 16, ROWS = COARSE_THREADS / SEG, HELD = 4;
    const int seg = tid % SEG, row0 = tid / SEG;
    T held[HELD];
#pragma unroll
    for (int i = 0; i < HELD; ++i) {
        const int col = seg + SEG * i;
        held[i] = m <= ROWS && row0 < m && col < m ? a.coarse_inverse[row0 * m + col] : T(0);
    }
    static_assert(HELD * SEG == ROWS, "a held row has at most ROWS columns");
    if (!P) {
        for (int i = tid; i < 27 * last; i += COARSE_THREADS) tabs[i / 27][i % 27] = inv_diag_entry<T>(i % 27, a.k[i / 27]);
        __syncthreads();
    }
    for (int l = 0; l < last; ++l) {
        coarse_stage<T, P>(a, l, false, lds, tabs[l]);
        coarse_restrict<T, P>(a, l, lds);
        __syncthreads();
    }
    {
        T* p = lds + a.off_p[last];
        T* r = lds + a.off_r[last];
        if (last == 0) {
            for (int i = tid; i < m; i += COARSE_THREADS) r[i] = a.rhs_in[i];
            __syncthreads();
        }
        if (m <= ROWS) {
            T s = T(0);
#pragma unroll
            for (int i = 0; i < HELD; ++i) s += held[i] * (seg + SEG * i < m ? r[seg + SEG * i] : T(0));
            s = row_sum16(s);
            if (row0 < m && seg == 0) p[row0] = s;
        } else {
            for (int row = row0; row < m; row += ROWS) {  // whole rows of 16 lanes stay together
                T s = T(0);
                for (int col = seg; col < m; col += SEG) s += a.coarse_inverse[row * m + col] * r[col];
                s = row_sum16(s);
                if (seg == 0) p[row] = s;
            }
        }
        __syncthreads();
        if (last == 0)
            for (int i = tid; i < m; i += COARSE_THREADS) a.p_out[i] = p[i];
    }
    for (int l = last - 1; l >= 0; --l) coarse_stage<T, P>(a, l, true, lds, tabs[l]);
}
