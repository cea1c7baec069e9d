// One smoothing stage of a 3D multigrid level in one launch (included by
// mgfast.hip, namespace afsi).
//
// A workgroup takes a TX x TY x 16 tile with a halo and runs up to four phases
// (red-black half-sweeps, or Jacobi sweeps) on it, with the prolongation of
// the coarse correction before the first phase or the residual restriction
// after the last one. Thread t = (y, pair j) owns the cell pair z = 2j, 2j + 1
// of every x plane of its column: both values, both right-hand sides of all
// planes stay in registers, so x neighbours and the pair's own neighbour are
// registers, and only y and outer z neighbours go through LDS: an update is
// three LDS reads, eight (Gauss-Seidel) or thirteen (Jacobi) floating-point
// operations and one LDS write. Jacobi updates in difference form,
// p + omega (b - sum w (p - nb)) / diag, as the unfused sweeps do: from
// (b + sum w nb) / diag the residual stagnates 1.6 to 1.8 times higher.
// LDS holds, per plane, the red cells of all columns, then the black ones, at
// index t: consecutive lanes read consecutive words whatever the row length,
// and a neighbour is a constant offset (y: +-HB, z: +-1).
//
// Phase s needs no bounds: a column's halo cells beyond the valid region hold
// values that are never used, because a phase moves that region in by one
// cell and the halo is as deep as the phases are many (one more for the
// restriction). Cells outside a closed domain are zero and stay zero (their
// 1/diag is zero). Reads beyond the first and last row of a plane land in the
// neighbouring planes (planes 0 and BX - 1 are never updated).
//
// Why: levels of up to 64^3 cells were bound by launches and barriers, the
// 128^3 sweeps by the LDS and VALU work of seven LDS accesses an update. The
// tile shape gives 256 workgroups at 64^3. Measured figures stand at
// FastRunner::WIDE_TILES in mgfast.hip. Bound now by latency: at 64^3 closed
// FP64 Jacobi, down stage, VALU issue takes 0.37 of the time with two waves
// per SIMD; at 128^3 FP32, up stage, 0.24, with 18 MB of HBM traffic in 11.6 us.

constexpr int TILE_Z = 16;

template <class T, int TX, int TY, int NPH, bool RESTRICT>
struct Tile3 {
    static constexpr int H = NPH + (RESTRICT ? 1 : 0);    // halo in x and y
    static constexpr int HZ = NPH + (RESTRICT ? 2 : 0);   // in z: even, so pairs are coarse children
    static constexpr int BX = TX + 2 * H, BY = TY + 2 * H, HB = TILE_Z / 2 + HZ;
    static constexpr int COLS = BY * HB;                          // columns, one thread each
    static constexpr int NT = (COLS + 63) / 64 * 64;
    static constexpr int TC = TY * TILE_Z / 2;                    // columns of the tile
    static constexpr size_t LDS = (size_t(BX) * 2 * COLS + (RESTRICT ? size_t(TX) * 2 * TC : 0)) * sizeof(T);
};

// One launch's arguments of one level.
template <class T>
struct StageArgs {
    const T* in;      // iterate (ignored when zero)
    const T* rhs;
    T* out;
    const T* coarse;  // correction to prolong first, or null
    T* restricted;    // coarse right-hand side to write, or null
    Dim32 d;
    W3<T> k;
    T omega;
    int32_t count;  // phases, the first one red
    int32_t zero;
};

__host__ __device__ inline int stage_tiles(const Dim32& d, int tx, int ty) {
    return ((d.n0 + tx - 1) / tx) * ((d.n1 + ty - 1) / ty) * ((d.n2 + TILE_Z - 1) / TILE_Z);
}

// Two cells loaded or stored at once, at any address that one cell may have.
template <class T> struct Pair2;
template <> struct Pair2<float> { typedef float type __attribute__((ext_vector_type(2), aligned(4))); };
template <> struct Pair2<double> { typedef double type __attribute__((ext_vector_type(2), aligned(8))); };

// g wrapped into [0, n): one addition where the axis is longer than a halo.
__device__ inline int wrap_near(int g, int n) {
    g = g < 0 ? g + n : (g >= n ? g - n : g);
    if (uint32_t(g) >= uint32_t(n)) g = ((g % n) + n) % n;
    return g;
}

// Gauss-Seidel value of a cell times its diagonal, from the sums of its z, y
// and x neighbours.
template <class T>
__device__ __forceinline__ T gs_sum(const W3<T>& k, T b, T zs, T ys, T xs) {
    return fma_of(k.w[0], xs, fma_of(k.w[1], ys, fma_of(k.w[2], zs, b)));
}

// The value. The row sweeps form it this way too, so they and the stages agree
// bit for bit. A plain product with the rounded reciprocal (lo = 0) lets the
// residual stagnate 1.1 to 1.2 times higher. Periodic levels have one
// reciprocal, and lo costs nothing there. On closed levels its selects cost 3
// to 11% of a cycle, so it is used only where the sweeps divide (z > ZROW), in
// tiles away from the ends of x, which need no selects.
template <class T>
__device__ __forceinline__ T gs_value(const W3<T>& k, T b, T zs, T ys, T xs, const Recip<T>& inv) {
    const T t = gs_sum(k, b, zs, ys, xs);
    return fma_of(t, inv.hi, t * inv.lo);
}

template <class T, bool P, bool GS, int TX, int TY, int NPH, bool RESTRICT>
__device__ __forceinline__ void stage_tile(const StageArgs<T>& a, int tile, T* lds) {
    using G = Tile3<T, TX, TY, NPH, RESTRICT>;
    using V2 = typename Pair2<T>::type;
    constexpr int H = G::H, HZ = G::HZ, BX = G::BX, HB = G::HB, COLS = G::COLS;
    constexpr int PL = 2 * COLS;  // LDS words per plane
    const Dim32 d = a.d;
    const W3<T> k = a.k;
    const int nty = (d.n1 + TY - 1) / TY, ntz = (d.n2 + TILE_Z - 1) / TILE_Z;
    const int tx = tile / (nty * ntz), rest = tile - tx * nty * ntz, ty = rest / ntz;
    const int x0 = tx * TX - H, y0 = ty * TY - H, z0 = (rest - ty * ntz) * TILE_Z - HZ;
    const int t = int(threadIdx.x);
    const bool column = t < COLS;
    const int y = t / HB, j = t - y * HB;
    int gy = y0 + y, gz = z0 + 2 * j;
    if (P) {
        gy = wrap_near(gy, d.n1);
        gz = wrap_near(gz, d.n2);
    }
    const bool inside = column && gy >= 0 && gy < d.n1 && gz >= 0 && gz < d.n2;
    const int sx = d.n1 * d.n2;
    // byte offset in a plane (32 bits: a uniform base with a lane offset is one instruction)
    const uint32_t pair = inside ? uint32_t(gy * d.n2 + gz) * uint32_t(sizeof(T)) : 0u;
    const auto load2 = [pair](const T* base) { return *reinterpret_cast<const V2*>(reinterpret_cast<const char*>(base) + pair); };
    const int q = (x0 + y0 + y) & 1;  // red's place in the pair on even box planes (odd planes: 1 - q)
    const auto plane_inside = [&](int x) { return P || (x0 + x >= 0 && x0 + x < d.n0); };

    // p and rhs of the column: red in A, black in B
    // (every load is issued before the first value is used: clamped addresses
    // and selects instead of branches)
    T A[BX], B[BX], RA[BX], RB[BX];
    {
        V2 p[BX], r[BX];
        int gx = P ? wrap_near(x0, d.n0) : x0;
        int row[BX];  // uniform
#pragma unroll
        for (int x = 0; x < BX; ++x) {
            row[x] = __builtin_amdgcn_readfirstlane((P ? gx : (gx < 0 ? 0 : (gx >= d.n0 ? d.n0 - 1 : gx))) * sx);
            gx = P && gx + 1 == d.n0 ? 0 : gx + 1;
        }
#pragma unroll
        for (int x = 0; x < BX; ++x) r[x] = load2(a.rhs + row[x]);
        if (a.zero) {
#pragma unroll
            for (int x = 0; x < BX; ++x) p[x] = V2{T(0), T(0)};
        } else {
#pragma unroll
            for (int x = 0; x < BX; ++x) p[x] = load2(a.in + row[x]);
        }
#pragma unroll
        for (int x = 0; x < BX; ++x) {
            const bool second = ((x & 1) ^ q) != 0, in = P || (inside && plane_inside(x));
            const T p0 = in ? p[x].x : T(0), p1 = in ? p[x].y : T(0), r0 = in ? r[x].x : T(0), r1 = in ? r[x].y : T(0);
            A[x] = second ? p1 : p0;
            B[x] = second ? p0 : p1;
            RA[x] = second ? r1 : r0;
            RB[x] = second ? r0 : r1;
        }
    }
    if constexpr (!RESTRICT) {
        if (a.coarse) {
            // q(c) = the coarse plane c interpolated in y and z at the pair;
            // plane 2m lies between coarse planes m - 1 and m, plane 2m + 1
            // between m and m + 1 (box plane 0 is an even plane)
            const int C0 = d.n0 / 2, C1 = d.n1 / 2, C2 = d.n2 / 2;
            const int ay = gy / 2 - 1 + (gy & 1), cz = gz / 2;
            const auto near = [](int c, int n) { return P ? (c < 0 ? c + n : (c >= n ? c - n : c)) : (c < 0 ? 0 : (c >= n ? n - 1 : c)); };
            const int ra = inside ? near(ay, C1) * C2 : 0, rb = inside ? near(ay + 1, C1) * C2 : 0;
            const int za = inside ? near(cz - 1, C2) : 0, zb = inside ? cz : 0, zc = inside ? near(cz + 1, C2) : 0;
            const T wy = (gy & 1) ? T(0.25) : T(0.75), lo = T(0.25), hi = T(0.75);
            const auto mix = [&](int c, T& even, T& odd) {
                const int cx = P ? c : (c < 0 ? 0 : (c >= C0 ? C0 - 1 : c));
                const T* s = a.coarse + cx * C1 * C2;
                const T a0 = s[ra + za], a1 = s[ra + zb], a2 = s[ra + zc];
                const T b0 = s[rb + za], b1 = s[rb + zb], b2 = s[rb + zc];
                const T e0 = a0 * lo + a1 * hi, e1 = b0 * lo + b1 * hi;
                const T o0 = a1 * hi + a2 * lo, o1 = b1 * hi + b2 * lo;
                even = e0 * (T(1) - wy) + e1 * wy;
                odd = o0 * (T(1) - wy) + o1 * wy;
            };
            int m = x0 / 2 - 1;  // x0 is even
            if (P) m = wrap_near(m, C0);
            const auto next = [&] { m = P && m + 1 == C0 ? 0 : m + 1; return m; };
            T pe, po, ce, co, ne, no;
            mix(m, pe, po);
            mix(next(), ce, co);
#pragma unroll
            for (int x = 0; x < BX; x += 2) {
                mix(next(), ne, no);
                const bool second = q != 0;
                const T e0 = pe * lo + ce * hi, o0 = po * lo + co * hi;
                const T e1 = ce * hi + ne * lo, o1 = co * hi + no * lo;
                const bool in0 = P || (inside && plane_inside(x)), in1 = P || (inside && plane_inside(x + 1));
                A[x] += in0 ? (second ? o0 : e0) : T(0);
                B[x] += in0 ? (second ? e0 : o0) : T(0);
                A[x + 1] += in1 ? (second ? e1 : o1) : T(0);
                B[x + 1] += in1 ? (second ? o1 : e1) : T(0);
                pe = ce; po = co; ce = ne; co = no;
            }
        }
    }
    T* own = lds + t;
    if (column) {
#pragma unroll
        for (int x = 0; x < BX; ++x) {
            own[x * PL] = A[x];
            own[x * PL + COLS] = B[x];
        }
    }
    const bool tiled = inside && y >= H && y < H + TY && y0 + y < d.n1 && 2 * j >= HZ && 2 * j < HZ + TILE_Z &&
                       z0 + 2 * j < d.n2;  // not a periodic copy beyond the domain
    T* const rhs_tile = lds + BX * PL;  // (plane, colour, column) of the tile, for the restriction
    if (RESTRICT && tiled) {
        T* r = rhs_tile + (y - H) * (TILE_Z / 2) + j - HZ / 2;
#pragma unroll
        for (int i = 0; i < TX; ++i) {
            r[2 * i * G::TC] = RA[H + i];
            r[(2 * i + 1) * G::TC] = RB[H + i];
        }
    }
    const bool plain = P || (x0 > 0 && x0 + BX < d.n0);  // no plane at or beyond an end
    // 1/diag of red on even planes (= black on odd ones) and the other way
    // round, for planes inside (mid) and at the ends (end) of a closed domain
    T mid[2], end[2], lo[2];
    if (P) {
        const Recip<T> r = recip(T(2) * (k.w[0] + k.w[1] + k.w[2]));
        mid[0] = mid[1] = end[0] = end[1] = r.hi;
        lo[0] = lo[1] = r.lo;
    } else {
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const int z = gz + (q ^ s);
            const int c = 3 * face_class(gy, d.n1) + face_class(z, d.n2);
            const Recip<T> m = recip(diag_entry<T>(9 + c, k));
            mid[s] = inside ? m.hi : T(0);
            end[s] = inside ? inv_diag_entry<T>(c, k) : T(0);
            lo[s] = inside && plain && d.n2 > ZROW ? m.lo : T(0);
        }
    }
    __syncthreads();

    const auto inverse = [&](int x, int s) -> T {
        if (plain) return mid[s];
        const int px = x0 + x;
        return px < 0 || px >= d.n0 ? T(0) : (px == 0 || px == d.n0 - 1 ? end[s] : mid[s]);
    };
    if constexpr (GS) {
        // the pair's outer z neighbour: above for the second cell, below for the first
        T* const zA = own + (q ? 1 : -1);
        T* const zB = own - (q ? 1 : -1);
        const auto value = [&](int x, int colour) -> T {
            // even planes: red is the pair's cell q; its neighbours are black
            const int s = (x & 1) ^ colour;
            const T* o = own + x * PL + (colour ? 0 : COLS);
            const T* z = (s ? zB : zA) + x * PL + (colour ? 0 : COLS);
            const T inner = colour ? A[x] : B[x];
            const T xs = colour ? A[x + 1] + A[x - 1] : B[x + 1] + B[x - 1];
            return gs_value<T>(k, colour ? RB[x] : RA[x], inner + *z, o[HB] + o[-HB], xs,
                               Recip<T>{inverse(x, s), lo[s]});
        };
#pragma unroll
        for (int s = 0; s < NPH; ++s) {
            if (s >= a.count) continue;
            // all LDS reads of a phase come before its writes: the compiler
            // cannot tell that they never meet
            if (column) {
#pragma unroll
                for (int x = 1 + s; x < BX - 1 - s; ++x) {
                    if (s & 1) B[x] = rb_relax(k, B[x], value(x, 1));
                    else A[x] = rb_relax(k, A[x], value(x, 0));
                }
#pragma unroll
                for (int x = 1 + s; x < BX - 1 - s; ++x) own[x * PL + (s & 1) * COLS] = (s & 1) ? B[x] : A[x];
            }
            __syncthreads();
        }
    } else {
        // Offsets of the y neighbours and of the outer z neighbour (of the cell
        // at place q of the pair, and of the other one) from the cell's plane,
        // for red; a missing neighbour's place is the cell's own. For black the
        // colours' places change roles.
        const auto place = [](bool there, int step, int colour) -> int {
            return there ? (colour ? 0 : COLS) + step : (colour ? COLS : 0);
        };
        const bool up = P || gy + 1 < d.n1, down = P || gy > 0;
        const bool za = P || (q ? gz + 2 < d.n2 : gz > 0), zb = P || (q ? gz > 0 : gz + 2 < d.n2);
        const int sa = q ? 1 : -1;
        const T *const yh0 = own + place(up, HB, 0), *const yh1 = own + place(up, HB, 1);
        const T *const yl0 = own + place(down, -HB, 0), *const yl1 = own + place(down, -HB, 1);
        const T *const za0 = own + place(za, sa, 0), *const za1 = own + place(za, sa, 1);
        const T *const zb0 = own + place(zb, -sa, 0), *const zb1 = own + place(zb, -sa, 1);
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            mid[s] *= a.omega;
            end[s] *= a.omega;
        }
        const auto value = [&](int x, int colour) -> T {
            const int s = (x & 1) ^ colour;
            const T c = colour ? B[x] : A[x], inner = colour ? A[x] : B[x];
            const T xl = colour ? A[x - 1] : B[x - 1], xh = colour ? A[x + 1] : B[x + 1];
            const T z = (s ? (colour ? zb1 : zb0) : (colour ? za1 : za0))[x * PL];
            const T zs = (inner - c) + (z - c);
            const T ys = ((colour ? yh1 : yh0)[x * PL] - c) + ((colour ? yl1 : yl0)[x * PL] - c);
            const T r = fma_of(k.w[0], (xh - c) + (xl - c), fma_of(k.w[1], ys, fma_of(k.w[2], zs, colour ? RB[x] : RA[x])));
            return fma_of(inverse(x, s), r, c);
        };
#pragma unroll
        for (int s = 0; s < NPH; ++s) {
            if (s >= a.count) continue;
            if (!plain) {  // planes -1 and n0 mirror the end planes (n0 and the tile's first plane are even)
#pragma unroll
                for (int x = 0; x < BX; ++x) {
                    if (x < H && (H - 1 - x) % TX == 0 && x0 + x == -1) {
                        A[x] = B[x + 1];
                        B[x] = A[x + 1];
                    }
                    if (x > H && (x - H) % 2 == 0 && x0 + x == d.n0) {
                        A[x] = B[x ? x - 1 : 0];
                        B[x] = A[x ? x - 1 : 0];
                    }
                }
            }
            if (column) {
                // new values replace plane x - 1 once plane x no longer reads it
                T na = A[s], nb = B[s];
#pragma unroll
                for (int x = 1 + s; x < BX - 1 - s; ++x) {
                    const T va = value(x, 0), vb = value(x, 1);
                    A[x - 1] = na;
                    B[x - 1] = nb;
                    na = va;
                    nb = vb;
                }
                A[BX - 2 - s] = na;
                B[BX - 2 - s] = nb;
            }
            __syncthreads();
            if (column) {
#pragma unroll
                for (int x = 1 + s; x < BX - 1 - s; ++x) {
                    own[x * PL] = A[x];
                    own[x * PL + COLS] = B[x];
                }
            }
            __syncthreads();
        }
    }

    if (tiled) {
#pragma unroll
        for (int x = H; x < H + TX; ++x) {
            if (x0 + x >= d.n0) continue;
            const bool second = ((x & 1) ^ q) != 0;
            V2 v;
            v.x = second ? B[x] : A[x];
            v.y = second ? A[x] : B[x];
            *reinterpret_cast<V2*>(reinterpret_cast<char*>(a.out + (x0 + x) * sx) + pair) = v;
        }
    }
    if constexpr (RESTRICT) {
        // One thread per coarse cell of the tile: the residual of its eight
        // children in difference form, summed in the order x, y, z (slowest
        // to fastest). The tile starts at even cells, so a child's colour is
        // the parity of its place and every LDS offset is a constant.
        constexpr int CZ = TILE_Z / 2, CELLS = (TX / 2) * (TY / 2) * CZ;
        for (int e = t; e < CELLS; e += G::NT) {
            const int cj = e % CZ, cy = e / CZ % (TY / 2), cx = e / (CZ * (TY / 2));
            const int fx = x0 + H + 2 * cx, fy = y0 + H + 2 * cy, fz = z0 + HZ + 2 * cj;
            if (fx >= d.n0 || fy >= d.n1 || fz >= d.n2) continue;
            const T* p = lds + (H + 2 * cx) * PL + (H + 2 * cy) * HB + HZ / 2 + cj;
            const T* r = rhs_tile + 2 * cx * 2 * G::TC + 2 * cy * CZ + cj;
            T v = T(0);
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                const int ax = c >> 2, ay = (c >> 1) & 1, az = c & 1, own_colour = (ax + ay + az) & 1;
                const T* q0 = p + ax * PL + ay * HB + own_colour * COLS;
                const T* o = p + ax * PL + ay * HB + (1 - own_colour) * COLS;
                const T w = *q0;
                T ap = T(0);
                if (P || fx + ax + 1 < d.n0) ap += k.w[0] * (w - o[PL]);
                if (P || fx + ax > 0) ap += k.w[0] * (w - o[-PL]);
                if (P || fy + ay + 1 < d.n1) ap += k.w[1] * (w - o[HB]);
                if (P || fy + ay > 0) ap += k.w[1] * (w - o[-HB]);
                if (P || fz + az + 1 < d.n2) ap += k.w[2] * (w - o[az ? 1 : 0]);
                if (P || fz + az > 0) ap += k.w[2] * (w - o[az ? 0 : -1]);
                v += r[(2 * ax + own_colour) * G::TC + ay * CZ] - ap;
            }
            a.restricted[(fx / 2 * (d.n1 / 2) + fy / 2) * (d.n2 / 2) + fz / 2] = v * T(0.125);
        }
    }
}

// Workgroup of a launch over one level. The relaxation, boundary type and
// smoother are uniform; workgroups are dealt to the XCDs in contiguous runs of
// tiles, so halos are re-read from one L2.
template <class T, bool P, bool GS, int TX, int TY, int NPH, bool RESTRICT>
__global__ void __launch_bounds__((Tile3<T, TX, TY, NPH, RESTRICT>::NT)) stage_kernel(StageArgs<T> a, int tiles) {
    extern __shared__ unsigned char raw[];
    stage_tile<T, P, GS, TX, TY, NPH, RESTRICT>(a, int(xcd_tile(blockIdx.x, tiles)), reinterpret_cast<T*>(raw));
}
