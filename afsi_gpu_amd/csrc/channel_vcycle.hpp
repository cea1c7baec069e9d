// Channel V-cycles in few launches: LDS tiles for the large levels, the rest
// of the hierarchy in the LDS of one workgroup. Included by channel.hip
// (after Dim2, Coef2, ch_apply and ch_diag) inside its anonymous namespace.
//
// A phase of a channel V-cycle (a half-sweep, a restriction) is far smaller
// than a launch: 512x128 FP64 cells are 0.5 MB, 0.1 us at the copy rate,
// against 2.4-5 us for a launch of any size. So launches, and the barriers
// and LDS latency inside them, are what a cycle costs:
//   * chf_tile: one launch runs up to CHF_MAX phases (half-sweeps of the
//     red-black smoother, sweeps of Jacobi) of a level on CHF_T x CHF_T
//     tiles, the halo staged once and the updated ring shrinking by one cell
//     per phase, with the prolongation before the first phase and the
//     residual restriction after the last one in the same launch. A V(2,2)
//     red-black or V(4,4) Jacobi level is two launches per cycle.
//   * chf_tail: the levels below run in one workgroup with every array in
//     LDS, for as many cycles as asked when level 0 itself fits.
// Measured figures stand at channel_cycles in channel.hip.
//
// Updates and the restricted residual use the difference form
// p + omega (b - sum w (p - nb)) / diag, with 1/diag from a nine-entry table
// (low end, interior, high end of each axis). Differences of neighbours are
// nearly exact and the quotient is a small correction, so a stored value
// carries little more than its own rounding; in the form (b + sum w nb) / diag
// the residual stagnates 1.45 to 3 times higher.
//
// Means of a periodic channel: A p has mean zero, so every residual has the
// mean of rhs[0], and so has its restriction. That mean is subtracted once, as
// level 0 is restricted; what is left below is rounding, which the coarse
// product drops (its inverse would return it as a shift of p). The mean of p
// is removed after the last cycle only: A 1 = 0, and smoothing, restriction
// and prolongation commute with a constant shift.

constexpr int CHF_T = 16;                    // tile edge
constexpr int CHF_MAX = 7;                   // phases per launch (halo CHF_MAX + 1 <= CHF_T / 2)
constexpr int CHF_NT = CHF_T * CHF_T;        // thread (i, j): rows i, i + 16 of the box, cell pair j
constexpr int CHF_B = CHF_T + 2 * (CHF_MAX + 1);
constexpr int CHF_PITCH = CHF_B + 1;
static_assert(CHF_B == 2 * CHF_T, "two rows and one pair of columns per thread");

constexpr int CHF_TAIL_NT = 1024;
constexpr size_t CHF_TAIL_LDS = 150 * 1024;  // of 160 KB; the tables and reductions take the rest
constexpr int CHF_TAIL_PAIRS = 2;            // cell pairs per thread: levels of at most 4096 cells

// Mean of `count` values from `parts` partial sums, `stride` apart, in every
// lane and in a fixed order.
__device__ inline double chf_mean(const double* __restrict__ partials, int parts, int stride, int count) {
    double v = 0.0;
    for (int b = int(threadIdx.x) % WAVE; b < parts; b += WAVE) v += partials[int64_t(b) * stride];
#pragma unroll
    for (int dd = 32; dd >= 1; dd >>= 1) v += __shfl_xor(v, dd, WAVE);
    return v / double(count);
}

// Phases of one smoothing stage.
__host__ __device__ inline int chf_phases(const afsi_mg2d_plan& pl) { return pl.smoother == 1 ? 2 * pl.nu : pl.nu; }

__host__ __device__ inline int chf_chunks(const afsi_mg2d_plan& pl) { return (chf_phases(pl) + CHF_MAX - 1) / CHF_MAX; }

__host__ __device__ inline int chf_tiles(const afsi_mg2d_plan& pl, int l) {
    return int(((pl.n[l][0] + CHF_T - 1) / CHF_T) * ((pl.n[l][1] + CHF_T - 1) / CHF_T));
}

template <class T>
__device__ inline Coef2<T> chf_coef(const afsi_mg2d_plan& pl, int l) {
    return coef2_of<T>(pl.h2[l][0], pl.h2[l][1], pl.inv_h2[l][0], pl.inv_h2[l][1]);
}

// Diagonal of a cell by its class per axis (0: x or y is the first, 1:
// interior, 2: last), in ch_diag's order.
template <class T, bool P>
__device__ inline T chf_diag(int cx, int cy, const Coef2<T>& k) {
    T g = T(0);
    if (P || cx != 2) g += k.ihx2;
    if (P || cx != 0) g += k.ihx2;
    if (cy != 2) g += k.ihy2;
    if (cy != 0) g += k.ihy2;
    if (!P && cx == 2) g += T(2) * k.ihx2;
    return g;
}

__device__ inline int chf_class(int i, int n) { return i == 0 ? 0 : (i == n - 1 ? 2 : 1); }

// A cell pair (y = 2j, 2j + 1 of one row) as one thread keeps it: cell 0 is
// the one that even red-black phases update, cell 1 the other (the order of
// the row's parity); Jacobi updates both in every phase. Values, addresses,
// right-hand sides and omega/diag stay in registers over all phases, and the
// pair's cells are each other's neighbour, so an update is three LDS reads,
// nine or ten operations and one LDS write. (Decoding the cell, its boundary
// class and its neighbours in every phase instead was bound by VALU issue:
// 26.7 us for a 128x32 tail, 6.7 us for a 256x64 tile launch.) A missing
// neighbour's address is the cell's own: its difference is zero.
template <class T>
struct ChfPair {
    int at[2], outer[2], up, down;  // LDS elements; up and down belong to cell 0
    T p[2], rhs[2], scale[2];       // scale: omega / diag
    T outlet;                       // 2/hx^2 in the outlet row of a closed channel (value -p beyond it), else 0
};

// The new value of cell o from the iterate `a`.
template <class T, bool P>
__device__ __forceinline__ T chf_update(const T* a, const ChfPair<T>& c, int o, T wx, T wy) {
    const int step = c.at[o] - c.at[0];
    const T p = c.p[o], dx = (a[c.up + step] - p) + (a[c.down + step] - p), dy = (a[c.outer[o]] - p) + (c.p[1 - o] - p);
    T r = fma_of(wy, dy, fma_of(wx, dx, c.rhs[o]));
    if (!P) r = fma_of(-c.outlet, p, r);
    return fma_of(c.scale[o], r, p);
}

// One launch's share of level l: tile `tile` of chunk `chunk` of the pre-
// (up = false) or post-smoothing (up = true) stage. Chunk c reads the buffer
// that chunk c - 1 wrote; p and tmp alternate, and both stages have the same
// number of chunks, so the level's iterate ends in p. The halo is even, so a
// thread's cell pairs are the children of coarse cells. A cell is updated in
// phase s while it lies more than s cells from the box edge. `mean` is
// subtracted from the restricted residual.
template <class T, bool P>
__device__ __forceinline__ void chf_tile(const afsi_mg2d_plan& pl, int l, int tile, int chunk, bool up, T mean, T* box,
                                         T* tab) {
    const Dim2 d{int(pl.n[l][0]), int(pl.n[l][1])};
    const Coef2<T> k = chf_coef<T>(pl, l);
    const bool gs = pl.smoother == 1;
    const int phases = chf_phases(pl), chunks = chf_chunks(pl);
    const int first = chunk * CHF_MAX, count = min(CHF_MAX, phases - first);
    const bool prolong = up && chunk == 0, restricts = !up && chunk == chunks - 1;
    const bool zero = !up && chunk == 0 && l > 0;
    const bool swap = ((chunk + (up ? chunks : 0)) & 1) != 0;
    const T* __restrict__ in = static_cast<const T*>(swap ? pl.tmp[l] : pl.p[l]);
    T* __restrict__ out = static_cast<T*>(swap ? pl.p[l] : pl.tmp[l]);
    const T* __restrict__ rhs = static_cast<const T*>(pl.rhs[l]);
    const int H = (count + (restricts ? 1 : 0) + 1) & ~1, span = CHF_T + 2 * H;
    const int nty = (d.ny + CHF_T - 1) / CHF_T;
    const int x0 = (tile / nty) * CHF_T - H, y0 = (tile % nty) * CHF_T - H;
    const int ti = int(threadIdx.x) / CHF_T, tj = int(threadIdx.x) % CHF_T;
    constexpr int SIZE = CHF_B * CHF_PITCH, ROWS = CHF_B / CHF_T;

    if (threadIdx.x < 9) tab[threadIdx.x] = T(1) / chf_diag<T, P>(int(threadIdx.x) / 3, int(threadIdx.x) % 3, k);
    const T* __restrict__ coarse = prolong ? static_cast<const T*>(pl.p[l + 1]) : nullptr;
    const int j = 2 * tj, gy = y0 + j;
    ChfPair<T> c[ROWS];
    int depth[ROWS][2], row[ROWS];  // depth 0: never updated; row: the global row, -1 outside the domain
#pragma unroll
    for (int q = 0; q < ROWS; ++q) {
        const int i = ti + q * CHF_T;
        int gx = x0 + i;
        if (P) gx = ((gx % d.nx) + d.nx) % d.nx;
        const bool held = i < span && j < span;
        const bool inside = held && gx >= 0 && gx < d.nx && gy >= 0 && gy < d.ny;  // pairs do not straddle walls
        row[q] = inside ? gx : -1;
        T v[2] = {T(0), T(0)}, b[2] = {T(0), T(0)};
        if (inside) {
            const int at = gx * d.ny + gy;
            if (!zero) {
                v[0] = in[at];
                v[1] = in[at + 1];
            }
            b[0] = rhs[at];
            b[1] = rhs[at + 1];
            if (prolong) {
                const int NX = d.nx / 2, NY = d.ny / 2, ax = gx / 2 - 1 + (gx & 1), Y = gy / 2;
                const T wx = (gx & 1) ? T(0.25) : T(0.75);
                T lo[2], mid[2], hi[2];
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    lo[s] = ch_coarse_value<T, P>(coarse, ax + s, Y - 1, NX, NY);
                    mid[s] = ch_coarse_value<T, P>(coarse, ax + s, Y, NX, NY);
                    hi[s] = ch_coarse_value<T, P>(coarse, ax + s, Y + 1, NX, NY);
                }
                const T lw = T(0.25), hw = T(0.75);
                v[0] += (lo[0] * lw + mid[0] * hw) * (T(1) - wx) + (lo[1] * lw + mid[1] * hw) * wx;
                v[1] += (mid[0] * hw + hi[0] * lw) * (T(1) - wx) + (mid[1] * hw + hi[1] * lw) * wx;
            }
        }
        const int at = i * CHF_PITCH + j;
        if (held) {
            box[at] = v[0];
            box[at + 1] = v[1];
            if (!gs) box[SIZE + at] = box[SIZE + at + 1] = T(0);
        }
        const int lead = gx & 1;  // even rows start with the even cell (gy is even)
        const int across = min(i, span - 1 - i);
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const int o = lead ^ s;
            const bool wall = o ? gy + 2 == d.ny : gy == 0;
            c[q].at[s] = held ? at + o : CHF_PITCH + 1;
            c[q].outer[s] = c[q].at[s] + (wall ? 0 : (o ? 1 : -1));
            c[q].p[s] = o ? v[1] : v[0];
            c[q].rhs[s] = o ? b[1] : b[0];
            depth[q][s] = inside ? min(across, min(j + o, span - 1 - j - o)) : 0;
        }
        c[q].up = c[q].at[0] + (P || gx + 1 != d.nx ? CHF_PITCH : 0);
        c[q].down = c[q].at[0] - (P || gx != 0 ? CHF_PITCH : 0);
        c[q].outlet = !P && gx + 1 == d.nx ? T(2) * k.ihx2 : T(0);
    }
    const T omega = gs ? T(1) : T(pl.omega);
    __syncthreads();
#pragma unroll
    for (int q = 0; q < ROWS; ++q)
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const int y = gy + ((row[q] & 1) ^ s), cx = P ? 1 : chf_class(row[q], d.nx);
            c[q].scale[s] = row[q] >= 0 ? omega * tab[3 * cx + chf_class(y, d.ny)] : T(0);
        }

    T* a = box;
    T* w = gs ? box : box + SIZE;
    for (int s = 0; s < count; ++s) {
        const int mine = (first + s) & 1;
#pragma unroll
        for (int q = 0; q < ROWS; ++q) {
            T v[2] = {c[q].p[0], c[q].p[1]};
#pragma unroll
            for (int o = 0; o < 2; ++o) {
                if ((gs && o != mine) || depth[q][o] <= s) continue;
                v[o] = chf_update<T, P>(a, c[q], o, k.ihx2, k.ihy2);
                w[c[q].at[o]] = v[o];
            }
            c[q].p[0] = v[0];
            c[q].p[1] = v[1];
        }
        __syncthreads();
        T* t = a; a = w; w = t;
    }

#pragma unroll
    for (int q = 0; q < ROWS; ++q) {
        const int i = ti + q * CHF_T;
        // rows of the tile, not of its periodic copies beyond the domain
        const bool mine = row[q] >= 0 && i >= H && i < H + CHF_T && x0 + i < d.nx && j >= H && j < H + CHF_T;
        T r[2] = {T(0), T(0)};
        if (mine) {
            const int at = i * CHF_PITCH + j, gx = row[q];
#pragma unroll
            for (int o = 0; o < 2; ++o) {
                const T* f = a + at + o;
                const T v = *f;
                out[gx * d.ny + gy + o] = v;
                if (!restricts) continue;
                T s = T(0);
                if (P || gx + 1 < d.nx) s -= k.ihx2 * (f[CHF_PITCH] - v);
                if (P || gx > 0) s += k.ihx2 * (v - f[-CHF_PITCH]);
                if (gy + o + 1 < d.ny) s -= k.ihy2 * (f[1] - v);
                if (gy + o > 0) s += k.ihy2 * (v - f[-1]);
                if (!P && gx == d.nx - 1) s += T(2) * k.ihx2 * v;
                r[o] = ((gx & 1) ? c[q].rhs[o ^ 1] : c[q].rhs[o]) - s;
            }
        }
        if (restricts) {  // rows 2X and 2X + 1 are lanes t and t + 16
            const T r10 = __shfl_down(r[0], CHF_T, WAVE), r11 = __shfl_down(r[1], CHF_T, WAVE);
            if (mine && !(i & 1))
                static_cast<T*>(pl.rhs[l + 1])[(row[q] / 2) * (d.ny / 2) + gy / 2] =
                    (((r[0] + r[1]) + r10) + r11) * T(0.25) - mean;
        }
    }
}

// ---- the lower levels in one workgroup ---------------------------------------
// LDS of level l: p as rows of ny + 2 words (an even pitch other than ny, a
// power of two as a rule, spreads rows over the banks), a second p for Jacobi,
// and rhs. The coarsest level keeps p and rhs in cell order.
__host__ __device__ inline int chf_box_cells(const afsi_mg2d_plan& pl, int l) {
    return int(pl.n[l][0] * (pl.n[l][1] + 2));
}

__host__ __device__ inline int chf_level_values(const afsi_mg2d_plan& pl, int l) {
    const int cells = int(pl.n[l][0] * pl.n[l][1]);
    if (l == pl.levels - 1) return 2 * cells;
    return cells + (pl.smoother == 1 ? 1 : 2) * chf_box_cells(pl, l);
}

// First level whose hierarchy fits the tail's LDS (the coarsest level, at
// most 512 cells, always does).
__host__ inline int chf_split(const afsi_mg2d_plan& pl, size_t value_bytes, size_t* bytes) {
    size_t need = 0;
    int l = pl.levels - 1;
    for (;; --l) {
        const size_t more = need + size_t(chf_level_values(pl, l)) * value_bytes;
        const bool fits = more <= CHF_TAIL_LDS && pl.n[l][0] * pl.n[l][1] <= 2 * CHF_TAIL_PAIRS * CHF_TAIL_NT;
        if (!fits) { ++l; break; }
        need = more;
        if (l == 0) break;
    }
    if (bytes) *bytes = need;
    return l;
}

// A tail level's extents, weights and LDS offsets, formed once per launch.
template <class T>
struct ChfLevel {
    int nx, ny, p, q, r;  // q < 0: no second iterate
    T wx, wy;             // 1/h^2
};

// Block-strided cells of a level by (x, y-pair): e / h for e < 2^13 through
// one float product (exact: the quotient is at least 1/(2h) from an integer).
struct ChfPairs {
    int h, n;
    float r;
    __device__ ChfPairs(int nx, int ny) : h(ny / 2), n(nx * (ny / 2)), r(1.0f / float(ny / 2)) {}
    __device__ void at(int e, int& x, int& j) const {
        x = int((float(e) + 0.5f) * r);
        j = e - x * h;
    }
};

// One smoothing stage of a level; the iterate enters and ends in p.
template <class T, bool P>
__device__ __forceinline__ void chf_smooth(const ChfLevel<T> v, bool gs, int phases, T omega, T* lds, const T* tab) {
    const ChfPairs pairs(v.nx, v.ny);
    const int pitch = v.ny + 2;
    T *a = lds + v.p, *w = gs ? a : lds + v.q;
    ChfPair<T> c[CHF_TAIL_PAIRS];
#pragma unroll
    for (int q = 0; q < CHF_TAIL_PAIRS; ++q) {
        const int e = int(threadIdx.x) + q * CHF_TAIL_NT;
        if (e >= pairs.n) continue;
        int x, j;
        pairs.at(e, x, j);
        const int above = (x + 1 < v.nx ? x + 1 : (P ? 0 : x)) * pitch;
        const int below = (x > 0 ? x - 1 : (P ? v.nx - 1 : x)) * pitch;
        const int lead = x & 1, cx = P ? 1 : chf_class(x, v.nx);
        const T* r = lds + v.r + x * v.ny + 2 * j;
        const T r0 = r[0], r1 = r[1];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const int o = lead ^ s, y = 2 * j + o, outer = o ? y + 1 : y - 1;
            c[q].at[s] = x * pitch + y + 1;
            c[q].outer[s] = x * pitch + (outer < 0 || outer == v.ny ? y : outer) + 1;
            c[q].p[s] = a[c[q].at[s]];
            c[q].scale[s] = omega * tab[3 * cx + chf_class(y, v.ny)];
            c[q].rhs[s] = o ? r1 : r0;
        }
        c[q].outlet = !P && x + 1 == v.nx ? T(2) * v.wx : T(0);
        c[q].up = above + 2 * j + lead + 1;
        c[q].down = below + 2 * j + lead + 1;
    }
    for (int s = 0; s < phases; ++s) {
        const int mine = s & 1;
#pragma unroll
        for (int q = 0; q < CHF_TAIL_PAIRS; ++q) {
            if (int(threadIdx.x) + q * CHF_TAIL_NT >= pairs.n) continue;
            T u[2] = {c[q].p[0], c[q].p[1]};
#pragma unroll
            for (int o = 0; o < 2; ++o) {
                if (gs && o != mine) continue;
                u[o] = chf_update<T, P>(a, c[q], o, v.wx, v.wy);
                w[c[q].at[o]] = u[o];
            }
            c[q].p[0] = u[0];
            c[q].p[1] = u[1];
        }
        __syncthreads();
        T* t = a; a = w; w = t;
    }
    if (a != lds + v.p) {
#pragma unroll
        for (int q = 0; q < CHF_TAIL_PAIRS; ++q)
            if (int(threadIdx.x) + q * CHF_TAIL_NT < pairs.n)
#pragma unroll
                for (int o = 0; o < 2; ++o) w[c[q].at[o]] = c[q].p[o];
        __syncthreads();
    }
}

// Shared tables of a tail workgroup.
template <class T>
struct ChfShared {
    ChfLevel<T> level[AFSI_MG_MAX_LEVELS];
    T tab[AFSI_MG_MAX_LEVELS][9];
    double red[CHF_TAIL_NT / WAVE];
};

// Levels l0..last of `cycles` V-cycles: rhs[l0] comes from global memory and
// p[l0] goes back there; l0 > 0 starts from zero, l0 == 0 from p[0].
template <class T, bool P>
__device__ __forceinline__ void chf_tail(const afsi_mg2d_plan& pl, int l0, int cycles, T* lds, ChfShared<T>& sh) {
    const int last = pl.levels - 1, tid = int(threadIdx.x), phases = chf_phases(pl);
    const bool gs = pl.smoother == 1;
    const T omega = gs ? T(1) : T(pl.omega);
    int total = 0;
    for (int l = l0; l <= last; ++l) {
        const int cells = int(pl.n[l][0] * pl.n[l][1]), box = l == last ? cells : chf_box_cells(pl, l);
        const bool two = !gs && l < last;
        if (tid == 0)
            sh.level[l] = ChfLevel<T>{int(pl.n[l][0]), int(pl.n[l][1]), total, two ? total + box : -1,
                                      total + (two ? 2 : 1) * box, T(pl.inv_h2[l][0]), T(pl.inv_h2[l][1])};
        if (l < last && tid < 9) sh.tab[l][tid] = T(1) / chf_diag<T, P>(tid / 3, tid % 3, chf_coef<T>(pl, l));
        total += chf_level_values(pl, l);
    }
    for (int i = tid; i < total; i += CHF_TAIL_NT) lds[i] = T(0);
    // rows of a small coarse inverse stay in registers: row ROWS * wave + i, column lane
    const int m = int(pl.coarse_cells), wave = tid / WAVE, lane = tid % WAVE;
    const T* A = static_cast<const T*>(pl.coarse_inverse);
    constexpr int ROWS = WAVE / (CHF_TAIL_NT / WAVE);
    T held[ROWS];
#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
        const int row = ROWS * wave + i;
        held[i] = m <= WAVE && row < m && lane < m ? A[row * m + lane] : T(0);
    }
    __syncthreads();
    const ChfLevel<T> top = sh.level[l0];
    {
        const T* rhs = static_cast<const T*>(pl.rhs[l0]);
        for (int i = tid; i < top.nx * top.ny; i += CHF_TAIL_NT) lds[top.r + i] = rhs[i];
        if (l0 == 0 && l0 < last) {
            const ChfPairs pairs(top.nx, top.ny);
            const T* src = static_cast<const T*>(pl.p[0]);
            for (int e = tid; e < pairs.n; e += CHF_TAIL_NT) {
                int x, j;
                pairs.at(e, x, j);
                const T v0 = src[x * top.ny + 2 * j], v1 = src[x * top.ny + 2 * j + 1];
                lds[top.p + x * (top.ny + 2) + 2 * j + 1] = v0;
                lds[top.p + x * (top.ny + 2) + 2 * j + 2] = v1;
            }
        }
    }
    __syncthreads();
    // mean of the n words at x (LDS), in every thread
    const auto mean_of = [&](const T* x, int n, int pitch) -> T {
        const float inverse = 1.0f / float(top.ny);
        double sum = 0.0;
        for (int i = tid; i < n; i += CHF_TAIL_NT) {
            const int r = int((float(i) + 0.5f) * inverse);
            sum += double(x[r * pitch + i - r * top.ny]);
        }
#pragma unroll
        for (int dd = 32; dd >= 1; dd >>= 1) sum += __shfl_xor(sum, dd, WAVE);
        if (lane == 0) sh.red[wave] = sum;
        __syncthreads();
        sum = 0.0;
        for (int w = 0; w < CHF_TAIL_NT / WAVE; ++w) sum += sh.red[w];
        return T(sum / double(n));
    };
    const int cells = top.nx * top.ny;
    const T rhs_mean = P && l0 == 0 && l0 < last ? mean_of(lds + top.r, cells, top.ny) : T(0);
    for (int cycle = 0; cycle < cycles; ++cycle) {
        for (int l = l0; l < last; ++l) {
            const ChfLevel<T> v = sh.level[l], c = sh.level[l + 1];
            chf_smooth<T, P>(v, gs, phases, omega, lds, sh.tab[l]);
            const int pitch = v.ny + 2;
            const float inverse = 1.0f / float(c.ny);
            for (int e = tid; e < c.nx * c.ny; e += CHF_TAIL_NT) {
                const int X = int((float(e) + 0.5f) * inverse), Y = e - X * c.ny;
                T res[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int x = 2 * X + (q >> 1), y = 2 * Y + (q & 1);
                    const T* f = lds + v.p + x * pitch + y + 1;
                    T s = T(0);
                    if (P || x + 1 < v.nx) s -= v.wx * (f[x + 1 < v.nx ? pitch : -x * pitch] - *f);
                    if (P || x > 0) s += v.wx * (*f - f[x > 0 ? -pitch : (v.nx - 1) * pitch]);
                    if (y + 1 < v.ny) s -= v.wy * (f[1] - *f);
                    if (y > 0) s += v.wy * (*f - f[-1]);
                    if (!P && x == v.nx - 1) s += T(2) * v.wx * *f;
                    res[q] = lds[v.r + x * v.ny + y] - s;
                }
                lds[c.r + e] = (((res[0] + res[1]) + res[2]) + res[3]) * T(0.25) - (l == 0 ? rhs_mean : T(0));
                if (l + 1 < last) lds[c.p + X * (c.ny + 2) + Y + 1] = T(0);
            }
            __syncthreads();
        }
        const ChfLevel<T> bottom = sh.level[last];
        if (m <= WAVE) {
            T x = lane < m ? lds[bottom.r + lane] : T(0);
            if (P) {
                T sum = x;
#pragma unroll
                for (int dd = 32; dd >= 1; dd >>= 1) sum += __shfl_xor(sum, dd, WAVE);
                x = lane < m ? x - sum / T(m) : T(0);
            }
#pragma unroll
            for (int i = 0; i < ROWS; ++i) {
                T acc = held[i] * x;
#pragma unroll
                for (int dd = 32; dd >= 1; dd >>= 1) acc += __shfl_xor(acc, dd, WAVE);
                if (lane == 0 && ROWS * wave + i < m) lds[bottom.p + ROWS * wave + i] = acc;
            }
        } else {
            T mean = T(0);
            if (P) {
                for (int c = lane; c < m; c += WAVE) mean += lds[bottom.r + c];
#pragma unroll
                for (int dd = 32; dd >= 1; dd >>= 1) mean += __shfl_xor(mean, dd, WAVE);
                mean /= T(m);
            }
            for (int row = wave; row < m; row += CHF_TAIL_NT / WAVE) {
                T acc = T(0);
                for (int c = lane; c < m; c += WAVE) acc += A[row * m + c] * (lds[bottom.r + c] - mean);
#pragma unroll
                for (int dd = 32; dd >= 1; dd >>= 1) acc += __shfl_xor(acc, dd, WAVE);
                if (lane == 0) lds[bottom.p + row] = acc;
            }
        }
        __syncthreads();
        for (int l = last - 1; l >= l0; --l) {
            const ChfLevel<T> v = sh.level[l], c = sh.level[l + 1];
            const int cp = l + 1 == last ? c.ny : c.ny + 2;
            const T* coarse = lds + c.p + (l + 1 == last ? 0 : 1);
            const ChfPairs pairs(v.nx, v.ny);
            const int pitch = v.ny + 2;
            for (int e = tid; e < pairs.n; e += CHF_TAIL_NT) {
                int x, Y;
                pairs.at(e, x, Y);
                const int ax = x / 2 - 1 + (x & 1);
                const T wx = (x & 1) ? T(0.25) : T(0.75);
                const int lo = Y > 0 ? Y - 1 : 0, hi = Y + 1 < c.ny ? Y + 1 : c.ny - 1;
                T even[2], odd[2];
#pragma unroll
                for (int s = 0; s < 2; ++s) {  // clamped at the inlet and walls, negated beyond the outlet
                    int xx = ax + s;
                    T sign = T(1);
                    if (P) {
                        xx = xx < 0 ? xx + c.nx : (xx >= c.nx ? xx - c.nx : xx);
                    } else {
                        sign = xx >= c.nx ? T(-1) : T(1);
                        xx = xx < 0 ? 0 : (xx >= c.nx ? c.nx - 1 : xx);
                    }
                    const T* row = coarse + xx * cp;
                    const T mid = sign * row[Y];
                    even[s] = (sign * row[lo]) * T(0.25) + mid * T(0.75);
                    odd[s] = mid * T(0.75) + (sign * row[hi]) * T(0.25);
                }
                T* f = lds + v.p + x * pitch + 2 * Y + 1;
                f[0] += even[0] * (T(1) - wx) + even[1] * wx;
                f[1] += odd[0] * (T(1) - wx) + odd[1] * wx;
            }
            __syncthreads();
            chf_smooth<T, P>(v, gs, phases, omega, lds, sh.tab[l]);
        }
    }
    const int pitch = l0 == last ? top.ny : top.ny + 2;
    const T* src = lds + top.p + (l0 == last ? 0 : 1);
    const float inverse = 1.0f / float(top.ny);
    const T mean = P && l0 == 0 ? mean_of(src, cells, pitch) : T(0);
    T* out = static_cast<T*>(pl.p[l0]);
    for (int i = tid; i < cells; i += CHF_TAIL_NT) {
        const int x = int((float(i) + 0.5f) * inverse), y = i - x * top.ny;
        out[i] = src[x * pitch + y] - mean;
    }
}
