// Row-wise assembly of the P1 quadrature operator (gfx950): the node-major
// CSR B_c of mac/assembled_transfer.py:1-8,
//   B_c[a, f] = sum_e sum_q W_eq N_qa phi_c(f - x_eq)   (a = cells[e, local]),
// and its face-major transpose for the three components together.
//
// Why by rows: contracted per cell into a hash table (assembled.hip) every
// site of a cell's stencil box costs a global atomic at a random slot, and
// the table then has to be compacted, sorted by key and sorted again for the
// transpose with 64-bit keys. A row of B_c is nonzero only in the box of the
// node's incident cells (some hundred to some thousand faces), which fits in
// LDS: one wave owns the row, adds the incident cells in ascending order and
// writes the nonzeros in face order. No atomics, no table, no first sort,
// and the sums are the same in every run.
//
// Per cell the points are first grouped by stencil base (cell_order_kernel,
// shared by the cell's nodes). Points of one base have the same 4x4x4 taps,
// so up to four of them are one v_mfma_f64_4x4x4: block y, row x, column z,
// and the four points as its inner dimension,
//   D[y][x][z] = sum_k (phi_x phi_y)_k (phi_z W N)_k,
// one tap per lane: 4 LDS reads and 2 products per lane for 256 tap products
// instead of 12 and 8. The lane's site gets one LDS add per four points.
//
// Bound: the chain of one wave per row (some 20 instructions per chunk of four
// points; VALU issue takes 0.21 of the time with 1.4 waves per SIMD), as many
// rows per CU as their boxes leave room for. 16200 cells of
// 64 points, 4185 nodes, 96^3 faces: all three matrices and transposes 0.93
// ms against 6.83 ms through the table; rows_kernel 427 us, against 785 us
// with the chunks found per node instead of once per cell, the site read and
// written back instead of added to, and one chunk at a time.
#include <algorithm>

#include "binshare.hpp"

namespace afsi {
namespace {

constexpr int PT_STRIDE = 13;     // 12 phi + W N per point; odd: rows spread over the banks
constexpr uint32_t ZERO_POINT = WAVE;  // a row of zeros after the points
constexpr int CELL_WAVES = 4;
constexpr int UNROLL = 4;              // chunks whose operands are read together; divides WAVE
// Chunk slots per cell: a cell of Q points has at most Q chunks.
__host__ __device__ inline int chunk_slots(int quad) { return (quad + UNROLL - 1) / UNROLL * UNROLL; }
// What LDS holds: 128 KB of sites + 6.6 KB of points. Rows beat the table
// wherever they fit. 64 points per cell: 0.28 / 2.78 ms for 468 nodes with
// rows up to 1320 sites, 0.34 / 5.12 ms up to 3808, 0.65 / 7.23 ms up to about
// 12000. Whole preparations with 4 points per tetrahedron: 0.46 / 2.12 ms for
// 384 cells on 32^3, 0.88 / 6.14 ms for 48000; with 3 per triangle: 0.66 /
// 4.20 ms for 20480.
constexpr int64_t ROW_SITES = 16384;

struct RowStats {  // int64 words, zeroed by the caller
    unsigned long long raw[3];
    long long max_sites;
    unsigned long long flag;  // 1: a span over 255, 2: invalid cell or box, 4: nonfinite entry
};

template <typename Op>
__device__ inline int wave_all(int v, Op op) {
#pragma unroll
    for (int m = 32; m > 0; m >>= 1) v = op(v, __shfl_xor(v, m));
    return v;
}

// One wave per (component, cell): the box of the points' bases, and the
// points of each base in chunks of at most four: x = four point numbers of 8
// bits, ZERO_POINT where there is none; y = the base relative to the box (8
// bits per axis), and in the first chunk's top byte the number of chunks less
// one. Groups by first appearance, points ascending; the list is filled with
// empty chunks.
__global__ void __launch_bounds__(CELL_WAVES* WAVE) cell_order_kernel(afsi_fe_geometry g,
                                                                      const int64_t* __restrict__ base,
                                                                      afsi_grid3 grid, uint2* __restrict__ chunks,
                                                                      int32_t* __restrict__ cell_box,
                                                                      RowStats* stats) {
    __shared__ unsigned long long part[CELL_WAVES];
    __shared__ uint32_t ids[CELL_WAVES][WAVE], offs[CELL_WAVES][WAVE];
    const int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE, c = blockIdx.y;
    const int Q = g.quad, A = g.nodes_per_cell, slots = chunk_slots(Q);
    const int64_t P = g.elements * Q;
    int64_t extent[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) extent[a] = grid.n[a] + (a == c ? 1 : 0);
    const auto least = [](int a, int b) { return min(a, b); };
    const auto most = [](int a, int b) { return max(a, b); };
    unsigned long long raw = 0;
    for (int64_t e = int64_t(blockIdx.x) * CELL_WAVES + wave; e < g.elements; e += int64_t(gridDim.x) * CELL_WAVES) {
        const int64_t first = int64_t(c) * P + e * Q;
        int b[3] = {0, 0, 0}, lo[3], span[3];
        bool bad = false;
        const bool mine = lane < Q;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const int64_t v = mine ? base[(first + lane) * 3 + a] : 0;
            bad = bad || v <= -(1 << 28) || v >= (1 << 28);
            b[a] = int(v);
        }
        if (lane < A) {
            const int64_t node = g.cells[e * A + lane];
            bad = bad || node < 0 || node >= g.node_count;
        }
        bool wide = false;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            lo[a] = wave_all(mine ? b[a] : 1 << 28, least);
            const int hi = wave_all(mine ? b[a] : -(1 << 28), most);
            span[a] = hi - lo[a];
            bad = bad || lo[a] < 0 || int64_t(hi) + 4 > extent[a];
            wide = wide || span[a] > 255;
        }
        if (__ballot(bad)) {
            if (lane == 0) atomicOr(&stats->flag, 2ull);
            continue;
        }
        if (lane == 0) {
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                cell_box[(int64_t(c) * g.elements + e) * 6 + a] = lo[a];
                cell_box[(int64_t(c) * g.elements + e) * 6 + 3 + a] = lo[a] + span[a] + 4;
            }
        }
        raw += (unsigned long long)(span[0] + 4) * (unsigned long long)(span[1] + 4) * (unsigned long long)(span[2] + 4);
        if (wide) {
            if (lane == 0) atomicOr(&stats->flag, 1ull);
            continue;
        }
        const uint32_t key = uint32_t(b[0] - lo[0]) | uint32_t(b[1] - lo[1]) << 8 | uint32_t(b[2] - lo[2]) << 16;
        unsigned long long todo = __ballot(mine);
        int start = 0, pos = 0;  // in slots of four per chunk
        while (todo) {
            const uint32_t k = __builtin_amdgcn_readlane(key, __builtin_ctzll(todo));
            const unsigned long long same = __ballot(mine && key == k);
            if (mine && key == k) pos = start + __popcll(same & ((1ull << lane) - 1));
            start += (__popcll(same) + 3) / 4 * 4;
            todo &= ~same;
        }
        // the wave's own words: LDS operations of a wave complete in order
        ids[wave][lane] = ZERO_POINT * 0x01010101u;
        offs[wave][lane] = 0;
        __builtin_amdgcn_wave_barrier();
        if (mine) {
            reinterpret_cast<uint8_t*>(ids[wave])[pos] = uint8_t(lane);
            offs[wave][pos / 4] = key;
        }
        __builtin_amdgcn_wave_barrier();
        uint2 chunk = make_uint2(ids[wave][lane], offs[wave][lane]);
        if (lane == 0) chunk.y |= uint32_t(start / 4 - 1) << 24;
        if (lane < slots) chunks[(int64_t(c) * g.elements + e) * slots + lane] = chunk;
        __builtin_amdgcn_wave_barrier();
    }
    if (lane == 0) part[wave] = raw;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < CELL_WAVES; ++w) raw += part[w];
        if (raw) atomicAdd(&stats->raw[c], raw);
    }
}

// Row r = c * nodes + a: the union of its cells' boxes (lo, width) and its
// number of sites.
__global__ void __launch_bounds__(256) row_box_kernel(afsi_fe_geometry g, const int32_t* __restrict__ cell_box,
                                                      int32_t* __restrict__ row_box, int64_t* __restrict__ sites,
                                                      RowStats* stats) {
    const int64_t rows = 3 * g.node_count;
    if (stats->flag) return;  // boxes of invalid cells were not written
    for (int64_t r = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; r < rows; r += int64_t(gridDim.x) * blockDim.x) {
        const int64_t c = r / g.node_count, a = r - c * g.node_count;
        int lo[3] = {1 << 30, 1 << 30, 1 << 30}, hi[3] = {0, 0, 0};
        const int32_t end = g.node_ptr[a + 1], begin = g.node_ptr[a];
        for (int32_t k = begin; k < end; ++k) {
            const int32_t* box = cell_box + (c * g.elements + g.node_items[k] / g.nodes_per_cell) * 6;
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                lo[d] = min(lo[d], box[d]);
                hi[d] = max(hi[d], box[3 + d]);
            }
        }
        int64_t n = begin < end ? 1 : 0;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            row_box[r * 6 + d] = lo[d];
            row_box[r * 6 + 3 + d] = hi[d] - lo[d];
            n *= hi[d] - lo[d];
        }
        sites[r] = n;
        if (n > 512) atomicMax(&stats->max_sites, (long long)n);
    }
}

__device__ inline int64_t row_of_block(int64_t rows) {
    // workgroups go round-robin over the 8 XCDs: each takes a contiguous run
    // of rows, whose nodes share cells, so their points are read from its L2
    const int64_t chunk = (rows + 7) / 8;
    return (blockIdx.x % 8) * chunk + blockIdx.x / 8;
}

// One wave per row: sites in LDS, then the nonzeros in face order to
// cols / vals at site_ptr[r - 1] (an upper bound) and their number.
__global__ void __launch_bounds__(WAVE) rows_kernel(afsi_fe_geometry g, const double* __restrict__ phi,
                                                    afsi_grid3 grid, const uint2* __restrict__ chunks,
                                                    const int32_t* __restrict__ cell_box,
                                                    const int32_t* __restrict__ row_box,
                                                    const int64_t* __restrict__ site_ptr,
                                                    int32_t* __restrict__ cols, double* __restrict__ vals,
                                                    int64_t* __restrict__ counts, RowStats* stats) {
    extern __shared__ double lds[];
    double* pts = lds;
    double* acc = lds + (WAVE + 1) * PT_STRIDE;
    const int64_t rows = 3 * g.node_count;
    const int64_t r = row_of_block(rows);
    if (blockIdx.x / 8 >= (rows + 7) / 8 || r >= rows) return;
    const int lane = threadIdx.x, Q = g.quad, A = g.nodes_per_cell, slots = chunk_slots(Q);
    const int64_t c = r / g.node_count, node = r - c * g.node_count;
    const int64_t P = g.elements * Q;
    const int l0 = row_box[r * 6], l1 = row_box[r * 6 + 1], l2 = row_box[r * 6 + 2];
    const int w1 = row_box[r * 6 + 4], w2 = row_box[r * 6 + 5];
    const int64_t out = r ? site_ptr[r - 1] : 0;
    const int sites = int(site_ptr[r] - out);
    for (int i = lane; i < sites; i += WAVE) acc[i] = 0.0;
    if (lane < PT_STRIDE) pts[ZERO_POINT * PT_STRIDE + lane] = 0.0;

    const int32_t begin = g.node_ptr[node], end = g.node_ptr[node + 1];
    // lane k holds incidence k of a batch of 64: item and box origin
    int item = 0, corner = 0;
    const auto fetch_items = [&](int32_t k0) {
        item = g.node_items[min(k0 + lane, end - 1)];
        const int32_t* box = cell_box + (c * g.elements + item / A) * 6;
        corner = ((box[0] - l0) * w1 + (box[1] - l1)) * w2 + (box[2] - l2);
    };
    // a cell's tables are one run of Q * 96 bytes: lanes read consecutive 16
    // bytes and the points keep their own order in LDS
    const double2* __restrict__ taps = reinterpret_cast<const double2*>(phi);
    double2 f[6];
    double weight = 0.0, basis = 0.0;
    uint2 chunk = make_uint2(0, 0);
    const auto fetch = [&](int it) {
        const int64_t e = it / A, first = c * P + e * Q;
        const int q = min(lane, Q - 1);
        chunk = chunks[(c * g.elements + e) * slots + min(lane, slots - 1)];
#pragma unroll
        for (int j = 0; j < 6; ++j) f[j] = taps[first * 6 + min(j * WAVE + lane, Q * 6 - 1)];
        weight = g.weights[e * Q + q];
        basis = g.values[q * A + (it - int(e) * A)];
    };
    int put[6];
#pragma unroll
    for (int j = 0; j < 6; ++j) {
        const int t = min(j * WAVE + lane, Q * 6 - 1);
        put[j] = t / 6 * PT_STRIDE + t % 6 * 2;
    }
    if (begin < end) {
        fetch_items(begin);
        fetch(__builtin_amdgcn_readlane(item, 0));
    }
    const int tx = lane >> 4, ty = (lane >> 2) & 3, tz = lane & 3;
    const int tap = (tx * w1 + ty) * w2 + tz;
    for (int32_t k = begin; k < end; ++k) {
        const int origin = __builtin_amdgcn_readlane(corner, (k - begin) % WAVE) + tap;
        __syncthreads();  // the last incidence's points are used up
#pragma unroll
        for (int j = 0; j < 6; ++j) {
            pts[put[j]] = f[j].x;
            pts[put[j] + 1] = f[j].y;
        }
        if (lane < Q) pts[lane * PT_STRIDE + 12] = weight * basis;
        const uint2 here = chunk;
        if (k + 1 < end) {  // the next incidence's points travel in registers meanwhile
            if ((k + 1 - begin) % WAVE == 0) fetch_items(k + 1);
            fetch(__builtin_amdgcn_readlane(item, (k + 1 - begin) % WAVE));
        }
        __syncthreads();
        // lane i: first site of chunk i
        const int corner_of = (int(here.y & 255u) * w1 + int(here.y >> 8 & 255u)) * w2 + int(here.y >> 16 & 255u);
        const int n = int(__builtin_amdgcn_readlane(here.y, 0) >> 24) + 1;
        for (int i = 0; i < n; i += UNROLL) {  // the slots are a multiple; the rest of a list is empty chunks
            double u[UNROLL], v[UNROLL];
#pragma unroll
            for (int j = 0; j < UNROLL; ++j) {
                // the lane's inner index is tx: point tx of the chunk
                const uint32_t q = __builtin_amdgcn_ubfe(__builtin_amdgcn_readlane(here.x, i + j), 8 * tx, 8);
                const double* p = pts + q * PT_STRIDE;
                u[j] = p[tz] * p[4 + ty];
                v[j] = p[8 + tz] * p[12];
            }
#pragma unroll
            for (int j = 0; j < UNROLL; ++j) {
                const double d = __builtin_amdgcn_mfma_f64_4x4x4f64(u[j], v[j], 0.0, 0, 0, 0);
                // 64 distinct sites, and LDS operations of a wave are done in
                // order: an add without a return has no latency to wait for
                unsafeAtomicAdd(acc + (origin + __builtin_amdgcn_readlane(corner_of, i + j)), d);
            }
        }
    }
    __syncthreads();
    const int64_t n1 = grid.n[1] + (c == 1 ? 1 : 0), n2 = grid.n[2] + (c == 2 ? 1 : 0);
    int count = 0;
    bool bad = false;
    for (int i0 = 0; i0 < sites; i0 += WAVE) {
        const int i = i0 + lane;
        const double v = i < sites ? acc[i] : 0.0;
        bad = bad || !isfinite(v);
        const unsigned long long some = __ballot(v != 0.0);
        if (v != 0.0) {
            const int64_t at = out + count + __popcll(some & ((1ull << lane) - 1));
            const int z = i % w2, xy = i / w2;
            const int y = xy % w1, x = xy / w1;
            cols[at] = int32_t((int64_t(l0 + x) * n1 + (l1 + y)) * n2 + (l2 + z));
            vals[at] = v;
        }
        count += __popcll(some);
    }
    if (__ballot(bad) && lane == 0) atomicOr(&stats->flag, 4ull);
    if (lane == 0) counts[r] = count;
}

// Rows to their place in the CSR, and the pairs to sort by face: key =
// component's first face + face, value = entry. end = inclusive row sums.
__global__ void __launch_bounds__(256) rows_place_kernel(int64_t rows, int64_t nodes, int64_t f1, int64_t f2,
                                                         const int64_t* __restrict__ site_ptr,
                                                         const int64_t* __restrict__ end,
                                                         const int32_t* __restrict__ cols_in,
                                                         const double* __restrict__ vals_in,
                                                         int32_t* __restrict__ row_ptr, int32_t* __restrict__ cols,
                                                         double* __restrict__ vals, int32_t* __restrict__ row_ids,
                                                         uint32_t* __restrict__ keys, uint32_t* __restrict__ entries) {
    const int lane = threadIdx.x % WAVE;
    for (int64_t r = (int64_t(blockIdx.x) * blockDim.x + threadIdx.x) / WAVE; r < rows;
         r += int64_t(gridDim.x) * blockDim.x / WAVE) {
        const int64_t c = r / nodes, a = r - c * nodes;
        const int64_t from = r ? site_ptr[r - 1] : 0, to = r ? end[r - 1] : 0, n = end[r] - to;
        const int64_t first = c ? end[c * nodes - 1] : 0;
        const uint32_t face0 = uint32_t(c == 0 ? 0 : c == 1 ? f1 : f2);
        if (lane == 0) {
            row_ptr[c * (nodes + 1) + a] = int32_t(to - first);
            if (a == nodes - 1) row_ptr[c * (nodes + 1) + nodes] = int32_t(end[r] - first);
        }
        for (int64_t i = lane; i < n; i += WAVE) {
            const int32_t col = cols_in[from + i];
            cols[to + i] = col;
            vals[to + i] = vals_in[from + i];
            row_ids[to + i] = int32_t(a);
            keys[to + i] = face0 + uint32_t(col);
            entries[to + i] = uint32_t(to + i);
        }
    }
}

// The transpose from the sorted entries; face pointers relative to their
// component's first entry.
__global__ void __launch_bounds__(256) rows_transpose_kernel(int64_t nnz, int64_t f1, int64_t f2, int64_t f3,
                                                             const int32_t* __restrict__ perm,
                                                             const int32_t* __restrict__ ptr,
                                                             const int32_t* __restrict__ row_ids,
                                                             const double* __restrict__ vals,
                                                             int32_t* __restrict__ face_ptr,
                                                             int32_t* __restrict__ nodes_t,
                                                             double* __restrict__ vals_t) {
    const int64_t step = int64_t(gridDim.x) * blockDim.x, t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    for (int64_t i = t; i < nnz; i += step) {
        const int32_t k = perm[i];
        nodes_t[i] = row_ids[k];
        vals_t[i] = vals[k];
    }
    for (int64_t i = t; i < f3 + 3; i += step) {  // one more pointer per component
        const int64_t c = i <= f1 ? 0 : i <= f2 + 1 ? 1 : 2;
        const int64_t first = c == 0 ? 0 : c == 1 ? f1 : f2;
        face_ptr[i] = ptr[i - c] - ptr[first];
    }
}

int check_rows(const afsi_fe_geometry* g, const afsi_grid3* grid) {
    AFSI_REQUIRE(g && g->cells && g->values && g->weights && g->node_ptr && g->node_items && grid,
                 "null row assembly argument");
    AFSI_REQUIRE(g->nodes_per_cell >= 1 && g->nodes_per_cell <= 4 && g->quad >= 1 && g->quad <= WAVE &&
                     g->elements > 0 && g->node_count > 0,
                 "row assembly takes cells of at most 4 nodes and 64 points");
    AFSI_REQUIRE(!grid->periodic, "the assembled operator requires a closed MAC box");
    // a wave per row, and a launch takes fewer than 2^32 threads
    AFSI_REQUIRE(g->elements < (int64_t(1) << 28) && WAVE * (3 * g->node_count + 7) < (int64_t(1) << 32),
                 "mesh too large for row assembly");
    return OK;
}

void face_offsets(const afsi_grid3& grid, int64_t f[4]) {
    f[0] = 0;
    for (int c = 0; c < 3; ++c) {
        int64_t n = 1;
        for (int a = 0; a < 3; ++a) n *= grid.n[a] + (a == c ? 1 : 0);
        f[c + 1] = f[c] + n;
    }
}

}  // namespace
}  // namespace afsi

using namespace afsi;

extern "C" {

int64_t afsi_p1_row_sites_limit(void) { return ROW_SITES; }

int afsi_p1_row_boxes_f64(const afsi_fe_geometry* g, const int64_t* base, const afsi_grid3* grid, uint64_t* chunks,
                          int32_t* cell_box, int32_t* row_box, int64_t* sites, int64_t* stats, void* stream) {
    if (int r = check_rows(g, grid)) return r;
    AFSI_REQUIRE(base && chunks && cell_box && row_box && sites && stats, "null row assembly argument");
    hipStream_t s = hipStream_t(stream);
    RowStats* st = reinterpret_cast<RowStats*>(stats);
    cell_order_kernel<<<dim3(grid_for(g->elements, CELL_WAVES, 1024), 3), CELL_WAVES * WAVE, 0, s>>>(
        *g, base, *grid, reinterpret_cast<uint2*>(chunks), cell_box, st);
    AFSI_LAUNCH_CHECK();
    row_box_kernel<<<grid_for(3 * g->node_count, 256, 8192), 256, 0, s>>>(*g, cell_box, row_box, sites, st);
    AFSI_LAUNCH_CHECK();
    return OK;
}

int afsi_p1_rows_f64(const afsi_fe_geometry* g, const double* phi, const afsi_grid3* grid, const uint64_t* chunks,
                     const int32_t* cell_box, const int32_t* row_box, const int64_t* site_ptr, int64_t max_sites,
                     int32_t* cols, double* vals, int64_t* counts, int64_t* stats, void* stream) {
    if (int r = check_rows(g, grid)) return r;
    AFSI_REQUIRE(phi && chunks && cell_box && row_box && site_ptr && cols && vals && counts && stats,
                 "null row assembly argument");
    AFSI_REQUIRE(reinterpret_cast<uintptr_t>(phi) % 16 == 0, "the stencil table must be aligned to 16 bytes");
    AFSI_REQUIRE(max_sites >= 0 && max_sites <= ROW_SITES, "a row's stencil box exceeds %lld sites",
                 (long long)ROW_SITES);
    const size_t bytes = (size_t(WAVE + 1) * PT_STRIDE + size_t(max_sites)) * sizeof(double);
    const void* fn = reinterpret_cast<const void*>(rows_kernel);
    if (int r = dynamic_lds(fn, bytes)) return r;
    const int64_t blocks = cdiv(3 * g->node_count, 8) * 8;
    rows_kernel<<<unsigned(blocks), WAVE, bytes, hipStream_t(stream)>>>(
        *g, phi, *grid, reinterpret_cast<const uint2*>(chunks), cell_box, row_box, site_ptr, cols, vals, counts, reinterpret_cast<RowStats*>(stats));
    AFSI_LAUNCH_CHECK();
    return OK;
}

size_t afsi_p1_rows_csr_workspace_bytes(const afsi_grid3* grid, int64_t nnz) {
    if (!grid || nnz < 0) return 0;
    int64_t f[4];
    face_offsets(*grid, f);
    const auto up = [](size_t b) { return (b + 255) & ~size_t(255); };
    return up(bin_workspace_bytes(nnz)) + 3 * up(size_t(nnz) * 4) + up(size_t(f[3] + 1) * 4);
}

int afsi_p1_rows_csr_f64(const afsi_grid3* grid, int64_t nodes, int64_t nnz, const int64_t* site_ptr,
                         const int64_t* row_end, const int32_t* cols_in, const double* vals_in, int32_t* row_ptr,
                         int32_t* cols, double* vals, int32_t* face_ptr, int32_t* face_nodes, double* face_vals,
                         void* workspace, size_t workspace_bytes, void* stream) {
    AFSI_REQUIRE(grid && site_ptr && row_end && cols_in && vals_in && row_ptr && cols && vals && face_ptr &&
                     face_nodes && face_vals && workspace,
                 "null row assembly argument");
    AFSI_REQUIRE(nodes > 0 && nnz >= 0 && nnz < (int64_t(1) << 31), "row assembly exceeds 2^31 entries");
    int64_t f[4];
    face_offsets(*grid, f);
    AFSI_REQUIRE(f[3] < (int64_t(1) << 31), "MAC grid too large for row assembly");
    AFSI_REQUIRE(workspace_bytes >= afsi_p1_rows_csr_workspace_bytes(grid, nnz), "row assembly workspace too small");
    hipStream_t s = hipStream_t(stream);
    const auto up = [](size_t b) { return (b + 255) & ~size_t(255); };
    char* w = static_cast<char*>(workspace);
    void* sort_ws = w;
    w += up(bin_workspace_bytes(nnz));
    uint32_t* sorted = reinterpret_cast<uint32_t*>(w);
    w += up(size_t(nnz) * 4);
    int32_t* perm = reinterpret_cast<int32_t*>(w);
    w += up(size_t(nnz) * 4);
    int32_t* row_ids = reinterpret_cast<int32_t*>(w);
    w += up(size_t(nnz) * 4);
    int32_t* ptr = reinterpret_cast<int32_t*>(w);
    uint32_t *keys, *entries;
    sort_key_slots(sort_ws, nnz, &keys, &entries);
    rows_place_kernel<<<grid_for(3 * nodes * WAVE, 256, 16384), 256, 0, s>>>(
        3 * nodes, nodes, f[1], f[2], site_ptr, row_end, cols_in, vals_in, row_ptr, cols, vals, row_ids, keys, entries);
    AFSI_LAUNCH_CHECK();
    if (int r = sort_pairs(nnz, f[3], sort_ws, sorted, perm, ptr, s)) return r;
    rows_transpose_kernel<<<grid_for(std::max(nnz, f[3] + 3), 256, 16384), 256, 0, s>>>(
        nnz, f[1], f[2], f[3], perm, ptr, row_ids, vals, face_ptr, face_nodes, face_vals);
    AFSI_LAUNCH_CHECK();
    return OK;
}

}  // extern "C"
