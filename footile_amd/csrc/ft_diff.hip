// ft_diff.hip -- the differentiable fill on gfx950: float32 analytic-coverage
// forward and a hand-written adjoint.  footile has no counterpart; the model
// (fixed dyadic flattening of cubics, winding-integral pixel coverage, SrcOver
// in path order) is specified by the FP64 oracle the tests compare against.
//
// Per step:
//   k_geometry   control points -> polygon vertices (16 per cubic, Bernstein),
//                edge lists per (path, row)
//   k_forward    one lane per pixel of a row tile: coverage of the image's
//                paths, 16 per round, from integer LDS cells and a prefix sum,
//                composite, the canvas and (in a step) its value before every
//                round, which the backward starts from
//   k_loss       L2 against a target: d loss / d canvas and the loss, summed on
//                the device in a fixed order
//   k_backward   the rounds last to first: coverage again, d loss / d alpha
//                per pixel and path, the colours' gradients summed over the
//                tile, and one lane per edge piece gathering its gradient from
//                the columns it touches
//   k_point_grad vertex gradients -> control point gradients
#include <algorithm>
#include <cstring>
#include <vector>

#include "ft_scan.h"

namespace ft {
namespace diff {

constexpr int DSEG = 16;          // segments per cubic
constexpr float EPS_W = 1e-5f;    // narrower pieces use the midpoint value

struct DScene {
    uint32_t n_images, W, H, n_paths;
    uint32_t n_vtx, n_cells;
    const uint32_t *pt_off;     // [n_paths + 1] first point of each path
    const uint32_t *vtx_off;    // [n_paths + 1] first vertex of each path
    const uint32_t *vtx_path;   // [n_vtx]
    const uint32_t *img_first;  // [n_images + 1] first path of each image
    float2 *vtx;                // [n_vtx]
    uint32_t *cell_cnt;         // [n_cells] edges per (path, row); first the differences
    uint32_t *cell_off;         // [n_cells]
    uint32_t *cell_cur;         // [n_cells]
    uint32_t *cell_edge;        // [cap_pairs] local edge index
    uint32_t cap_pairs;
};

// Bernstein weights at t = j / 16: integers over 4096, exact in f32.
__device__ inline void bern(int j, float w[4]) {
    const float u = (float)(DSEG - j), t = (float)j;
    w[0] = u * u * u / 4096.0f;
    w[1] = 3.0f * u * u * t / 4096.0f;
    w[2] = 3.0f * u * t * t / 4096.0f;
    w[3] = t * t * t / 4096.0f;
}

__device__ __forceinline__ float clamp01(float u) { return __builtin_amdgcn_fmed3f(u, 0.0f, 1.0f); }

// The row piece of an edge: its part within row Y, oriented top to bottom.
struct Piece {
    bool live;
    bool down;       // the edge descends from its first to its second vertex
    float sign;      // +1 descending, -1 ascending
    float xa, xb;    // x at the piece's top and bottom
    float h;         // piece height
};

__device__ inline Piece piece_of(float2 p, float2 q, int Y) {
    Piece r;
    r.live = false;
    r.down = q.y > p.y;
    r.sign = r.down ? 1.0f : -1.0f;
    r.xa = r.xb = r.h = 0.0f;
    if (p.y == q.y) return r;
    const float2 t = r.down ? p : q, b = r.down ? q : p;
    const float ya = t.y > (float)Y ? t.y : (float)Y;
    const float yb = b.y < (float)(Y + 1) ? b.y : (float)(Y + 1);
    if (!(yb > ya)) return r;
    const float sl = (b.x - t.x) / (b.y - t.y);
    r.xa = t.x + (ya - t.y) * sl;
    r.xb = t.x + (yb - t.y) * sl;
    r.h = yb - ya;
    r.live = true;
    return r;
}

// Gradients of one piece's sign * h * M, given S1 = sum dA M, Sa = sum dA
// dM/du_a, Sb = sum dA dM/du_b over the pixels of the row (u = X1 - x at the
// piece's top and bottom).  x_a and x_b are linear in the edge's ends, so
// over all the rows between them d/dy of an end is -slope times its d/dx: a
// piece adds the d/dx of both ends, and only the row that holds an end adds
// that end's own d/dy terms.  The slope enters once per edge (vertex_grad).
// That is 2.2 atomics per piece instead of 4.
struct EdgeGrad {
    float xp, xq;  // d/dx of the first and second vertex
    float yp, yq;  // their rows' own d/dy terms
    bool has_p, has_q;
};

__device__ __forceinline__ EdgeGrad piece_grad(float2 p, float2 q, int Y, float S1, float Sa, float Sb) {
    const bool down = q.y > p.y;
    const float2 t = down ? p : q, b = down ? q : p;
    const bool top = t.y > (float)Y, bot = b.y < (float)(Y + 1);  // the ends lie inside the row
    const float ya = top ? t.y : (float)Y, yb = bot ? b.y : (float)(Y + 1);
    const float dy = b.y - t.y, h = yb - ya, idy = 1.0f / dy, hsl = h * ((b.x - t.x) / dy);
    const float fa = (ya - t.y) * idy, fb = (yb - t.y) * idy;  // where the piece lies on the edge
    const float s = down ? 1.0f : -1.0f, sh = -s * h;
    const float xt = sh * fmaf(1.0f - fa, Sa, (1.0f - fb) * Sb), xb = sh * fmaf(fa, Sa, fb * Sb);
    const float yt = -s * fmaf(hsl, Sa, S1), yz = s * fmaf(-hsl, Sb, S1);
    EdgeGrad g;
    g.xp = down ? xt : xb;
    g.xq = down ? xb : xt;
    g.yp = down ? yt : yz;
    g.yq = down ? yz : yt;
    g.has_p = down ? top : bot;
    g.has_q = down ? bot : top;
    return g;
}

// One DPP step of a wavefront float scan: v + (v of the source lane, or 0).
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ float dpp_add(float v) {
    const int src = __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, ROW_MASK, 0xf, false);
    return v + __builtin_bit_cast(float, src);
}

// Sums over the 64 lanes (all active), returned to every lane: inclusive
// scans with DPP (row_shr 1, 2, 4, 8 within rows of 16 lanes, then
// row_bcast:15 and row_bcast:31), read from lane 63.
__device__ inline void wave_sum3(float &a, float &b, float &c) {
#define FT_DPP3(CTRL, RM) a = dpp_add<CTRL, RM>(a); b = dpp_add<CTRL, RM>(b); c = dpp_add<CTRL, RM>(c);
    FT_DPP3(0x111, 0xf)
    FT_DPP3(0x112, 0xf)
    FT_DPP3(0x114, 0xf)
    FT_DPP3(0x118, 0xf)
    FT_DPP3(0x142, 0xa)
    FT_DPP3(0x143, 0xc)
#undef FT_DPP3
    a = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, a), 63));
    b = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, b), 63));
    c = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, c), 63));
}

// ---------------------------------------------------------------------------
// Geometry
// ---------------------------------------------------------------------------
// Vertex v of a path with control points P: the start point, then the points
// t = 1/16 .. 1 of each cubic.
__device__ __forceinline__ float2 path_vertex(const float2 *P, uint32_t v) {
    if (!v) return P[0];
    const uint32_t c = (v - 1) / DSEG;
    float w[4];
    bern((int)((v - 1) % DSEG) + 1, w);
    const float2 p0 = P[3 * c], p1 = P[3 * c + 1], p2 = P[3 * c + 2], p3 = P[3 * c + 3];
    return make_float2(w[0] * p0.x + w[1] * p1.x + w[2] * p2.x + w[3] * p3.x,
                       w[0] * p0.y + w[1] * p1.y + w[2] * p2.y + w[3] * p3.y);
}

__global__ __launch_bounds__(BLOCK) void k_vertices(DScene S, const float2 *points, DevStatus *st) {
    for (uint32_t v = blockIdx.x * BLOCK + threadIdx.x; v < S.n_vtx; v += gridDim.x * BLOCK) {
        const uint32_t k = S.vtx_path[v];
        if (k >= S.n_paths) {
            raise_err(st, FT_EDEVICE);
            continue;
        }
        S.vtx[v] = path_vertex(points + S.pt_off[k], v - S.vtx_off[k]);
    }
}

// Clears a run's look-back words and status.  Needed before the first run and
// after a failed one only: k_forward leaves the words clear for the next
// k_geometry, and a run without errors leaves no error (2 us and a gap per
// call of some 110 us otherwise).
__global__ __launch_bounds__(BLOCK) void k_clear_run(unsigned long long *lb, uint32_t n_lb, DevStatus *st,
                                                     uint32_t *host_err) {
    for (uint32_t i = threadIdx.x; i < n_lb; i += BLOCK) lb[i] = 0;
    status_begin(st, threadIdx.x, host_err);
}

// Rows [r0, r1] an edge overlaps within [0, H); false when none.
__device__ inline bool edge_row_range(float2 a, float2 b, uint32_t H, uint32_t &r0, uint32_t &r1) {
    if (!(a.y != b.y)) return false;  // horizontal, or NaN
    float lo = a.y < b.y ? a.y : b.y, hi = a.y < b.y ? b.y : a.y;
    if (!(hi > 0.0f) || !(lo < (float)H)) return false;
    lo = lo < 0.0f ? 0.0f : lo;
    hi = hi > (float)H ? (float)H : hi;
    const float f0 = floorf(lo), f1 = ceilf(hi) - 1.0f;
    if (f1 < f0) return false;
    r0 = (uint32_t)f0;
    r1 = (uint32_t)f1 < H - 1 ? (uint32_t)f1 : H - 1;
    return r0 <= r1;
}

__device__ inline void edge_at(const DScene &S, uint32_t v, uint32_t &k, float2 &a, float2 &b) {
    k = S.vtx_path[v];
    const uint32_t vb = S.vtx_off[k], V = S.vtx_off[k + 1] - vb, local = v - vb;
    a = S.vtx[v];
    b = S.vtx[local + 1 < V ? v + 1 : vb];
}

// Clears the cell counters, the scans' look-back words, the status and (when
// given) the gradients.
__global__ __launch_bounds__(BLOCK) void k_clear_cells(DScene S, float4 *gedge, float *gcol, unsigned long long *lb,
                                                       uint32_t n_lb, DevStatus *st, uint32_t *host_err) {
    uint32_t n = S.n_cells > S.n_vtx ? S.n_cells : S.n_vtx;
    n = n > 4 * S.n_paths ? n : 4 * S.n_paths;
    n = n > n_lb ? n : n_lb;
    for (uint32_t i = blockIdx.x * BLOCK + threadIdx.x; i < n; i += gridDim.x * BLOCK) {
        if (i < n_lb) lb[i] = 0;
        if (i < S.n_cells) {
            S.cell_cnt[i] = 0;
            S.cell_cur[i] = 0;
        }
        if (gedge && i < S.n_vtx) gedge[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (gcol && i < 4 * S.n_paths) gcol[i] = 0.0f;
    }
    if (blockIdx.x == 0) status_begin(st, threadIdx.x, host_err);
}

__global__ __launch_bounds__(BLOCK) void k_rows(DScene S, DevStatus *st) {
    for (uint32_t v = blockIdx.x * BLOCK + threadIdx.x; v < S.n_vtx; v += gridDim.x * BLOCK) {
        uint32_t k, r0, r1;
        float2 a, b;
        edge_at(S, v, k, a, b);
        if (!edge_row_range(a, b, S.H, r0, r1)) continue;
        // +1 at the first row's cell, -1 at the cell after the last row (the
        // next path's first row when r1 is the last row): the inclusive scan
        // over all cells is then the edge count of every (path, row)
        const uint64_t c = (uint64_t)k * S.H;
        atomicAdd(&S.cell_cnt[c + r0], 1u);
        if (c + r1 + 1 < S.n_cells) atomicAdd(&S.cell_cnt[c + r1 + 1], 0xFFFFFFFFu);
    }
}

// Exclusive scan of x over the block's BLOCK threads, and the total.  Every
// thread calls it; s_w is free again when it returns.
__device__ __forceinline__ uint32_t block_excl(uint32_t x, uint32_t *s_w, uint32_t &total) {
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const uint32_t incl = wave_incl_dpp<false>(x);
    if (lane == 63) s_w[wid] = incl;
    __syncthreads();
    uint32_t pre = incl - x;
    total = 0;
#pragma unroll
    for (int w = 0; w < BLOCK / 64; ++w) {
        pre += w < wid ? s_w[w] : 0u;
        total += s_w[w];
    }
    __syncthreads();
    return pre;
}

// The whole geometry in one launch, for layouts whose paths have at most
// GEOM_EDGES edges: a block takes `per` consecutive paths, writes their
// vertices and counts their (edge, row) pairs, takes its place in the pair
// list by look-back, and then per path and GEOM_ROWS of the rows between its
// first and last counts the rows' edges in LDS, scans them into the cells' list
// offsets and hands out the list slots with LDS cursors; the other rows get
// counts of 0, whose offsets nothing reads.  (Up to a row per thread they cost
// nothing, and the span is not made: 0.8 of 8.3 us for 24 paths of 120 rows.)
// Order within a list is free: coverage is an integer sum.  It also clears the
// gradients (gedge null: none).  It replaces a clear over all cells, a vertex
// pass, atomics per edge on the cells, two scans over all cells and a kernel
// that tested every edge of a path against every row: 545 -> 173 us of a
// 64-image step with 17,500 paths, 85 us in six launches -> 18 us in one for
// 256 paths, 110 -> 16 us for a 1000x600 image of 128 paths.  4,096 figures of
// 24 pixels in an image of 9,000 rows: 63 us, 530 with counts and offsets of
// all rows by this kernel, 290 by the general form, which took images past
// 8,192 rows.  A path's work is a chain of a few barriers, so a launch of few
// paths is bound by latency.
constexpr uint32_t GEOM_EDGES = 2048, GEOM_ROWS = 8192, GEOM_BLOCKS = 1024;
constexpr uint32_t GEOM_SPANS = 64;  // paths of a block whose spans are kept; the others take all rows
constexpr uint32_t EDGE_LANES = 4;  // threads per edge in the fill, on every fourth of its rows

__global__ __launch_bounds__(BLOCK) void k_geometry(DScene S, const float2 *points, float4 *gedge, float *gcol,
                                                    uint32_t per, unsigned long long *lb, DevStatus *st) {
    extern __shared__ uint32_t s_row[];  // [min(H, GEOM_ROWS) + 1]: differences, counts, then list cursors
    __shared__ uint32_t s_w[BLOCK / 64], s_tk;
    __shared__ unsigned long long s_base;
    __shared__ uint32_t s_up[GEOM_SPANS], s_end[GEOM_SPANS];  // a path's rows [H - s_up, s_end)
    const uint32_t tid = threadIdx.x;
    if (tid == 0) s_tk = lookback_ticket(lb);
    if (tid < GEOM_SPANS) s_up[tid] = s_end[tid] = 0;
    __syncthreads();
    const uint32_t b = s_tk;
    const uint32_t k0 = b * per, k1 = k0 + per < S.n_paths ? k0 + per : S.n_paths;
    // vertices, then the pairs of the paths' edges
    for (uint32_t k = k0; k < k1; ++k) {
        const uint32_t vb = S.vtx_off[k], V = S.vtx_off[k + 1] - vb;
        for (uint32_t v = tid; v < V; v += BLOCK) {
            S.vtx[vb + v] = path_vertex(points + S.pt_off[k], v);
            if (gedge) gedge[vb + v] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        }
        if (gcol && tid < 4) gcol[4 * (uint64_t)k + tid] = 0.0f;
    }
    __syncthreads();
    unsigned long long mine = 0;
    for (uint32_t k = k0; k < k1; ++k) {
        const uint32_t vb = S.vtx_off[k], V = S.vtx_off[k + 1] - vb;
        uint32_t up = 0, end = 0;  // rows from the first on; the row after the last
        for (uint32_t e = tid; e < V; e += BLOCK) {
            uint32_t r0, r1;
            if (!edge_row_range(S.vtx[vb + e], S.vtx[vb + (e + 1 < V ? e + 1 : 0u)], S.H, r0, r1)) continue;
            mine += r1 - r0 + 1;
            up = S.H - r0 > up ? S.H - r0 : up;
            end = r1 + 1 > end ? r1 + 1 : end;
        }
        if ((k - k0 < GEOM_SPANS) & (S.H > BLOCK)) {
            up = wave_incl_dpp<true>(up);
            end = wave_incl_dpp<true>(end);
            if ((tid & 63) == 63) {
                atomicMax(&s_up[k - k0], up);
                atomicMax(&s_end[k - k0], end);
            }
        }
    }
    // at most GEOM_EDGES edges of FT_MAX_WIDTH rows per path: one path's pairs fit 32 bits, a block's need not
    const unsigned long long wsum = wave_incl_t<unsigned long long, false>(mine);
    __shared__ unsigned long long s_sum[BLOCK / 64];
    if ((tid & 63) == 63) s_sum[tid >> 6] = wsum;
    __syncthreads();
    if (tid < 64) {
        unsigned long long tot = 0;
#pragma unroll
        for (int w = 0; w < BLOCK / 64; ++w) tot += s_sum[w];
        const unsigned long long pre = lookback_prefix<unsigned long long, false>(lb, b, tot, st);
        if (tid == 0) {
            s_base = pre + tot <= S.cap_pairs ? pre : ~0ull;
            if (k1 == S.n_paths && k0 < S.n_paths) {  // the run's total
                const unsigned long long all = pre + tot;
                st->n_pairs = all < 0xFFFFFFFFull ? (uint32_t)all : 0xFFFFFFFFu;
                if (all > S.cap_pairs) {
                    atomicOr(&st->overflow, 2u);
                    st->need_pairs = all < 0xFFFFFFFFull ? (uint32_t)all : 0xFFFFFFFFu;
                }
            }
        }
    }
    __syncthreads();
    if (s_base == ~0ull) return;  // no room: the run is repeated with more
    uint32_t base = (uint32_t)s_base;
    for (uint32_t k = k0; k < k1; ++k) {
        const uint32_t vb = S.vtx_off[k], V = S.vtx_off[k + 1] - vb;
        // the rows [w0, w0 + h) of an edge, counted from w0
        auto window = [&](uint32_t e, uint32_t w0, uint32_t h, uint32_t &r0, uint32_t &r1) {
            if (!edge_row_range(S.vtx[vb + e], S.vtx[vb + (e + 1 < V ? e + 1 : 0u)], S.H, r0, r1)) return false;
            if ((r0 >= w0 + h) | (r1 < w0)) return false;
            r0 = r0 > w0 ? r0 - w0 : 0u;
            r1 = r1 - w0 < h ? r1 - w0 : h - 1;
            return true;
        };
        const bool kept = (k - k0 < GEOM_SPANS) & (S.H > BLOCK);
        const uint32_t lo = kept ? S.H - s_up[k - k0] : 0u, end = kept ? s_end[k - k0] : S.H;
        for (uint32_t r = tid; r < lo; r += BLOCK) S.cell_cnt[(uint64_t)k * S.H + r] = 0;
        for (uint32_t r = end > lo ? end + tid : S.H; r < S.H; r += BLOCK) S.cell_cnt[(uint64_t)k * S.H + r] = 0;
        for (uint32_t w0 = lo; w0 < end; w0 += GEOM_ROWS) {
            const uint32_t h = end - w0 < GEOM_ROWS ? end - w0 : GEOM_ROWS;
            for (uint32_t r = tid; r <= h; r += BLOCK) s_row[r] = 0;
            __syncthreads();
            for (uint32_t e = tid; e < V; e += BLOCK) {
                uint32_t r0, r1;
                if (!window(e, w0, h, r0, r1)) continue;
                atomicAdd(&s_row[r0], 1u);
                atomicAdd(&s_row[r1 + 1], 0xFFFFFFFFu);
            }
            __syncthreads();
            // thread t's rows [a, z): counts from the differences, then offsets
            const uint32_t rows_per = (h + BLOCK - 1) / BLOCK;
            const uint32_t a = tid * rows_per < h ? tid * rows_per : h;
            const uint32_t z = a + rows_per < h ? a + rows_per : h;
            uint32_t d = 0, total;
            for (uint32_t r = a; r < z; ++r) d += s_row[r];
            uint32_t cnt = block_excl(d, s_w, total);
            const uint32_t before = cnt;
            uint32_t sum = 0;
            for (uint32_t r = a; r < z; ++r) {
                cnt += s_row[r];
                sum += cnt;
            }
            uint32_t at = base + block_excl(sum, s_w, total);
            cnt = before;
            const uint64_t c0 = (uint64_t)k * S.H + w0;
            for (uint32_t r = a; r < z; ++r) {
                cnt += s_row[r];
                S.cell_cnt[c0 + r] = cnt;
                S.cell_off[c0 + r] = at;
                s_row[r] = at;
                at += cnt;
            }
            __syncthreads();
            for (uint32_t i = tid; i < V * EDGE_LANES; i += BLOCK) {
                const uint32_t e = i / EDGE_LANES;
                uint32_t r0, r1;
                if (!window(e, w0, h, r0, r1)) continue;
                for (uint32_t r = r0 + i % EDGE_LANES; r <= r1; r += EDGE_LANES)
                    S.cell_edge[atomicAdd(&s_row[r], 1u)] = e;
            }
            base += total;
            __syncthreads();
        }
    }
}

// The general form, for longer paths: k_vertices, k_rows (differences on the
// cells), two scans over the cells, and k_fill_cells.
//
// FILL_LANES threads per edge, each taking every FILL_LANES-th run of
// FILL_ROWS rows, with the run's FILL_ROWS slot reservations (returning
// atomics on the cells' cursors) in flight together: a tall edge does not
// wait on one atomic per row in turn.
constexpr uint32_t FILL_LANES = 4, FILL_ROWS = 8;

__global__ __launch_bounds__(BLOCK) void k_fill_cells(DScene S, DevStatus *st) {
    if (run_failed(st)) return;
    if (st->n_pairs > S.cap_pairs) {
        if (blockIdx.x == 0 && threadIdx.x == 0) {
            atomicOr(&st->overflow, 2u);
            st->need_pairs = st->n_pairs;
        }
        return;
    }
    const uint64_t n_items = (uint64_t)S.n_vtx * FILL_LANES;
    for (uint64_t t = (uint64_t)blockIdx.x * BLOCK + threadIdx.x; t < n_items; t += (uint64_t)gridDim.x * BLOCK) {
        const uint32_t v = (uint32_t)(t / FILL_LANES), q = (uint32_t)(t % FILL_LANES);
        uint32_t k, r0, r1;
        float2 a, b;
        edge_at(S, v, k, a, b);
        if (!edge_row_range(a, b, S.H, r0, r1)) continue;
        const uint32_t local = v - S.vtx_off[k];
        const uint64_t c0 = (uint64_t)k * S.H;
        for (uint32_t rb = r0 + q * FILL_ROWS; rb <= r1; rb += FILL_LANES * FILL_ROWS) {
            uint32_t at[FILL_ROWS];
#pragma unroll
            for (uint32_t u = 0; u < FILL_ROWS; ++u)
                at[u] = rb + u <= r1 ? S.cell_off[c0 + rb + u] + atomicAdd(&S.cell_cur[c0 + rb + u], 1u) : 0u;
#pragma unroll
            for (uint32_t u = 0; u < FILL_ROWS; ++u) {
                if (rb + u > r1) break;
                if (at[u] < S.cap_pairs)
                    S.cell_edge[at[u]] = local;
                else
                    raise_err(st, FT_EDEVICE);
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Forward, loss, backward
// ---------------------------------------------------------------------------
// ---------------------------------------------------------------------------
// Coverage by cells.  A block owns a tile of blockDim.x pixels (64 to
// TILE_MAX) of one row of one image and takes the image's paths SEG at a
// time.  One thread per row piece adds the piece's coverage *differences* to
// the path's row of LDS cells: only the columns the piece's ramp touches, so
// a piece costs its x extent instead of the tile's width, and a 64-lane
// prefix sum then gives every pixel's coverage.  (Evaluating every piece that
// touches a wavefront's columns on all of its pixels took 3.84 ms for 64
// images of 256x256 with 17,500 paths, most of it on pixels outside the
// ramp; this form takes 1.03 ms, and 74 us instead of 297 for one 512x512
// image of 256 paths.  What is left is VALU work, 95 % of the SIMDs' issue
// rate for the 64 images: per path and pixel about 9 instructions of prefix
// sum and 9 of composite.)
//
// Cells are integers in units of 2^-26 (an i32 add): the sum does not depend
// on the order of the pieces, so the same inputs give the same canvas
// whichever kernel computes it, and a column of n pieces is within n 2^-27 of
// its products' sum.  i32 holds |A| < 32; a (path, row) with more than HEAVY
// pieces takes 64-bit cells of 2^-38.
//
// A pixel has a gradient only where its coverage is not 0, so a column that a
// ramp touches by less than 2^-27 would lose it (the tip of a figure that
// reaches 1e-4 into a pixel has a gradient of 1e-4 there).  What rounding took
// from a ramp column of a share under TINY is therefore listed, and added to
// the column's coverage.  A path with a piece less than TINY high, or with
// more such columns than the list has room for, takes 64-bit cells of 2^-56.
// (At cells of 2^-24 for all, without this, gradients of a 512x512 scene were
// 8.2e-6 from FP64 instead of 4.4e-6.  With 64-bit cells for all those paths,
// one round in 30, a forward of 24 paths in 200x120 took 1.4 us
// longer: its slowest row decides.)
//
// Every 64-column chunk of a row stands alone: a piece left of a chunk adds
// its whole signed height to the chunk's first cell, so no carry passes
// between wavefronts.
// ---------------------------------------------------------------------------
constexpr uint32_t SEG = 16;         // paths per round
// Pixels per block.  k_forward is held to the VGPRs with which a SIMD takes 5
// wavefronts, and blocks of 4 wavefronts fill them where blocks of 8 leave one
// empty: an earlier form took 229 us for a 1000x600 image with 256, 250 with
// 512, 233 with 128.
constexpr uint32_t TILE_MAX = 256;
constexpr uint32_t ROW_PATHS = 256;  // paths whose cell counts are staged at once
constexpr uint32_t HEAVY = 31;       // pieces of one path in one row past which cells are 64-bit
constexpr int RAMP_LANE = 8;         // ramps of at most this many columns are walked by one lane
constexpr float CELL_ONE = 0x1p26f;
constexpr float HEAVY_ONE = 0x1p38f;     // at most 2^24 pieces: |A| < 2^24
constexpr float FINE_ONE = 0x1p56f;      // at most HEAVY pieces: |A| < 32
constexpr float TINY = 0x1p4f;           // of CELL_ONE: a share of 2^-22
constexpr uint32_t FIX_MAX = 32;         // listed columns per round

// The paths of a staging round that have pieces in the row, in path order:
// only they are rounded up to SEG and walked.  (A path without pieces leaves
// the row's canvas as it is.  With all paths walked, a scene of small figures
// paid for every figure in every row: 1,024 of 24 pixels in 512x512 took 271
// us a forward and 790 a step, now 71 and 143; 256 paths across the image 113
// and 349, now 102 and 326.)
struct RowLds {
    __align__(16) uint32_t pb[ROW_PATHS + 4];  // exclusive scan of their piece counts; the total to the last round's end
    __align__(16) uint8_t path[ROW_PATHS];     // their index among the staged paths; 0 to the last round's end
    uint32_t dl[ROW_PATHS];                    // list position of a path's piece e: dl + e
    uint2 vtx[ROW_PATHS];                      // first vertex and number of vertices
    uint32_t heavy[ROW_PATHS / SEG];           // per round: bit j, its path j has more than HEAVY pieces
    // per round parity: x: bit j, path j has a piece that is no number here,
    // bit 16 + j, it takes 64-bit cells; y: listed columns
    __align__(8) uint2 mark[2];
    uint2 fix[FIX_MAX];                        // path << 16 | column; the share rounding took, in cell units
    uint32_t n;                                // how many
};

// Row Y of the n <= ROW_PATHS paths from global path kbase.  Every thread
// calls it, between barriers of the caller.
__device__ void stage_row(const DScene &S, uint32_t kbase, uint32_t n, int Y, RowLds &R) {
    const uint32_t lane = threadIdx.x;
    if (lane >= 64) return;
    constexpr uint32_t PER = ROW_PATHS / 64;
    uint32_t c[PER], o[PER];
    uint2 v[PER];
#pragma unroll
    for (uint32_t i = 0; i < PER; ++i) {
        if (64 * i >= n) break;  // (uniform)
        const uint32_t p = 64 * i + lane, k = kbase + (p < n ? p : 0u);
        const uint64_t cell = (uint64_t)k * S.H + (uint32_t)Y;
        c[i] = S.cell_cnt[cell];
        v[i] = make_uint2(S.vtx_off[k], S.vtx_off[k + 1]);
        c[i] = p < n ? c[i] : 0u;
        // (of many paths most have none here, and their offsets are not loaded:
        // 1,118 -> 415 us in a scene of small figures; with few paths the loads
        // are cheap and a second round trip is not)
        o[i] = 0;
        if (n <= 64 || c[i]) o[i] = S.cell_off[cell];
    }
    if (lane < ROW_PATHS / SEG) R.heavy[lane] = 0;
    if (lane < 2) R.mark[lane] = make_uint2(0u, 0u);
    uint32_t first = 0, rank = 0;  // pieces and paths before
#pragma unroll
    for (uint32_t i = 0; i < PER; ++i) {
        if (64 * i >= n) break;
        const unsigned long long live = __ballot(c[i] != 0u);
        const uint32_t incl = wave_incl_dpp<false>(c[i]), pre = first + incl - c[i];
        if (c[i]) {
            const uint32_t r = rank + __builtin_amdgcn_mbcnt_hi((uint32_t)(live >> 32),
                                                                __builtin_amdgcn_mbcnt_lo((uint32_t)live, 0u));
            R.pb[r] = pre;
            R.path[r] = (uint8_t)(64 * i + lane);
            R.dl[r] = o[i] - pre;
            R.vtx[r] = make_uint2(v[i].x, v[i].y - v[i].x);
            if (c[i] > HEAVY) atomicOr(&R.heavy[r / SEG], 1u << (r % SEG));
        }
        first += (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
        rank += (uint32_t)__popcll(live);
    }
    // the rest of the last round
    if (lane <= SEG && rank + lane <= ROW_PATHS) {
        R.pb[rank + lane] = first;
        if (rank + lane < ROW_PATHS) R.path[rank + lane] = 0;
    }
    if (lane == 0) R.n = rank;
}

// Piece e of round s (staged paths [s * SEG, s * SEG + SEG)).
struct PieceRef {
    uint32_t j;     // path within the round, NO_IDX: none
    uint32_t edge;  // the path's edge
};

__device__ __forceinline__ PieceRef piece_ref(const DScene &S, const RowLds &R, uint32_t s, uint32_t e) {
    const uint32_t end = R.pb[(s + 1) * SEG];
    PieceRef r;
    r.j = NO_IDX;
    r.edge = 0;
    if (e >= end) return r;
    uint32_t j = 0;  // the last path of the round that starts at or before e
#pragma unroll
    for (uint32_t i = 0; i < SEG; i += 4) {
        const uint4 q = *reinterpret_cast<const uint4 *>(&R.pb[s * SEG + i]);
        j += (q.x <= e ? 1u : 0u) + (q.y <= e ? 1u : 0u) + (q.z <= e ? 1u : 0u) + (q.w <= e ? 1u : 0u);
    }
    r.j = j - 1;
    r.edge = S.cell_edge[R.dl[s * SEG + r.j] + e];
    return r;
}

// The two vertices of a piece's edge.
struct PieceVtx {
    float2 p, q;
    uint32_t ip;  // index of the first
};

__device__ __forceinline__ PieceVtx piece_vtx(const DScene &S, const RowLds &R, uint32_t s, const PieceRef &r,
                                              uint32_t &bad) {
    const uint32_t t = s * SEG + (r.j != NO_IDX ? r.j : 0u);
    const uint32_t vb = R.vtx[t].x, V = R.vtx[t].y;
    bad |= r.edge < V ? 0u : 1u;
    const uint32_t e = r.edge < V ? r.edge : 0u;
    PieceVtx v;
    v.ip = vb + e;
    v.p = S.vtx[v.ip];
    v.q = S.vtx[vb + (e + 1 < V ? e + 1 : 0u)];
    return v;
}

// A piece against the tile: its coverage M is 0 left of its ramp, 1 right of
// it.  [c0, c1) are the ramp's columns within the tile (c1 <= c0: none), and
// from column max(c0, c1) on the piece counts whole.
struct Ramp {
    float lo, hi, w, inv, z;  // x range, its width, 1 / w (0: narrow, the midpoint's value), signed height
    int c0, c1;
    bool live, nan;
};

__device__ __forceinline__ Ramp ramp_of(const Piece &r, float xb0, int tw) {
    Ramp m;
    m.lo = r.xa < r.xb ? r.xa : r.xb;
    m.hi = r.xa < r.xb ? r.xb : r.xa;
    m.z = r.sign * r.h;
    m.w = m.hi - m.lo;
    m.nan = r.live & !(m.w < __builtin_inff());  // a NaN or unbounded x
    m.live = r.live & !m.nan & (m.lo < xb0 + (float)tw);
    m.inv = m.w < EPS_W ? 0.0f : 1.0f / m.w;
    const float f0 = floorf(m.lo) - xb0, f1 = ceilf(m.hi) - xb0;
    m.c0 = f0 > 0.0f ? (f0 < (float)tw ? (int)f0 : tw) : 0;
    m.c1 = f1 > 0.0f ? (f1 < (float)tw ? (int)f1 : tw) : 0;
    return m;
}

// M at the pixel whose right border is X1, within the ramp: the mean of
// clamp(u, 0, 1) for u from X1 - hi to X1 - lo; a and b are the clamped ends,
// `in` the ramp's length within the pixel and `past` that left of it.  Both
// come from the x's and not from the u's: in column 0, where x is finer than
// 1 - x, the u's difference over the ramp's width is off by 2^-24 / w.
// The quotient is the correctly rounded one (a product with 1 / w corrected
// by its remainder): M close to 0 or 1 decides whether a pixel has a
// gradient.
__device__ __forceinline__ float ramp_mean(const Ramp &m, float X1, float &a, float &b, float &in, float &past) {
    const float lo = X1 - m.hi, hi = X1 - m.lo, X0 = X1 - 1.0f;
    a = clamp01(lo);
    b = clamp01(hi);
    in = fminf(m.hi, X1) - fmaxf(m.lo, X0);
    past = fmaxf(X0 - m.lo, 0.0f);
    if (m.inv == 0.0f) return clamp01((lo + hi) * 0.5f);
    const float I = in * (a + b) * 0.5f + past;
    const float q = I * m.inv;
    return fmaf(fmaf(-q, m.w, I), m.inv, q);
}
__device__ __forceinline__ float ramp_cover(const Ramp &m, float X1) {
    float a, b, in, past;
    return ramp_mean(m, X1, a, b, in, past);
}

// v rounded to a whole number: a share in cell units, |v| at most a cell's
// one (64-bit cells: 2^56, in two exact halves, the conversion of the whole
// being twice as long).
template <typename T>
__device__ __forceinline__ T cell_of(float v) {
    if constexpr (sizeof(T) == 8) {
        const float h = rintf(v * 0x1p-28f);
        return (T)(int)h * ((T)1 << 28) + __float2int_rn(fmaf(-h, 0x1p28f, v));
    } else {
        return __float2int_rn(v);
    }
}
template <typename T>
__device__ __forceinline__ void cell_add(T *c, T v) {
    if constexpr (sizeof(T) == 8)
        atomicAdd(reinterpret_cast<unsigned long long *>(c), (unsigned long long)v);
    else
        atomicAdd(c, v);
}

// Adds one piece per lane to row_at of the cells (the wavefront's lanes all
// call it, those without a piece with m.live false), in units of 1 / one.  A
// ramp of more than RAMP_LANE columns is evaluated by the whole wavefront, one
// column per lane, so that one long near-horizontal piece does not hold up 63
// lanes.  fix(c, r): column c lost r to rounding (32-bit cells, TINY shares:
// the shares of a ramp rise with its columns, so those are its first ones).
template <typename T, class Fix>
__device__ __forceinline__ void scatter_piece(T *cells, uint32_t row_at, const Ramp &m, float xb0, int tw, float one,
                                              Fix &&fix) {
    constexpr bool FIX = sizeof(T) == 4;
    const float zs = m.z * one;
    const int n = m.c1 - m.c0;
    const bool wide = m.live & (n > RAMP_LANE);
    T prev = 0;
    float least = TINY;
    if (m.live & !wide) {
        for (int c = m.c0; c < m.c1; ++c) {
            const float v = zs * ramp_cover(m, xb0 + (float)(c + 1));
            const T q = cell_of<T>(v);
            if (FIX) least = fminf(least, fabsf(v));
            cell_add(&cells[row_at + c], q - ((c & 63) ? prev : (T)0));
            prev = q;
        }
    }
    unsigned long long todo = __ballot(wide);
    while (todo) {
        const int l = __ffsll((long long)todo) - 1;
        todo &= todo - 1;
        auto bc = [l](float v) {
            return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), l));
        };
        Ramp w;
        w.lo = bc(m.lo);
        w.hi = bc(m.hi);
        w.w = w.hi - w.lo;
        w.inv = bc(m.inv);
        const float wz = bc(zs);
        const int w0 = __builtin_amdgcn_readlane(m.c0, l), w1 = __builtin_amdgcn_readlane(m.c1, l);
        const uint32_t at = (uint32_t)__builtin_amdgcn_readlane((int)row_at, l);
        const int lane = threadIdx.x & 63;
        for (int c = w0 + lane; c < w1; c += 64) {
            const T q = cell_of<T>(wz * ramp_cover(w, xb0 + (float)(c + 1)));
            const T b = ((c > w0) & ((c & 63) != 0)) ? cell_of<T>(wz * ramp_cover(w, xb0 + (float)c)) : (T)0;
            cell_add(&cells[at + c], q - b);
        }
    }
    if (!m.live) return;
    if (wide) {
        prev = cell_of<T>(zs * ramp_cover(m, xb0 + (float)m.c1));  // the last ramp column's value
        if (FIX) least = fabsf(zs * ramp_cover(m, xb0 + (float)(m.c0 + 1)));
    }
    // from the column after the ramp on: whole
    const T whole = cell_of<T>(zs);
    const int t = m.c1 > m.c0 ? m.c1 : m.c0;
    if (t < tw) cell_add(&cells[row_at + t], whole - ((t & 63) ? prev : (T)0));
    for (int c = (t | 63) + 1; c < tw; c += 64) cell_add(&cells[row_at + c], whole);
    if (FIX && least < TINY) {
        for (int c = m.c0; c < m.c1; ++c) {
            const float v = zs * ramp_cover(m, xb0 + (float)(c + 1));
            if (!(fabsf(v) < TINY)) break;
            if (v != 0.0f) fix(c, v - rintf(v));
        }
    }
}

// Coverage A[j] of round s's paths at this thread's pixel, from the first
// blockDim.x pieces (ref, first: one per thread, loaded by the caller ahead of
// time) and any further ones.  cells: SEG rows of pitch `pitch`, zero on
// entry; with ZERO zero again on exit, behind a barrier, else the caller's to
// use: each thread has read its own column.  Every thread calls it.
template <bool ZERO, uint32_t TW>
__device__ __forceinline__ void round_cover(const DScene &S, RowLds &R, uint32_t s, const PieceRef &ref,
                                            const Piece &first, int Y, float xb0, int *cells,
                                            float A[SEG], uint32_t &bad) {
    const int tid = threadIdx.x, tw = TW ? (int)TW : (int)blockDim.x;
    const uint32_t pitch = (uint32_t)tw + 1;
    const uint32_t base = R.pb[s * SEG], end = R.pb[(s + 1) * SEG];
    const uint32_t heavy = R.heavy[s];
    for (uint32_t eb = base; eb < end; eb += (uint32_t)tw) {
        if (eb + ((uint32_t)tid & ~63u) >= end) break;  // no piece for this wavefront
        PieceRef r = ref;
        Piece pc = first;
        if (eb != base) {
            r = piece_ref(S, R, s, eb + (uint32_t)tid);
            const PieceVtx u = piece_vtx(S, R, s, r, bad);
            pc = piece_of(u.p, u.q, Y);
        }
        pc.live &= r.j != NO_IDX;
        const uint32_t j = r.j != NO_IDX ? r.j : 0u;
        pc.live &= ((heavy >> j) & 1u) == 0u;
        const Ramp m = ramp_of(pc, xb0, tw);
        const bool low = m.live & (fabsf(m.z) < TINY / CELL_ONE);
        if (m.nan | low) atomicOr(&R.mark[s & 1].x, (m.nan ? 1u : 0x10000u) << j);
        scatter_piece<int>(cells, j * pitch, m, xb0, tw, CELL_ONE, [&](int c, float r) {
            const uint32_t k = atomicAdd(&R.mark[s & 1].y, 1u);
            if (k < FIX_MAX)
                R.fix[k] = make_uint2(j << 16 | (uint32_t)c, __builtin_bit_cast(uint32_t, r));
            else
                atomicOr(&R.mark[s & 1].x, 0x10000u << j);
        });
    }
    __syncthreads();
    const uint2 mark = R.mark[s & 1];
    uint32_t c[SEG];
#pragma unroll
    for (uint32_t j = 0; j < SEG; ++j) {
        c[j] = (uint32_t)cells[j * pitch + tid];
        if (ZERO) cells[j * pitch + tid] = 0;
    }
#pragma unroll
    for (uint32_t j = 0; j < SEG; ++j) A[j] = (float)(int)wave_incl_dpp<false>(c[j]) * (1.0f / CELL_ONE);
    if (mark.x | mark.y | heavy) {  // (uniform)
        const uint32_t n_fix = mark.y < FIX_MAX ? mark.y : FIX_MAX;
        for (uint32_t k = 0; k < n_fix; ++k) {
            const uint2 f = R.fix[k];
            const float r = (f.x & 0xFFFFu) == (uint32_t)tid ? __builtin_bit_cast(float, f.y) : 0.0f;
            const uint32_t path = (uint32_t)__builtin_amdgcn_readfirstlane((int)(f.x >> 16));
#pragma unroll
            for (uint32_t j = 0; j < SEG; ++j) A[j] = j == path ? fmaf(r, 1.0f / CELL_ONE, A[j]) : A[j];
        }
        const uint32_t wide = heavy | (mark.x >> 16);
        uint32_t poison = mark.x;
        if (wide) {  // one path at a time, in 64-bit cells over the same LDS
            long long *c64 = reinterpret_cast<long long *>(cells);
            for (uint32_t j = 0; j < SEG; ++j) {
                if (!((wide >> j) & 1u)) continue;
                const bool many = ((heavy >> j) & 1u) != 0;
                const float one = many ? HEAVY_ONE : FINE_ONE;
                __syncthreads();  // the cells, or the path before's, are read
                c64[tid] = 0;
                __syncthreads();
                const uint32_t e0 = R.pb[s * SEG + j], e1 = R.pb[s * SEG + j + 1];
                for (uint32_t eb = e0; eb < e1; eb += (uint32_t)tw) {  // whole blocks: scatter_piece is collective
                    const uint32_t e = eb + (uint32_t)tid;
                    PieceRef r = piece_ref(S, R, s, e < e1 ? e : NO_IDX);
                    const PieceVtx u = piece_vtx(S, R, s, r, bad);
                    Piece pc = piece_of(u.p, u.q, Y);
                    pc.live &= r.j != NO_IDX;
                    const Ramp m = ramp_of(pc, xb0, tw);
                    if (m.nan) atomicOr(&R.mark[s & 1].x, 1u << j);
                    scatter_piece<long long>(c64, 0u, m, xb0, tw, one, [](int, float) {});
                }
                __syncthreads();
                const long long sum = (long long)wave_incl_t<unsigned long long, false>((unsigned long long)c64[tid]);
                const float a = (float)sum * (many ? 1.0f / HEAVY_ONE : 1.0f / FINE_ONE);
#pragma unroll
                for (uint32_t k = 0; k < SEG; ++k) A[k] = k == j ? a : A[k];
            }
            __syncthreads();
            if (ZERO) c64[tid] = 0;
            poison = R.mark[s & 1].x;
        }
        // a piece without an x takes its path's whole row (coverage past 1, and so no gradient)
#pragma unroll
        for (uint32_t j = 0; j < SEG; ++j) A[j] = ((poison >> j) & 1u) ? 2.0f : A[j];
    }
    if (tid == 0) R.mark[(s + 1) & 1] = make_uint2(0u, 0u);
    if (ZERO) __syncthreads();
}

__device__ __forceinline__ float alpha_cover(float A) { return __builtin_amdgcn_fmed3f(fabsf(A), 0.0f, 1.0f); }

// The paths of round s: their number, and their index among the staged paths
// (path j's: byte j), uniform.
struct RoundPaths {
    uint32_t n, w[SEG / 4];
    __device__ __forceinline__ uint32_t at(uint32_t j) const { return (w[j / 4] >> (8 * (j % 4))) & 0xFFu; }
};
__device__ __forceinline__ RoundPaths round_paths(const RowLds &R, uint32_t s, uint32_t n_live) {
    static_assert(SEG == 16, "one 16-byte read");
    const uint4 q = *reinterpret_cast<const uint4 *>(&R.path[s * SEG]);
    RoundPaths r;
    r.n = n_live - s * SEG < SEG ? n_live - s * SEG : SEG;
    r.w[0] = (uint32_t)__builtin_amdgcn_readfirstlane((int)q.x);
    r.w[1] = (uint32_t)__builtin_amdgcn_readfirstlane((int)q.y);
    r.w[2] = (uint32_t)__builtin_amdgcn_readfirstlane((int)q.z);
    r.w[3] = (uint32_t)__builtin_amdgcn_readfirstlane((int)q.w);
    return r;
}

// Colour of the round's path j, or zero past its last one (staged: the
// colours of the staged paths).  Uniform: scalar loads, and no branch between
// a round's paths.
__device__ __forceinline__ float4 round_colour(const float4 *__restrict__ staged, const RoundPaths &rp, uint32_t j) {
    const float4 c = staged[rp.at(j)];
    const uint32_t m = j < rp.n ? 0xFFFFFFFFu : 0u;
    auto sel = [m](float v) { return __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, v) & m); };
    return make_float4(sel(c.x), sel(c.y), sel(c.z), sel(c.w));
}

// A kernel's start: the image's first path and number of paths, and false when
// an earlier kernel of the run failed, in one round trip to memory.
__device__ __forceinline__ bool image_begin(const DScene &S, const DevStatus *st, uint32_t im, uint32_t &k0,
                                            uint32_t &np) {
    const uint32_t e = st->err, o = st->overflow, k1 = S.img_first[im + 1];
    k0 = S.img_first[im];
    np = k1 - k0;
    asm volatile("" ::"s"(e), "s"(o), "s"(k0), "s"(k1));
    return (e | o) == 0u;
}

// The canvas of one tile of one row: the image's paths with pieces there
// composited over transparent pixels, SEG at a time, with the next round's
// pieces loaded while a round is composited.  With ck it also leaves the
// canvas before every round but the image's first, as checkpoint (staged
// paths before it) / SEG + round, at slot (image row) * ck_pitch + X; canvas
// may be null.  One block also clears the n_lb look-back words of the geometry
// (done by now) for the next run and, with `report`, reports the status.
//
// TW: the tile's width where it is TILE_MAX (any wider than 192 pixels), else
// 0 and the block's.  As a constant it makes the LDS rows' addresses offsets of
// one register instead of sixteen (when it came in 1.17 -> 1.13 ms for 64
// images of 256x256, 86 -> 83 us for 512x512; k_backward 3.57 -> 3.19 ms).
template <uint32_t TW>
__global__ __launch_bounds__(TILE_MAX, 5) void k_forward(DScene S, const float4 *__restrict__ colours,
                                                      float4 *__restrict__ canvas, float4 *__restrict__ ck,
                                                      uint32_t ck_pitch, uint64_t ck_stride, DevStatus *st,
                                                      unsigned long long *__restrict__ lb, uint32_t n_lb,
                                                      HostStatus *__restrict__ report) {
    extern __shared__ __align__(16) int s_cells[];
    __shared__ RowLds R;
    if ((blockIdx.x | blockIdx.y | blockIdx.z) == 0) {
        if (report) report_status(report, st, nullptr, nullptr, 0);
        for (uint32_t i = threadIdx.x; i < n_lb; i += blockDim.x) lb[i] = 0;
    }
    const uint32_t tw = TW ? TW : blockDim.x, pitch = tw + 1;
    const uint32_t X = blockIdx.x * tw + threadIdx.x, Y = blockIdx.y, im = blockIdx.z;
    uint32_t k0, np;
    if (!image_begin(S, st, im, k0, np)) return;
    const float xb0 = (float)(blockIdx.x * tw);
    const uint64_t slot = ((uint64_t)im * S.H + Y) * ck_pitch + X;
    const bool in = X < S.W;
    uint32_t bad = 0;
    float4 C = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    for (uint32_t i = threadIdx.x; i < SEG * pitch; i += tw) s_cells[i] = 0;
    for (uint32_t ja = 0; ja < np; ja += ROW_PATHS) {
        const uint32_t n = np - ja < ROW_PATHS ? np - ja : ROW_PATHS;
        __syncthreads();  // the previous paths' staging is no longer read
        stage_row(S, k0 + ja, n, (int)Y, R);
        __syncthreads();
        const uint32_t n_live = (uint32_t)__builtin_amdgcn_readfirstlane((int)R.n), rounds = (n_live + SEG - 1) / SEG;
        if (!rounds) continue;
        const float4 *const staged = colours + k0 + ja;
        PieceRef ref = piece_ref(S, R, 0, R.pb[0] + threadIdx.x);
        PieceVtx v = piece_vtx(S, R, 0, ref, bad);
        PieceRef nref = ref;
        if (rounds > 1) nref = piece_ref(S, R, 1, R.pb[SEG] + threadIdx.x);
        for (uint32_t s = 0; s < rounds; ++s) {
            const PieceRef cur = ref;
            const Piece first = piece_of(v.p, v.q, (int)Y);
            if (s + 1 < rounds) {  // the next round's vertices, and the one after's edge
                ref = nref;
                v = piece_vtx(S, R, s + 1, ref, bad);
                if (s + 2 < rounds) nref = piece_ref(S, R, s + 2, R.pb[(s + 2) * SEG] + threadIdx.x);
            }
            const RoundPaths rp = round_paths(R, s, n_live);
            float A[SEG];
            round_cover<true, TW>(S, R, s, cur, first, (int)Y, xb0, s_cells, A, bad);
            const uint32_t j0 = ja + s * SEG;
            if (ck && j0 && in) ck[(uint64_t)(j0 / SEG) * ck_stride + slot] = C;
#pragma unroll
            for (uint32_t j = 0; j < SEG; ++j) {
                const float4 c = round_colour(staged, rp, j);
                const float al = alpha_cover(A[j]), keep = fmaf(-c.w, al, 1.0f);
                C = make_float4(fmaf(C.x, keep, c.x * al), fmaf(C.y, keep, c.y * al), fmaf(C.z, keep, c.z * al),
                                fmaf(C.w, keep, c.w * al));
            }
        }
    }
    if (bad) raise_err(st, FT_EDEVICE);
    if (canvas && in) canvas[((uint64_t)im * S.H + Y) * S.W + X] = C;
}

// The loss, and grad = 2 (C - T) / N: a sum of squared differences per block,
// and their sum in a fixed order by the block that finishes last, so that a
// step and a separate ft_diff_loss of the same canvas give the same value.
// VEC floats per load (4 where every pointer is aligned for it).  LOSS_GRID
// blocks, one per CU with LOSS_UNROLL loads of each kind in flight: their adds
// to the one counter go by quickly.  (1,024 blocks of single floats and a
// second kernel for the sum: 5.1 + 5.2 us for 512x512, 55 + 5 for 64 images of
// 256x256; now 7.5 and 46.)
constexpr uint32_t LOSS_GRID = 256;
constexpr int LOSS_UNROLL = 4;
template <int VEC>
__global__ __launch_bounds__(BLOCK) void k_loss(const float *canvas, const float *target, float *grad, uint64_t n,
                                                unsigned long long *partial, uint32_t *done, double *loss) {
    __shared__ double s_w[BLOCK / 64];
    __shared__ uint32_t s_last;
    struct __align__(4 * VEC) Vec {
        float v[VEC];
    };
    const Vec *const vc = reinterpret_cast<const Vec *>(canvas), *const vt = reinterpret_cast<const Vec *>(target);
    Vec *const vg = reinterpret_cast<Vec *>(grad);
    const uint64_t nv = n / VEC, stride = (uint64_t)LOSS_GRID * BLOCK;  // (n is a multiple of 4)
    double acc = 0.0;
    const float scale = (float)(2.0 / (double)n);
    for (uint64_t i = (uint64_t)blockIdx.x * BLOCK + threadIdx.x; i < nv; i += LOSS_UNROLL * stride) {
        Vec c[LOSS_UNROLL], t[LOSS_UNROLL];
#pragma unroll
        for (int u = 0; u < LOSS_UNROLL; ++u) {
            const uint64_t k = i + u * stride;
            if (k < nv) {
                c[u] = vc[k];
                t[u] = vt[k];
            }
        }
#pragma unroll
        for (int u = 0; u < LOSS_UNROLL; ++u) {
            const uint64_t k = i + u * stride;
            if (k >= nv) continue;
            Vec g;
#pragma unroll
            for (int x = 0; x < VEC; ++x) {
                const float r = c[u].v[x] - t[u].v[x];
                acc += (double)r * (double)r;
                g.v[x] = scale * r;
            }
            if (grad) vg[k] = g;
        }
    }
    auto block_sum = [&](double v) {  // (thread 0's)
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
        if ((threadIdx.x & 63) == 0) s_w[threadIdx.x >> 6] = v;
        __syncthreads();
        double t = 0.0;
        for (int w = 0; w < BLOCK / 64; ++w) t += s_w[w];
        return t;
    };
    const double mine = block_sum(acc);
    if (threadIdx.x == 0) {
        __hip_atomic_store(&partial[blockIdx.x], __builtin_bit_cast(unsigned long long, mine), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        s_last = atomicAdd(done, 1u) == LOSS_GRID - 1 ? 1u : 0u;
    }
    __syncthreads();
    if (!s_last) return;
    static_assert(LOSS_GRID == BLOCK, "one partial per thread");
    const unsigned long long p = __hip_atomic_load(&partial[threadIdx.x], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const double all = block_sum(__builtin_bit_cast(double, p));
    if (threadIdx.x == 0) {
        *loss = all;
        *done = 0;  // for the next run
    }
}

// Sums of 64 values over the wavefront's lanes at once, as a tree that
// halves the number of registers at each level instead of reducing every
// value on its own (141 instructions for 64 values; 6 DPP adds each would be
// 384).  sum2 takes two values: lanes below 32 of the result hold a's sums
// over lane pairs (l, l + 32), the others b's; sum_rows does the same over
// row pairs of 16 lanes, and sum_dpp within a row, where the DPP pattern
// CTRL mirrors the lanes and `hi` is the lane bit that decides.
__device__ __forceinline__ float sum2(float a, float b) {
    const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b),
                                                    false, false);
    return __builtin_bit_cast(float, (uint32_t)r[0]) + __builtin_bit_cast(float, (uint32_t)r[1]);
}
__device__ __forceinline__ float sum_rows(float a, float b) {
    const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b),
                                                    false, false);
    return __builtin_bit_cast(float, (uint32_t)r[0]) + __builtin_bit_cast(float, (uint32_t)r[1]);
}
template <int CTRL>
__device__ __forceinline__ float sum_dpp(float a, float b, bool hi) {
    const float give = hi ? a : b;
    const int got = __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, give), CTRL, 0xf, 0xf, true);
    return (hi ? b : a) + __builtin_bit_cast(float, got);
}

// Suffix sums within rows of 16 lanes (row_shl 1, 2, 4, 8): lane i's is the
// sum of lanes i .. i | 15.
__device__ __forceinline__ float row_suffix(float v) {
    v = dpp_add<0x101, 0xf>(v);
    v = dpp_add<0x102, 0xf>(v);
    v = dpp_add<0x104, 0xf>(v);
    return dpp_add<0x108, 0xf>(v);
}

// The sum of dA over the columns [t, 64) of a chunk from its 64 row suffixes.
// Only columns at or right of t are added, so a sum whose terms are zero is
// zero and a large (or unbounded) dA left of t does not touch it: as the
// difference of two prefix sums of the chunk it kept their rounding.
__device__ __forceinline__ float chunk_right(const float *suf, int t) {
    const float r1 = suf[16], r2 = suf[32], r3 = suf[48];
    return ((suf[t] + (t < 16 ? r1 : 0.0f)) + (t < 32 ? r2 : 0.0f)) + (t < 48 ? r3 : 0.0f);
}

// A piece's S1 = sum dA M, S2 = sum dA dM/dx_lo, S3 = sum dA dM/dx_hi terms
// of one column (dA: the pixel's d loss / d coverage; the partials are with
// respect to u = X1 - x, so S2 goes with the larger x).  The partials are
// (M - a) / w and (b - M) / w; written out, with w = in + past + the length
// right of the pixel, they are sums of positive terms: M - a would keep M's
// rounding, which 1 / w multiplies.
__device__ __forceinline__ void ramp_grad(const Ramp &m, float X1, float g, float &S1, float &S2, float &S3) {
    float a, b, in, past;
    const float M = ramp_mean(m, X1, a, b, in, past);
    S1 = fmaf(g, M, S1);
    if (m.inv == 0.0f) {  // narrow: half of the slope each
        const float half = ((M > 0.0f) & (M < 1.0f)) ? 0.5f : 0.0f;
        S2 += g * half;
        S3 += g * half;
        return;
    }
    const float r = in * m.inv, even = 0.5f * r * r, g2 = g * m.inv * m.inv;
    S2 = fmaf(g2, past * (1.0f - a), fmaf(g, even, S2));
    S3 = fmaf(g2, fmaxf(m.hi - X1, 0.0f) * b, fmaf(g, even, S3));
}

// One tile of one row, the image's rounds of SEG paths last to first.  With f
// the pixel's d loss / d canvas, everything the paths' gradients need of the
// canvas is the scalar q_j = f . (canvas under path j), and of the paths above
// the scalar T_j, the product of their 1 - alpha (the same for every channel):
//     d loss / d alpha_j  = T_j (f . c_j - c_j.w q_j)
//     d loss / d c_j      = sum over pixels of T_j alpha_j (f.x, f.y, f.z, f.w - q_j)
// q starts from the round's checkpoint (k_forward's) and runs forward over
// the round; T runs backward.  So a path costs a pixel about 20 operations
// beside its coverage, where re-compositing four channels cost twice that.
//
// The paths' dA and its suffix sums per 16 columns go to LDS, and one thread
// per piece gathers its sums: the ramp's columns one by one, and all columns
// right of it from the suffix sums (chunk_right).  (Evaluating each piece on all 64
// pixels of every wavefront it touches and reducing the three sums over the
// wavefront took 18.4 ms for 64 images of 256x256 with 17,500 paths; this
// form takes 2.86 ms, and 205-231 us instead of 869 for one 512x512 image of
// 256 paths (where its buffers come to lie decides between the two, for a
// reason not found).  Adding four vertex gradients per piece instead of
// EdgeGrad's two and its ends took 4.5 ms and 332 us.)  What bounds it is VALU issue (79 % of the SIMDs' rate for
// the 64 images, 50-56 % for the one, whose 1,024 blocks are one pass of the
// chip) and the waits on LDS and barriers.  Four wavefronts per SIMD are asked
// for: with three blocks per CU those 1,024 run in two passes (370 us).
template <uint32_t TW>
__global__ __launch_bounds__(TILE_MAX, 4) void k_backward(DScene S, const float4 *__restrict__ colours,
                                                       const float4 *__restrict__ grad_canvas,
                                                       const float4 *__restrict__ ck, uint32_t ck_pitch,
                                                       uint64_t ck_stride, float4 *__restrict__ gedge,
                                                       float *__restrict__ gcol, DevStatus *st) {
    extern __shared__ __align__(16) int s_cells[];  // cells, then the suffix sums of dA; then dA
    __shared__ RowLds R;
    __shared__ float s_gc[64];  // the round's colour gradients, in sum-tree order
    const uint32_t tw = TW ? TW : blockDim.x, pitch = tw + 1;
    const int tid = threadIdx.x, lane = tid & 63;
    const uint32_t X = blockIdx.x * tw + threadIdx.x, Y = blockIdx.y, im = blockIdx.z;
    uint32_t k0, np;
    if (!image_begin(S, st, im, k0, np)) return;
    const float xb0 = (float)(blockIdx.x * tw);
    const uint64_t slot = ((uint64_t)im * S.H + Y) * ck_pitch + X;
    const bool in = X < S.W;
    float *const s_suf = reinterpret_cast<float *>(s_cells);
    float *const s_dA = s_suf + SEG * pitch;
    uint32_t bad = 0;
    const float4 zero = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    const float4 f = in ? grad_canvas[((uint64_t)im * S.H + Y) * S.W + X] : zero;
    float T = 1.0f;
    for (uint32_t i = threadIdx.x; i < SEG * pitch; i += tw) s_cells[i] = 0;
    if (tid < 64) s_gc[tid] = 0.0f;
    for (uint32_t chunk = (np + ROW_PATHS - 1) / ROW_PATHS; chunk-- > 0;) {
        const uint32_t ja = chunk * ROW_PATHS;
        const uint32_t n = np - ja < ROW_PATHS ? np - ja : ROW_PATHS;
        __syncthreads();  // the previous paths' staging is no longer read
        stage_row(S, k0 + ja, n, (int)Y, R);
        __syncthreads();
        const uint32_t n_live = (uint32_t)__builtin_amdgcn_readfirstlane((int)R.n), rounds = (n_live + SEG - 1) / SEG;
        if (!rounds) continue;
        const float4 *const staged = colours + k0 + ja;
        PieceRef ref = piece_ref(S, R, rounds - 1, R.pb[(rounds - 1) * SEG] + threadIdx.x);
        PieceVtx v = piece_vtx(S, R, rounds - 1, ref, bad);
        PieceRef nref = ref;
        if (rounds > 1) nref = piece_ref(S, R, rounds - 2, R.pb[(rounds - 2) * SEG] + threadIdx.x);
        for (uint32_t s = rounds; s-- > 0;) {
            const uint32_t j0 = ja + s * SEG;
            const float4 C = in && j0 ? ck[(uint64_t)(j0 / SEG) * ck_stride + slot] : zero;
            const PieceRef cur = ref;
            const PieceVtx cv = v;
            if (s > 0) {  // the next round's vertices, and the one after's edge
                ref = nref;
                v = piece_vtx(S, R, s - 1, ref, bad);
                if (s > 1) nref = piece_ref(S, R, s - 2, R.pb[(s - 2) * SEG] + threadIdx.x);
            }
            float A[SEG];
            round_cover<false, TW>(S, R, s, cur, piece_of(cv.p, cv.q, (int)Y), (int)Y, xb0, s_cells, A, bad);
            const RoundPaths rp = round_paths(R, s, n_live);
            float q[SEG];  // f . canvas under path j
            // f . c_j - c_j.w q_j, made again in the second pass: kept beside q it
            // spilled 16 more registers (3.77 ms instead of 3.57 for 64 images when it was tried)
            auto d_of = [&](const float4 &c, float qj) {
                return fmaf(-c.w, qj, fmaf(f.w, c.w, fmaf(f.z, c.z, fmaf(f.y, c.y, f.x * c.x))));
            };
            float qr = fmaf(f.w, C.w, fmaf(f.z, C.z, fmaf(f.y, C.y, f.x * C.x)));
#pragma unroll
            for (uint32_t j = 0; j < SEG; ++j) {
                const float4 c = round_colour(staged, rp, j);
                q[j] = qr;
                qr = fmaf(alpha_cover(A[j]), d_of(c, qr), qr);  // = al f . c_j + (1 - c_j.w al) q_j
            }
            float z[SEG / 2];
            const bool b3 = (lane & 8) != 0, b2 = (lane & 4) != 0, b1 = (lane & 2) != 0, b0 = (lane & 1) != 0;
#pragma unroll
            for (uint32_t jp = SEG / 2; jp-- > 0;) {
                float r[2][4];
#pragma unroll
                for (uint32_t h = 2; h-- > 0;) {
                    const uint32_t j = 2 * jp + h;
                    const float4 c = round_colour(staged, rp, j);
                    // (else the first pass's alpha and d stay in registers: 3.19 ms, 3.03 so, when it came in)
                    asm("" : "+v"(A[j]), "+v"(q[j]));
                    const float al = alpha_cover(A[j]);
                    const float dal = T * d_of(c, q[j]), V = T * al;
                    const bool part = (fabsf(A[j]) < 1.0f) & (A[j] != 0.0f);
                    const float dA = part ? (A[j] > 0.0f ? dal : -dal) : 0.0f;
                    r[h][0] = V * f.x;
                    r[h][1] = V * f.y;
                    r[h][2] = V * f.z;
                    r[h][3] = V * (f.w - q[j]);
                    T *= fmaf(-c.w, al, 1.0f);
                    s_dA[j * pitch + tid] = dA;
                    s_suf[j * pitch + tid] = row_suffix(dA);
                }
                const float x0 = sum2(r[0][0], r[1][0]), x1 = sum2(r[0][1], r[1][1]);
                const float x2 = sum2(r[0][2], r[1][2]), x3 = sum2(r[0][3], r[1][3]);
                z[jp] = sum_dpp<0x140>(sum_rows(x0, x1), sum_rows(x2, x3), b3);  // row_mirror
            }
#pragma unroll
            for (uint32_t i = 0; i < 4; ++i) z[i] = sum_dpp<0x141>(z[2 * i], z[2 * i + 1], b2);  // row_half_mirror
#pragma unroll
            for (uint32_t i = 0; i < 2; ++i) z[i] = sum_dpp<0x1B>(z[2 * i], z[2 * i + 1], b1);  // quad_perm 3,2,1,0
            // lane: path 2 (4 b0 + 2 b1 + b2) + (lane >> 5), channel 2 b3 + (lane >> 4 & 1)
            const float gc = sum_dpp<0xB1>(z[0], z[1], b0);  // quad_perm 1,0,3,2
            if (gc != 0.0f) atomicAdd(&s_gc[lane], gc);
            __syncthreads();
            if (tid < 64) {
                const float g = s_gc[tid];
                const uint32_t j = 2 * (4 * (tid & 1) + (tid & 2) + ((tid >> 2) & 1)) + (tid >> 5);
                const uint32_t ch = ((tid >> 2) & 2) + ((tid >> 4) & 1);
                s_gc[tid] = 0.0f;
                if (g != 0.0f && j < rp.n)
                    atomicAdd(&gcol[4 * (uint64_t)(k0 + ja + R.path[s * SEG + j]) + ch], g);
            }
            // the pieces' gradients
            const uint32_t base = R.pb[s * SEG], end = R.pb[(s + 1) * SEG];
            for (uint32_t eb = base; eb < end; eb += tw) {
                if (eb + ((uint32_t)tid & ~63u) >= end) break;  // no piece for this wavefront
                PieceRef pr = cur;
                PieceVtx pv = cv;
                if (eb != base) {
                    pr = piece_ref(S, R, s, eb + threadIdx.x);
                    pv = piece_vtx(S, R, s, pr, bad);
                }
                Piece pc = piece_of(pv.p, pv.q, (int)Y);
                pc.live &= pr.j != NO_IDX;
                const Ramp m = ramp_of(pc, xb0, (int)tw);
                const uint32_t at = (pr.j != NO_IDX ? pr.j : 0u) * pitch;
                const bool wide = m.live & (m.c1 - m.c0 > RAMP_LANE);
                float S1 = 0.0f, S2 = 0.0f, S3 = 0.0f;
                if (m.live & !wide)
                    for (int c = m.c0; c < m.c1; ++c) ramp_grad(m, xb0 + (float)(c + 1), s_dA[at + c], S1, S2, S3);
                unsigned long long todo = __ballot(wide);
                while (todo) {  // a long ramp: one column per lane
                    const int l = __ffsll((long long)todo) - 1;
                    todo &= todo - 1;
                    auto bc = [l](float u) {
                        return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, u), l));
                    };
                    Ramp w;
                    w.lo = bc(m.lo);
                    w.hi = bc(m.hi);
                    w.w = w.hi - w.lo;
                    w.inv = bc(m.inv);
                    const int w0 = __builtin_amdgcn_readlane(m.c0, l), w1 = __builtin_amdgcn_readlane(m.c1, l);
                    const uint32_t wat = (uint32_t)__builtin_amdgcn_readlane((int)at, l);
                    float a1 = 0.0f, a2 = 0.0f, a3 = 0.0f;
                    for (int c = w0 + lane; c < w1; c += 64)
                        ramp_grad(w, xb0 + (float)(c + 1), s_dA[wat + c], a1, a2, a3);
                    wave_sum3(a1, a2, a3);
                    S1 = lane == l ? a1 : S1;
                    S2 = lane == l ? a2 : S2;
                    S3 = lane == l ? a3 : S3;
                }
                if (m.live) {  // the columns right of the ramp
                    const int t = m.c1 > m.c0 ? m.c1 : m.c0;
                    if (t < (int)tw) S1 += chunk_right(s_suf + at + (t & ~63), t & 63);
                    for (int c = (t | 63) + 1; c < (int)tw; c += 64) S1 += chunk_right(s_suf + at + c, 0);
                    if ((S1 != 0.0f) | (S2 != 0.0f) | (S3 != 0.0f)) {
                        const bool flip = pc.xa < pc.xb;  // S2 goes with the larger x
                        const EdgeGrad g =
                            piece_grad(pv.p, pv.q, (int)Y, S1, flip ? S3 : S2, flip ? S2 : S3);
                        atomicAdd(&gedge[pv.ip].x, g.xp);
                        atomicAdd(&gedge[pv.ip].y, g.xq);
                        if (g.has_p) atomicAdd(&gedge[pv.ip].z, g.yp);
                        if (g.has_q) atomicAdd(&gedge[pv.ip].w, g.yq);
                    }
                }
            }
            __syncthreads();
#pragma unroll
            for (uint32_t j = 0; j < SEG; ++j) s_cells[j * pitch + tid] = 0;
            __syncthreads();
        }
    }
    if (bad) raise_err(st, FT_EDEVICE);
}

// The edge gradients of a path's edge e, with the y gradients completed by
// the slope's share: (x, y) of its first vertex, (x, y) of its second.
__device__ __forceinline__ float4 edge_grad(const DScene &S, const float4 *gedge, uint32_t vb, uint32_t V,
                                            uint32_t e) {
    const float4 g = gedge[vb + e];
    const float2 p = S.vtx[vb + e], q = S.vtx[vb + (e + 1 < V ? e + 1 : 0u)];
    const float sl = (q.x - p.x) / (q.y - p.y);
    // (an edge without pieces, a horizontal one among them, has no gradient)
    return make_float4(g.x, g.x != 0.0f ? fmaf(-sl, g.x, g.z) : g.z, g.y, g.y != 0.0f ? fmaf(-sl, g.y, g.w) : g.w);
}

// Control point gradients from edge gradients: the sum over the point's
// cubics' vertices of their Bernstein weights times the vertex's gradient,
// which is its two edges' shares.  DSEG lanes per point, one per vertex of a
// cubic; a vertex's second edge is its neighbour's first.  (One thread per
// point walked its 16 or 32 vertices one after another, a chain of loads and
// divisions: 7.0 us for 200x120, 8.8 for 512x512 and 60 for 64 images, now
// 4.0, 4.2 and 62.)  One block also reports the run's status, every other
// kernel of the run being done.
__global__ __launch_bounds__(BLOCK) void k_point_grad(DScene S, const float4 *gedge, float2 *gpts, uint32_t n_pts,
                                                      const uint32_t *pt_path, const DevStatus *st,
                                                      HostStatus *report) {
    static_assert(DSEG == 16, "a point's lanes are one DPP row");
    if (blockIdx.x == 0) report_status(report, st, nullptr, nullptr, 0);
    const uint32_t q = threadIdx.x % DSEG;  // vertex q + 1 of the cubic
    constexpr uint32_t PTS = BLOCK / DSEG;
    for (uint32_t mb = blockIdx.x * PTS; mb < n_pts; mb += gridDim.x * PTS) {
        const uint32_t m = mb + threadIdx.x / DSEG;
        const bool on = m < n_pts;
        const uint32_t k = pt_path[on ? m : 0u];
        const uint32_t local = on ? m - S.pt_off[k] : 0u;
        const uint32_t n_cub = (S.pt_off[k + 1] - S.pt_off[k] - 1) / 3;
        const uint32_t vb = S.vtx_off[k], V = S.vtx_off[k + 1] - vb;
        float2 acc = make_float2(0.0f, 0.0f);
        if (local == 0 && q == 0) {
            const float4 g = edge_grad(S, gedge, vb, V, 0), l = edge_grad(S, gedge, vb, V, V - 1);
            acc = make_float2(g.x + l.z, g.y + l.w);
        }
        // the point is control r of cubic c (and control 0 of cubic c + 1 when r == 3)
#pragma unroll
        for (int pass = 0; pass < 2; ++pass) {
            const bool has = pass == 0 ? local != 0 : (local % 3 == 0) & (local / 3 < n_cub);
            const uint32_t c = pass == 0 ? (local ? (local - 1) / 3 : 0u) : (has ? local / 3 : 0u);
            const uint32_t r = pass == 0 ? (local ? (local - 1) % 3 + 1 : 0u) : 0u;
            if (pass == 1 && !__any(has)) continue;
            const float4 in = edge_grad(S, gedge, vb, V, c * DSEG + q);  // the edge into vertex c * DSEG + q + 1
            // and the one out of it: the next lane's, the last lane's its own
            float2 out = make_float2(__shfl_down(in.x, 1, DSEG), __shfl_down(in.y, 1, DSEG));
            if (q == DSEG - 1) {
                const float4 e = edge_grad(S, gedge, vb, V, (c + 1) * DSEG);
                out = make_float2(e.x, e.y);
            }
            float w[4];
            bern((int)q + 1, w);
            const float wr = r == 0 ? w[0] : (r == 1 ? w[1] : (r == 2 ? w[2] : w[3]));
            acc.x += has ? wr * (in.z + out.x) : 0.0f;
            acc.y += has ? wr * (in.w + out.y) : 0.0f;
        }
#pragma unroll
        for (int o = DSEG / 2; o > 0; o >>= 1) {
            acc.x += __shfl_xor(acc.x, o, DSEG);
            acc.y += __shfl_xor(acc.y, o, DSEG);
        }
        if (on & (q == 0)) gpts[m] = acc;
    }
}

}  // namespace diff
}  // namespace ft

// ---------------------------------------------------------------------------
// Host side and C ABI
// ---------------------------------------------------------------------------
using namespace ft;
using namespace ft::diff;

struct ft_diff {
    hipStream_t stream = nullptr;
    uint32_t n_images = 0, W = 0, H = 0, n_paths = 0, max_paths = 0;
    uint32_t n_pts = 0, n_vtx = 0;
    uint32_t max_path_vtx = 0;  // most vertices (edges) of one path
    uint64_t n_cells = 0, canvas_floats = 0;
    uint32_t *d_pt_off = nullptr, *d_vtx_off = nullptr, *d_vtx_path = nullptr, *d_img_first = nullptr,
             *d_pt_path = nullptr;
    float2 *d_vtx = nullptr;
    float4 *d_gedge = nullptr;  // per edge: see EdgeGrad
    uint32_t *d_cell_cnt = nullptr, *d_cell_off = nullptr, *d_cell_cur = nullptr, *d_cell_edge = nullptr;
    uint32_t cap_pairs = 0;
    size_t cap_tiles = 0;
    unsigned long long *d_lb = nullptr;  // scan look-back words
    float4 *d_ck = nullptr;
    uint32_t ck_pitch = 0;  // checkpoint pixels per row
    uint64_t ck_stride = 0;  // and per checkpoint
    unsigned long long *d_partial = nullptr;  // [LOSS_GRID] loss partials (doubles)
    uint32_t *d_done = nullptr;   // blocks of k_loss done: 0 between its runs
    double *h_loss = nullptr;     // pinned: the summed loss, written by k_loss
    DevStatus *d_status = nullptr;
    HostStatus *h_status = nullptr;  // pinned: written by a run's last kernel
    bool clean = false;  // d_lb and d_status are as k_clear_run leaves them
};

namespace {

#define FD_HIP(call)                                 \
    do {                                             \
        if ((call) != hipSuccess) return FT_EDEVICE; \
    } while (0)

template <typename T>
ft_status dalloc(T *&p, size_t n) {
    if (p) (void)hipFree(p);
    p = nullptr;
    return hipMalloc(reinterpret_cast<void **>(&p), (n ? n : 1) * sizeof(T)) == hipSuccess ? FT_OK : FT_ENOMEM;
}

DScene scene_of(const ft_diff *d) {
    DScene S;
    S.n_images = d->n_images;
    S.W = d->W;
    S.H = d->H;
    S.n_paths = d->n_paths;
    S.n_vtx = d->n_vtx;
    S.n_cells = (uint32_t)d->n_cells;
    S.pt_off = d->d_pt_off;
    S.vtx_off = d->d_vtx_off;
    S.vtx_path = d->d_vtx_path;
    S.img_first = d->d_img_first;
    S.vtx = d->d_vtx;
    S.cell_cnt = d->d_cell_cnt;
    S.cell_off = d->d_cell_off;
    S.cell_cur = d->d_cell_cur;
    S.cell_edge = d->d_cell_edge;
    S.cap_pairs = d->cap_pairs;
    return S;
}

uint32_t grid_of(uint64_t n) {
    uint64_t g = (n + BLOCK - 1) / BLOCK;
    return (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(g, GRID_MAX));
}

// Blocks of k_geometry (0: the scene takes the general form).
uint32_t geometry_blocks(const ft_diff *d) {
    if (d->max_path_vtx > GEOM_EDGES || !d->n_paths) return 0;
    const uint32_t per = (d->n_paths + GEOM_BLOCKS - 1) / GEOM_BLOCKS;
    return (d->n_paths + per - 1) / per;
}

// Geometry for one parameter set: vertices, per-(path, row) edge lists.
ft_status launch_geometry(ft_diff *d, const float *points, bool clear_grads, float *gcol) {
    hipStream_t s = d->stream;
    DScene S = scene_of(d);
    float4 *const gedge = clear_grads ? d->d_gedge : nullptr;
    if (!clear_grads) gcol = nullptr;
    const float2 *const pts = reinterpret_cast<const float2 *>(points);
    uint32_t *const host_err = &d->h_status->late_err;
    const bool clean = d->clean;
    d->clean = false;  // until this run is known to have left them so
    if (const uint32_t blocks = geometry_blocks(d)) {
        const uint32_t per = (d->n_paths + GEOM_BLOCKS - 1) / GEOM_BLOCKS;
        if (!clean)
            k_clear_run<<<1, BLOCK, 0, s>>>(d->d_lb, (uint32_t)lookback_words(blocks), d->d_status, host_err);
        const size_t lds = (std::min(d->H, GEOM_ROWS) + 1) * sizeof(uint32_t);
        k_geometry<<<blocks, BLOCK, lds, s>>>(S, pts, gedge, gcol, per, d->d_lb, d->d_status);
        FD_HIP(hipGetLastError());
        return FT_OK;
    }
    const uint32_t n_lb = (uint32_t)(4 * d->cap_tiles);  // look-back words of the two cell scans
    const uint64_t n_clear = std::max<uint64_t>(std::max<uint64_t>(d->n_cells, d->n_vtx),
                                                std::max<uint64_t>(4ull * d->n_paths, n_lb));
    k_clear_cells<<<grid_of(n_clear), BLOCK, 0, s>>>(S, gedge, gcol, d->d_lb, n_lb, d->d_status, host_err);
    k_vertices<<<grid_of(d->n_vtx), BLOCK, 0, s>>>(S, pts, d->d_status);
    k_rows<<<grid_of(d->n_vtx), BLOCK, 0, s>>>(S, d->d_status);
    const uint32_t nc = (uint32_t)d->n_cells;
    scan_launch<uint32_t, false>(s, scan_resident_blocks(), d->d_cell_cnt, d->d_cell_cnt, nullptr, nc, nc, d->d_lb,
                                 nullptr, d->d_status, false, true);
    scan_launch<uint32_t, false>(s, scan_resident_blocks(), d->d_cell_cnt, d->d_cell_off, nullptr, nc, nc,
                                 d->d_lb + 2 * d->cap_tiles, &d->d_status->n_pairs, d->d_status, false, false);
    k_fill_cells<<<grid_of((size_t)d->n_vtx * FILL_LANES), BLOCK, 0, s>>>(S, d->d_status);
    FD_HIP(hipGetLastError());
    return FT_OK;
}

// The run's one host wait.  Its kernels have written the status (and the
// summed loss) to host memory: two copies behind the last kernel cost 8 us of
// a step that then took 390.
ft_status finish(ft_diff *d) {
    FD_HIP(hipStreamSynchronize(d->stream));
    const uint32_t late = d->h_status->late_err;
    d->h_status->late_err = 0;
    if (d->h_status->st.err) return (ft_status)d->h_status->st.err;
    if (late) return (ft_status)late;
    if (d->h_status->st.overflow) return (ft_status)0x100;
    d->clean = geometry_blocks(d) != 0;
    return FT_OK;
}

ft_status grow_pairs(ft_diff *d) {
    const uint64_t need = (uint64_t)d->h_status->st.need_pairs;
    const uint64_t cap = need + need / 4 + 4096;
    if (cap >= 0xFFFFFFFFull) return FT_ENOMEM;
    ft_status st = dalloc(d->d_cell_edge, cap);
    if (st) return st;
    d->cap_pairs = (uint32_t)cap;
    return FT_OK;
}

// Tiles of the forward and the backward: at most TILE_MAX pixels of a row, in
// whole wavefronts.
uint32_t tiles_of(const ft_diff *d) { return (d->W + TILE_MAX - 1) / TILE_MAX; }
uint32_t tile_width(const ft_diff *d) {
    const uint32_t n = tiles_of(d);
    return ((d->W + n - 1) / n + 63) / 64 * 64;
}

// canvas may be null; keep: also the checkpoints that the backward needs;
// last: no later kernel reports the run's status.
ft_status launch_forward(ft_diff *d, const float *colours, float *canvas, bool keep, bool last) {
    const uint32_t blocks = geometry_blocks(d);
    const uint32_t tw = tile_width(d);
    const size_t lds = (size_t)SEG * (tw + 1) * sizeof(int);
    (tw == TILE_MAX ? k_forward<TILE_MAX> : k_forward<0>)<<<dim3(tiles_of(d), d->H, d->n_images), tw, lds, d->stream>>>(
        scene_of(d), reinterpret_cast<const float4 *>(colours), reinterpret_cast<float4 *>(canvas),
        keep ? d->d_ck : nullptr, d->ck_pitch, d->ck_stride, d->d_status, d->d_lb,
        blocks ? (uint32_t)lookback_words(blocks) : 0u, last ? d->h_status : nullptr);
    FD_HIP(hipGetLastError());
    return FT_OK;
}

ft_status run_forward(ft_diff *d, const float *points, const float *colours, float *canvas) {
    for (int attempt = 0; attempt < 3; ++attempt) {
        ft_status st = launch_geometry(d, points, false, nullptr);
        if (st) return st;
        if ((st = launch_forward(d, colours, canvas, false, true))) return st;
        st = finish(d);
        if (st != (ft_status)0x100) return st;
        if ((st = grow_pairs(d))) return st;
    }
    return FT_ENOMEM;
}

// Enqueues the loss (to h_loss) and its gradient.
ft_status launch_loss(ft_diff *d, const float *canvas, const float *target, float *grad) {
    const uintptr_t low = reinterpret_cast<uintptr_t>(canvas) | reinterpret_cast<uintptr_t>(target) |
                          reinterpret_cast<uintptr_t>(grad);
    (low & 15u ? k_loss<1> : k_loss<4>)<<<LOSS_GRID, BLOCK, 0, d->stream>>>(canvas, target, grad, d->canvas_floats,
                                                                           d->d_partial, d->d_done, d->h_loss);
    FD_HIP(hipGetLastError());
    return FT_OK;
}

ft_status run_loss(ft_diff *d, const float *canvas, const float *target, float *grad, double *loss) {
    ft_status st = launch_loss(d, canvas, target, grad);
    if (!st) {
        FD_HIP(hipStreamSynchronize(d->stream));
        if (loss) *loss = *d->h_loss / (double)d->canvas_floats;
    }
    return st;
}

// Enqueues the backward kernels, after a forward of the same points and
// colours that left its checkpoints.
ft_status launch_backward(ft_diff *d, const float *colours, const float *grad_canvas, float *grad_points,
                          float *grad_colours) {
    DScene S = scene_of(d);
    const uint32_t tw = tile_width(d);
    const size_t lds = 2 * (size_t)SEG * (tw + 1) * sizeof(float);
    (tw == TILE_MAX ? k_backward<TILE_MAX> : k_backward<0>)<<<dim3(tiles_of(d), d->H, d->n_images), tw, lds, d->stream>>>(
        S, reinterpret_cast<const float4 *>(colours), reinterpret_cast<const float4 *>(grad_canvas), d->d_ck,
        d->ck_pitch, d->ck_stride, d->d_gedge, grad_colours, d->d_status);
    k_point_grad<<<grid_of((uint64_t)d->n_pts * DSEG), BLOCK, 0, d->stream>>>(
        S, d->d_gedge, reinterpret_cast<float2 *>(grad_points),
                                                             d->n_pts, d->d_pt_path, d->d_status, d->h_status);
    FD_HIP(hipGetLastError());
    return FT_OK;
}

ft_status run_backward(ft_diff *d, const float *points, const float *colours, const float *grad_canvas,
                       float *grad_points, float *grad_colours) {
    for (int attempt = 0; attempt < 3; ++attempt) {
        ft_status st = launch_geometry(d, points, true, grad_colours);
        if (!st) st = launch_forward(d, colours, nullptr, true, false);
        if (!st) st = launch_backward(d, colours, grad_canvas, grad_points, grad_colours);
        if (st) return st;
        st = finish(d);
        if (st != (ft_status)0x100) return st;
        if ((st = grow_pairs(d))) return st;
    }
    return FT_ENOMEM;
}

// forward (leaving checkpoints), loss and backward on one geometry, with one
// host wait; a pair overflow turns the later kernels into no-ops, and the
// step is run again with room for the pairs.
ft_status run_step(ft_diff *d, const float *points, const float *colours, const float *target, float *canvas,
                   float *grad_canvas, float *grad_points, float *grad_colours, double *loss) {
    for (int attempt = 0; attempt < 3; ++attempt) {
        ft_status st = launch_geometry(d, points, true, grad_colours);
        if (st) return st;
        if ((st = launch_forward(d, colours, canvas, true, false))) return st;
        if ((st = launch_loss(d, canvas, target, grad_canvas))) return st;
        if ((st = launch_backward(d, colours, grad_canvas, grad_points, grad_colours))) return st;
        st = finish(d);
        if (st == FT_OK && loss) *loss = *d->h_loss / (double)d->canvas_floats;
        if (st != (ft_status)0x100) return st;
        if ((st = grow_pairs(d))) return st;
    }
    return FT_ENOMEM;
}

}  // namespace

extern "C" {

ft_status ft_diff_new(const ft_diff_layout *L, ft_diff **out) {
    if (!L || !out || !L->path_image || !L->path_cubics || !L->n_images || !L->width || !L->height ||
        (L->flags & ~FT_DIFF_KEEP_COVERAGE))
        return FT_EINVAL;
    if (L->width > FT_MAX_WIDTH || L->height > FT_MAX_WIDTH) return FT_ENOTSUP;
    std::vector<uint32_t> pt_off(L->n_paths + 1), vtx_off(L->n_paths + 1), img_first(L->n_images + 1);
    uint64_t np = 0, nv = 0;
    for (uint32_t k = 0; k < L->n_paths; ++k) {
        if (L->path_image[k] >= L->n_images || (k && L->path_image[k] < L->path_image[k - 1])) return FT_EINVAL;
        if (L->path_cubics[k] == 0 || L->path_cubics[k] > (1u << 20)) return FT_EINVAL;
        pt_off[k] = (uint32_t)np;
        vtx_off[k] = (uint32_t)nv;
        np += 1 + 3ull * L->path_cubics[k];
        nv += 1 + (uint64_t)DSEG * L->path_cubics[k];
        if (np >= 0x7FFFFFFFull || nv >= 0x7FFFFFFFull) return FT_ENOTSUP;
    }
    pt_off[L->n_paths] = (uint32_t)np;
    vtx_off[L->n_paths] = (uint32_t)nv;
    uint32_t max_paths = 0;
    {
        uint32_t k = 0;
        for (uint32_t i = 0; i <= L->n_images; ++i) {
            while (k < L->n_paths && L->path_image[k] < i) ++k;
            img_first[i] = k;
        }
        for (uint32_t i = 0; i < L->n_images; ++i) max_paths = std::max(max_paths, img_first[i + 1] - img_first[i]);
    }
    const uint64_t cells = (uint64_t)L->n_paths * L->height;
    if (cells >= 0xFFFFFFFFull) return FT_ENOTSUP;
    std::vector<uint32_t> vtx_path(nv), pt_path(np);
    for (uint32_t k = 0; k < L->n_paths; ++k) {
        for (uint32_t v = vtx_off[k]; v < vtx_off[k + 1]; ++v) vtx_path[v] = k;
        for (uint32_t m = pt_off[k]; m < pt_off[k + 1]; ++m) pt_path[m] = k;
    }
    ft_diff *d = new ft_diff();
    d->n_images = L->n_images;
    d->W = L->width;
    d->H = L->height;
    d->n_paths = L->n_paths;
    d->max_paths = max_paths;
    d->n_pts = (uint32_t)np;
    d->n_vtx = (uint32_t)nv;
    for (uint32_t k = 0; k < L->n_paths; ++k) d->max_path_vtx = std::max(d->max_path_vtx, vtx_off[k + 1] - vtx_off[k]);
    d->n_cells = cells;
    d->canvas_floats = 4ull * L->n_images * L->width * L->height;
    d->ck_pitch = (d->W + 15) / 16 * 16;
    d->ck_stride = (uint64_t)d->ck_pitch * d->H * d->n_images;
    const uint64_t n_ck = std::max<uint64_t>(1, (max_paths + SEG - 1) / SEG);
    d->cap_tiles = (cells + SCAN_TILE_MIN - 1) / SCAN_TILE_MIN + 1;
    d->cap_pairs = (uint32_t)std::min<uint64_t>(0xFFFFFFF0ull, 8 * nv + 4096);
    ft_status st;
    if (hipStreamCreateWithFlags(&d->stream, hipStreamNonBlocking) != hipSuccess) st = FT_EDEVICE;
    else if ((st = dalloc(d->d_pt_off, L->n_paths + 1)) || (st = dalloc(d->d_vtx_off, L->n_paths + 1)) ||
             (st = dalloc(d->d_vtx_path, nv)) || (st = dalloc(d->d_pt_path, np)) ||
             (st = dalloc(d->d_img_first, L->n_images + 1)) || (st = dalloc(d->d_vtx, nv)) ||
             (st = dalloc(d->d_gedge, nv)) || (st = dalloc(d->d_cell_cnt, cells)) ||
             (st = dalloc(d->d_cell_off, cells)) || (st = dalloc(d->d_cell_cur, cells)) ||
             (st = dalloc(d->d_cell_edge, d->cap_pairs)) || (st = dalloc(d->d_lb, std::max<size_t>(4 * d->cap_tiles, lookback_words(GEOM_BLOCKS)))) ||
             (st = dalloc(d->d_ck, n_ck * d->ck_stride)) || (st = dalloc(d->d_partial, LOSS_GRID)) ||
             (st = dalloc(d->d_status, 1)) || (st = dalloc(d->d_done, 1)))
        ;
    else if (hipMemset(d->d_done, 0, sizeof(uint32_t)) != hipSuccess)
        st = FT_EDEVICE;
    else if (hipHostMalloc(reinterpret_cast<void **>(&d->h_loss), sizeof(double), hipHostMallocCoherent) !=
                 hipSuccess ||
             hipHostMalloc(reinterpret_cast<void **>(&d->h_status), sizeof(HostStatus), hipHostMallocCoherent) !=
                 hipSuccess)
        st = FT_ENOMEM;
    else if (hipMemcpy(d->d_pt_off, pt_off.data(), pt_off.size() * 4, hipMemcpyHostToDevice) != hipSuccess ||
             hipMemcpy(d->d_vtx_off, vtx_off.data(), vtx_off.size() * 4, hipMemcpyHostToDevice) != hipSuccess ||
             hipMemcpy(d->d_vtx_path, vtx_path.data(), nv * 4, hipMemcpyHostToDevice) != hipSuccess ||
             hipMemcpy(d->d_pt_path, pt_path.data(), np * 4, hipMemcpyHostToDevice) != hipSuccess ||
             hipMemcpy(d->d_img_first, img_first.data(), img_first.size() * 4, hipMemcpyHostToDevice) != hipSuccess)
        st = FT_EDEVICE;
    else {
        *d->h_status = HostStatus{};
        st = FT_OK;
    }
    if (st) {
        ft_diff_free(d);
        return st;
    }
    *out = d;
    return FT_OK;
}

void ft_diff_free(ft_diff *d) {
    if (!d) return;
    void *bufs[] = {d->d_pt_off,   d->d_vtx_off,  d->d_vtx_path, d->d_pt_path,   d->d_img_first, d->d_vtx,
                    d->d_gedge,     d->d_cell_cnt, d->d_cell_off, d->d_cell_cur,  d->d_cell_edge, d->d_lb,
                    d->d_ck,       d->d_partial,  d->d_status,   d->d_done};
    for (void *b : bufs)
        if (b) (void)hipFree(b);
    if (d->h_loss) (void)hipHostFree(d->h_loss);
    if (d->h_status) (void)hipHostFree(d->h_status);
    if (d->stream) (void)hipStreamDestroy(d->stream);
    delete d;
}

ft_status ft_diff_info(const ft_diff *d, uint64_t *n_points, uint64_t *n_paths, uint64_t *canvas_floats) {
    if (!d) return FT_EINVAL;
    if (n_points) *n_points = d->n_pts;
    if (n_paths) *n_paths = d->n_paths;
    if (canvas_floats) *canvas_floats = d->canvas_floats;
    return FT_OK;
}

ft_status ft_diff_forward(ft_diff *d, const float *points, const float *colours, float *canvas) {
    if (!d || !points || !colours || !canvas) return FT_EINVAL;
    return run_forward(d, points, colours, canvas);
}

ft_status ft_diff_loss(ft_diff *d, const float *canvas, const float *target, float *grad_canvas, double *loss) {
    if (!d || !canvas || !target) return FT_EINVAL;
    return run_loss(d, canvas, target, grad_canvas, loss);
}

ft_status ft_diff_backward(ft_diff *d, const float *points, const float *colours, const float *grad_canvas,
                           float *grad_points, float *grad_colours) {
    if (!d || !points || !colours || !grad_canvas || !grad_points || !grad_colours) return FT_EINVAL;
    return run_backward(d, points, colours, grad_canvas, grad_points, grad_colours);
}

ft_status ft_diff_step(ft_diff *d, const float *points, const float *colours, const float *target, float *canvas,
                       float *grad_canvas, float *grad_points, float *grad_colours, double *loss) {
    if (!d || !points || !colours || !target || !canvas || !grad_canvas || !grad_points || !grad_colours)
        return FT_EINVAL;
    return run_step(d, points, colours, target, canvas, grad_canvas, grad_points, grad_colours, loss);
}

}  // extern "C"
