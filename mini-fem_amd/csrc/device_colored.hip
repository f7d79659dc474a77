// Drop-in GPU twins of the reference's per-iteration entry points:
//   assembly()        -> mf_assembly / mf_assembly_ex   (COLORING semantics)
//   prec_init()       -> mf_prec_init
//   prec_inversion()  -> mf_prec_inversion
//   compute_double_norm() -> mf_norm
// The assembly goes row by row (k_assemble_rows): the per-entry summation order is the color
// order, i.e. the reference COLORING build's element order. What the rows cannot do goes on, in
// the same order, in launches after them that ordinarily return at once (k_entry_* with
// elemToEdge, else k_assemble_left). Under stream capture, without
// memory for its workspace, for patterns thinner than the elements' couplings and for large lap
// meshes with elemToEdge it is one
// launch per color with 16 lanes per element (one per element block): elements of one color
// share no node, so their scatter-adds never touch the same CSR entry and each pass is
// race-free and deterministic, in the same order.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <type_traits>
#include <vector>

#include "device_common.h"
#include "minifem.h"

namespace {

constexpr int kBlock = 256;

// CSR position of the (j,k) pair of one element: elemToEdge when present, else the
// reference's row search (src/assembly.cc:415-421).
__device__ __forceinline__ int elem_position(const int *__restrict__ row,
                                             const int *__restrict__ col,
                                             const int *__restrict__ e2e, int e, int nj, int nk,
                                             int q)
{
    if (e2e) return e2e[(int64_t)e * 16 + q];
    for (int l = row[nj - 1]; l < row[nj]; l++)
        if (col[l] == nk) return l;
    return -1;
}

// Element e's (j,k) block, q = 4j + k.
template <int OP, int PREC>
__device__ __forceinline__ void
elem_block(const double *__restrict__ coord, const double *__restrict__ coef, int4 v, int e, int q,
           double (&out)[OP == MF_OP_ELA ? 9 : 1])
{
    const int j = q >> 2, k = q & 3;
    double c[4][3], g[4][3];
    mf::load_coords(coord, v, c);
    mf::elem_grad(c, g);
    float gj[3], gk[3];
#pragma unroll
    for (int d = 0; d < 3; d++) {
        gj[d] = (float)g[j][d];
        gk[d] = (float)g[k][d];
    }
    if constexpr (OP == MF_OP_LAP) {
        const double kd = coef ? coef[e] : 1.0;
        if (PREC == MF_PREC_FP64) {
            const double x = mf::lap_entry(g[j], g[k]);
            out[0] = coef ? kd * x : x;
        } else {
            const float x = (float)kd * mf::lap_entry(gj, gk);
            out[0] = (double)x;
        }
    } else {
        const mf::ElaCoef kc = mf::ela_coef(coef, e);
        if (PREC == MF_PREC_FP64) {
            mf::ela_block(g[j], g[k], kc.cd, kc.co, kc.cm, out);
        } else {
            float b[9];
            mf::ela_block(gj, gk, (float)kc.cd, (float)kc.co, (float)kc.cm, b);
#pragma unroll
            for (int r = 0; r < 9; r++) out[r] = (double)b[r];
        }
    }
}

// Adds that block into its CSR entry. The 16 lanes of an element compute its gradients
// alike.
template <int OP, int PREC>
__device__ __forceinline__ void
add_block(const double *__restrict__ coord, const double *__restrict__ coef, double *values,
          const int *__restrict__ row, const int *__restrict__ col, const int4 *__restrict__ e2n,
          const int *__restrict__ e2e, int e, int q)
{
    constexpr int D = OP == MF_OP_ELA ? 9 : 1;
    const int4 v = e2n[e];
    const int n[4] = {v.x, v.y, v.z, v.w};
    const int p = elem_position(row, col, e2e, e, n[q >> 2], n[q & 3], q);
    if (p < 0) return;
    double b[D];
    elem_block<OP, PREC>(coord, coef, v, e, q, b);
    double *out = values + (int64_t)p * D;
#pragma unroll
    for (int r = 0; r < D; r++) out[r] += b[r];
}

struct ColorOffsets {
    int n;
    int off[MF_MAX_COLOR + 1];
};

// What the rows leave for the launches after them. Each workgroup reports in a slot of its
// own: some thousand atomics on one address took longer than a small call's rows (40 us).
constexpr int kTableGrid = 1024, kRowsGridMax = 4096;
struct RowsCtl {
    int odd;                       // set by the rows, cleared by the table
    int top[kTableGrid];           // the largest node id of each table workgroup's elements
    unsigned found[kRowsGridMax];  // table entries of each rows workgroup that are elements
    int left;                      // whether the rows left the call (k_entry_lists)
};

// Whether the rows left a call of nE elements to what follows them: they found something odd,
// or not 4 table entries per element. Called by a whole workgroup of BT threads; s: one word of
// LDS per thread.
template <int BT>
__device__ bool rows_verdict(const RowsCtl *ctl, int groups, int nE, unsigned long long *s)
{
    unsigned long long n = 0;
    for (int w = threadIdx.x; w < groups; w += BT) n += ctl->found[w];
    s[threadIdx.x] = n;
    __syncthreads();
    for (int w = BT / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) s[threadIdx.x] += s[threadIdx.x + w];
        __syncthreads();
    }
    return ctl->odd || s[0] != 4ull * (unsigned long long)nE;
}

__global__ void __launch_bounds__(kBlock) k_fill(double *__restrict__ p, int64_t n, double v)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (; i < n; i += stride) p[i] = v;
}

// One color: 16 lanes per element, lane q adds block q. Elements of one color share no
// node, so no two lanes of a launch touch the same entry; each entry receives its elements'
// blocks in color order, as in the reference COLORING build.
template <int OP, int PREC>
__global__ void __launch_bounds__(kBlock)
    k_assemble_color(const double *__restrict__ coord, const double *__restrict__ coef,
                     double *values, const int *__restrict__ row,
                     const int *__restrict__ col, const int4 *__restrict__ e2n,
                     const int *__restrict__ e2e, int first, int count)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (int64_t)count * 16) return;
    add_block<OP, PREC>(coord, coef, values, row, col, e2n, e2e, first + (int)(t >> 4), (int)(t & 15));
}

// ---- the whole assembly row by row ------------------------------------------------------
//
// One launch per color reads and writes every CSR block once per element that holds it (an
// off-diagonal block 5 times on a Kuhn cube, a diagonal one 24 times): 1.58 ms of the 1.83
// of an ela 60^3 call. Row by row, a block is summed in registers and written once. What a
// row needs is its elements in ascending order, and the coloring gives that without sorting
// or counting: a node has at most one element of each color, and a color's elements come
// before the next color's. So a table with one slot per node and color, filled with plain
// stores, lists every row's elements in order. The table is never cleared: a slot counts
// only if it names an element of its color that holds the node, and the slots that elements
// own are always written.
//
// The call does not say how many nodes there are, and a part of a mesh may keep the ids of the
// whole. The first nnz / 8 nodes (rows have 15 entries in the mean, so those are all unless ids
// are left out) have the line of their id in the table; a node past them has the line, after
// those, of a quarter of its row's start. The row of a node of an element has 4 entries or more
// (the element's own couplings), so no two such nodes share a line, and nnz / 4 lines hold them
// whatever the ids. Without those lines the launch after the rows took such a call: ela 40^3
// with ids eight times as far 62,000 us, so 337. All nodes by their rows' starts: lap 100^3
// 1,560 -> 1,889, ela 60^3 353 -> 369.
// What the rows cannot do is left to the launches after them (k_entry_*, k_assemble_left), which
// otherwise return at once: an elemToEdge entry outside its node's row, a diagonal entry that not
// all of the node's elements share, elements that repeat a node, and, past the first nnz / 8
// nodes, rows of fewer entries than an element's couplings.
//
// ela 60^3 1,830 -> 416 us, lap 31^3 with elemToEdge 148 -> 53 (the two prec
// calls included); ela 60^3: k_row_table 63 us, k_assemble_rows 293.

// The color of element e, one of the n from e0 (the same for the whole wave) on: e0's by
// bisection, then the few that the n span.
__device__ __forceinline__ int color_of(const ColorOffsets &co, int e0, int e, int n)
{
    int a = 0, b = co.n - 1;
    while (a < b) {
        const int m = (a + b + 1) >> 1;
        if (co.off[m] <= e0) a = m;
        else b = m - 1;
    }
    int c = a;
    for (int k = a + 1; k < co.n && co.off[k] < e0 + n; k++)
        if (co.off[k] <= e) c = k;
    return c;
}

// The lines of the table of a call of nnz entries: by id, then by the row's start.
__host__ __device__ constexpr int direct_lines(int nnz) { return nnz / 8 + 1; }
__host__ __device__ constexpr int table_lines(int nnz) { return direct_lines(nnz) + nnz / 4 + 1; }

// The line of node i (0-based); -1 where its row starts outside the entries.
__device__ __forceinline__ int line_of(int i, const int *__restrict__ row, int nnz)
{
    if (i < direct_lines(nnz)) return i;
    const int start = row[i];
    return start >= 0 && start <= nnz ? direct_lines(nnz) + (start >> 2) : -1;
}

__global__ void __launch_bounds__(kBlock)
    k_row_table(ColorOffsets co, const int4 *__restrict__ e2n, const int *__restrict__ row, int nE,
                int nnz, int width, int *__restrict__ table, int *__restrict__ head,
                RowsCtl *__restrict__ ctl)
{
    __shared__ int smax[kBlock / 64];
    int top = 0;
    const int lane = threadIdx.x & 63;
    // with elemToEdge, empty lists for k_entry_lists (here rather than in one more launch; head
    // has a whole number of 16 bytes)
    if (head)
        for (int64_t z = (int64_t)blockIdx.x * kBlock + threadIdx.x; z < ((int64_t)nnz + 3) / 4;
             z += (int64_t)gridDim.x * kBlock)
            reinterpret_cast<int4 *>(head)[z] = make_int4(-1, -1, -1, -1);
    for (int64_t first = ((int64_t)blockIdx.x * kBlock + threadIdx.x) & ~63ll; first < nE;
         first += (int64_t)gridDim.x * kBlock) {
        const int e0 = __builtin_amdgcn_readfirstlane((int)first), e = e0 + lane;
        const int c = color_of(co, e0, e, 64);
        if (e >= nE) continue;
        const int4 q = e2n[e];
        const int v[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int i = v[k] - 1;
            top = top > v[k] ? top : v[k];
            const int line = i < 0 ? -1 : line_of(i, row, nnz);
            if (line >= 0) table[(int64_t)line * width + c] = e;
        }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const int t = __shfl_xor(top, o);
        top = top > t ? top : t;
    }
    if (lane == 0) smax[threadIdx.x >> 6] = top;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kBlock / 64; w++) top = top > smax[w] ? top : smax[w];
        ctl->top[blockIdx.x] = top;
        if (blockIdx.x == 0) ctl->odd = 0;
    }
}

// Four rows per wave, 16 lanes each, one wave per workgroup. A row's elements are staged SL
// at a time, one lane each: the gradients with the row's own vertex first and the
// coefficients (ela), or the row's four products (lap). Then a lane per entry finds the
// elements that hold its column, as bits in order, and sums their blocks. The diagonal block
// of ela, which every element adds to, is summed apart: its six distinct values are formed
// by the lanes of the elements and added up by six lanes.
// What bounds it is latency: a row's loads depend on each other (row bounds, table, elements,
// coordinates), and the stage leaves 7 to 9 waves to a CU. So the first three are loaded
// three, two and one step ahead.
template <int OP, int PREC, bool EDGES, int KC>
__global__ void __launch_bounds__(64)
    k_assemble_rows(ColorOffsets co, const double *__restrict__ coord,
                    const double *__restrict__ coef, double *__restrict__ values,
                    const int *__restrict__ row, const int *__restrict__ col,
                    const int4 *__restrict__ e2n, const int *__restrict__ e2e, int nnz,
                    const int *__restrict__ table, RowsCtl *__restrict__ ctl, int tables)
{
    using T = typename std::conditional<PREC == MF_PREC_FP64, double, float>::type;
    constexpr bool ELA = OP == MF_OP_ELA;
    constexpr int D = ELA ? 9 : 1;
    constexpr int SL = 24;                                   // elements staged at a time
    constexpr int CH = (MF_MAX_COLOR + SL - 1) / SL;         // chunks of the longest row
    constexpr int S = ELA ? (sizeof(T) == 8 ? 18 : 20) : 4;  // values per element
    constexpr int PAD = 16 / (int)sizeof(T);                 // groups start on different banks
    constexpr int H = (SL + 15) / 16;                        // staged elements per lane
    __shared__ __align__(16) T s_stage[4][(SL + 1) * S + PAD];
    __shared__ int4 s_ids[4][SL + 1];
    __shared__ int4 s_node[4][16 * KC + 1];  // a row's elements in order: their vertices,
    __shared__ int s_list[4][16 * KC];       // and 4 e + the row's vertex
    __shared__ uint32_t s_seen[4][CH * 4];   // matched bits per chunk and vertex
    const int l = threadIdx.x & 15, g = threadIdx.x >> 4;
    T *stage = s_stage[g];
    for (int q = l; q < S; q += 16) stage[SL * S + q] = (T)0;
    int lo[KC], hi[KC];
#pragma unroll
    for (int k = 0; k < KC; k++) {
        const int c = l + 16 * k;
        lo[k] = c < co.n ? co.off[c] : 0;
        hi[k] = c < co.n ? co.off[c + 1] : 0;
    }
    int N = 0;
    for (int w = threadIdx.x; w < tables; w += 64) N = N > ctl->top[w] ? N : ctl->top[w];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const int t = __shfl_xor(N, o);
        N = N > t ? N : t;
    }
    N = __builtin_amdgcn_readfirstlane(N);
    const int quads = (N + 3) / 4;
    // the XCD of a workgroup walks its eighth of the rows: neighbouring rows share elements
    const int per = (quads + 7) / 8, xcd = blockIdx.x & 7, step = gridDim.x >> 3;
    const int stop = per < quads - xcd * per ? per : quads - xcd * per;
    unsigned found = 0;
    int odd = 0;
    // row bounds three steps ahead, table slots two, elements one; past the end, row 0's
    auto row_of = [&](int s) { return s < stop ? 4 * (xcd * per + s) + g : N; };
    auto bounds = [&](int s, int &r0, int &r1) {
        const int i = row_of(s), ic = i < N ? i : 0;
        r0 = row[ic];
        r1 = row[ic + 1];
    };
    auto slots = [&](int s, int (&e)[KC]) {
        const int i = row_of(s), q = line_of(i < N ? i : 0, row, nnz), line = q < 0 ? 0 : q;
#pragma unroll
        for (int k = 0; k < KC; k++) e[k] = table[(int64_t)line * (16 * KC) + l + 16 * k];
    };
    auto elements = [&](const int (&e)[KC], int4 (&q)[KC]) {
#pragma unroll
        for (int k = 0; k < KC; k++) q[k] = e2n[e[k] >= lo[k] && e[k] < hi[k] ? e[k] : 0];
    };
    int s = blockIdx.x >> 3;
    int r0, r1, r0n, r1n, e[KC], en[KC];
    int4 nd[KC];
    bounds(s, r0, r1);
    bounds(s + step, r0n, r1n);
    slots(s, e);
    slots(s + step, en);
    elements(e, nd);
    for (; s < stop; s += step) {
        const int i = row_of(s);
        if (i >= N || r0 < 0 || r1 < r0 || r1 > nnz) {
            if (i < N) odd = 1;
            r0 = r1 = 0;
        }
        const int len = r1 - r0;
        const int key0 = EDGES ? r0 + l : l < len ? col[r0 + l] : 0;
        mf::wave_sync();  // the previous rows' reads
        int L = 0;
#pragma unroll
        for (int k = 0; k < KC; k++) {
            const int4 q = nd[k];
            const int at = q.x == i + 1 ? 0 : q.y == i + 1 ? 1 : q.z == i + 1 ? 2 : q.w == i + 1 ? 3 : -1;
            const bool ok = i < N && e[k] >= lo[k] && e[k] < hi[k] && at >= 0;
            const uint32_t bits = (uint32_t)(__ballot(ok) >> (16 * g)) & 0xFFFFu;
            if (ok) {
                const int r = L + __builtin_popcount(bits & ((1u << l) - 1));
                s_list[g][r] = e[k] << 2 | at;
                s_node[g][r] = q;
            }
            L += __builtin_popcount(bits);
        }
        if (l == 0) found += L;
        // the next steps' loads
#pragma unroll
        for (int k = 0; k < KC; k++) e[k] = en[k];
        elements(e, nd);
        slots(s + 2 * step, en);
        int r0m, r1m;
        bounds(s + 2 * step, r0m, r1m);

        const int nch = (L + SL - 1) / SL, npass = (len + 15) / 16;
        for (int strict = 0; strict < 2; strict++) {
            int matched = 0;
            double dsum = 0.0;        // ela: lane q < 6, the q-th distinct diagonal value
            int dpos = -1;            // this lane's entry when it is the diagonal
            for (int q = l; q < CH * 4; q += 16) s_seen[g][q] = 0;
            for (int pass = 0; pass < npass; pass++) {
                const int p = r0 + l + 16 * pass;
                bool ent = p < r1;
                const int key = EDGES ? p : pass == 0 ? key0 : ent ? col[p] : 0;
                if (strict)  // a repeated column: its first entry takes the blocks
                    for (int t = r0; t < p && ent; t++) ent = col[t] != key;
                double acc[D];
#pragma unroll
                for (int q = 0; q < D; q++) acc[q] = 0.0;
                for (int ch = 0; ch < nch; ch++) {
                    const int Lc = L - ch * SL < SL ? L - ch * SL : SL;
                    if (nch > 1 || pass == 0) {
                        mf::wave_sync();  // the list is written, the previous chunk read
                        // the loads of both of a lane's elements go out together
                        double c[H][4][3], kl[H];
                        mf::ElaCoef kc[H];
                        int4 ids[H];
                        int jj[H];
#pragma unroll
                        for (int h = 0; h < H; h++) {
                            const int sl = l + 16 * h < Lc ? l + 16 * h : 0;
                            const int ej = s_list[g][ch * SL + sl], el = ej >> 2;
                            jj[h] = ej & 3;
                            ids[h] = s_node[g][ch * SL + sl];
                            mf::load_coords(coord, ids[h], c[h]);
                            kl[h] = 1.0;
                            if constexpr (ELA) kc[h] = mf::ela_coef(coef, el);
                            else if (coef) kl[h] = coef[el];
                            if (EDGES) ids[h] = mf::load_four(e2e + ((int64_t)el * 4 + jj[h]) * 4);
                        }
#pragma unroll
                        for (int h = 0; h < H; h++) {
                            const int sl = l + 16 * h, j = jj[h];
                            if (sl >= SL) continue;
                            int4 id = ids[h];
                            if (sl >= Lc) {  // past the chunk: nothing to match
                                s_ids[g][sl] = make_int4(-1, -1, -1, -1);
                                continue;
                            }
                            double gr[4][3];
                            mf::elem_grad(c[h], gr);
                            if (EDGES) {
                                const int w[4] = {id.x, id.y, id.z, id.w};
#pragma unroll
                                for (int q = 0; q < 4; q++) odd |= w[q] >= 0 && (w[q] < r0 || w[q] >= r1);
                            }
                            // the row's vertex first
                            const int idj = j == 0 ? id.x : j == 1 ? id.y : j == 2 ? id.z : id.w;
                            if (j == 1) id.y = id.x;
                            if (j == 2) id.z = id.x;
                            if (j == 3) id.w = id.x;
                            id.x = idj;
                            s_ids[g][sl] = id;
                            T gt[4][3];
#pragma unroll
                            for (int d = 0; d < 3; d++) {
                                const double a = j == 0 ? gr[0][d] : j == 1 ? gr[1][d] : j == 2 ? gr[2][d] : gr[3][d];
                                gt[0][d] = (T)a;
                                gt[1][d] = (T)(j == 1 ? gr[0][d] : gr[1][d]);
                                gt[2][d] = (T)(j == 2 ? gr[0][d] : gr[2][d]);
                                gt[3][d] = (T)(j == 3 ? gr[0][d] : gr[3][d]);
                            }
                            T *o = stage + sl * S;
                            if constexpr (ELA) {
#pragma unroll
                                for (int v = 0; v < 4; v++) {
#pragma unroll
                                    for (int d = 0; d < 3; d++) o[4 * v + d] = gt[v][d];
                                }
                                o[3] = (T)kc[h].cd;
                                o[16] = (T)kc[h].co;
                                o[17] = (T)kc[h].cm;
                            } else {
#pragma unroll
                                for (int v = 0; v < 4; v++) {
                                    const T x = mf::lap_entry(gt[0], gt[v]);
                                    o[v] = PREC == MF_PREC_FP64 && !coef ? x : (T)kl[h] * x;
                                }
                            }
                        }
                        mf::wave_sync();
                    }
                    // bit s of m[k]: the chunk's s-th element holds this entry as its vertex k
                    uint32_t m[4] = {0, 0, 0, 0};
#pragma unroll 8
                    for (int q = 0; q < SL; q++) {
                        const int4 id = s_ids[g][q];
                        m[0] |= (uint32_t)(id.x == key) << q;
                        m[1] |= (uint32_t)(id.y == key) << q;
                        m[2] |= (uint32_t)(id.z == key) << q;
                        m[3] |= (uint32_t)(id.w == key) << q;
                    }
                    if (!ent) m[0] = m[1] = m[2] = m[3] = 0;
                    if (!EDGES) {
#pragma unroll
                        for (int k = 0; k < 4; k++) {
                            matched += __builtin_popcount(m[k]);
                            if (m[k]) atomicOr(&s_seen[g][4 * ch + k], m[k]);
                        }
                    }
                    uint32_t todo = m[1] | m[2] | m[3];
                    if (m[0]) {
                        // the diagonal entry, of every element and of nothing else
                        if (todo || m[0] != (1u << Lc) - 1) odd = 1;
                        dpos = p;
                    }
                    // two elements at a time; the one that an odd count lacks is slot SL, all
                    // zeros, whose +0.0 leave the sums as they are
                    while (todo) {
                        int q[2], v[2];
#pragma unroll
                        for (int u = 0; u < 2; u++) {
                            q[u] = todo ? __builtin_ctz(todo) : SL;
                            todo &= todo - 1;
                            v[u] = (m[1] >> q[u]) & 1 ? 1 : (m[2] >> q[u]) & 1 ? 2 : 3;
                        }
                        if constexpr (ELA) {
                            T ga[2][3], gk[2][3], k0[2], k1[2], k2[2];
#pragma unroll
                            for (int u = 0; u < 2; u++) {
                                const T *o = stage + q[u] * S;
#pragma unroll
                                for (int w = 0; w < 3; w++) {
                                    ga[u][w] = o[w];
                                    gk[u][w] = o[4 * v[u] + w];
                                }
                                k0[u] = o[3];
                                k1[u] = o[16];
                                k2[u] = o[17];
                            }
#pragma unroll
                            for (int u = 0; u < 2; u++) {
                                T bl[9];
                                mf::ela_block(ga[u], gk[u], k0[u], k1[u], k2[u], bl);
#pragma unroll
                                for (int w = 0; w < 9; w++) acc[w] += (double)bl[w];
                            }
                        } else {
                            const T x0 = stage[q[0] * S + v[0]], x1 = stage[q[1] * S + v[1]];
                            acc[0] += (double)x0;
                            acc[0] += (double)x1;
                        }
                    }
                    // the stage is needed for nothing else in this chunk: the diagonal values
                    // of its elements go over their gradients
                    if (nch > 1 ? pass == 0 : pass == npass - 1) {
                        mf::wave_sync();
                        if constexpr (ELA) {
#pragma unroll
                            for (int h = 0; h < H; h++) {
                                const int sl = l + 16 * h;
                                if (sl >= Lc) continue;
                                T *o = stage + sl * S;
                                const T x = o[0], y = o[1], z = o[2], cd = o[3], c1 = o[16], cm = o[17];
                                const T p00 = x * x, p11 = y * y, p22 = z * z;
                                o[0] = p00 * cd + p11 * cm + p22 * cm;
                                o[1] = x * y * c1;
                                o[2] = x * z * c1;
                                o[3] = p00 * cm + p11 * cd + p22 * cm;
                                o[4] = y * z * c1;
                                o[5] = p00 * cm + p11 * cm + p22 * cd;
                            }
                            mf::wave_sync();
                        }
                        if (l < (ELA ? 6 : 1)) {
                            for (int q = 0; q < Lc; q += 4) {
                                T x[4];
#pragma unroll
                                for (int u = 0; u < 4; u++) x[u] = stage[(q + u < Lc ? q + u : SL) * S + l];
#pragma unroll
                                for (int u = 0; u < 4; u++) dsum += (double)x[u];
                            }
                        }
                        mf::wave_sync();
                    }
                }
                if (p < r1 && dpos != p) {
                    double *o = values + (int64_t)p * D;
                    if constexpr (ELA) {
#pragma unroll
                        for (int q = 0; q < 4; q++)
                            *reinterpret_cast<mf::Two *>(o + 2 * q) = mf::Two{acc[2 * q], acc[2 * q + 1]};
                        o[8] = acc[8];
                    } else {
                        o[0] = acc[0];
                    }
                }
            }
            // the diagonal block: six sums hold its nine values
            const uint32_t own = (uint32_t)(__ballot(dpos >= 0) >> (16 * g)) & 0xFFFFu;
            const double v = __shfl(dsum, ELA ? (int)((0x542431210ull >> (4 * (l < 9 ? l : 0))) & 15) : 0, 16);
            if (own) {
                const int pd = __shfl(dpos, __builtin_ctz(own), 16);
                if (EDGES && (own & (own - 1))) odd = 1;  // two entries
                if (l < D) values[(int64_t)pd * D + l] = v;
            }
            if (EDGES) break;
            // a vertex matched by two entries: a column stands twice in the row
#pragma unroll
            for (int o = 8; o > 0; o >>= 1) matched += __shfl_xor(matched, o, 16);
            mf::wave_sync();
            int seen = 0;
            for (int q = l; q < CH * 4; q += 16) seen += __builtin_popcount(s_seen[g][q]);
#pragma unroll
            for (int o = 8; o > 0; o >>= 1) seen += __shfl_xor(seen, o, 16);
            mf::wave_sync();
            if (!__ballot(matched != seen)) break;
            __threadfence();  // the second pass stores some of the first's entries from other lanes
        }
        r0 = r0n;
        r1 = r1n;
        r0n = r0m;
        r1n = r1m;
    }
    if (__ballot(odd) && threadIdx.x == 0) atomicOr(&ctl->odd, 1);
#pragma unroll
    for (int o = 32; o >= 16; o >>= 1) found += __shfl_xor(found, o);
    if (threadIdx.x == 0) ctl->found[blockIdx.x] = (unsigned)found;
    // what no row of a node covers: zeros
    const int first = row[0], last = row[N];
    const int64_t z0 = (int64_t)first * D, z1 = (int64_t)(last > 0 ? last : 0) * D;
    const int64_t total = (int64_t)nnz * D, stride = (int64_t)gridDim.x * 64;
    for (int64_t z = (int64_t)blockIdx.x * 64 + threadIdx.x; z < z0 && z < total; z += stride) values[z] = 0.0;
    for (int64_t z = z1 + (int64_t)blockIdx.x * 64 + threadIdx.x; z < total; z += stride) values[z] = 0.0;
}

// ---- any elemToEdge, entry by entry, for a call that the rows left
//
// Every block is put into a list of its CSR entry, and a lane per entry sums its list in
// ascending order of element and block: what the serial loop gives, whatever the positions are.
// The lists lie in the bytes that held the rows' table. All positions reversed, ela 40^3: 757
// us, with a slot per entry and color instead, in four times the workspace, 768.
constexpr int kListGrid = 256, kListThreads = 512, kSumThreads = 128;

__global__ void __launch_bounds__(kListThreads)
    k_entry_lists(const int *__restrict__ e2e, int nE, int nnz, int *__restrict__ head,
                  int *__restrict__ next, RowsCtl *__restrict__ ctl, int groups)
{
    __shared__ unsigned long long s[kListThreads];
    const bool left = rows_verdict<kListThreads>(ctl, groups, nE, s);
    if (blockIdx.x == 0 && threadIdx.x == 0) ctl->left = left;
    if (!left) return;
    const int64_t stride = (int64_t)gridDim.x * kListThreads;
    for (int64_t t = (int64_t)blockIdx.x * kListThreads + threadIdx.x; t < (int64_t)nE * 4; t += stride) {
        const int4 p = mf::load_four(e2e + t * 4);
        const int at[4] = {p.x, p.y, p.z, p.w};
        int nx[4];
#pragma unroll
        for (int k = 0; k < 4; k++)
            nx[k] = at[k] >= 0 && at[k] < nnz ? atomicExch(head + at[k], (int)(t * 4 + k)) : -1;
        reinterpret_cast<int4 *>(next)[t] = make_int4(nx[0], nx[1], nx[2], nx[3]);
    }
}

template <int OP, int PREC>
__global__ void __launch_bounds__(kSumThreads)
    k_entry_sum(const double *__restrict__ coord, const double *__restrict__ coef,
                double *__restrict__ values, const int4 *__restrict__ e2n, int nnz,
                const int *__restrict__ head, const int *__restrict__ next,
                const RowsCtl *__restrict__ ctl)
{
    if (!ctl->left) return;
    constexpr int D = OP == MF_OP_ELA ? 9 : 1;
    constexpr int SORT = 16;  // blocks sorted at a time
    __shared__ int s_block[SORT][kSumThreads];
    auto sorted = [&](int i) -> int & { return s_block[i][threadIdx.x]; };
    for (int64_t p = (int64_t)blockIdx.x * kSumThreads + threadIdx.x; p < nnz;
         p += (int64_t)gridDim.x * kSumThreads) {
        double acc[D];
#pragma unroll
        for (int r = 0; r < D; r++) acc[r] = 0.0;
        for (int last = -1, n = SORT; n == SORT;) {
            // the SORT lowest blocks past the last one
            n = 0;
            for (int t = head[p]; t >= 0; t = next[t]) {
                if (t <= last || (n == SORT && t > sorted(SORT - 1))) continue;
                int i = n < SORT ? n++ : SORT - 1;
                for (; i > 0 && sorted(i - 1) > t; i--) sorted(i) = sorted(i - 1);
                sorted(i) = t;
            }
            for (int i = 0; i < n; i++) {
                last = sorted(i);
                double b[D];
                elem_block<OP, PREC>(coord, coef, e2n[last >> 4], last >> 4, last & 15, b);
#pragma unroll
                for (int r = 0; r < D; r++) acc[r] += b[r];
            }
        }
#pragma unroll
        for (int r = 0; r < D; r++) values[p * D + r] = acc[r];
    }
}

// ---- the colors, for a call without elemToEdge that the rows left
//
// One launch that takes the colors in turn, and no workgroup waits for another: each owns every
// kLeftGrid-th row, looks through all elements of a color for vertices of its own, and adds their
// blocks once the color is listed, 16 lanes an element. Lanes of one element that share an entry
// (a vertex stands twice in it) add in order, on one lane. Reading the elements kLeftGrid times is
// what it costs; a workgroup a CU is the best (ela 40^3 with one element that repeats a vertex 1,045
// us, 128 of them 1,708, 512 1,272; one launch per color 519, all colors in one workgroup 61,700).
constexpr int kLeftGrid = 256, kLeftThreads = 1024;

template <int OP, int PREC>
__global__ void __launch_bounds__(kLeftThreads)
    k_assemble_left(ColorOffsets co, const double *__restrict__ coord,
                    const double *__restrict__ coef, double *values, const int *__restrict__ row,
                    const int *__restrict__ col, const int4 *__restrict__ e2n, int nnz,
                    const RowsCtl *__restrict__ ctl, int tables, int groups)
{
    constexpr int D = OP == MF_OP_ELA ? 9 : 1;
    constexpr int PER = 4, STEP = PER * kLeftThreads, LIST = 2 * STEP;
    __shared__ unsigned long long s[kLeftThreads];
    if (!rows_verdict<kLeftThreads>(ctl, groups, co.off[co.n], s)) return;
    __shared__ int s_list[LIST], s_n;
    const int w = blockIdx.x, tid = threadIdx.x, l = tid & 15;
    auto own = [&](int v) { return (unsigned)v % kLeftGrid == (unsigned)w; };
    int N = 0;
    for (int t = 0; t < tables; t++) N = N > ctl->top[t] ? N : ctl->top[t];
    for (int64_t v = w + (int64_t)(tid >> 4) * kLeftGrid; v <= N; v += (kLeftThreads / 16) * kLeftGrid) {
        if (v == 0) continue;
        const int64_t a = (int64_t)(row[v - 1] > 0 ? row[v - 1] : 0) * D;
        const int64_t b = (int64_t)(row[v] < nnz ? row[v] : nnz) * D;
        for (int64_t z = a + l; z < b; z += 16) values[z] = 0.0;
    }
    if (tid == 0) s_n = 0;
    for (int c = 0; c < co.n; c++) {
        for (int64_t first = co.off[c]; first < co.off[c + 1]; first += STEP) {
            __syncthreads();  // the list's places are free
#pragma unroll
            for (int u = 0; u < PER; u++) {
                const int64_t e = first + u * kLeftThreads + tid;
                if (e >= co.off[c + 1]) continue;
                const int4 q = e2n[e];
                if (own(q.x) || own(q.y) || own(q.z) || own(q.w)) s_list[atomicAdd(&s_n, 1)] = (int)e;
            }
            __syncthreads();
            const int n = s_n;
            if (n <= LIST - STEP && first + STEP < co.off[c + 1]) continue;
            for (int i = tid >> 4; i < n; i += kLeftThreads / 16) {
                const int e = s_list[i], j = l >> 2, k = l & 3;
                const int4 q = e2n[e];
                const int v[4] = {q.x, q.y, q.z, q.w};
                const int nj = j == 0 ? v[0] : j == 1 ? v[1] : j == 2 ? v[2] : v[3];
                const int nk = k == 0 ? v[0] : k == 1 ? v[1] : k == 2 ? v[2] : v[3];
                int p = nj > 0 && own(nj) ? elem_position(row, col, nullptr, e, nj, nk, l) : -1;
                if (p >= nnz) p = -1;
                bool twice = false;
#pragma unroll
                for (int m = 1; m < 16; m++) twice |= p >= 0 && __shfl_xor(p, m, 16) == p;
                const bool serial = (__ballot(twice) >> (tid & 48)) & 0xFFFFu;
                for (int t = serial ? 0 : l; t < (serial ? 16 : l + 1); t++) {
                    const int pt = serial ? __shfl(p, t, 16) : p;
                    if (pt < 0 || (serial && l > 0)) continue;
                    double b[D];
                    elem_block<OP, PREC>(coord, coef, q, e, t, b);
                    double *o = values + (int64_t)pt * D;
#pragma unroll
                    for (int r = 0; r < D; r++) o[r] += b[r];
                }
            }
            __syncthreads();  // this color's sums, and the list, before the next one's
            if (tid == 0) s_n = 0;
        }
    }
}

// prec_init, src/preconditioner.cc:52-87: the diagonal entry's d values, or zeros. 16 lanes
// per row: they look at 16 columns at once, and the values of a row go through consecutive
// lanes (a lane per row, each zeroing and copying 72 bytes of its own, took 54 us for ela
// 60^3; this takes 16).
__global__ void __launch_bounds__(kBlock)
    k_prec_init(double *__restrict__ prec, const double *__restrict__ values,
                const int *__restrict__ row, const int *__restrict__ col, int N, int dim)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t i = t >> 4;
    const int l = (int)(t & 15), g = (threadIdx.x >> 4) & 3;
    if (i >= N) return;
    int at = -1;
    for (int b = row[i], e = row[i + 1]; b < e; b += 16) {
        const bool hit = b + l < e && col[b + l] - 1 == i;
        const uint32_t bits = (uint32_t)(__ballot(hit) >> (16 * g)) & 0xFFFFu;
        if (bits) {
            at = b + __builtin_ctz(bits);
            break;
        }
    }
    if (l < dim) prec[i * dim + l] = at >= 0 ? values[(int64_t)at * dim + l] : 0.0;
}

__global__ void __launch_bounds__(kBlock) k_prec_inv_lap(double *__restrict__ prec, int N)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < N) prec[i] = 1.0 / prec[i];
}

// prec_inversion for ela: one ela_invert_prec per node (src/preconditioner.cc:44-46).
__global__ void __launch_bounds__(kBlock)
    k_prec_inv_ela(double *__restrict__ prec, const int *__restrict__ row,
                   const int *__restrict__ col, const int *__restrict__ cb, int N,
                   int *__restrict__ singular)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    double blk[9];
    double *p = prec + (int64_t)i * 9;
#pragma unroll
    for (int q = 0; q < 9; q++) blk[q] = p[q];
    int mask = 0;
    if (cb) {
        mask = (cb[i] != 0 ? 1 : 0) | (cb[(int64_t)N + i] != 0 ? 2 : 0) |
               (cb[2 * (int64_t)N + i] != 0 ? 4 : 0);
    }
    bool hasDiag = false;
    for (int l = row[i]; l < row[i + 1]; l++)
        if (col[l] == i + 1) { hasDiag = true; break; }
    const int info = mf::ela_invert_block(blk, mask, hasDiag);
#pragma unroll
    for (int q = 0; q < 9; q++) p[q] = blk[q];
    if (info != 0 && singular) atomicAdd(singular, 1);
}

// Deterministic sum of squares: fixed grid, fixed per-thread stride order, fixed LDS
// tree; then one block folds the partials in index order.
constexpr int kNormBlocks = 1024;

__global__ void __launch_bounds__(kBlock)
    k_sumsq_partial(const double *__restrict__ x, int64_t n, double *__restrict__ part)
{
    __shared__ double s[kBlock];
    double acc = 0.0;
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n;
         i += (int64_t)kNormBlocks * kBlock)
        acc += x[i] * x[i];
    s[threadIdx.x] = acc;
    __syncthreads();
    for (int w = kBlock / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) s[threadIdx.x] += s[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = s[0];
}

__global__ void __launch_bounds__(kBlock) k_sumsq_final(double *__restrict__ part)
{
    __shared__ double s[kBlock];
    double acc = 0.0;
    for (int i = threadIdx.x; i < kNormBlocks; i += kBlock) acc += part[i];
    s[threadIdx.x] = acc;
    __syncthreads();
    for (int w = kBlock / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) s[threadIdx.x] += s[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[0] = s[0];
}

inline unsigned grid_for(int64_t n) { return (unsigned)((n + kBlock - 1) / kBlock); }

// The zero fill and one launch per color.
template <int OP, int PREC>
int launch_colors(const double *coord, const double *coef, double *values, const int *row,
                  const int *col, const int *e2n, const int *e2e, int nbElem, int nbEdges,
                  const int *colorToElem, int nbColors, hipStream_t s)
{
    const int64_t nv = (int64_t)nbEdges * (OP == MF_OP_ELA ? 9 : 1);
    if (nv > 0) {
        hipLaunchKernelGGL(k_fill, dim3(std::min(grid_for(nv), 8192u)), dim3(kBlock), 0, s, values,
                           nv, 0.0);
        MF_CHECK_LAUNCH();
    }
    for (int c = 0; c < nbColors && nbElem > 0; c++) {
        const int first = colorToElem[c], count = colorToElem[c + 1] - first;
        if (count <= 0) continue;
        hipLaunchKernelGGL((k_assemble_color<OP, PREC>), dim3(grid_for((int64_t)count * 16)),
                           dim3(kBlock), 0, s, coord, coef, values, row, col,
                           reinterpret_cast<const int4 *>(e2n), e2e, first, count);
        MF_CHECK_LAUNCH();
    }
    return MF_OK;
}

template <int OP, int PREC, bool EDGES>
void launch_rows_width(int kc, const ColorOffsets &co, const double *coord, const double *coef,
                       double *values, const int *row, const int *col, const int4 *e2n,
                       const int *e2e, int nnz, const int *table, RowsCtl *ctl, int tables,
                       int groups, hipStream_t s)
{
    const dim3 g((unsigned)groups), b(64);
    if (kc == 2)
        hipLaunchKernelGGL((k_assemble_rows<OP, PREC, EDGES, 2>), g, b, 0, s, co, coord, coef,
                           values, row, col, e2n, e2e, nnz, table, ctl, tables);
    else if (kc == 4)
        hipLaunchKernelGGL((k_assemble_rows<OP, PREC, EDGES, 4>), g, b, 0, s, co, coord, coef,
                           values, row, col, e2n, e2e, nnz, table, ctl, tables);
    else
        hipLaunchKernelGGL((k_assemble_rows<OP, PREC, EDGES, 8>), g, b, 0, s, co, coord, coef,
                           values, row, col, e2n, e2e, nnz, table, ctl, tables);
}

// The row-by-row assembly; false when it does not apply (the caller then runs the colors): a
// stream under capture, whose graph would have to own the workspace; no memory for the
// table; element ids that do not leave the bits it needs; or fewer than two entries per
// element, which a pattern of the elements' couplings has (2.4 to 2.5 on cubes and Delaunay
// meshes) and one of, say, the diagonals alone has not. Nor does lap with elemToEdge past
// kLapEdgesElems elements take it: the colors add 8 bytes an entry without a search, and the rows
// read elemToEdge in 16-byte pieces out of order (us, rows and colors: 60^3 396 and 433, 75^3 830
// and 830, 80^3 1,037 and 1,006, 100^3 2,130 and 1,901; ela 90^3 1,639 and 5,574).
constexpr int kLapEdgesElems = 2500000;

template <int OP, int PREC>
bool launch_rows(const double *coord, const double *coef, double *values, const int *row,
                 const int *col, const int *e2n, const int *e2e, int nbElem, int nnz,
                 const int *colorToElem, int nbColors, hipStream_t s, int *status)
{
    if (nbElem >= 1 << 27 || nnz / 2 < nbElem) return false;
    if (OP == MF_OP_LAP && e2e && nbElem > kLapEdgesElems) return false;
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &cap) != hipSuccess || cap != hipStreamCaptureStatusNone) {
        (void)hipGetLastError();
        return false;
    }
    ColorOffsets co;
    co.n = nbColors;
    std::memcpy(co.off, colorToElem, (size_t)(nbColors + 1) * sizeof(int));
    const int kc = nbColors <= 32 ? 2 : nbColors <= 64 ? 4 : 8, width = 16 * kc;
    const int tables = (int)std::min<unsigned>(kTableGrid, grid_for(nbElem));
    // as many workgroups as a CU's LDS holds (ela, FP64: 8; else 16 cover the latency), at
    // most one per four rows of 4 entries, a multiple of 8 (one share per XCD)
    constexpr int kPerCu = OP == MF_OP_ELA && PREC == MF_PREC_FP64 ? 8 : 16;
    static_assert(256 * kPerCu <= kRowsGridMax, "one slot per workgroup");
    const int groups = (int)std::min<int64_t>(256 * kPerCu, ((int64_t)nnz / 16 + 8) / 8 * 8);
    // the control block and the table, whose bytes then hold the lists of k_entry_lists, their
    // heads before it
    const size_t heads = e2e ? (size_t)nnz : 0;
    const size_t slots = std::max((size_t)table_lines(nnz) * width, e2e ? (size_t)nbElem * 16 : 0);
    mf::Workspace ws(mf::Workspace::padded(sizeof(RowsCtl)) + mf::Workspace::padded(heads * sizeof(int)) +
                         mf::Workspace::padded(slots * sizeof(int)), s);
    if (!ws.ok()) return false;
    RowsCtl *ctl = ws.cut<RowsCtl>(1);
    int *head = e2e ? ws.cut<int>(heads) : nullptr, *table = ws.cut<int>(slots);
    const int4 *en = reinterpret_cast<const int4 *>(e2n);
    hipLaunchKernelGGL(k_row_table, dim3((unsigned)tables), dim3(kBlock), 0, s, co, en, row, nbElem,
                       nnz, width, table, head, ctl);
    if (e2e) {
        launch_rows_width<OP, PREC, true>(kc, co, coord, coef, values, row, col, en, e2e, nnz, table,
                                          ctl, tables, groups, s);
        hipLaunchKernelGGL(k_entry_lists, dim3(kListGrid), dim3(kListThreads), 0, s, e2e, nbElem, nnz,
                           head, table, ctl, groups);
        hipLaunchKernelGGL((k_entry_sum<OP, PREC>), dim3(2048), dim3(kSumThreads), 0, s, coord, coef,
                           values, en, nnz, head, table, ctl);
    } else {
        launch_rows_width<OP, PREC, false>(kc, co, coord, coef, values, row, col, en, e2e, nnz, table,
                                           ctl, tables, groups, s);
        hipLaunchKernelGGL((k_assemble_left<OP, PREC>), dim3(kLeftGrid), dim3(kLeftThreads), 0, s, co,
                           coord, coef, values, row, col, en, nnz, ctl, tables, groups);
    }
    *status = hipGetLastError() == hipSuccess ? MF_OK : MF_ERR_HIP;
    return true;
}

template <int OP, int PREC>
int assemble(const double *coord, const double *coef, double *values, const int *row,
             const int *col, const int *e2n, const int *e2e, int nbElem, int nbEdges,
             const int *colorToElem, int nbColors, hipStream_t s)
{
    int status = MF_OK;
    if (nbElem > 0 && nbEdges > 0 &&
        launch_rows<OP, PREC>(coord, coef, values, row, col, e2n, e2e, nbElem, nbEdges, colorToElem,
                              nbColors, s, &status))
        return status;
    return launch_colors<OP, PREC>(coord, coef, values, row, col, e2n, e2e, nbElem, nbEdges,
                                   colorToElem, nbColors, s);
}

}  // namespace

// Scratch of the allocation-free norm (mf_norm_noalloc): the kNormBlocks per-workgroup
// partial sums of k_sumsq_partial, folded in place by k_sumsq_final. 8 KiB, held by
// every GPU the library runs on until the process ends, each GPU its own copy at its own
// address. Host code never passes `scratch` itself (a host-side stand-in): it uses the
// per-device address resolved by hipGetSymbolAddress below.
static __device__ __align__(256) double scratch[kNormBlocks];

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
double *g_scratch[kMaxDevices] = {};

// The device address of `scratch` on the current device `dev`, resolved once per device
// (at mf_device_init, or on the first allocation-free call on a device that skipped it).
int norm_scratch(int dev, double **out)
{
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (dev < 0 || dev >= kMaxDevices) return MF_ERR_HIP;
    if (!g_scratch[dev]) {
        void *p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return MF_ERR_HIP;
        g_scratch[dev] = static_cast<double *>(p);
    }
    *out = g_scratch[dev];
    return MF_OK;
}

}  // namespace

extern "C" const char *mf_status_string(int status)
{
    switch (status) {
    case MF_OK: return "ok";
    case MF_ERR_ARG: return "invalid argument";
    case MF_ERR_IO: return "file missing, truncated or unwritable";
    case MF_ERR_COLORS: return "Not enough colors (more than 128)";
    case MF_ERR_NNZ: return "CSR pattern larger than the nnz capacity";
    case MF_ERR_HIP: return "HIP runtime error or no GPU";
    case MF_ERR_NOMEM: return "allocation failed";
    case MF_ERR_BUDGET: return "request exceeds the HBM budget";
    case MF_ERR_STATE: return "object used in the wrong state";
    default: return "unknown status";
    }
}

extern "C" int mf_version(void) { return 1; }

extern "C" int mf_device_count(void)
{
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess) return MF_ERR_HIP;
    return n;
}

extern "C" int mf_device_init(int device)
{
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || device < 0 || device >= n) return MF_ERR_HIP;
    if (hipSetDevice(device) != hipSuccess) return MF_ERR_HIP;
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, device) != hipSuccess) return MF_ERR_HIP;
    if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0) {
        std::fprintf(stderr, "minifem: device %d is %s, this library is built for gfx950\n",
                     device, prop.gcnArchName);
        return MF_ERR_HIP;
    }
    (void)mf::workspace_pool();  // made here rather than in a call's first use
    double *unused = nullptr;
    return norm_scratch(device, &unused);
}

extern "C" int mf_assembly_ex(const double *coord, const double *coef, double *values,
                              const int *row, const int *col, const int *elemToNode,
                              const int *elemToEdge, int nbElem, int nbEdges,
                              int operatorDim, int operatorID, const int *colorToElem,
                              int nbColors, int precision, void *stream)
{
    if (nbElem < 0 || nbEdges < 0 || nbColors < 0 || nbColors > MF_MAX_COLOR) return MF_ERR_ARG;
    if (!(operatorID == MF_OP_LAP && operatorDim == 1) &&
        !(operatorID == MF_OP_ELA && operatorDim == 9))
        return MF_ERR_ARG;
    if (precision != MF_PREC_FP64 && precision != MF_PREC_MIXED) return MF_ERR_ARG;
    if (!values || (nbElem > 0 && (!coord || !elemToNode || !colorToElem || !row ||
                                   (!elemToEdge && !col))))
        return MF_ERR_ARG;
    if (nbElem > 0 && (colorToElem[0] != 0 || colorToElem[nbColors] != nbElem)) return MF_ERR_ARG;
    for (int c = 0; c < nbColors; c++)
        if (colorToElem[c + 1] < colorToElem[c]) return MF_ERR_ARG;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    const bool fp64 = precision == MF_PREC_FP64;
    if (operatorID == MF_OP_LAP)
        return fp64 ? assemble<MF_OP_LAP, MF_PREC_FP64>(coord, coef, values, row, col, elemToNode,
                                                        elemToEdge, nbElem, nbEdges, colorToElem,
                                                        nbColors, s)
                    : assemble<MF_OP_LAP, MF_PREC_MIXED>(coord, coef, values, row, col, elemToNode,
                                                         elemToEdge, nbElem, nbEdges, colorToElem,
                                                         nbColors, s);
    return fp64 ? assemble<MF_OP_ELA, MF_PREC_FP64>(coord, coef, values, row, col, elemToNode,
                                                    elemToEdge, nbElem, nbEdges, colorToElem,
                                                    nbColors, s)
                : assemble<MF_OP_ELA, MF_PREC_MIXED>(coord, coef, values, row, col, elemToNode,
                                                     elemToEdge, nbElem, nbEdges, colorToElem,
                                                     nbColors, s);
}

extern "C" int mf_assembly(const double *coord, double *values, const int *row,
                           const int *col, const int *elemToNode, const int *elemToEdge,
                           int nbElem, int nbEdges, int operatorDim, int operatorID,
                           const int *colorToElem, int nbColors, void *stream)
{
    return mf_assembly_ex(coord, nullptr, values, row, col, elemToNode, elemToEdge, nbElem,
                          nbEdges, operatorDim, operatorID, colorToElem, nbColors,
                          MF_PREC_FP64, stream);
}

extern "C" int mf_prec_init(double *prec, const double *values, const int *row,
                            const int *col, int nbNodes, int operatorDim, void *stream)
{
    if (nbNodes < 0 || (operatorDim != 1 && operatorDim != 9)) return MF_ERR_ARG;
    if (nbNodes == 0) return MF_OK;
    if (!prec || !values || !row || !col) return MF_ERR_ARG;
    hipLaunchKernelGGL(k_prec_init, dim3(grid_for((int64_t)nbNodes * 16)), dim3(kBlock), 0,
                       reinterpret_cast<hipStream_t>(stream), prec, values, row, col, nbNodes,
                       operatorDim);
    MF_CHECK_LAUNCH();
    return MF_OK;
}

extern "C" int mf_prec_inversion(double *prec, const int *row, const int *col,
                                 const int *checkBounds, int nbNodes, int operatorID,
                                 int *singular, void *stream)
{
    if (nbNodes < 0 || (operatorID != MF_OP_LAP && operatorID != MF_OP_ELA)) return MF_ERR_ARG;
    if (nbNodes == 0) return MF_OK;
    if (!prec) return MF_ERR_ARG;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    if (operatorID == MF_OP_LAP) {
        hipLaunchKernelGGL(k_prec_inv_lap, dim3(grid_for(nbNodes)), dim3(kBlock), 0, s, prec,
                           nbNodes);
    } else {
        if (!row || !col) return MF_ERR_ARG;
        hipLaunchKernelGGL(k_prec_inv_ela, dim3(grid_for(nbNodes)), dim3(kBlock), 0, s, prec,
                           row, col, checkBounds, nbNodes, singular);
    }
    MF_CHECK_LAUNCH();
    return MF_OK;
}

extern "C" int mf_norm(const double *x, int64_t n, double *result, void *stream)
{
    if (n < 0 || !result || (n > 0 && !x)) return MF_ERR_ARG;
    if (n == 0) { *result = 0.0; return MF_OK; }
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    double *part = nullptr;
    if (hipMallocAsync(reinterpret_cast<void **>(&part), kNormBlocks * sizeof(double), s) !=
        hipSuccess)
        return MF_ERR_NOMEM;
    hipLaunchKernelGGL(k_sumsq_partial, dim3(kNormBlocks), dim3(kBlock), 0, s, x, n, part);
    hipLaunchKernelGGL(k_sumsq_final, dim3(1), dim3(kBlock), 0, s, part);
    double h = 0.0;
    hipError_t e1 = hipMemcpyAsync(&h, part, sizeof(double), hipMemcpyDeviceToHost, s);
    hipError_t e2 = hipStreamSynchronize(s);
    hipError_t e3 = hipFreeAsync(part, s);
    hipError_t e4 = hipStreamSynchronize(s);
    if (e1 != hipSuccess || e2 != hipSuccess || e3 != hipSuccess || e4 != hipSuccess)
        return MF_ERR_HIP;
    *result = __builtin_sqrt(h);
    return MF_OK;
}

extern "C" int mf_norm_noalloc(const double *x, int64_t n, double *result, void *stream)
{
    if (n < 0 || !result || (n > 0 && !x)) return MF_ERR_ARG;
    if (n == 0) { *result = 0.0; return MF_OK; }
    int dev = 0;
    double *part = nullptr;
    if (hipGetDevice(&dev) != hipSuccess) return MF_ERR_HIP;
    const int st = norm_scratch(dev, &part);
    if (st != MF_OK) return st;
    // the same two kernels and order as mf_norm: every workgroup writes its own partial
    // (zero when it sums nothing), so nothing in the scratch has to be cleared first
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    hipLaunchKernelGGL(k_sumsq_partial, dim3(kNormBlocks), dim3(kBlock), 0, s, x, n, part);
    hipLaunchKernelGGL(k_sumsq_final, dim3(1), dim3(kBlock), 0, s, part);
    double h = 0.0;
    if (hipGetLastError() != hipSuccess ||
        hipMemcpyAsync(&h, part, sizeof(double), hipMemcpyDeviceToHost, s) != hipSuccess ||
        hipStreamSynchronize(s) != hipSuccess)
        return MF_ERR_HIP;
    *result = __builtin_sqrt(h);
    return MF_OK;
}
