// Device-side mesh setup, bit-exact twins of the host setup (src/matrix.cc:25-91,
// DC_create_nodeToElem as called at src/main.cc:243-250, and the greedy coloring of
// src/coloring.cc:46-109): for meshes that arrive at a server already resident on the GPU.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cstdint>

#include "device_common.h"
#include "minifem.h"

namespace {

// Each vertex's turn at its node (in any order) and the nodes' counts.
__global__ void k_count_nodes(const int *__restrict__ e2n, int64_t n4, int N, int *__restrict__ cnt,
                              int *__restrict__ turn, int *__restrict__ bad)
{
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= n4) return;
    const int v = e2n[q] - 1;
    if (v < 0 || v >= N) {
        *bad = 1;
        return;
    }
    turn[q] = atomicAdd(cnt + v, 1);
}

__global__ void k_fill_nodes(const int *__restrict__ e2n, int64_t n4, const int *__restrict__ index,
                             const int *__restrict__ turn, int *__restrict__ value)
{
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= n4) return;
    value[index[e2n[q] - 1] + turn[q]] = (int)(q >> 2);
}

// Nodes with up to kListElems elements get 16 lanes, each with up to kListOwn of the
// elements; longer lists go through one lane.
constexpr int kListOwn = 4, kListElems = 16 * kListOwn;

// Each node's element list in ascending order, by each element's rank in its list.
__global__ void __launch_bounds__(256)
k_sort_lists(const int *__restrict__ index, int N, int *__restrict__ value)
{
    __shared__ int s_list[16][kListElems + 1];
    const int l = threadIdx.x & 15, g = threadIdx.x >> 4;
    const int i = blockIdx.x * 16 + g;
    if (i >= N) return;
    const int b = index[i], L = index[i + 1] - b;
    if (L > kListElems) {
        if (l > 0) return;
        for (int a = b + 1; a < b + L; a++) {
            const int x = value[a];
            int c = a - 1;
            while (c >= b && value[c] > x) {
                value[c + 1] = value[c];
                c--;
            }
            value[c + 1] = x;
        }
        return;
    }
    int own[kListOwn], rank[kListOwn];
#pragma unroll
    for (int h = 0; h < kListOwn; h++) {
        const int j = l + 16 * h;
        own[h] = j < L ? value[b + j] : 0;
        rank[h] = 0;
        if (j < L) s_list[g][j] = own[h];
    }
    mf::wave_sync();
    for (int q = 0; q < L; q++) {
        const int x = s_list[g][q];
#pragma unroll
        for (int h = 0; h < kListOwn; h++)
            rank[h] += x < own[h] || (x == own[h] && q < l + 16 * h);
    }
#pragma unroll
    for (int h = 0; h < kListOwn; h++)
        if (l + 16 * h < L) value[b + rank[h]] = own[h];
}

// Row i in first-seen order: node i's elements ascending, each element's vertices in
// order, a column appended when not seen yet (src/matrix.cc:67-85). With out == nullptr
// only the length is counted.
__device__ int row_columns(int i, const int *__restrict__ index, const int *__restrict__ value,
                           const int *__restrict__ e2n, int *out, int cap)
{
    int len = 0;
    for (int j = index[i]; j < index[i + 1]; j++) {
        const int el = value[j];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int c = e2n[(int64_t)el * 4 + k];  // 1-based, as col[] stores it
            bool seen = false;
            if (out) {
                for (int q = 0; q < len; q++) seen |= out[q] == c;
            } else {
                // count pass: compare against the earlier vertices of earlier elements
                for (int j2 = index[i]; j2 <= j && !seen; j2++) {
                    const int el2 = value[j2];
                    const int kmax = j2 == j ? k : 4;
                    for (int k2 = 0; k2 < kmax; k2++) seen |= e2n[(int64_t)el2 * 4 + k2] == c;
                }
            }
            if (!seen) {
                if (out && len < cap) out[len] = c;
                len++;
            }
        }
    }
    return len;
}

// The rows' lengths and, for k_row_fill, which vertices of each row's elements are new: bit k
// of flags[j] for vertex k of incidence j. 16 lanes per row, each with up to kListOwn of its
// elements, all of which they look through in LDS. (A lane per row that looked through the
// lists in memory took 1.2 ms for a 50^3 cube's lengths and 0.26 for its columns; these two
// take 83 and 20 us.)
__global__ void __launch_bounds__(256)
k_row_len(const int *__restrict__ index, const int *__restrict__ value, const int *__restrict__ e2n,
          int N, int *__restrict__ len, uint8_t *__restrict__ flags)
{
    __shared__ int4 s_elem[16][kListElems + 1];  // rows start on different banks
    const int l = threadIdx.x & 15, g = threadIdx.x >> 4;
    const int i = blockIdx.x * 16 + g;
    if (i >= N) return;
    const int b = index[i], L = index[i + 1] - b;
    if (L > kListElems) {  // more than the lanes hold: one lane through the lists in memory
        if (l == 0) len[i] = row_columns(i, index, value, e2n, nullptr, 0);
        return;
    }
    int4 own[kListOwn];
    uint32_t fresh[kListOwn];
#pragma unroll
    for (int h = 0; h < kListOwn; h++) {
        const int j = l + 16 * h;
        own[h] = j < L ? mf::load_four(e2n + (int64_t)value[b + j] * 4) : make_int4(0, 0, 0, 0);
        if (j < L) s_elem[g][j] = own[h];
        const int4 v = own[h];
        fresh[h] = 1u | (v.y != v.x) << 1 | (v.z != v.x && v.z != v.y) << 2 |
                   (v.w != v.x && v.w != v.y && v.w != v.z) << 3;
    }
    mf::wave_sync();
    for (int q = 0; q < L; q++) {
        const int4 c = s_elem[g][q];
#pragma unroll
        for (int h = 0; h < kListOwn; h++) {
            if (16 * h >= L) break;
            const int4 v = own[h];
            const uint32_t same = (uint32_t)(v.x == c.x || v.x == c.y || v.x == c.z || v.x == c.w) |
                                  (uint32_t)(v.y == c.x || v.y == c.y || v.y == c.z || v.y == c.w) << 1 |
                                  (uint32_t)(v.z == c.x || v.z == c.y || v.z == c.z || v.z == c.w) << 2 |
                                  (uint32_t)(v.w == c.x || v.w == c.y || v.w == c.z || v.w == c.w) << 3;
            if (q < l + 16 * h) fresh[h] &= ~same;
        }
    }
    int n = 0;
#pragma unroll
    for (int h = 0; h < kListOwn; h++) {
        const int j = l + 16 * h;
        if (j >= L) continue;
        flags[b + j] = (uint8_t)fresh[h];
        n += __builtin_popcount(fresh[h]);
    }
#pragma unroll
    for (int o = 8; o > 0; o >>= 1) n += __shfl_xor(n, o, 16);
    if (l == 0) len[i] = n;
}

__global__ void __launch_bounds__(256)
k_row_fill(const int *__restrict__ index, const int *__restrict__ value, const int *__restrict__ e2n,
           const int *__restrict__ row, int N, const uint8_t *__restrict__ flags, int *__restrict__ col)
{
    const int l = threadIdx.x & 15;
    const int i = blockIdx.x * 16 + (threadIdx.x >> 4);
    if (i >= N) return;
    const int b = index[i], L = index[i + 1] - b;
    if (L > kListElems) {
        if (l == 0)
            row_columns(i, index, value, e2n, col + row[i], row[i + 1] - row[i]);
        return;
    }
    int at = row[i];
    for (int j0 = 0; j0 < L; j0 += 16) {
        const int j = j0 + l;
        const uint32_t f = j < L ? flags[b + j] : 0u;
        const int n = __builtin_popcount(f);
        int scan = n;  // inclusive, over the row's lanes
#pragma unroll
        for (int o = 1; o < 16; o <<= 1) {
            const int t = __shfl_up(scan, o, 16);
            if (l >= o) scan += t;
        }
        int p = at + scan - n;
        if (f) {
            const int4 q = mf::load_four(e2n + (int64_t)value[b + j] * 4);
            const int v[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
            for (int k = 0; k < 4; k++)
                if ((f >> k) & 1) col[p++] = v[k];
        }
        at += __shfl(scan, 15, 16);
    }
}

// elemToEdge (src/matrix.cc:25-52): for each element, the 16 CSR positions of its (i, j)
// vertex pairs, row-major. A lane looks through one row for the four columns of an element,
// four entries at a time.
__global__ void k_elem_to_edge(const int *__restrict__ row, const int *__restrict__ col,
                               const int *__restrict__ e2n, int nE, int *__restrict__ e2e)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (int64_t)nE * 4) return;
    const int4 v = mf::load_four(e2n + (t >> 2) * 4);
    const int i = (int)(t & 3), a = (i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w) - 1;
    int4 p = make_int4(-1, -1, -1, -1);
    int left = 4;
    for (int q0 = row[a], e = row[a + 1]; q0 < e && left > 0; q0 += 4) {
        int c[4];
#pragma unroll
        for (int u = 0; u < 4; u++) c[u] = col[q0 + u < e ? q0 + u : e - 1];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int q = q0 + u < e ? q0 + u : e - 1;
            if (p.x < 0 && c[u] == v.x) { p.x = q; left--; }
            if (p.y < 0 && c[u] == v.y) { p.y = q; left--; }
            if (p.z < 0 && c[u] == v.z) { p.z = q; left--; }
            if (p.w < 0 && c[u] == v.w) { p.w = q; left--; }
        }
    }
    *reinterpret_cast<mf::Four *>(e2e + t * 4) = mf::Four{p.x, p.y, p.z, p.w};
}

inline dim3 grid_for(int64_t n, int bt) { return dim3((unsigned)((n + bt - 1) / bt)); }

// ---- greedy first-fit coloring (src/coloring.cc:46-81), exact, level by level ----
//
// Element e takes the lowest color that no lower-index element sharing a node with it
// holds. At node v the elements are listed in ascending order (nodeToElem), so e's color
// depends on v's list only up to e. Once every element before e in each of its nodes'
// lists is colored, e's color is fixed: the first color missing from the OR of its nodes'
// color masks, each mask holding the colors of the elements colored at that node so far
// (the host scan's per-node masks). Elements become ready in levels: level 0 has no lower
// neighbour at all, and an element is ready once its predecessor at each node is colored.
// Two elements ready in the same level never share a node (the later one's predecessor
// at a shared node would be uncolored), so one level colors its elements in parallel, and
// the result is the sequential scan's, bit for bit. The 100^3 cube needs 2,750 levels of
// about 2,100 elements each, one launch per level.

// Per element: at each distinct node, the element that follows it in the node's list
// (-1: none), and the number of distinct nodes where an element precedes it.
__global__ void k_color_links(const int4 *__restrict__ e2n, int nE, const int *__restrict__ index,
                              const int *__restrict__ value, int4 *__restrict__ next,
                              int *__restrict__ npre)
{
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= nE) return;
    const int4 q = e2n[e];
    const int v[4] = {q.x - 1, q.y - 1, q.z - 1, q.w - 1};
    int nx[4] = {-1, -1, -1, -1}, np = 0;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        bool dup = false;
#pragma unroll
        for (int j = 0; j < k; j++) dup |= v[j] == v[k];
        if (dup) continue;  // a node the element repeats counts once
        const int b = index[v[k]], en = index[v[k] + 1];
        int lo = b, hi = en;  // first entry >= e
        while (lo < hi) {
            const int m = (lo + hi) >> 1;
            if (value[m] < e) lo = m + 1;
            else hi = m;
        }
        int last = lo;  // past e's entries (two when the element repeats the node)
        while (last < en && value[last] == e) last++;
        np += lo > b;
        if (last < en) nx[k] = value[last];
    }
    next[e] = make_int4(nx[0], nx[1], nx[2], nx[3]);
    npre[e] = np;
}

__global__ void k_color_seed(const int *__restrict__ npre, int nE, int *__restrict__ front,
                             int *__restrict__ count)
{
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e < nE && npre[e] == 0) front[atomicAdd(count, 1)] = e;
}

// One level per launch: launches on one stream run in order, which orders the levels, and
// each level spreads over kLevelBlocks workgroups (a level's cost is its chain of memory
// round trips, so more CUs keep more of them in flight). Level L reads its list from
// front[L & 1] and its length from counts[L % 3], appends the next level to
// front[(L + 1) & 1] and counts[(L + 1) % 3], and clears counts[(L + 2) % 3] for level L + 1.
// status: [1] elements colored, [2] nonzero when an element needs more than MF_MAX_COLOR
// colors.
constexpr int kLevelThreads = 256, kLevelBlocks = 32, kLevelsPerCheck = 64;

__global__ void __launch_bounds__(kLevelThreads)
k_color_level(const int4 *__restrict__ e2n, const int4 *__restrict__ next,
              const int *__restrict__ npre, int *__restrict__ cnt, const int *__restrict__ cur,
              int *__restrict__ nxt, int *__restrict__ counts, int L, ulonglong2 *masks,
              int *__restrict__ part, int *__restrict__ status)
{
    const int n = counts[L % 3];
    const int gt = blockIdx.x * kLevelThreads + threadIdx.x;
    if (gt == 0) {
        counts[(L + 2) % 3] = 0;
        if (n > 0) atomicAdd(status + 1, n);
    }
    for (int i = gt; i < n; i += kLevelBlocks * kLevelThreads) {
        const int e = cur[i];
        const int4 q = e2n[e], nq = next[e];
        const int v[4] = {q.x - 1, q.y - 1, q.z - 1, q.w - 1};
        const int c[4] = {nq.x, nq.y, nq.z, nq.w};
        ulonglong2 m[4];
        int old[4], np[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            m[k] = masks[v[k]];
            old[k] = c[k] >= 0 ? atomicAdd(cnt + c[k], 1) : 0;
            np[k] = c[k] >= 0 ? npre[c[k]] : 0;
        }
        const uint64_t lo = m[0].x | m[1].x | m[2].x | m[3].x;
        const uint64_t hi = m[0].y | m[1].y | m[2].y | m[3].y;
        int color = ~lo ? __builtin_ctzll(~lo) : ~hi ? 64 + __builtin_ctzll(~hi) : 128;
        if (color >= MF_MAX_COLOR) {
            atomicOr(status + 2, 1);
            color = MF_MAX_COLOR - 1;  // keeps the levels going; the call fails
        }
        part[e] = color;
        const uint64_t blo = color < 64 ? 1ull << color : 0ull;
        const uint64_t bhi = color < 64 ? 0ull : 1ull << (color - 64);
        // no other element of this level holds these nodes (a repeated node gets the same
        // value twice)
#pragma unroll
        for (int k = 0; k < 4; k++) masks[v[k]] = make_ulonglong2(m[k].x | blo, m[k].y | bhi);
#pragma unroll
        for (int k = 0; k < 4; k++) {
            // no successor at this node, or c[k] still waits for another node
            if (c[k] < 0 || old[k] + 1 != np[k]) continue;
            nxt[atomicAdd(counts + (L + 1) % 3, 1)] = c[k];
        }
    }
}

// The same colors without a launch per level, for meshes that stay within 60 of them. An
// element's word collects the masks of its nodes (bits 0-59) and who has delivered them (bit
// 60 + k: its k-th vertex's predecessor has, or there is none). An element that takes color c
// adds it to the mask of each of its nodes, one atomic that returns the mask before, and
// hands that mask with its own color to the node's next element, one atomic that returns
// what the others have handed it. Whoever delivers last has the whole word, hence the color,
// in the returned value, and goes on with that element: two round trips per element of the
// chain, no element is looked at before it is ready, and nobody waits for anybody.
//
// A wave keeps its ready elements in LDS, with their vertices and successors, which it loads
// along with the second atomic. It stops after kChainHops elements of its longest chain, and
// the ready ones go to the next launch's list, which spreads them over all waves again: on
// average an element readies one other, so a few waves' queues grow while most run dry. 50^3
// and 100^3 cubes, the whole coloring: 16.5 and 35 ms level by level, 5.1 and 21 ms with 64
// hops a launch, 3.7 and 13.9 with 32, 3.8 and 11.0 with 20, 3.9 and 10.8 with 16.
constexpr int kChainColors = 60, kChainHops = 20, kChainWaves = 1792, kChainQueue = 128;
constexpr int kChainsPerCheck = 8;
// More elements than this at one node, and greedy coloring may need more than 60 colors
// (Kuhn cubes: 24 elements at a node, 30 colors): then level by level from the start.
constexpr int kChainValence = 40;
constexpr uint64_t kChainMask = (1ull << kChainColors) - 1;

// Per element: the element after it at each distinct node, 4 times its index plus the node's
// place in it (-1: none); its word with the vertices that have no predecessor delivered; the
// elements with none at all go to the first list. status[3]: some node has too many elements.
__global__ void k_chain_links(const int4 *__restrict__ e2n, int nE, const int *__restrict__ index,
                              const int *__restrict__ value, int4 *__restrict__ next,
                              unsigned long long *__restrict__ word, int *__restrict__ front,
                              int *__restrict__ count, int *__restrict__ status)
{
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= nE) return;
    const int4 q = e2n[e];
    const int v[4] = {q.x, q.y, q.z, q.w};
    int nx[4] = {-1, -1, -1, -1};
    uint64_t w = 0;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        bool dup = false;
#pragma unroll
        for (int j = 0; j < k; j++) dup |= v[j] == v[k];
        const int b = index[v[k] - 1], en = index[v[k]];
        if (en - b > kChainValence) status[3] = 1;
        int lo = b, hi = en;  // first entry >= e
        while (lo < hi) {
            const int m = (lo + hi) >> 1;
            if (value[m] < e) lo = m + 1;
            else hi = m;
        }
        if (dup || lo == b) w |= 1ull << (kChainColors + k);
        if (dup) continue;  // a node the element repeats counts once
        int last = lo;
        while (last < en && value[last] == e) last++;
        if (last < en) {
            const int s = value[last];
            const int4 t = e2n[s];
            nx[k] = s << 2 | (t.x == v[k] ? 0 : t.y == v[k] ? 1 : t.z == v[k] ? 2 : 3);
        }
    }
    next[e] = make_int4(nx[0], nx[1], nx[2], nx[3]);
    word[e] = w;
    if (w >> kChainColors == 15) front[atomicAdd(count, 1)] = e;
}

__global__ void __launch_bounds__(64)
k_color_chains(const int4 *__restrict__ e2n, const int4 *__restrict__ next,
               unsigned long long *word, unsigned long long *mask, const int *__restrict__ cur,
               int *__restrict__ nxt, int *__restrict__ counts, int L, int *__restrict__ part,
               int *__restrict__ status)
{
    __shared__ int q_elem[2][kChainQueue];
    __shared__ int4 q_node[2][kChainQueue], q_next[2][kChainQueue];
    __shared__ unsigned long long q_word[2][kChainQueue];
    const int lane = threadIdx.x;
    const int n = counts[L % 3];
    if (blockIdx.x == 0 && lane == 0) counts[(L + 2) % 3] = 0;
    if (status[3]) return;  // for the levels
    int colored = 0, fill = 0;
    bool over = false;
    // colors element e of every lane that is on; the elements that became ready go to
    // queue[to], or past its end to the next launch's list
    auto color = [&](bool on, int e, int4 nd, int4 sc, uint64_t w, int to) {
        const int v[4] = {nd.x, nd.y, nd.z, nd.w}, s[4] = {sc.x, sc.y, sc.z, sc.w};
        const uint64_t open = ~w & kChainMask;
        const int c = open ? __builtin_ctzll(open) : kChainColors - 1;
        const uint64_t bit = 1ull << c;
        uint64_t m[4] = {0, 0, 0, 0}, old[4] = {~0ull, ~0ull, ~0ull, ~0ull};
        // the successors' records as scalars (an array of vectors stays in scratch)
        int nx[4], ny[4], nz[4], nw[4], sx[4], sy[4], sz[4], sw[4];
        if (on) {
            over |= !open;
            colored++;
            part[e] = c;
#pragma unroll
            for (int k = 0; k < 4; k++)
                if (s[k] >= 0) m[k] = atomicOr(mask + (v[k] - 1), bit);
        }
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int t = on && s[k] >= 0 ? s[k] >> 2 : e;
            const int4 a = e2n[t], b = next[t];
            nx[k] = a.x; ny[k] = a.y; nz[k] = a.z; nw[k] = a.w;
            sx[k] = b.x; sy[k] = b.y; sz[k] = b.z; sw[k] = b.w;
        }
        if (on) {
#pragma unroll
            for (int k = 0; k < 4; k++) {
                if (s[k] < 0) continue;
                m[k] |= bit | 1ull << (kChainColors + (s[k] & 3));
                old[k] = atomicOr(word + (s[k] >> 2), m[k]);
            }
        }
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const bool ready = on && s[k] >= 0 && old[k] >> kChainColors != 15 &&
                               (old[k] | m[k]) >> kChainColors == 15;
            const uint64_t b = __ballot(ready);
            if (ready) {
                const int at = fill + __builtin_popcountll(b & ((1ull << lane) - 1));
                if (at < kChainQueue) {
                    q_elem[to][at] = s[k] >> 2;
                    q_node[to][at] = make_int4(nx[k], ny[k], nz[k], nw[k]);
                    q_next[to][at] = make_int4(sx[k], sy[k], sz[k], sw[k]);
                    q_word[to][at] = old[k] | m[k];
                } else {
                    nxt[atomicAdd(counts + (L + 1) % 3, 1)] = s[k] >> 2;
                }
            }
            fill += __builtin_popcountll(b);
        }
    };
    // this wave's share of the list
    const int per = (n + gridDim.x - 1) / gridDim.x;
    const int b0 = blockIdx.x * per, b1 = b0 + per < n ? b0 + per : n;
    for (int b = b0; b < b1; b += 64) {
        const bool on = b + lane < b1;
        const int e = on ? cur[b + lane] : 0;
        color(on, e, e2n[e], next[e], word[e], 0);
    }
    int now = 0;
    for (int hop = 1; hop < kChainHops && fill > 0; hop++, now ^= 1) {
        const int have = fill < kChainQueue ? fill : kChainQueue;
        fill = 0;
        mf::wave_sync();
        for (int b = 0; b < have; b += 64) {
            const bool on = b + lane < have;
            const int i = on ? b + lane : 0;
            color(on, q_elem[now][i], q_node[now][i], q_next[now][i], q_word[now][i], now ^ 1);
        }
    }
    const int have = fill < kChainQueue ? fill : kChainQueue;
    mf::wave_sync();
    for (int b = 0; b < have; b += 64)
        if (b + lane < have) nxt[atomicAdd(counts + (L + 1) % 3, 1)] = q_elem[now][b + lane];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) colored += __shfl_xor(colored, o);
    if (lane == 0 && colored) atomicAdd(status + 1, colored);
    if (__ballot(over) && lane == 0) atomicOr(status + 2, 1);
}

__global__ void k_iota(int *__restrict__ a, int n)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) a[i] = i;
}

// Elements sorted by (color, index): position i holds element order[i], whose new index
// is i (the stable counting sort of src/coloring.cc:27-42 and DC_create_permutation).
// Each color's first position goes to colorToElem.
__global__ void k_color_perm(const int *__restrict__ key, const int *__restrict__ order, int nE,
                             int *__restrict__ perm, int *__restrict__ c2e)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nE) return;
    perm[order[i]] = i;
    if (i == 0 || key[i] != key[i - 1]) c2e[key[i]] = i;
    if (i == nE - 1) c2e[key[i] + 1] = nE;
}

__global__ void k_check_perm(const int *__restrict__ perm, int n, int *__restrict__ bad)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n && (perm[i] < 0 || perm[i] >= n)) atomicOr(bad, 1);
}

// row i of src to row perm[i] of dst
template <typename T>
__global__ void k_permute_rows(const T *__restrict__ src, const int *__restrict__ perm, int n,
                               int dim, T *__restrict__ dst)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (int64_t)n * dim) return;
    const int64_t i = t / dim, d = t - i * dim;
    dst[(int64_t)perm[i] * dim + d] = src[t];
}

using mf::Workspace;

struct DevBuf {
    void *p = nullptr;
    ~DevBuf() { (void)hipFree(p); }
    template <typename T>
    T *get() const { return static_cast<T *>(p); }
};

// Waits for the stream when it goes out of scope: declared after the DevBufs of a call, it
// runs before they free their memory, on every return path.
struct StreamDrain {
    hipStream_t s;
    ~StreamDrain() { (void)hipStreamSynchronize(s); }
};

inline int dev_alloc(DevBuf &b, size_t bytes)
{
    return mf::device_alloc(&b.p, std::max<size_t>(bytes, 16));
}

// The device arrays of one coloring.
struct ColoringWork {
    const int4 *e2n;
    int nE, N;
    int *index, *value;  // nodeToElem
    int4 *next;
    int *front[2];
    ulonglong2 *masks;            // 16 bytes a node; the chains use 8 of them
    unsigned long long *words;    // 8 bytes an element; the levels keep two counts there
    int *counts, *status, *part;
};

int read_ints(int *dst, const int *src, int n, hipStream_t s)
{
    return hipMemcpyAsync(dst, src, n * sizeof(int), hipMemcpyDeviceToHost, s) == hipSuccess &&
                   hipStreamSynchronize(s) == hipSuccess
               ? MF_OK
               : MF_ERR_HIP;
}

// Colors by chains; *done stays false for a mesh that needs the levels (more than
// kChainColors colors, or too many elements at a node to expect fewer).
int color_by_chains(const ColoringWork &w, hipStream_t s, bool *done)
{
    unsigned long long *mask = reinterpret_cast<unsigned long long *>(w.masks);
    if (hipMemsetAsync(mask, 0, (size_t)w.N * sizeof(*mask), s) != hipSuccess ||
        hipMemsetAsync(w.counts, 0, 7 * sizeof(int), s) != hipSuccess)
        return MF_ERR_HIP;
    hipLaunchKernelGGL(k_chain_links, grid_for(w.nE, 256), dim3(256), 0, s, w.e2n, w.nE, w.index,
                       w.value, w.next, w.words, w.front[0], w.counts, w.status);
    int L = 0, h[7] = {0, 0, 0, 0, 0, 0, 0};
    do {
        if (L > w.nE) return MF_ERR_ARG;  // every launch colors an element or is the last
        for (int b = 0; b < kChainsPerCheck; b++, L++)
            hipLaunchKernelGGL(k_color_chains, dim3(kChainWaves), dim3(64), 0, s, w.e2n, w.next,
                               w.words, mask, w.front[L & 1], w.front[(L + 1) & 1], w.counts, L,
                               w.part, w.status);
        if (hipGetLastError() != hipSuccess || read_ints(h, w.counts, 7, s) != MF_OK) return MF_ERR_HIP;
        if (h[3 + 2] || h[3 + 3]) return MF_OK;  // for the levels
    } while (h[L % 3] > 0);
    if (h[3 + 1] != w.nE) return MF_ERR_ARG;  // not every element became ready
    *done = true;
    return MF_OK;
}

int color_by_levels(const ColoringWork &w, hipStream_t s)
{
    int *npre = reinterpret_cast<int *>(w.words), *cnt = npre + w.nE;
    if (hipMemsetAsync(cnt, 0, (size_t)w.nE * sizeof(int), s) != hipSuccess ||
        hipMemsetAsync(w.masks, 0, (size_t)w.N * sizeof(ulonglong2), s) != hipSuccess ||
        hipMemsetAsync(w.counts, 0, 7 * sizeof(int), s) != hipSuccess)
        return MF_ERR_HIP;
    hipLaunchKernelGGL(k_color_links, grid_for(w.nE, 256), dim3(256), 0, s, w.e2n, w.nE, w.index,
                       w.value, w.next, npre);
    hipLaunchKernelGGL(k_color_seed, grid_for(w.nE, 256), dim3(256), 0, s, npre, w.nE, w.front[0],
                       w.counts);
    if (hipGetLastError() != hipSuccess) return MF_ERR_HIP;
    // levels in batches of kLevelsPerCheck launches, then a look at the next level's
    // length: launches past the last level find an empty list and return at once
    int L = 0, remaining = 1;
    while (remaining > 0) {
        if (L > w.nE) return MF_ERR_ARG;  // more levels than elements cannot happen
        for (int b = 0; b < kLevelsPerCheck; b++, L++)
            hipLaunchKernelGGL(k_color_level, dim3(kLevelBlocks), dim3(kLevelThreads), 0, s, w.e2n,
                               w.next, npre, cnt, w.front[L & 1], w.front[(L + 1) & 1], w.counts, L,
                               w.masks, w.part, w.status);
        if (hipGetLastError() != hipSuccess || read_ints(&remaining, w.counts + L % 3, 1, s) != MF_OK)
            return MF_ERR_HIP;
    }
    int hs[3] = {0, 0, 0};
    if (read_ints(hs, w.status, 3, s) != MF_OK) return MF_ERR_HIP;
    if (hs[2]) return MF_ERR_COLORS;
    return hs[1] == w.nE ? MF_OK : MF_ERR_ARG;  // not every element became ready
}

}  // namespace

extern "C" int mf_dev_coloring_creation(const int *elemToNode, int *colorPart, int *colorPerm,
                                        int nbElem, int nbNodes, int *colorToElem,
                                        int *nbColors, void *stream)
{
    if (nbElem < 0 || nbNodes < 0 || !colorPerm || !colorToElem || !nbColors ||
        (nbElem > 0 && !elemToNode) || (reinterpret_cast<uintptr_t>(elemToNode) & 15))
        return MF_ERR_ARG;  // elements are read as 16-byte rows
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    if (nbElem == 0) {
        *nbColors = 0;
        const int z = 0;
        if (hipMemcpyAsync(colorToElem, &z, sizeof(int), hipMemcpyHostToDevice, s) != hipSuccess ||
            hipStreamSynchronize(s) != hipSuccess)
            return MF_ERR_HIP;
        return MF_OK;
    }
    const size_t nE = (size_t)nbElem, N = (size_t)nbNodes;
    // index, value, next, the two lists, masks and words (or predecessor counts), the colors
    // when the caller does not keep them; later the sort's keys, elements and scratch
    const auto pad = [](size_t b) { return Workspace::padded(b); };
    size_t sort_bytes = 0;
    if (hipcub::DeviceRadixSort::SortPairs(nullptr, sort_bytes, (const int *)nullptr, (int *)nullptr,
                                           (const int *)nullptr, (int *)nullptr, nbElem, 0, 7, s) !=
        hipSuccess)
        return MF_ERR_HIP;
    Workspace ws(pad((N + 1) * sizeof(int)) + pad(4 * nE * sizeof(int)) + pad(nE * sizeof(int4)) +
                     2 * pad(nE * sizeof(int)) + pad(N * sizeof(ulonglong2)) +
                     pad(nE * sizeof(unsigned long long)) + pad(7 * sizeof(int)) +
                     4 * pad(nE * sizeof(int)) + pad(sort_bytes + 1), s);
    const StreamDrain drain{s};
    if (!ws.ok()) return MF_ERR_NOMEM;
    ColoringWork w;
    w.e2n = reinterpret_cast<const int4 *>(elemToNode);
    w.nE = nbElem;
    w.N = nbNodes;
    w.index = ws.cut<int>(N + 1);
    w.value = ws.cut<int>(4 * nE);
    w.next = ws.cut<int4>(nE);
    w.front[0] = ws.cut<int>(nE);
    w.front[1] = ws.cut<int>(nE);
    w.masks = ws.cut<ulonglong2>(N);
    w.words = ws.cut<unsigned long long>(nE);
    w.counts = ws.cut<int>(7);  // counts[3], status[4]
    w.status = w.counts + 3;
    int *own = ws.cut<int>(nE);
    w.part = colorPart ? colorPart : own;
    // nodeToElem (each node's elements ascending), as the host's
    int st = mf_dev_create_nodeToElem(elemToNode, nbElem, nbNodes, w.index, w.value, stream);
    if (st != MF_OK) return st;
    bool done = false;
    if (nbElem < 1 << 29) st = color_by_chains(w, s, &done);
    if (st == MF_OK && !done) st = color_by_levels(w, s);
    if (st != MF_OK) return st;
    // stable sort of the element ids by color: 7 key bits (colors < 128)
    int *kout = ws.cut<int>(nE), *vin = ws.cut<int>(nE), *vout = ws.cut<int>(nE);
    void *tmp = ws.cut<unsigned char>(sort_bytes + 1);
    hipLaunchKernelGGL(k_iota, grid_for(nbElem, 256), dim3(256), 0, s, vin, nbElem);
    if (hipcub::DeviceRadixSort::SortPairs(tmp, sort_bytes, w.part, kout, vin, vout, nbElem, 0, 7, s) !=
        hipSuccess)
        return MF_ERR_HIP;
    hipLaunchKernelGGL(k_color_perm, grid_for(nbElem, 256), dim3(256), 0, s, kout, vout, nbElem,
                       colorPerm, colorToElem);
    if (hipGetLastError() != hipSuccess) return MF_ERR_HIP;
    int last = 0;
    if (hipMemcpyAsync(&last, kout + nE - 1, sizeof(int), hipMemcpyDeviceToHost, s) != hipSuccess ||
        hipStreamSynchronize(s) != hipSuccess)
        return MF_ERR_HIP;
    *nbColors = last + 1;
    return MF_OK;
}

extern "C" int mf_dev_create_nodeToElem(const int *elemToNode, int nbElem, int nbNodes, int *index,
                                        int *value, void *stream)
{
    if (nbElem < 0 || nbNodes < 0 || !index || (nbElem > 0 && (!elemToNode || !value)))
        return MF_ERR_ARG;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    const int64_t n4 = (int64_t)nbElem * 4;
    const int N = nbNodes;
    size_t scan_bytes = 0;
    if (hipcub::DeviceScan::ExclusiveSum(nullptr, scan_bytes, (const int *)nullptr, (int *)nullptr,
                                         N + 1, s) != hipSuccess)
        return MF_ERR_HIP;
    const size_t counts = ((size_t)N + 2) * sizeof(int);  // and the flag
    Workspace ws(Workspace::padded(counts) + Workspace::padded((size_t)n4 * sizeof(int) + 1) +
                     Workspace::padded(scan_bytes + 1), s);
    const StreamDrain drain{s};
    if (!ws.ok()) return MF_ERR_NOMEM;
    int *cnt = ws.cut<int>((size_t)N + 2), *bad = cnt + N + 1;
    int *turn = ws.cut<int>((size_t)n4 + 1);
    void *tmp = ws.cut<unsigned char>(scan_bytes + 1);
    if (hipMemsetAsync(cnt, 0, counts, s) != hipSuccess) return MF_ERR_HIP;
    int hbad = 0;
    if (n4 > 0) {
        hipLaunchKernelGGL(k_count_nodes, grid_for(n4, 256), dim3(256), 0, s, elemToNode, n4, N, cnt,
                           turn, bad);
        if (hipGetLastError() != hipSuccess ||
            hipMemcpyAsync(&hbad, bad, sizeof(int), hipMemcpyDeviceToHost, s) != hipSuccess ||
            hipStreamSynchronize(s) != hipSuccess)
            return MF_ERR_HIP;
    }
    if (hbad) return MF_ERR_ARG;  // a node id outside 1..N
    if (hipcub::DeviceScan::ExclusiveSum(tmp, scan_bytes, cnt, index, N + 1, s) != hipSuccess)
        return MF_ERR_HIP;
    if (n4 > 0) {
        hipLaunchKernelGGL(k_fill_nodes, grid_for(n4, 256), dim3(256), 0, s, elemToNode, n4, index,
                           turn, value);
        hipLaunchKernelGGL(k_sort_lists, grid_for(N, 16), dim3(256), 0, s, index, N, value);
        if (hipGetLastError() != hipSuccess) return MF_ERR_HIP;
    }
    return hipStreamSynchronize(s) == hipSuccess ? MF_OK : MF_ERR_HIP;
}

extern "C" int mf_dev_create_nodeToNode(int *row, int *col, const int *n2eIndex,
                                        const int *n2eValue, const int *elemToNode, int nbNodes,
                                        int nbEdges, void *stream)
{
    if (!row || nbNodes < 0 || nbEdges < 0 || (nbNodes > 0 && (!n2eIndex || !elemToNode)))
        return MF_ERR_ARG;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    const int N = nbNodes;
    int inc = 0, nnz = 0;  // entries of all the nodes' lists; of all rows
    if (N > 0 && (hipMemcpyAsync(&inc, n2eIndex + N, sizeof(int), hipMemcpyDeviceToHost, s) != hipSuccess ||
                  hipStreamSynchronize(s) != hipSuccess))
        return MF_ERR_HIP;
    size_t scan_bytes = 0;
    if (hipcub::DeviceScan::ExclusiveSum(nullptr, scan_bytes, (const int *)nullptr, (int *)nullptr,
                                         N + 1, s) != hipSuccess)
        return MF_ERR_HIP;
    const size_t lens = Workspace::padded(((size_t)N + 1) * sizeof(int)),
                 marks = Workspace::padded((size_t)std::max(inc, 0) + 1);
    Workspace ws(lens + marks + Workspace::padded(scan_bytes + 1), s);
    const StreamDrain drain{s};
    if (!ws.ok()) return MF_ERR_NOMEM;
    int *len = ws.cut<int>((size_t)N + 1);
    uint8_t *flags = ws.cut<uint8_t>((size_t)std::max(inc, 0) + 1);
    void *tmp = ws.cut<unsigned char>(scan_bytes + 1);
    if (hipMemsetAsync(len + N, 0, sizeof(int), s) != hipSuccess) return MF_ERR_HIP;
    if (N > 0)
        hipLaunchKernelGGL(k_row_len, grid_for(N, 16), dim3(256), 0, s, n2eIndex, n2eValue, elemToNode, N,
                           len, flags);
    if (hipGetLastError() != hipSuccess ||
        hipcub::DeviceScan::ExclusiveSum(tmp, scan_bytes, len, row, N + 1, s) != hipSuccess ||
        hipMemcpyAsync(&nnz, row + N, sizeof(int), hipMemcpyDeviceToHost, s) != hipSuccess ||
        hipStreamSynchronize(s) != hipSuccess)
        return MF_ERR_HIP;
    if (nnz > nbEdges) return MF_ERR_NNZ;  // the pattern does not fit col[]
    if (N > 0 && nnz > 0) {
        if (!col) return MF_ERR_ARG;
        hipLaunchKernelGGL(k_row_fill, grid_for(N, 16), dim3(256), 0, s, n2eIndex, n2eValue, elemToNode, row,
                           N, flags, col);
        if (hipGetLastError() != hipSuccess) return MF_ERR_HIP;
    }
    return hipStreamSynchronize(s) == hipSuccess ? nnz : MF_ERR_HIP;
}

extern "C" int mf_dev_create_elemToEdge(const int *row, const int *col, const int *elemToNode,
                                        int *elemToEdge, int nbElem, void *stream)
{
    if (nbElem < 0 || (nbElem > 0 && (!row || !col || !elemToNode || !elemToEdge)))
        return MF_ERR_ARG;
    if (nbElem == 0) return MF_OK;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    hipLaunchKernelGGL(k_elem_to_edge, grid_for((int64_t)nbElem * 4, 256), dim3(256), 0, s, row, col,
                       elemToNode, nbElem, elemToEdge);
    if (hipGetLastError() != hipSuccess) return MF_ERR_HIP;
    return hipStreamSynchronize(s) == hipSuccess ? MF_OK : MF_ERR_HIP;
}

namespace {

template <typename T>
int dev_permute_rows(T *tab, const int *perm, int n, int dim, hipStream_t s)
{
    if (n < 0 || dim <= 0 || (n > 0 && (!tab || !perm))) return MF_ERR_ARG;
    if (n == 0) return MF_OK;
    DevBuf tmp, bad;
    const StreamDrain drain{s};
    if (dev_alloc(tmp, (size_t)n * dim * sizeof(T)) != MF_OK || dev_alloc(bad, sizeof(int)) != MF_OK)
        return MF_ERR_NOMEM;
    if (hipMemsetAsync(bad.p, 0, sizeof(int), s) != hipSuccess) return MF_ERR_HIP;
    hipLaunchKernelGGL(k_check_perm, grid_for(n, 256), dim3(256), 0, s, perm, n, bad.get<int>());
    int hbad = 0;
    if (hipGetLastError() != hipSuccess ||
        hipMemcpyAsync(&hbad, bad.p, sizeof(int), hipMemcpyDeviceToHost, s) != hipSuccess ||
        hipStreamSynchronize(s) != hipSuccess)
        return MF_ERR_HIP;
    if (hbad) return MF_ERR_ARG;  // tab unchanged, as the host twin leaves it
    const int64_t total = (int64_t)n * dim;
    if (hipMemcpyAsync(tmp.p, tab, (size_t)total * sizeof(T), hipMemcpyDeviceToDevice, s) != hipSuccess)
        return MF_ERR_HIP;
    hipLaunchKernelGGL(k_permute_rows<T>, grid_for(total, 256), dim3(256), 0, s, tmp.get<T>(), perm,
                       n, dim, tab);
    if (hipGetLastError() != hipSuccess) return MF_ERR_HIP;
    return hipStreamSynchronize(s) == hipSuccess ? MF_OK : MF_ERR_HIP;
}

}  // namespace

extern "C" int mf_dev_permute_int_2d(int *tab, const int *perm, int n, int dim, void *stream)
{
    return dev_permute_rows(tab, perm, n, dim, reinterpret_cast<hipStream_t>(stream));
}

extern "C" int mf_dev_permute_double_2d(double *tab, const int *perm, int n, int dim, void *stream)
{
    return dev_permute_rows(tab, perm, n, dim, reinterpret_cast<hipStream_t>(stream));
}
