// Consumer of the iteration's outputs: block-Jacobi preconditioned conjugate gradients
// on the assembled operator. The reference assembles values and prec every iteration
// but stops before the solve ("solver & update", src/main.cc:353); this closes the loop
// on the GPU.
//
// Operator: the dofs masked by checkBounds (the Dirichlet dofs ela_invert_prec masks,
// src/Fortran/elasclpr.f:29-32; lap masks a node when any of its three flags is set)
// are fixed: K = P A P + (I - P), with P zeroing masked dofs. prec is the block inverse
// of K's diagonal blocks exactly as prec_inversion leaves it (masked rows/columns unit),
// so z = prec r is the block-Jacobi step. Diagonal blocks of ela are symmetric, so the
// Fortran column-major and C row-major views of prec coincide.
//
// One iteration is three launches, each reading what it needs once; the scalars stay on the
// device:
//   q = K p with the partial sums of p.q           (k_spmv_lap, k_spmv_ela_staged:
//                                                   16 lanes per row)
//   x += alpha p, r -= alpha q, z = M r with the partial sums of r.z and r.r
//                                                  (k_update_prec_dot)
//   p = z + beta p and its masked copy P p, and the next iteration's scalars  (k_direction)
// Every workgroup of the second and third sums the launch before's partials for itself, in
// one fixed order, instead of waiting for a launch that sums them: 2,048 partials are 16 KB
// of L2 reads each, less than the start of a launch (an iteration of lap 41^3 27 -> 22 us, of
// ela 80^3 in the plan's order 185 -> 176, 100^3 351 -> 320).
// The product reads each row's blocks as one contiguous stream: the 16 lanes of a row
// take its blocks in turn (consecutive lanes, consecutive 72- or 8-byte blocks), then
// sum their three (one) partial rows in a fixed butterfly; the columns are gathered
// from the masked copy of the direction, one gather per block. Dot products are
// deterministic: a fixed grid, a fixed tree per workgroup, the workgroup partials summed
// in a fixed tree.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <type_traits>

#include "device_common.h"
#include "minifem.h"

namespace {

constexpr int kBT = 256;          // threads per workgroup
// lanes per row in the operator product; for lap 8 took 82 against 87 us per 100^3 iteration
// in the plan's order but 217 against 204 us in the shuffled one, 4 was slower in both
constexpr int kGroup = 16;
constexpr int kMaxGrid = 2048;    // workgroups of the reducing kernels (partials per sum)
// Iterations enqueued between two looks at the state: a look leaves the GPU idle for 30 us, an
// iteration enqueued past the end costs 8, so 12, then a quarter of those so far, up to 32.
// Eight each time, and these (us): lap 41^3, 20 iterations 544 and 508, 136 3143 and 2887; lap
// 9^3, 46 iterations 889 and 778; ela 40^3, 304 iterations 11186 and 10327.
constexpr int kBatch = 12, kMaxBatch = 32;

// The iteration's scalars, on the device: the host enqueues iterations without waiting
// for them and reads this after every batch. There are two: an iteration reads one and
// k_direction writes the other, so no workgroup reads what another one writes. Once done is
// set, every kernel of the iterations already enqueued returns at once.
struct CgState {
    double rz, rr, tol, bnorm;
    int it, max_it;
    int done;  // 0 running; 1 converged or max_it reached; 2 p.q <= 0 (breakdown)
    int pad;
};

// Per node: bit e set when dof e is fixed (ela); lap: all three bits when any flag is set.
// With an order, entry t describes node order[t].
__global__ void k_mask_bits(const int *__restrict__ cb, int N, bool ela, const int *__restrict__ order,
                            uint8_t *__restrict__ m)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= N) return;
    const int i = order ? order[t] : t;
    uint8_t b = 0;
    if (cb) {
        const int f0 = cb[i] != 0, f1 = cb[(int64_t)N + i] != 0, f2 = cb[2 * (int64_t)N + i] != 0;
        b = ela ? (uint8_t)(f0 | f1 << 1 | f2 << 2) : (uint8_t)((f0 | f1 | f2) ? 7 : 0);
    }
    m[t] = b;
}

// Sum of x over the 16 lanes of a row, on every one of them (cross-lane moves of the vector
// unit, which leave the LDS to the operands).
__device__ __forceinline__ double row16_sum(double x)
{
    auto moved = [](double v, auto ctrl) {
        union {
            double d;
            int i[2];
        } u{v}, w;
#pragma unroll
        for (int k = 0; k < 2; k++)
            w.i[k] = __builtin_amdgcn_update_dpp(0, u.i[k], decltype(ctrl)::value, 0xF, 0xF, true);
        return w.d;
    };
    x += moved(x, std::integral_constant<int, 0xB1>{});   // lanes 1 0 3 2 of each four
    x += moved(x, std::integral_constant<int, 0x4E>{});   // lanes 2 3 0 1
    x += moved(x, std::integral_constant<int, 0x141>{});  // the other four of each eight
    x += moved(x, std::integral_constant<int, 0x140>{});  // the other eight
    return x;
}

// Fixed-order sums of NV values over a workgroup's kBT threads, on every thread; s: 4 NV
// words of LDS.
template <int NV>
__device__ __forceinline__ void block_sums(double *s, double (&v)[NV])
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
    for (int k = 0; k < NV; k++) {
        v[k] = row16_sum(v[k]);
        v[k] += __shfl_xor(v[k], 16);
        v[k] += __shfl_xor(v[k], 32);
        if (lane == 0) s[4 * k + w] = v[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NV; k++) v[k] = (s[4 * k] + s[4 * k + 1]) + (s[4 * k + 2] + s[4 * k + 3]);
    __syncthreads();
}

// The sums of NV arrays of n partials (part, part + kMaxGrid, ...), on every thread.
template <int NV>
__device__ __forceinline__ void part_sums(double *s, const double *__restrict__ part, int n,
                                          double (&v)[NV])
{
#pragma unroll
    for (int k = 0; k < NV; k++) v[k] = 0.0;
    for (int i = threadIdx.x; i < n; i += kBT)
#pragma unroll
        for (int k = 0; k < NV; k++) v[k] += part[k * kMaxGrid + i];
    block_sums<NV>(s, v);
}

// The lap product: q = K p over rows i = group, group + groups, ...; part[blockIdx.x] = this
// workgroup's share of p.q. The columns are gathered from pm = P p (fixed dofs already zero),
// so an entry costs its own load and one gather; a fixed row takes p's own value.
__global__ void __launch_bounds__(kBT)
    k_spmv_lap(const int *__restrict__ row, const int *__restrict__ col,
               const double *__restrict__ values, const uint8_t *__restrict__ mask, int N,
               const double *__restrict__ pm, const double *__restrict__ p, double *__restrict__ q,
               double *__restrict__ part, const CgState *__restrict__ cs)
{
    if (cs && cs->done) return;
    __shared__ double s[4];
    const int l = threadIdx.x % kGroup;
    const int groups = gridDim.x * (kBT / kGroup);
    double pq = 0.0;
    for (int i = blockIdx.x * (kBT / kGroup) + threadIdx.x / kGroup; i < N; i += groups) {
        const int q0 = row[i], q1 = row[i + 1];
        const unsigned mi = mask[i];
        const double pi = p[i];
        double acc = 0.0;
        for (int k = q0 + l; k < q1; k += kGroup) acc += values[k] * pm[col[k] - 1];
        acc = row16_sum(acc);
        if (l == 0) {
            const double qi = mi & 1u ? pi : acc;
            q[i] = qi;
            pq += pi * qi;
        }
    }
    double t[1] = {pq};
    block_sums<1>(s, t);
    if (threadIdx.x == 0) part[blockIdx.x] = t[0];
}

// The ela product with the value stream staged through LDS: a wave's four row groups own
// four consecutive rows, whose blocks are one contiguous segment of values; the wave
// reads it in chunks of kChunk blocks with consecutive lanes on consecutive 16-byte
// pieces (a lane that reads its own 72-byte block touches each line with several lanes and
// several instructions), then every lane takes its row's blocks from LDS in turn, every
// 16th, as the lanes of the lap product take entries. Only this wave reads its LDS region, and
// LDS operations of one wave complete in order, so no workgroup barrier is needed.
constexpr int kChunk = 64;
__global__ void __launch_bounds__(kBT)
    k_spmv_ela_staged(const int *__restrict__ row, const int *__restrict__ col,
                      const double *__restrict__ values, const uint8_t *__restrict__ mask, int N,
                      const double *__restrict__ pm, const double *__restrict__ p,
                      double *__restrict__ q, double *__restrict__ part, const CgState *__restrict__ cs)
{
    if (cs && cs->done) return;
    __shared__ double s[4];
    __shared__ __align__(16) double stage[kBT / 64][kChunk * 9];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int l = lane & (kGroup - 1), g = lane / kGroup;
    const int stride = gridDim.x * (kBT / kGroup);
    double *st = stage[w];
    double pq = 0.0;
    for (int r0 = blockIdx.x * (kBT / kGroup) + w * (64 / kGroup); r0 < N; r0 += stride) {
        const int i = r0 + g;
        const bool on = i < N;
        const int ic = on ? i : r0;
        const int q0 = row[ic], q1 = on ? row[ic + 1] : q0;
        const int s0 = row[r0], s1 = row[r0 + (64 / kGroup) < N ? r0 + (64 / kGroup) : N];
        const unsigned mi = mask[ic];
        double pi[3], acc[3];
#pragma unroll
        for (int d = 0; d < 3; d++) {
            pi[d] = p[(int64_t)ic * 3 + d];
            acc[d] = 0.0;
        }
        int k = q0 + l;  // this lane's next block: q0 + l, q0 + l + 16, ...
        for (int c0 = s0; c0 < s1; c0 += kChunk) {
            const int nb = s1 - c0 < kChunk ? s1 - c0 : kChunk, nd = nb * 9;
            const double *src = values + (int64_t)c0 * 9;
            for (int d = 2 * lane; d < nd; d += 128) {
                if (d + 1 < nd) {
                    const mf::Two v = *reinterpret_cast<const mf::Two *>(src + d);
                    st[d] = v.x;
                    st[d + 1] = v.y;
                } else {
                    st[d] = src[d];
                }
            }
            __builtin_amdgcn_wave_barrier();
            for (; k < q1 && k < c0 + nb; k += kGroup) {
                const int j = col[k] - 1;
                const double *b = st + (k - c0) * 9;
                const double x0 = pm[(int64_t)j * 3], x1 = pm[(int64_t)j * 3 + 1],
                             x2 = pm[(int64_t)j * 3 + 2];
#pragma unroll
                for (int d = 0; d < 3; d++)
                    acc[d] += b[3 * d] * x0 + b[3 * d + 1] * x1 + b[3 * d + 2] * x2;
            }
            __builtin_amdgcn_wave_barrier();
        }
#pragma unroll
        for (int d = 0; d < 3; d++) acc[d] = row16_sum(acc[d]);
        if (l == 0 && on) {
#pragma unroll
            for (int d = 0; d < 3; d++) {
                const double qi = (mi >> d) & 1u ? pi[d] : acc[d];
                q[(int64_t)i * 3 + d] = qi;
                pq += pi[d] * qi;
            }
        }
    }
    double t[1] = {pq};
    block_sums<1>(s, t);
    if (threadIdx.x == 0) part[blockIdx.x] = t[0];
}

// z = M r of node i, from its residual; adds r.z and r.r to v[0] and v[1]
template <bool ELA>
__device__ __forceinline__ void prec_node(const double *__restrict__ prec, const uint8_t *__restrict__ mask,
                                          int i, const double (&r)[ELA ? 3 : 1], double *__restrict__ z,
                                          double &rz, double &rr)
{
    if constexpr (ELA) {
        const double *m = prec + (int64_t)i * 9;
        const double z0 = m[0] * r[0] + m[1] * r[1] + m[2] * r[2];
        const double z1 = m[3] * r[0] + m[4] * r[1] + m[5] * r[2];
        const double z2 = m[6] * r[0] + m[7] * r[1] + m[8] * r[2];
        z[(int64_t)i * 3] = z0;
        z[(int64_t)i * 3 + 1] = z1;
        z[(int64_t)i * 3 + 2] = z2;
        rz += r[0] * z0 + r[1] * z1 + r[2] * z2;
        rr += r[0] * r[0] + r[1] * r[1] + r[2] * r[2];
    } else {
        // a masked lap node's row of K is the identity, so its prec is 1
        const double zi = mask[i] ? r[0] : prec[i] * r[0];
        z[i] = zi;
        rz += r[0] * zi;
        rr += r[0] * r[0];
    }
}

// r = P b - q, z = M r; part: shares of r.z, r.r and (P b).(P b)
template <bool ELA>
__global__ void __launch_bounds__(kBT)
    k_start(const double *__restrict__ b, const double *__restrict__ q,
            const double *__restrict__ prec, const uint8_t *__restrict__ mask, int N,
            double *__restrict__ r, double *__restrict__ z, double *__restrict__ part)
{
    constexpr int D = ELA ? 3 : 1;
    __shared__ double s[12];
    double v[3] = {0.0, 0.0, 0.0};
    for (int i = blockIdx.x * kBT + threadIdx.x; i < N; i += gridDim.x * kBT) {
        const unsigned mi = mask[i];
        double rv[D];
#pragma unroll
        for (int d = 0; d < D; d++) {
            const int64_t k = (int64_t)i * D + d;
            const double bi = (mi >> d) & 1u ? 0.0 : b[k];
            rv[d] = bi - q[k];
            r[k] = rv[d];
            v[2] += bi * bi;
        }
        prec_node<ELA>(prec, mask, i, rv, z, v[0], v[1]);
    }
    block_sums<3>(s, v);
    if (threadIdx.x == 0)
        for (int k = 0; k < 3; k++) part[k * kMaxGrid + blockIdx.x] = v[k];
}

// x += alpha p, r -= alpha q (alpha = r.z / p.q, from the product's partials), then z = M r;
// part: shares of r.z and r.r. p.q <= 0 stops the iteration before x moves.
template <bool ELA>
__global__ void __launch_bounds__(kBT)
    k_update_prec_dot(const CgState *__restrict__ cs, const double *__restrict__ pqPart, int nPart,
                      const double *__restrict__ p, const double *__restrict__ q,
                      double *__restrict__ x, double *__restrict__ r,
                      const double *__restrict__ prec, const uint8_t *__restrict__ mask, int N,
                      double *__restrict__ z, double *__restrict__ part, int *__restrict__ broken)
{
    constexpr int D = ELA ? 3 : 1;
    if (cs->done) return;
    __shared__ double s[8];
    double pq[1];
    part_sums<1>(s, pqPart, nPart, pq);
    if (!(pq[0] > 0.0)) {  // K is not positive definite on p (or p = 0)
        if (blockIdx.x == 0 && threadIdx.x == 0) *broken = 1;
        return;
    }
    const double alpha = cs->rz / pq[0];
    double v[2] = {0.0, 0.0};
    for (int i = blockIdx.x * kBT + threadIdx.x; i < N; i += gridDim.x * kBT) {
        double rv[D];
#pragma unroll
        for (int d = 0; d < D; d++) {
            const int64_t k = (int64_t)i * D + d;
            x[k] += alpha * p[k];
            rv[d] = r[k] - alpha * q[k];
            r[k] = rv[d];
        }
        prec_node<ELA>(prec, mask, i, rv, z, v[0], v[1]);
    }
    block_sums<2>(s, v);
    if (threadIdx.x == 0)
        for (int k = 0; k < 2; k++) part[k * kMaxGrid + blockIdx.x] = v[k];
}

// The end of an iteration: r.z and r.r of the updated residual from the partials, beta = r.z
// (new) / r.z (old), the next state (the solve stops at max_it or convergence), and, when it
// goes on, p = z + beta p and pm = P p (pm may be null). Without a state cs (the start): p = z
// and the first state, from k_start's partials, h its constants.
__global__ void __launch_bounds__(kBT)
    k_direction(const CgState *__restrict__ cs, CgState h, CgState *__restrict__ next, double rtol,
                const double *__restrict__ part, int nPart, const int *__restrict__ broken,
                const double *__restrict__ z, const uint8_t *__restrict__ mask, int D,
                double *__restrict__ p, double *__restrict__ pm, int64_t n)
{
    __shared__ double s[12];
    const bool first = blockIdx.x == 0 && threadIdx.x == 0;
    double beta = 0.0;
    if (cs) {
        h = *cs;
        if (h.done || *broken) {
            if (first) {
                if (!h.done) h.done = 2;
                *next = h;
            }
            return;
        }
        double v[2];
        part_sums<2>(s, part, nPart, v);
        beta = v[0] / h.rz;
        h.rz = v[0];
        h.rr = v[1];
        h.it += 1;
        h.done = h.it >= h.max_it || !(sqrt(h.rr) > h.tol) ? 1 : 0;
    } else {
        double v[3];
        part_sums<3>(s, part, nPart, v);
        h.rz = v[0];
        h.rr = v[1];
        h.bnorm = sqrt(v[2]) > 0.0 ? sqrt(v[2]) : 1.0;
        h.tol = rtol * h.bnorm;
        h.it = 0;
        h.done = h.max_it > 0 && sqrt(h.rr) > h.tol ? 0 : 1;
    }
    if (first) *next = h;
    if (h.done) return;
    for (int64_t i = (int64_t)blockIdx.x * kBT + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBT) {
        const double v = cs ? z[i] + beta * p[i] : z[i];
        p[i] = v;
        if (pm) pm[i] = (mask[i / D] >> (i % D)) & 1u ? 0.0 : v;
    }
}

// pm = P x
__global__ void __launch_bounds__(kBT)
    k_masked(const double *__restrict__ x, const uint8_t *__restrict__ mask, int D,
             double *__restrict__ pm, int64_t n)
{
    for (int64_t i = (int64_t)blockIdx.x * kBT + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBT)
        pm[i] = (mask[i / D] >> (i % D)) & 1u ? 0.0 : x[i];
}

// ---- the system in another node order (mf_pcg_ordered)

// inv[order[t]] = t; flag = 1 when some order[t] lies outside [0, N)
__global__ void k_order_invert(const int *__restrict__ order, int N, int *__restrict__ inv, int *flag)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= N) return;
    const int i = order[t];
    if (i < 0 || i >= N) *flag = 1;
    else inv[i] = t;
}

// len[t] = length of row order[t]; len[N] = 0 (the exclusive scan then ends in nnz); flag = 1
// for a negative length and when order repeats a node (some inv[order[t]] then names another t)
__global__ void k_order_rowlen(const int *__restrict__ order, const int *__restrict__ inv,
                               const int *__restrict__ row, int N, int *__restrict__ len, int *flag)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t > N) return;
    int l = 0;
    if (t < N) {
        const int i = order[t];
        if (i >= 0 && i < N) {
            l = row[i + 1] - row[i];
            if (l < 0 || inv[i] != t) *flag = 1;
        }
    }
    len[t] = l;
}

// flag = 1 for a column outside 1..N
__global__ void k_check_cols(const int *__restrict__ col, int64_t nnz, int N, int *flag)
{
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < nnz; k += stride)
        if (col[k] < 1 || col[k] > N) *flag = 1;
}

// New row t = old row order[t], its entries in their own order, columns renumbered, the
// columns of fixed dofs zero (m: the mask in the new order): the product then gathers the
// direction itself, and needs no masked copy of it. 16 lanes take a row 16 entries at a time:
// each lane the column of one, then all of them the entries' values, one contiguous run on both
// sides, in 16-byte pieces (the first read before the columns, so that both are in flight). A
// piece asks the lanes of its entries for their masks and is stored once, as it is to stay
// (311 us for ela 80^3; the pieces as they were read, fixed dofs zeroed by more stores, 325; a
// block per lane word by word 386: rows of 1 KB in random order).
template <int DD>
__global__ void __launch_bounds__(kBT)
    k_order_csr(const int *__restrict__ order, const int *__restrict__ inv,
                const int *__restrict__ row, const int *__restrict__ col,
                const double *__restrict__ values, const int *__restrict__ rowp,
                const uint8_t *__restrict__ m, int N, int *__restrict__ colp,
                double *__restrict__ valp)
{
    const int l = threadIdx.x % kGroup, g = (threadIdx.x >> 4) & 3;
    const int groups = gridDim.x * (kBT / kGroup);
    for (int t = blockIdx.x * (kBT / kGroup) + threadIdx.x / kGroup; t < N; t += groups) {
        const int i = order[t], src = row[i], n = row[i + 1] - src, dst = rowp[t];
        for (int c0 = 0; c0 < n; c0 += kGroup) {
            const bool on = c0 + l < n;
            const double *from = values + (int64_t)(src + c0) * DD;
            double *to = valp + (int64_t)(dst + c0) * DD;
            if constexpr (DD == 1) {
                const double v = on ? from[l] : 0.0;
                const int j = on ? inv[col[src + c0 + l] - 1] : 0;
                if (on) {
                    colp[dst + c0 + l] = j + 1;
                    to[l] = m[j] ? 0.0 : v;
                }
            } else {
                constexpr int CP = (kGroup * DD / 2 + kGroup - 1) / kGroup;
                const int nd = min(n - c0, kGroup) * DD;
                mf::Two v[CP];
#pragma unroll
                for (int k = 0; k < CP; k++) {
                    const int d = 2 * (l + kGroup * k);
                    if (d + 1 < nd) v[k] = *reinterpret_cast<const mf::Two *>(from + d);
                    else v[k] = mf::Two{d < nd ? from[d] : 0.0, 0.0};
                }
                const int j = on ? inv[col[src + c0 + l] - 1] : 0;
                const unsigned mj = on ? m[j] : 0;
                if (on) colp[dst + c0 + l] = j + 1;
                const bool any = (__ballot(mj != 0) >> (16 * g)) & 0xFFFFu;
#pragma unroll
                for (int k = 0; k < CP; k++) {
                    const int d = 2 * (l + kGroup * k);
                    if (any) {  // entry d / 9, its column d % 3
                        const unsigned a = __shfl(mj, min(d / 9, kGroup - 1), kGroup),
                                       b = __shfl(mj, min((d + 1) / 9, kGroup - 1), kGroup);
                        if ((a >> (d % 3)) & 1u) v[k].x = 0.0;
                        if ((b >> ((d + 1) % 3)) & 1u) v[k].y = 0.0;
                    }
                    if (d + 1 < nd) *reinterpret_cast<mf::Two *>(to + d) = v[k];
                    else if (d < nd) to[d] = v[k].x;
                }
            }
        }
    }
}

// out[t W + w] = in[order[t] W + w] (gather) or the reverse (scatter)
__global__ void k_order_rows(const int *__restrict__ order, int64_t total, int W, bool gather,
                             const double *__restrict__ in, double *__restrict__ out)
{
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= total) return;
    const int64_t t = k / W, w = k % W, o = (int64_t)order[t] * W + w;
    if (gather) out[k] = in[o];
    else out[o] = in[k];
}

inline dim3 g1(int64_t n) { return dim3((unsigned)((n + kBT - 1) / kBT)); }
inline int grid_for(int64_t items) { return (int)std::max<int64_t>(1, std::min<int64_t>(kMaxGrid, (items + kBT - 1) / kBT)); }

}  // namespace

// The solve on one numbering of the nodes. copied: the system is k_order_csr's copy, whose
// columns of fixed dofs are zero, so the direction itself takes the place of its masked copy.
static int pcg_core(bool ela, bool copied, int nbNodes, const int *row, const int *col,
                    const double *values, const double *prec, const uint8_t *mask,
                    const double *b, double *x, double rtol, int maxIter, int *iterations,
                    double *relResidual, hipStream_t s)
{
    const int D = ela ? 3 : 1;
    const int64_t n = (int64_t)nbNodes * D;
    // r, z, p, q, pm = P p (not for a copy); 1 + 3 arrays of kMaxGrid partials; two states;
    // the breakdown flag
    const size_t vec = mf::Workspace::padded((size_t)n * sizeof(double));
    mf::Workspace ws((copied ? 4 : 5) * vec + mf::Workspace::padded(4 * kMaxGrid * sizeof(double)) +
                         mf::Workspace::padded(2 * sizeof(CgState)) + mf::Workspace::padded(sizeof(int)), s);
    if (!ws.ok()) return MF_ERR_NOMEM;
    double *r = ws.cut<double>(n), *z = ws.cut<double>(n), *p = ws.cut<double>(n), *q = ws.cut<double>(n);
    double *pm = copied ? nullptr : ws.cut<double>(n);
    double *pqPart = ws.cut<double>(4 * kMaxGrid), *part = pqPart + kMaxGrid;
    CgState *cs = ws.cut<CgState>(2);
    int *broken = ws.cut<int>(1);
    const int gSpmv = (int)std::max<int64_t>(1, std::min<int64_t>(kMaxGrid, ((int64_t)nbNodes * kGroup + kBT - 1) / kBT));
    const int gNode = grid_for(nbNodes), gDof = grid_for(n);
    // out = K in, from in and its masked copy in_m (state: skipped once the solve is done)
    auto spmv = [&](const double *in_m, const double *in, double *out, const CgState *c) {
        auto kern = ela ? k_spmv_ela_staged : k_spmv_lap;
        hipLaunchKernelGGL(kern, dim3(gSpmv), dim3(kBT), 0, s, row, col, values, mask, nbNodes,
                           copied ? in : in_m, in, out, pqPart, c);
    };
    CgState h{};
    h.max_it = maxIter;
    auto direction = [&](const CgState *c, CgState *next) {
        hipLaunchKernelGGL(k_direction, dim3(gDof), dim3(kBT), 0, s, c, h, next, rtol, part, gNode,
                           broken, z, mask, D, p, pm, n);
    };
    // r = P b - K x; z = M r; p = z
    const int zero = 0;
    if (hipMemcpyAsync(broken, &zero, sizeof(int), hipMemcpyHostToDevice, s) != hipSuccess) return MF_ERR_HIP;
    if (!copied) hipLaunchKernelGGL(k_masked, dim3(gDof), dim3(kBT), 0, s, x, mask, D, pm, n);
    spmv(pm, x, q, nullptr);  // its p.q partials are not used
    if (ela)
        hipLaunchKernelGGL(k_start<true>, dim3(gNode), dim3(kBT), 0, s, b, q, prec, mask, nbNodes, r, z, part);
    else
        hipLaunchKernelGGL(k_start<false>, dim3(gNode), dim3(kBT), 0, s, b, q, prec, mask, nbNodes, r, z, part);
    direction(nullptr, cs);
    // the iterations, enqueued a batch at a time; k_direction counts each one and decides, as
    // the loop condition would, whether another one runs
    int done = 0, sent = 0, batch = kBatch;
    do {
        for (int k = 0; k < batch && sent < maxIter; k++, sent++) {
            const CgState *c = cs + (sent & 1);
            spmv(pm, p, q, c);
            if (ela)
                hipLaunchKernelGGL(k_update_prec_dot<true>, dim3(gNode), dim3(kBT), 0, s, c, pqPart,
                                   gSpmv, p, q, x, r, prec, mask, nbNodes, z, part, broken);
            else
                hipLaunchKernelGGL(k_update_prec_dot<false>, dim3(gNode), dim3(kBT), 0, s, c, pqPart,
                                   gSpmv, p, q, x, r, prec, mask, nbNodes, z, part, broken);
            direction(c, cs + ((sent + 1) & 1));
        }
        if (hipGetLastError() != hipSuccess ||
            hipMemcpyAsync(&h, cs + (sent & 1), sizeof(h), hipMemcpyDeviceToHost, s) != hipSuccess ||
            hipStreamSynchronize(s) != hipSuccess) {
            (void)hipStreamSynchronize(s);
            return MF_ERR_HIP;
        }
        done = h.done;
        batch = std::max(kBatch, std::min(sent / 4, kMaxBatch));
    } while (!done);
    if (iterations) *iterations = h.it;
    if (relResidual) *relResidual = std::sqrt(h.rr) / h.bnorm;
    return MF_OK;
}

extern "C" int mf_pcg(int operatorID, int nbNodes, const int *row, const int *col,
                      const double *values, const double *prec, const int *checkBounds,
                      const double *b, double *x, double rtol, int maxIter, int *iterations,
                      double *relResidual, void *stream)
{
    const bool ela = operatorID == MF_OP_ELA;
    if ((operatorID != MF_OP_LAP && !ela) || nbNodes < 0 || !row || !values || !prec || !b || !x ||
        maxIter < 0 || !(rtol > 0.0))
        return MF_ERR_ARG;
    if (iterations) *iterations = 0;
    if (relResidual) *relResidual = 0.0;
    if (nbNodes == 0) return MF_OK;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    mf::Workspace ws(mf::Workspace::padded((size_t)nbNodes), s);
    if (!ws.ok()) return MF_ERR_NOMEM;
    uint8_t *mask = ws.cut<uint8_t>(nbNodes);
    hipLaunchKernelGGL(k_mask_bits, g1(nbNodes), dim3(kBT), 0, s, checkBounds, nbNodes, ela,
                       (const int *)nullptr, mask);
    return pcg_core(ela, false, nbNodes, row, col, values, prec, mask, b, x, rtol, maxIter, iterations,
                    relResidual, s);
}

extern "C" int mf_pcg_ordered(int operatorID, int nbNodes, const int *row, const int *col,
                              const double *values, const double *prec, const int *checkBounds,
                              const int *order, const double *b, double *x, double rtol,
                              int maxIter, int *iterations, double *relResidual, void *stream)
{
    const bool ela = operatorID == MF_OP_ELA;
    if ((operatorID != MF_OP_LAP && !ela) || nbNodes < 0 || !row || !values || !prec || !b || !x ||
        !order || maxIter < 0 || !(rtol > 0.0))
        return MF_ERR_ARG;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    if (iterations) *iterations = 0;
    if (relResidual) *relResidual = 0.0;
    const int N = nbNodes, D = ela ? 3 : 1, DD = D * D;
    if (N == 0) return MF_OK;
    int ends[2] = {0, 0};  // row[0], row[N]
    if (hipMemcpyAsync(&ends[0], row, sizeof(int), hipMemcpyDeviceToHost, s) != hipSuccess ||
        hipMemcpyAsync(&ends[1], row + N, sizeof(int), hipMemcpyDeviceToHost, s) != hipSuccess ||
        hipStreamSynchronize(s) != hipSuccess)
        return MF_ERR_HIP;
    const int nnz = ends[1];
    if (ends[0] != 0 || nnz < 0 || (nnz > 0 && !col)) return MF_ERR_ARG;
    size_t scan_bytes = 0;
    if (hipcub::DeviceScan::ExclusiveSum(nullptr, scan_bytes, (const int *)nullptr, (int *)nullptr,
                                         N + 1, s) != hipSuccess)
        return MF_ERR_HIP;
    const auto pad = [](size_t v) { return mf::Workspace::padded(v); };
    mf::Workspace ws(256 + pad(4 * (size_t)N) + 2 * pad(4 * ((size_t)N + 1)) + pad(4 * (size_t)nnz) +
                         pad(8 * (size_t)nnz * DD) + pad(8 * (size_t)N * DD) +
                         2 * pad(8 * (size_t)N * D) + pad((size_t)N) + pad(scan_bytes + 1), s);
    if (!ws.ok()) return MF_ERR_NOMEM;
    int *flag = ws.cut<int>(1), *inv = ws.cut<int>(N), *len = ws.cut<int>((size_t)N + 1),
        *rowp = ws.cut<int>((size_t)N + 1), *colp = ws.cut<int>(nnz);
    double *valp = ws.cut<double>((size_t)nnz * DD), *precp = ws.cut<double>((size_t)N * DD),
           *bp = ws.cut<double>((size_t)N * D), *xp = ws.cut<double>((size_t)N * D);
    uint8_t *mask = ws.cut<uint8_t>(N);
    void *scan = ws.cut<unsigned char>(scan_bytes + 1);
    // the copies below write where row and order say: order must be a permutation of
    // 0..N-1 (every index in range, no repeats), every row length >= 0 (with row[0] = 0 and
    // row[N] = nnz, each new row then lies inside 0..nnz) and every column in 1..N
    int bad = 0;
    if (hipMemcpyAsync(flag, &bad, sizeof(int), hipMemcpyHostToDevice, s) != hipSuccess) return MF_ERR_HIP;
    hipLaunchKernelGGL(k_order_invert, g1(N), dim3(kBT), 0, s, order, N, inv, flag);
    hipLaunchKernelGGL(k_order_rowlen, g1((int64_t)N + 1), dim3(kBT), 0, s, order, inv, row, N, len, flag);
    if (nnz > 0)
        hipLaunchKernelGGL(k_check_cols, dim3(grid_for(nnz)), dim3(kBT), 0, s, col, (int64_t)nnz, N, flag);
    if (hipGetLastError() != hipSuccess ||
        hipMemcpyAsync(&bad, flag, sizeof(int), hipMemcpyDeviceToHost, s) != hipSuccess ||
        hipStreamSynchronize(s) != hipSuccess)
        return MF_ERR_HIP;
    if (bad) return MF_ERR_ARG;
    if (hipcub::DeviceScan::ExclusiveSum(scan, scan_bytes, len, rowp, N + 1, s) != hipSuccess)
        return MF_ERR_HIP;
    hipLaunchKernelGGL(k_mask_bits, g1(N), dim3(kBT), 0, s, checkBounds, N, ela, order, mask);
    const int g = (int)std::max<int64_t>(1, std::min<int64_t>(kMaxGrid, ((int64_t)N * kGroup + kBT - 1) / kBT));
    if (ela)
        hipLaunchKernelGGL(k_order_csr<9>, dim3(g), dim3(kBT), 0, s, order, inv, row, col, values,
                           rowp, mask, N, colp, valp);
    else
        hipLaunchKernelGGL(k_order_csr<1>, dim3(g), dim3(kBT), 0, s, order, inv, row, col, values,
                           rowp, mask, N, colp, valp);
    hipLaunchKernelGGL(k_order_rows, g1((int64_t)N * DD), dim3(kBT), 0, s, order, (int64_t)N * DD, DD,
                       true, prec, precp);
    hipLaunchKernelGGL(k_order_rows, g1((int64_t)N * D), dim3(kBT), 0, s, order, (int64_t)N * D, D,
                       true, b, bp);
    hipLaunchKernelGGL(k_order_rows, g1((int64_t)N * D), dim3(kBT), 0, s, order, (int64_t)N * D, D,
                       true, x, xp);
    int st = hipGetLastError() == hipSuccess ? MF_OK : MF_ERR_HIP;
    if (st == MF_OK)
        st = pcg_core(ela, true, N, rowp, colp, valp, precp, mask, bp, xp, rtol, maxIter, iterations,
                      relResidual, s);
    if (st == MF_OK) {
        hipLaunchKernelGGL(k_order_rows, g1((int64_t)N * D), dim3(kBT), 0, s, order, (int64_t)N * D, D,
                           false, xp, x);
        if (hipGetLastError() != hipSuccess || hipStreamSynchronize(s) != hipSuccess) st = MF_ERR_HIP;
    }
    return st;
}
