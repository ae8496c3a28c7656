// FP64 / FP32 MLFMA matvec kernels for gfx950 (64-wide wavefronts).
//
// Workspaces are laid out [box][cur][comp][K] so that consecutive threads
// (consecutive k-space samples) touch consecutive addresses.  RWG functions are
// stored in leaf-major order (internal index i); perm[i] is the reference index
// used by the caller's x and y vectors.  The far-field kernels are templates on
// the real type R of the patterns, tables and workspaces (double or float);
// they accumulate in R.  Solver vectors x, y and the near field stay FP64.
#include <algorithm>
#include <complex>

#include "kernels.hpp"
#include <stdexcept>

#include "cplx.hpp"

namespace mlfma {

// Blocks are dispatched round-robin over the 8 XCDs of the MI355X; remap the
// linear block id so that every XCD works on one contiguous (Morton-ordered)
// range of boxes and its L2 sees the shared source boxes.
__device__ __forceinline__ int xcd_remap(int lin, int total) {
    const int per = total >> 3, rem = total & 7;
    const int x = lin & 7, s = lin >> 3;
    return x * per + min(x, rem) + s;
}

// Window order of n items x nt tiles: items go in windows of wc, and inside
// a window the tile index is the slow one, so the workgroups that run at
// once on one XCD work on the same tile of wc neighbouring items (which
// share most of their inputs in that XCD's L2); wc = 1 is item-major order.
__device__ __forceinline__ void window_order(int lin, int n, int nt, int wc, int& item, int& tile) {
    const int span = wc * nt;
    const int win = lin / span, r = lin - win * span;
    const int w = min(wc, n - win * wc);
    tile = r / w;
    item = win * wc + (r - tile * w);
}

// ---------------------------------------------------------------- aggregation
// Code/ProcessMLFMM.h:33-56 (mexp), J and M currents of PMCHWT in one pass.
// One workgroup per leaf, threads over the K samples (blockDim = K rounded up
// to a wavefront, at most 512), so that a workgroup streams whole pattern rows
// [i][3][K] of its leaf from HBM.  Leaves are taken largest first.  The leaf's
// x values are gathered into LDS in chunks, which keeps the dependent
// perm -> x loads out of the pattern stream.  RB right-hand sides share each
// pattern load: solver vectors are RHS-fastest (unknown u, rhs r at
// u * ldr + r) and workspace current c = rr * NCUR + cur.
template <typename R, int NCUR, int RB>
__global__ __launch_bounds__(512) void k_aggregate(int K, int N, int ldr, int r0, const int* __restrict__ order,
                                                   const int* __restrict__ leaf_ptr, const int* __restrict__ perm,
                                                   const cplx_t<R>* __restrict__ Vs, const double2* __restrict__ x,
                                                   cplx_t<R>* __restrict__ Sm) {
    using C = cplx_t<R>;
    constexpr int NC = NCUR * RB;
    constexpr int CHUNK = NC <= 2 ? 128 : 64;
    __shared__ C xl[NC][CHUNK];
    const int leaf = order[blockIdx.x];
    const int i0 = leaf_ptr[leaf], i1 = leaf_ptr[leaf + 1];
    for (int q0 = 0; q0 < K; q0 += blockDim.x) {
        const int q = q0 + threadIdx.x;
        const bool act = q < K;
        C acc[NC][3];
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int d = 0; d < 3; ++d) acc[c][d] = C{0, 0};
        for (int b = i0; b < i1; b += CHUNK) {
            const int n = min(CHUNK, i1 - b);
            __syncthreads();
            for (int e = threadIdx.x; e < n * NC; e += blockDim.x) {
                const int j = e / NC, c = e - j * NC;
                const int rr = c / NCUR, cur = c - rr * NCUR;
                narrow(x[((size_t)cur * N + perm[b + j]) * ldr + r0 + rr], xl[c][j]);
            }
            __syncthreads();
            if (act) {
                const C* v = Vs + (size_t)b * 3 * K + q;
                const size_t s3 = (size_t)3 * K;
                int j = 0;
                for (; j + 1 < n; j += 2) {
                    const C a0 = v[0], a1 = v[K], a2 = v[2 * K];
                    const C b0 = v[s3], b1 = v[s3 + K], b2 = v[s3 + 2 * K];
#pragma unroll
                    for (int c = 0; c < NC; ++c) {
                        const C xa = xl[c][j], xb = xl[c][j + 1];
                        cfma(acc[c][0], a0, xa);
                        cfma(acc[c][1], a1, xa);
                        cfma(acc[c][2], a2, xa);
                        cfma(acc[c][0], b0, xb);
                        cfma(acc[c][1], b1, xb);
                        cfma(acc[c][2], b2, xb);
                    }
                    v += 2 * s3;
                }
                if (j < n) {
                    const C a0 = v[0], a1 = v[K], a2 = v[2 * K];
#pragma unroll
                    for (int c = 0; c < NC; ++c) {
                        const C xa = xl[c][j];
                        cfma(acc[c][0], a0, xa);
                        cfma(acc[c][1], a1, xa);
                        cfma(acc[c][2], a2, xa);
                    }
                }
            }
        }
        if (act) {
            C* s = Sm + (size_t)leaf * NC * 3 * K + q;
#pragma unroll
            for (int c = 0; c < NC; ++c)
#pragma unroll
                for (int d = 0; d < 3; ++d) s[(size_t)(c * 3 + d) * K] = acc[c][d];
        }
    }
}

// The single-vector aggregation where there are few leaves: a workgroup takes
// 64 samples of one leaf and its four wavefronts every fourth RWG each, so a
// leaf is spread over K / 64 workgroups; the wavefronts' sums are added in a
// fixed order through LDS.
template <typename R, int NCUR>
__global__ __launch_bounds__(256) void k_aggregate_t(int K, int N, int tiles, const int* __restrict__ order,
                                                     const int* __restrict__ leaf_ptr, const int* __restrict__ perm,
                                                     const cplx_t<R>* __restrict__ Vs, const double2* __restrict__ x,
                                                     cplx_t<R>* __restrict__ Sm) {
    using C = cplx_t<R>;
    constexpr int CHUNK = 256, D = NCUR * 3;
    __shared__ C xl[NCUR][CHUNK];
    __shared__ C red[3][D][64];
    const int leaf = order[blockIdx.x / tiles];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int q = (blockIdx.x % tiles) * 64 + lane;
    const bool act = q < K;
    const int i0 = leaf_ptr[leaf], i1 = leaf_ptr[leaf + 1];
    C acc[D];
#pragma unroll
    for (int d = 0; d < D; ++d) acc[d] = C{0, 0};
    const size_t s3 = (size_t)3 * K;
    for (int b = i0; b < i1; b += CHUNK) {
        const int n = min(CHUNK, i1 - b);
        __syncthreads();
        for (int e = threadIdx.x; e < n; e += 256) {
            const int r = perm[b + e];
#pragma unroll
            for (int c = 0; c < NCUR; ++c) narrow(x[(size_t)c * N + r], xl[c][e]);
        }
        __syncthreads();
        if (act) {
            const C* v = Vs + (size_t)(b + wave) * s3 + q;
            int j = wave;
            for (; j + 12 < n; j += 16, v += 16 * s3) {
                C a[4][3];
#pragma unroll
                for (int u = 0; u < 4; ++u)
#pragma unroll
                    for (int d = 0; d < 3; ++d) a[u][d] = v[(size_t)(4 * u) * s3 + (size_t)d * K];
#pragma unroll
                for (int u = 0; u < 4; ++u)
#pragma unroll
                    for (int c = 0; c < NCUR; ++c)
#pragma unroll
                        for (int d = 0; d < 3; ++d) cfma(acc[c * 3 + d], a[u][d], xl[c][j + 4 * u]);
            }
            for (; j < n; j += 4, v += 4 * s3) {
                const C a0 = v[0], a1 = v[K], a2 = v[2 * (size_t)K];
#pragma unroll
                for (int c = 0; c < NCUR; ++c) {
                    cfma(acc[c * 3 + 0], a0, xl[c][j]);
                    cfma(acc[c * 3 + 1], a1, xl[c][j]);
                    cfma(acc[c * 3 + 2], a2, xl[c][j]);
                }
            }
        }
    }
    if (wave > 0)
#pragma unroll
        for (int d = 0; d < D; ++d) red[wave - 1][d][lane] = acc[d];
    __syncthreads();
    if (wave == 0 && act) {
        C* s = Sm + (size_t)leaf * D * K + q;
#pragma unroll
        for (int d = 0; d < D; ++d) {
            C a = acc[d];
#pragma unroll
            for (int w = 0; w < 3; ++w) a.x += red[w][d][lane].x, a.y += red[w][d][lane].y;
            s[(size_t)d * K] = a;
        }
    }
}

// One workgroup per leaf needs enough leaves: 7,680 RWG in 56 leaves (PMCHWT,
// FP64, both wavenumbers, 346 MB of patterns) take 310 us that way and 88 us in
// sample tiles, 480 RWG 7.1 and 5.0 us.  With 3,200 leaves (300,000 RWG,
// 4.9 GB) whole rows stream slightly better, 917 against 944 us.  Near the line,
// FP64 PMCHWT, whole rows and tiles in us: 512 leaves 309 and 252, 768 leaves
// 235 and 232, 824 leaves 679 and 674, 1,272 leaves 209 and 223, 1,968 leaves
// 967 and 1,046; FP32 with leaves of 19 RWG leans to whole rows earlier (768
// leaves 27 and 32), with leaves of 90 later (1,392 leaves 520 and 484).
constexpr int kAggTileLeaves = 1024;

template <typename R>
void launch_aggregate_b(hipStream_t st, int ncur, int rb, int nleaf, int K, int N, int ldr, int r0, const int* order,
                        const int* leaf_ptr, const int* perm, const cplx_t<R>* Vs, const double2* x,
                        cplx_t<R>* Sm) {
    if (nleaf == 0) return;
    if (rb == 1 && ldr == 1 && nleaf < kAggTileLeaves) {
        const int tiles = (K + 63) / 64;
        if (ncur == 1) k_aggregate_t<R, 1><<<nleaf * tiles, 256, 0, st>>>(K, N, tiles, order, leaf_ptr, perm, Vs, x, Sm);
        else k_aggregate_t<R, 2><<<nleaf * tiles, 256, 0, st>>>(K, N, tiles, order, leaf_ptr, perm, Vs, x, Sm);
        return;
    }
    const int threads = std::min(512, (K + 63) / 64 * 64);
#define AGG(NCUR, RB) k_aggregate<R, NCUR, RB><<<nleaf, threads, 0, st>>>(K, N, ldr, r0, order, leaf_ptr, perm, Vs, x, Sm)
    if (ncur == 1) {
        if (rb == 1) AGG(1, 1);
        else if (rb == 2) AGG(1, 2);
        else if (rb == 4) AGG(1, 4);
        else AGG(1, 8);
    } else {
        if (rb == 1) AGG(2, 1);
        else if (rb == 2) AGG(2, 2);
        else if (rb == 4) AGG(2, 4);
        else if constexpr (sizeof(R) == 4) AGG(2, 8);
        else throw std::invalid_argument("FP64 aggregation: at most 4 right-hand sides per pass");
    }
#undef AGG
}

template <typename R>
void launch_aggregate(hipStream_t st, int ncur, int nleaf, int K, int N, const int* order, const int* leaf_ptr,
                      const int* perm, const cplx_t<R>* Vs, const double2* x, cplx_t<R>* Sm) {
    launch_aggregate_b<R>(st, ncur, 1, nleaf, K, N, 1, 0, order, leaf_ptr, perm, Vs, x, Sm);
}

// ---------------------------------------------------------------- interpolation
// Code/ProcessMLFMM.h:61-107 (m2m): 3x3 Lagrange taps into the child grid, then
// the octant phase shift, summed over the children of each parent.  A thread
// owns one parent sample and CPT of the nc x 3 workspace columns (one
// wavefront per column group); the q tiles of one parent
// are consecutive after the XCD remap, so they share that XCD's L2 copy of the
// children's workspaces.
template <typename R, int NC, int CPT>
__global__ __launch_bounds__(64 * NC * 3 / CPT) void k_m2m(int nparent, int qtiles, int Kp, int Kc,
                                                 const int* __restrict__ son_ptr, const int* __restrict__ son_idx,
                                                 const int* __restrict__ oct_child, const int* __restrict__ tap,
                                                 const R* __restrict__ w, const cplx_t<R>* __restrict__ shup,
                                                 const cplx_t<R>* __restrict__ Smc, cplx_t<R>* __restrict__ Smp) {
    using C = cplx_t<R>;
    const int lin = xcd_remap(blockIdx.x, nparent * qtiles);
    const int p = lin / qtiles;
    const int q = (lin % qtiles) * 64 + (threadIdx.x & 63);
    const int c0 = (threadIdx.x >> 6) * CPT;   // first workspace column of this thread
    if (q >= Kp) return;
    int t[9];
    R ww[9];
#pragma unroll
    for (int s = 0; s < 9; ++s) {
        t[s] = tap[(size_t)s * Kp + q];
        ww[s] = w[(size_t)s * Kp + q];
    }
    C acc[CPT];
#pragma unroll
    for (int d = 0; d < CPT; ++d) acc[d] = C{0, 0};
    for (int j = son_ptr[p]; j < son_ptr[p + 1]; ++j) {
        const int c = son_idx[j];
        const C e = shup[(size_t)oct_child[c] * Kp + q];
        const C* S = Smc + ((size_t)c * NC * 3 + c0) * Kc;
#pragma unroll
        for (int d = 0; d < CPT; ++d) {
            const C* sd = S + (size_t)d * Kc;
            C r = C{0, 0};
#pragma unroll
            for (int k = 0; k < 9; ++k) {
                const C f = sd[t[k]];
                r.x += f.x * ww[k];
                r.y += f.y * ww[k];
            }
            cfma(acc[d], e, r);
        }
    }
    C* o = Smp + ((size_t)p * NC * 3 + c0) * Kp + q;
#pragma unroll
    for (int d = 0; d < CPT; ++d) o[(size_t)d * Kp] = acc[d];
}

template <typename R>
void launch_m2m(hipStream_t st, int ncur, int nparent, int Kp, int Kc, const int* son_ptr, const int* son_idx,
                const int* octant_child, const int* tap, const R* w, const cplx_t<R>* shift_up, const cplx_t<R>* Sm_child,
                cplx_t<R>* Sm_parent) {
    if (nparent == 0) return;
    const int qt = (Kp + 63) / 64;
#define M2M(NC, CPT)                                                                                                  \
    k_m2m<R, NC, CPT><<<nparent * qt, 64 * NC * 3 / CPT, 0, st>>>(nparent, qt, Kp, Kc, son_ptr, son_idx,             \
                                                                  octant_child, tap, w, shift_up, Sm_child, Sm_parent)
    if (ncur == 1) M2M(1, 3);
    else if (ncur == 2) M2M(2, 3);
    else if (ncur == 4) M2M(4, 3);
    else if (ncur == 8) M2M(8, 3);
    else if constexpr (sizeof(R) == 4) M2M(16, 6);
    else throw std::invalid_argument("FP64 far field: at most 8 workspace currents per pass");
#undef M2M
}

// Code/ProcessMLFMM.h:61-107 (m2m) in separable form: the 3x3 stencil of parent
// sample (i, j) is child rows th_tap[i][a] x child columns ph_tap[j][b] with
// weights th_w[i][a] ph_w[j][b], so theta comes first, U(i, m) = sum_a th_w[i][a]
// S_c(th_tap[i][a], m), then phi, r(i, j) = sum_b ph_w[j][b] U(i, ph_tap[j][b]),
// and shift x r is added child after child.  About half the loads and
// multiply-adds of the 9-tap form; the sums are regrouped, which changes only
// rounding.  A wavefront takes RW rows of a parent and CPT of the nc x 3
// columns.  Theta: its lanes run over the child's columns and it walks the
// window of child rows that its parent rows take (win_*: row_windows of the
// theta stencil), so a child sample is loaded once per group of RW rows and
// added to the RW rows in registers, the next row's loads in flight.  (Parent
// row by parent row each child sample was loaded about four times: C5, 64
// right-hand sides, 4.4 ms per matvec, now 3.3.)  Phi: the rows go through the
// wavefront's own LDS (no barrier), lanes over (row, parent column) pairs, JJ
// outputs per thread kept in registers over the children.
template <typename R, int CPT, int RW, int JJ>
__global__ __launch_bounds__(256) void k_m2m_row(int nc, int Lp, int Lc, int ncb, const int* __restrict__ son_ptr,
                                                 const int* __restrict__ son_idx,
                                                 const int* __restrict__ oct_child,
                                                 const int* __restrict__ win_ptr, const int* __restrict__ win_row,
                                                 const R* __restrict__ win_w, const int* __restrict__ ph_tap,
                                                 const R* __restrict__ ph_w, const cplx_t<R>* __restrict__ shup,
                                                 const cplx_t<R>* __restrict__ Smc, cplx_t<R>* __restrict__ Smp) {
    using C = cplx_t<R>;
    extern __shared__ __align__(16) unsigned char m2m_lds[];
    const int pfn = 2 * Lp, psn = 2 * Lc, Kp = Lp * pfn, Kc = Lc * psn;
    const int nrg = (Lp + RW - 1) / RW;   // row groups per parent
    const int lin = xcd_remap(blockIdx.x, (int)gridDim.x);
    const int cb = lin % ncb, g = (lin / ncb) % nrg, p = lin / (ncb * nrg);   // one parent's workgroups are consecutive
    const int i0 = g * RW, nr = min(RW, Lp - i0);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int c0 = (cb * (int)(blockDim.x >> 6) + wave) * CPT;
    C* U = reinterpret_cast<C*>(m2m_lds) + (size_t)wave * CPT * RW * psn;   // [CPT][RW][2 Lc]
    // phi-pass outputs of this thread (t = lane + 64 jj, clamped past the last)
    int pj[JJ][3];
    R wj[JJ][3];
    C out[JJ][CPT];
#pragma unroll
    for (int jj = 0; jj < JJ; ++jj) {
        const int t = min(lane + 64 * jj, nr * pfn - 1);
        const int r = t / pfn, j = t - r * pfn;
#pragma unroll
        for (int b = 0; b < 3; ++b) {
            pj[jj][b] = r * psn + ph_tap[3 * j + b];
            wj[jj][b] = ph_w[3 * j + b];
        }
#pragma unroll
        for (int d = 0; d < CPT; ++d) out[jj][d] = C{0, 0};
    }
    const int k0 = win_ptr[g], k1 = win_ptr[g + 1];
    const int s0 = son_ptr[p], s1 = son_ptr[p + 1];
    if (s0 == s1) return;   // (every box of a parent level has a child)
    auto load = [&](const C* S, int m, int k, C (&v)[CPT]) {
        const int at = win_row[min(k, k1 - 1)] * psn + m;
#pragma unroll
        for (int d = 0; d < CPT; ++d) v[d] = S[(size_t)d * Kc + at];
    };
    auto block = [&](int s) { return Smc + ((size_t)son_idx[s] * nc * 3 + c0) * Kc; };
    // four rows in flight; the first two of the next 64 columns or child are
    // loaded before this one's phi pass
    C va[CPT], vb[CPT], vc[CPT], vd[CPT];
    const C* S = block(s0);
    load(S, min(lane, psn - 1), k0, va);
    load(S, min(lane, psn - 1), k0 + 1, vb);
    for (int s = s0; s < s1; ++s) {
        const C* Sn = block(min(s + 1, s1 - 1));
        for (int mb = 0; mb < psn; mb += 64) {
            const int m = min(mb + lane, psn - 1);
            C acc[RW][CPT];
#pragma unroll
            for (int r = 0; r < RW; ++r)
#pragma unroll
                for (int d = 0; d < CPT; ++d) acc[r][d] = C{0, 0};
            auto add = [&](int k, const C (&v)[CPT]) {
#pragma unroll
                for (int r = 0; r < RW; ++r) {
                    const R w = win_w[(size_t)k * RW + r];
#pragma unroll
                    for (int d = 0; d < CPT; ++d) {
                        acc[r][d].x = fma(w, v[d].x, acc[r][d].x);
                        acc[r][d].y = fma(w, v[d].y, acc[r][d].y);
                    }
                }
            };
            for (int k = k0; k < k1; k += 4) {
                load(S, m, k + 2, vc);
                load(S, m, k + 3, vd);
                __builtin_amdgcn_sched_barrier(0);
                add(k, va);
                if (k + 1 < k1) add(k + 1, vb);
                const bool more = k + 4 < k1, same = mb + 64 < psn;   // uniform
                const C* Sl = more || same ? S : Sn;
                const int ml = more ? m : min((same ? mb + 64 : 0) + lane, psn - 1);
                load(Sl, ml, more ? k + 4 : k0, va);
                load(Sl, ml, more ? k + 5 : k0 + 1, vb);
                __builtin_amdgcn_sched_barrier(0);
                if (k + 2 < k1) add(k + 2, vc);
                if (k + 3 < k1) add(k + 3, vd);
            }
            if (mb + lane < psn)
#pragma unroll
                for (int d = 0; d < CPT; ++d)
#pragma unroll
                    for (int r = 0; r < RW; ++r) U[(d * RW + r) * psn + m] = acc[r][d];
        }
        S = Sn;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // other lanes of this wavefront wrote U
        const C* sh = shup + (size_t)oct_child[son_idx[s]] * Kp + (size_t)i0 * pfn;
#pragma unroll
        for (int jj = 0; jj < JJ; ++jj) {
            const C e = sh[min(lane + 64 * jj, nr * pfn - 1)];
#pragma unroll
            for (int d = 0; d < CPT; ++d) {
                const C u0 = U[d * RW * psn + pj[jj][0]], u1 = U[d * RW * psn + pj[jj][1]],
                        u2 = U[d * RW * psn + pj[jj][2]];
                C r;
                r.x = u0.x * wj[jj][0] + u1.x * wj[jj][1] + u2.x * wj[jj][2];
                r.y = u0.y * wj[jj][0] + u1.y * wj[jj][1] + u2.y * wj[jj][2];
                cfma(out[jj][d], e, r);
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // U is read before the next child's rows replace it
    }
    C* o = Smp + ((size_t)p * nc * 3 + c0) * Kp + (size_t)i0 * pfn;
#pragma unroll
    for (int jj = 0; jj < JJ; ++jj)
        if (lane + 64 * jj < nr * pfn)
#pragma unroll
            for (int d = 0; d < CPT; ++d) o[(size_t)d * Kp + lane + 64 * jj] = out[jj][d];
}

// Parent rows per group: 4 up to rows of 64 samples, 2 up to 192, then 1 (with
// 4 outputs per thread; 6 for 2 rows).  4 rows of 65 to 96 samples take 6
// outputs as well and run slower (FP64: one wavefront per SIMD, 76 against 45
// us at 2 rows; FP32 39 against 34), 1 row of 129 to 192 slower than 2 (64.5
// against 51).  0 (the caller takes the 9-tap kernel) where a row has more than
// 256 samples or does not fit 64 KB of LDS.
int m2m_rows(int Lp, int Lc) {
    const size_t row = (size_t)3 * 2 * Lc * sizeof(double2);
    if (2 * Lp > 256 || row > 64 * 1024) return 0;
    if (2 * Lp <= 64 && 4 * row <= 64 * 1024) return 4;
    if (2 * Lp <= 192 && 2 * row <= 64 * 1024) return 2;
    return 1;
}

template <typename R>
void launch_m2m_row(hipStream_t st, int ncur, int nparent, int Lp, int Lc, int rw, const int* son_ptr,
                    const int* son_idx, const int* octant_child, const int* win_ptr, const int* win_row,
                    const R* win_w, const int* ph_tap, const R* ph_w, const cplx_t<R>* shift_up,
                    const cplx_t<R>* Sm_child, cplx_t<R>* Sm_parent) {
    if (nparent == 0) return;
    constexpr int CPT = 3;
    const size_t lds = (size_t)CPT * rw * 2 * Lc * sizeof(cplx_t<R>);   // per wavefront
    const int JJ = (rw * 2 * Lp + 63) / 64;
    if ((rw != 1 && rw != 2 && rw != 4) || JJ > (rw == 2 ? 6 : 4) || lds > 64 * 1024)
        throw std::invalid_argument("separable interpolation: rows per wavefront out of range");
    int G = std::min(4, ncur);   // wavefronts (column groups) per workgroup
    while (G > 1 && G * lds > 64 * 1024) G /= 2;
    const int ncb = ncur / G;
    const unsigned grid = (unsigned)nparent * ((Lp + rw - 1) / rw) * ncb;
#define M2MR(RW, J)                                                                                                   \
    k_m2m_row<R, CPT, RW, J><<<grid, 64 * G, G * lds, st>>>(ncur, Lp, Lc, ncb, son_ptr, son_idx, octant_child,        \
                                                            win_ptr, win_row, win_w, ph_tap, ph_w, shift_up,          \
                                                            Sm_child, Sm_parent)
    if (rw == 4) {
        if (JJ <= 2) M2MR(4, 2);
        else if (JJ == 3) M2MR(4, 3);
        else M2MR(4, 4);
    } else if (rw == 2) {
        if (JJ <= 3) M2MR(2, 3);
        else if (JJ == 4) M2MR(2, 4);
        else M2MR(2, 6);
    } else {
        M2MR(1, 4);
    }
#undef M2MR
}

// Anterpolation from the parent level as a separable pass (the transpose of
// k_m2m_row): for box b with parent P and octant o, child sample (i, j) gets
//   sum over (parent row ip, wt) with th_tap[ip][a] = i, (parent column jp, wp)
//   with ph_tap[jp][b] = j of  wt wp shift_o(ip, jp) P(ip, jp),
// the same products as the fused gather (Code/ProcessMLFMM.h:152-202) with the
// sums regrouped (theta first), which changes only rounding; it adds into Bm,
// which the translation wrote before.  A wavefront takes RW child rows of one
// box and CPT of the nc x 3 columns.  Theta: its lanes run over the parent's
// columns and it walks the window of parent rows that touch its child rows
// (win_*: per group of RW rows the parent rows, ascending, with RW weights
// each), so every parent sample is loaded and shifted once per group and
// added to the RW rows in registers, the next row's loads in flight.  (Child
// row by child row, each parent sample was loaded three times behind scalar
// table loads: C5, 64 right-hand sides, 6.0 ms per matvec, now 4.5.)  Phi: the
// rows go through the wavefront's own LDS (no barrier), lanes over (row, child
// column) pairs, MT taps per child column padded with weight 0.
template <typename R, int CPT, int RW, int MT>
__global__ __launch_bounds__(256) void k_l2l_row(int nc, int Lp, int Lc, int ncb, const int* __restrict__ parent,
                                                 const int* __restrict__ oct, const int* __restrict__ win_ptr,
                                                 const int* __restrict__ win_row, const R* __restrict__ win_w,
                                                 const int* __restrict__ ap_tap, const R* __restrict__ ap_w,
                                                 const cplx_t<R>* __restrict__ shdn,
                                                 const cplx_t<R>* __restrict__ Bmp, cplx_t<R>* __restrict__ Bm) {
    using C = cplx_t<R>;
    extern __shared__ __align__(16) unsigned char l2l_lds[];
    const int pfn = 2 * Lp, psn = 2 * Lc, Kp = Lp * pfn, Kc = Lc * psn;
    const int nrg = (Lc + RW - 1) / RW;   // row groups per box
    const int lin = xcd_remap(blockIdx.x, (int)gridDim.x);
    const int cb = lin % ncb, g = (lin / ncb) % nrg, b = lin / (ncb * nrg);   // one box's workgroups are consecutive
    const int r0 = g * RW, nr = min(RW, Lc - r0);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int c0 = (cb * (int)(blockDim.x >> 6) + wave) * CPT;
    C* V = reinterpret_cast<C*>(l2l_lds) + (size_t)wave * CPT * RW * pfn;   // [CPT][RW][2 Lp]
    const C* P = Bmp + ((size_t)parent[b] * nc * 3 + c0) * Kp;
    const C* sh = shdn + (size_t)oct[b] * Kp;
    const int k0 = win_ptr[g], k1 = win_ptr[g + 1];
    for (int jb = 0; jb < pfn; jb += 64) {
        const int jp = min(jb + lane, pfn - 1);
        C acc[RW][CPT];
#pragma unroll
        for (int r = 0; r < RW; ++r)
#pragma unroll
            for (int d = 0; d < CPT; ++d) acc[r][d] = C{0, 0};
        auto load = [&](int k, C& e, C (&v)[CPT]) {
            const int kp = win_row[min(k, k1 - 1)] * pfn + jp;
            e = sh[kp];
#pragma unroll
            for (int d = 0; d < CPT; ++d) v[d] = P[(size_t)d * Kp + kp];
        };
        auto add = [&](int k, const C& e, const C (&v)[CPT]) {
            R w[RW];
#pragma unroll
            for (int r = 0; r < RW; ++r) w[r] = win_w[(size_t)k * RW + r];
#pragma unroll
            for (int d = 0; d < CPT; ++d) {
                const C t = cmul(e, v[d]);
#pragma unroll
                for (int r = 0; r < RW; ++r) {
                    acc[r][d].x = fma(w[r], t.x, acc[r][d].x);
                    acc[r][d].y = fma(w[r], t.y, acc[r][d].y);
                }
            }
        };
        C ea, eb, va[CPT], vb[CPT];
        load(k0, ea, va);
        for (int k = k0; k < k1; k += 2) {
            load(k + 1, eb, vb);
            __builtin_amdgcn_sched_barrier(0);
            add(k, ea, va);
            load(k + 2, ea, va);
            __builtin_amdgcn_sched_barrier(0);
            if (k + 1 < k1) add(k + 1, eb, vb);
        }
        if (jb + lane < pfn)
#pragma unroll
            for (int d = 0; d < CPT; ++d)
#pragma unroll
                for (int r = 0; r < RW; ++r) V[(d * RW + r) * pfn + jp] = acc[r][d];
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // other lanes of this wavefront wrote V
    C* O = Bm + ((size_t)b * nc * 3 + c0) * Kc + (size_t)r0 * psn;
    for (int t = lane; t < nr * psn; t += 64) {
        const int r = t / psn, jc = t - r * psn;
        C o[CPT];
#pragma unroll
        for (int d = 0; d < CPT; ++d) o[d] = O[(size_t)d * Kc + t];
        int ti[MT];
        R tw[MT];
#pragma unroll
        for (int k = 0; k < MT; ++k) {
            ti[k] = r * pfn + ap_tap[k * psn + jc];
            tw[k] = ap_w[k * psn + jc];
        }
#pragma unroll
        for (int d = 0; d < CPT; ++d) {
            C s = C{0, 0};
#pragma unroll
            for (int k = 0; k < MT; ++k) {
                const C v = V[d * RW * pfn + ti[k]];
                s.x = fma(tw[k], v.x, s.x);
                s.y = fma(tw[k], v.y, s.y);
            }
            o[d].x += s.x;
            o[d].y += s.y;
            O[(size_t)d * Kc + t] = o[d];
        }
    }
}

// Child rows per group and the LDS of one wavefront (3 columns, FP64) decide
// whether the pass applies: 4 rows up to 2 Lp = 340, 2 up to 682, else none
// (0: the translation then fuses the anterpolation), and at most 8 taps.
int l2l_rows(int Lp, int taps) {
    if (taps > 8) return 0;
    const size_t row = (size_t)3 * 2 * Lp * sizeof(double2);
    return 4 * row <= 64 * 1024 ? 4 : (2 * row <= 64 * 1024 ? 2 : 0);
}

// taps that the phi pass is compiled for
int l2l_taps(int rw, int taps) { return rw == 2 || taps > 6 ? 8 : std::max(taps, 5); }

template <typename R>
void launch_l2l_row(hipStream_t st, int ncur, int nbox, int Lp, int Lc, int rw, int taps, const int* parent,
                    const int* oct, const int* win_ptr, const int* win_row, const R* win_w, const int* ap_tap,
                    const R* ap_w, const cplx_t<R>* shift_dn, const cplx_t<R>* Bm_parent, cplx_t<R>* Bm) {
    if (nbox == 0) return;
    constexpr int CPT = 3;
    const size_t lds = (size_t)CPT * rw * 2 * Lp * sizeof(cplx_t<R>);   // per wavefront
    if ((rw != 2 && rw != 4) || lds > 64 * 1024 || taps != l2l_taps(rw, taps))
        throw std::invalid_argument("separable anterpolation: rows per wavefront out of range");
    int G = std::min(4, ncur);   // wavefronts (column groups) per workgroup
    while (G > 1 && G * lds > 64 * 1024) G /= 2;
    const int ncb = ncur / G;
    const unsigned grid = (unsigned)nbox * ((Lc + rw - 1) / rw) * ncb;
#define L2LR(RW, MT)                                                                                                  \
    k_l2l_row<R, CPT, RW, MT><<<grid, 64 * G, G * lds, st>>>(ncur, Lp, Lc, ncb, parent, oct, win_ptr, win_row, win_w, \
                                                             ap_tap, ap_w, shift_dn, Bm_parent, Bm)
    if (rw == 2) L2LR(2, 8);
    else if (taps == 5) L2LR(4, 5);
    else if (taps == 6) L2LR(4, 6);
    else L2LR(4, 8);
#undef L2LR
}

// ---------------------------------------------------------------- translation + anterpolation
// Code/ProcessMLFMM.h:112-147 (m2l, quadrature weight folded into TFw) and
// :152-202 (l2l) in gather form: each child sample sums the parent samples whose
// 9-tap stencil contains it (transposed table, ascending parent sample), so no
// atomics and a fixed summation order.
template <typename R, int NC>
__global__ __launch_bounds__(256) void k_m2l_l2l(int nbox, int K, int ktiles, const int* __restrict__ dr_ptr,
                                                 const int* __restrict__ dr_idx, const int* __restrict__ dr_vec,
                                                 const cplx_t<R>* __restrict__ TFw, const cplx_t<R>* __restrict__ Sm,
                                                 int Kp, const int* __restrict__ parent, const int* __restrict__ oct,
                                                 const int* __restrict__ t_ptr, const int* __restrict__ t_kp,
                                                 const R* __restrict__ t_w, const cplx_t<R>* __restrict__ shdn,
                                                 const cplx_t<R>* __restrict__ Bmp, cplx_t<R>* __restrict__ Bm) {
    using C = cplx_t<R>;
    const int lin = xcd_remap(blockIdx.x, nbox * ktiles);
    const int b = lin / ktiles;
    const int q = (lin % ktiles) * blockDim.x + threadIdx.x;
    if (q >= K) return;
    C acc[NC][3];
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int d = 0; d < 3; ++d) acc[c][d] = C{0, 0};
    for (int j = dr_ptr[b]; j < dr_ptr[b + 1]; ++j) {
        const C T = TFw[(size_t)dr_vec[j] * K + q];
        const C* S = Sm + (size_t)dr_idx[j] * NC * 3 * K + q;
#pragma unroll
        for (int cc = 0; cc < NC; ++cc)
#pragma unroll
            for (int d = 0; d < 3; ++d) cfma(acc[cc][d], T, S[(size_t)(cc * 3 + d) * K]);
    }
    if (Bmp != nullptr) {
        const int pb = parent[b];
        const C* sh = shdn + (size_t)oct[b] * Kp;
        const C* P = Bmp + (size_t)pb * NC * 3 * Kp;
        for (int j = t_ptr[q]; j < t_ptr[q + 1]; ++j) {
            const int kp = t_kp[j];
            C e = sh[kp];
            e.x *= t_w[j];
            e.y *= t_w[j];
#pragma unroll
            for (int cc = 0; cc < NC; ++cc)
#pragma unroll
                for (int d = 0; d < 3; ++d) cfma(acc[cc][d], e, P[(size_t)(cc * 3 + d) * Kp + kp]);
        }
    }
    C* o = Bm + (size_t)b * NC * 3 * K + q;
#pragma unroll
    for (int cc = 0; cc < NC; ++cc)
#pragma unroll
        for (int d = 0; d < 3; ++d) o[(size_t)(cc * 3 + d) * K] = acc[cc][d];
}

template <typename R>
void launch_m2l_l2l(hipStream_t st, int ncur, int nbox, int K, const int* dr_ptr, const int* dr_idx,
                    const int* dr_vec, const cplx_t<R>* TFw, const cplx_t<R>* Sm, int Kp, const int* parent,
                    const int* octant, const int* t_ptr, const int* t_kp, const R* t_w, const cplx_t<R>* shift_down,
                    const cplx_t<R>* Bm_parent, cplx_t<R>* Bm) {
    const int kt = (K + 255) / 256;
    dim3 grid(kt * nbox);
#define M2L(NC) k_m2l_l2l<R, NC><<<grid, 256, 0, st>>>(nbox, K, kt, dr_ptr, dr_idx, dr_vec, TFw, Sm, Kp, parent, octant, t_ptr, t_kp, t_w, shift_down, Bm_parent, Bm)
    if (ncur == 1) M2L(1);
    else if (ncur == 2) M2L(2);
    else if (ncur == 4) M2L(4);
    else if (ncur == 8) M2L(8);
    else if constexpr (sizeof(R) == 4) M2L(16);
    else throw std::invalid_argument("FP64 far field: at most 8 workspace currents per pass");
#undef M2L
}

// Sibling-cluster form of the same product: a thread owns one sample q, CPT of
// the nc x 3 workspace columns and all NM (1..4) children of one parent.  It
// walks the union of their distant-relative lists in ascending box order,
// reading each source box's CPT values once and applying them to every member
// with that member's translation vector; a member without the source in its
// list reads the all-zero row the table keeps after its last vector, so the
// member loop has no branches (a member's sum thus runs over its own list in
// ascending box order, plus exact zeros).  The interpolation from the parent
// reads each parent value once for all members.  No LDS and no barriers.
// SP = 2 (FP32): a lane owns two neighbouring samples and loads both with one
// 16-byte load.  An 8-byte load keeps the L1 busy as long as a 16-byte one (16
// against 18 to 20 cycles per wavefront and CU, measured on 64 consecutive
// values), and that data path bounds this kernel.
template <typename R, int SP>
struct SampleVec {
    using type = cplx_t<R>;
};
template <>
struct SampleVec<float, 2> {
    using type = float4;
};
__device__ __forceinline__ float2 sample_of(float4 v, int s) { return s ? make_float2(v.z, v.w) : make_float2(v.x, v.y); }
__device__ __forceinline__ float2 sample_of(float2 v, int) { return v; }
__device__ __forceinline__ double2 sample_of(double2 v, int) { return v; }

template <typename R, int CPT, int SP, int NM>
__device__ __forceinline__ void m2l_cl_body(int nc, int cl, int K, int q, int c0, const int* __restrict__ cl_child,
                                            const int* __restrict__ cl_ptr, const int* __restrict__ cl_src,
                                            const int* __restrict__ cl_vec, const cplx_t<R>* __restrict__ TFw,
                                            const cplx_t<R>* __restrict__ Sm, int Kp, const int* __restrict__ parent,
                                            const int* __restrict__ oct, const int* __restrict__ t_ptr,
                                            const int* __restrict__ t_kp, const R* __restrict__ t_w,
                                            const cplx_t<R>* __restrict__ shdn, const cplx_t<R>* __restrict__ Bmp,
                                            cplx_t<R>* __restrict__ Bm) {
    using C = cplx_t<R>;
    using V = typename SampleVec<R, SP>::type;   // SP samples (q is a multiple of SP, K is even: aligned)
    int child[NM];
#pragma unroll
    for (int k = 0; k < NM; ++k) child[k] = cl_child[cl * 4 + k];
    C acc[NM][CPT][SP];
#pragma unroll
    for (int k = 0; k < NM; ++k)
#pragma unroll
        for (int j = 0; j < CPT; ++j)
#pragma unroll
            for (int p = 0; p < SP; ++p) acc[k][j][p] = C{0, 0};
    const int u0 = cl_ptr[cl], u1 = cl_ptr[cl + 1];
    // software pipeline over two register sets: the next source's values and
    // its members' translation samples are loaded into one set while the
    // other is applied
    V sa[CPT], sb[CPT], ta[NM], tb[NM];
    auto fetch = [&](V (&s)[CPT], V (&t)[NM], int u) {
        const int4 v = *reinterpret_cast<const int4*>(cl_vec + (size_t)u * 4);
        const int vk[4] = {v.x, v.y, v.z, v.w};
        const C* S = Sm + ((size_t)cl_src[u] * nc * 3 + c0) * K + q;
#pragma unroll
        for (int j = 0; j < CPT; ++j) s[j] = *reinterpret_cast<const V*>(S + (size_t)j * K);
#pragma unroll
        for (int k = 0; k < NM; ++k) t[k] = *reinterpret_cast<const V*>(TFw + (size_t)vk[k] * K + q);
    };
    auto apply = [&](const V (&s)[CPT], const V (&t)[NM]) {
#pragma unroll
        for (int k = 0; k < NM; ++k)
#pragma unroll
            for (int j = 0; j < CPT; ++j)
#pragma unroll
                for (int p = 0; p < SP; ++p) cmac(acc[k][j][p], sample_of(t[k], p), sample_of(s[j], p));
    };
    // Sources go in pairs, so that every apply has the other set's loads in
    // flight; the prefetch after a pair is unconditional (the last source is
    // read again past the end), so every path reaches an apply with the same
    // loads outstanding, and the scheduling barriers keep the compiler from
    // sinking the loads to their uses.
    int u = u0;
    if (u < u1) fetch(sa, ta, u);
    for (; u + 1 < u1; u += 2) {
        fetch(sb, tb, u + 1);
        __builtin_amdgcn_sched_barrier(0);
        apply(sa, ta);
        fetch(sa, ta, min(u + 2, u1 - 1));
        __builtin_amdgcn_sched_barrier(0);
        apply(sb, tb);
    }
    if (u < u1) apply(sa, ta);
    if (Bmp != nullptr) {
        const C* P = Bmp + ((size_t)parent[child[0]] * nc * 3 + c0) * Kp;   // siblings share the parent
        const C* sh[NM];
#pragma unroll
        for (int k = 0; k < NM; ++k) sh[k] = shdn + (size_t)oct[child[k]] * Kp;
#pragma unroll
        for (int p = 0; p < SP; ++p)
            for (int j = t_ptr[q + p]; j < t_ptr[q + p + 1]; ++j) {
                const int kp = t_kp[j];
                const R w = t_w[j];
                C pv[CPT];
#pragma unroll
                for (int jj = 0; jj < CPT; ++jj) pv[jj] = P[(size_t)jj * Kp + kp];
#pragma unroll
                for (int k = 0; k < NM; ++k) {
                    C e = sh[k][kp];
                    e.x *= w;
                    e.y *= w;
#pragma unroll
                    for (int jj = 0; jj < CPT; ++jj) cfma(acc[k][jj][p], e, pv[jj]);
                }
            }
    }
#pragma unroll
    for (int k = 0; k < NM; ++k) {
        C* o = Bm + ((size_t)child[k] * nc * 3 + c0) * K + q;
#pragma unroll
        for (int j = 0; j < CPT; ++j) {
            if constexpr (SP == 2)
                *reinterpret_cast<V*>(o + (size_t)j * K) =
                    make_float4(acc[k][j][0].x, acc[k][j][0].y, acc[k][j][SP - 1].x, acc[k][j][SP - 1].y);
            else
                o[(size_t)j * K] = acc[k][j][0];
        }
    }
}

// All-sibling clusters with LDS-staged translation samples (FP32): a cluster
// is every child of one parent (NM <= 8 members; with up to 4 a parent of 5-8
// children needs two clusters, which read the union's sources twice), a
// thread owns one sample q and CPT = 6 columns.  The translation samples of
// the members for kS sources at a time are staged in LDS by the whole
// workgroup, so each is read from memory once per workgroup instead of once
// per column-group wavefront, and a source costs a wavefront CPT vector loads
// (its workspace values) and NM LDS reads.  The staging is double-buffered
// (the next chunk's samples are loaded into registers during the current
// chunk's products, one barrier per chunk); the last chunk is padded with
// zero samples, and members without a source read the table's zero row, so
// the product loop has no branches.  Per sample and member the sums run over
// the same sources in the same order as the other cluster forms (plus exact
// zeros), so the results are identical.
constexpr int kClsS = 4;   // sources per staged chunk (8 spills registers)

template <int NC, int G, int NM>
__device__ __forceinline__ void m2l_cls_body(int cl, int K, int kt, int c0, float2 (*tfs)[kClsS][8][64],
                                             const int* __restrict__ cl_child, const int* __restrict__ cl_ptr,
                                             const int* __restrict__ cl_src, const int* __restrict__ cl_vec,
                                             const float2* __restrict__ TFw, const float2* __restrict__ Sm, int Kp,
                                             const int* __restrict__ parent, const int* __restrict__ oct,
                                             const int* __restrict__ t_ptr, const int* __restrict__ t_kp,
                                             const float* __restrict__ t_w, const float2* __restrict__ shdn,
                                             const float2* __restrict__ Bmp, float2* __restrict__ Bm) {
    using C = float2;
    constexpr int CPT = NC * 3 / G;
    constexpr int NTH = 64 * G;
    constexpr int NE = kClsS * NM * 64, EPT = (NE + NTH - 1) / NTH;   // staged samples per chunk, per thread
    const int lane = threadIdx.x & 63;
    const int q = kt * 64 + lane, qc = min(q, K - 1);   // lanes past K compute on clamped data, store nothing
    int child[NM];
#pragma unroll
    for (int k = 0; k < NM; ++k) child[k] = cl_child[cl * 8 + k];
    C acc[NM][CPT];
#pragma unroll
    for (int k = 0; k < NM; ++k)
#pragma unroll
        for (int j = 0; j < CPT; ++j) acc[k][j] = C{0, 0};
    const int u0 = cl_ptr[cl], u1 = cl_ptr[cl + 1];
    const int nchunk = (u1 - u0 + kClsS - 1) / kClsS;
    // staging: entry e = (s, k, l) of chunk c -> tfs[b][s][k][l]
    C tv[EPT];
    auto stage_load = [&](int c) {
#pragma unroll
        for (int i = 0; i < EPT; ++i) {
            const int e = min((int)threadIdx.x + NTH * i, NE - 1);
            const int s = e / (NM * 64), k = (e / 64) % NM, l = e % 64;
            const int u = u0 + c * kClsS + s;
            const int vid = cl_vec[(size_t)min(u, u1 - 1) * 8 + k];
            const C v = TFw[(size_t)vid * K + min(kt * 64 + l, K - 1)];
            tv[i] = u < u1 ? v : C{0, 0};   // the last chunk's padding applies exact zeros
        }
    };
    auto stage_store = [&](int b) {
#pragma unroll
        for (int i = 0; i < EPT; ++i) {
            const int e = (int)threadIdx.x + NTH * i;
            if (NE % NTH == 0 || e < NE) {
                const int s = e / (NM * 64), k = (e / 64) % NM, l = e % 64;
                tfs[b][s][k][l] = tv[i];
            }
        }
    };
    C sa[CPT], sb[CPT];
    auto fetch = [&](C (&sv)[CPT], int u) {
        const C* S = Sm + ((size_t)cl_src[min(u, u1 - 1)] * NC * 3 + c0) * K + qc;
#pragma unroll
        for (int j = 0; j < CPT; ++j) sv[j] = S[(size_t)j * K];
    };
    auto apply = [&](const C (&sv)[CPT], int b, int s) {
#pragma unroll
        for (int k = 0; k < NM; ++k) {
            const C t = tfs[b][s][k][lane];
#pragma unroll
            for (int j = 0; j < CPT; ++j) cmac(acc[k][j], t, sv[j]);
        }
    };
    if (nchunk > 0) {
        stage_load(0);
        stage_store(0);
        fetch(sa, u0);
        __syncthreads();
        for (int c = 0; c < nchunk; ++c) {
            const int b = c & 1, ub = u0 + c * kClsS;
            stage_load(c + 1 < nchunk ? c + 1 : c);   // the last chunk reloads itself (never stored)
            // kClsS is even: the chunk's first source is in set A
#pragma unroll
            for (int s = 0; s < kClsS; s += 2) {
                fetch(sb, ub + s + 1);
                __builtin_amdgcn_sched_barrier(0);
                apply(sa, b, s);
                fetch(sa, ub + s + 2);
                __builtin_amdgcn_sched_barrier(0);
                apply(sb, b, s + 1);
            }
            if (c + 1 < nchunk) stage_store(b ^ 1);
            __syncthreads();
        }
    }
    if (Bmp != nullptr) {
        const C* P = Bmp + ((size_t)parent[child[0]] * NC * 3 + c0) * Kp;   // siblings share the parent
        const C* sh[NM];
#pragma unroll
        for (int k = 0; k < NM; ++k) sh[k] = shdn + (size_t)oct[child[k]] * Kp;
        for (int j = t_ptr[qc]; j < t_ptr[qc + 1]; ++j) {
            const int kp = t_kp[j];
            const float w = t_w[j];
            C pv[CPT];
#pragma unroll
            for (int jj = 0; jj < CPT; ++jj) pv[jj] = P[(size_t)jj * Kp + kp];
#pragma unroll
            for (int k = 0; k < NM; ++k) {
                C e = sh[k][kp];
                e.x *= w;
                e.y *= w;
#pragma unroll
                for (int jj = 0; jj < CPT; ++jj) cfma(acc[k][jj], e, pv[jj]);
            }
        }
    }
    if (q >= K) return;
#pragma unroll
    for (int k = 0; k < NM; ++k) {
        C* o = Bm + ((size_t)child[k] * NC * 3 + c0) * K + q;
#pragma unroll
        for (int j = 0; j < CPT; ++j) o[(size_t)j * K] = acc[k][j];
    }
}

template <int NC, int G>
__global__ __launch_bounds__(64 * G) void k_m2l_cls(int ncl, int K, int ktiles, int wc,
                                                    const int* __restrict__ cl_child, const int* __restrict__ cl_ptr,
                                                    const int* __restrict__ cl_src, const int* __restrict__ cl_vec,
                                                    const float2* __restrict__ TFw, const float2* __restrict__ Sm,
                                                    int Kp, const int* __restrict__ parent,
                                                    const int* __restrict__ oct, const int* __restrict__ t_ptr,
                                                    const int* __restrict__ t_kp, const float* __restrict__ t_w,
                                                    const float2* __restrict__ shdn, const float2* __restrict__ Bmp,
                                                    float2* __restrict__ Bm) {
    __shared__ float2 tfs[2][kClsS][8][64];
    constexpr int CPT = NC * 3 / G;
    int cl, kt;
    window_order(xcd_remap(blockIdx.x, ncl * ktiles), ncl, ktiles, wc, cl, kt);
    const int c0 = (threadIdx.x >> 6) * CPT;
    // members are packed first; the count is uniform over the workgroup
    int nm = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k) nm += cl_child[cl * 8 + k] >= 0 ? 1 : 0;
#define M2LS(NM)                                                                                                      \
    m2l_cls_body<NC, G, NM>(cl, K, kt, c0, tfs, cl_child, cl_ptr, cl_src, cl_vec, TFw, Sm, Kp, parent, oct, t_ptr,   \
                            t_kp, t_w, shdn, Bmp, Bm)
    switch (nm) {
        case 8: M2LS(8); break;
        case 7: M2LS(7); break;
        case 6: M2LS(6); break;
        case 5: M2LS(5); break;
        case 4: M2LS(4); break;
        case 3: M2LS(3); break;
        case 2: M2LS(2); break;
        default: M2LS(1); break;
    }
#undef M2LS
}

template <typename R>
void launch_m2l_cls(hipStream_t st, int ncur, int ncl, int K, const int* cl_child, const int* cl_ptr,
                    const int* cl_src, const int* cl_vec, const cplx_t<R>* TFw, const cplx_t<R>* Sm, int Kp,
                    const int* parent, const int* octant, const int* t_ptr, const int* t_kp, const R* t_w,
                    const cplx_t<R>* shift_down, const cplx_t<R>* Bm_parent, cplx_t<R>* Bm) {
    if constexpr (sizeof(R) == 8) {
        throw std::invalid_argument("LDS-staged cluster translation: FP32 far field only");
    } else {
        if (ncl == 0) return;
        const int kt = (K + 63) / 64;
        constexpr int wc = 128;
#define M2LS_L(NC)                                                                                                    \
    k_m2l_cls<NC, NC / 2><<<ncl * kt, 32 * NC, 0, st>>>(ncl, K, kt, wc, cl_child, cl_ptr, cl_src, cl_vec, TFw, Sm,   \
                                                         Kp, parent, octant, t_ptr, t_kp, t_w, shift_down,            \
                                                         Bm_parent, Bm)
        if (ncur == 4) M2LS_L(4);
        else if (ncur == 8) M2LS_L(8);
        else if (ncur == 16) M2LS_L(16);
        else throw std::invalid_argument("LDS-staged cluster translation: 4, 8 or 16 workspace currents per pass");
#undef M2LS_L
    }
}

// A workgroup's wavefronts take consecutive clusters, all with one sample tile
// and one group of CPT columns, and the launch goes window by window of wc
// workgroups: tile, then column group, then clusters.  The wavefronts that run
// at once on one XCD so read 64 samples x CPT columns of the boxes around wc
// neighbouring clusters, which its L2 holds, and neighbouring clusters share
// sources in the L1.  With a cluster's column groups as the wavefronts of one
// workgroup the tile's boxes took four times that and a quarter of the reads
// missed the L2: C5 at 64 right-hand sides 30.2 ms per matvec, 29.3 in this
// order, 27.5 with two samples per lane as well.  What is left is shared by the
// L1 (10 loads of 18 cycles per source) and the vector unit (192 cycles of FMA).
template <typename R, int CPT, int SP>
__global__ __launch_bounds__(256) void k_m2l_cl(int nc, int ncl, int K, int ktiles, int wc,
                                                const int* __restrict__ cl_child,
                                                const int* __restrict__ cl_ptr, const int* __restrict__ cl_src,
                                                const int* __restrict__ cl_vec, const cplx_t<R>* __restrict__ TFw,
                                                const cplx_t<R>* __restrict__ Sm, int Kp,
                                                const int* __restrict__ parent, const int* __restrict__ oct,
                                                const int* __restrict__ t_ptr, const int* __restrict__ t_kp,
                                                const R* __restrict__ t_w, const cplx_t<R>* __restrict__ shdn,
                                                const cplx_t<R>* __restrict__ Bmp, cplx_t<R>* __restrict__ Bm) {
    const int W = blockDim.x >> 6, ncg = nc * 3 / CPT, nq = (ncl + W - 1) / W;
    int quad, tile;
    window_order(xcd_remap(blockIdx.x, (int)gridDim.x), nq, ktiles * ncg, wc, quad, tile);
    const int kt = tile / ncg, c0 = (tile - kt * ncg) * CPT;
    const int cl = quad * W + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int q = (kt * 64 + (threadIdx.x & 63)) * SP;
    if (cl >= ncl || q >= K) return;
    // members are packed first; the count is uniform over the wavefront
    const int4 ch = *reinterpret_cast<const int4*>(cl_child + (size_t)cl * 4);
    const int nm = (ch.y >= 0) + (ch.z >= 0) + (ch.w >= 0) + 1;
#define M2LB(NM)                                                                                                      \
    m2l_cl_body<R, CPT, SP, NM>(nc, cl, K, q, c0, cl_child, cl_ptr, cl_src, cl_vec, TFw, Sm, Kp, parent, oct, t_ptr,     \
                            t_kp, t_w, shdn, Bmp, Bm)
    if (nm == 4) M2LB(4);
    else if (nm == 3) M2LB(3);
    else if (nm == 2) M2LB(2);
    else M2LB(1);
#undef M2LB
}

template <typename R>
void launch_m2l_cl(hipStream_t st, int ncur, int ncl, int K, const int* cl_child, const int* cl_ptr,
                   const int* cl_src, const int* cl_vec, const cplx_t<R>* TFw, const cplx_t<R>* Sm, int Kp,
                   const int* parent, const int* octant, const int* t_ptr, const int* t_kp, const R* t_w,
                   const cplx_t<R>* shift_down, const cplx_t<R>* Bm_parent, cplx_t<R>* Bm) {
    if (ncl == 0) return;
    if (ncur != 1 && ncur != 2 && ncur != 4 && ncur != 8 && (ncur != 16 || sizeof(R) == 8))
        throw std::invalid_argument("FP64 far field: at most 8 workspace currents per pass");
    // Columns x samples per thread.  From 4 currents 6 x 2 in FP32 and 6 x 1 in
    // FP64 (16-byte loads both): whole matvec of C5 at 64 right-hand sides, FP32:
    // 6 x 2 27.5 ms, 6 x 1 29.3, 12 x 1 28.5, 3 x 2 28.4, 8 x 2 31.8 (spills into
    // the accumulator file); FP64 lossy sphere at 13: 6 x 1 5.57, 3 x 1 5.77.
    // A level that so has fewer than 1024 wavefronts, one per SIMD, takes one
    // sample per lane, and below 512 of those 3 columns: a wavefront's walk through
    // its sources then bounds the time (5,070 EFIE unknowns in 56 leaves, 64
    // right-hand sides in passes of 8: 236 us of translation with 6 x 2, 180 with 6
    // x 1, 143 with 3 x 1; 52,920 in 824 leaves, 4 of them: 216, 161, 161).  One
    // vector: PMCHWT of 15k unknowns 401 us with 3 columns, 409 with the wide form.
    constexpr bool f64 = sizeof(R) == 8;
    const long long cols = (long long)ncl * ncur / 2;   // wavefronts per sample tile, 6 columns each
    const bool wide = ncur >= 4;
    // pairs need rows of whole pairs (K = 2 L^2 is even)
    const int sp = !f64 && wide && (K & 1) == 0 && cols * ((K + 127) / 128) >= 1024 ? 2 : 1;
    const int kt = (K + 64 * sp - 1) / (64 * sp);
    const int cpt = (wide || (!f64 && ncur == 2)) && cols * kt >= 512 ? 6 : 3;
    const int ncg = ncur * 3 / cpt;
    // Wavefronts (neighbouring clusters) per workgroup; single ones where a level
    // does not give each SIMD four wavefronts.
    const int W = !wide || (long long)ncl * kt * ncg < 4096 ? 1 : 4;
    const int nq = (ncl + W - 1) / W;
    // clusters per window: 512 (measured 27.5 at 512 and 1024, 27.9 at 256), 128 below 4 currents
    const int wc = wide ? 512 / W : 128;
#define M2LC(CPT, SP)                                                                                                 \
    k_m2l_cl<R, CPT, SP><<<nq * kt * ncg, 64 * W, 0, st>>>(ncur, ncl, K, kt, wc, cl_child, cl_ptr, cl_src, cl_vec,   \
                                                           TFw, Sm, Kp, parent, octant, t_ptr, t_kp, t_w,             \
                                                           shift_down, Bm_parent, Bm)
    if (cpt == 3) M2LC(3, 1);
    else if (sp == 1) M2LC(6, 1);
    else if constexpr (!f64) M2LC(6, 2);
#undef M2LC
}

// ---------------------------------------------------------------- disaggregation
// Code/MLFMM.cpp:211-227: w_m += (k eta/4pi)(k/4pi) sum_k Vfmj_m . Bm_leaf.
// Each wavefront owns ROWS consecutive RWG rows (internal order) and streams
// their patterns together, lanes over k, then one wavefront reduction per row
// and right-hand side.  Rows run over the whole RWG range, so small and large
// leaves load the GPU alike.  With RB right-hand sides each pattern load
// serves RB workspaces (current rr of the leaf).
template <typename R, int ROWS, int RB>
__global__ __launch_bounds__(256) void k_disagg_pec(int N, int K, int ldr, int r0, const int* __restrict__ leaf_of,
                                                    const int* __restrict__ perm, const cplx_t<R>* __restrict__ Vf,
                                                    const cplx_t<R>* __restrict__ Bm, double2 c,
                                                    double2* __restrict__ y) {
    using C = cplx_t<R>;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int i00 = (blockIdx.x * 4 + wave) * ROWS;
    if (i00 >= N) return;
    const C* V[ROWS];
    const C* B[ROWS];
    C s[ROWS][RB];
#pragma unroll
    for (int u = 0; u < ROWS; ++u) {
        const int i = min(i00 + u, N - 1);   // rows past N repeat row N-1 and are not written
        V[u] = Vf + (size_t)i * 3 * K;
        B[u] = Bm + (size_t)leaf_of[i] * RB * 3 * K;
#pragma unroll
        for (int rr = 0; rr < RB; ++rr) s[u][rr] = C{0, 0};
    }
    for (int q = lane; q < K; q += 64) {
#pragma unroll
        for (int u = 0; u < ROWS; ++u) {
            const C v0 = V[u][q], v1 = V[u][K + q], v2 = V[u][2 * K + q];
#pragma unroll
            for (int rr = 0; rr < RB; ++rr) {
                const C* b = B[u] + (size_t)rr * 3 * K;
                cfma(s[u][rr], v0, b[q]);
                cfma(s[u][rr], v1, b[K + q]);
                cfma(s[u][rr], v2, b[2 * K + q]);
            }
        }
    }
#pragma unroll
    for (int u = 0; u < ROWS; ++u)
#pragma unroll
        for (int rr = 0; rr < RB; ++rr) s[u][rr] = wave_sum(s[u][rr]);
    // lane u * RB + rr writes row u, right-hand side rr
    if (lane < ROWS * RB) {
        const int u = lane / RB, rr = lane - u * RB;
        C v = s[0][0];
#pragma unroll
        for (int uu = 0; uu < ROWS; ++uu)
#pragma unroll
            for (int q = 0; q < RB; ++q)
                if (uu == u && q == rr) v = s[uu][q];
        if (i00 + u < N) {
            double2* yp = y + (size_t)perm[i00 + u] * ldr + r0 + rr;
            double2 t = *yp;
            cfma(t, c, widen(v));
            *yp = t;
        }
    }
}

// Single-vector disaggregation, both equations (Code/MLFMM.cpp:211-227,
// :285-351).  A wavefront streams ROWS consecutive RWG rows together; rows of
// one leaf share its effective vectors: PEC E = B, PMCHWT (the K integral
// sum (-khat x V).B with khat = -kp is sum V.(kp x B)) for the J and M outputs
//   E_J = a B_J - c kp x B_M,   E_M = c kp x B_J + b B_M
// with a, b, c the wavenumber's constants over the common factor `scale`, which
// multiplies the sums in FP64 (k1: a = b = c = 1).  In FP32 mode the constants
// keep their FP64 value as two FP32 parts, and each wavenumber's sums are added
// in FP64: constants rounded to FP32 scaled every row of an output alike, by up
// to 2^-24, which sums of independent roundings stay below.  216,000 PMCHWT
// unknowns, FP32 product: rounded constants 2.23 ms, as here 2.25, E formed in
// FP64 2.29, and the four sums with B_J, B_M and their curls kept apart 2.57.
// Forming E once per ROWS rows in place of one row's L and K sums cuts the L2
// reads of B, which bounded the row-per-wavefront form (7,680 RWG, 346 MB of
// patterns: 98 us, now 76).  KS = 4: the block's wavefronts split the samples of
// the same rows instead, for few rows (480 RWG, PEC: 11.7 us with four rows a
// wavefront, 4.1 with one a block).
template <typename R>
struct WideConst {   // an FP64 constant, as the sum of two FP32 ones in FP32 mode
    cplx_t<R> hi, lo;
    WideConst(double2 v) {
        hi = cplx_t<R>{(R)v.x, (R)v.y};
        lo = cplx_t<R>{(R)(v.x - (double)hi.x), (R)(v.y - (double)hi.y)};
    }
    __device__ __forceinline__ cplx_t<R> times(cplx_t<R> x) const {
        if constexpr (sizeof(R) == 8) return cmul(hi, x);
        cplx_t<R> p = cmul(lo, x);
        cmac(p, hi, x);   // the low part is added before the product is rounded
        return p;
    }
};

template <typename R>
struct DisaggWave {
    int K;
    const cplx_t<R>*Vf, *Bm;
    const R* kp;
    WideConst<R> a, b, c;
};

// (FP32 PMCHWT by whole rows: three wavefronts per SIMD asked for, 181 registers without)
template <typename R, bool PM, int ROWS, int KS>
__global__ __launch_bounds__(256, sizeof(R) == 4 && PM && ROWS == 4 && KS == 1 ? 3 : 1) void k_disagg_one(
    int N, int nw, int ldr, int r0, const int* __restrict__ leaf_of, const int* __restrict__ perm, DisaggWave<R> w0,
    DisaggWave<R> w1, double2 scale, double2* __restrict__ y) {
    using C = cplx_t<R>;
    constexpr int NO = PM ? 2 : 1;
    constexpr bool APART = PM && sizeof(R) == 4;   // each wavenumber's sums are added in FP64
    __shared__ double2 red[4][ROWS * NO];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int i00 = (KS == 1 ? blockIdx.x * 4 + wave : blockIdx.x) * ROWS;
    if (KS == 1 && i00 >= N) return;
    int leaf[ROWS];
#pragma unroll
    for (int u = 0; u < ROWS; ++u) leaf[u] = __builtin_amdgcn_readfirstlane(leaf_of[min(i00 + u, N - 1)]);
    C s[ROWS][NO];
#pragma unroll
    for (int u = 0; u < ROWS; ++u)
#pragma unroll
        for (int o = 0; o < NO; ++o) s[u][o] = C{0, 0};
    auto leave = [&](bool add) {   // the sums so far into red, or added to what is there
#pragma unroll
        for (int u = 0; u < ROWS; ++u)
#pragma unroll
            for (int o = 0; o < NO; ++o) s[u][o] = wave_sum(s[u][o]);
        if (lane == 0)
#pragma unroll
            for (int u = 0; u < ROWS; ++u)
#pragma unroll
                for (int o = 0; o < NO; ++o) {
                    double2& r = red[wave][u * NO + o];
                    r = add ? cadd(r, widen(s[u][o])) : widen(s[u][o]);
                }
    };
    for (int w = 0; w < nw; ++w) {
        const DisaggWave<R> W = w == 0 ? w0 : w1;
        const int K = W.K;
        for (int q = lane + (KS == 1 ? 0 : 64 * wave); q < K; q += 64 * KS) {
            C v[ROWS][3];
#pragma unroll
            for (int u = 0; u < ROWS; ++u) {
                const C* V = W.Vf + (size_t)min(i00 + u, N - 1) * 3 * K + q;   // rows past N repeat N-1
#pragma unroll
                for (int d = 0; d < 3; ++d) v[u][d] = V[(size_t)d * K];
            }
            C e[NO][3];
#pragma unroll
            for (int u = 0; u < ROWS; ++u) {
                if (u == 0 || leaf[u] != leaf[u - 1]) {   // uniform over the wavefront
                    const C* B = W.Bm + (size_t)leaf[u] * NO * 3 * K + q;
#pragma unroll
                    for (int d = 0; d < 3; ++d) e[0][d] = B[(size_t)d * K];
                    if constexpr (PM) {
                        const R kx = W.kp[q], ky = W.kp[K + q], kz = W.kp[2 * K + q];
                        const C j0 = e[0][0], j1 = e[0][1], j2 = e[0][2];
                        const C m0 = B[(size_t)3 * K], m1 = B[(size_t)4 * K], m2 = B[(size_t)5 * K];
                        // kp x B
                        const C cj[3] = {csub(cscale(j2, ky), cscale(j1, kz)), csub(cscale(j0, kz), cscale(j2, kx)),
                                         csub(cscale(j1, kx), cscale(j0, ky))};
                        const C cm[3] = {csub(cscale(m2, ky), cscale(m1, kz)), csub(cscale(m0, kz), cscale(m2, kx)),
                                         csub(cscale(m1, kx), cscale(m0, ky))};
                        const C m[3] = {m0, m1, m2};
#pragma unroll
                        for (int d = 0; d < 3; ++d) {
                            e[0][d] = csub(W.a.times(e[0][d]), W.c.times(cm[d]));
                            e[NO - 1][d] = cadd(W.c.times(cj[d]), W.b.times(m[d]));
                        }
                    }
                }
#pragma unroll
                for (int o = 0; o < NO; ++o)
#pragma unroll
                    for (int d = 0; d < 3; ++d) cfma(s[u][o], v[u][d], e[o][d]);
            }
        }
        if (APART && w == 0) {
            leave(false);
#pragma unroll
            for (int u = 0; u < ROWS; ++u)
#pragma unroll
                for (int o = 0; o < NO; ++o) s[u][o] = C{0, 0};
        }
    }
    leave(APART);
    if (KS > 1) {
        __syncthreads();
        if (wave > 0) return;
    } else {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // lane 0 of this wavefront wrote red
    }
    if (lane < ROWS * NO) {   // lane u * NO + o writes row u, output o
        const int u = lane / NO, o = lane - u * NO;
        double2 v = red[wave][lane];
        if (KS > 1)
            for (int k = 1; k < 4; ++k) v = cadd(v, red[k][lane]);
        if (i00 + u < N) {
            double2* yp = y + ((size_t)o * N + perm[i00 + u]) * ldr + r0;
            double2 t = *yp;
            cfma(t, scale, v);
            *yp = t;
        }
    }
}

// Rows per wavefront and sample split by the number of rows: very few rows take
// one row a block, more take four rows a block whose wavefronts split the
// samples, and from 16,384 rows a wavefront takes four whole rows (300,000 RWG:
// 809 us, 6.0 TB/s).  Measured, FP64, PEC and PMCHWT, in us: one row against four
// rows split, 1,080 RWG 9.1 / 11.0 and 22 / 25, 3,000 RWG 14.9 / 16.5 and 47 / 49,
// 7,680 RWG 30.6 / 31.3 and 103 / 91; four rows split against four whole rows,
// 7,680 RWG 31.3 / 31.2 and 91 / 113, 18,750 RWG 64 / 68 and 176 / 196, 147,000
// RWG 401 / 413 and 1,242 / 1,317 (FP32 690 / 671).  The split form loses only in
// FP32 PMCHWT at large sizes, so the upper line could lie higher elsewhere.
template <typename R, bool PM>
void disagg_one(hipStream_t st, int N, int nw, int ldr, int r0, const int* leaf_of, const int* perm,
                const DisaggWave<R>& w0, const DisaggWave<R>& w1, double2 scale, double2* y) {
    if (N >= 16384)
        k_disagg_one<R, PM, 4, 1><<<(N + 15) / 16, 256, 0, st>>>(N, nw, ldr, r0, leaf_of, perm, w0, w1, scale, y);
    else if (N >= 2048)
        k_disagg_one<R, PM, 4, 4><<<(N + 3) / 4, 256, 0, st>>>(N, nw, ldr, r0, leaf_of, perm, w0, w1, scale, y);
    else
        k_disagg_one<R, PM, 1, 4><<<N, 256, 0, st>>>(N, nw, ldr, r0, leaf_of, perm, w0, w1, scale, y);
}

template <typename R>
void launch_disagg_pec_b(hipStream_t st, int rb, int N, int K, int ldr, int r0, const int* leaf_of, const int* perm,
                         const cplx_t<R>* Vf, const cplx_t<R>* Bm, double2 c, double2* y) {
#define DIS(ROWS, RB)                                                                                      \
    k_disagg_pec<R, ROWS, RB><<<(N + 4 * ROWS - 1) / (4 * ROWS), 256, 0, st>>>(N, K, ldr, r0, leaf_of, perm, Vf, \
                                                                               Bm, c, y)
    if (rb == 1) {
        const double2 one = make_double2(1.0, 0.0);
        const DisaggWave<R> w{K, Vf, Bm, nullptr, one, one, one};
        disagg_one<R, false>(st, N, 1, ldr, r0, leaf_of, perm, w, w, c, y);
    } else if (rb == 2) DIS(2, 2);
    else if (rb == 4) DIS(1, 4);
    else DIS(1, 8);
#undef DIS
}

template <typename R>
void launch_disagg_pec(hipStream_t st, int N, int K, const int* leaf_of, const int* perm, const cplx_t<R>* Vf,
                       const cplx_t<R>* Bm, double2 c, double2* y) {
    launch_disagg_pec_b<R>(st, 1, N, K, 1, 0, leaf_of, perm, Vf, Bm, c, y);
}

// Code/MLFMM.cpp:285-351.  The K integral sum (-khat x V).B with khat = -kp is
// evaluated as sum V.(kp x B).  Sums of RB right-hand sides: s[rr] = {LJ, KJ, LM, KM}.
template <typename R, int RB>
__device__ __forceinline__ void far_sums(int K, const cplx_t<R>* __restrict__ V, const cplx_t<R>* __restrict__ B,
                                         const R* __restrict__ kp, int lane, cplx_t<R> (&s)[RB][4]) {
    using C = cplx_t<R>;
    for (int q = lane; q < K; q += 64) {
        const R kx = kp[q], ky = kp[K + q], kz = kp[2 * K + q];
        const C v0 = V[q], v1 = V[K + q], v2 = V[2 * K + q];
#pragma unroll
        for (int rr = 0; rr < RB; ++rr) {
            const C* BJ = B + (size_t)rr * 6 * K;
            const C* BM = BJ + (size_t)3 * K;
            const C j0 = BJ[q], j1 = BJ[K + q], j2 = BJ[2 * K + q];
            const C m0 = BM[q], m1 = BM[K + q], m2 = BM[2 * K + q];
            cfma(s[rr][0], v0, j0);
            cfma(s[rr][0], v1, j1);
            cfma(s[rr][0], v2, j2);
            cfma(s[rr][2], v0, m0);
            cfma(s[rr][2], v1, m1);
            cfma(s[rr][2], v2, m2);
            // kp x B
            const C cj0 = csub(cscale(j2, ky), cscale(j1, kz));
            const C cj1 = csub(cscale(j0, kz), cscale(j2, kx));
            const C cj2 = csub(cscale(j1, kx), cscale(j0, ky));
            const C cm0 = csub(cscale(m2, ky), cscale(m1, kz));
            const C cm1 = csub(cscale(m0, kz), cscale(m2, kx));
            const C cm2 = csub(cscale(m1, kx), cscale(m0, ky));
            cfma(s[rr][1], v0, cj0);
            cfma(s[rr][1], v1, cj1);
            cfma(s[rr][1], v2, cj2);
            cfma(s[rr][3], v0, cm0);
            cfma(s[rr][3], v1, cm1);
            cfma(s[rr][3], v2, cm2);
        }
    }
}

// One wavefront per RWG row over the whole RWG range (four rows per block).
template <typename R, int RB>
__global__ __launch_bounds__(256) void k_disagg_pmchwt(int ldr, int r0, const int* __restrict__ leaf_of,
                                                       const int* __restrict__ perm, PmchwtFarArgs<R> a,
                                                       double2* __restrict__ y) {
    using C = cplx_t<R>;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int i = blockIdx.x * 4 + wave;
    if (i >= a.N) return;
    const int leaf = leaf_of[i];
    C s1[RB][4], s2[RB][4];
#pragma unroll
    for (int rr = 0; rr < RB; ++rr)
#pragma unroll
        for (int f = 0; f < 4; ++f) s1[rr][f] = s2[rr][f] = C{0, 0};
    far_sums<R, RB>(a.K1, a.Vf1 + (size_t)i * 3 * a.K1, a.B1 + (size_t)leaf * RB * 6 * a.K1, a.kp1, lane, s1);
    far_sums<R, RB>(a.K2, a.Vf2 + (size_t)i * 3 * a.K2, a.B2 + (size_t)leaf * RB * 6 * a.K2, a.kp2, lane, s2);
#pragma unroll
    for (int rr = 0; rr < RB; ++rr)
#pragma unroll
        for (int f = 0; f < 4; ++f) {
            s1[rr][f] = wave_sum(s1[rr][f]);
            s2[rr][f] = wave_sum(s2[rr][f]);
        }
    if (lane < RB) {
        C t1[4], t2[4];
#pragma unroll
        for (int f = 0; f < 4; ++f) t1[f] = s1[0][f], t2[f] = s2[0][f];
#pragma unroll
        for (int rr = 1; rr < RB; ++rr)
            if (lane == rr)
#pragma unroll
                for (int f = 0; f < 4; ++f) t1[f] = s1[rr][f], t2[f] = s2[rr][f];
        const double2 L1J = widen(t1[0]), K1J = widen(t1[1]), L1M = widen(t1[2]), K1M = widen(t1[3]);
        const double2 L2J = widen(t2[0]), K2J = widen(t2[1]), L2M = widen(t2[2]), K2M = widen(t2[3]);
        const int r = perm[i];
        double2* pj = y + (size_t)r * ldr + r0 + lane;
        double2* pm = y + ((size_t)a.N + r) * ldr + r0 + lane;
        double2 wj = *pj, wm = *pm;
        // Code/MLFMM.cpp:339-349
        wj = cadd(wj, cmul(a.c1, L1J));
        wj = csub(wj, cmul(a.c1, K1M));
        wm = cadd(wm, cmul(a.c1, K1J));
        wm = cadd(wm, cmul(a.c1, L1M));
        wj = cadd(wj, cmul(cmul(a.c2, a.etai), L2J));
        wj = csub(wj, cmul(a.c2, K2M));
        wm = cadd(wm, cmul(a.c2, K2J));
        wm = cadd(wm, cmul(cmul(a.c2, L2M), a.inv_etai));
        *pj = wj;
        *pm = wm;
    }
}

template <typename R>
void launch_disagg_pmchwt_b(hipStream_t st, int rb, int ldr, int r0, const int* leaf_of, const int* perm,
                            const PmchwtFarArgs<R>& a, double2* y) {
    const int blocks = (a.N + 3) / 4;
    if (rb == 1) {
        using Z = std::complex<double>;
        auto z = [](double2 v) { return Z(v.x, v.y); };
        auto d = [](Z v) { return make_double2(v.real(), v.imag()); };
        const double2 one = make_double2(1.0, 0.0);
        const Z c = z(a.c2) / z(a.c1);
        const DisaggWave<R> w0{a.K1, a.Vf1, a.B1, a.kp1, one, one, one};
        const DisaggWave<R> w1{a.K2, a.Vf2, a.B2, a.kp2, d(c * z(a.etai)), d(c * z(a.inv_etai)), d(c)};
        disagg_one<R, true>(st, a.N, 2, ldr, r0, leaf_of, perm, w0, w1, a.c1, y);
    } else if (rb == 2) k_disagg_pmchwt<R, 2><<<blocks, 256, 0, st>>>(ldr, r0, leaf_of, perm, a, y);
    else if (rb == 4) k_disagg_pmchwt<R, 4><<<blocks, 256, 0, st>>>(ldr, r0, leaf_of, perm, a, y);
    else if constexpr (sizeof(R) == 4) k_disagg_pmchwt<R, 8><<<blocks, 256, 0, st>>>(ldr, r0, leaf_of, perm, a, y);
    else throw std::invalid_argument("FP64 disaggregation: at most 4 right-hand sides per pass");
}

template <typename R>
void launch_disagg_pmchwt(hipStream_t st, const int* leaf_of, const int* perm, const PmchwtFarArgs<R>& a,
                          double2* y) {
    launch_disagg_pmchwt_b<R>(st, 1, 1, 0, leaf_of, perm, a, y);
}

__global__ void k_narrow(size_t n, const double2* __restrict__ in, float2* __restrict__ out) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        narrow(in[i], out[i]);
}

void launch_narrow(hipStream_t st, size_t n, const double2* in, float2* out) {
    if (n == 0) return;
    const size_t blocks = std::min<size_t>((n + 255) / 256, 65536);
    k_narrow<<<(unsigned)blocks, 256, 0, st>>>(n, in, out);
}

#define MLFMA_FAR_INSTANTIATE(R)                                                                                    \
    template void launch_aggregate<R>(hipStream_t, int, int, int, int, const int*, const int*, const int*,         \
                                      const cplx_t<R>*, const double2*, cplx_t<R>*);                                      \
    template void launch_m2m<R>(hipStream_t, int, int, int, int, const int*, const int*, const int*, const int*,   \
                                const R*, const cplx_t<R>*, const cplx_t<R>*, cplx_t<R>*);                                     \
    template void launch_m2l_l2l<R>(hipStream_t, int, int, int, const int*, const int*, const int*, const cplx_t<R>*,  \
                                    const cplx_t<R>*, int, const int*, const int*, const int*, const int*, const R*,   \
                                    const cplx_t<R>*, const cplx_t<R>*, cplx_t<R>*);                                           \
    template void launch_disagg_pec<R>(hipStream_t, int, int, const int*, const int*, const cplx_t<R>*, const cplx_t<R>*,  \
                                       double2, double2*);                                                        \
    template void launch_disagg_pmchwt<R>(hipStream_t, const int*, const int*, const PmchwtFarArgs<R>&, double2*); \
    template void launch_aggregate_b<R>(hipStream_t, int, int, int, int, int, int, int, const int*, const int*,     \
                                        const int*, const cplx_t<R>*, const double2*, cplx_t<R>*);                \
    template void launch_disagg_pec_b<R>(hipStream_t, int, int, int, int, int, const int*, const int*,             \
                                         const cplx_t<R>*, const cplx_t<R>*, double2, double2*);                  \
    template void launch_disagg_pmchwt_b<R>(hipStream_t, int, int, int, const int*, const int*,                    \
                                            const PmchwtFarArgs<R>&, double2*);                                   \
    template void launch_m2m_row<R>(hipStream_t, int, int, int, int, int, const int*, const int*, const int*,      \
                                    const int*, const int*, const R*, const int*, const R*, const cplx_t<R>*,     \
                                    const cplx_t<R>*, cplx_t<R>*);                                                \
    template void launch_m2l_cls<R>(hipStream_t, int, int, int, const int*, const int*, const int*, const int*,      \
                                    const cplx_t<R>*, const cplx_t<R>*, int, const int*, const int*, const int*,  \
                                    const int*, const R*, const cplx_t<R>*, const cplx_t<R>*, cplx_t<R>*);        \
    template void launch_m2l_cl<R>(hipStream_t, int, int, int, const int*, const int*, const int*, const int*,      \
                                   const cplx_t<R>*, const cplx_t<R>*, int, const int*, const int*, const int*,   \
                                   const int*, const R*, const cplx_t<R>*, const cplx_t<R>*, cplx_t<R>*);       \
    template void launch_l2l_row<R>(hipStream_t, int, int, int, int, int, int, const int*, const int*, const int*,  \
                                    const int*, const R*, const int*, const R*, const cplx_t<R>*,                 \
                                    const cplx_t<R>*, cplx_t<R>*);
MLFMA_FAR_INSTANTIATE(double)
MLFMA_FAR_INSTANTIATE(float)
#undef MLFMA_FAR_INSTANTIATE

// ---------------------------------------------------------------- near field
// Code/MLFMM.cpp:228-231 (PEC) and :354-366 (PMCHWT).  All near blocks of one
// target leaf form a single column-major nt x C_t matrix per plane (PMCHWT:
// z11, zK, z22 with z12 = -zK, z21 = zK, Code/Zmartix.h:611-614), so one
// workgroup streams one contiguous range of HBM.  For nt < BS the BS threads
// form G = BS / nt column groups of nt rows and group g takes the columns
// c = g (mod G): thread tid reads entry c * nt + tid, so the workgroup reads
// consecutive addresses; U columns per thread are in flight at once.  The
// group partials are summed in LDS in a fixed order.  x is gathered into LDS
// CH columns at a time.  Entries are stored in S (double or float) and
// accumulated in FP64.  SPLIT: a workgroup takes the column range of one
// NearDev::split item instead of the whole block row and leaves its rows'
// partial sums in `part`, which k_near_fold adds up.
template <typename S, int P, int BS, int U, int CH, bool SPLIT>
__global__ __launch_bounds__(BS) void k_near(NearDev nd, const cplx_t<S>* __restrict__ Z,
                                             const double2* __restrict__ x, double2* __restrict__ y,
                                             double2* __restrict__ part) {
    constexpr int NX = (P == 3) ? 2 : 1;
    __shared__ double2 xs[NX][CH];
    __shared__ double2 red[NX][BS];
    const int4 it = SPLIT ? nd.split[blockIdx.x] : make_int4(nd.order[blockIdx.x], 0, 0, 0);
    const int t = it.x;
    const int i0 = nd.leaf_ptr[t], nt = nd.leaf_ptr[t + 1] - i0;
    if (nt == 0) return;
    const int C = nd.tgt_cols[t];
    const int ca = SPLIT ? it.y : 0, cb = SPLIT ? it.z : C;   // this workgroup's columns
    if (SPLIT) part += nd.part_ptr[t] + (size_t)it.w * NX * nt;
    const int* cref = nd.colref + nd.col_ptr[t];
    const int plane = C * nt;   // < 2^31: one target's block row
    const cplx_t<S>* Zt = Z + nd.tgt_off[t];
    const int span = nt < BS ? nt : BS;
    const int G = BS / span;
    const int g = threadIdx.x / span, rl = threadIdx.x - g * span;
    for (int r0 = 0; r0 < nt; r0 += span) {
        const int row = r0 + rl;
        const bool act = g < G && row < nt;
        double2 aJ = {0, 0}, aM = {0, 0};
        for (int c0 = ca; c0 < cb; c0 += CH) {
            const int cl = min(CH, cb - c0);
            __syncthreads();
            for (int c = threadIdx.x; c < cl; c += BS) {
                const int r = cref[c0 + c];
                xs[0][c] = x[r];
                if (P == 3) xs[NX - 1][c] = x[nd.N + r];
            }
            __syncthreads();
            if (act) {
                const cplx_t<S>* z = Zt + c0 * nt + row;
                const int step = G * nt;
                int c = g;
                if (P == 1) {
                    for (; c + (U - 1) * G < cl; c += U * G) {
                        double2 zz[U];
#pragma unroll
                        for (int u = 0; u < U; ++u) zz[u] = widen(z[c * nt + u * step]);
#pragma unroll
                        for (int u = 0; u < U; ++u) cfma(aJ, zz[u], xs[0][c + u * G]);
                    }
                    for (; c < cl; c += G) cfma(aJ, widen(z[c * nt]), xs[0][c]);
                } else {
                    for (; c + (U - 1) * G < cl; c += U * G) {
                        double2 p[U], k[U], m[U];
#pragma unroll
                        for (int u = 0; u < U; ++u) {
                            const int o = c * nt + u * step;
                            p[u] = widen(z[o]);
                            k[u] = widen(z[o + plane]);
                            m[u] = widen(z[o + 2 * plane]);
                        }
#pragma unroll
                        for (int u = 0; u < U; ++u) {
                            const double2 xJ = xs[0][c + u * G], xM = xs[NX - 1][c + u * G];
                            cfma(aJ, p[u], xJ);
                            cfms(aJ, k[u], xM);
                            cfma(aM, k[u], xJ);
                            cfma(aM, m[u], xM);
                        }
                    }
                    for (; c < cl; c += G) {
                        const int o = c * nt;
                        const double2 p0 = widen(z[o]), k0 = widen(z[o + plane]), m0 = widen(z[o + 2 * plane]);
                        const double2 xJ = xs[0][c], xM = xs[NX - 1][c];
                        cfma(aJ, p0, xJ);
                        cfms(aJ, k0, xM);
                        cfma(aM, k0, xJ);
                        cfma(aM, m0, xM);
                    }
                }
            }
        }
        // row `q` of the leaf is done (column groups folded)
        auto put = [&](int q, double2 sJ, double2 sM) {
            if (SPLIT) {
                part[q] = sJ;
                if (P == 3) part[nt + q] = sM;
            } else {
                const int r = nd.perm[i0 + q];
                y[r] = sJ;
                if (P == 3) y[nd.N + r] = sM;
            }
        };
        if (G > 1) {   // nt < BS: a single row pass, fold the column groups
            red[0][threadIdx.x] = aJ;
            if (P == 3) red[NX - 1][threadIdx.x] = aM;
            __syncthreads();
            if (threadIdx.x < nt) {
                double2 sJ = red[0][threadIdx.x], sM = red[NX - 1][threadIdx.x];
                for (int h = 1; h < G; ++h) {
                    sJ = cadd(sJ, red[0][h * nt + threadIdx.x]);
                    if (P == 3) sM = cadd(sM, red[NX - 1][h * nt + threadIdx.x]);
                }
                put(threadIdx.x, sJ, sM);
            }
        } else if (act) {   // G == 1: threads past nt hold no row
            put(row, aJ, aM);
        }
    }
}

// y of the split near product: each row's partial sums in item order.
template <int P>
__global__ __launch_bounds__(256) void k_near_fold(NearDev nd, const int* __restrict__ leaf_of,
                                                   const double2* __restrict__ part, double2* __restrict__ y) {
    constexpr int NX = (P == 3) ? 2 : 1;
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= NX * nd.N) return;
    const int cur = e / nd.N, i = e - cur * nd.N;
    const int t = leaf_of[i], i0 = nd.leaf_ptr[t], nt = nd.leaf_ptr[t + 1] - i0;
    const size_t p0 = nd.part_ptr[t];
    const int cnt = (int)((nd.part_ptr[t + 1] - p0) / ((size_t)NX * nt));
    const double2* p = part + p0 + (size_t)cur * nt + (i - i0);
    const size_t step = (size_t)NX * nt;
    double2 s = p[0];
    int k = 1;
    for (; k + 7 < cnt; k += 8) {   // eight loads in flight
        double2 a[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) a[u] = p[(size_t)(k + u) * step];
#pragma unroll
        for (int u = 0; u < 8; ++u) s = cadd(s, a[u]);
    }
    for (; k < cnt; ++k) s = cadd(s, p[(size_t)k * step]);
    y[(size_t)cur * nd.N + nd.perm[i]] = s;
}

template <typename S>
void launch_near(hipStream_t st, const NearDev& nd, const cplx_t<S>* Z, const double2* x, double2* y) {
    if (nd.nleaf == 0) return;
    const int nsplit = sizeof(S) == 8 ? nd.nsplit : nd.nsplit32;
    if (nsplit > 0) {   // few or large leaves (Engine::build_near_split)
        const int NX = nd.planes == 1 ? 1 : 2, fb = (NX * nd.N + 255) / 256;
        if (nd.planes == 1) {
            k_near<S, 1, 512, 8, 1024, true><<<nsplit, 512, 0, st>>>(nd, Z, x, y, nd.part);
            k_near_fold<1><<<fb, 256, 0, st>>>(nd, nd.leaf_of, nd.part, y);
        } else {
            k_near<S, 3, 512, 4, 512, true><<<nsplit, 512, 0, st>>>(nd, Z, x, y, nd.part);
            k_near_fold<3><<<fb, 256, 0, st>>>(nd, nd.leaf_of, nd.part, y);
        }
        return;
    }
    if (nd.planes == 1) k_near<S, 1, 512, 8, 1024, false><<<nd.nleaf, 512, 0, st>>>(nd, Z, x, y, nullptr);
    else k_near<S, 3, 512, 4, 512, false><<<nd.nleaf, 512, 0, st>>>(nd, Z, x, y, nullptr);
}
template void launch_near<double>(hipStream_t, const NearDev&, const double2*, const double2*, double2*);
template void launch_near<float>(hipStream_t, const NearDev&, const float2*, const double2*, double2*);

// Batched near product: RB right-hand sides per pass over the entries (vectors
// RHS-fastest, element (u, r) at u * ldr + r).  Same column-group scheme as
// k_near with 256 threads; the x chunk is staged as [column][rhs] and each
// thread keeps RB (PMCHWT: 2 RB) FP64 accumulators.
template <typename S, int P, int RB, int U, int CH>
__global__ __launch_bounds__(256) void k_near_b(NearDev nd, int ldr, int r0, const cplx_t<S>* __restrict__ Z,
                                                const double2* __restrict__ x, double2* __restrict__ y) {
    constexpr int NX = (P == 3) ? 2 : 1;
    constexpr int BS = 256;
    __shared__ double2 xs[NX][CH][RB];
    __shared__ double2 red[NX][BS];
    const int t = nd.order[blockIdx.x];
    const int i0 = nd.leaf_ptr[t], nt = nd.leaf_ptr[t + 1] - i0;
    if (nt == 0) return;
    const int C = nd.tgt_cols[t];
    const int* cref = nd.colref + nd.col_ptr[t];
    const int plane = C * nt;
    const cplx_t<S>* Zt = Z + nd.tgt_off[t];
    const int span = nt < BS ? nt : BS;
    const int G = BS / span;
    const int g = threadIdx.x / span, rl = threadIdx.x - g * span;
    for (int rs = 0; rs < nt; rs += span) {
        const int row = rs + rl;
        const bool act = g < G && row < nt;
        double2 aJ[RB], aM[RB];
#pragma unroll
        for (int rr = 0; rr < RB; ++rr) aJ[rr] = aM[rr] = make_double2(0.0, 0.0);
        for (int c0 = 0; c0 < C; c0 += CH) {
            const int cl = min(CH, C - c0);
            __syncthreads();
            for (int e = threadIdx.x; e < cl * RB; e += BS) {
                const int c = e / RB, rr = e - c * RB;
                const int r = cref[c0 + c];
                xs[0][c][rr] = x[(size_t)r * ldr + r0 + rr];
                if (P == 3) xs[NX - 1][c][rr] = x[((size_t)nd.N + r) * ldr + r0 + rr];
            }
            __syncthreads();
            if (act) {
                const cplx_t<S>* z = Zt + c0 * nt + row;
                const int step = G * nt;
                int c = g;
                for (; c + (U - 1) * G < cl; c += U * G) {
                    double2 p[U], k[U], m[U];
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        const int o = c * nt + u * step;
                        p[u] = widen(z[o]);
                        if (P == 3) {
                            k[u] = widen(z[o + plane]);
                            m[u] = widen(z[o + 2 * plane]);
                        }
                    }
#pragma unroll
                    for (int u = 0; u < U; ++u)
#pragma unroll
                        for (int rr = 0; rr < RB; ++rr) {
                            const double2 xJ = xs[0][c + u * G][rr];
                            cfma(aJ[rr], p[u], xJ);
                            if (P == 3) {
                                const double2 xM = xs[NX - 1][c + u * G][rr];
                                cfms(aJ[rr], k[u], xM);
                                cfma(aM[rr], k[u], xJ);
                                cfma(aM[rr], m[u], xM);
                            }
                        }
                }
                for (; c < cl; c += G) {
                    const int o = c * nt;
                    const double2 p0 = widen(z[o]);
                    double2 k0 = p0, m0 = p0;
                    if (P == 3) {
                        k0 = widen(z[o + plane]);
                        m0 = widen(z[o + 2 * plane]);
                    }
#pragma unroll
                    for (int rr = 0; rr < RB; ++rr) {
                        const double2 xJ = xs[0][c][rr];
                        cfma(aJ[rr], p0, xJ);
                        if (P == 3) {
                            const double2 xM = xs[NX - 1][c][rr];
                            cfms(aJ[rr], k0, xM);
                            cfma(aM[rr], k0, xJ);
                            cfma(aM[rr], m0, xM);
                        }
                    }
                }
            }
        }
        // fold the column groups one right-hand side at a time
#pragma unroll
        for (int rr = 0; rr < RB; ++rr) {
            if (G > 1) {
                __syncthreads();
                red[0][threadIdx.x] = aJ[rr];
                if (P == 3) red[NX - 1][threadIdx.x] = aM[rr];
                __syncthreads();
                if (threadIdx.x < nt) {
                    double2 sJ = red[0][threadIdx.x], sM = red[NX - 1][threadIdx.x];
                    for (int h = 1; h < G; ++h) {
                        sJ = cadd(sJ, red[0][h * nt + threadIdx.x]);
                        if (P == 3) sM = cadd(sM, red[NX - 1][h * nt + threadIdx.x]);
                    }
                    const size_t r = nd.perm[i0 + threadIdx.x];
                    y[r * ldr + r0 + rr] = sJ;
                    if (P == 3) y[((size_t)nd.N + r) * ldr + r0 + rr] = sM;
                }
            } else if (act) {
                const size_t r = nd.perm[i0 + row];
                y[r * ldr + r0 + rr] = aJ[rr];
                if (P == 3) y[((size_t)nd.N + r) * ldr + r0 + rr] = aM[rr];
            }
        }
    }
}

template <typename S>
void launch_near_b(hipStream_t st, int rb, int ldr, int r0, const NearDev& nd, const cplx_t<S>* Z, const double2* x,
                   double2* y) {
    if (nd.nleaf == 0) return;
    if (rb == 1) {
        if (ldr == 1 && r0 == 0) launch_near<S>(st, nd, Z, x, y);
        else if (nd.planes == 1) k_near_b<S, 1, 1, 8, 512><<<nd.nleaf, 256, 0, st>>>(nd, ldr, r0, Z, x, y);
        else k_near_b<S, 3, 1, 4, 256><<<nd.nleaf, 256, 0, st>>>(nd, ldr, r0, Z, x, y);
    } else if (nd.planes == 1) {
        if (rb == 2) k_near_b<S, 1, 2, 8, 512><<<nd.nleaf, 256, 0, st>>>(nd, ldr, r0, Z, x, y);
        else if (rb == 4) k_near_b<S, 1, 4, 4, 256><<<nd.nleaf, 256, 0, st>>>(nd, ldr, r0, Z, x, y);
        else k_near_b<S, 1, 8, 4, 256><<<nd.nleaf, 256, 0, st>>>(nd, ldr, r0, Z, x, y);
    } else {
        if (rb == 2) k_near_b<S, 3, 2, 2, 256><<<nd.nleaf, 256, 0, st>>>(nd, ldr, r0, Z, x, y);
        else k_near_b<S, 3, 4, 2, 128><<<nd.nleaf, 256, 0, st>>>(nd, ldr, r0, Z, x, y);
    }
}
template void launch_near_b<double>(hipStream_t, int, int, int, const NearDev&, const double2*, const double2*,
                                    double2*);
template void launch_near_b<float>(hipStream_t, int, int, int, const NearDev&, const float2*, const double2*,
                                   double2*);

}  // namespace mlfma
