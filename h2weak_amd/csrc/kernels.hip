// kernels.hip -- gfx950 kernels of libh2w.
//
// This file is compiled with -ffp-contract=off so that the kernel entries
// and the ACA residual updates round like the reference's scalar code
// (no fused multiply-add); the streaming GEMV and BLAS-1 loops ask for fused
// multiply-adds explicitly with fma().
#include <hip/hip_runtime.h>

#include <cfloat>
#include <climits>
#include <type_traits>

#include "h2w_internal.hpp"
#include "h2w_device.hpp"

namespace h2w {

namespace {

constexpr double kPI = 3.141592653589793238462643383279502884;

// ------------------------------------------------------------------ kernel entry
// A(i,j) of the reference's userkernel::getMatrixEntry for choice 0 (IE) and
// 1 (RBF): 1D/codes/kernel.hpp:108-185, 2D/codes/kernel.hpp:118-228,299-318,
// 3D/codes/kernel.hpp:123-192.  Off-diagonal entries depend on the pair's
// distance; i == j returns the diagonal rule (kp.diag).
// Flop weights (add/mul = 1, sqrt/log/div = 1 each): 3D IE 9, 3D RBF 10.
__device__ __forceinline__ double koff(int dim, int choice, double dx, double dy, double dz) {
    const double a = 0.0001;
    if (dim == 1) {
        double R = fabs(dx);
        if (choice == 0) return log(R);
        return R < a ? R / a : a / R;
    } else if (dim == 2) {
        double R2 = dx * dx + dy * dy;
        if (choice == 0) return (-1.0 / (2 * kPI)) * 0.5 * log(R2);
        double R = sqrt(R2);
        return R < a ? R / a : a / R;
    } else {
        double R2 = dx * dx + dy * dy + dz * dz;
        double R = sqrt(R2);
        if (choice == 0) return 1.0 / (4.0 * kPI * R);
        if (R < a) return (R * log(R) - 1.0) / (a * log(a) - 1.0);
        return (1.0 * log(R)) / log(a);
    }
}

struct PointI {
    double x, y, z;
    int i;
};
__device__ __forceinline__ PointI load_point(const KParams &kp, int i) {
    PointI p;
    p.i = i;
    p.x = kp.px[i];
    p.y = kp.dim > 1 ? kp.py[i] : 0.0;
    p.z = kp.dim > 2 ? kp.pz[i] : 0.0;
    return p;
}
__device__ __forceinline__ double kentry(const KParams &kp, const PointI &p, int j) {
    if (p.i == j) return kp.diag;
    double dx = p.x - kp.px[j];
    double dy = kp.dim > 1 ? p.y - kp.py[j] : 0.0;
    double dz = kp.dim > 2 ? p.z - kp.pz[j] : 0.0;
    return koff(kp.dim, kp.choice, dx, dy, dz);
}
__device__ __forceinline__ double kentry2(const KParams &kp, int i, int j) {
    return kentry(kp, load_point(kp, i), j);
}

// ------------------------------------------------------------------ reductions (wave64)
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}
// argmax of |v| with first-index tie break; (a = |v|, idx, sv = signed v)
struct AMax {
    double a;
    int idx;
    double sv;
};
__device__ __forceinline__ void amax_merge(AMax &x, const AMax &y) {
    if (y.a > x.a || (y.a == x.a && y.idx < x.idx)) x = y;
}
__device__ __forceinline__ AMax wave_amax(AMax v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        AMax w;
        w.a = __shfl_xor(v.a, o, 64);
        w.idx = __shfl_xor(v.idx, o, 64);
        w.sv = __shfl_xor(v.sv, o, 64);
        amax_merge(v, w);
    }
    return v;
}
__device__ __forceinline__ void amax_update(AMax &m, double v, int idx) {
    double a = fabs(v);
    if (a > m.a || (a == m.a && idx < m.idx)) {
        m.a = a;
        m.idx = idx;
        m.sv = v;
    }
}

template <int NT>
struct BlockRed {
    static constexpr int NW = NT / 64;
    double s0[NW], s1[NW];
    double a[NW], sv[NW];
    int idx[NW];
};

// block-wide (sum, sum, argmax); all threads receive the result
template <int NT>
__device__ __forceinline__ void block_reduce(BlockRed<NT> &sh, double &s0, double &s1, AMax &m) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    s0 = wave_sum(s0);
    s1 = wave_sum(s1);
    m = wave_amax(m);
    __syncthreads();
    if (lane == 0) {
        sh.s0[w] = s0;
        sh.s1[w] = s1;
        sh.a[w] = m.a;
        sh.idx[w] = m.idx;
        sh.sv[w] = m.sv;
    }
    __syncthreads();
    s0 = 0.0;
    s1 = 0.0;
    m.a = -1.0;
    m.idx = INT_MAX;
    m.sv = 0.0;
    for (int q = 0; q < BlockRed<NT>::NW; ++q) {
        s0 += sh.s0[q];
        s1 += sh.s1[q];
        AMax o{sh.a[q], sh.idx[q], sh.sv[q]};
        amax_merge(m, o);
    }
}

// ------------------------------------------------------------------ batched ACA
// Restates LowRank::ACA_only_nodes / ACA_only_nodesCUR (2D/codes/aca.hpp:158-446)
// and ACA_only_nodesUV (1D/codes/aca.hpp:40-156), which share the pivot loop:
//   - first row (in order) whose max |entry| exceeds 1e-36 starts the cross,
//   - pivot column = first argmax of |residual row| over unused columns,
//   - u = residual column / pivot, next row = first argmax of |residual column|
//     over unused rows,
//   - stop when |u||v| <= tol * normS or rank = min(m, n), or when |u| or |v|
//     falls below 1e-36 (that step is dropped),
//   - normS^2 += (|u||v|)^2 + 2 sum_{l<=new} |<U_l,u><V_l,v>| (the sum includes
//     the newest term, as the reference's loop does, 2D/codes/aca.hpp:404-409).
// Residual rows/columns subtract the previous terms one by one in rank order
// with separate multiply and subtract, as the reference does.
// One pivot step of every block of a batch is two launches, a row pass and a
// column pass over tiles of all of them: a cross reads the (m + n) k entries of
// its earlier terms at step k, and a level has few blocks near the root and small
// ones near the leaves, so only all blocks together fill the chip at every level.
// (One workgroup per block, with only the blocks of m + n > 8192 spread: the vertex
// level of 64 blocks of m + n up to 8192 took 208 ms at N = 20011, now 13 ms for its
// 272 steps; assemblies 572 -> 180 ms there, 32^3 grid at tol 1e-10 2440 -> 560 ms.)
// Batches of small blocks only keep that form (k_aca_small).
// U and V columns live in a workspace pool shared by the batch: each step reserves
// a column pair with an atomic bump; the column offsets go to the job's table.
// Per-block state lives in WideState; a finished block (converged, exhausted, or out
// of workspace: status 1, re-run by the host) is skipped by every later launch.
constexpr int kChunk = 512;

__device__ __forceinline__ bool aca_reserve(int64_t *tab, int k, int m, int n, int tcap,
                                            unsigned long long *ws_top, int64_t ws_cap, int64_t *sh_off) {
    if (threadIdx.x == 0) {
        int64_t off = -1;
        if (k < tcap) {
            unsigned long long o = atomicAdd(ws_top, (unsigned long long)(m + n));
            if ((int64_t)o + m + n <= ws_cap) off = (int64_t)o;
        }
        *sh_off = off;
        if (off >= 0) {
            tab[2 * k] = off;
            tab[2 * k + 1] = off + m;
        }
    }
    __syncthreads();
    return *sh_off >= 0;
}

// The same cross with one workgroup per block and every step in one launch, for batches of small blocks (the driver's
// rule): their steps of two launches are latency, 17 us of launch, state and first loads a step against 10 us here.
__global__ __launch_bounds__(256) void k_aca_small(const AcaJob *__restrict__ jobs, const int32_t *__restrict__ idx,
                                            double *__restrict__ ws, int64_t ws_cap, unsigned long long *ws_top,
                                            int64_t *__restrict__ tab_all, uint8_t *__restrict__ flags,
                                            int32_t *__restrict__ rank_out, int32_t *__restrict__ status_out,
                                            int32_t *__restrict__ rowpiv, int32_t *__restrict__ colpiv, KParams kp,
                                            double tol, double *__restrict__ hist_all) {
    constexpr int NT = 256;
    const AcaJob jb = jobs[blockIdx.x];
    const int m = jb.m, n = jb.n, tcap = jb.tcap;
    double *hist = hist_all + 2 * jb.piv;  // per accepted step: |u||v|, normS after the step
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    constexpr int NW = NT / 64;
    const int32_t *rows = idx + jb.rows;
    const int32_t *cols = idx + jb.cols;
    int64_t *tab = tab_all + jb.tab;
    uint8_t *ru = flags + jb.wsF;
    uint8_t *cu = ru + m;
    int32_t *rp_out = rowpiv + jb.piv;
    int32_t *cp_out = colpiv + jb.piv;
    __shared__ double coef[kChunk];
    __shared__ int64_t cofs[kChunk];
    __shared__ BlockRed<NT> red;
    __shared__ double dacc[NW];
    __shared__ int64_t sh_off;

    if (m == 0 || n == 0 || tcap == 0) {
        if (tid == 0) {
            rank_out[blockIdx.x] = 0;
            status_out[blockIdx.x] = 0;
        }
        return;
    }
    for (int i = tid; i < m; i += NT) ru[i] = 0;
    for (int s = tid; s < n; s += NT) cu[s] = 0;
    const int mn = min(m, n);
    if (!aca_reserve(tab, 0, m, n, tcap, ws_top, ws_cap, &sh_off)) {
        if (tid == 0) {
            rank_out[blockIdx.x] = 0;
            status_out[blockIdx.x] = 1;
        }
        return;
    }
    double *U0 = ws + sh_off;
    double *V0 = U0 + m;

    // ---- first row with a nonzero entry
    int l = 0, cp = -1;
    double piv = 0.0;
    for (l = 0; l < m; ++l) {
        PointI pr = load_point(kp, rows[l]);
        AMax am{-1.0, INT_MAX, 0.0};
        for (int s = tid; s < n; s += NT) {
            double v = kentry(kp, pr, cols[s]);
            V0[s] = v;
            amax_update(am, v, s);
        }
        double d0 = 0.0, d1 = 0.0;
        block_reduce<NT>(red, d0, d1, am);
        if (am.idx != INT_MAX && am.a > 1e-36) {
            cp = am.idx;
            piv = am.sv;
            break;
        }
    }
    if (l == m) {
        if (tid == 0) {
            rank_out[blockIdx.x] = 0;
            status_out[blockIdx.x] = 0;
        }
        return;
    }
    int rp = l;
    // ---- first column
    double un2 = 0.0, vn2 = 0.0;
    AMax an{-1.0, INT_MAX, 0.0};
    {
        PointI pc = load_point(kp, cols[cp]);
        for (int t = tid; t < m; t += NT) {
            double c = kentry(kp, pc, rows[t]);  // A(rows[t], cols[cp]) (symmetric entry)
            double u = c / piv;
            U0[t] = u;
            un2 += u * u;
            if (t != rp) amax_update(an, c, t);
        }
        for (int s = tid; s < n; s += NT) vn2 += V0[s] * V0[s];
    }
    block_reduce<NT>(red, un2, vn2, an);
    if (tid == 0) {
        rp_out[0] = rp;
        cp_out[0] = cp;
        ru[rp] = 1;
        cu[cp] = 1;
    }
    int rank = 1;
    int status = 0;
    double normS = 0.0;
    double un = sqrt(un2), vn = sqrt(vn2);
    int next_rp = an.idx;
    if (tid == 0) {
        hist[0] = un * vn;
        hist[1] = 0.0;
    }
    __syncthreads();

    while (un * vn > tol * normS && rank < mn) {
        rp = next_rp;
        if (rp == INT_MAX) break;
        if (!aca_reserve(tab, rank, m, n, tcap, ws_top, ws_cap, &sh_off)) {
            status = 1;
            break;
        }
        double *Ur = ws + sh_off;
        double *Vr = Ur + m;
        const int nch = (rank + kChunk - 1) / kChunk;
        // ---- residual row -> V column `rank`
        PointI pr = load_point(kp, rows[rp]);
        AMax am{-1.0, INT_MAX, 0.0};
        vn2 = 0.0;
        for (int ch = 0; ch < nch; ++ch) {
            const int l0 = ch * kChunk, l1 = min(rank, l0 + kChunk);
            for (int q = l0 + tid; q < l1; q += NT) {
                coef[q - l0] = ws[tab[2 * q] + rp];
                cofs[q - l0] = tab[2 * q + 1];
            }
            __syncthreads();
            for (int s = tid; s < n; s += NT) {
                double r = ch == 0 ? kentry(kp, pr, cols[s]) : Vr[s];
                for (int q = l0; q < l1; ++q) r -= coef[q - l0] * ws[cofs[q - l0] + s];
                Vr[s] = r;
                if (ch == nch - 1) {
                    vn2 += r * r;
                    if (!cu[s]) amax_update(am, r, s);
                }
            }
            __syncthreads();
        }
        double dummy = 0.0;
        block_reduce<NT>(red, vn2, dummy, am);
        if (am.idx == INT_MAX) break;
        cp = am.idx;
        piv = am.sv;
        // ---- residual column -> U column `rank`
        PointI pc = load_point(kp, cols[cp]);
        an = AMax{-1.0, INT_MAX, 0.0};
        un2 = 0.0;
        for (int ch = 0; ch < nch; ++ch) {
            const int l0 = ch * kChunk, l1 = min(rank, l0 + kChunk);
            for (int q = l0 + tid; q < l1; q += NT) {
                coef[q - l0] = ws[tab[2 * q + 1] + cp];
                cofs[q - l0] = tab[2 * q];
            }
            __syncthreads();
            for (int t = tid; t < m; t += NT) {
                double c = ch == 0 ? kentry(kp, pc, rows[t]) : Ur[t];
                for (int q = l0; q < l1; ++q) c -= coef[q - l0] * ws[cofs[q - l0] + t];
                if (ch == nch - 1) {
                    double u = c / piv;
                    Ur[t] = u;
                    un2 += u * u;
                    if (t != rp && !ru[t]) amax_update(an, c, t);
                } else {
                    Ur[t] = c;
                }
            }
            __syncthreads();
        }
        block_reduce<NT>(red, un2, dummy, an);
        un = sqrt(un2);
        vn = sqrt(vn2);
        if (un < 1e-36 || vn < 1e-36) break;
        if (tid == 0) {
            rp_out[rank] = rp;
            cp_out[rank] = cp;
            ru[rp] = 1;
            cu[cp] = 1;
        }
        ++rank;
        next_rp = an.idx;
        // ---- normS update: dots of the new term with every term
        double acc = 0.0;
        for (int q = wv; q < rank; q += NW) {
            const double *Uq = ws + tab[2 * q];
            const double *Vq = ws + tab[2 * q + 1];
            double du = 0.0, dv = 0.0;
            for (int t = lane; t < m; t += 64) du += Uq[t] * Ur[t];
            for (int s = lane; s < n; s += 64) dv += Vq[s] * Vr[s];
            du = wave_sum(du);
            dv = wave_sum(dv);
            acc += fabs(du * dv);
        }
        if (lane == 0) dacc[wv] = acc;
        __syncthreads();
        double S = 0.0;
        for (int q = 0; q < NW; ++q) S += dacc[q];
        double uv = un * vn;
        normS = sqrt(normS * normS + uv * uv + 2.0 * S);
        if (tid == 0) {
            hist[2 * (rank - 1)] = uv;
            hist[2 * (rank - 1) + 1] = normS;
        }
        __syncthreads();
    }
    if (tid == 0) {
        rank_out[blockIdx.x] = rank;
        status_out[blockIdx.x] = status;
    }
}


// A tile of the wide passes: 256 threads x 2 consecutive entries (one 16-byte load per earlier term),
// kWideU terms in flight twice over: 64 KB of loads outstanding per workgroup.  Large levels are bound by
// the bytes of the earlier terms (a row pass over 1617 tiles at rank 150 reads 1.0 GB in 195 us, 5.1 TB/s;
// that level of 64 blocks takes 28 ms, with 2048 entries per workgroup and eight loads in flight it took
// 121 ms), small ones by the 10 us that a pass's chain of dependent accesses takes.  (Four waves per SIMD by a register limit spilled: 45 ms; the offsets and
// weights through LDS instead of lane broadcasts, and the sums through the LDS crossbar: 31 ms.)
constexpr int kWideTile = 512;
constexpr int kWideU = 8;

// space for one (U, V) pair; both columns start 16-byte aligned and hold an even number of entries
__device__ __forceinline__ bool wide_take(WideState &st, const AcaJob &jb, int cap, int64_t *tab,
                                          unsigned long long *ws_top, int64_t ws_cap) {
    const int64_t mp = (jb.m + 1) & ~1, np = (jb.n + 1) & ~1;
    if (st.rank >= cap) return false;
    const int64_t off = (int64_t)atomicAdd(ws_top, (unsigned long long)(mp + np));
    if (off + mp + np > ws_cap) return false;
    st.off = off;
    tab[2 * st.rank] = off;
    tab[2 * st.rank + 1] = off + mp;
    return true;
}
__device__ __forceinline__ void wide_reserve(WideState &st, const AcaJob &jb, int cap, int64_t *tab,
                                             unsigned long long *ws_top, int64_t ws_cap) {
    if (!wide_take(st, jb, cap, tab, ws_top, ws_cap)) {
        st.status = 1;
        st.done = 1;
    }
}

// first launch: clear the used-row/column flags, reserve step 0, start the first-row search
__global__ __launch_bounds__(256) void k_wide_init(const AcaJob *__restrict__ jobs, const WideBlk *__restrict__ blk,
                                                   WideState *__restrict__ state, uint8_t *__restrict__ flags,
                                                   int64_t *__restrict__ tab_all, unsigned long long *ws_top,
                                                   int64_t ws_cap) {
    const AcaJob jb = jobs[blockIdx.x];
    const int tot = jb.m + jb.n;
    for (int e = threadIdx.x; e < tot; e += 256) flags[jb.wsF + e] = 0;
    if (threadIdx.x == 0) {
        WideState st{};
        st.next_rp = INT_MAX;
        st.done = (jb.m == 0 || jb.n == 0 || jb.tcap == 0);
        st.kfix = jb.pad;
        if (!st.done) wide_reserve(st, jb, blk[blockIdx.x].cap, tab_all + jb.tab, ws_top, ws_cap);
        state[blockIdx.x] = st;
    }
}

// Values handed from the workgroups of a pass to the one that finishes its block, within one launch:
// agent-scope accesses go past the caches that the XCDs do not share, every wave waits for its stores (s_waitcnt 0)
// before the barrier behind which the arrival is counted, and the last workgroup reads behind its own count.  That
// order is gfx950's; the memory model's form of it (release and acquire at agent scope on the count) also writes back
// whatever the XCD's L2 holds dirty, the residual rows and columns among it: assembly of 20011 3D points 76.6 -> 93.1
// ms, of 40000 2D points 34.3 -> 36.8.
__device__ __forceinline__ void st_agent(double *p, double v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ double ld_agent(const double *p) {
    return __hip_atomic_load(const_cast<double *>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// every tile's partials (sum of squares, first argmax) of one block
__device__ __forceinline__ void wide_reduce(const double *part, int t0, int nt, BlockRed<256> &red, double &ss,
                                            AMax &am) {
    ss = 0.0;
    am = AMax{-1.0, INT_MAX, 0.0};
    for (int w = threadIdx.x; w < nt; w += 256) {
        const double *p = part + 4 * (int64_t)(t0 + w);
        ss += ld_agent(p);
        AMax o{ld_agent(p + 1), (int)ld_agent(p + 2), ld_agent(p + 3)};
        amax_merge(am, o);
    }
    double dummy = 0.0;
    block_reduce<256>(red, ss, dummy, am);
}

// the pivot column of a row pass (first step: a row with a nonzero entry, else the next row)
__device__ __forceinline__ void wide_row_end(WideState &st, const AcaJob &jb, double vn2, const AMax &am) {
    if (st.rank == 0) {
        if (am.idx != INT_MAX && am.a > 1e-36) {
            st.cp = am.idx;
            st.piv = am.sv;
            st.vn2 = vn2;
            st.found = 1;
        } else if (++st.l >= jb.m) {
            st.done = 1;  // every row is zero: rank 0
        } else {
            st.rp = st.l;
        }
    } else if (am.idx == INT_MAX) {
        st.closing = 1;  // no unused column left
    } else {
        st.cp = am.idx;
        st.piv = am.sv;
        st.vn2 = vn2;
    }
}

// Acceptance of a step after its column pass, and what the next step does.
__device__ __forceinline__ void wide_accept(WideState &st, const AcaJob &jb, const WideBlk &wb, double un2,
                                            const AMax &an, uint8_t *flags, int32_t *rowpiv, int32_t *colpiv,
                                            double *hist, int64_t *tab, unsigned long long *ws_top, int64_t ws_cap,
                                            double tol) {
    const double un = sqrt(un2), vn = sqrt(st.vn2);
    uint8_t *ru = flags + jb.wsF, *cu = ru + jb.m;
    const int mn = min(jb.m, jb.n);
    const bool fixed = st.kfix > 1 && st.dots_rank >= 0;  // (dots_rank < 0: the fixed phase was judged)
    if (st.rank > 0 && (un < 1e-36 || vn < 1e-36)) {
        st.done = 1;  // the step is dropped
        if (fixed && st.rank >= 2) st.status = 3;
        return;
    }
    rowpiv[jb.piv + st.rank] = st.rp;
    colpiv[jb.piv + st.rank] = st.cp;
    ru[st.rp] = 1;
    cu[st.cp] = 1;
    st.un = un;
    st.vn = vn;
    st.next_rp = an.idx;
    ++st.rank;
    hist[2 * (st.rank - 1)] = un * vn;
    hist[2 * (st.rank - 1) + 1] = 0.0;
    st.rp = st.next_rp;
    if (fixed) {
        // fixed phase: no normS update and no stopping test until kfix steps are taken (the stopping
        // rule is applied afterwards to all of them at once, from their Gram products)
        st.dots_rank = st.rank;
        if (st.rank >= st.kfix || st.rank >= mn || st.next_rp == INT_MAX) {
            st.done = 1;
            st.status = st.rank >= st.kfix && st.rank < mn && st.next_rp != INT_MAX ? 2 : 3;
        } else {
            wide_reserve(st, jb, wb.cap, tab, ws_top, ws_cap);
        }
    } else if (st.rank == 1) {
        // the first term enters without a normS update (normS stays 0)
        st.normS = 0.0;
        if (!(un * vn > 0.0 && st.rank < mn) || st.next_rp == INT_MAX) st.done = 1;
        else wide_reserve(st, jb, wb.cap, tab, ws_top, ws_cap);
    } else if (st.rank >= mn || st.next_rp == INT_MAX) {
        st.closing = 1;
    } else if (!wide_take(st, jb, wb.cap, tab, ws_top, ws_cap)) {
        st.closing = 2;
    }
}

// One pass of a pivot step over every block, one workgroup per tile of 512 entries.
// COL = 0: residual row rp -> V slot of the current step; COL = 1: residual column cp -> U slot (divided
// by the pivot).  Each workgroup also leaves the sum of squares and the first argmax over unused entries
// of its tile, and its share of the inner products of the newest accepted term with every term (V columns
// in the row pass, U columns in the column pass): the residual and the products read the same earlier
// columns, so reading them once serves both.  The products decide whether the newest term was the last
// one, so the step taken beside them is a step ahead of the stopping rule: the workgroup that ends the
// column pass applies the rule first and drops the step where the rule ends the block.  (Products in a
// pass of their own, and separate launches for the reductions: six launches and two reads per step.)
// A block that cannot take another step whatever the rule says (every row or column used, no workspace)
// is closing: its last passes form the products only.
// The workgroup that arrives last on a block's counter reduces the tiles' partials, in tile order.
template <int COL>
__global__ __launch_bounds__(256) void k_wide_pass(const AcaJob *__restrict__ jobs, const WideBlk *__restrict__ blk,
                                                   const int2 *__restrict__ tiles, const int32_t *__restrict__ idx,
                                                   const double *wsr, double *ws, int64_t *tab_all, uint8_t *flags,
                                                   WideState *state, double *part, double *pdot,
                                                   uint32_t *__restrict__ arrived, int32_t *__restrict__ rowpiv,
                                                   int32_t *__restrict__ colpiv, double *__restrict__ hist_all,
                                                   unsigned long long *ws_top, int64_t ws_cap, KParams kp, double tol) {
    typedef double D2 __attribute__((ext_vector_type(2)));
    const int2 bt = tiles[blockIdx.x];
    WideState st = state[bt.x];
    if (st.done || (COL && st.rank == 0 && !st.found)) return;
    const AcaJob jb = jobs[bt.x];
    const WideBlk wb = blk[bt.x];
    const int len = COL ? jb.m : jb.n;
    const int nt = COL ? wb.nct : wb.nrt;
    const int rank = st.rank;
    const bool resid = !st.closing;
    const bool dots = rank >= 2 && st.dots_rank != rank;  // the newest term's products are due
    int64_t *tab = tab_all + jb.tab;
    __shared__ double wpart[4][kChunk];
    __shared__ BlockRed<256> red;
    __shared__ int last;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int s = bt.y * kWideTile + 2 * threadIdx.x;
    const bool in0 = s < len, in1 = s + 1 < len;
    const int sl = in0 ? s : 0;  // (threads past the end read the column's first entries and use none of them)
    const int pr = COL ? st.cp : st.rp;
    const int32_t *run_i = idx + (COL ? jb.rows : jb.cols);
    const int j0 = run_i[sl], j1 = run_i[in1 ? s + 1 : sl];
    double r0 = 0.0, r1 = 0.0;
    double *out = ws + st.off + (COL ? 0 : (jb.m + 1) & ~1);
    D2 w = {0.0, 0.0};
    if (dots && in0) w = *(const D2 *)(wsr + tab[2 * (rank - 1) + (COL ? 0 : 1)] + s);
    double *pd = pdot + wb.pd + (int64_t)(COL ? wb.nrt + bt.y : bt.y) * wb.cap;
    // The earlier terms' column offsets and coefficients (this tile's residual row or column at their
    // pivots): lane q of a wave holds those of term l0 + q, the next 64 terms' are on their way, and each
    // term's are broadcast from there.  Groups of kWideU columns are loaded two ahead, unconditionally, so
    // that the waits count exactly the loads in flight; past the last term they read its column again
    // (at rank 0 the step's own, unwritten one) and are masked.
    auto term = [&](int l) { return *(const longlong2 *)(tab + 2 * max(0, min(l + lane, rank - 1))); };
    auto weight = [&](const longlong2 &o, int l) {
        return resid && l + lane < rank ? wsr[(COL ? o.y : o.x) + pr] : 0.0;
    };
    auto lane_of = [&](int64_t v, int l) -> int64_t {
        const int lo = __builtin_amdgcn_readlane((int)v, l), hi = __builtin_amdgcn_readlane((int)(v >> 32), l);
        return ((int64_t)hi << 32) | (uint32_t)lo;
    };
    D2 A[kWideU], B[kWideU];
    auto load = [&](D2(&v)[kWideU], const longlong2 &o, int q) {
#pragma unroll
        for (int u = 0; u < kWideU; ++u) v[u] = *(const D2 *)(wsr + lane_of(COL ? o.x : o.y, q + u) + sl);
    };
    auto use = [&](D2(&v)[kWideU], double cf, int l0, int q) {
        if (l0 + q + kWideU > rank) {
#pragma unroll
            for (int u = 0; u < kWideU; ++u)
                if (l0 + q + u >= rank) v[u] = (D2)0.0;
        }
#pragma unroll
        for (int u = 0; u < kWideU; ++u) {
            const double c = __longlong_as_double(lane_of(__double_as_longlong(cf), q + u));
            r0 -= c * v[u].x;
            r1 -= c * v[u].y;
        }
        if (dots) {
            typedef double D8 __attribute__((ext_vector_type(kWideU)));
            D8 p;
#pragma unroll
            for (int u = 0; u < kWideU; ++u) p[u] = fma(v[u].y, w.y, v[u].x * w.x);
            // sums over the wave: three exchanges that halve the values per lane, then three plain ones
            int ui = 0;
#pragma unroll
            for (int k = kWideU, o = 1; k > 1; k >>= 1, o <<= 1) {
                const bool hi = lane & o;
#pragma unroll
                for (int i = 0; i < k / 2; ++i) {
                    const double snd = hi ? p[i] : p[i + k / 2];
                    const double keep = hi ? p[i + k / 2] : p[i];
                    p[i] = keep + (o == 1 ? fold_lane<1>(snd) : o == 2 ? fold_lane<2>(snd) : fold_lane<4>(snd));
                }
                ui += hi ? k / 2 : 0;
            }
            const double t = sum_halves(p[0] + fold_lane<8>(p[0]));
            if (lane < kWideU) wpart[wv][((l0 + q) & (kChunk - 1)) + ui] = t;
        }
    };
    longlong2 o0 = term(0), o1 = term(64);
    double cf0 = weight(o0, 0);
    load(A, o0, 0);
    load(B, o0, kWideU);
    if (resid) {
        // (the entries' own loads and logarithms pass behind the first groups; a closing block has no row
        // or column pr)
        const PointI p = load_point(kp, (idx + (COL ? jb.cols : jb.rows))[pr]);
        r0 = kentry(kp, p, j0);
        r1 = kentry(kp, p, j1);
    }
    for (int l0 = 0; l0 < rank; l0 += 64) {
        const double cf1 = weight(o1, l0 + 64);
        const longlong2 o2 = term(l0 + 128);
        for (int q = 0; q < 64 && l0 + q < rank; q += 2 * kWideU) {
            const bool nx = q + 2 * kWideU == 64;
            const longlong2 on{nx ? o1.x : o0.x, nx ? o1.y : o0.y};
            const int qn = (q + 2 * kWideU) & 63;
            use(A, cf0, l0, q);
            load(A, on, qn);
            use(B, cf0, l0, q + kWideU);
            load(B, on, qn + kWideU);
        }
        o0 = o1;
        o1 = o2;
        cf0 = cf1;
        if (dots && (l0 + 64 >= rank || ((l0 + 64) & (kChunk - 1)) == 0)) {
            // the waves' sums of up to kChunk terms
            const int f0 = l0 / kChunk * kChunk, nq = min(rank - f0, kChunk);
            __syncthreads();
            for (int q = threadIdx.x; q < nq; q += 256)
                st_agent(pd + f0 + q, (wpart[0][q] + wpart[1][q]) + (wpart[2][q] + wpart[3][q]));
            __syncthreads();
        }
    }
    double ss = 0.0, dummy = 0.0;
    AMax am{-1.0, INT_MAX, 0.0};
    if (resid) {
        const uint8_t *used = flags + jb.wsF + (COL ? 0 : jb.m);
        double v0 = in0 ? r0 : 0.0, v1 = in1 ? r1 : 0.0;
        if (in0 && !used[s] && !(COL && s == st.rp)) amax_update(am, v0, s);
        if (in1 && !used[s + 1] && !(COL && s + 1 == st.rp)) amax_update(am, v1, s + 1);
        if (COL) {
            v0 = v0 / st.piv;
            v1 = in1 ? v1 / st.piv : 0.0;
        }
        if (in0) {
            ss = v0 * v0 + v1 * v1;
            *(D2 *)(out + s) = D2{v0, v1};  // (the padding entry of an odd column is zero)
        }
    }
    block_reduce<256>(red, ss, dummy, am);
    if (threadIdx.x == 0) {
        double *p = part + 4 * (int64_t)((COL ? wb.ct0 : wb.rt0) + bt.y);
        st_agent(p, ss);
        st_agent(p + 1, am.a);
        st_agent(p + 2, (double)am.idx);
        st_agent(p + 3, am.sv);
    }
    // every partial of this workgroup is at the coherence point before its arrival is counted
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (threadIdx.x == 0) last = atomicAdd(arrived + bt.x, 1u) == (uint32_t)(nt - 1);
    __syncthreads();
    if (!last) return;

    // ---- the block's last workgroup of this pass
    wide_reduce(part, COL ? wb.ct0 : wb.rt0, nt, red, ss, am);
    if (!COL) {
        if (threadIdx.x != 0) return;
        arrived[bt.x] = 0;
        if (resid) wide_row_end(st, jb, ss, am);
        if (st.closing && !dots) st.done = 1;  // nothing left to form
        state[bt.x] = st;
        return;
    }
    double *hist = hist_all + 2 * jb.piv;
    const int mn = min(jb.m, jb.n);
    if (dots) {
        double S = 0.0;
        for (int q = threadIdx.x; q < rank; q += 256) {
            double du = 0.0, dv = 0.0;
            const double *pv = pdot + wb.pd + q, *pu = pv + (int64_t)wb.nrt * wb.cap;
#pragma unroll 8
            for (int t = 0; t < wb.nrt; ++t) dv += ld_agent(pv + (int64_t)t * wb.cap);
#pragma unroll 8
            for (int t = 0; t < wb.nct; ++t) du += ld_agent(pu + (int64_t)t * wb.cap);
            S += fabs(du * dv);
        }
        AMax none{-1.0, INT_MAX, 0.0};
        block_reduce<256>(red, S, dummy, none);
        const double uv = st.un * st.vn;
        st.normS = sqrt(st.normS * st.normS + uv * uv + 2.0 * S);
        st.dots_rank = rank;
        const bool more = uv > tol * st.normS && rank < mn;
        if (threadIdx.x == 0) hist[2 * (rank - 1) + 1] = st.normS;
        if (!more || st.closing) {
            st.done = 1;
            if (more && st.closing == 2) st.status = 1;  // out of workspace before the rule was met
        }
    }
    if (threadIdx.x != 0) return;
    arrived[bt.x] = 0;
    if (!st.done)
        wide_accept(st, jb, wb, ss, am, flags, rowpiv, colpiv, hist, tab, ws_top, ws_cap, tol);
    state[bt.x] = st;
}

__global__ void k_wide_finish(const WideState *__restrict__ state, int nb, int32_t *__restrict__ rank_out,
                              int32_t *__restrict__ status_out, int32_t *__restrict__ ndone) {
    int done = 0;
    for (int b = threadIdx.x; b < nb; b += blockDim.x) {
        rank_out[b] = state[b].rank;
        status_out[b] = state[b].status;
        done += state[b].done;
    }
    done = (int)wave_sum((double)done);
    if (threadIdx.x == 0) *ndone = done;
}

// Gram products of the terms of a parked block: one workgroup per 64 x 64 tile of term pairs
// (q in tile qi, k in tile ki, qi <= ki); each thread accumulates 4 x 4 dot products of U
// columns, then of V columns, over 32-entry slabs staged in LDS.  prod = |<U_q,U_k>||<V_q,V_k>|
// for q <= k (packed lower-triangular by k).
constexpr int kGramT = 64, kGramS = 32;
__device__ __forceinline__ void gram_tile(const double *ws, const int64_t *tab, int part, int len, int q0, int nq,
                                          int k0, int nk, double (&acc)[4][4]) {
    __shared__ double sq[kGramS][kGramT + 1], sk[kGramS][kGramT + 1];
    const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;  // q = q0 + 4 tx + a, k = k0 + 4 ty + b
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b) acc[a][b] = 0.0;
    for (int t0 = 0; t0 < len; t0 += kGramS) {
        __syncthreads();
        for (int e = threadIdx.x; e < kGramS * kGramT; e += 256) {
            const int c = e / kGramS, t = e % kGramS;  // column c of the tile, entry t of the slab
            const bool tin = t0 + t < len;
            sq[t][c] = (c < nq && tin) ? ws[tab[2 * (q0 + c) + part] + t0 + t] : 0.0;
            sk[t][c] = (c < nk && tin) ? ws[tab[2 * (k0 + c) + part] + t0 + t] : 0.0;
        }
        __syncthreads();
#pragma unroll 4
        for (int t = 0; t < kGramS; ++t) {
            double x[4], y[4];
#pragma unroll
            for (int a = 0; a < 4; ++a) x[a] = sq[t][4 * tx + a];
#pragma unroll
            for (int b = 0; b < 4; ++b) y[b] = sk[t][4 * ty + b];
#pragma unroll
            for (int a = 0; a < 4; ++a)
#pragma unroll
                for (int b = 0; b < 4; ++b) acc[a][b] = fma(x[a], y[b], acc[a][b]);
        }
    }
}
__global__ __launch_bounds__(256) void k_wide_gram(const GramJob *__restrict__ gj, const AcaJob *__restrict__ jobs,
                                                   const WideState *__restrict__ state, const double *__restrict__ ws,
                                                   const int64_t *__restrict__ tab_all, double *__restrict__ prod) {
    const GramJob g = gj[blockIdx.x];
    const AcaJob jb = jobs[g.blk];
    const int K = state[g.blk].rank;
    const int64_t *tab = tab_all + jb.tab;
    const int q0 = g.qi * kGramT, k0 = g.ki * kGramT;
    const int nq = min(kGramT, K - q0), nk = min(kGramT, K - k0);
    double gu[4][4], gv[4][4];
    gram_tile(ws, tab, 0, jb.m, q0, nq, k0, nk, gu);
    gram_tile(ws, tab, 1, jb.n, q0, nq, k0, nk, gv);
    const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const int q = q0 + 4 * tx + a, k = k0 + 4 * ty + b;
            if (q < K && k < K && q <= k) prod[g.off + (int64_t)k * (k + 1) / 2 + q] = fabs(gu[a][b]) * fabs(gv[a][b]);
        }
}

// decisions of the host on the judged blocks (one thread per block)
__global__ void k_wide_judge(const AcaJob *__restrict__ jobs, const WideBlk *__restrict__ blk, int nb,
                             WideState *__restrict__ state,
                             const int32_t *__restrict__ final_rank, const double *__restrict__ normS_in,
                             int64_t *__restrict__ tab_all, unsigned long long *ws_top, int64_t ws_cap) {
    for (int b = blockIdx.x * blockDim.x + threadIdx.x; b < nb; b += gridDim.x * blockDim.x) {
        const int fr = final_rank[b];
        if (fr == -2) continue;
        WideState st = state[b];
        st.dots_rank = -1;  // (the fixed phase is over)
        if (fr >= 0) {
            st.rank = fr;
            st.done = 1;
            st.status = 0;
        } else {
            // the stopping rule did not hold within the fixed phase: continue adaptively
            st.normS = normS_in[b];
            st.dots_rank = st.rank;
            st.done = 0;
            st.status = 0;
            st.kfix = 0;
            st.rp = st.next_rp;
            wide_reserve(st, jobs[b], blk[b].cap, tab_all + jobs[b].tab, ws_top, ws_cap);
        }
        state[b] = st;
    }
}

// sampled entries of finished blocks against their cross approximation
__global__ __launch_bounds__(64) void k_aca_sample(const AcaJob *__restrict__ jobs, const int32_t *__restrict__ rank,
                                                   const int32_t *__restrict__ idx, const double *__restrict__ ws,
                                                   const int64_t *__restrict__ tab_all, KParams kp, int ns,
                                                   double *__restrict__ err2, double *__restrict__ ref2) {
    const AcaJob jb = jobs[blockIdx.x];
    const int r = rank[blockIdx.x];
    const int64_t *tab = tab_all + jb.tab;
    double e2 = 0.0, a2 = 0.0;
    if (jb.m > 0 && jb.n > 0)
        for (int q = threadIdx.x; q < ns; q += 64) {
            // (i, j) from a 64-bit mix of (block, sample)
            uint64_t h = ((uint64_t)blockIdx.x << 32) ^ (uint64_t)q ^ 0x9E3779B97F4A7C15ull;
            h ^= h >> 33;
            h *= 0xff51afd7ed558ccdull;
            h ^= h >> 33;
            h *= 0xc4ceb9fe1a85ec53ull;
            h ^= h >> 33;
            const int i = (int)(h % (uint64_t)jb.m), j = (int)((h >> 32) % (uint64_t)jb.n);
            const double a = kentry2(kp, idx[jb.rows + i], idx[jb.cols + j]);
            double v = 0.0;
            for (int k = 0; k < r; ++k) v = fma(ws[tab[2 * k] + i], ws[tab[2 * k + 1] + j], v);
            e2 += (a - v) * (a - v);
            a2 += a * a;
        }
    e2 = wave_sum(e2);
    a2 = wave_sum(a2);
    if (threadIdx.x == 0) {
        err2[blockIdx.x] = e2;
        ref2[blockIdx.x] = a2;
    }
}

// L (unit lower) and R (upper) of the cross: L(i,j) = U_j[rb_i], R(j,i) = V_j[cb_i]
// (2D/codes/aca.hpp:419-445)
__global__ void k_lr_extract(const LrJob *__restrict__ jobs, const double *__restrict__ ws,
                             const int64_t *__restrict__ tab_all, const int32_t *__restrict__ rowpiv,
                             const int32_t *__restrict__ colpiv, double *__restrict__ out) {
    const LrJob jb = jobs[blockIdx.x];
    const int r = jb.rank;
    double *L = out + jb.out;
    double *R = L + (int64_t)r * r;
    const int64_t *tab = tab_all + jb.tab;
    for (int e = threadIdx.x; e < r * r; e += blockDim.x) {
        int i = e % r, j = e / r;  // row i, column j
        double lv = 0.0, rv = 0.0;
        if (i == j) lv = 1.0;
        else if (j < i) lv = ws[tab[2 * j] + rowpiv[jb.piv + i]];
        if (i <= j) rv = ws[tab[2 * i + 1] + colpiv[jb.piv + j]];
        L[e] = lv;
        R[e] = rv;
    }
}

// L and R again from a skeleton's pivots, for an operator that no longer holds them: elimination of the pivot block in
// pivot order.  Every entry takes the products of the earlier terms in rank order, multiplied and subtracted separately,
// as the cross's residual rows and columns do, so the factors are the cross's to the last bit.
// Eight pivots at a time: their columns one after another, their rows by a thread per column, then every other entry
// with all eight products from one load.  64 skeletons of rank up to 465: 4.1 ms (one pivot at a time, bound by those
// loads, 15.1 ms).
constexpr int kLrB = 8;
__global__ __launch_bounds__(1024) void k_lr_form(const LrFormJob *__restrict__ jobs, const int32_t *__restrict__ idx,
                                                  double *__restrict__ out, KParams kp) {
    const LrFormJob jb = jobs[blockIdx.x];
    const int k = jb.k;
    const int64_t ld = k;
    double *L = out + jb.out;
    double *R = L + ld * k;
    for (int e = threadIdx.x; e < k * k; e += 1024) {
        const int i = e % k, j = e / k;
        R[e] = kentry2(kp, idx[jb.ir + i], idx[jb.ic + j]);
        L[e] = i == j ? 1.0 : 0.0;
    }
    const int ti = threadIdx.x & 63, tj = threadIdx.x >> 6;
    for (int q0 = 0; q0 < k; q0 += kLrB) {
        const int q1 = min(q0 + kLrB, k);
        for (int q = q0; q < q1; ++q) {
            __syncthreads();
            const double piv = R[q * ld + q];
            for (int i = q + 1 + threadIdx.x; i < k; i += 1024) L[q * ld + i] = R[q * ld + i] / piv;
            __syncthreads();
            const int j = q + 1 + (tj & 7);  // (at most seven columns; two waves each)
            if (j < q1) {
                const double v = R[j * ld + q];
                for (int i = q + 1 + ti + 64 * (tj >> 3); i < k; i += 128) R[j * ld + i] -= L[q * ld + i] * v;
            }
        }
        if (q1 == k) break;
        __syncthreads();
        for (int j = q1 + threadIdx.x; j < k; j += 1024) {
            double r[kLrB];
#pragma unroll
            for (int u = 0; u < kLrB; ++u) {
                r[u] = R[j * ld + q0 + u];
#pragma unroll
                for (int v = 0; v < u; ++v) r[u] -= L[(q0 + v) * ld + q0 + u] * r[v];
                R[j * ld + q0 + u] = r[u];
            }
        }
        __syncthreads();
        for (int i = q1 + ti; i < k; i += 64) {
            double l[kLrB];
#pragma unroll
            for (int u = 0; u < kLrB; ++u) l[u] = L[(q0 + u) * ld + i];
#pragma unroll 2
            for (int j = q1 + tj; j < k; j += 16) {
                const double *r = R + j * ld + q0;
                double x = R[j * ld + i];
#pragma unroll
                for (int u = 0; u < kLrB; ++u) x -= l[u] * r[u];
                R[j * ld + i] = x;
            }
        }
    }
    __syncthreads();
    for (int e = threadIdx.x; e < k * k; e += 1024)
        if (e % k > e / k) R[e] = 0.0;
}

__global__ void k_pack_pivots(const LrJob *__restrict__ jobs, const int32_t *__restrict__ rowpiv,
                              const int32_t *__restrict__ colpiv, const double *__restrict__ hist,
                              int32_t *__restrict__ prow, int32_t *__restrict__ pcol, double *__restrict__ phist) {
    const LrJob jb = jobs[blockIdx.x];
    for (int k = threadIdx.x; k < jb.rank; k += blockDim.x) {
        prow[jb.pk + k] = rowpiv[jb.piv + k];
        pcol[jb.pk + k] = colpiv[jb.piv + k];
        phist[2 * ((int64_t)jb.pk + k)] = hist[2 * (jb.piv + k)];
        phist[2 * ((int64_t)jb.pk + k) + 1] = hist[2 * (jb.piv + k) + 1];
    }
}

__global__ void k_slot_points(const int32_t *__restrict__ pid, int64_t n, const double *__restrict__ px,
                              const double *__restrict__ py, const double *__restrict__ pz, double *__restrict__ xd,
                              double *__restrict__ yd, double *__restrict__ zd, float *__restrict__ x,
                              float *__restrict__ y, float *__restrict__ z, float *__restrict__ xl,
                              float *__restrict__ yl, float *__restrict__ zl) {
    const int64_t v = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (v >= n) return;
    const int32_t i = pid[v];
    const double a = i < 0 ? 0.0 : px[i], b = i < 0 ? 0.0 : py[i], c = i < 0 ? 0.0 : pz[i];
    xd[v] = a;
    yd[v] = b;
    zd[v] = c;
    x[v] = (float)a;
    y[v] = (float)b;
    z[v] = (float)c;
    xl[v] = (float)(a - (double)(float)a);
    yl[v] = (float)(b - (double)(float)b);
    zl[v] = (float)(c - (double)(float)c);
}

// A = K(rows, cols), column-major (getMatrix, 3D/codes/kernel.hpp:58-71)
__global__ void k_eval(const EvalJob *__restrict__ jobs, const int32_t *__restrict__ idx, double *__restrict__ A,
                       KParams kp) {
    const EvalJob jb = jobs[blockIdx.x];
    const int64_t tot = (int64_t)jb.m * jb.n;
    const int32_t *rows = idx + jb.rows;
    const int32_t *cols = idx + jb.cols;
    for (int64_t e = threadIdx.x; e < tot; e += blockDim.x) {
        int i = (int)(e % jb.m), j = (int)(e / jb.m);
        A[jb.a + (int64_t)j * jb.lda + i] = kentry2(kp, rows[i], cols[j]);
    }
}

// E = K(S, Ic) R^{-1} L^{-1} (m x r) and its transpose.  For the far field this
// is L2P (3D/codes/HODLR3Dtree.hpp:1926-1927); for the vertex-sharing field it
// is the transpose of M2M_ver = (L R)^{-T} K(Ic, S) (:2110-2133), the same
// matrix since the kernel is symmetric.  One thread per row of S.
// kSolveB columns are solved together: each earlier column's entry is loaded once
// for all of them, their sums are independent chains, and the triangle's entries
// (the same for every row) come by scalar loads of consecutive elements.
// (One column at a time, a load of E and a dependent subtraction per multiply:
// 13.1 -> 1.8 ms for the transfers at 3D N = 20011, 42.7 -> 4.9 ms at 32^3, tol 1e-10.)
constexpr int kSolveB = 8;
__global__ __launch_bounds__(64) void k_xfer(const XferJob *__restrict__ jobs, const int32_t *__restrict__ idx,
                                             const double *__restrict__ lr, double *__restrict__ A, KParams kp) {
    const XferJob jb = jobs[blockIdx.x];
    const int m = jb.m, r = jb.r;
    const int64_t ldr = jb.ldr;
    const int64_t lde = jb.lde, ldet = jb.ldet;
    const double *L = lr + jb.lr;
    const double *R = L + ldr * ldr;
    const int32_t *S = idx + jb.s;
    const int32_t *Ic = idx + jb.ic;
    for (int t = threadIdx.x; t < m; t += blockDim.x) {
        double *E = A + jb.e + t;
        double *ET = A + jb.et + t * ldet;
        const PointI p = load_point(kp, S[t]);
        double s[kSolveB], e[kSolveB];
        // X R = K(S_t, Ic)
        for (int k0 = 0; k0 < r; k0 += kSolveB) {
#pragma unroll
            for (int u = 0; u < kSolveB; ++u) s[u] = kentry(kp, p, Ic[min(k0 + u, r - 1)]);
            for (int q0 = 0; q0 < k0; q0 += kSolveB) {
#pragma unroll
                for (int v = 0; v < kSolveB; ++v) e[v] = E[(q0 + v) * lde];
#pragma unroll
                for (int u = 0; u < kSolveB; ++u) {
                    const double *Rk = R + min(k0 + u, r - 1) * ldr + q0;
#pragma unroll
                    for (int v = 0; v < kSolveB; ++v) s[u] = fma(-e[v], Rk[v], s[u]);
                }
            }
#pragma unroll
            for (int u = 0; u < kSolveB; ++u) {
                const double *Rk = R + min(k0 + u, r - 1) * ldr + k0;
                if (k0 + u < r) {
#pragma unroll
                    for (int v = 0; v < kSolveB; ++v)
                        if (v < u) s[u] = fma(-s[v], Rk[v], s[u]);
                    s[u] = s[u] / Rk[u];
                    E[(k0 + u) * lde] = s[u];
                }
            }
        }
        // Y L = X, from the last columns
        for (int k0 = (r - 1) / kSolveB * kSolveB; k0 >= 0; k0 -= kSolveB) {
#pragma unroll
            for (int u = 0; u < kSolveB; ++u) s[u] = E[min(k0 + u, r - 1) * lde];
            int q0 = k0 + kSolveB;
            for (; q0 + kSolveB <= r; q0 += kSolveB) {
#pragma unroll
                for (int v = 0; v < kSolveB; ++v) e[v] = E[(q0 + v) * lde];
#pragma unroll
                for (int u = 0; u < kSolveB; ++u) {
                    const double *Lk = L + (k0 + u) * ldr + q0;
#pragma unroll
                    for (int v = 0; v < kSolveB; ++v) s[u] = fma(-e[v], Lk[v], s[u]);
                }
            }
            for (; q0 < r; ++q0) {
                const double eq = E[q0 * lde];
#pragma unroll
                for (int u = 0; u < kSolveB; ++u) s[u] = fma(-eq, L[(k0 + u) * ldr + q0], s[u]);
            }
#pragma unroll
            for (int u = kSolveB - 1; u >= 0; --u) {
                if (k0 + u < r) {
                    const double *Lk = L + (k0 + u) * ldr + k0;
#pragma unroll
                    for (int v = 0; v < kSolveB; ++v)
                        if (v > u && k0 + v < r) s[u] = fma(-s[v], Lk[v], s[u]);
                    s[u] = s[u] / Lk[u];
                    E[(k0 + u) * lde] = s[u];
                    ET[k0 + u] = s[u];
                }
            }
        }
    }
}

// A = R^{-1} L^{-1} K(Ir, V) (r x n), one thread per column: the semi-nested
// vertex block's row factor with the two triangular solves of the reference's
// apply (3D/codes/HODLR3Dtree.hpp:2341-2344) folded in at assembly.  kSolveB rows
// are solved together, as in k_xfer (4.9 -> 0.9 ms at 3D N = 20000, tol 1e-8).
__global__ __launch_bounds__(64) void k_cur(const CurJob *__restrict__ jobs, const int32_t *__restrict__ idx,
                                            const double *__restrict__ lr, double *__restrict__ A, KParams kp) {
    const CurJob jb = jobs[blockIdx.x];
    const int r = jb.r, n = jb.n;
    const double *L = lr + jb.lr;
    const double *R = L + (int64_t)r * r;
    const int32_t *Ir = idx + jb.ir;
    const int32_t *Vv = idx + jb.v;
    for (int t = threadIdx.x; t < n; t += blockDim.x) {
        double *a = A + jb.a + (int64_t)t * jb.lda;
        const PointI p = load_point(kp, Vv[t]);
        double s[kSolveB];
        for (int k0 = 0; k0 < r; k0 += kSolveB) {
#pragma unroll
            for (int u = 0; u < kSolveB; ++u) s[u] = kentry(kp, p, Ir[min(k0 + u, r - 1)]);
            for (int q = 0; q < k0; ++q) {
                const double aq = a[q];
                const double *Lq = L + (int64_t)q * r + k0;
#pragma unroll
                for (int u = 0; u < kSolveB; ++u) s[u] = fma(-aq, Lq[min(u, r - 1 - k0)], s[u]);
            }
#pragma unroll
            for (int u = 0; u < kSolveB; ++u)
                if (k0 + u < r) {
#pragma unroll
                    for (int v = 0; v < kSolveB; ++v)
                        if (v < u) s[u] = fma(-s[v], L[(int64_t)(k0 + v) * r + k0 + u], s[u]);
                    s[u] = s[u] / L[(int64_t)(k0 + u) * r + k0 + u];
                    a[k0 + u] = s[u];
                }
        }
        for (int k0 = (r - 1) / kSolveB * kSolveB; k0 >= 0; k0 -= kSolveB) {
#pragma unroll
            for (int u = 0; u < kSolveB; ++u) s[u] = a[min(k0 + u, r - 1)];
            for (int q = k0 + kSolveB; q < r; ++q) {
                const double aq = a[q];
                const double *Rq = R + (int64_t)q * r + k0;
#pragma unroll
                for (int u = 0; u < kSolveB; ++u) s[u] = fma(-aq, Rq[u], s[u]);
            }
#pragma unroll
            for (int u = kSolveB - 1; u >= 0; --u)
                if (k0 + u < r) {
#pragma unroll
                    for (int v = 0; v < kSolveB; ++v)
                        if (v > u && k0 + v < r) s[u] = fma(-s[v], R[(int64_t)(k0 + v) * r + k0 + u], s[u]);
                    s[u] = s[u] / R[(int64_t)(k0 + u) * r + k0 + u];
                    a[k0 + u] = s[u];
                }
        }
    }
}

// Products of consecutive transfers (a box's skeleton to a descendant's, several levels down), once per
// assembly: one workgroup per block of at most a few hundred rows and columns.  Transfers have entries well
// above one whose products cancel, so the products are carried as unevaluated pairs (lo: the low parts of the
// blocks from offset lo0 on) and rounded once: with plain products the operator of a 1D system with
// N = 250000 was four times further from the dense one (1.2e-12 for 3.3e-13).
// most receives the largest entry (infinity for one that is not finite), by which the caller decides whether the
// products are used.
__global__ __launch_bounds__(256) void k_compose(const ComposeJob *__restrict__ jobs, double *A, double *lo,
                                                 int64_t lo0, unsigned long long *most) {
    const ComposeJob jb = jobs[blockIdx.x];
    double mc = 0.0;
    for (int e = threadIdx.x; e < jb.m * jb.n; e += 256) {
        const int i = e % jb.m, j = e / jb.m;
        double v = jb.k == 0 ? A[jb.a + (int64_t)j * jb.lda + i] : 0.0, r = 0.0;
        for (int q = 0; q < jb.k; ++q) {
            const int64_t o = jb.a + (int64_t)q * jb.lda + i;
            const double x = A[o], y = A[jb.b + (int64_t)j * jb.ldb + q];
            const double p = x * y, pe = fma(x, y, -p);
            const double t = v + p, z = t - v;
            r += ((v - (t - z)) + (p - z)) + (pe + lo[o - lo0] * y);
            v = t;
        }
        const double h = v + r;
        A[jb.d + (int64_t)j * jb.ldd + i] = h;
        lo[jb.d - lo0 + (int64_t)j * jb.ldd + i] = (v - h) + r;
        if (jb.dt >= 0) A[jb.dt + (int64_t)i * jb.ldt + j] = h;
        mc = fabs(h) <= DBL_MAX ? fmax(mc, fabs(h)) : HUGE_VAL;
    }
    // the largest entry (the bits of doubles that are not negative are in their order)
    for (int o = 32; o > 0; o >>= 1) mc = fmax(mc, __shfl_xor(mc, o, 64));
    if ((threadIdx.x & 63) == 0) atomicMax(most, (unsigned long long)__double_as_longlong(mc));
}

// ------------------------------------------------------------------ batched skinny GEMV
// One workgroup (4 waves) per item of <= 128 rows.  Each lane loads VEC
// consecutive rows of a column with one 16-byte load (VEC = 2 for FP64, 4 for
// FP32); ceil(rows / VEC) lanes, rounded up to a power of two, cover a column,
// so a wave load reads 64/lpc whole columns.  The waves split the columns of
// every term.  Partial sums are combined across the wave's column groups with
// cross-lane adds, then across the waves in LDS, and added to y exclusively
// or atomically.  Blocks are column-major with leading dimensions padded to a
// multiple of 4, so every VEC group is aligned and stays inside the column.
// ROLE 1 (the fused M2L + near-field launch) also forms the transposed products
// of the symmetric terms; 0 (transfer passes) and 2 (semi-nested column factors)
// only name the instance so that profiles separate the launches.  UNR is the
// number of columns each lane loads per iteration.  Bit 1 of an item's flags
// selects the operator pool A1 (the inner operator of the refinement) instead
// of A0.
// The column loop of an item walks (term, column) iterations with a wave-uniform
// cursor; each iteration is UNR column loads per lane.  Two iterations are in flight:
// the loads of the next are issued before the current one is multiplied.  Every load
// is unconditional (lanes out of range address past the buffer's end), so the
// compiler's waits count exactly the outstanding operations.
// WPI waves share an item: 4, whose sums meet in LDS, or 1, four items per workgroup.
template <typename T, int VEC, int ROLE, int UNR, int WPI>
__global__ __launch_bounds__(256) void k_bgemv(const GItem *__restrict__ items, int nitems,
                                               const GTerm *__restrict__ terms, const T *__restrict__ A0,
                                               const T *__restrict__ A1, T *vec) {
    typedef T V __attribute__((ext_vector_type(VEC)));
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int item = WPI == 4 ? blockIdx.x : 4 * blockIdx.x + wave;
    if (WPI == 1 && item >= nitems) return;
    const int wv = WPI == 4 ? wave : 0;
    const GItem it = items[item];
    const CGTerm *const tms = (const CGTerm *)terms;
    const T *__restrict__ A = (it.flags & 2) ? A1 : A0;
    const int rows = it.rows;
    // (the fused launch gives a column at least UNR lanes, so that its transposed sums
    // end on UNR distinct lanes; the extra lanes of a short tile are inactive)
    int lpc = ROLE == 1 ? UNR : 1;
    while (lpc * VEC < rows) lpc <<= 1;
    const int cpw = 64 / lpc;
    const int q = lane / lpc, r0 = (lane % lpc) * VEC;
    const bool act = r0 < rows;
    __shared__ T part[WPI == 4 ? 4 : 1][kRowTile];
    V acc = (V)0;
    // this tile's own input rows: the x of the transposed products of symmetric terms
    T xb[VEC];
#pragma unroll
    for (int v = 0; v < VEC; ++v) xb[v] = (ROLE == 1 && act && r0 + v < rows) ? vec[it.xb + r0 + v] : T(0);
    const int64_t lda = it.lda;
    // a wave takes chunks of cpw UNR consecutive columns, lane group q the UNR columns
    // c0 + q UNR + u (one vector load of their x); the four waves take every fourth chunk
    const int chunk = cpw * UNR;
    const uint32_t roff = (uint32_t)((it.row0 + (act ? r0 : 0)) * sizeof(T));  // this lane's rows in a column
    struct Iter {
        V av[UNR];
        T xv[UNR];
        int cols, cb;
        int64_t t;
    };
    int tt = it.t0, c0 = wv * chunk;  // next iteration: term, first column of the wave's chunk
    auto settle = [&]() {
        while (tt < it.t1 && c0 >= tms[tt].cols) {
            ++tt;
            c0 = wv * chunk;
        }
    };
    // loads of the next iteration (past the last one: a term's resources with no valid lane)
    auto load = [&](Iter &B) -> bool {
        const bool has = tt < it.t1;
        const GTerm tm = term_at(tms, has ? tt : it.t1 - 1);
        B.cols = has ? tm.cols : 0;
        B.cb = c0 + q * UNR;
        B.t = tm.t;
        const __amdgpu_buffer_rsrc_t ra = buf_rsrc(A + tm.a, (uint32_t)((int64_t)tm.cols * lda * sizeof(T)));
        const __amdgpu_buffer_rsrc_t rx = buf_rsrc(vec + tm.x, (uint32_t)(B.cols * sizeof(T)));
#pragma unroll
        for (int u = 0; u < UNR; ++u) {
            const int cc = B.cb + u;
            const bool ok = act && cc < B.cols;
            B.av[u] = buf_ld16_nt<V>(ra, ok ? (uint32_t)(cc * lda * sizeof(T)) + roff : kOutOfRange);
        }
        // (columns past the term's end within the group read neighbouring values or zeros:
        // their A entries are zero and they are dropped below)
        buf_ld_n<T, UNR>(B.xv, rx, act && B.cb < B.cols ? (uint32_t)(B.cb * sizeof(T)) : kOutOfRange);
        if (has) {
            c0 += WPI * chunk;
            settle();
        }
        return has;
    };
    auto compute = [&](const Iter &B) {
#pragma unroll
        for (int u = 0; u < UNR; ++u) {
            const T xu = B.cb + u < B.cols ? B.xv[u] : T(0);
#pragma unroll
            for (int v = 0; v < VEC; ++v) acc[v] = fma(B.av[u][v], xu, acc[v]);
        }
        if (ROLE == 1) {
            // columns cb + u of the block dotted with this tile's rows of x, summed over the
            // lpc lanes that hold them, and added to the partner box's output y_p (offset t)
            // with atomics.  A butterfly first halves the UNR values per exchange (lane bit o
            // keeps one half, sends the other), so that after log2 UNR exchanges lane l holds
            // column ui(l) summed over its UNR-lane group; plain exchanges then finish the
            // sums, and the first UNR lanes of every column group add them (non-symmetric
            // terms, t < 0, add nothing).
            // (a vector, not an array: the selects below then pick values, where selects
            // between array elements become a dynamically indexed array)
            typedef T VU __attribute__((ext_vector_type(UNR)));
            VU tp;
#pragma unroll
            for (int u = 0; u < UNR; ++u) {
                tp[u] = T(0);
#pragma unroll
                for (int v = 0; v < VEC; ++v) tp[u] = fma(B.av[u][v], xb[v], tp[u]);
            }
            int ui = 0;
#pragma unroll
            for (int k = UNR, o = 1; k > 1; k >>= 1, o <<= 1) {
                const bool hi = lane & o;
#pragma unroll
                for (int i = 0; i < k / 2; ++i) {
                    const T snd = hi ? tp[i] : tp[i + k / 2];
                    const T keep = hi ? tp[i + k / 2] : tp[i];
                    tp[i] = keep + xor_lane_n(snd, o);
                }
                ui += hi ? k / 2 : 0;
            }
#pragma unroll
            for (int o = UNR; o < 64; o <<= 1)
                if (o < lpc) tp[0] += xor_lane_n(tp[0], o);
            const int cc = B.cb + ui;
            if ((lane % lpc) < UNR && cc < B.cols && B.t >= 0) atomicAdd(vec + B.t + cc, tp[0]);
        }
    };
    // (an iteration loaded past the last one reads nothing and adds nothing: both halves
    // run unconditionally, so the loop has a single path for the waits)
    Iter B0, B1;
    settle();
    bool h0 = load(B0);
    load(B1);
    while (h0) {
        compute(B0);
        h0 = load(B0);
        compute(B1);
        load(B1);
    }
#pragma unroll
    for (int v = 0; v < VEC; ++v)
        for (int o = lpc; o < 64; o <<= 1) acc[v] += __shfl_xor(acc[v], o, 64);
    if (WPI == 1) {
        if (q == 0 && act)
#pragma unroll
            for (int v = 0; v < VEC; ++v) {
                T *y = vec + it.y + r0 + v;
                if (r0 + v >= rows) continue;
                if (it.flags & 5) atomicAdd(y, acc[v]);
                else *y += acc[v];
            }
        return;
    }
    if (q == 0 && act)
#pragma unroll
        for (int v = 0; v < VEC; ++v)
            if (r0 + v < kRowTile) part[threadIdx.x >> 6][r0 + v] = acc[v];
    __syncthreads();
    if (threadIdx.x < rows) {
        const int t = threadIdx.x;
        T s = part[0][t] + part[1][t] + part[2][t] + part[3][t];
        T *y = vec + it.y + t;
        if (it.flags & 5) atomicAdd(y, s);  // split items; fused items (transposes land in y too)
        else *y += s;
    }
}

// ------------------------------------------------------------------ batched skinny GEMM, kNR right-hand sides
// The same work items as k_bgemv, on a vector pool holding kNR right-hand
// sides per slot (element (slot, rhs) at slot * kNR + rhs): every item is a
// small dense product Y[rows x kNR] += A[rows x cols] X[cols x kNR] on the
// matrix cores (16x16x4 MFMA, FP32 or FP64).
//
// Lane l (m = l % 16, q = l / 16) reads VEC consecutive rows of column c0 + q
// with one 16-byte load: rows VEC m .. VEC m + VEC-1 of a 16 VEC-row group (a
// quarter-wave reads 256 contiguous bytes of a column).  Component u of that
// vector is the MFMA's A(m, q) for the strided row set {VEC m + u}, so VEC
// MFMAs consume one load and X(c0 + q, m) -- kNR contiguous elements per
// column -- is the B operand of all of them.  An MFMA's D(row(q, v), m) then
// belongs to item row  group * 16 VEC + VEC row(q, v) + u, where row(q, v) =
// 4q + v (FP32) or q + 4v (FP64) are the two instructions' result layouts,
// checked on gfx950.
template <typename T>
struct Mfma16;
template <>
struct Mfma16<float> {
    typedef float v4 __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ v4 op(float a, float b, v4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int q, int v) { return 4 * q + v; }
};
template <>
struct Mfma16<double> {
    typedef double v4 __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ v4 op(double a, double b, v4 c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int q, int v) { return q + 4 * v; }
};

// One pass over an item's terms for `rows` of its rows, from h0 on: NG slabs of RG = 16 VEC rows.  The terms are cut
// into 16-column groups (never across a term); of WPI waves each takes every WPI-th group, the next group's loads
// in flight while one is multiplied (raw buffer loads: out-of-range lanes read zeros, no branch guards them).
// The terms of an item (64 of them at a time) sit one per lane, and a group's term is found by a ballot over the
// running group counts: a cursor over descriptors in memory waited on two or three dependent scalar loads a
// group, and those waits cover the LDS counter too.  MFMAs over columns past the term or rows past the pass are
// left out, four at a time.  SYM: the transposed products of symmetric terms as well (below).
// Transfers of a 16-wide product against 128-row items by 4-column chunks from a scalar cursor (FP64, the same
// lists, then those of wide_items): 32^3 grid at 1e-10 193 -> 187 -> 161 us, 3D N = 20011 148 -> 114 -> 102, 2D
// N = 90000 422 -> 370 -> 348, 2D semi-nested N = 40000 207 -> 156, 16^3 77 -> 55, 1D N = 65536 147 -> 110.
template <typename T, int VEC, int NG, bool SYM, int WPI>
__device__ __forceinline__ void bgemm_rows(const GItem &it, int h0, int rows, const GTerm *__restrict__ terms,
                                           const T *__restrict__ A, T *vec, T *smem) {
    typedef typename Mfma16<T>::v4 V4;
    typedef T VL __attribute__((ext_vector_type(VEC)));
    constexpr int RG = 16 * VEC;         // rows of a slab
    constexpr int NS = RG / 4;           // MFMA k-steps of a slab's transposed product
    constexpr int LDR = RG + VEC;        // LDS column of a slab, padded by 16 bytes
    constexpr int SLB = SYM ? 16 * LDR : 16 * RG;  // one slab buffer (or its rows' sums)
    constexpr uint32_t kNoRow = 0x80000000u;  // past any group's size, also with its column offsets added
    const int lane = threadIdx.x & 63;
    const int wv = WPI == 4 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0;
    const int m = lane & 15, q = lane >> 4;
    const int64_t lda = it.lda;
    T *const mine = smem + wv * NG * SLB;  // this wave's buffers, [NG][16][LDR]
    // lane (q, m), element v of the transposed product is column q + 4 v of the group: whole 256- or 512-byte
    // runs per atomic instruction (the FP32 MFMA's row 4 q + v takes its A rows in that order)
    const int tc = sizeof(T) == 8 ? m : (m >> 2) + 4 * (m & 3);
    // X_b(RG g + 4 s + q, m) (zero beyond the rows)
    T xb[SYM ? NG * NS : 1];
    const __amdgpu_buffer_rsrc_t rb = buf_rsrc(vec + (it.xb + h0) * kNR, (uint32_t)(rows * kNR * sizeof(T)));
#pragma unroll
    for (int s = 0; s < (SYM ? NG * NS : 0); ++s) xb[s] = buf_ld<T>(rb, (uint32_t)(((4 * s + q) * kNR + m) * sizeof(T)));
    V4 acc[NG * VEC];
#pragma unroll
    for (int a = 0; a < NG * VEC; ++a) acc[a] = (V4)0;
    uint32_t off[NG][4];
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
        for (int j = 0; j < 4; ++j)
            off[g][j] = RG * g + VEC * m < rows
                            ? (uint32_t)(((4 * j + q) * lda + it.row0 + h0 + RG * g + VEC * m) * sizeof(T))
                            : kNoRow;
    const uint32_t xoff = (uint32_t)((q * kNR + m) * sizeof(T));
    // the window: terms w0 .. w0 + 63, lane k holding term w0 + k and the groups up to its end
    int w0 = it.t0, ends = 0, total = 0, cols = 0;
    int64_t ta = 0, tx = 0, tp = 0;
    auto window = [&]() {
        const bool in = w0 + lane < it.t1;
        const GTerm t = terms[in ? w0 + lane : it.t0];
        ta = t.a;
        tx = t.x;
        tp = t.t;
        cols = in ? t.cols : 0;
        // (wait for them here: a wait left to the loop would be for every load in flight)
        asm volatile("" : "+v"(ta), "+v"(tx), "+v"(tp), "+v"(cols));
        ends = (cols + 15) >> 4;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int u = __shfl_up(ends, o, 64);
            ends += lane >= o ? u : 0;
        }
        total = __builtin_amdgcn_readlane(ends, 63);
    };
    window();
    int G = wv;  // next group of this wave, counted in the window
    auto lane64 = [](int64_t v, int k) {
        const uint32_t lo = __builtin_amdgcn_readlane((int)(uint32_t)v, k), hi = __builtin_amdgcn_readlane((int)(v >> 32), k);
        return (int64_t)(((uint64_t)hi << 32) | lo);
    };
    struct Group {
        VL av[NG][4];
        T bx[4];
        int64_t t;
        int left;  // columns of the term from the group's first one, 0: no group
    };
    auto load = [&](Group &S) {
        while (G >= total && w0 + 64 < it.t1) {
            G -= total;
            w0 += 64;
            window();
        }
        const bool has = G < total;
        const int k = has ? (int)__builtin_ctzll(__ballot(ends > G)) : 0;
        const int nc = __builtin_amdgcn_readlane(cols, k);
        const int c0 = has ? 16 * (G - __builtin_amdgcn_readlane(ends, k) + ((nc + 15) >> 4)) : 0;
        const int64_t t = lane64(tp, k);
        S.left = has ? nc - c0 : 0;
        S.t = SYM && t >= 0 ? t + c0 : -1;
        const int n = min(S.left, 16);
        const __amdgpu_buffer_rsrc_t ra = buf_rsrc(A + lane64(ta, k) + c0 * lda, (uint32_t)(n * lda * sizeof(T)));
        const __amdgpu_buffer_rsrc_t rx = buf_rsrc(vec + (lane64(tx, k) + c0) * kNR, (uint32_t)(n * kNR * sizeof(T)));
        const uint32_t xo = opaque_off(xoff);  // (row steps fold into the loads: hoisted, each would be a register)
#pragma unroll
        for (int j = 0; j < 4; ++j) S.bx[j] = buf_ld<T>(rx, xo + (uint32_t)(4 * j * kNR * sizeof(T)));
#pragma unroll
        for (int g = 0; g < NG; ++g)
#pragma unroll
            for (int j = 0; j < 4; ++j) S.av[g][j] = buf_ldv_nt<VL>(ra, off[g][j]);
        G += WPI;
    };
    auto wave_sync = [] {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    auto put = [&](const Group &S, int g) {
        T *sl = mine + g * SLB;
#pragma unroll
        for (int j = 0; j < 4; ++j) *(VL *)&sl[(4 * j + q) * LDR + VEC * m] = S.av[g][j];
    };
    auto direct = [&](const Group &S, int g) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (4 * j < S.left)
#pragma unroll
                for (int e = 0; e < VEC; ++e) acc[g * VEC + e] = Mfma16<T>::op(S.av[g][j][e], S.bx[j], acc[g * VEC + e]);
    };
    // the transposed product of a group, added to the partner's output after the next loads are issued: loads
    // and atomics share a counter that retires in order, and a wait for loads behind atomics is one for both
    struct Out {
        V4 y;
        int64_t t;
        int left;
    };
    auto compute = [&](const Group &S) {
        Out o{(V4)0, S.t, S.t >= 0 ? S.left : 0};
        if (SYM && S.t >= 0) {
            V4 y[2] = {(V4)0, (V4)0};  // (two chains of the transposed MFMAs)
#pragma unroll
            for (int g = 0; g < NG; ++g) put(S, g);
            wave_sync();
#pragma unroll
            for (int g = 0; g < NG; ++g) {
                T tr[NS];
#pragma unroll
                for (int s = 0; s < NS; ++s) tr[s] = mine[g * SLB + tc * LDR + 4 * s + q];
                direct(S, g);  // (the LDS round trip overlaps the direct products)
#pragma unroll
                for (int s = 0; s < NS; ++s)
                    if (RG * g + 4 * s < rows) y[s & 1] = Mfma16<T>::op(tr[s], xb[g * NS + s], y[s & 1]);
            }
            wave_sync();  // (the next group's slabs overwrite these)
            o.y = y[0] + y[1];
        } else {
#pragma unroll
            for (int g = 0; g < NG; ++g) direct(S, g);
        }
        return o;
    };
    auto flush = [&](const Out &o) {
        if (!SYM) return;
        const __amdgpu_buffer_rsrc_t ry =
            buf_rsrc(vec + (o.left > 0 ? o.t : 0) * kNR, (uint32_t)(min(o.left, 16) * kNR * sizeof(T)));
        const uint32_t xo = opaque_off(xoff);
#pragma unroll
        for (int v = 0; v < 4; ++v) buf_atomic_add(ry, xo + (uint32_t)(4 * v * kNR * sizeof(T)), o.y[v]);
    };
    // two groups rotate (one loaded past the last reads nothing and adds nothing)
    Group S0, S1;
    load(S0);
    load(S1);
    while (S0.left > 0) {
        const Out o0 = compute(S0);
        load(S0);
        flush(o0);
        const Out o1 = compute(S1);
        load(S1);
        flush(o1);
    }
    auto row_of = [&](int g, int e, int v) { return RG * g + VEC * Mfma16<T>::row(q, v) + e; };
    T *y = vec + (it.y + h0) * kNR;
    const bool atomic = SYM || (it.flags & 1);
    if constexpr (WPI == 1) {
#pragma unroll
        for (int g = 0; g < NG; ++g)
#pragma unroll
            for (int e = 0; e < VEC; ++e)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int r = row_of(g, e, v);
                    if (r >= rows) continue;
                    if (atomic) atomicAdd(y + r * kNR + m, acc[g * VEC + e][v]);
                    else y[r * kNR + m] += acc[g * VEC + e][v];
                }
    } else {
        // the four waves' direct products, summed through LDS (each wave's rows lie in its own buffers)
        wave_sync();
#pragma unroll
        for (int g = 0; g < NG; ++g)
#pragma unroll
            for (int e = 0; e < VEC; ++e)
#pragma unroll
                for (int v = 0; v < 4; ++v) mine[row_of(g, e, v) * kNR + m] = acc[g * VEC + e][v];
        __syncthreads();
        for (int e = threadIdx.x; e < rows * kNR; e += 256) {
            const T sum = (smem[e] + smem[NG * SLB + e]) + (smem[2 * NG * SLB + e] + smem[3 * NG * SLB + e]);
            if (atomic) atomicAdd(y + e, sum);
            else y[e] += sum;
        }
    }
}
// A pass's rows: as many as two slabs of 16-byte loads hold (64 in FP64, 128 in FP32), the last rows of an item
// in the narrowest slab that holds them (a box of 20 rows takes one 32-row slab, one of 10 a 16-row slab of
// 8- or 4-byte loads).
template <typename T>
constexpr int kPassRows = 2 * 16 * (16 / sizeof(T));
template <typename T, bool SYM, int WPI>
__device__ __forceinline__ void bgemm_pass(const GItem &it, int h0, const GTerm *__restrict__ terms,
                                           const T *__restrict__ A, T *vec, T *smem) {
    constexpr int VMAX = 16 / sizeof(T);
    const int left = min(it.rows - h0, kPassRows<T>);
    if (left > 16 * VMAX) bgemm_rows<T, VMAX, 2, SYM, WPI>(it, h0, left, terms, A, vec, smem);
    else if (left <= 16) bgemm_rows<T, 1, 1, SYM, WPI>(it, h0, left, terms, A, vec, smem);
    else if (VMAX == 4 && left <= 32) bgemm_rows<T, 2, 1, SYM, WPI>(it, h0, left, terms, A, vec, smem);
    else bgemm_rows<T, VMAX, 1, SYM, WPI>(it, h0, left, terms, A, vec, smem);
}

// WPI 4: one item per workgroup; WPI 1: one item per wave (launches of many small items: no cross-wave
// reduction, four items in flight per workgroup), nitems bounds the last one.  blockIdx.y: the pass.
template <typename T, int ROLE, int WPI>
__global__ __launch_bounds__(256) void k_bgemm(const GItem *__restrict__ items, int nitems,
                                               const GTerm *__restrict__ terms, const T *__restrict__ A0,
                                               const T *__restrict__ A1, const T *const *__restrict__ tab, T *vec) {
    const int idx = WPI == 4 ? (int)blockIdx.x : 4 * (int)blockIdx.x + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (idx >= nitems) return;  // (WPI 1 only: whole waves, and no barrier follows)
    const GItem it = items[idx];
    const int h0 = blockIdx.y * kPassRows<T>;
    if (h0 >= it.rows) return;
    // batched systems: pool pair of system flags >> 8 from the table
    const T *__restrict__ A = tab ? tab[2 * (it.flags >> 8) + ((it.flags >> 1) & 1)] : ((it.flags & 2) ? A1 : A0);
    if constexpr (WPI == 4) {
        __shared__ __attribute__((aligned(16))) T smem[4 * kPassRows<T> * kNR];
        bgemm_pass<T, false, 4>(it, h0, terms, A, vec, smem);
    } else {
        bgemm_pass<T, false, 1>(it, h0, terms, A, vec, nullptr);
    }
}

// Direct and transposed products of the stored blocks in one read, kNR right-hand sides
// (the fused M2L + near-field launch of the multi-vector pass).  One item (box b, rows <= 128) per
// workgroup, its rows in passes of up to RG NG (RG = 16 VEC).  The item's terms K(b, p) are cut into
// 16-column groups (never across a term); wave wv takes groups wv, wv + 4, ...  A group is NG slabs of
// RG rows x 16 columns, loaded in the direct product's layout (lane (m, q): VEC consecutive rows of column
// 4 j + q, j < 4: 16-byte loads, 256-byte runs per column; the next group in flight) and multiplied into
// the pass's rows (as k_bgemm: A(m, q) = K(VEC m + e, 4 j + q), B(q, m) = X_p(4 j + q, m)).  For a
// symmetric term (t >= 0) the wave also writes the slabs to its LDS buffers and reads them back with a
// column per lane % 16 and a row per lane / 16, the A operand of K^T: with B(q, m) = X_b(4 s + q, m), held in
// registers, it forms the 16 x kNR block Y_p(c0 .. c0 + 15, :) += K(rows, c0 ..)^T X_b and adds it to the
// partner's output with atomics.  MFMAs over columns past the term or rows past the pass are left out, four at
// a time.  The item's own rows are added atomically too (other items' transposes land in them).  Each
// stored element is read once per pass, where k_bgemm + k_bgemm_tl read it twice.
// The terms of an item (64 of them at a time) sit one per lane, and a group's term is found by a ballot over
// the running group counts: a cursor over descriptors in memory waited on two or three dependent scalar
// loads a group, and those waits cover the LDS counter too.
// FP64: 64 MFMA flops per stored element (direct and transposed, 16 right-hand sides) against
// 8 bytes, so the launch needs both HBM and the FP64 matrix cores (78.6 TFLOP/s) at once;
// launch bounds cap it at 256 registers a lane (two waves per SIMD).
// Measured against slabs of 128-row items from a scalar cursor, with the atomics before the next loads (the same
// lists), FP64 / FP32: 32^3 grid at 1e-10 (1.9 GB) 517 / 277 -> 492 / 255 us, 3D N = 20011 258 / 148 -> 231 /
// 129, 2D N = 90000 328 / 195 -> 317 / 162; with the lists of wide_items 448 / 232, 204 / 113, 292 / 143.
// Without loads from HBM it takes 440 us on the first, without the partner's atomics 350, with the direct
// products only 155 (MFMA time 105 each way): the matrix pipe and the atomics share the bound.
template <typename T>
__global__ __launch_bounds__(256, 2) void k_bgemm_sym(const GItem *__restrict__ items, const GTerm *__restrict__ terms,
                                                      const T *__restrict__ A0, const T *__restrict__ A1,
                                                      const T *const *__restrict__ tab, T *vec) {
    constexpr int VMAX = 16 / sizeof(T);
    __shared__ __attribute__((aligned(16))) T smem[4 * 2 * 16 * (16 * VMAX + VMAX)];
    const GItem it = items[blockIdx.x];
    const T *__restrict__ A = tab ? tab[2 * (it.flags >> 8) + ((it.flags >> 1) & 1)] : ((it.flags & 2) ? A1 : A0);
    for (int h0 = 0; h0 < it.rows; h0 += kPassRows<T>) {
        if (h0 > 0) __syncthreads();  // (the sums of the pass before are still read)
        bgemm_pass<T, true, 4>(it, h0, terms, A, vec, smem);
    }
}

// Transposed products of the symmetric blocks on the 16-wide path:
// Y[j, n] += sum_i K[i, row0 + j] X[i, n] for an item's output rows j (box p) and
// terms K(b, p) (leading dimension tm.ld, inner dimension tm.cols = r_b), through LDS.
// The MFMA's A operand wants an output row (a column of K) per lane % 16 and the inner
// index per lane / 16, while K's contiguous direction is the inner one: loading that
// layout directly reads 64-byte runs per column.  Instead a slab is 16 VEC inner
// indices (256 bytes of every column); wave w owns output groups w and w + 4 (16 rows each) of the item and reads
// its 16-column groups slab by slab with 16 lanes per column (whole 256-byte runs),
// writes them to its own LDS region and reads them back in the MFMA's A layout (lane
// (m, q): VEC inner indices of column 16 g + m).  The next slab's loads are in flight
// while a slab is multiplied: the slab's B operands are loaded before them, since
// vector loads retire in order.  No wave reads another wave's region, and every wave
// writes only its own output rows.
template <typename T, int LPC>
__global__ __launch_bounds__(256) void k_bgemm_tl(const GItem *__restrict__ items, const GTerm *__restrict__ terms,
                                                  const T *__restrict__ A0, const T *__restrict__ A1,
                                                  const T *const *__restrict__ tab, T *vec) {
    typedef typename Mfma16<T>::v4 V4;
    constexpr int VEC = 16 / sizeof(T);
    constexpr int SL = LPC * VEC;      // inner indices of one slab (LPC lanes per column)
    constexpr int LD = SL + VEC;       // LDS row: one column's slab, padded by 16 bytes
    constexpr int CPL = 64 / LPC;      // columns per load instruction
    constexpr int NJ = 16 / CPL;       // load instructions per 16-column group
    constexpr int NSUB = LPC / 4;      // MFMA k-steps (4 VEC inner indices) per slab
    constexpr int U = 16 / LPC;        // slabs per iteration
    typedef T VL __attribute__((ext_vector_type(VEC)));
    __shared__ __attribute__((aligned(16))) T lds[4][U][32][LD];
    const GItem it = items[blockIdx.x];
    const CGTerm *const tms = (const CGTerm *)terms;
    const T *__restrict__ A = tab ? tab[2 * (it.flags >> 8) + ((it.flags >> 1) & 1)] : ((it.flags & 2) ? A1 : A0);
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int rows = it.rows;
    const int ng = (rows + 15) >> 4;
    const int m = lane & 15, q = lane >> 4;       // MFMA operand lane
    const int il = lane % LPC, cl = lane / LPC;   // load lane: inner chunk, column
    // Items of one or two groups split their slabs over the waves instead: wave w takes
    // group w % ng and every ns-th slab from the (w / ng)-th, and the partial products are
    // summed through LDS at the end.
    const int ns = ng <= 2 ? 4 / ng : 1;
    const int g0 = ns > 1 ? wv % ng : wv;  // first group of this wave (the second is wv + 4)
    const int nown = ns > 1 ? 1 : (wv < ng) + (wv + 4 < ng);
    if (nown == 0) return;  // (ns == 1 only: no barrier follows)
    V4 acc[2] = {(V4)0, (V4)0};
    int lt = it.t0, lk = ns > 1 ? wv / ng : 0;  // next slab to load (term, slab of the term)
    auto settle = [&]() {
        while (lt < it.t1) {
            const int nk = (tms[lt].cols + SL - 1) / SL;
            if (lk < nk) break;
            lk -= nk;
            ++lt;
        }
    };
    struct Slab {
        int64_t x;         // input offset
        int cols, i0;      // inner size, first inner index
        int okm, vlim;     // lanes' valid loads, valid inner indices from this lane's first
    };
    Slab S[U];
    VL L[U][2][NJ];
    // load the next slab into L[u] (past the last slab it still loads, from the last term,
    // and the loads are dropped: loads under a branch, or values used at once, would make
    // the next wait drain all of them)
    auto next = [&](int u) -> bool {
        settle();
        const bool has = lt < it.t1;
        const GTerm tm = term_at(tms, has ? lt : it.t1 - 1);
        S[u].x = tm.x;
        S[u].cols = tm.cols;
        S[u].i0 = has ? lk * SL : tm.cols;
        const int io = S[u].i0 + VEC * il;
        S[u].okm = 0;
        S[u].vlim = tm.cols - io;
#pragma unroll
        for (int gi = 0; gi < 2; ++gi)
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const int c = 16 * (gi ? wv + 4 : g0) + cl + CPL * j;  // item row = column of the block
                const bool ok = gi < nown && c < rows && io < tm.cols;
                S[u].okm |= ok ? 1 << (NJ * gi + j) : 0;
                L[u][gi][j] = ld_nt((const VL *)(A + tm.a + (ok ? (int64_t)(it.row0 + c) * tm.ld + io : 0)));
            }
        lk += has ? ns : 0;
        return has;
    };
    auto wave_sync = [] {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    bool more = false;
#pragma unroll
    for (int u = 0; u < U; ++u) more |= next(u);
    while (more) {
        // staged with every entry outside the block set to zero, so that the B operands of
        // inner indices beyond the block (clamped loads of a valid x) multiply zeros
        T bx[U][NSUB][VEC];
        Slab C[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
#pragma unroll
            for (int gi = 0; gi < 2; ++gi)
#pragma unroll
                for (int j = 0; j < NJ; ++j) {
                    VL v = L[u][gi][j];
#pragma unroll
                    for (int e = 0; e < VEC; ++e)
                        v[e] = ((S[u].okm >> (NJ * gi + j)) & 1) && e < S[u].vlim ? v[e] : T(0);
                    *(VL *)&lds[wv][u][16 * gi + cl + CPL * j][VEC * il] = v;
                }
#pragma unroll
            for (int s = 0; s < NSUB; ++s) {
                const int i = S[u].i0 + 4 * VEC * s + VEC * q;
#pragma unroll
                for (int e = 0; e < VEC; ++e) bx[u][s][e] = vec[(S[u].x + min(i + e, S[u].cols - 1)) * kNR + m];
            }
            C[u] = S[u];
        }
        more = false;
#pragma unroll
        for (int u = 0; u < U; ++u) more |= next(u);
        wave_sync();
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (C[u].i0 < C[u].cols)  // (a slab past the last one multiplies nothing)
#pragma unroll
                for (int s = 0; s < NSUB; ++s)
#pragma unroll
                    for (int gi = 0; gi < 2; ++gi)
                        if (gi < nown) {
                            const VL a = *(const VL *)&lds[wv][u][16 * gi + m][4 * VEC * s + VEC * q];
#pragma unroll
                            for (int e = 0; e < VEC; ++e) acc[gi] = Mfma16<T>::op(a[e], bx[u][s][e], acc[gi]);
                        }
        wave_sync();
    }
    if (ns > 1) {
        // partial products of group g0 from waves g0, g0 + ng, ..: summed by wave g0
        T(*red)[kNR] = (T(*)[kNR])&lds[wv][0][0][0];
#pragma unroll
        for (int v = 0; v < 4; ++v) red[Mfma16<T>::row(q, v)][m] = acc[0][v];
        __syncthreads();
        if (wv >= ng) return;
        for (int o = wv + ng; o < 4; o += ng) {
            T(*ro)[kNR] = (T(*)[kNR])&lds[o][0][0][0];
#pragma unroll
            for (int v = 0; v < 4; ++v) acc[0][v] += ro[Mfma16<T>::row(q, v)][m];
        }
    }
#pragma unroll
    for (int gi = 0; gi < 2; ++gi)
        if (gi < nown) {
            T *y = vec + it.y * kNR + m;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int r = 16 * (gi ? wv + 4 : g0) + Mfma16<T>::row(q, v);
                if (r < rows) {
                    if (it.flags & 1) atomicAdd(y + (int64_t)r * kNR, acc[gi][v]);
                    else y[(int64_t)r * kNR] += acc[gi][v];
                }
            }
        }
}

// leading sub-block copies from the FP32 pool into the inner-operator buffer
__global__ void k_copy32(const CopyJob *__restrict__ jobs, const float *__restrict__ src, float *dst) {
    const CopyJob jb = jobs[blockIdx.x];
    const int64_t tot = (int64_t)jb.m * jb.n;
    for (int64_t e = threadIdx.x; e < tot; e += blockDim.x) {
        int i = (int)(e % jb.m), j = (int)(e / jb.m);
        dst[jb.dst + (int64_t)j * jb.ldd + i] = src[jb.src + (int64_t)j * jb.lds + i];
    }
}

// ------------------------------------------------------------------ on-the-fly P2P / M2L
// The near-field and M2L terms of a work list are blocks of plain kernel entries
// K(target points, source points); this kernel evaluates them instead of reading
// them.  Target row r of an item is vector slot it.y + r, source column c of a
// term is slot tm.x + c; the slot tables give each slot's point.  VALU-bound:
// per entry 3 sub + 3 mul/fma + sqrt + log (3D RBF) and the diagonal test.
__device__ __forceinline__ float koff_f(int dim, int choice, float dx, float dy, float dz) {
    const float a = 1.0e-4f;
    if (dim == 1) {
        float R = fabsf(dx);
        if (choice == 0) return __logf(R);
        return R < a ? R * 1.0e4f : a / R;
    } else if (dim == 2) {
        float R2 = dx * dx + dy * dy;
        if (choice == 0) return -0.0795774715459476679f * __logf(R2);  // -(1/2pi) * 0.5 * log R^2
        float R = sqrtf(R2);
        return R < a ? R * 1.0e4f : a / R;
    } else {
        float R2 = dx * dx + dy * dy + dz * dz;
        if (choice == 0) return 0.0795774715459476679f * rsqrtf(R2);  // 1 / (4 pi R)
        float R = sqrtf(R2);
        float lr = __logf(R);
        // (R log R - 1) / (a log a - 1) below a, log R / log a above
        return R < a ? (R * lr - 1.0f) * -0.9990798135f : lr * -0.1085736205f;
    }
}

template <typename T>
__device__ __forceinline__ T koff_t(int dim, int choice, T dx, T dy, T dz);
template <>
__device__ __forceinline__ float koff_t<float>(int dim, int choice, float dx, float dy, float dz) {
    return koff_f(dim, choice, dx, dy, dz);
}
template <>
__device__ __forceinline__ double koff_t<double>(int dim, int choice, double dx, double dy, double dz) {
    return koff(dim, choice, dx, dy, dz);
}

// Coordinate differences: FP64 directly; FP32 from (hi, lo) pairs, where the
// hi difference of two nearby points is exact or nearly so and the lo
// difference restores the digits plain FP32 coordinates would lose.
template <typename T>
struct Coords {
    const T *x, *y, *z;
    const float *xl, *yl, *zl;
};

// FP32 entries from the squared distance R2 (1D: the distance R): the common case of each
// kernel (otf_val32) and the case of points closer than a = 1e-4 (otf_near32, RBF only;
// otf_rare32 says whether it applies).  log R = log2(R^2) ln2 / 2, so the common 3D and 2D
// cases need no square root; hardware log2 / rsq / rcp (about 1 ulp; arguments are never
// denormal: R >= 1e-4 in the common case).
template <int DIM, int CH>
__device__ __forceinline__ float otf_val32(float R2) {
    constexpr float kLn2 = 0.69314718055994531f;
    if constexpr (DIM == 3) {
        if constexpr (CH == 0) return 0.0795774715459476679f * __builtin_amdgcn_rsqf(R2);  // 1 / (4 pi R)
        return __builtin_amdgcn_logf(R2) * (float)(0.5 * 0.69314718055994531 / -9.2103403719761836);  // log R / log a
    } else if constexpr (DIM == 2) {
        if constexpr (CH == 0) return (-0.0795774715459476679f * kLn2) * __builtin_amdgcn_logf(R2);  // -(1/4pi) log R^2
        return 1.0e-4f * __builtin_amdgcn_rsqf(R2);  // a / R
    } else {
        if constexpr (CH == 0) return kLn2 * __builtin_amdgcn_logf(R2);  // log R (R2 holds R)
        return 1.0e-4f * __builtin_amdgcn_rcpf(R2);                     // a / R
    }
}
template <int DIM, int CH>
__device__ __forceinline__ bool otf_rare32(float R2) {
    if constexpr (CH == 0) return false;
    return DIM == 1 ? R2 < 1.0e-4f : R2 < 1.0e-8f;
}
template <int DIM>
__device__ __forceinline__ float otf_near32(float R2) {
    const float R = DIM == 1 ? R2 : sqrtf(R2);
    if constexpr (DIM == 3) return (R * logf(R) - 1.0f) * -0.9990798135f;  // (R log R - 1) / (a log a - 1)
    return R * 1.0e4f;                                                       // R / a
}

// One source point of a tile: coordinates (FP32: hi and lo parts), its value and point id.
template <typename T>
struct OtfSrc;
template <>
struct OtfSrc<float> {
    float x, y, z, xl, yl, zl, v;
    int pid;
};
template <>
struct OtfSrc<double> {
    double x, y, z, v;
    int pid, pad;
};

template <typename T>
struct OtfTgt {
    T x, y, z;
    float xl, yl, zl;
    int pid;
};

template <typename T>
__device__ __forceinline__ OtfTgt<T> otf_target(const Coords<T> &C, const int32_t *pid, int dim, int64_t ts) {
    OtfTgt<T> t;
    t.x = C.x[ts];
    t.y = dim > 1 ? C.y[ts] : T(0);
    t.z = dim > 2 ? C.z[ts] : T(0);
    t.xl = t.yl = t.zl = 0.f;
    if (C.xl) {
        t.xl = C.xl[ts];
        t.yl = dim > 1 ? C.yl[ts] : 0.f;
        t.zl = dim > 2 ? C.zl[ts] : 0.f;
    }
    t.pid = pid[ts];
    return t;
}

// Entries K(t0, q) and K(t1, q) of two target rows and one source, accumulated with the
// source's value.  DIAG: the diagonal rule where the points are the same (a tile holding one
// of the item's own points: the near-field self blocks).  The FP32 case for points closer
// than a is a branch the wave takes only when one of its lanes needs it.
template <typename T, int DIM, int CH, bool DIAG>
__device__ __forceinline__ void otf_pair(const OtfTgt<T> &t0, const OtfTgt<T> &t1, const OtfSrc<T> &q, T diag,
                                         T &acc0, T &acc1) {
    T v0, v1;
    if constexpr (sizeof(T) == 4) {
        float r0, r1;
        if constexpr (DIM == 1) {
            r0 = fabsf((t0.x - q.x) + (t0.xl - q.xl));
            r1 = fabsf((t1.x - q.x) + (t1.xl - q.xl));
        } else {
            const float ax = (t0.x - q.x) + (t0.xl - q.xl), bx = (t1.x - q.x) + (t1.xl - q.xl);
            const float ay = (t0.y - q.y) + (t0.yl - q.yl), by = (t1.y - q.y) + (t1.yl - q.yl);
            r0 = fmaf(ay, ay, ax * ax);
            r1 = fmaf(by, by, bx * bx);
            if constexpr (DIM == 3) {
                const float az = (t0.z - q.z) + (t0.zl - q.zl), bz = (t1.z - q.z) + (t1.zl - q.zl);
                r0 = fmaf(az, az, r0);
                r1 = fmaf(bz, bz, r1);
            }
        }
        v0 = otf_val32<DIM, CH>(r0);
        v1 = otf_val32<DIM, CH>(r1);
        if constexpr (CH != 0) {
            const bool n0 = otf_rare32<DIM, CH>(r0), n1 = otf_rare32<DIM, CH>(r1);
            if (__ballot(n0 || n1)) {
                if (n0) v0 = otf_near32<DIM>(r0);
                if (n1) v1 = otf_near32<DIM>(r1);
            }
        }
    } else {
        // the stored operator's own formula (koff), so the FP64 products agree to rounding
        v0 = koff(DIM, CH, t0.x - q.x, t0.y - q.y, t0.z - q.z);
        v1 = koff(DIM, CH, t1.x - q.x, t1.y - q.y, t1.z - q.z);
    }
    if constexpr (DIAG) {
        v0 = q.pid == t0.pid ? diag : v0;
        v1 = q.pid == t1.pid ? diag : v1;
    }
    acc0 = fma(v0, q.v, acc0);
    acc1 = fma(v1, q.v, acc1);
}

// P2P / M2L on the fly, tiled.  One workgroup per item (<= 128 target rows).  Source
// points of the item's terms are staged 256 at a time in LDS (coordinates, value, id: one
// coalesced load per source instead of one broadcast load per source and target row).
// Thread t owns target rows g and g + h (h = ceil(rows / 2), g = t mod h) in registers and
// the sources k = sub, sub + nsub, ... of each tile (sub = t / h, nsub = 256 / h), so every
// source read from LDS feeds two entries; the partial sums of the nsub source subsets are
// added through LDS at the end.  A tile is checked once for points of the item itself (the
// near-field self blocks); only such tiles test every entry for the diagonal.
constexpr int kOtfTile = 256;
template <typename T, int DIM, int CH>
__global__ __launch_bounds__(256) void k_otf(const GItem *__restrict__ items, const GTerm *__restrict__ terms,
                                             Coords<T> C, const int32_t *__restrict__ pid, T diag, T *vec) {
    constexpr int dim = DIM;
    __shared__ OtfSrc<T> tile[kOtfTile];
    __shared__ T part[2 * 256];
    __shared__ int tpmin, tpmax;
    const GItem it = items[blockIdx.x];
    const int R = it.rows;
    const int h = (R + 1) >> 1;
    const int nsub = 256 / h;
    const int t = threadIdx.x;
    const bool act = t < nsub * h;
    const int g = act ? t % h : 0, sub = act ? t / h : 0;
    const bool two = g + h < R;
    const OtfTgt<T> t0 = otf_target<T>(C, pid, dim, it.y + g);
    const OtfTgt<T> t1 = otf_target<T>(C, pid, dim, it.y + (two ? g + h : g));
    if (t == 0) {
        tpmin = INT_MAX;
        tpmax = INT_MIN;
    }
    __syncthreads();
    if (t < R) {
        const int p = pid[it.y + t];
        atomicMin(&tpmin, p);
        atomicMax(&tpmax, p);
    }
    __syncthreads();
    const int pmin = tpmin, pmax = tpmax;
    T acc0 = 0, acc1 = 0;
    for (int tt = it.t0; tt < it.t1; ++tt) {
        const GTerm tm = terms[tt];
        for (int c0 = 0; c0 < tm.cols; c0 += kOtfTile) {
            const int n = min(kOtfTile, tm.cols - c0);
            __syncthreads();  // (the previous tile is no longer read)
            bool own = false;
            if (t < n) {
                const int64_t sl = tm.x + c0 + t;
                OtfSrc<T> q;
                q.x = C.x[sl];
                q.y = dim > 1 ? C.y[sl] : T(0);
                q.z = dim > 2 ? C.z[sl] : T(0);
                if constexpr (sizeof(T) == 4) {
                    q.xl = C.xl ? C.xl[sl] : 0.f;
                    q.yl = dim > 1 && C.yl ? C.yl[sl] : 0.f;
                    q.zl = dim > 2 && C.zl ? C.zl[sl] : 0.f;
                }
                q.v = vec[sl];
                q.pid = pid[sl];
                tile[t] = q;
                own = q.pid >= pmin && q.pid <= pmax;
            }
            const bool diag_tile = __syncthreads_or(own);
            if (!act) continue;
            if (!diag_tile) {
                for (int k = sub; k < n; k += nsub) otf_pair<T, DIM, CH, false>(t0, t1, tile[k], diag, acc0, acc1);
            } else {
                for (int k = sub; k < n; k += nsub) otf_pair<T, DIM, CH, true>(t0, t1, tile[k], diag, acc0, acc1);
            }
        }
    }
    // partial sums of the source subsets: part[sub * R + row]
    __syncthreads();
    if (act) {
        part[sub * R + g] = acc0;
        if (two) part[sub * R + g + h] = acc1;
    }
    __syncthreads();
    if (t < R) {
        T sum = 0;
        for (int q = 0; q < nsub; ++q) sum += part[q * R + t];
        T *y = vec + it.y + t;
        if (it.flags & 1) atomicAdd(y, sum);
        else *y += sum;
    }
}

// ------------------------------------------------------------------ small vector kernels
__global__ void k_to_fp32(const double *a, float *b, int64_t n) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        b[i] = (float)a[i];
}
__global__ void k_to_fp64(const float *a, double *b, int64_t n) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        b[i] = (double)a[i];
}
// Read-only stream (the read bandwidth a streaming kernel is compared with): chunks of
// kStreamUnr x 256 16-byte words, one chunk per workgroup and trip (lane t loads words
// t, t + 256, ... of the chunk, all nontemporal and issued before any is used), chunks
// strided over the grid.  The words are folded into one that is written only when it
// equals a value it practically never takes, so the loads stay live and nothing is written.
constexpr int kStreamUnr = 8;
typedef uint32_t Word16 __attribute__((ext_vector_type(4)));
__global__ __launch_bounds__(256) void k_stream_read(const Word16 *__restrict__ p, int64_t nchunks,
                                                     uint32_t *__restrict__ out) {
    uint32_t acc = 0;
    for (int64_t c = blockIdx.x; c < nchunks; c += gridDim.x) {
        const Word16 *q = p + c * (kStreamUnr * 256) + threadIdx.x;
        Word16 w[kStreamUnr];
#pragma unroll
        for (int u = 0; u < kStreamUnr; ++u) w[u] = __builtin_nontemporal_load(q + u * 256);
#pragma unroll
        for (int u = 0; u < kStreamUnr; ++u) acc = (acc ^ w[u].x ^ w[u].y) + (w[u].z ^ w[u].w);
    }
    if (acc == 0x9E3779B9u) out[blockIdx.x] = acc;
}

template <typename T>
__global__ void k_fill(T *a, int64_t n, T v) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        a[i] = v;
}
template <typename T>
__global__ void k_permute_in(const double *x, int64_t ldx, T *xt, int64_t ldt, const int32_t *perm, int64_t N) {
    const int r = blockIdx.y;
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < N; t += (int64_t)gridDim.x * blockDim.x)
        xt[r * ldt + t] = (T)x[r * ldx + perm[t]];
}
// What comes before the launches of a product, in one pass: the pool's input from scale x (tree order, or
// input order through perm; scale / sqrt(*norm2) where a norm is given), a copy of it where the caller keeps
// one, and zeros in everything the product accumulates into.  x may lie in py (an entry is read before it is zeroed, by the same thread).
template <typename T>
__global__ __launch_bounds__(256) void k_begin(const double *x, double scale, const double *norm2, double *copy,
                                               const int32_t *perm, T *px, int64_t N, T *py, int64_t len) {
    if (norm2) scale /= sqrt(*norm2);
    const int64_t step = (int64_t)gridDim.x * 256;
    for (int64_t i = blockIdx.x * (int64_t)256 + threadIdx.x; i < max(N, len); i += step) {
        if (i < N) {
            const double v = scale * x[perm ? perm[i] : i];
            if (copy) copy[i] = v;
            px[i] = (T)v;
        }
        if (i < len) py[i] = T(0);
    }
}
template <typename T>
__global__ void k_permute_out(const T *yt, int64_t ldt, double *y, int64_t ldy, const int32_t *perm, int64_t N) {
    const int r = blockIdx.y;
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < N; t += (int64_t)gridDim.x * blockDim.x)
        y[r * ldy + perm[t]] = (double)yt[r * ldt + t];
}

// Dense rows of A x with entries evaluated on the fly (getTruePoten,
// 3D/codes/HODLR3Dtree.hpp:2630-2643).  64 rows per workgroup, 4 column
// groups; source coordinates and x staged through LDS.
__global__ __launch_bounds__(256) void k_dense_rows(const int32_t *__restrict__ rows, int64_t nrows,
                                                    const double *__restrict__ xt, double *__restrict__ y, int64_t N,
                                                    KParams kp) {
    __shared__ double sx[256], sy[256], sz[256], sq[256];
    __shared__ double part[4][64];
    const int lane = threadIdx.x & 63, g = threadIdx.x >> 6;
    const int64_t r = blockIdx.x * 64LL + lane;
    const bool active = r < nrows;
    const int i = active ? (rows ? rows[r] : (int)r) : 0;
    PointI p = load_point(kp, i);
    double acc = 0.0;
    for (int64_t j0 = 0; j0 < N; j0 += 256) {
        int64_t j = j0 + threadIdx.x;
        __syncthreads();
        if (j < N) {
            sx[threadIdx.x] = kp.px[j];
            sy[threadIdx.x] = kp.dim > 1 ? kp.py[j] : 0.0;
            sz[threadIdx.x] = kp.dim > 2 ? kp.pz[j] : 0.0;
            sq[threadIdx.x] = xt[j];
        }
        __syncthreads();
        const int nj = (int)min<int64_t>(256, N - j0);
        for (int q = g; q < nj; q += 4) {
            int jj = (int)(j0 + q);
            double v = (jj == i) ? kp.diag : koff(kp.dim, kp.choice, p.x - sx[q], p.y - sy[q], p.z - sz[q]);
            acc = fma(v, sq[q], acc);
        }
    }
    part[g][lane] = acc;
    __syncthreads();
    if (g == 0 && active) y[r] = part[0][lane] + part[1][lane] + part[2][lane] + part[3][lane];
}

// ------------------------------------------------------------------ BLAS-1 for Arnoldi (FP64)
// x += sign V c
__global__ void k_mgemv(const double *__restrict__ V, int64_t ldv, int k, const double *__restrict__ h,
                        double *__restrict__ w, int64_t n, double sign) {
    __shared__ double hs[1024];
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i - threadIdx.x < n;
         i += (int64_t)gridDim.x * blockDim.x) {
        double acc = 0.0;
        for (int l0 = 0; l0 < k; l0 += 1024) {
            int l1 = min(k, l0 + 1024);
            __syncthreads();
            for (int l = l0 + threadIdx.x; l < l1; l += blockDim.x) hs[l - l0] = h[l];
            __syncthreads();
            if (i < n)
                for (int l = l0; l < l1; ++l) acc = fma(V[(int64_t)l * ldv + i], hs[l - l0], acc);
        }
        if (i < n) w[i] += sign * acc;
    }
}
// One pass of the Arnoldi process over a vector w of n rows, 256 R rows per workgroup, rows in registers:
//   w = src                      (the product's FP32 output, when src is given)
//   w -= sum_l V_l sub[l]        for the ns columns from s0 on
//   out[l] = V_l . w             for the nd columns from d0 on, or out[0] = w . w when norm is set
// A Gram-Schmidt step (dots, subtraction with the second dots, second subtraction with the norm) is three
// such launches; the workgroup that arrives last sums the others' dots, in workgroup order, and copies
// nhost numbers from all_h, then out, to page-locked host memory, then seq to flag, which the host polls.
// (Dots, their reduction and each subtraction as launches of their own, and a copy to the host, were eight
// launches of 4 to 5 us and 30 us of idle GPU while the host waited, rotated and launched.)
constexpr int kCgsCols = 128;  // columns whose coefficients, or sums, are in LDS at a time
template <int R, typename S>
__global__ __launch_bounds__(256) void k_cgs(const double *__restrict__ V, int64_t ldv, const S *src, double *w,
                                             int64_t n, int s0, int ns, const double *__restrict__ sub, int d0, int nd,
                                             int norm, double *partial, uint32_t *arrived, double *out, int last_sums,
                                             const double *all_h, int nhost, double *host, uint64_t *flag,
                                             uint64_t seq) {
    __shared__ double hs[256];
    __shared__ double wpart[4][kCgsCols];
    __shared__ int last;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, tid = threadIdx.x;
    const int64_t i0 = blockIdx.x * (int64_t)(256 * R) + tid;
    double x[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int64_t i = i0 + 256 * r;
        x[r] = i < n ? (src ? (double)src[i] : w[i]) : 0.0;
    }
    for (int l0 = 0; l0 < ns; l0 += kCgsCols) {
        const int nl = min(ns - l0, kCgsCols);
        __syncthreads();
        for (int l = tid; l < nl; l += 256) hs[l] = sub[l0 + l];
        __syncthreads();
        const double *v = V + (int64_t)(s0 + l0) * ldv;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int64_t i = i0 + 256 * r;
            if (i >= n) continue;
            double a = 0.0;
#pragma unroll 8
            for (int l = 0; l < nl; ++l) a = fma(v[(int64_t)l * ldv + i], hs[l], a);
            x[r] -= a;
        }
    }
    if (src || ns > 0)
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int64_t i = i0 + 256 * r;
            if (i < n) w[i] = x[r];
        }
    const int nt = norm ? 1 : nd;
    if (norm) {
        double a = 0.0;
#pragma unroll
        for (int r = 0; r < R; ++r) a = fma(x[r], x[r], a);
        a = wave_sum(a);
        if (lane == 0) wpart[wv][0] = a;
        __syncthreads();
        if (tid == 0)
            st_agent(partial + blockIdx.x, (wpart[0][0] + wpart[1][0]) + (wpart[2][0] + wpart[3][0]));
    }
    for (int l0 = 0; l0 < nd && !norm; l0 += kCgsCols) {
        const int nl = min(nd - l0, kCgsCols);
        const double *v = V + (int64_t)(d0 + l0) * ldv;
        for (int l = 0; l < nl; l += 8) {
            typedef double D8 __attribute__((ext_vector_type(8)));
            D8 p = (D8)0.0;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int64_t i = i0 + 256 * r;
                const int64_t ii = i < n ? i : 0;  // (x is zero there)
#pragma unroll
                for (int u = 0; u < 8; ++u) p[u] = fma(v[(int64_t)min(l + u, nl - 1) * ldv + ii], x[r], p[u]);
            }
            int ui = 0;
#pragma unroll
            for (int k = 8, o = 1; k > 1; k >>= 1, o <<= 1) {
                const bool hi = lane & o;
#pragma unroll
                for (int q = 0; q < k / 2; ++q) {
                    const double snd = hi ? p[q] : p[q + k / 2];
                    const double keep = hi ? p[q + k / 2] : p[q];
                    p[q] = keep + (o == 1 ? fold_lane<1>(snd) : o == 2 ? fold_lane<2>(snd) : fold_lane<4>(snd));
                }
                ui += hi ? k / 2 : 0;
            }
            const double t = sum_halves(p[0] + fold_lane<8>(p[0]));
            if (lane < 8 && l + ui < nl) wpart[wv][l + ui] = t;
        }
        __syncthreads();
        for (int l = tid; l < nl; l += 256)
            st_agent(partial + (int64_t)blockIdx.x * nd + l0 + l,
                     (wpart[0][l] + wpart[1][l]) + (wpart[2][l] + wpart[3][l]));
        __syncthreads();
    }
    if (!last_sums) return;
    __builtin_amdgcn_s_waitcnt(0);  // (the partials are at the coherence point before the arrival is counted)
    __syncthreads();
    if (tid == 0) last = atomicAdd(arrived, 1u) == gridDim.x - 1;
    __syncthreads();
    if (!last) return;
    if (tid == 0) *arrived = 0;
    // K threads side by side on the columns, 256 / K shares of the workgroups each
    int K = 1;
    while (K < nt && K < 256) K <<= 1;
    const int share = tid / K, nsh = 256 / K;
    for (int l0 = 0; l0 < nt; l0 += K) {
        const int l = l0 + tid % K;
        double a = 0.0;
        if (l < nt)
#pragma unroll 8
            for (int b = share; b < (int)gridDim.x; b += nsh) a += ld_agent(partial + (int64_t)b * nt + l);
        __syncthreads();
        hs[tid] = a;
        __syncthreads();
        if (tid < K && l < nt) {
            double t = 0.0;
            for (int q = 0; q < nsh; ++q) t += hs[q * K + tid];
            out[l] = t;
            if (host) __hip_atomic_store(host + nhost + l, t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    }
    if (!host) return;
    for (int q = tid; q < nhost; q += 256)
        __hip_atomic_store(host + q, all_h[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (tid == 0) __hip_atomic_store(flag, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}
// the sums of many workgroups' dots of many columns, one wave per column
__global__ __launch_bounds__(64) void k_cgs_sums(const double *__restrict__ partial, int nblk, int nd,
                                                 double *__restrict__ out) {
    const int l = blockIdx.x;
    double a = 0.0;
    for (int b = threadIdx.x; b < nblk; b += 64) a += partial[(int64_t)b * nd + l];
    a = wave_sum(a);
    if (threadIdx.x == 0) out[l] = a;
}
__global__ void k_axpby(double a, const double *__restrict__ x, double b, double *__restrict__ y, int64_t n) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        y[i] = b == 0.0 ? a * x[i] : a * x[i] + b * y[i];
}

__global__ void k_scal(double a, double *y, int64_t n) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        y[i] *= a;
}


// ------------------------------------------------------------------ kNR-wide vectors (interleaved N x kNR)
// element (t, r) at t * kNR + r; one dot product, norm or update per column r
template <typename T>
__global__ void k_gather_m(const double *__restrict__ X, int64_t ldx, int nrhs, const int32_t *__restrict__ perm,
                           int64_t N, T *__restrict__ dst) {
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < N * kNR; e += (int64_t)gridDim.x * blockDim.x) {
        const int64_t t = e / kNR;
        const int r = (int)(e % kNR);
        const int64_t src = perm ? perm[t] : t;
        dst[e] = r < nrhs ? (T)X[src + r * ldx] : T(0);
    }
}
template <typename T>
__global__ void k_scatter_m(const T *__restrict__ src, int64_t N, double *__restrict__ Y, int64_t ldy, int nrhs,
                            const int32_t *__restrict__ perm) {
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < N * kNR; e += (int64_t)gridDim.x * blockDim.x) {
        const int64_t t = e / kNR;
        const int r = (int)(e % kNR);
        if (r < nrhs) Y[(perm ? perm[t] : t) + r * ldy] = (double)src[e];
    }
}
// ---- lockstep solves: S systems x kNR columns.  A lockstep vector holds the
// systems' interleaved tree-order vectors one after another (n slots in all);
// column (s, r) is right-hand side r of system s, seg[t] the system of slot t
// (NULL: a single system).  Dot products reduce per block of slots (blk[b] =
// first and one-past-last slot, all in one system), then per system over the
// system's blocks sblk[s] .. sblk[s+1]-1.
// partial[(j * nblk + b) * kNR + r] = sum over block b of V_j(t, r) w(t, r)
__global__ __launch_bounds__(256) void k_bdot16(const double *__restrict__ V, int64_t ldv,
                                                const double *__restrict__ w, const int2 *__restrict__ blk,
                                                double *__restrict__ partial) {
    const int b = blockIdx.x, j = blockIdx.y, nblk = gridDim.x;
    const double *v = V + (int64_t)j * ldv;
    const int2 rg = blk[b];
    const int r = threadIdx.x & 15;
    double acc = 0.0;
    for (int64_t e = (int64_t)rg.x * kNR + threadIdx.x; e < (int64_t)rg.y * kNR; e += 256) acc = fma(v[e], w[e], acc);
    acc += __shfl_xor(acc, 16, 64);
    acc += __shfl_xor(acc, 32, 64);
    __shared__ double sh[4][kNR];
    if ((threadIdx.x & 63) < 16) sh[threadIdx.x >> 6][r] = acc;
    __syncthreads();
    if (threadIdx.x < 16)
        partial[((int64_t)j * nblk + b) * kNR + r] = sh[0][r] + sh[1][r] + sh[2][r] + sh[3][r];
}
// out[(j * S + s) * kNR + r] = sum over system s's blocks
__global__ __launch_bounds__(256) void k_bdot16_reduce(const double *__restrict__ partial, int nblk,
                                                       const int32_t *__restrict__ sblk, double *__restrict__ out) {
    const int j = blockIdx.x, sy = blockIdx.y, S = gridDim.y;
    const int r = threadIdx.x & 15, q = threadIdx.x >> 4;
    double acc = 0.0;
#pragma unroll 8
    for (int b = sblk[sy] + q; b < sblk[sy + 1]; b += 16) acc += partial[((int64_t)j * nblk + b) * kNR + r];
    acc += __shfl_xor(acc, 16, 64);
    acc += __shfl_xor(acc, 32, 64);
    __shared__ double sh[4][kNR];
    if ((threadIdx.x & 63) < 16) sh[threadIdx.x >> 6][r] = acc;
    __syncthreads();
    if (threadIdx.x < 16) out[((int64_t)j * S + sy) * kNR + r] = sh[0][r] + sh[1][r] + sh[2][r] + sh[3][r];
}
// w(t, r) += sign * sum_j V_j(t, r) h(j, seg(t), r)
__global__ __launch_bounds__(256) void k_bgemv16(const double *__restrict__ V, int64_t ldv, int k,
                                                 const double *__restrict__ h, int S, double sign,
                                                 double *__restrict__ w, int64_t n, const int32_t *__restrict__ seg) {
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n * kNR; e += (int64_t)gridDim.x * blockDim.x) {
        const int64_t col = (seg ? (int64_t)seg[e / kNR] * kNR : 0) + (e % kNR);
        double acc = 0.0;
        for (int l = 0; l < k; ++l) acc = fma(V[(int64_t)l * ldv + e], h[(int64_t)l * S * kNR + col], acc);
        w[e] += sign * acc;
    }
}
// A subtraction and the dot products that follow it in the Arnoldi process, in one pass over a block's slots:
// w(t, r) -= sum_{l < k} V_l(t, r) h(l, s, r), then partial as k_bdot16's for the nd columns of V, or of w with
// itself (nd = 0).  A thread's entries share one column, so its products need no exchange until the end, and it
// reads back only entries of w that it wrote.  Bound by the reads of V: 14 columns of 55000 slots take 33 us, as the
// subtraction and the dots in two launches do (17 each); without dots, for the norm, 20 us.  (The entries of 24
// columns kept in registers between the two: two waves per SIMD, 2% slower solves.)
__global__ __launch_bounds__(256) void k_bsub_dot16(const double *__restrict__ V, int64_t ldv, int k,
                                                    const double *__restrict__ h, int S, double *w, int nd,
                                                    const int2 *__restrict__ blk, const int32_t *__restrict__ seg,
                                                    double *__restrict__ partial) {
    const int b = blockIdx.x, nblk = gridDim.x;
    const int2 rg = blk[b];
    const int r = threadIdx.x & 15, wv = threadIdx.x >> 6;
    const int64_t e0 = (int64_t)rg.x * kNR + threadIdx.x, e1 = (int64_t)rg.y * kNR;
    const int64_t col = (seg ? (int64_t)seg[rg.x] * kNR : 0) + r;
    for (int64_t e = e0; e < e1; e += 1024) {
        double acc[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
        for (int l = 0; l < k; ++l) {
            const double c = h[(int64_t)l * S * kNR + col];
            const double *v = V + (int64_t)l * ldv;
#pragma unroll
            for (int u = 0; u < 4; ++u) acc[u] = fma(v[min(e + 256 * u, e1 - 1)], c, acc[u]);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (e + 256 * u < e1) w[e + 256 * u] -= acc[u];
    }
    constexpr int kG = 4, kL = 16;  // columns at a time, columns per round of LDS
    __shared__ double sh[4][kL][kNR];
    const int nt = nd > 0 ? nd : 1;
    for (int j0 = 0; j0 < nt; j0 += kL) {
        for (int j1 = j0; j1 < min(j0 + kL, nt); j1 += kG) {
            double acc[kG] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
            for (int64_t e = e0; e < e1; e += 256) {
                const double x = w[e];
#pragma unroll
                for (int u = 0; u < kG; ++u)
                    acc[u] = fma(nd > 0 ? V[(int64_t)min(j1 + u, nd - 1) * ldv + e] : x, x, acc[u]);
            }
#pragma unroll
            for (int u = 0; u < kG; ++u) {
                acc[u] += __shfl_xor(acc[u], 16, 64);
                acc[u] += __shfl_xor(acc[u], 32, 64);
                if ((threadIdx.x & 63) < 16) sh[wv][j1 - j0 + u][r] = acc[u];
            }
        }
        __syncthreads();
        for (int q = threadIdx.x; q < min(kL, nt - j0) * kNR; q += 256) {
            const int j = q / kNR, c = q % kNR;
            partial[((int64_t)(j0 + j) * nblk + b) * kNR + c] = sh[0][j][c] + sh[1][j][c] + sh[2][j][c] + sh[3][j][c];
        }
        __syncthreads();
    }
}
// A space shared by every column of a one-system lockstep vector (the deflation space): k vectors
// of n slots, stored row-major (Cs[t * k + q]), so that the k values of a slot are contiguous.
// Both products with it are tall-skinny GEMMs and run on the FP64 matrix cores (16x16x4 MFMA:
// lane l supplies A(l % 16, l / 16) and B(l / 16, l % 16) and holds D(l / 16 + 4 v, l % 16), v < 4).
//
// partial[(q * nblk + b) * kNR + r] = sum over block b's slots of Cs(t, q) w(t, r), for the
// kSdTiles 16-vector tiles q = qg .. qg + 16 kSdTiles - 1 of this workgroup (grid.y covers k):
// D(16 q x 16 r) += A(16 q x 4 t) B(4 t x 16 r) with A(m, j) = Cs(t0 + j, q0 + m), B(j, n) = w(t0 + j, n);
// the four waves take every fourth group of 4 slots and are summed through LDS (the reduction over
// blocks is k_bdot16_reduce's).
constexpr int kSdTiles = 8;
__global__ __launch_bounds__(256) void k_sdot16(const double *__restrict__ Cs, int k, const double *__restrict__ w,
                                                const int2 *__restrict__ blk, double *__restrict__ partial) {
    typedef double v4 __attribute__((ext_vector_type(4)));
    const int b = blockIdx.x, nblk = gridDim.x;
    const int qg = blockIdx.y * 16 * kSdTiles;
    const int nz = min(kSdTiles, (k - qg + 15) / 16);
    const int2 rg = blk[b];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int m = lane & 15, j = lane >> 4;
    v4 acc[kSdTiles];
#pragma unroll
    for (int z = 0; z < kSdTiles; ++z) acc[z] = (v4)0.0;
#pragma unroll 2
    for (int t0 = rg.x + 4 * wv; t0 < rg.y; t0 += 16) {
        const int t = t0 + j;
        const bool ok = t < rg.y;
        const double bv = ok ? w[(int64_t)t * kNR + m] : 0.0;
        const double *c = Cs + (int64_t)t * k + qg + m;
        double av[kSdTiles];
#pragma unroll
        for (int z = 0; z < kSdTiles; ++z) av[z] = (z < nz && ok && qg + 16 * z + m < k) ? c[16 * z] : 0.0;
#pragma unroll
        for (int z = 0; z < kSdTiles; ++z)
            if (z < nz) acc[z] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[z], bv, acc[z], 0, 0, 0);
    }
    // waves 2, 3 -> waves 0, 1 -> wave 0
    __shared__ double sh[2][kSdTiles][4][64];
    if (wv >= 2)
#pragma unroll
        for (int z = 0; z < kSdTiles; ++z)
#pragma unroll
            for (int v = 0; v < 4; ++v) sh[wv - 2][z][v][lane] = acc[z][v];
    __syncthreads();
    if (wv < 2)
#pragma unroll
        for (int z = 0; z < kSdTiles; ++z)
#pragma unroll
            for (int v = 0; v < 4; ++v) acc[z][v] += sh[wv][z][v][lane];
    __syncthreads();
    if (wv == 1)
#pragma unroll
        for (int z = 0; z < kSdTiles; ++z)
#pragma unroll
            for (int v = 0; v < 4; ++v) sh[0][z][v][lane] = acc[z][v];
    __syncthreads();
    if (wv == 0)
#pragma unroll
        for (int z = 0; z < kSdTiles; ++z)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int q = qg + 16 * z + j + 4 * v;
                if (z < nz && q < k) partial[((int64_t)q * nblk + b) * kNR + m] = acc[z][v] + sh[0][z][v][lane];
            }
}
// w(t, r) += sign * sum_q Cs(t, q) h(q, seg(t), r)   (the shared space, row-major as above; with several
// systems every system's slots carry its own space, h holds the coefficients of every system).
// A wave takes 64 slots, four tiles of 16: D_i(16 t x 16 r) += A_i(16 t x 4 q) B(4 q x 16 r) with
// A_i(m, j) = Cs(t0 + 16 i + m, q), B(j, n) = h(q, s, n), q = q0 + j, one B load serving the four tiles;
// 16 vectors per trip, their 20 loads issued before the 16 MFMAs.  Slots of several systems in one
// group of 64 are taken once per system with the other systems' rows zeroed.
__global__ __launch_bounds__(256) void k_supd16(const double *__restrict__ Cs, int k, const double *__restrict__ h,
                                                int S, double sign, double *__restrict__ w, int64_t n,
                                                const int32_t *__restrict__ seg) {
    typedef double v4 __attribute__((ext_vector_type(4)));
    const int lane = threadIdx.x & 63;
    const int m = lane & 15, j = lane >> 4;
    const int64_t ngrp = (n + 63) / 64;
    for (int64_t g = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); g < ngrp; g += (int64_t)gridDim.x * 4) {
        const int64_t t0 = g * 64;
        const int s_lo = seg ? seg[t0] : 0;
        const int s_hi = seg ? seg[min(t0 + 63, n - 1)] : 0;
        const double *c[4];
        bool rok[4];
        int s_row[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int64_t ta = t0 + 16 * i + m;  // this lane's A row of tile i
            rok[i] = ta < n;
            s_row[i] = seg && rok[i] ? seg[ta] : 0;
            c[i] = Cs + (rok[i] ? ta : 0) * k;
        }
        v4 acc[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] = (v4)0.0;
        for (int sy = s_lo; sy <= s_hi; ++sy) {
            const double *hq = h + (int64_t)sy * kNR + m;
            const int64_t hs = (int64_t)S * kNR;
            bool mine[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) mine[i] = rok[i] && s_row[i] == sy;
            for (int q0 = 0; q0 < k; q0 += 16) {
                double av[4][4], bv[4];
                // (a tile's four loads read the same 16 lines: issued one after another)
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        const int q = q0 + 4 * u + j;
                        av[i][u] = (mine[i] && q < k) ? c[i][q] : 0.0;
                    }
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int q = q0 + 4 * u + j;
                    bv[u] = q < k ? hq[q * hs] : 0.0;
                }
#pragma unroll
                for (int u = 0; u < 4; ++u)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        acc[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[i][u], bv[u], acc[i], 0, 0, 0);
            }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int64_t t = t0 + 16 * i + j + 4 * v;
                if (t < n) w[t * kNR + m] += sign * acc[i][v];
            }
    }
}
// dst[t * k + q] = src[q * n + t]: k column-major vectors of n entries to row-major
__global__ void k_to_rowmajor(const double *__restrict__ src, int64_t n, int k, double *__restrict__ dst) {
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n * k; e += (int64_t)gridDim.x * blockDim.x)
        dst[e] = src[(e % k) * n + e / k];
}

// dst(t, r) = sc(seg(t), r) * src(t, r), or with norm2 that over sqrt(norm2(seg(t), r)), zero where either is zero
__global__ void k_bscale16(const double *__restrict__ src, const double *__restrict__ sc,
                           const double *__restrict__ norm2, double *dst, int64_t n, const int32_t *__restrict__ seg) {
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n * kNR; e += (int64_t)gridDim.x * blockDim.x) {
        const int64_t c = (seg ? (int64_t)seg[e / kNR] * kNR : 0) + (e % kNR);
        double f = sc[c];
        if (norm2) f = f != 0.0 && norm2[c] > 0.0 ? f / sqrt(norm2[c]) : 0.0;
        dst[e] = f * src[e];
    }
}


// batch vector pool <-> lockstep vectors: lockstep slot t lives at pool slot map[t]
template <typename T>
__global__ void k_map_in(const double *__restrict__ X, const int32_t *__restrict__ map, int64_t n, T *__restrict__ pool) {
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n * kNR; e += (int64_t)gridDim.x * blockDim.x)
        pool[(int64_t)map[e / kNR] * kNR + e % kNR] = (T)X[e];
}
template <typename T>
__global__ void k_map_out(const T *__restrict__ pool, const int32_t *__restrict__ map, int64_t n, double *__restrict__ Y) {
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n * kNR; e += (int64_t)gridDim.x * blockDim.x)
        Y[e] = (double)pool[(int64_t)map[e / kNR] * kNR + e % kNR];
}
// column-major caller blocks <-> lockstep vectors: lockstep slot t reads row src[t] of a block with
// leading dimension ld[t] (per-system blocks concatenated), columns r < nrhs
__global__ void k_gather_b(const double *__restrict__ X, const int64_t *__restrict__ src, const int32_t *__restrict__ ld,
                           int nrhs, int64_t n, double *__restrict__ dst) {
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n * kNR; e += (int64_t)gridDim.x * blockDim.x) {
        const int64_t t = e / kNR;
        const int r = (int)(e % kNR);
        dst[e] = r < nrhs ? X[src[t] + (int64_t)r * ld[t]] : 0.0;
    }
}
__global__ void k_scatter_b(const double *__restrict__ src_v, const int64_t *__restrict__ src,
                            const int32_t *__restrict__ ld, int nrhs, int64_t n, double *__restrict__ Y) {
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n * kNR; e += (int64_t)gridDim.x * blockDim.x) {
        const int64_t t = e / kNR;
        const int r = (int)(e % kNR);
        if (r < nrhs) Y[src[t] + (int64_t)r * ld[t]] = src_v[e];
    }
}


// ------------------------------------------------------------------ rank predictor
// A 16-64-64-64-1 perceptron with GELU (erf form) activations predicting
// log2(1 + rank) of an ACA block from its geometry features.  BF16 parameters
// (expanded to FP32 in LDS), FP32 accumulation, one thread per block.
// Parameter layout: W1 (F x H, row-major: input-major), b1, W2 (H x H), b2,
// W3 (H x H), b3, w4 (H), b4.
constexpr int kRF = 16, kRH = 64;
constexpr int kRP = kRF * kRH + kRH + 2 * (kRH * kRH + kRH) + kRH + 1;
__device__ __forceinline__ float bf16_f32(uint16_t v) { return __uint_as_float((uint32_t)v << 16); }
__device__ __forceinline__ float gelu_erf(float x) { return 0.5f * x * (1.0f + erff(x * 0.70710678118654752f)); }

__global__ __launch_bounds__(256) void k_rank_mlp(const float *__restrict__ feat, int n,
                                                  const uint16_t *__restrict__ w, float *__restrict__ out) {
    __shared__ float sw[kRP];
    for (int q = threadIdx.x; q < kRP; q += blockDim.x) sw[q] = bf16_f32(w[q]);
    __syncthreads();
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float *W1 = sw, *b1 = W1 + kRF * kRH, *W2 = b1 + kRH, *b2 = W2 + kRH * kRH, *W3 = b2 + kRH;
    const float *b3 = W3 + kRH * kRH, *w4 = b3 + kRH, *b4 = w4 + kRH;
    float x[kRF], h1[kRH], h2[kRH];
#pragma unroll
    for (int f = 0; f < kRF; ++f) x[f] = feat[(int64_t)i * kRF + f];
#pragma unroll
    for (int o = 0; o < kRH; ++o) {
        float a = b1[o];
#pragma unroll
        for (int f = 0; f < kRF; ++f) a = fmaf(x[f], W1[f * kRH + o], a);
        h1[o] = gelu_erf(a);
    }
#pragma unroll
    for (int o = 0; o < kRH; ++o) {
        float a = b2[o];
#pragma unroll
        for (int k = 0; k < kRH; ++k) a = fmaf(h1[k], W2[k * kRH + o], a);
        h2[o] = gelu_erf(a);
    }
#pragma unroll
    for (int o = 0; o < kRH; ++o) {
        float a = b3[o];
#pragma unroll
        for (int k = 0; k < kRH; ++k) a = fmaf(h2[k], W3[k * kRH + o], a);
        h1[o] = gelu_erf(a);
    }
    float y = b4[0];
#pragma unroll
    for (int k = 0; k < kRH; ++k) y = fmaf(h1[k], w4[k], y);
    out[i] = y;
}

inline int grid_for(int64_t n, int nt = 256, int cap = 8192) {
    int64_t g = (n + nt - 1) / nt;
    if (g < 1) g = 1;
    if (g > cap) g = cap;
    return (int)g;
}

}  // namespace

// ------------------------------------------------------------------ launch wrappers
void launch_lr_extract(const LrJob *jobs, int njobs, const double *ws, const int64_t *tab, const int32_t *rowpiv,
                       const int32_t *colpiv, double *out, hipStream_t s) {
    if (njobs > 0)
        hipLaunchKernelGGL(k_lr_extract, dim3(njobs), dim3(256), 0, s, jobs, ws, tab, rowpiv, colpiv, out);
}
void launch_lr_form(const LrFormJob *jobs, int njobs, const int32_t *idx, double *out, KParams kp, hipStream_t s) {
    if (njobs > 0) hipLaunchKernelGGL(k_lr_form, dim3(njobs), dim3(1024), 0, s, jobs, idx, out, kp);
}
void launch_pack_pivots(const LrJob *jobs, int njobs, const int32_t *rowpiv, const int32_t *colpiv, const double *hist,
                        int32_t *prow, int32_t *pcol, double *phist, hipStream_t s) {
    if (njobs > 0)
        hipLaunchKernelGGL(k_pack_pivots, dim3(njobs), dim3(64), 0, s, jobs, rowpiv, colpiv, hist, prow, pcol, phist);
}
void launch_slot_points(const int32_t *pid, int64_t n, const double *px, const double *py, const double *pz, double *xd,
                        double *yd, double *zd, float *x, float *y, float *z, float *xl, float *yl, float *zl,
                        hipStream_t s) {
    if (n > 0)
        hipLaunchKernelGGL(k_slot_points, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, pid, n, px, py, pz, xd, yd,
                           zd, x, y, z, xl, yl, zl);
}
void launch_eval(const EvalJob *jobs, int njobs, const int32_t *idx, double *A, KParams kp, hipStream_t s) {
    if (njobs > 0) hipLaunchKernelGGL(k_eval, dim3(njobs), dim3(256), 0, s, jobs, idx, A, kp);
}
void launch_xfer(const XferJob *jobs, int njobs, const int32_t *idx, const double *lr, double *A, KParams kp,
                 hipStream_t s) {
    if (njobs > 0) hipLaunchKernelGGL(k_xfer, dim3(njobs), dim3(64), 0, s, jobs, idx, lr, A, kp);
}
void launch_cur(const CurJob *jobs, int njobs, const int32_t *idx, const double *lr, double *A, KParams kp,
                hipStream_t s) {
    if (njobs > 0) hipLaunchKernelGGL(k_cur, dim3(njobs), dim3(64), 0, s, jobs, idx, lr, A, kp);
}
template <typename T, int ROLE>
static void launch_bgemv_r(const GItem *items, int nitems, const GTerm *terms, const T *A0, const T *A1, T *vec,
                           int unr, bool per_wave, hipStream_t s) {
    constexpr int VEC = sizeof(T) == 8 ? 2 : 4;
    auto go = [&](auto U) {
        constexpr int UNR = decltype(U)::value;
        if (per_wave)
            hipLaunchKernelGGL((k_bgemv<T, VEC, ROLE, UNR, 1>), dim3((nitems + 3) / 4), dim3(256), 0, s, items, nitems,
                               terms, A0, A1, vec);
        else
            hipLaunchKernelGGL((k_bgemv<T, VEC, ROLE, UNR, 4>), dim3(nitems), dim3(256), 0, s, items, nitems, terms, A0,
                               A1, vec);
    };
    if (unr <= 2) go(std::integral_constant<int, 2>{});
    else if (unr >= 8) go(std::integral_constant<int, 8>{});
    else go(std::integral_constant<int, 4>{});
}
template <typename T>
static void launch_bgemv_t(const GItem *items, int nitems, const GTerm *terms, const T *A0, const T *A1, T *vec,
                           int role, int unr, bool per_wave, hipStream_t s) {
    if (nitems <= 0) return;
    if (!A1) A1 = A0;
    if (role == 1) launch_bgemv_r<T, 1>(items, nitems, terms, A0, A1, vec, unr, per_wave, s);
    else if (role == 2) launch_bgemv_r<T, 2>(items, nitems, terms, A0, A1, vec, unr, per_wave, s);
    else launch_bgemv_r<T, 0>(items, nitems, terms, A0, A1, vec, unr, per_wave, s);
}
void launch_compose(const ComposeJob *jobs, int njobs, double *A, double *lo, int64_t lo0, unsigned long long *most,
                    hipStream_t s) {
    if (njobs > 0) hipLaunchKernelGGL(k_compose, dim3(njobs), dim3(256), 0, s, jobs, A, lo, lo0, most);
}
void launch_copy32(const CopyJob *jobs, int njobs, const float *src, float *dst, hipStream_t s) {
    if (njobs > 0) hipLaunchKernelGGL(k_copy32, dim3(njobs), dim3(256), 0, s, jobs, src, dst);
}
void launch_bgemv64(const GItem *items, int nitems, const GTerm *terms, const double *A0, const double *A1,
                    double *vec, int role, int unr, bool per_wave, hipStream_t s) {
    launch_bgemv_t<double>(items, nitems, terms, A0, A1, vec, role, unr, per_wave, s);
}
void launch_bgemv32(const GItem *items, int nitems, const GTerm *terms, const float *A0, const float *A1,
                    float *vec, int role, int unr, bool per_wave, hipStream_t s) {
    launch_bgemv_t<float>(items, nitems, terms, A0, A1, vec, role, unr, per_wave, s);
}
template <typename T>
static void launch_otf_t(const GItem *items, int nitems, const GTerm *terms, Coords<T> C, const SlotPoints &sp, T *vec,
                         hipStream_t s) {
    if (nitems <= 0) return;
    const T diag = (T)sp.diag;
    const int key = sp.dim * 2 + (sp.choice != 0);
#define H2W_OTF(D, CH) \
    hipLaunchKernelGGL((k_otf<T, D, CH>), dim3(nitems), dim3(256), 0, s, items, terms, C, sp.pid, diag, vec)
    switch (key) {
        case 2: H2W_OTF(1, 0); break;
        case 3: H2W_OTF(1, 1); break;
        case 4: H2W_OTF(2, 0); break;
        case 5: H2W_OTF(2, 1); break;
        case 6: H2W_OTF(3, 0); break;
        default: H2W_OTF(3, 1); break;
    }
#undef H2W_OTF
}
void launch_otf32(const GItem *items, int nitems, const GTerm *terms, SlotPoints sp, float *vec, hipStream_t s) {
    launch_otf_t<float>(items, nitems, terms, Coords<float>{sp.x, sp.y, sp.z, sp.xl, sp.yl, sp.zl}, sp, vec, s);
}
void launch_otf64(const GItem *items, int nitems, const GTerm *terms, SlotPoints sp, double *vec, hipStream_t s) {
    launch_otf_t<double>(items, nitems, terms, Coords<double>{sp.xd, sp.yd, sp.zd, nullptr, nullptr, nullptr}, sp,
                         vec, s);
}
void launch_to_fp32(const double *a, float *b, int64_t n, hipStream_t s) {
    if (n > 0) hipLaunchKernelGGL(k_to_fp32, dim3(grid_for(n)), dim3(256), 0, s, a, b, n);
}
void launch_to_fp64(const float *a, double *b, int64_t n, hipStream_t s) {
    if (n > 0) hipLaunchKernelGGL(k_to_fp64, dim3(grid_for(n)), dim3(256), 0, s, a, b, n);
}
int64_t stream_chunk_bytes() { return (int64_t)kStreamUnr * 256 * 16; }
void launch_stream_read(const void *p, int64_t bytes, uint32_t *out, int grid, hipStream_t s) {
    hipLaunchKernelGGL(k_stream_read, dim3(grid), dim3(256), 0, s, (const Word16 *)p, bytes / stream_chunk_bytes(), out);
}
void launch_fill(double *a, int64_t n, double v, hipStream_t s) {
    if (n > 0) hipLaunchKernelGGL(k_fill<double>, dim3(grid_for(n)), dim3(256), 0, s, a, n, v);
}
void launch_fill32(float *a, int64_t n, float v, hipStream_t s) {
    if (n > 0) hipLaunchKernelGGL(k_fill<float>, dim3(grid_for(n)), dim3(256), 0, s, a, n, v);
}
void launch_begin64(const double *x, double scale, const double *norm2, double *copy, const int32_t *perm, double *px,
                    int64_t N, double *py, int64_t len, hipStream_t s) {
    hipLaunchKernelGGL(k_begin<double>, dim3(grid_for(std::max(N, len), 256, 2048)), dim3(256), 0, s, x, scale, norm2, copy,
                       perm, px, N, py, len);
}
void launch_begin32(const double *x, double scale, const double *norm2, double *copy, const int32_t *perm, float *px,
                    int64_t N, float *py, int64_t len, hipStream_t s) {
    hipLaunchKernelGGL(k_begin<float>, dim3(grid_for(std::max(N, len), 256, 2048)), dim3(256), 0, s, x, scale, norm2, copy,
                       perm, px, N, py, len);
}
void launch_permute_in(const double *x, int64_t ldx, double *xt, int64_t ldt, const int32_t *perm, int64_t N,
                       int nrhs, hipStream_t s) {
    hipLaunchKernelGGL(k_permute_in<double>, dim3(grid_for(N, 256, 2048), nrhs), dim3(256), 0, s, x, ldx, xt, ldt,
                       perm, N);
}
void launch_permute_out(const double *yt, int64_t ldt, double *y, int64_t ldy, const int32_t *perm, int64_t N,
                        int nrhs, hipStream_t s) {
    hipLaunchKernelGGL(k_permute_out<double>, dim3(grid_for(N, 256, 2048), nrhs), dim3(256), 0, s, yt, ldt, y, ldy,
                       perm, N);
}
void launch_permute_out32(const float *yt, int64_t ldt, double *y, int64_t ldy, const int32_t *perm, int64_t N,
                          int nrhs, hipStream_t s) {
    hipLaunchKernelGGL(k_permute_out<float>, dim3(grid_for(N, 256, 2048), nrhs), dim3(256), 0, s, yt, ldt, y, ldy,
                       perm, N);
}
void launch_dense_rows(const int32_t *rows, int64_t nrows, const double *xt, double *y, int64_t N, KParams kp,
                       hipStream_t s) {
    if (nrows > 0)
        hipLaunchKernelGGL(k_dense_rows, dim3((unsigned)((nrows + 63) / 64)), dim3(256), 0, s, rows, nrows, xt, y, N,
                           kp);
}
// rows per thread: up to 256 workgroups, whose dots one workgroup still sums in a few microseconds
static int cgs_rows(int64_t n) { return n <= 131072 ? 2 : n <= 262144 ? 4 : 8; }
int cgs_blocks(int64_t n) { return (int)((n + 256 * cgs_rows(n) - 1) / (256 * cgs_rows(n))); }
void launch_cgs(const CgsArgs &a, hipStream_t s) {
    const int nb = cgs_blocks(a.n), nt = a.norm ? 1 : a.nd;
    if (nt <= 0) return;
    // the last workgroup's share: nb nt numbers from one compute unit, 2 us up to about 16384 of them
    const int last = a.norm || a.host || (int64_t)nb * nt <= 16384;
    auto go = [&](auto R, const auto *src) {
        hipLaunchKernelGGL((k_cgs<decltype(R)::value, std::decay_t<decltype(*src)>>), dim3(nb), dim3(256), 0, s, a.V,
                           a.ldv, src, a.w, a.n, a.s0, a.ns, a.sub, a.d0, a.nd, a.norm, a.partial, a.arrived, a.out,
                           last, a.all_h, a.nhost, a.host, a.flag, a.seq);
    };
    auto rows = [&](const auto *src) {
        switch (cgs_rows(a.n)) {
        case 2: go(std::integral_constant<int, 2>{}, src); break;
        case 4: go(std::integral_constant<int, 4>{}, src); break;
        default: go(std::integral_constant<int, 8>{}, src);
        }
    };
    if (a.src32) rows(a.src32);
    else rows((const double *)nullptr);
    if (!last) hipLaunchKernelGGL(k_cgs_sums, dim3(nt), dim3(64), 0, s, a.partial, nb, nt, a.out);
}
void launch_vec_update(const double *V, int64_t ldv, int k, const double *c, double *x, int64_t n, hipStream_t s) {
    if (k > 0) hipLaunchKernelGGL(k_mgemv, dim3(grid_for(n, 256, 4096)), dim3(256), 0, s, V, ldv, k, c, x, n, 1.0);
}
void launch_axpby(double a, const double *x, double b, double *y, int64_t n, hipStream_t s) {
    hipLaunchKernelGGL(k_axpby, dim3(grid_for(n)), dim3(256), 0, s, a, x, b, y, n);
}
void launch_scal(double a, double *y, int64_t n, hipStream_t s) {
    hipLaunchKernelGGL(k_scal, dim3(grid_for(n)), dim3(256), 0, s, a, y, n);
}


template <typename T, int ROLE>
static void launch_bgemm_r(const GItem *items, int nitems, const GTerm *terms, const T *A0, const T *A1,
                           const T *const *tab, T *vec, bool per_wave, hipStream_t s) {
    constexpr int np = kRowTile / kPassRows<T>;
    if (per_wave)
        hipLaunchKernelGGL((k_bgemm<T, ROLE, 1>), dim3((nitems + 3) / 4, np), dim3(256), 0, s, items, nitems, terms, A0, A1,
                           tab, vec);
    else
        hipLaunchKernelGGL((k_bgemm<T, ROLE, 4>), dim3(nitems, np), dim3(256), 0, s, items, nitems, terms, A0, A1, tab,
                           vec);
}
template <typename T>
static void launch_bgemm_t(const GItem *items, int nitems, const GTerm *terms, const T *A0, const T *A1,
                           const T *const *tab, T *vec, int role, bool per_wave, hipStream_t s) {
    if (nitems <= 0) return;
    if (!A1) A1 = A0;
    if (role == 1) launch_bgemm_r<T, 1>(items, nitems, terms, A0, A1, tab, vec, per_wave, s);
    else if (role == 2) launch_bgemm_r<T, 2>(items, nitems, terms, A0, A1, tab, vec, per_wave, s);
    else launch_bgemm_r<T, 0>(items, nitems, terms, A0, A1, tab, vec, per_wave, s);
}
void launch_bgemm64(const GItem *items, int nitems, const GTerm *terms, const double *A0, const double *A1,
                    double *vec, int role, bool per_wave, hipStream_t s) {
    launch_bgemm_t<double>(items, nitems, terms, A0, A1, nullptr, vec, role, per_wave, s);
}
void launch_bgemm32(const GItem *items, int nitems, const GTerm *terms, const float *A0, const float *A1, float *vec,
                    int role, bool per_wave, hipStream_t s) {
    launch_bgemm_t<float>(items, nitems, terms, A0, A1, nullptr, vec, role, per_wave, s);
}
void launch_bgemm64_tab(const GItem *items, int nitems, const GTerm *terms, const double *const *tab, double *vec,
                        int role, bool per_wave, hipStream_t s) {
    launch_bgemm_t<double>(items, nitems, terms, nullptr, nullptr, tab, vec, role, per_wave, s);
}
void launch_bgemm32_tab(const GItem *items, int nitems, const GTerm *terms, const float *const *tab, float *vec,
                        int role, bool per_wave, hipStream_t s) {
    launch_bgemm_t<float>(items, nitems, terms, nullptr, nullptr, tab, vec, role, per_wave, s);
}
void launch_gather_m64(const double *X, int64_t ldx, int nrhs, const int32_t *perm, int64_t N, double *dst,
                       hipStream_t s) {
    hipLaunchKernelGGL(k_gather_m<double>, dim3(grid_for(N * kNR)), dim3(256), 0, s, X, ldx, nrhs, perm, N, dst);
}
void launch_gather_m32(const double *X, int64_t ldx, int nrhs, const int32_t *perm, int64_t N, float *dst,
                       hipStream_t s) {
    hipLaunchKernelGGL(k_gather_m<float>, dim3(grid_for(N * kNR)), dim3(256), 0, s, X, ldx, nrhs, perm, N, dst);
}
void launch_scatter_m64(const double *src, int64_t N, double *Y, int64_t ldy, int nrhs, const int32_t *perm,
                        hipStream_t s) {
    hipLaunchKernelGGL(k_scatter_m<double>, dim3(grid_for(N * kNR)), dim3(256), 0, s, src, N, Y, ldy, nrhs, perm);
}
void launch_scatter_m32(const float *src, int64_t N, double *Y, int64_t ldy, int nrhs, const int32_t *perm,
                        hipStream_t s) {
    hipLaunchKernelGGL(k_scatter_m<float>, dim3(grid_for(N * kNR)), dim3(256), 0, s, src, N, Y, ldy, nrhs, perm);
}
void launch_bdot16(const double *V, int64_t ldv, int k, const double *w, const int2 *blk, int nblk, double *partial,
                   hipStream_t s) {
    if (k > 0) hipLaunchKernelGGL(k_bdot16, dim3(nblk, k), dim3(256), 0, s, V, ldv, w, blk, partial);
}
void launch_bdot16_reduce(const double *partial, int nblk, int k, const int32_t *sblk, int S, double *out,
                          hipStream_t s) {
    if (k > 0) hipLaunchKernelGGL(k_bdot16_reduce, dim3(k, S), dim3(256), 0, s, partial, nblk, sblk, out);
}
void launch_bgemv16(const double *V, int64_t ldv, int k, const double *h, int S, double sign, double *w, int64_t n,
                    const int32_t *seg, hipStream_t s) {
    if (k > 0)
        hipLaunchKernelGGL(k_bgemv16, dim3(grid_for(n * kNR, 256, 4096)), dim3(256), 0, s, V, ldv, k, h, S, sign, w, n,
                           seg);
}
void launch_sdot16(const double *Cs, int k, const double *w, const int2 *blk, int nblk, double *partial, hipStream_t s) {
    if (k > 0)
        hipLaunchKernelGGL(k_sdot16, dim3(nblk, (k + 16 * kSdTiles - 1) / (16 * kSdTiles)), dim3(256), 0, s, Cs, k, w, blk,
                           partial);
}
void launch_supd16(const double *Cs, int k, const double *h, int S, double sign, double *w, int64_t n,
                   const int32_t *seg, hipStream_t s) {
    if (k > 0 && n > 0)
        hipLaunchKernelGGL(k_supd16, dim3((unsigned)std::min<int64_t>((n + 255) / 256, 8192)), dim3(256), 0, s, Cs, k, h, S,
                           sign, w, n, seg);
}
void launch_to_rowmajor(const double *src, int64_t n, int k, double *dst, hipStream_t s) {
    if (k > 0) hipLaunchKernelGGL(k_to_rowmajor, dim3(grid_for(n * k, 256, 4096)), dim3(256), 0, s, src, n, k, dst);
}
void launch_bsub_dot16(const double *V, int64_t ldv, int k, const double *h, int S, double *w, int nd, const int2 *blk,
                       int nblk, const int32_t *seg, double *partial, hipStream_t s) {
    hipLaunchKernelGGL(k_bsub_dot16, dim3(nblk), dim3(256), 0, s, V, ldv, k, h, S, w, nd, blk, seg, partial);
}
void launch_bscale16(const double *src, const double *sc, const double *norm2, double *dst, int64_t n,
                     const int32_t *seg, hipStream_t s) {
    hipLaunchKernelGGL(k_bscale16, dim3(grid_for(n * kNR)), dim3(256), 0, s, src, sc, norm2, dst, n, seg);
}
void launch_map_in64(const double *X, const int32_t *map, int64_t n, double *pool, hipStream_t s) {
    hipLaunchKernelGGL(k_map_in<double>, dim3(grid_for(n * kNR)), dim3(256), 0, s, X, map, n, pool);
}
void launch_map_in32(const double *X, const int32_t *map, int64_t n, float *pool, hipStream_t s) {
    hipLaunchKernelGGL(k_map_in<float>, dim3(grid_for(n * kNR)), dim3(256), 0, s, X, map, n, pool);
}
void launch_map_out64(const double *pool, const int32_t *map, int64_t n, double *Y, hipStream_t s) {
    hipLaunchKernelGGL(k_map_out<double>, dim3(grid_for(n * kNR)), dim3(256), 0, s, pool, map, n, Y);
}
void launch_map_out32(const float *pool, const int32_t *map, int64_t n, double *Y, hipStream_t s) {
    hipLaunchKernelGGL(k_map_out<float>, dim3(grid_for(n * kNR)), dim3(256), 0, s, pool, map, n, Y);
}
void launch_gather_b(const double *X, const int64_t *src, const int32_t *ld, int nrhs, int64_t n, double *dst,
                     hipStream_t s) {
    hipLaunchKernelGGL(k_gather_b, dim3(grid_for(n * kNR)), dim3(256), 0, s, X, src, ld, nrhs, n, dst);
}
void launch_scatter_b(const double *v, const int64_t *src, const int32_t *ld, int nrhs, int64_t n, double *Y,
                      hipStream_t s) {
    hipLaunchKernelGGL(k_scatter_b, dim3(grid_for(n * kNR)), dim3(256), 0, s, v, src, ld, nrhs, n, Y);
}
void launch_rank_mlp(const float *feat, int n, const uint16_t *w, float *out, hipStream_t s) {
    if (n > 0) hipLaunchKernelGGL(k_rank_mlp, dim3((n + 255) / 256), dim3(256), 0, s, feat, n, w, out);
}
void launch_aca_small(const AcaJob *jobs, int njobs, const int32_t *idx, double *ws, int64_t ws_cap,
                      unsigned long long *ws_top, int64_t *tab, uint8_t *flags, int32_t *rank, int32_t *status,
                      int32_t *rowpiv, int32_t *colpiv, KParams kp, double tol, double *hist, hipStream_t s) {
    if (njobs > 0)
        hipLaunchKernelGGL(k_aca_small, dim3(njobs), dim3(256), 0, s, jobs, idx, ws, ws_cap, ws_top, tab, flags, rank,
                           status, rowpiv, colpiv, kp, tol, hist);
}
void launch_wide_init(const AcaJob *jobs, const WideBlk *blk, int nb, WideState *state, uint8_t *flags, int64_t *tab,
                      unsigned long long *ws_top, int64_t ws_cap, hipStream_t s) {
    hipLaunchKernelGGL(k_wide_init, dim3(nb), dim3(256), 0, s, jobs, blk, state, flags, tab, ws_top, ws_cap);
}
int wide_tile() { return kWideTile; }
void launch_wide_step(const AcaJob *jobs, const WideArgs &w, const int32_t *idx, double *ws, int64_t *tab,
                      uint8_t *flags, WideState *state, int32_t *rowpiv, int32_t *colpiv, double *hist,
                      unsigned long long *ws_top, int64_t ws_cap, KParams kp, double tol, hipStream_t s) {
    hipLaunchKernelGGL(k_wide_pass<0>, dim3(w.nrow), dim3(256), 0, s, jobs, w.blk, w.tiles, idx, ws, ws, tab, flags,
                       state, w.part, w.pdot, w.arrived, rowpiv, colpiv, hist, ws_top, ws_cap, kp, tol);
    hipLaunchKernelGGL(k_wide_pass<1>, dim3(w.ncol), dim3(256), 0, s, jobs, w.blk, w.tiles + w.nrow, idx, ws, ws, tab,
                       flags, state, w.part, w.pdot, w.arrived, rowpiv, colpiv, hist, ws_top, ws_cap, kp, tol);
}
void launch_wide_finish(const WideState *state, int nb, int32_t *rank_out, int32_t *status_out, int32_t *ndone,
                        hipStream_t s) {
    hipLaunchKernelGGL(k_wide_finish, dim3(1), dim3(64), 0, s, state, nb, rank_out, status_out, ndone);
}
void launch_wide_gram(const GramJob *gj, int njobs, const AcaJob *jobs, const WideState *state, const double *ws,
                      const int64_t *tab, double *prod, hipStream_t s) {
    if (njobs > 0) hipLaunchKernelGGL(k_wide_gram, dim3(njobs), dim3(256), 0, s, gj, jobs, state, ws, tab, prod);
}
void launch_wide_judge(const AcaJob *jobs, const WideBlk *blk, int nb, WideState *state, const int32_t *final_rank,
                       const double *normS_in, int64_t *tab, unsigned long long *ws_top, int64_t ws_cap, hipStream_t s) {
    if (nb > 0)
        hipLaunchKernelGGL(k_wide_judge, dim3((nb + 63) / 64), dim3(64), 0, s, jobs, blk, nb, state, final_rank, normS_in,
                           tab, ws_top, ws_cap);
}
void launch_aca_sample(const AcaJob *jobs, int nb, const int32_t *rank, const int32_t *idx, const double *ws,
                       const int64_t *tab, KParams kp, int ns, double *err2, double *ref2, hipStream_t s) {
    if (nb > 0) hipLaunchKernelGGL(k_aca_sample, dim3(nb), dim3(64), 0, s, jobs, rank, idx, ws, tab, kp, ns, err2, ref2);
}
template <typename T>
static void launch_bgemm_tl(const GItem *items, int nitems, const GTerm *terms, const T *A0, const T *A1,
                            const T *const *tab, T *vec, int narrow, hipStream_t s) {
    if (nitems <= 0) return;
    if (narrow)
        hipLaunchKernelGGL((k_bgemm_tl<T, 4>), dim3(nitems), dim3(256), 0, s, items, terms, A0, A1 ? A1 : A0, tab, vec);
    else
        hipLaunchKernelGGL((k_bgemm_tl<T, 16>), dim3(nitems), dim3(256), 0, s, items, terms, A0, A1 ? A1 : A0, tab, vec);
}
void launch_bgemm_sym64(const GItem *items, int nitems, const GTerm *terms, const double *A0, const double *A1,
                        const double *const *tab, double *vec, hipStream_t s) {
    if (nitems > 0)
        hipLaunchKernelGGL(k_bgemm_sym<double>, dim3(nitems), dim3(256), 0, s, items, terms, A0, A1 ? A1 : A0, tab, vec);
}
void launch_bgemm_sym32(const GItem *items, int nitems, const GTerm *terms, const float *A0, const float *A1,
                        const float *const *tab, float *vec, hipStream_t s) {
    if (nitems > 0)
        hipLaunchKernelGGL(k_bgemm_sym<float>, dim3(nitems), dim3(256), 0, s, items, terms, A0, A1 ? A1 : A0, tab, vec);
}
void launch_bgemm_t64(const GItem *items, int nitems, const GTerm *terms, const double *A0, const double *A1,
                      const double *const *tab, double *vec, int narrow, hipStream_t s) {
    launch_bgemm_tl<double>(items, nitems, terms, A0, A1, tab, vec, narrow, s);
}
void launch_bgemm_t32(const GItem *items, int nitems, const GTerm *terms, const float *A0, const float *A1,
                      const float *const *tab, float *vec, int narrow, hipStream_t s) {
    launch_bgemm_tl<float>(items, nitems, terms, A0, A1, tab, vec, narrow, s);
}
}  // namespace h2w
