// h2w_ops.hip -- host orchestration of libh2w: assembly, matvec, GMRES and
// the C ABI declared in include/h2w.h.
//
// Device layout (one handle):
//   points  px/py/pz    tree-order coordinates (FP64)
//   mat64 / mat32       one pool with every stored operator, column-major,
//                       32-element aligned; mat32 is the FP32 shadow at the
//                       same element offsets
//   vec64 / vec32       one pool with x and y in tree order, then the outgoing
//                       (o) and incoming (u) skeleton vectors of every family,
//                       level and box, then the semi-nested pair vectors (t)
// A matvec is a fixed sequence of batched-GEMV launches over work lists built
// once at assembly (up pass per level, one M2L + near-field launch, down pass
// per level, leaf down, semi-nested CUR down).
#include <hip/hip_runtime.h>

#include <atomic>
#include <mutex>
#include <thread>

#include <algorithm>
#include <array>
#include <atomic>
#include <deque>
#include <chrono>
#include <cmath>
#include <complex>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <numeric>
#include <string>
#include <vector>

#include "h2w_handle.hpp"

namespace h2w {

static thread_local std::string g_err;
void set_error(const std::string &m) { g_err = m; }

}  // namespace h2w

namespace h2w {
namespace {

int ref_nlevels(int dim, int64_t N, int n_max, bool grid) {
    if (grid && dim > 1) {
        int n = (int)std::llround(dim == 2 ? std::sqrt((double)N) : std::cbrt((double)N));
        int p = (int)std::llround(dim == 2 ? std::sqrt((double)n_max) : std::cbrt((double)n_max));
        if (dim == 2) return (int)std::ceil(2.0 * std::log(double(n) / p) / std::log(4));
        return (int)std::ceil(3 * std::log(double(n) / p) / std::log(8));
    }
    return (int)std::ceil(std::log(double(N) / n_max) / std::log((double)(1 << dim)));
}

// GL-16 nodes/weights by Newton on P_16, for the IE diagonal's Kii
// (*/codes/integral{1,2,3}d.hpp; Gauss_Legendre_Nodes_and_Weights.hpp:471-523)
void gl16(double *nodes, double *weights) {
    const int n = 16;
    double pos[8], wts[8];
    for (int i = 0; i < 8; ++i) {
        double x = std::cos(kPI * (i + 0.75) / (n + 0.5));
        double dp = 1.0;
        for (int it = 0; it < 100; ++it) {
            double p0 = 1.0, p1 = x;
            for (int k = 2; k <= n; ++k) {
                double p2 = ((2.0 * k - 1.0) * x * p1 - (k - 1.0) * p0) / k;
                p0 = p1;
                p1 = p2;
            }
            dp = n * (x * p1 - p0) / (x * x - 1.0);
            double dx = p1 / dp;
            x -= dx;
            if (std::fabs(dx) < 1e-17) break;
        }
        double p0 = 1.0, p1 = x;
        for (int k = 2; k <= n; ++k) {
            double p2 = ((2.0 * k - 1.0) * x * p1 - (k - 1.0) * p0) / k;
            p0 = p1;
            p1 = p2;
        }
        dp = n * (x * p1 - p0) / (x * x - 1.0);
        pos[i] = x;
        wts[i] = 2.0 / ((1.0 - x * x) * dp * dp);
    }
    for (int i = 0; i < 8; ++i) {
        int s = 7 - i;
        nodes[2 * i] = -pos[s];
        nodes[2 * i + 1] = pos[s];
        weights[2 * i] = weights[2 * i + 1] = wts[s];
    }
}

// Diagonal of the complex kernels.  3D Helmholtz (choice 2): 500 sqrt(N) (3D/codes/kernel.hpp:132-144).
// 2D Hankel (choice 10): (1 + 15 log N + Kii) / h^2 with h = N^(-1/2) and the complex
// Kii = 4 GL16^2 of (i/4) H0^(1)(R) = (i J0(R) - Y0(R)) / 4 on [0, h/2]^2 (2D/codes/kernel.hpp:126-135,
// 2D/codes/integral2d.hpp:16-57,60-90).
void diag_value_c(int dim, int choice, int64_t N, double &re, double &im) {
    if (choice == 2) {
        re = 500.0 * std::sqrt(double(N));
        im = 0.0;
        return;
    }
    double nd[16], w[16];
    gl16(nd, w);
    const double h = 1.0 / std::sqrt(double(N));
    const double cx = 0.5 * (0.5 * h), Lx = cx;
    double kr = 0.0, ki = 0.0;
    for (int i = 0; i < 16; ++i)
        for (int j = 0; j < 16; ++j) {
            const double tx = cx * nd[i] + Lx, ty = cx * nd[j] + Lx;
            const double R = std::sqrt(tx * tx + ty * ty);
            kr += w[i] * w[j] * (-::y0(R) / 4.0);
            ki += w[i] * w[j] * (::j0(R) / 4.0);
        }
    kr *= cx * cx * 4;
    ki *= cx * cx * 4;
    const double h2 = std::pow(h, 2.0);
    re = (1.0 + 15.0 * std::log(double(N)) + kr) / h2;
    im = ki / h2;
    (void)dim;
}

// diagonal value of A (the i == j branch of getMatrixEntry):
// IE: (1 + Kii) / h^dim with Kii = 2^dim * GL16^dim of the integrand on [0, h/2]^dim,
// h = N^(-1/dim) (1D/codes/kernel.hpp:95-114, 2D/codes/kernel.hpp:101-122, 3D/codes/kernel.hpp:101-129);
// RBF: 1D sqrt(2N) (reference_compat) / 2D 1 / 3D sqrt(N).
double diag_value(int dim, int choice, int64_t N, int compat) {
    if (choice == 1) {
        if (dim == 1) return std::sqrt(double(compat ? 2 * N : N));
        if (dim == 2) return 1.0;
        return std::sqrt(double(N));
    }
    double nd[16], w[16];
    gl16(nd, w);
    double h = dim == 1 ? 1.0 / double(N) : (dim == 2 ? 1.0 / std::sqrt(double(N)) : 1.0 / std::cbrt(double(N)));
    double cx = 0.5 * (0.5 * h), Lx = cx;
    double res = 0.0;
    if (dim == 1) {
        for (int i = 0; i < 16; ++i) res += w[i] * std::log(std::fabs(1.0 * (cx * nd[i] + Lx)));
        res *= cx;
        res *= 2;
        return (1.0 + res) / h;
    }
    if (dim == 2) {
        double c = -1.0 / (2 * kPI);
        for (int i = 0; i < 16; ++i)
            for (int j = 0; j < 16; ++j) {
                double tx = cx * nd[i] + Lx, ty = cx * nd[j] + Lx;
                res += w[i] * w[j] * (c * 0.5 * std::log(tx * tx + ty * ty));
            }
        res *= (cx * cx);
        res *= 4;
        return (1.0 + res) / std::pow(h, 2.0);
    }
    for (int i = 0; i < 16; ++i)
        for (int j = 0; j < 16; ++j)
            for (int k = 0; k < 16; ++k) {
                double tx = cx * nd[i] + Lx, ty = cx * nd[j] + Lx, tz = cx * nd[k] + Lx;
                res += (w[i] * w[j] * w[k] * (1.0 / ((4 * kPI) * std::sqrt(tx * tx + ty * ty + tz * tz))));
            }
    res *= (cx * cx * cx);
    res *= 8;
    return (1.0 + res) / std::pow(h, 3.0);
}

// ------------------------------------------------------------------ batched ACA driver
// Runs every block through the device ACA.  A batch shares one workspace pool
// from which each block takes one (U, V) column pair per step; batches are
// admitted by an estimated rank (rank_hint), and a block that runs out of pool
// is re-run in a later batch with a larger estimate (alone if needed).
struct AcaPool {
    DevBuf<double> ws;
    DevBuf<unsigned long long> top;
    int64_t cap = 0;  // doubles
    // the wide cross: tiles, states and partials of a batch, kept over the batches of an assembly
    DevBuf<uint8_t> wide;  // a batch's tables and partials of the passes (run_wide), one allocation
    // a batch's jobs, index lists and results, also kept over the assembly's batches
    DevBuf<uint8_t> flags;
    DevBuf<int32_t> idx, rank, stat, rp, cp, prow, pcol;
    DevBuf<double> hist, phist;
    DevBuf<int64_t> tab;
    DevBuf<AcaJob> jobs;
    DevBuf<LrJob> lrj;
    // L and R of the batches so far, part by part (offsets in elements)
    std::deque<DevBuf<double>> lr;
    std::vector<std::pair<int64_t, int64_t>> lr_part;  // first element, elements
    int64_t lr_len = 0;
};

// The workspace holds the U and V columns of every block of a batch.  It is sized
// to what the blocks at hand are estimated to need (within the budget: opts or
// half of the free device memory, at most 96 GB) and grows when a later call
// needs more, so small systems do not pay for a large allocation.
void ensure_pool(Handle &h, AcaPool &P, int64_t need_doubles) {
    int64_t budget = h.opts.workspace_bytes;
    if (budget <= 0) {
        size_t fr = 0, tot = 0;
        H2W_HIP(hipMemGetInfo(&fr, &tot));
        budget = std::min<int64_t>((int64_t)96 << 30, (int64_t)(fr / 2) + P.cap * 8);
        budget = std::max<int64_t>(budget, (int64_t)64 << 20);
    }
    const int64_t want = std::min<int64_t>(budget / 8, std::max<int64_t>(need_doubles + need_doubles / 4, 8 << 20));
    if (P.cap >= want) return;
    P.ws.release();
    P.cap = want;
    P.ws.alloc(P.cap);
    if (!P.top.p) P.top.alloc(1);
}

// Geometry features of an ACA block for the rank predictor: family, level, row and
// column counts, the box's and the partners' point counts, the interaction set's
// size and centre separations (in box half-widths), how much of their boxes the
// points fill, and the box centre.  All of order one.
void block_features(const Handle &h, int fam, int j, int b, const std::vector<int32_t> &partners, int64_t m,
                    int64_t n, AcaBlock &B) {
    const Plan &P = h.plan;
    const double hw = P.L / double(1 << j);
    auto centre = [&](int bx, int d) { return d < P.dim ? -P.L + (2.0 * P.icoord[j][bx][d] + 1.0) * hw : 0.0; };
    auto fill = [&](int bx) {
        const auto &bb = P.bbox[j][bx];
        if (bb[0] > bb[3]) return 0.0;
        double e = 0.0;
        for (int d = 0; d < P.dim; ++d) e += bb[3 + d] - bb[d];
        return e / (P.dim * 2.0 * hw);
    };
    double sum_d = 0.0, min_d = 0.0, sum_fill = 0.0;
    int64_t pcount = 0;
    for (size_t q = 0; q < partners.size(); ++q) {
        const int p = partners[q];
        double d2 = 0.0;
        for (int d = 0; d < 3; ++d) d2 += (centre(p, d) - centre(b, d)) * (centre(p, d) - centre(b, d));
        const double dist = std::sqrt(d2) / hw;
        sum_d += dist;
        min_d = q == 0 ? dist : std::min(min_d, dist);
        sum_fill += fill(p);
        pcount += P.bcount[j][p];
    }
    const double np = (double)partners.size();
    float *f = B.feat.data();
    f[0] = fam == 0;
    f[1] = fam == 1;
    f[2] = fam == 2;
    f[3] = (float)(j / 8.0);
    f[4] = (float)(std::log2(1.0 + m) / 16.0);
    f[5] = (float)(std::log2(1.0 + n) / 20.0);
    f[6] = (float)(std::log2(1.0 + P.bcount[j][b]) / 16.0);
    f[7] = (float)(std::log2(1.0 + pcount) / 20.0);
    f[8] = (float)(np / 64.0);
    f[9] = (float)(np > 0 ? sum_d / np / 8.0 : 0.0);
    f[10] = (float)(min_d / 8.0);
    f[11] = (float)fill(b);
    f[12] = (float)(np > 0 ? sum_fill / np : 0.0);
    for (int d = 0; d < 3; ++d) f[13 + d] = (float)(centre(b, d) / P.L);
    B.has_feat = true;
}

// The cross of a batch's blocks (device copies of the jobs at djobs).  Blocks with a
// fixed-rank phase (AcaJob.pad = kfix > 1, from the rank model) first take kfix pivot steps
// without the normS update and stopping test -- every launch enqueued at once, no host reads
// in between -- and are then judged by the reference's own stopping rule, applied to all their
// steps at once: the normS sequence follows from the Gram products |<U_q,U_k>||<V_q,V_k>| of
// their terms, the block ends at the first step the rule stops (the pivots up to there are the
// ones the adaptive cross takes, since the rule never influences a pivot) or, when the rule
// holds for every step (rank under-predicted), it continues adaptively from there.  Adaptive
// steps are enqueued 16 at a time; between groups the host reads how many blocks are done.
// Every step advances a block's rank, moves its first-row search on, or finishes it, so the
// loop ends within max(m) + max(tcap) + 1 steps.
void run_wide(Handle &h, const std::vector<AcaJob> &jobs, const std::vector<int> &est, const AcaJob *djobs,
              const int32_t *didx, AcaPool &pool, int64_t *dtab, uint8_t *dflags, int32_t *drank, int32_t *dstat, int32_t *drp,
              int32_t *dcp, double *dhist, double tol) {
    hipStream_t s = h.stream;
    const int nb = (int)jobs.size();
    int maxm = 0, maxt = 0, maxfix = 0;
    // tiles of every block, and room for the inner products of twice its estimated rank and more
    const int T = wide_tile();
    std::vector<WideBlk> wb(nb);
    std::vector<int2> rt, ct;
    int64_t pd = 0;
    for (int q = 0; q < nb; ++q) {
        const AcaJob &J = jobs[q];
        maxm = std::max(maxm, J.m);
        maxt = std::max(maxt, J.tcap);
        maxfix = std::max(maxfix, J.pad);
        WideBlk &W = wb[q];
        W.nrt = (J.n + T - 1) / T;
        W.nct = (J.m + T - 1) / T;
        W.cap = std::min(J.tcap, std::max(4 * est[q], 256));
        W.pad = 0;
        W.rt0 = (int)rt.size();
        W.ct0 = (int)ct.size();
        W.pd = pd;
        pd += (int64_t)(W.nrt + W.nct) * W.cap;
        for (int t = 0; t < W.nrt; ++t) rt.push_back(int2{q, t});
        for (int t = 0; t < W.nct; ++t) ct.push_back(int2{q, t});
    }
    const int nrow = (int)rt.size(), ncol = (int)ct.size();
    for (WideBlk &W : wb) W.ct0 += nrow;
    rt.insert(rt.end(), ct.begin(), ct.end());
    size_t wlen = 0;
    auto part = [&](size_t bytes) {
        const size_t o = wlen;
        wlen += (bytes + 255) / 256 * 256;
        return o;
    };
    const size_t o_blk = part(nb * sizeof(WideBlk)), o_tiles = part(rt.size() * sizeof(int2)),
                 o_state = part(nb * sizeof(WideState)), o_part = part(rt.size() * 32), o_dot = part(pd * 8),
                 o_done = part(4), o_arr = part(nb * 4);
    pool.wide.ensure(std::max<size_t>(wlen, 256));
    WideBlk *dblk = reinterpret_cast<WideBlk *>(pool.wide.p + o_blk);
    int2 *dtiles = reinterpret_cast<int2 *>(pool.wide.p + o_tiles);
    WideState *dst = reinterpret_cast<WideState *>(pool.wide.p + o_state);
    int32_t *ddone = reinterpret_cast<int32_t *>(pool.wide.p + o_done);
    uint32_t *darr = reinterpret_cast<uint32_t *>(pool.wide.p + o_arr);
    H2W_HIP(hipMemcpyAsync(dblk, wb.data(), nb * sizeof(WideBlk), hipMemcpyHostToDevice, s));
    if (!rt.empty()) H2W_HIP(hipMemcpyAsync(dtiles, rt.data(), rt.size() * sizeof(int2), hipMemcpyHostToDevice, s));
    H2W_HIP(hipMemsetAsync(darr, 0, nb * sizeof(uint32_t), s));
    const WideArgs W{dblk, dtiles, nrow, ncol, reinterpret_cast<double *>(pool.wide.p + o_part),
                     reinterpret_cast<double *>(pool.wide.p + o_dot), darr};
    launch_wide_init(djobs, dblk, nb, dst, dflags, dtab, pool.top.p, pool.cap, s);
    auto step = [&]() {
        if (nrow > 0 && ncol > 0)
            launch_wide_step(djobs, W, didx, pool.ws.p, dtab, dflags, dst, drp, dcp, dhist, pool.top.p, pool.cap, h.kp,
                             tol, s);
    };
    // (the step after the last accepted one is taken beside its inner products)
    const int64_t limit = (int64_t)maxm + maxt + 2;
    int64_t steps = 0;
    if (maxfix > 1) {
        // ---- fixed phase (a block whose first rows are zero spends steps on its first-row search:
        // enqueue more until every block has parked or ended)
        std::vector<WideState> hs(nb);
        int64_t todo = maxfix;
        while (true) {
            for (int64_t c = 0; c < todo; ++c, ++steps) step();
            H2W_HIP(hipGetLastError());
            H2W_HIP(hipMemcpyAsync(hs.data(), dst, (size_t)nb * sizeof(WideState), hipMemcpyDeviceToHost, s));
            H2W_HIP(hipStreamSynchronize(s));
            int running = 0;
            for (auto &w : hs) running += !w.done;
            if (running == 0) break;
            if (steps > limit) throw Error{H2W_EHIP, "wide cross (fixed phase) did not finish within its step bound"};
            todo = 16;
        }
        // ---- Gram products of the judged blocks (status 2: parked at kfix, 3: ended inside the phase)
        std::vector<GramJob> gj;
        std::vector<int64_t> poff(nb, -1);
        int64_t plen = 0;
        for (int b = 0; b < nb; ++b) {
            if (hs[b].status != 2 && hs[b].status != 3) continue;
            const int K = hs[b].rank;
            poff[b] = plen;
            plen += (int64_t)K * (K + 1) / 2;
            const int nt = (K + 63) / 64;
            for (int ki = 0; ki < nt; ++ki)
                for (int qi = 0; qi <= ki; ++qi) gj.push_back(GramJob{b, qi, ki, 0, poff[b]});
        }
        std::vector<int32_t> fin(nb, -2);
        std::vector<double> nrm(nb, 0.0);
        if (!gj.empty()) {
            DevBuf<GramJob> dgj;
            DevBuf<double> dprod;
            dgj.upload(gj, s);
            dprod.alloc(std::max<int64_t>(plen, 1));
            launch_wide_gram(dgj.p, (int)gj.size(), djobs, dst, pool.ws.p, dtab, dprod.p, s);
            H2W_HIP(hipGetLastError());
            std::vector<double> prod(plen);
            H2W_HIP(hipMemcpyAsync(prod.data(), dprod.p, plen * 8, hipMemcpyDeviceToHost, s));
            H2W_HIP(hipStreamSynchronize(s));
            for (int b = 0; b < nb; ++b) {
                if (poff[b] < 0) continue;
                const int K = hs[b].rank;
                const int64_t ho = 2 * jobs[b].piv;
                std::vector<double> hb(2 * (size_t)K);
                H2W_HIP(hipMemcpyAsync(hb.data(), dhist + ho, 2 * (size_t)K * 8, hipMemcpyDeviceToHost, s));
                H2W_HIP(hipStreamSynchronize(s));
                // the reference's recurrence (2D/codes/aca.hpp:404-409): the first term enters with
                // normS = 0; term k adds (|u_k||v_k|)^2 + 2 sum_{q <= k} |<U_q,u_k>||<V_q,v_k>|
                const int mn = std::min(jobs[b].m, jobs[b].n);
                double normS = 0.0;
                int stop = -1;
                for (int k = 0; k < K; ++k) {
                    const double uv = hb[2 * k];
                    if (k > 0) {
                        double S = 0.0;
                        const double *pk = prod.data() + poff[b] + (int64_t)k * (k + 1) / 2;
                        for (int q = 0; q <= k; ++q) S += pk[q];
                        normS = std::sqrt(normS * normS + uv * uv + 2.0 * S);
                    }
                    hb[2 * k + 1] = normS;
                    if (!(uv > tol * normS && k + 1 < mn)) {
                        stop = k + 1;
                        break;
                    }
                }
                const int kept = stop > 0 ? stop : K;
                if (stop > 0 || hs[b].status == 3) {
                    fin[b] = kept;
                    h.rank_fix_extra_steps += K - kept;
                } else {
                    fin[b] = -1;  // continue adaptively
                    nrm[b] = normS;
                    h.rank_fix_resumed++;
                }
                h.rank_fix_blocks++;
                H2W_HIP(hipMemcpyAsync(dhist + ho, hb.data(), 2 * (size_t)kept * 8, hipMemcpyHostToDevice, s));
                H2W_HIP(hipStreamSynchronize(s));
            }
            DevBuf<int32_t> dfin;
            DevBuf<double> dnrm;
            dfin.upload(fin, s);
            dnrm.upload(nrm, s);
            launch_wide_judge(djobs, dblk, nb, dst, dfin.p, dnrm.p, dtab, pool.top.p, pool.cap, s);
            H2W_HIP(hipGetLastError());
            H2W_HIP(hipStreamSynchronize(s));
        }
    }
    while (true) {
        if (steps == 0)
            for (int c = 0; c < 16; ++c, ++steps) step();
        launch_wide_finish(dst, nb, drank, dstat, ddone, s);
        H2W_HIP(hipGetLastError());
        int nd = 0;
        H2W_HIP(hipMemcpyAsync(&nd, ddone, 4, hipMemcpyDeviceToHost, s));
        H2W_HIP(hipStreamSynchronize(s));
        if (nd == nb) break;
        if (steps > limit) throw Error{H2W_EHIP, "wide cross did not finish within its step bound"};
        for (int c = 0; c < 16; ++c, ++steps) step();
    }
    // sampled entries of the fixed-rank blocks against their cross approximation
    if (maxfix > 1) {
        std::vector<int> sel;
        for (int b = 0; b < nb; ++b)
            if (jobs[b].pad > 1) sel.push_back(b);
        DevBuf<double> e2, a2;
        e2.alloc(nb);
        a2.alloc(nb);
        launch_aca_sample(djobs, nb, drank, didx, pool.ws.p, dtab, h.kp, 256, e2.p, a2.p, s);
        H2W_HIP(hipGetLastError());
        std::vector<double> he(nb), ha(nb);
        std::vector<int32_t> hst(nb);
        H2W_HIP(hipMemcpyAsync(he.data(), e2.p, nb * 8, hipMemcpyDeviceToHost, s));
        H2W_HIP(hipMemcpyAsync(ha.data(), a2.p, nb * 8, hipMemcpyDeviceToHost, s));
        H2W_HIP(hipMemcpyAsync(hst.data(), dstat, nb * 4, hipMemcpyDeviceToHost, s));
        H2W_HIP(hipStreamSynchronize(s));
        for (int b : sel)
            if (hst[b] == 0 && ha[b] > 0.0)
                h.rank_fix_sampled_err = std::max(h.rank_fix_sampled_err, std::sqrt(he[b] / ha[b]));
    }
}

void run_aca(Handle &h, std::vector<AcaBlock> &blocks, int rank_hint, AcaPool &pool) {
    if (blocks.empty()) return;
    const double tol = std::pow(10.0, -1.0 * h.tol_pow);
    hipStream_t s = h.stream;
    const bool verbose = std::getenv("H2W_VERBOSE") != nullptr;
    std::vector<int> est(blocks.size());
    for (size_t b = 0; b < blocks.size(); ++b) {
        int mn = (int)std::min(blocks[b].rows.size(), blocks[b].cols.size());
        est[b] = std::min(mn, std::max(1, rank_hint));
    }
    std::vector<size_t> todo(blocks.size());
    std::iota(todo.begin(), todo.end(), 0);
    // learned rank estimates: the workspace each block reserves, and rank-homogeneous batches
    // (blocks in descending predicted rank); the cross itself still stops at the tolerance
    bool pred = h.rank_model.p != nullptr;
    for (auto &B : blocks) pred = pred && B.has_feat;
    std::vector<float> plog;
    if (pred) {
        const int nb = (int)blocks.size();
        std::vector<float> F((size_t)nb * kRankFeatures);
        for (int b = 0; b < nb; ++b) std::copy(blocks[b].feat.begin(), blocks[b].feat.end(), &F[(size_t)b * kRankFeatures]);
        DevBuf<float> dF, dO;
        dF.upload(F, s);
        dO.alloc(nb);
        launch_rank_mlp(dF.p, nb, h.rank_model.p, dO.p, s);
        H2W_HIP(hipGetLastError());
        plog.resize(nb);
        H2W_HIP(hipMemcpyAsync(plog.data(), dO.p, (size_t)nb * 4, hipMemcpyDeviceToHost, s));
        H2W_HIP(hipStreamSynchronize(s));
        for (int b = 0; b < nb; ++b) {
            const int mn = (int)std::min(blocks[b].rows.size(), blocks[b].cols.size());
            const double pr = std::max(0.0, std::exp2((double)plog[b]) - 1.0);
            est[b] = std::max(1, std::min(mn, (int)std::ceil(1.2 * pr) + 4));
        }
        std::stable_sort(todo.begin(), todo.end(), [&](size_t a, size_t c) { return est[a] > est[c]; });
    }
    const std::vector<int> est0 = est;
    // fixed-rank phase of the wide cross: 3 % above the predicted rank plus 2 steps (H2W_NO_FIXED_RANK
    // keeps the adaptive cross throughout)
    const bool fixed_off = std::getenv("H2W_NO_FIXED_RANK") != nullptr;
    auto kfix_of = [&](size_t b) {
        const double pr = pred ? std::max(0.0, std::exp2((double)plog[b]) - 1.0) : 0.0;
        return std::max(2, (int)std::lround(1.03 * pr) + 2);
    };
    // complex kernels: workspace, L and R in complex elements (two doubles each), every block through
    // the one-workgroup cross
    const bool cx = h.cplx;
    const int esz = cx ? 2 : 1;
    int64_t need = 0;
    // a block's workspace: a column pair (each padded to an even length) per term, and the step ahead
    auto space_of = [&](size_t b) {
        const int64_t mp = (blocks[b].rows.size() + 1) / 2 * 2, np = (blocks[b].cols.size() + 1) / 2 * 2;
        return (mp + np) * (int64_t)(est[b] + 1);
    };
    for (size_t b = 0; b < blocks.size(); ++b) need += space_of(b);
    ensure_pool(h, pool, need * esz);
    h.aca_pool_bytes = std::max<int64_t>(h.aca_pool_bytes, pool.cap * 8);
    DevBuf<uint8_t> &flags = pool.flags;
    DevBuf<int32_t> &didx = pool.idx, &drank = pool.rank, &dstat = pool.stat, &drp = pool.rp, &dcp = pool.cp;
    DevBuf<double> &dhist = pool.hist;
    DevBuf<int64_t> &dtab = pool.tab;
    DevBuf<AcaJob> &djobs = pool.jobs;
    DevBuf<LrJob> &dlr = pool.lrj;
    const size_t kBig = 16384;    // complex kernels: m + n above which a block gets a 1024-thread workgroup
    // m + n above which a block with a predicted rank takes a fixed-rank phase (H2W_WIDE_MIN overrides):
    // its judgement costs host work per block, which small blocks do not repay
    const size_t kHuge = cx ? SIZE_MAX
                            : std::getenv("H2W_WIDE_MIN") ? (size_t)std::atoll(std::getenv("H2W_WIDE_MIN")) : 8192;
    // m + n up to which a batch's blocks take every step in one launch, a workgroup each (k_aca_small): a step there
    // is shorter than two launches, while a workgroup alone is slower on longer rows (blocks of m + n above 8192
    // for a fixed-rank phase never are).  Assemblies, all in tiles / to 256 / 512 / 1024 / 2048: 1D N = 1584 at 1e-12
    // 6.4 / 5.4 / 5.1 / 4.9 / 5.4 ms, 1D N = 8000 11.4 / 10.7 / 10.0 / 9.9 / 9.9, 2D N = 1600 8.6 / 7.4 / 7.2 / 7.0 /
    // 7.0, 2D N = 4000 14.0 / 13.8 / 13.7 / 14.0 / 19.6, 3D N = 2000 9.4 / 9.1 / 8.2 / 10.1 / 10.8.  (1D ranks are 20
    // to 40, so that longer rows are still cheap to a workgroup alone.)
    const size_t kSmall = h.plan.dim == 1 ? 1024 : 512;
    while (!todo.empty()) {
        std::vector<size_t> rerun;
        size_t pos = 0;
        while (pos < todo.size()) {
            std::vector<size_t> batch;
            int64_t need = 0, isz = 0;
            while (pos < todo.size()) {
                size_t b = todo[pos];
                const AcaBlock &B = blocks[b];
                const int64_t nb = space_of(b);
                if (!batch.empty() && need + nb > pool.cap / esz) break;
                batch.push_back(b);
                need += nb;
                isz += (int64_t)(B.rows.size() + B.cols.size());
                ++pos;
                if (batch.size() >= 65535) break;
            }
            // the largest blocks first
            auto mn_of = [&](size_t b) { return blocks[b].rows.size() + blocks[b].cols.size(); };
            std::stable_partition(batch.begin(), batch.end(), [&](size_t b) { return mn_of(b) > kBig; });
            std::stable_partition(batch.begin(), batch.end(), [&](size_t b) { return mn_of(b) > kHuge; });
            size_t nhuge = 0, nbig = 0;
            while (nhuge < batch.size() && mn_of(batch[nhuge]) > kHuge) ++nhuge;
            nbig = nhuge;
            while (nbig < batch.size() && mn_of(batch[nbig]) > kBig) ++nbig;
            std::vector<AcaJob> jobs(batch.size());
            std::vector<int32_t> idx;
            idx.reserve(isz);
            int64_t fo = 0, po = 0, to = 0;
            for (size_t q = 0; q < batch.size(); ++q) {
                const AcaBlock &B = blocks[batch[q]];
                AcaJob &J = jobs[q];
                J.m = (int32_t)B.rows.size();
                J.n = (int32_t)B.cols.size();
                J.tcap = std::min(std::min(J.m, J.n), 8192);
                // large blocks with a predicted rank: a fixed-rank phase of about that many steps
                J.pad = (pred && q < nhuge && !fixed_off) ? std::min(J.tcap, kfix_of(batch[q])) : 0;
                J.rows = (int64_t)idx.size();
                idx.insert(idx.end(), B.rows.begin(), B.rows.end());
                J.cols = (int64_t)idx.size();
                idx.insert(idx.end(), B.cols.begin(), B.cols.end());
                J.tab = to;
                to += 2LL * J.tcap;
                J.wsF = fo;
                fo += align_up((int64_t)(J.m + J.n), 64);
                J.piv = po;
                po += J.tcap;
            }
            bool small = !cx;
            for (size_t q = 0; q < batch.size() && small; ++q)
                small = mn_of(batch[q]) <= std::min(kSmall, kHuge) && jobs[q].pad <= 1;
            flags.ensure(std::max<int64_t>(fo, 1));
            dtab.ensure(std::max<int64_t>(to, 1));
            didx.upload(idx, s);
            djobs.upload(jobs, s);
            drank.ensure(batch.size());
            dstat.ensure(batch.size());
            drp.ensure(std::max<int64_t>(po, 1));
            dcp.ensure(std::max<int64_t>(po, 1));
            dhist.ensure(std::max<int64_t>(2 * po, 2));
            H2W_HIP(hipMemsetAsync(pool.top.p, 0, sizeof(unsigned long long), s));
            ++h.aca_batches;
            double tb = now_s();
            if (cx) {
                double2 *wsc = reinterpret_cast<double2 *>(pool.ws.p);
                if (nbig > 0)
                    launch_aca_c(djobs.p, (int)nbig, didx.p, wsc, pool.cap / 2, pool.top.p, dtab.p, flags.p, drank.p,
                                 dstat.p, drp.p, dcp.p, h.kpc, tol, dhist.p, 1, s);
                if (batch.size() > nbig)
                    launch_aca_c(djobs.p + nbig, (int)(batch.size() - nbig), didx.p, wsc, pool.cap / 2, pool.top.p,
                                 dtab.p, flags.p, drank.p + nbig, dstat.p + nbig, drp.p, dcp.p, h.kpc, tol, dhist.p, 0, s);
            } else if (small) {
                launch_aca_small(djobs.p, (int)batch.size(), didx.p, pool.ws.p, pool.cap, pool.top.p, dtab.p, flags.p,
                                 drank.p, dstat.p, drp.p, dcp.p, h.kp, tol, dhist.p, s);
            } else {
                std::vector<int> best(batch.size());
                for (size_t q = 0; q < batch.size(); ++q) best[q] = est[batch[q]];
                run_wide(h, jobs, best, djobs.p, didx.p, pool, dtab.p, flags.p, drank.p, dstat.p, drp.p, dcp.p, dhist.p,
                         tol);
            }
            H2W_HIP(hipGetLastError());
            std::vector<int32_t> rk(batch.size()), st(batch.size());
            H2W_HIP(hipMemcpyAsync(rk.data(), drank.p, rk.size() * 4, hipMemcpyDeviceToHost, s));
            H2W_HIP(hipMemcpyAsync(st.data(), dstat.p, st.size() * 4, hipMemcpyDeviceToHost, s));
            H2W_HIP(hipStreamSynchronize(s));
            if (verbose) {
                int mr = 0, nov = 0;
                for (size_t q = 0; q < batch.size(); ++q) {
                    mr = std::max(mr, rk[q]);
                    nov += st[q] != 0;
                }
                std::fprintf(stderr, "[h2w]   aca batch: %zu blocks (%zu big), max rank %d, %d re-run, %.3f s\n",
                             batch.size(), nbig, mr, nov, now_s() - tb);
            }
            std::vector<LrJob> lj;
            std::vector<size_t> lb;
            int64_t lo = 0, pk = 0;
            for (size_t q = 0; q < batch.size(); ++q) {
                size_t b = batch[q];
                if (st[q] != 0) {
                    int mn = (int)std::min(blocks[b].rows.size(), blocks[b].cols.size());
                    if (batch.size() == 1 && est[b] >= mn)
                        throw Error{H2W_ENOMEM, "ACA workspace pool too small for one block"};
                    est[b] = std::min(mn, std::max(est[b] * 4, rk[q] * 2));
                    rerun.push_back(b);
                    h.aca_reruns++;
                    continue;
                }
                AcaBlock &B = blocks[b];
                B.rank = rk[q];
                if (B.has_feat) {
                    h.sample_feat.push_back(B.feat);
                    h.sample_rank.push_back(rk[q]);
                }
                if (pred) {
                    h.rank_pred_blocks++;
                    h.rank_pred_under += rk[q] > est0[b];
                    h.rank_pred_abs_log2 += std::fabs((double)plog[b] - std::log2(1.0 + rk[q]));
                }
                if (rk[q] > 0) {
                    LrJob J;
                    J.tab = jobs[q].tab;
                    J.piv = jobs[q].piv;
                    J.m = jobs[q].m;
                    J.n = jobs[q].n;
                    J.rank = rk[q];
                    J.pk = (int32_t)pk;
                    pk += rk[q];
                    J.out = lo;
                    lo += 2LL * rk[q] * rk[q];
                    lj.push_back(J);
                    lb.push_back(b);
                }
            }
            if (!lj.empty()) {
                if (pk > INT32_MAX) throw Error{H2W_ENOMEM, "too many pivots in one batch"};
                dlr.upload(lj, s);
                // L and R stay on the device, where the transfers are made from them
                pool.lr.emplace_back();
                DevBuf<double> &part = pool.lr.back();
                part.alloc(lo * esz);
                pool.lr_part.push_back({pool.lr_len, lo});
                if (cx)
                    launch_lr_extract_c(dlr.p, (int)lj.size(), reinterpret_cast<const double2 *>(pool.ws.p), dtab.p,
                                        drp.p, dcp.p, reinterpret_cast<double2 *>(part.p), s);
                else launch_lr_extract(dlr.p, (int)lj.size(), pool.ws.p, dtab.p, drp.p, dcp.p, part.p, s);
                pool.prow.ensure(pk);
                pool.pcol.ensure(pk);
                pool.phist.ensure(2 * pk);
                launch_pack_pivots(dlr.p, (int)lj.size(), drp.p, dcp.p, dhist.p, pool.prow.p, pool.pcol.p, pool.phist.p,
                                   s);
                H2W_HIP(hipGetLastError());
                std::vector<int32_t> rp(pk), cp(pk);
                std::vector<double> hs(2 * pk);
                H2W_HIP(hipMemcpyAsync(hs.data(), pool.phist.p, 2 * pk * 8, hipMemcpyDeviceToHost, s));
                H2W_HIP(hipMemcpyAsync(rp.data(), pool.prow.p, pk * 4, hipMemcpyDeviceToHost, s));
                H2W_HIP(hipMemcpyAsync(cp.data(), pool.pcol.p, pk * 4, hipMemcpyDeviceToHost, s));
                H2W_HIP(hipStreamSynchronize(s));
                for (size_t q = 0; q < lj.size(); ++q) {
                    AcaBlock &B = blocks[lb[q]];
                    const int64_t o = lj[q].pk, r = lj[q].rank;
                    B.rb.assign(rp.begin() + o, rp.begin() + o + r);
                    B.cb.assign(cp.begin() + o, cp.begin() + o + r);
                    B.hist.assign(hs.begin() + 2 * o, hs.begin() + 2 * (o + r));
                    B.lr = pool.lr_len + lj[q].out;
                }
                pool.lr_len += lo;
            }
        }
        todo.swap(rerun);
        if (!todo.empty()) {
            // re-runs go with larger estimates: let the workspace grow to hold them
            int64_t need2 = 0;
            for (size_t b : todo) need2 += space_of(b);
            ensure_pool(h, pool, need2 * esz);
        }
    }
}

std::vector<int32_t> range_list(int64_t start, int64_t count) {
    std::vector<int32_t> v(count);
    for (int64_t i = 0; i < count; ++i) v[i] = (int32_t)(start + i);
    return v;
}

// far field, bottom-up NCA (3D/codes/HODLR3Dtree.hpp:1872-1939)
void far_nca(Handle &h, AcaPool &pool) {
    const Plan &P = h.plan;
    auto &F = h.fam[0];
    F.assign(P.nL + 1, FamLevel());
    if (P.dim == 1) return;
    for (int j = P.nL; j >= 2; --j) {
        FamLevel &fl = F[j];
        fl.nb = P.nboxes[j];
        fl.S.resize(fl.nb);
        for (int b = 0; b < fl.nb; ++b) {
            if (j == P.nL) fl.S[b] = range_list(P.bstart[j][b], P.bcount[j][b]);
            else
                for (int c = 0; c < P.nchild; ++c) {
                    auto &ir = F[j + 1].Ir[b * P.nchild + c];
                    fl.S[b].insert(fl.S[b].end(), ir.begin(), ir.end());
                }
        }
        std::vector<AcaBlock> blocks(fl.nb);
        for (int b = 0; b < fl.nb; ++b) {
            blocks[b].rows = fl.S[b];
            const auto far = P.far_of(j, b);
            for (int f : far) blocks[b].cols.insert(blocks[b].cols.end(), fl.S[f].begin(), fl.S[f].end());
            block_features(h, 0, j, b, far, (int64_t)blocks[b].rows.size(), (int64_t)blocks[b].cols.size(), blocks[b]);
        }
        // the far rank is bounded by the row-set size (children's skeletons)
        int hint = 0;
        for (auto &B : blocks) hint = std::max<int>(hint, (int)B.rows.size());
        run_aca(h, blocks, hint, pool);
        fl.rank.resize(fl.nb);
        fl.Ir.resize(fl.nb);
        fl.Ic.resize(fl.nb);
        fl.lr.assign(fl.nb, -1);
        fl.hist.resize(fl.nb);
        for (int b = 0; b < fl.nb; ++b) {
            AcaBlock &B = blocks[b];
            fl.rank[b] = B.rank;
            fl.hist[b] = std::move(B.hist);
            for (int q = 0; q < B.rank; ++q) {
                fl.Ir[b].push_back(B.rows[B.rb[q]]);
                fl.Ic[b].push_back(B.cols[B.cb[q]]);
            }
            fl.lr[b] = B.lr;
        }
        if (std::getenv("H2W_VERBOSE")) std::fprintf(stderr, "[h2w]  far level %d done\n", j);
    }
}

// vertex-sharing field, top-down NCA with the parent's column pivots appended
// (3D/codes/HODLR3Dtree.hpp:2062-2107; 1D/codes/HODLR1Dtree.hpp:231-276)
void vertex_nca(Handle &h, AcaPool &pool) {
    const Plan &P = h.plan;
    auto &F = h.fam[1];
    F.assign(P.nL + 1, FamLevel());
    for (int j = 1; j <= P.nL; ++j) {
        FamLevel &fl = F[j];
        fl.nb = P.nboxes[j];
        std::vector<AcaBlock> blocks(fl.nb);
        for (int b = 0; b < fl.nb; ++b) {
            blocks[b].rows = range_list(P.bstart[j][b], P.bcount[j][b]);
            const auto ver = P.vert_of(j, b);
            for (int v : ver) {
                auto r = range_list(P.bstart[j][v], P.bcount[j][v]);
                blocks[b].cols.insert(blocks[b].cols.end(), r.begin(), r.end());
            }
            if (j > 1) {
                auto &pic = F[j - 1].Ic[b / P.nchild];
                blocks[b].cols.insert(blocks[b].cols.end(), pic.begin(), pic.end());
            }
            block_features(h, 1, j, b, ver, (int64_t)blocks[b].rows.size(), (int64_t)blocks[b].cols.size(), blocks[b]);
        }
        // ranks shrink with the box size: start from twice the parent level's largest rank
        int hint = std::max(16, h.opts.rank_cap);
        if (j > 1) {
            hint = 0;
            for (int r : F[j - 1].rank) hint = std::max(hint, r);
            hint = std::max(16, 2 * hint);
        }
        run_aca(h, blocks, hint, pool);
        fl.rank.resize(fl.nb);
        fl.Ir.resize(fl.nb);
        fl.Ic.resize(fl.nb);
        fl.lr.assign(fl.nb, -1);
        fl.hist.resize(fl.nb);
        for (int b = 0; b < fl.nb; ++b) {
            AcaBlock &B = blocks[b];
            fl.rank[b] = B.rank;
            fl.hist[b] = std::move(B.hist);
            for (int q = 0; q < B.rank; ++q) {
                fl.Ir[b].push_back(B.rows[B.rb[q]]);
                fl.Ic[b].push_back(B.cols[B.cb[q]]);
            }
            fl.lr[b] = B.lr;
        }
        if (std::getenv("H2W_VERBOSE")) std::fprintf(stderr, "[h2w]  vertex level %d done\n", j);
    }
    for (int j = 1; j <= P.nL; ++j) {
        FamLevel &fl = F[j];
        fl.S.assign(fl.nb, {});
        for (int b = 0; b < fl.nb; ++b) {
            if (j == P.nL) fl.S[b] = range_list(P.bstart[j][b], P.bcount[j][b]);
            else
                for (int c = 0; c < P.nchild; ++c) {
                    auto &ir = F[j + 1].Ir[b * P.nchild + c];
                    fl.S[b].insert(fl.S[b].end(), ir.begin(), ir.end());
                }
        }
    }
}

// semi-nested vertex blocks: one cross approximation per directed pair and level
// (3D/codes/HODLR3Dtree.hpp:2250-2321; 1D/codes/HODLR1Dtree.hpp:418-443)
void cur_pairs(Handle &h, AcaPool &pool) {
    const Plan &P = h.plan;
    h.pairs.clear();
    std::vector<AcaBlock> blocks;
    for (int j = 1; j <= P.nL; ++j)
        for (int b = 0; b < P.nboxes[j]; ++b)
            for (int v : (h.variant == H2W_NON_NESTED ? P.il[j][b] : P.vert_of(j, b))) {
                Pair p;
                p.level = j;
                p.b = b;
                p.v = v;
                p.rank = 0;
                h.pairs.push_back(p);
                AcaBlock B;
                B.rows = range_list(P.bstart[j][b], P.bcount[j][b]);
                B.cols = range_list(P.bstart[j][v], P.bcount[j][v]);
                block_features(h, 2, j, b, {v}, (int64_t)B.rows.size(), (int64_t)B.cols.size(), B);
                blocks.push_back(std::move(B));
            }
    run_aca(h, blocks, std::max(16, h.opts.rank_cap), pool);
    for (size_t q = 0; q < blocks.size(); ++q) {
        Pair &p = h.pairs[q];
        AcaBlock &B = blocks[q];
        p.rank = B.rank;
        for (int k = 0; k < B.rank; ++k) {
            p.Ir.push_back(B.rows[B.rb[k]]);
            p.Ic.push_back(B.cols[B.cb[k]]);
        }
        p.lr = B.lr;
    }
}

// The rows of a transfer (columns of a CUR row factor) are independent: sub-jobs of
// 64 rows (columns) spread one large box over many workgroups.
std::vector<XferJob> split_xfer(const std::vector<XferJob> &in) {
    std::vector<XferJob> out;
    for (const XferJob &J : in)
        for (int r0 = 0; r0 < J.m; r0 += 64) {
            XferJob K = J;
            K.m = std::min(64, J.m - r0);
            K.s = J.s + r0;
            K.e = J.e + r0;
            K.et = J.et + (int64_t)r0 * J.ldet;
            out.push_back(K);
        }
    return out;
}
std::vector<CurJob> split_cur(const std::vector<CurJob> &in) {
    std::vector<CurJob> out;
    for (const CurJob &J : in)
        for (int c0 = 0; c0 < J.n; c0 += 64) {
            CurJob K = J;
            K.n = std::min(64, J.n - c0);
            K.v = J.v + c0;
            K.a = J.a + (int64_t)c0 * J.lda;
            out.push_back(K);
        }
    return out;
}

// ------------------------------------------------------------------ work lists
constexpr int64_t kItemWork = 128 * 4096;  // elements of A per GEMV item before column chunking

void add_item(WorkList &W, int64_t y, int rows, const std::vector<TermSpec> &terms, bool atomic, int lda = -1,
              int row_base = 0, int pool = 0) {
    if (rows <= 0 || terms.empty()) return;
    if (lda < 0) lda = rows;
    int64_t C = 0;
    for (auto &t : terms) C += t.cols;
    if (C == 0) return;
    for (int r0 = 0; r0 < rows; r0 += kRowTile) {
        int tr = std::min(kRowTile, rows - r0);
        if ((int64_t)tr * C <= kItemWork) {
            GItem it;
            it.y = y + r0;
            it.xb = 0;
            it.rows = tr;
            it.lda = lda;
            it.row0 = row_base + r0;
            it.t0 = (int32_t)W.terms.size();
            for (auto &t : terms)
                if (t.cols > 0) W.terms.push_back(GTerm{t.a, t.x, -1, t.cols, 0});
            it.t1 = (int32_t)W.terms.size();
            it.flags = (atomic ? 1 : 0) | (pool << 1);
            W.items.push_back(it);
        } else {
            // column chunks accumulate atomically
            const int64_t maxc = std::max<int64_t>(1, kItemWork / kRowTile);
            GItem it;
            it.rows = tr;
            it.lda = lda;
            it.row0 = row_base + r0;
            it.y = y + r0;
            it.xb = 0;
            it.flags = 1 | (pool << 1);
            int64_t used = 0;
            it.t0 = (int32_t)W.terms.size();
            for (auto &t : terms) {
                for (int64_t c0 = 0; c0 < t.cols;) {
                    int64_t take = std::min<int64_t>(t.cols - c0, maxc - used);
                    W.terms.push_back(GTerm{t.a + c0 * lda, t.x + c0, -1, (int32_t)take, 0});
                    used += take;
                    c0 += take;
                    if (used == maxc) {
                        it.t1 = (int32_t)W.terms.size();
                        W.items.push_back(it);
                        it.t0 = it.t1;
                        used = 0;
                    }
                }
            }
            it.t1 = (int32_t)W.terms.size();
            if (it.t1 > it.t0) W.items.push_back(it);
        }
    }
}

// rank at which the ACA would have stopped for tolerance tau: the first accepted
// step k >= 1 with |u_k||v_k| <= tau * normS_k ends the cross (2D/codes/aca.hpp:363)
// Items whose terms are never split by columns: a row tile's terms are grouped into
// items of at most kItemWork elements (a tile split over several items accumulates
// atomically).  Terms keep their t (a symmetric term's transposed-product output).
void add_item_whole(WorkList &W, int64_t y, int64_t xb, int rows, const std::vector<TermSpec> &terms, int lda,
                    int pool) {
    if (rows <= 0) return;
    std::vector<const TermSpec *> ts;
    for (auto &t : terms)
        if (t.cols > 0) ts.push_back(&t);
    if (ts.empty()) return;
    for (int r0 = 0; r0 < rows; r0 += kRowTile) {
        const int tr = std::min(kRowTile, rows - r0);
        std::vector<std::pair<size_t, size_t>> groups;  // [first, last) of ts per item
        size_t g0 = 0;
        int64_t work = 0;
        for (size_t q = 0; q < ts.size(); ++q) {
            const int64_t w = (int64_t)tr * ts[q]->cols;
            if (q > g0 && work + w > kItemWork) {
                groups.push_back({g0, q});
                g0 = q;
                work = 0;
            }
            work += w;
        }
        groups.push_back({g0, ts.size()});
        for (auto &g : groups) {
            GItem it;
            it.y = y + r0;
            it.xb = xb + r0;
            it.rows = tr;
            it.lda = lda;
            it.row0 = r0;
            it.t0 = (int32_t)W.terms.size();
            for (size_t q = g.first; q < g.second; ++q) {
                const TermSpec &t = *ts[q];
                W.terms.push_back(GTerm{t.a, t.x, t.t, t.cols, t.ld});
            }
            it.t1 = (int32_t)W.terms.size();
            it.flags = (groups.size() > 1 ? 1 : 0) | (pool << 1);
            W.items.push_back(it);
        }
    }
}

// Terms of an item whose blocks and vector segments follow one another become one: a box's blocks with
// consecutive partner boxes (their segments are in box order), a semi-nested box's pairs.  The kernels walk
// an item's terms one by one, about 1 us a term and wave from the next term's descriptor to its data, so
// short ones cost them most of their time: fused launch of the 16^3 grid (leaves of 8 points) 63 -> 22 us,
// 2D semi-nested 400 x 400 106 -> 101 us, its column factors 111 -> 106 us, 3D semi-nested N = 20000
// 110 -> 104 us; 16-wide 276 -> 258 us at 3D N = 20011.
void merge_terms(WorkList &W) {
    size_t n = 0;
    for (GItem &it : W.items) {
        const size_t t0 = n;
        for (int32_t k = it.t0; k < it.t1; ++k) {
            const GTerm t = W.terms[k];
            GTerm *p = n > t0 ? &W.terms[n - 1] : nullptr;
            const bool sym = t.t >= 0;
            if (p && (p->t >= 0) == sym && t.a == p->a + (int64_t)p->cols * it.lda && t.x == p->x + p->cols &&
                (!sym || t.t == p->t + p->cols) && t.ld == p->ld)
                p->cols += t.cols;
            else W.terms[n++] = t;
        }
        it.t0 = (int32_t)t0;
        it.t1 = (int32_t)n;
    }
    W.terms.resize(n);
}

// A launch of few large items leaves part of the GPU idle while the last of them stream: the transfer
// passes near the root, the semi-nested factors of the large boxes beside the small ones', and the fused
// M2L + near-field launch of anything but the largest systems.  Items above twice the launch's mean at
// about so many items are split by columns (the pieces accumulate atomically): 2048 for transfers and
// column factors, where an item is one column run, and 8192 for the fused launch, whose items are runs of
// blocks and accumulate atomically anyway.
// Measured (fused launch, FP64, unsplit / 2048 / 4096 / 8192 / 16384 items): 3D N = 20011 279 / 166 / 139 /
// 137 / 141 us, 32^3 grid at 1e-10 472 / 363 / 343 / 323 / 313 us, 2D N = 90000 191 / 195 / 176 / 174 /
// 178 us; complex 32^3 product 879 / 884 / 736 / 726 / 653 us.  The 16-wide launch likes larger
// pieces (wide_items).  The
// leaf launch of the 2D semi-nested 400 x 400 grid (more than 2048 items, some of 4 MB) 214 -> 137 us.
constexpr int64_t kMinItems = 2048, kMinPiece = 128 * 64;
constexpr int64_t kMinItemsFused = 8192, kMinPieceFused = 128 * 128;
void rebalance(WorkList &W) {
    merge_terms(W);
    const bool fused = W.role == 1;
    int64_t E = 0;
    for (auto &it : W.items)
        for (int32_t k = it.t0; k < it.t1; ++k) E += (int64_t)it.rows * W.terms[k].cols;
    const int64_t target = std::min(kItemWork, std::max<int64_t>(E / (fused ? kMinItemsFused : kMinItems),
                                                                 fused ? kMinPieceFused : kMinPiece));
    WorkList out;
    out.role = W.role;
    out.stage = W.stage;
    out.step = W.step;
    out.items.reserve(W.items.size());
    out.terms.reserve(W.terms.size());
    for (const GItem &it : W.items) {
        int64_t work = 0;
        for (int32_t k = it.t0; k < it.t1; ++k) work += (int64_t)it.rows * W.terms[k].cols;
        GItem nt = it;
        nt.t0 = (int32_t)out.terms.size();
        if (work <= 2 * target) {
            out.terms.insert(out.terms.end(), W.terms.begin() + it.t0, W.terms.begin() + it.t1);
            nt.t1 = (int32_t)out.terms.size();
            out.items.push_back(nt);
            continue;
        }
        // equal pieces of whole 16-column groups; a piece ends early rather than cut a term in two
        const int64_t np = (work + target - 1) / target;
        const int64_t maxc = align_up((work / it.rows + np - 1) / np, 16);
        nt.flags |= 1;
        int64_t used = 0;
        auto close = [&]() {
            nt.t1 = (int32_t)out.terms.size();
            if (nt.t1 > nt.t0) out.items.push_back(nt);
            nt.t0 = nt.t1;
            used = 0;
        };
        for (int32_t k = it.t0; k < it.t1; ++k) {
            const GTerm &t = W.terms[k];
            if (used > 0 && t.cols <= maxc && used + t.cols > maxc + maxc / 4) close();
            for (int64_t c0 = 0; c0 < t.cols;) {
                const int64_t left = t.cols - c0;
                const int64_t take = left <= maxc + maxc / 4 - used ? left : maxc - used;
                out.terms.push_back(
                    GTerm{t.a + c0 * it.lda, t.x + c0, t.t >= 0 ? t.t + c0 : -1, (int32_t)take, t.ld});
                used += take;
                c0 += take;
                if (used >= maxc) close();
            }
        }
        close();
    }
    W = std::move(out);
}

// One group of boxes whose pairwise blocks are stored once per unordered pair (the
// M2L blocks of one family and level, or the near field): box b has output offset
// y[b], input offset x[b] and size r[b]; up[b] lists the stored blocks K(b, p), p > b
// (r[b] x r[p], leading dimension pad_ld(r[b])), self[b] the block K(b, b) or -1.
struct SymGroup {
    std::vector<int64_t> y, x;
    std::vector<int> r;
    std::vector<std::vector<std::pair<int, int64_t>>> up;
    std::vector<int64_t> self;
    int pool = 0;
};
// The three lists of such a group: fused items (box b: y_b += K(b, p) x_p over its stored
// blocks, and each block's K(b, p)^T x_b added to y_p; in the single-vector product every
// fused item accumulates atomically, since its rows also receive the transposed products of
// other items), the
// 16-wide path's transposed items (box p: y_p += K(b, p)^T X_b, b < p) and the on-the-fly
// path's directed items.
struct SymLists {
    WorkList fused, trans, otf;
};
void sym_lists(const SymGroup &G, SymLists &L) {
    const int nb = (int)G.r.size();
    std::vector<std::vector<std::pair<int, int64_t>>> down(nb);
    for (int b = 0; b < nb; ++b)
        for (auto &pe : G.up[b]) down[pe.first].push_back({b, pe.second});
    const size_t item0 = L.fused.items.size();
    for (int b = 0; b < nb; ++b) {
        if (G.r[b] <= 0) continue;
        std::vector<TermSpec> t;
        if (G.self[b] >= 0) t.push_back(TermSpec{G.self[b], G.x[b], G.r[b]});
        for (auto &pe : G.up[b]) {
            TermSpec ts{pe.second, G.x[pe.first], G.r[pe.first]};
            ts.t = G.y[pe.first];
            t.push_back(ts);
        }
        add_item_whole(L.fused, G.y[b], G.x[b], G.r[b], t, (int)pad_ld(G.r[b]), G.pool);
    }
    // (flag bit 2: the single-vector kernel adds y atomically; the 16-wide path applies the
    // transposes in a later launch and keeps exclusive writers)
    for (size_t q = item0; q < L.fused.items.size(); ++q) L.fused.items[q].flags |= 4;
    for (int p = 0; p < nb; ++p) {
        std::vector<TermSpec> t;
        for (auto &be : down[p]) {
            TermSpec ts{be.second, G.x[be.first], G.r[be.first]};
            ts.ld = (int32_t)pad_ld(G.r[be.first]);
            t.push_back(ts);
        }
        add_item_whole(L.trans, G.y[p], 0, G.r[p], t, (int)pad_ld(G.r[p]), G.pool);
    }
    for (int b = 0; b < nb; ++b) {
        std::vector<TermSpec> t;
        if (G.self[b] >= 0) t.push_back(TermSpec{0, G.x[b], G.r[b]});
        for (auto &pe : G.up[b]) t.push_back(TermSpec{0, G.x[pe.first], G.r[pe.first]});
        for (auto &be : down[b]) t.push_back(TermSpec{0, G.x[be.first], G.r[be.first]});
        add_item(L.otf, G.y[b], G.r[b], t, false, (int)pad_ld(G.r[b]));
    }
}

int inner_rank(const std::vector<double> &hist, int rank, double tau) {
    for (int k = 1; k < rank && 2 * k + 1 < (int)hist.size(); ++k)
        if (hist[2 * k] <= tau * hist[2 * k + 1]) return k + 1;
    return rank;
}

}  // namespace

// The 16-wide path's items of a launch, appended to items, whose entries from item0 on are the single-vector
// path's: consecutive pieces of one row tile (their terms follow one another) are put together again.  A workgroup
// of the 16-wide kernels reads 16 input rows per item row, and sums and adds as many at the end: about 5 us an item
// beside its data.  Fused launches (role 1) up to a 2048th of the launch's elements, the others up to 256 columns,
// four 16-column groups per wave.  Measured, FP64, uncombined first:
//   fused, 4096 / 2048 / 1024 items: 32^3 grid at 1e-10 492, 452 / 448 / 458 us, 3D N = 20011 231, 229 / 204 / 202,
//     2D N = 90000 317, 297 / 292 / 304;
//   transfers of a product, 128 / 256 / 512 columns: 32^3 188, 168 / 161 / 154 us, 3D N = 20011 114, 106 / 102 / 101,
//     2D N = 90000 369, 352 / 348 / 352, 2D semi-nested N = 40000 156, 156 / 157 / 158, 16^3 55, 55 / 56 / 59.
//     (By elements instead, a 512th of the launch: the semi-nested one, a few tall boxes among many, 172.)
// Returns the number of items appended; 0 where nothing combines.
int64_t wide_items(std::vector<GItem> &items, int64_t item0, const std::vector<GTerm> &terms, int role) {
    const int64_t end = (int64_t)items.size();
    auto work = [&](const GItem &it) {
        int64_t w = 0;
        for (int32_t k = it.t0; k < it.t1; ++k) w += (int64_t)it.rows * terms[k].cols;
        return w;
    };
    int64_t E = 0, sum = 0;
    for (int64_t q = item0; q < end; ++q) E += work(items[q]);
    const int64_t share = E / 2048 + E / 8192;
    for (int64_t q = item0; q < end; ++q) {
        const GItem it = items[q];
        const int64_t w = work(it);
        const int64_t most = role == 1 ? share : 256 * (int64_t)it.rows;
        GItem &l = items.back();
        if (q > item0 && l.y == it.y && l.xb == it.xb && l.rows == it.rows && l.lda == it.lda && l.row0 == it.row0 &&
            l.flags == it.flags && l.t1 == it.t0 && sum + w <= most) {
            l.t1 = it.t1;
            sum += w;
        } else {
            items.push_back(it);
            sum = w;
        }
    }
    const int64_t n = (int64_t)items.size() - end;
    if (n < end - item0) return n;
    items.resize(end);
    return 0;
}
void Launch::set_wide(std::vector<GItem> &items, const std::vector<GTerm> &terms) {
    const int64_t n = (int64_t)items.size();
    nitemsm = wide_items(items, item0, terms, role);
    item0m = nitemsm ? n : item0;
    if (!nitemsm) nitemsm = nitems;
    int64_t e = 0;
    for (int64_t q = item0; q < item0 + nitems; ++q)
        for (int32_t k = items[q].t0; k < items[q].t1; ++k) e += (int64_t)items[q].rows * terms[k].cols;
    avg_item_elemsm = e / nitemsm;
}

namespace {
// wide: the 16-wide path dispatches these lists by items of its own
void upload_lists(std::vector<WorkList> &WL, LaunchSet &LS, bool wide, hipStream_t s) {
    std::vector<GItem> items;
    std::vector<GTerm> terms;
    LS.launches.clear();
    LS.elems.clear();
    for (auto &W : WL) {
        if (W.items.empty()) continue;
        Launch Lh;
        Lh.item0 = (int64_t)items.size();
        Lh.nitems = (int64_t)W.items.size();
        Lh.term0 = (int64_t)terms.size();
        Lh.nterms = (int64_t)W.terms.size();
        Lh.role = W.role;
        Lh.stage = W.stage;
        Lh.step = W.step;
        int64_t e = 0, sc = 0;
        for (auto &tm : W.terms) sc += tm.cols;
        Lh.avg_cols = W.terms.empty() ? 0 : (int)(sc / (int64_t)W.terms.size());
        for (auto it : W.items) {
            for (int q = it.t0; q < it.t1; ++q) e += (int64_t)it.rows * W.terms[q].cols;
            it.t0 += (int32_t)Lh.term0;
            it.t1 += (int32_t)Lh.term0;
            items.push_back(it);
        }
        terms.insert(terms.end(), W.terms.begin(), W.terms.end());
        Lh.avg_item_elems = e / Lh.nitems;
        if (wide) Lh.set_wide(items, terms);
        LS.launches.push_back(Lh);
        LS.elems.push_back(e);
    }
    LS.d_items.upload(items, s);
    LS.d_terms.upload(terms, s);
    LS.h_items = std::move(items);
    LS.h_terms = std::move(terms);
}

// ------------------------------------------------------------------ the refinement's inner operator
// Every box keeps the leading pivots at which its cross would have stopped for
// tolerance 10^-irp (from the ACA history); its M2L blocks are compact copies of
// the leading sub-blocks of the stored FP32 M2L blocks, its transfers are
// recomputed from the leading blocks of L and R.  Lives in its own FP32 buffer
// (work items flagged with pool 1); rebuilt by h2w_set_inner_tolerance and the
// autotuner.

void build_inner(Handle &h, double irp) {
    drop_graph(h, H2W_FP32_INNER);
    ++h.inner_gen;
    const Plan &P = h.plan;
    hipStream_t s = h.stream;
    // the inner buffers and lists are freed and reallocated below: nothing queued may still read them
    H2W_HIP(hipStreamSynchronize(s));
    const int nfam_lo[2] = {2, 1};
    const bool fam_on[2] = {P.dim >= 2 && h.variant != H2W_NON_NESTED, h.variant == H2W_NESTED};
    const int nleaf = P.nboxes[P.nL];
    auto &m2l = h.m2l;
    auto &nearb = h.nearb;
    h.inner.launches.clear();
    h.inner_elems = 0;
    h.mat32in.release();
    // ---- inner operator of the refinement: each box keeps the leading pivots at which its
    // cross would have stopped for tolerance 10^-ir_tol_pow; its M2L blocks are the leading
    // sub-blocks of the stored ones, its transfers are recomputed from the leading L, R blocks
    const bool inner_on = h.opts.fp32_shadow && irp > 0 && irp < h.tol_pow;
    int64_t in_len = 0;
    auto take_in = [&](int64_t elems) {
        int64_t o = in_len;
        in_len += align_up(elems, 32);
        return o;
    };
    // compact copies of the inner M2L sub-blocks: (index into m2l, offset in the inner region)
    std::vector<std::pair<size_t, int64_t>> m2l_in;
    if (inner_on) {
        const double tau = std::pow(10.0, -1.0 * irp);
        for (int f = 0; f < 2; ++f) {
            if (!fam_on[f]) continue;
            for (int j = nfam_lo[f]; j <= P.nL; ++j) {
                FamLevel &fl = h.fam[f][j];
                fl.kin.assign(fl.nb, 0);
                for (int b = 0; b < fl.nb; ++b)
                    fl.kin[b] = fl.rank[b] > 0 ? inner_rank(fl.hist[b], fl.rank[b], tau) : 0;
            }
            // inner transfers: rows are the children's leading pivots, each child's segment
            // padded to a multiple of 4 rows so every row tile stays aligned
            for (int j = nfam_lo[f]; j <= P.nL; ++j) {
                FamLevel &fl = h.fam[f][j];
                fl.ein_off.assign(fl.nb, -1);
                fl.eint_off.assign(fl.nb, -1);
                for (int b = 0; b < fl.nb; ++b) {
                    int64_t m = 0;
                    if (j == P.nL) m = P.bcount[j][b];
                    else
                        for (int c = 0; c < P.nchild; ++c) m += pad_ld(h.fam[f][j + 1].kin[b * P.nchild + c]);
                    if (m * fl.kin[b] == 0) continue;
                    fl.ein_off[b] = take_in(pad_ld(m) * fl.kin[b]);
                    fl.eint_off[b] = take_in(pad_ld(fl.kin[b]) * m);
                }
            }
        }
        for (size_t q = 0; q < m2l.size(); ++q) {
            const M2LBlk &m = m2l[q];
            const FamLevel &fl = h.fam[m.f][m.j];
            // (the blocks of one box one after another, as in the full operator)
            if (q > 0 && (m2l[q - 1].f != m.f || m2l[q - 1].j != m.j || m2l[q - 1].b != m.b)) in_len = align_up(in_len, 32);
            if (fl.kin[m.b] > 0 && fl.kin[m.p] > 0) {
                m2l_in.push_back({q, in_len});
                in_len += pad_ld(fl.kin[m.b]) * fl.kin[m.p];
            }
        }
        in_len = align_up(in_len, 32);
    }
    if (inner_on) h.mat32in.alloc(std::max<int64_t>(in_len, 32));
    if (inner_on && in_len > 0) H2W_HIP(hipMemsetAsync(h.mat32in.p, 0, in_len * 4, s));
    if (inner_on && in_len > 0) {
        std::vector<int32_t> idx;
        std::vector<XferJob> xj;
        LrForm lr;  // (unless the assembly's are still there)
        for (int f = 0; f < 2; ++f) {
            if (!fam_on[f]) continue;
            for (int j = nfam_lo[f]; j <= P.nL; ++j) {
                FamLevel &fl = h.fam[f][j];
                for (int b = 0; b < fl.nb; ++b) {
                    if (fl.ein_off[b] < 0) continue;
                    const int k = fl.kin[b];
                    const int64_t lro = h.d_lr.p ? fl.lr[b] : lr.add(fl.Ir[b].data(), fl.Ic[b].data(), k);
                    const int64_t icq = (int64_t)idx.size();
                    idx.insert(idx.end(), fl.Ic[b].begin(), fl.Ic[b].begin() + k);
                    int64_t m = 0;
                    if (j == P.nL) m = P.bcount[j][b];
                    else
                        for (int c = 0; c < P.nchild; ++c) m += pad_ld(h.fam[f][j + 1].kin[b * P.nchild + c]);
                    const int lde = (int)pad_ld(m), ldet = (int)pad_ld(k);
                    auto add_job = [&](const int32_t *S, int ms, int64_t row) {
                        if (ms == 0) return;
                        XferJob J;
                        J.r = k;
                        J.m = ms;
                        J.s = (int64_t)idx.size();
                        idx.insert(idx.end(), S, S + ms);
                        J.ic = icq;
                        J.lr = lro;  // (the leading k x k blocks of L and R)
                        J.ldr = h.d_lr.p ? fl.rank[b] : k;
                        J.pad = 0;
                        J.e = fl.ein_off[b] + row;
                        J.et = fl.eint_off[b] + row * ldet;
                        J.lde = lde;
                        J.ldet = ldet;
                        xj.push_back(J);
                    };
                    if (j == P.nL) {
                        auto rl = range_list(P.bstart[j][b], P.bcount[j][b]);
                        add_job(rl.data(), (int)rl.size(), 0);
                    } else {
                        int64_t row = 0;
                        for (int c = 0; c < P.nchild; ++c) {
                            const int cc = b * P.nchild + c;
                            const int kc = h.fam[f][j + 1].kin[cc];
                            add_job(h.fam[f][j + 1].Ir[cc].data(), kc, row);
                            row += pad_ld(kc);
                        }
                    }
                }
            }
        }
        DevBuf<int32_t> didx;
        DevBuf<double> tmp;
        DevBuf<XferJob> dxj;
        didx.upload(idx, s);
        xj = split_xfer(xj);
        dxj.upload(xj, s);
        tmp.alloc(in_len);
        H2W_HIP(hipMemsetAsync(tmp.p, 0, in_len * 8, s));
        lr.run(h, s);
        launch_xfer(dxj.p, (int)xj.size(), didx.p, h.d_lr.p ? h.d_lr.p : lr.out.p, tmp.p, h.kp, s);
        H2W_HIP(hipGetLastError());
        launch_to_fp32(tmp.p, h.mat32in.p, in_len, s);
        H2W_HIP(hipGetLastError());
        // compact copies of the leading M2L sub-blocks
        std::vector<CopyJob> cj;
        for (auto &pr : m2l_in) {
            const M2LBlk &m = m2l[pr.first];
            const FamLevel &fl = h.fam[m.f][m.j];
            CopyJob J;
            J.src = m.off;
            J.dst = pr.second;
            J.m = fl.kin[m.b];
            J.n = fl.kin[m.p];
            J.lds = (int32_t)pad_ld(fl.rank[m.b]);
            J.ldd = (int32_t)pad_ld(fl.kin[m.b]);
            cj.push_back(J);
        }
        DevBuf<CopyJob> dcj;
        dcj.upload(cj, s);
        launch_copy32(dcj.p, (int)cj.size(), h.mat32.p, h.mat32in.p, s);
        H2W_HIP(hipGetLastError());
        H2W_HIP(hipStreamSynchronize(s));
    }

    if (inner_on) {
        const int64_t base = 0;  // offsets into the inner buffer (items flagged with pool 1)
        std::vector<WorkList> IL;
        {
            WorkList W;
            for (int f = 0; f < 2; ++f) {
                if (!fam_on[f] || P.nL < nfam_lo[f]) continue;
                FamLevel &fl = h.fam[f][P.nL];
                for (int b = 0; b < fl.nb; ++b)
                    if (fl.eint_off[b] >= 0)
                        add_item(W, fl.o_off[b], fl.kin[b],
                                 {TermSpec{base + fl.eint_off[b], h.off_x + P.bstart[P.nL][b], (int32_t)P.bcount[P.nL][b]}},
                                 false, (int)pad_ld(fl.kin[b]), 0, 1);
            }
            for (auto &p : h.pairs)
                if (p.rank > 0)
                    add_item(W, p.t_off, p.rank,
                             {TermSpec{p.ar_off, h.off_x + P.bstart[p.level][p.v], (int32_t)P.bcount[p.level][p.v]}},
                             false, (int)pad_ld(p.rank));
            IL.push_back(std::move(W));
        }
        for (int j = P.nL - 1; j >= 1; --j) {
            WorkList W;
            W.step = P.nL - j;
            for (int f = 0; f < 2; ++f) {
                if (!fam_on[f] || j < nfam_lo[f]) continue;
                FamLevel &fl = h.fam[f][j];
                FamLevel &ch = h.fam[f][j + 1];
                for (int b = 0; b < fl.nb; ++b) {
                    if (fl.eint_off[b] < 0) continue;
                    const int64_t ldet = pad_ld(fl.kin[b]);
                    std::vector<TermSpec> t;
                    int64_t col = 0;
                    for (int c = 0; c < P.nchild; ++c) {
                        const int cc = b * P.nchild + c;
                        if (ch.kin[cc] > 0)
                            t.push_back(TermSpec{base + fl.eint_off[b] + col * ldet, ch.o_off[cc], (int32_t)ch.kin[cc]});
                        col += pad_ld(ch.kin[cc]);
                    }
                    add_item(W, fl.o_off[b], fl.kin[b], t, false, (int)ldet, 0, 1);
                }
            }
            IL.push_back(std::move(W));
        }
        {
            // the inner M2L blocks (compact leading sub-blocks, one per unordered pair, second
            // pool) and the stored near field, both directions in one fused launch
            SymLists SL;
            for (int f = 0; f < 2; ++f) {
                if (!fam_on[f]) continue;
                for (int j = nfam_lo[f]; j <= P.nL; ++j) {
                    FamLevel &fl = h.fam[f][j];
                    SymGroup G;
                    G.y.assign(fl.u_off.begin(), fl.u_off.end());
                    G.x.assign(fl.o_off.begin(), fl.o_off.end());
                    G.r = fl.kin;
                    G.up.assign(fl.nb, {});
                    G.self.assign(fl.nb, -1);
                    G.pool = 1;
                    for (auto &pr : m2l_in) {
                        const M2LBlk &m = m2l[pr.first];
                        if (m.f == f && m.j == j) G.up[m.b].push_back({m.p, base + pr.second});
                    }
                    sym_lists(G, SL);
                }
            }
            {
                SymGroup G;
                G.y.resize(nleaf);
                G.x.resize(nleaf);
                G.r.resize(nleaf);
                G.up.assign(nleaf, {});
                G.self.assign(nleaf, -1);
                for (int b = 0; b < nleaf; ++b) {
                    G.y[b] = h.off_y + P.bstart[P.nL][b];
                    G.x[b] = h.off_x + P.bstart[P.nL][b];
                    G.r[b] = (int)P.bcount[P.nL][b];
                }
                for (auto &nb : nearb) {
                    if (nb.n == nb.b) G.self[nb.b] = nb.off;
                    else G.up[nb.b].push_back({nb.n, nb.off});
                }
                sym_lists(G, SL);
            }
            SL.fused.role = 1;
            SL.fused.stage = 1;
            IL.push_back(std::move(SL.fused));
            SL.trans.role = 3;
            SL.trans.stage = 1;
            SL.trans.step = 1;
            std::vector<WorkList> tl;
            tl.push_back(std::move(SL.trans));
            upload_lists(tl, h.inner_trans, false, s);
        }
        for (int j = 1; j <= P.nL - 1; ++j) {
            WorkList W;
            W.stage = 2;
            W.step = P.nL - j;
            for (int f = 0; f < 2; ++f) {
                if (!fam_on[f] || j < nfam_lo[f]) continue;
                FamLevel &fl = h.fam[f][j];
                FamLevel &ch = h.fam[f][j + 1];
                for (int b = 0; b < fl.nb; ++b) {
                    if (fl.ein_off[b] < 0) continue;
                    int64_t m = 0;
                    for (int c = 0; c < P.nchild; ++c) m += pad_ld(ch.kin[b * P.nchild + c]);
                    int64_t row = 0;
                    for (int c = 0; c < P.nchild; ++c) {
                        const int cc = b * P.nchild + c;
                        if (ch.kin[cc] > 0)
                            add_item(W, ch.u_off[cc], ch.kin[cc],
                                     {TermSpec{base + fl.ein_off[b], fl.u_off[b], (int32_t)fl.kin[b]}}, false,
                                     (int)pad_ld(m), (int)row, 1);
                        row += pad_ld(ch.kin[cc]);
                    }
                }
            }
            IL.push_back(std::move(W));
        }
        {
            WorkList W;
            W.stage = 2;
            for (int b = 0; b < nleaf; ++b) {
                std::vector<TermSpec> t;
                for (int f = 0; f < 2; ++f) {
                    if (!fam_on[f] || P.nL < nfam_lo[f]) continue;
                    FamLevel &fl = h.fam[f][P.nL];
                    if (fl.ein_off[b] >= 0) t.push_back(TermSpec{base + fl.ein_off[b], fl.u_off[b], (int32_t)fl.kin[b]});
                }
                add_item(W, h.off_y + P.bstart[P.nL][b], (int)P.bcount[P.nL][b], t, false,
                         (int)pad_ld(P.bcount[P.nL][b]), 0, 1);
            }
            IL.push_back(std::move(W));
        }
        if (!h.pairs.empty()) {
            WorkList W;
            W.role = 2;
            W.stage = 3;
            std::vector<std::vector<std::vector<TermSpec>>> per(P.nL + 1);
            for (int j = 1; j <= P.nL; ++j) per[j].assign(P.nboxes[j], {});
            for (auto &p : h.pairs)
                if (p.rank > 0) per[p.level][p.b].push_back(TermSpec{p.ac_off, p.t_off, (int32_t)p.rank});
            for (int j = 1; j <= P.nL; ++j)
                for (int b = 0; b < P.nboxes[j]; ++b)
                    add_item(W, h.off_y + P.bstart[j][b], (int)P.bcount[j][b], per[j][b], true,
                             (int)pad_ld(P.bcount[j][b]));
            IL.push_back(std::move(W));
        }
        for (auto &W : IL)
            rebalance(W);
        upload_lists(IL, h.inner, true, s);
        h.inner_elems = 0;
        for (auto e : h.inner.elems) h.inner_elems += e;
    } else {
        h.inner.launches.clear();
        h.inner_elems = 0;
    }
    H2W_HIP(hipStreamSynchronize(s));
    h.ir_exp = inner_on ? irp : 0.0;
}

// ------------------------------------------------------------------ assembly

void assemble_operators(Handle &h, double t0, DevBuf<double> &scratch);

void assemble(Handle &h) {
    drop_graphs(h);
    double t0 = now_s();
    h.aca_reruns = h.aca_batches = 0;
    h.aca_pool_bytes = 0;
    h.rank_pred_blocks = h.rank_pred_under = 0;
    h.rank_pred_abs_log2 = 0.0;
    h.rank_fix_blocks = h.rank_fix_resumed = 0;
    h.rank_fix_extra_steps = 0;
    h.rank_fix_sampled_err = 0.0;
    h.sample_feat.clear();
    h.sample_rank.clear();
    const bool verbose = std::getenv("H2W_VERBOSE") != nullptr;
    auto phase = [&](const char *what) {
        if (verbose) {
            (void)hipStreamSynchronize(h.stream);
            std::fprintf(stderr, "[h2w] %-28s %8.3f s\n", what, now_s() - t0);
        }
    };
    const Plan &P = h.plan;
    DevBuf<double> scratch;  // the crosses' workspace, reused
    {
        AcaPool pool;
        if (P.dim >= 2 && h.variant != H2W_NON_NESTED) far_nca(h, pool);
        else h.fam[0].assign(P.nL + 1, FamLevel());
        phase("far NCA");
        if (h.variant == H2W_NESTED) vertex_nca(h, pool);
        else {
            h.fam[1].assign(P.nL + 1, FamLevel());
            cur_pairs(h, pool);
        }
        phase("vertex NCA / CUR");
        const int64_t es = h.cplx ? 2 : 1;
        h.d_lr.alloc(pool.lr_len * es);
        for (size_t q = 0; q < pool.lr.size(); ++q)
            H2W_HIP(hipMemcpyAsync(h.d_lr.p + pool.lr_part[q].first * es, pool.lr[q].p, pool.lr_part[q].second * es * 8,
                                   hipMemcpyDeviceToDevice, h.stream));
        H2W_HIP(hipStreamSynchronize(h.stream));
        scratch.swap(pool.ws);
    }
    assemble_operators(h, t0, scratch);
}

// The transfer passes near the root are launches of a few hundred kilobytes, one after another, 3 to 4 us
// each whatever they hold (all of a 1D system with N = 2048).  Levels B .. T-1 can be one
// launch each way: their skeletons go straight to those of their descendants at level T and back, by the
// products of the transfers between them.  Such blocks hold a full row of blocks each, so that every level
// of the group has as many bytes as the widest; a group grows while the launches it saves outweigh the bytes
// it adds, and while no block is so large that the launch would cut it into pieces that accumulate
// atomically (a box's outgoing vector stays one sum in one order).  Returns the groups from the leaves up as
// (T, B), B = T - 1 for a level by itself (real kernels; the inner operator keeps its own chain).
// Measured, products without / with: 1D N = 2048 62 / 48 us.
constexpr double kLaunchUs = 3.0, kBytesPerUs = 4.0e6;
// A group ends before the first level whose composites have entries above this.  Rounding in a chain of transfers
// perturbs the skeleton charges between two levels, and the next transfer reproduces the far field of whatever
// charges it is given; rounding in a composite of large entries of both signs is not so absorbed.  At 512 it stays at
// 1e-13.  (1D, uniform points, N = 70003 at 1e-12, entries to 2e4: the product of a random vector 1.9e-13 from the
// dense one by the chain, 6.4e-13 with composites, and the residual of a solve from x0 = 1 3e-7 / 1e-5; N = 2048,
// entries to 330: 1.1e-13 both.)
constexpr double kComposeMost = 512.0;
std::vector<std::pair<int, int>> level_groups(const Handle &h, const int (&lo)[2], const bool (&on)[2]) {
    const Plan &P = h.plan;
    std::vector<std::pair<int, int>> G;
    for (int T = P.nL; T > 1;) {
        int best = T - 1;
        double gain = 0.0, extra = 0.0;  // elements, each way
        int levels = 0;
        for (int j = T - 1; j >= 1 && !h.cplx; --j) {
            bool any = false, fits = true;
            for (int f = 0; f < 2; ++f) {
                if (!on[f] || j < lo[f]) continue;
                const FamLevel &fl = h.fam[f][j], &ft = h.fam[f][T];
                const int64_t nd = (int64_t)1 << (P.dim * (T - j));
                for (int b = 0; b < fl.nb; ++b) {
                    if (fl.rank[b] == 0) continue;
                    any = true;
                    int64_t R = 0;
                    for (int64_t c = b * nd; c < (b + 1) * nd; ++c) R += ft.rank[c];
                    fits = fits && std::min<int64_t>(fl.rank[b], kRowTile) * R <= 2 * kMinPiece;
                    extra += (double)fl.rank[b] * (double)(R - (int64_t)fl.S[b].size());
                }
            }
            if (j < T - 1 && !fits) break;
            levels += any;
            const double g = 2.0 * (levels - 1) * kLaunchUs - 2.0 * 8.0 * extra / kBytesPerUs;
            if (g > gain) {
                gain = g;
                best = j;
            }
        }
        G.push_back({T, best});
        T = best;
    }
    return G;
}

// Everything after the skeletons: pools, transfer / M2L / near-field / CUR blocks,
// the FP32 shadow, work lists and the inner operator.  Reads h.fam (ranks, pivots,
// L and R, ACA histories, row sets S) and h.pairs only, so it also rebuilds an
// operator from saved skeletons.  scratch: device memory to use, replaced if too small, released when done with.
void assemble_operators(Handle &h, double t0, DevBuf<double> &scratch) {
    const bool verbose = std::getenv("H2W_VERBOSE") != nullptr;
    auto phase = [&](const char *what) {
        if (verbose) {
            (void)hipStreamSynchronize(h.stream);
            std::fprintf(stderr, "[h2w] %-28s %8.3f s\n", what, now_s() - t0);
        }
    };
    const Plan &P = h.plan;
    hipStream_t s = h.stream;
    const int nfam_lo[2] = {2, 1};  // first level of each family
    const bool fam_on[2] = {P.dim >= 2 && h.variant != H2W_NON_NESTED, h.variant == H2W_NESTED};

    // ---- vector pool: x, y, skeleton vectors
    int64_t vo = 0;
    h.off_x = vo;
    vo += align_up(P.N, 32);
    h.off_y = vo;
    vo += align_up(P.N, 32);
    for (int f = 0; f < 2; ++f) {
        if (!fam_on[f]) continue;
        for (int j = nfam_lo[f]; j <= P.nL; ++j) {
            FamLevel &fl = h.fam[f][j];
            fl.o_off.resize(fl.nb);
            fl.u_off.resize(fl.nb);
            // o segments of one parent's children are contiguous (the parent's up input)
            for (int b = 0; b < fl.nb; ++b) {
                fl.o_off[b] = vo;
                vo += fl.rank[b];
            }
            vo = align_up(vo, 32);
            for (int b = 0; b < fl.nb; ++b) {
                fl.u_off[b] = vo;
                vo += fl.rank[b];
            }
            vo = align_up(vo, 32);
        }
    }
    for (auto &p : h.pairs) {
        p.t_off = vo;
        vo += p.rank;
    }
    h.vec_len = align_up(std::max<int64_t>(vo, 1), 32);

    // ---- matrix pool offsets
    int64_t mo = 0;
    auto take = [&](int64_t elems) {
        int64_t o = mo;
        mo += align_up(elems, 32);
        return o;
    };
    auto run = [&](int64_t elems) {  // right behind the block before (columns are multiples of 4 elements)
        int64_t o = mo;
        mo += elems;
        return o;
    };
    double memory = 0.0;
    for (int f = 0; f < 2; ++f) {
        if (!fam_on[f]) continue;
        for (int j = nfam_lo[f]; j <= P.nL; ++j) {
            FamLevel &fl = h.fam[f][j];
            fl.e_off.assign(fl.nb, -1);
            fl.et_off.assign(fl.nb, -1);
            for (int b = 0; b < fl.nb; ++b) {
                int64_t m = (int64_t)fl.S[b].size(), r = fl.rank[b];
                memory += 2.0 * (double)(m * r);
                if (m * r == 0) continue;
                fl.e_off[b] = take(pad_ld(m) * r);
                fl.et_off[b] = take(pad_ld(r) * m);
            }
        }
    }
    const int64_t xfer_len = mo;
    // the transfers of every level into a pool
    auto form_transfers = [&](double *A) {
        std::vector<int32_t> idx;
        std::vector<XferJob> xj;
        for (int f = 0; f < 2; ++f) {
            if (!fam_on[f]) continue;
            for (int j = nfam_lo[f]; j <= P.nL; ++j) {
                FamLevel &fl = h.fam[f][j];
                for (int b = 0; b < fl.nb; ++b) {
                    if (fl.e_off[b] < 0) continue;
                    XferJob J;
                    J.m = (int32_t)fl.S[b].size();
                    J.r = fl.rank[b];
                    J.s = (int64_t)idx.size();
                    idx.insert(idx.end(), fl.S[b].begin(), fl.S[b].end());
                    J.ic = (int64_t)idx.size();
                    idx.insert(idx.end(), fl.Ic[b].begin(), fl.Ic[b].end());
                    J.lr = fl.lr[b];
                    J.ldr = J.r;
                    J.pad = 0;
                    J.e = fl.e_off[b];
                    J.et = fl.et_off[b];
                    J.lde = (int32_t)pad_ld(J.m);
                    J.ldet = (int32_t)pad_ld(J.r);
                    xj.push_back(J);
                }
            }
        }
        DevBuf<int32_t> didx;
        DevBuf<XferJob> dxj;
        didx.upload(idx, s);
        xj = split_xfer(xj);
        dxj.upload(xj, s);
        if (h.cplx)
            launch_xfer_c(dxj.p, (int)xj.size(), didx.p, reinterpret_cast<const double2 *>(h.d_lr.p),
                          reinterpret_cast<double2 *>(A), h.kpc, s);
        else launch_xfer(dxj.p, (int)xj.size(), didx.p, h.d_lr.p, A, h.kp, s);
        H2W_HIP(hipGetLastError());
        H2W_HIP(hipStreamSynchronize(s));
    };
    auto &m2l = h.m2l;
    m2l.clear();
    for (int f = 0; f < 2; ++f) {
        if (!fam_on[f]) continue;
        for (int j = nfam_lo[f]; j <= P.nL; ++j) {
            FamLevel &fl = h.fam[f][j];
            for (int b = 0; b < fl.nb; ++b) {
                // (in box order, one after another: neighbouring partners then form one run of columns)
                auto partners = f == 0 ? P.far_of(j, b) : P.vert_of(j, b);
                std::sort(partners.begin(), partners.end());
                for (int p : partners) {
                    int64_t e = (int64_t)fl.rank[b] * fl.rank[p];
                    memory += (double)e;  // the reference counts both directions
                    // K(Ir_p, Ir_b) = K(Ir_b, Ir_p)^T entry for entry (the kernel depends on |x - y|
                    // only): one block per unordered pair, the lower-numbered box's
                    if (e == 0 || p < b) continue;
                    m2l.push_back(M2LBlk{f, j, b, p, run(pad_ld(fl.rank[b]) * fl.rank[p])});
                }
                mo = align_up(mo, 32);
            }
        }
    }
    auto &nearb = h.nearb;
    nearb.clear();
    const int nleaf = P.nboxes[P.nL];
    const bool count_near = !(P.dim == 1 && h.variant == H2W_SEMI_NESTED);  // 1D findMemory_sn skips it
    for (int b = 0; b < nleaf; ++b) {
        std::vector<int32_t> lst = P.near[b];
        lst.push_back(b);
        std::sort(lst.begin(), lst.end());
        for (int n : lst) {
            int64_t e = P.bcount[P.nL][b] * P.bcount[P.nL][n];
            if (count_near) memory += (double)e;
            if (e == 0 || n < b) continue;  // one block per unordered pair (self blocks kept)
            nearb.push_back(NearBlk{b, n, run(pad_ld(P.bcount[P.nL][b]) * P.bcount[P.nL][n])});
        }
        mo = align_up(mo, 32);
    }
    for (auto &p : h.pairs) {
        int64_t mb = P.bcount[p.level][p.b], nv = P.bcount[p.level][p.v];
        if (P.dim == 1) memory += (double)(mb * p.rank + (int64_t)p.rank * nv);  // U + V
        else memory += 2.0 * p.rank * p.rank + (double)(mb * p.rank + (int64_t)p.rank * nv);  // L + R + Ac + Ar
        p.ac_off = p.ar_off = -1;
        if (p.rank == 0) continue;
        p.ar_off = take(pad_ld(p.rank) * nv);
    }
    // (the pairs of one box are consecutive, and so are their intermediate vectors: one run of columns)
    for (size_t q = 0; q < h.pairs.size(); ++q) {
        Pair &p = h.pairs[q];
        if (q > 0 && (h.pairs[q - 1].level != p.level || h.pairs[q - 1].b != p.b)) mo = align_up(mo, 32);
        if (p.rank > 0) p.ac_off = run(pad_ld(P.bcount[p.level][p.b]) * p.rank);
    }
    mo = align_up(mo, 32);
    // composite transfers of the groups of several levels: per box c at T the blocks of all its ancestors of
    // the group side by side (down), per box above T - 1 its descendants' blocks transposed (up; at T - 1
    // that is the transfer itself)
    auto groups = level_groups(h, nfam_lo, fam_on);
    auto ancestor = [&](int c, int T, int j) { return c >> (P.dim * (T - j)); };
    auto first_at = [&](int b, int j, int T) { return (int)((int64_t)b << (P.dim * (T - j))); };
    auto rank_at = [&](int f, int b, int j, int T) {
        int64_t R = 0;
        for (int c = first_at(b, j, T); c < first_at(b + 1, j, T); ++c) R += h.fam[f][T].rank[c];
        return R;
    };
    // room for the groups' blocks from `base` on; returns its length
    auto place_composites = [&](int64_t base) {
        mo = base;
        for (auto [T, B] : groups)
            for (int f = 0; f < 2 && B < T - 1; ++f) {
                if (!fam_on[f]) continue;
                FamLevel &ft = h.fam[f][T];
                ft.c_off.assign(ft.nb, -1);
                for (int c = 0; c < ft.nb; ++c) {
                    int64_t n = 0;
                    for (int j = T - 1; j >= std::max(B, nfam_lo[f]); --j) n += h.fam[f][j].rank[ancestor(c, T, j)];
                    if (ft.rank[c] > 0 && n > 0) ft.c_off[c] = take(pad_ld(ft.rank[c]) * n);
                }
                for (int j = T - 2; j >= std::max(B, nfam_lo[f]); --j) {
                    FamLevel &fl = h.fam[f][j];
                    fl.ct_off.assign(fl.nb, -1);
                    for (int b = 0; b < fl.nb; ++b) {
                        const int64_t R = rank_at(f, b, j, T);
                        if (fl.rank[b] > 0 && R > 0) fl.ct_off[b] = take(pad_ld(fl.rank[b]) * R);
                    }
                }
            }
        return mo - base;
    };
    // the blocks placed from `base` on (len elements) from the transfers in A, level by level away from T (block (c, a)
    // from block (c, a's child)), with scratch at lo; returns the largest entry of every level
    auto form_composites = [&](double *A, int64_t base, int64_t len, double *lo) {
        std::vector<ComposeJob> jobs;
        std::vector<std::array<int64_t, 3>> runs;  // level, its jobs
        for (auto [T, B] : groups)
            for (int j = T - 1; j >= B && B < T - 1; --j) {
                const int64_t job0 = (int64_t)jobs.size();
                for (int f = 0; f < 2; ++f) {
                    if (!fam_on[f] || j < nfam_lo[f]) continue;
                    const FamLevel &fl = h.fam[f][j], &ft = h.fam[f][T];
                    for (int c = 0; c < ft.nb; ++c) {
                        const int a = ancestor(c, T, j);
                        if (ft.c_off[c] < 0 || fl.rank[a] == 0) continue;
                        int64_t row = 0, col = 0;  // of the child's rows in a's transfer, of the block in c's run
                        const int ch = ancestor(c, T, j + 1);
                        for (int q = a * P.nchild; q < ch; ++q) row += h.fam[f][j + 1].rank[q];
                        for (int i = T - 1; i > j; --i) col += h.fam[f][i].rank[ancestor(c, T, i)];
                        const int kc = h.fam[f][j + 1].rank[ch];
                        if (kc == 0) continue;
                        ComposeJob J;
                        J.m = ft.rank[c];
                        J.n = fl.rank[a];
                        J.ldd = (int32_t)pad_ld(J.m);
                        J.d = ft.c_off[c] + col * J.ldd;
                        J.dt = -1;
                        J.ldt = (int32_t)pad_ld(J.n);
                        J.pad = 0;
                        J.lda = J.ldb = (int32_t)pad_ld((int64_t)fl.S[a].size());
                        if (j == T - 1) {
                            J.k = 0;
                            J.a = fl.e_off[a] + row;
                            J.b = 0;
                        } else {
                            J.k = kc;
                            J.lda = J.ldd;
                            J.a = J.d - (int64_t)kc * J.ldd;  // (c, ch), the block before
                            J.b = fl.e_off[a] + row;
                            J.dt = fl.ct_off[a] + (ft.o_off[c] - ft.o_off[first_at(a, j, T)]) * J.ldt;
                        }
                        jobs.push_back(J);
                    }
                }
                runs.push_back({j, job0, (int64_t)jobs.size()});
            }
        // the blocks' low parts, the largest entry of each level, the jobs
        const int64_t nj = (int64_t)(jobs.size() * sizeof(ComposeJob) / 8);
        unsigned long long *dmost = reinterpret_cast<unsigned long long *>(lo + len);
        ComposeJob *dj = reinterpret_cast<ComposeJob *>(dmost + P.nL + 1);
        if (nj > 0) H2W_HIP(hipMemcpyAsync(dj, jobs.data(), (size_t)nj * 8, hipMemcpyHostToDevice, s));
        // (a block across a box without a skeleton is never formed, but is a factor of the next level's: zero, low
        // part included)
        H2W_HIP(hipMemsetAsync(lo, 0, (len + P.nL + 1) * 8, s));
        for (auto &r : runs)
            launch_compose(dj + r[1], (int)(r[2] - r[1]), A, lo, base, dmost + r[0], s);
        H2W_HIP(hipGetLastError());
        std::vector<double> most(P.nL + 1);
        H2W_HIP(hipMemcpyAsync(most.data(), dmost, (P.nL + 1) * 8, hipMemcpyDeviceToHost, s));
        H2W_HIP(hipStreamSynchronize(s));
        return most;
    };
    // Composites come last in the pool, once it is known which are used (kComposeMost): they are formed where the other
    // blocks will be, or in scratch where that is too small.  Up to 2 MB is taken for them beforehand.
    const int64_t pool_len = mo;
    int64_t comp_len = place_composites(xfer_len);
    const int64_t spare = std::min<int64_t>(comp_len, 1 << 18);
    int64_t need = 2 * comp_len + P.nL + 1;  // blocks, low parts, largest entries, jobs
    for (auto [T, B] : groups)
        for (int f = 0; f < 2; ++f)
            if (B < T - 1 && fam_on[f]) need += (int64_t)(T - B) * h.fam[f][T].nb * (int64_t)(sizeof(ComposeJob) / 8);
    const bool inside = xfer_len + need <= pool_len;
    // scratch for them; where the device has none left, every level is a launch of its own instead
    auto room = [&]() {
        try {
            scratch.ensure(xfer_len + need);
            return true;
        } catch (const Error &) {
            (void)hipGetLastError();
            std::vector<std::pair<int, int>> single;
            for (int T = P.nL; T > 1; --T) single.push_back({T, T - 1});
            groups = std::move(single);
            comp_len = 0;
            return false;
        }
    };
    if (comp_len == 0 || inside) scratch.release();
    else room();
    h.memory = memory;
    // (complex kernels: pools of (re, im) pairs at the same element offsets)
    const int esz = h.cplx ? 2 : 1;
    h.mat64.alloc(std::max<int64_t>(pool_len + spare, 32) * esz);
    H2W_HIP(hipMemsetAsync(h.mat64.p, 0, h.mat64.n * 8, s));
    h.vec64.alloc(h.vec_len * esz);
    if (h.cplx) h.vec32.release();
    else h.vec32.alloc(h.vec_len);
    {
        // the point of every vector slot, for on-the-fly near-field / M2L evaluation
        std::vector<int32_t> pid(h.vec_len, -1);
        for (int64_t t = 0; t < P.N; ++t) pid[h.off_x + t] = pid[h.off_y + t] = (int32_t)t;
        for (int f = 0; f < 2; ++f) {
            if (!fam_on[f]) continue;
            for (int j = nfam_lo[f]; j <= P.nL; ++j) {
                FamLevel &fl = h.fam[f][j];
                for (int b = 0; b < fl.nb; ++b)
                    for (int k = 0; k < fl.rank[b]; ++k) pid[fl.o_off[b] + k] = pid[fl.u_off[b] + k] = fl.Ir[b][k];
            }
        }
        h.spid.upload(pid, s);
        for (DevBuf<float> *v : {&h.sx32, &h.sy32, &h.sz32, &h.sxl, &h.syl, &h.szl}) v->ensure(h.vec_len);
        for (DevBuf<double> *v : {&h.sx64, &h.sy64, &h.sz64}) v->ensure(h.vec_len);
        launch_slot_points(h.spid.p, h.vec_len, h.d_px.p, h.d_py.p, h.d_pz.p, h.sx64.p, h.sy64.p, h.sz64.p, h.sx32.p,
                           h.sy32.p, h.sz32.p, h.sxl.p, h.syl.p, h.szl.p, s);
        H2W_HIP(hipGetLastError());
        H2W_HIP(hipStreamSynchronize(s));
        h.sp.x = h.sx32.p;
        h.sp.y = h.sy32.p;
        h.sp.z = h.sz32.p;
        h.sp.xl = h.sxl.p;
        h.sp.yl = h.syl.p;
        h.sp.zl = h.szl.p;
        h.sp.xd = h.sx64.p;
        h.sp.yd = h.sy64.p;
        h.sp.zd = h.sz64.p;
        h.sp.pid = h.spid.p;
        h.sp.dim = P.dim;
        h.sp.choice = h.choice;
        h.sp.diag = h.diag;
    }

    // ---- evaluate operators on the device
    form_transfers(h.mat64.p);
    if (comp_len > 0) {
        double *A = h.mat64.p;
        if (!inside) {
            A = scratch.p;
            H2W_HIP(hipMemcpyAsync(A, h.mat64.p, xfer_len * 8, hipMemcpyDeviceToDevice, s));
            H2W_HIP(hipMemsetAsync(A + xfer_len, 0, comp_len * 8, s));
        }
        const auto most = form_composites(A, xfer_len, comp_len, A + xfer_len + comp_len);
        std::vector<std::pair<int, int>> kept;
        for (auto [T, B] : groups) {
            int low = T - 1;  // the group's levels from here on are kept
            while (low > B && most[low - 1] <= kComposeMost) --low;
            kept.push_back({T, low});
            for (int q = low; q > B; --q) kept.push_back({q, q - 1});
        }
        const bool all = kept == groups;
        const int64_t comp_trial = comp_len;
        groups = std::move(kept);
        comp_len = place_composites(pool_len);
        if (comp_len > spare && (!inside || room())) {  // (not two pools at a time)
            if (inside) {
                H2W_HIP(hipMemcpyAsync(scratch.p, A, (xfer_len + comp_trial) * 8, hipMemcpyDeviceToDevice, s));
                A = scratch.p;
            }
            H2W_HIP(hipStreamSynchronize(s));
            h.mat64.alloc(pool_len + comp_len);
            H2W_HIP(hipMemsetAsync(h.mat64.p, 0, h.mat64.n * 8, s));
            H2W_HIP(hipMemcpyAsync(h.mat64.p, A, xfer_len * 8, hipMemcpyDeviceToDevice, s));
        }
        double *M = h.mat64.p;
        if (all && comp_len > 0) H2W_HIP(hipMemcpyAsync(M + pool_len, A + xfer_len, comp_len * 8, hipMemcpyDeviceToDevice, s));
        else if (comp_len > 0) form_composites(M, pool_len, comp_len, A + xfer_len);
        if (M == A) H2W_HIP(hipMemsetAsync(M + xfer_len, 0, need * 8, s));
        H2W_HIP(hipStreamSynchronize(s));
        scratch.release();
    }
    h.mat_len = std::max<int64_t>(pool_len + comp_len, 32);
    if (!h.pairs.empty()) {
        // semi-nested row factors
        std::vector<int32_t> idx;
        std::vector<CurJob> cj;
        for (auto &p : h.pairs) {
            if (p.rank == 0) continue;
            CurJob J;
            J.r = p.rank;
            J.n = (int32_t)P.bcount[p.level][p.v];
            J.ir = (int64_t)idx.size();
            idx.insert(idx.end(), p.Ir.begin(), p.Ir.end());
            J.v = (int64_t)idx.size();
            auto vr = range_list(P.bstart[p.level][p.v], J.n);
            idx.insert(idx.end(), vr.begin(), vr.end());
            J.lr = p.lr;
            J.a = p.ar_off;
            J.lda = (int32_t)pad_ld(J.r);
            J.pad = 0;
            cj.push_back(J);
        }
        DevBuf<int32_t> didx;
        DevBuf<CurJob> dcj;
        didx.upload(idx, s);
        cj = split_cur(cj);
        dcj.upload(cj, s);
        if (h.cplx)
            launch_cur_c(dcj.p, (int)cj.size(), didx.p, reinterpret_cast<const double2 *>(h.d_lr.p),
                         reinterpret_cast<double2 *>(h.mat64.p), h.kpc, s);
        else launch_cur(dcj.p, (int)cj.size(), didx.p, h.d_lr.p, h.mat64.p, h.kp, s);
        H2W_HIP(hipGetLastError());
        H2W_HIP(hipStreamSynchronize(s));
    }
    phase("transfer operators");
    {
        // plain entry blocks: M2L, near field, semi-nested column factors
        std::vector<int32_t> idx;
        std::vector<EvalJob> ej;
        auto add = [&](const std::vector<int32_t> &r, const std::vector<int32_t> &c, int64_t off) {
            EvalJob J;
            J.m = (int32_t)r.size();
            J.n = (int32_t)c.size();
            J.lda = (int32_t)pad_ld(J.m);
            J.pad = 0;
            J.rows = (int64_t)idx.size();
            idx.insert(idx.end(), r.begin(), r.end());
            J.cols = (int64_t)idx.size();
            idx.insert(idx.end(), c.begin(), c.end());
            J.a = off;
            ej.push_back(J);
        };
        DevBuf<int32_t> didx;
        DevBuf<EvalJob> dej;
        auto flush = [&]() {
            if (ej.empty()) return;
            didx.upload(idx, s);
            dej.upload(ej, s);
            if (h.cplx) launch_eval_c(dej.p, (int)ej.size(), didx.p, reinterpret_cast<double2 *>(h.mat64.p), h.kpc, s);
            else launch_eval(dej.p, (int)ej.size(), didx.p, h.mat64.p, h.kp, s);
            H2W_HIP(hipGetLastError());
            H2W_HIP(hipStreamSynchronize(s));
            idx.clear();
            ej.clear();
        };
        for (auto &m : m2l) {
            add(h.fam[m.f][m.j].Ir[m.b], h.fam[m.f][m.j].Ir[m.p], m.off);
            if (idx.size() > ((size_t)64 << 20)) flush();
        }
        for (auto &nb : nearb) {
            add(range_list(P.bstart[P.nL][nb.b], P.bcount[P.nL][nb.b]),
                range_list(P.bstart[P.nL][nb.n], P.bcount[P.nL][nb.n]), nb.off);
            if (idx.size() > ((size_t)64 << 20)) flush();
        }
        for (auto &p : h.pairs) {
            if (p.rank == 0) continue;
            add(range_list(P.bstart[p.level][p.b], P.bcount[p.level][p.b]), p.Ic, p.ac_off);
            if (idx.size() > ((size_t)64 << 20)) flush();
        }
        flush();
    }
    phase("M2L / near / CUR blocks");
    if (h.opts.fp32_shadow) {
        h.mat32.alloc(h.mat_len);
        launch_to_fp32(h.mat64.p, h.mat32.p, h.mat_len, s);
        H2W_HIP(hipGetLastError());
    } else {
        h.mat32.release();
    }
    // ---- GEMV work lists, one per launch of the matvec
    std::vector<WorkList> WL;
    auto fam_up_item = [&](WorkList &W, int f, int j, int b, int64_t src) {
        FamLevel &fl = h.fam[f][j];
        if (fl.et_off[b] < 0) return;
        add_item(W, fl.o_off[b], fl.rank[b], {TermSpec{fl.et_off[b], src, (int32_t)fl.S[b].size()}}, false,
                 (int)pad_ld(fl.rank[b]));
    };
    // up, leaf level (and semi-nested row factors, which read x directly)
    {
        WorkList W;
        for (int f = 0; f < 2; ++f) {
            if (!fam_on[f] || P.nL < nfam_lo[f]) continue;
            for (int b = 0; b < P.nboxes[P.nL]; ++b) fam_up_item(W, f, P.nL, b, h.off_x + P.bstart[P.nL][b]);
        }
        for (auto &p : h.pairs)
            if (p.rank > 0)
                add_item(W, p.t_off, p.rank,
                         {TermSpec{p.ar_off, h.off_x + P.bstart[p.level][p.v], (int32_t)P.bcount[p.level][p.v]}},
                         false, (int)pad_ld(p.rank));
        WL.push_back(std::move(W));
    }
    // up, levels nL-1 .. 1 (the levels of a group in one launch)
    for (auto [T, B] : groups) {
        WorkList W;
        W.step = P.nL - (T - 1);
        for (int f = 0; f < 2; ++f) {
            if (!fam_on[f]) continue;
            for (int b = 0; T - 1 >= nfam_lo[f] && b < P.nboxes[T - 1]; ++b)
                fam_up_item(W, f, T - 1, b, h.fam[f][T].o_off[b * P.nchild]);
            for (int j = T - 2; j >= std::max(B, nfam_lo[f]); --j) {
                const FamLevel &fl = h.fam[f][j];
                for (int b = 0; b < fl.nb; ++b)
                    if (fl.ct_off[b] >= 0)
                        add_item(W, fl.o_off[b], fl.rank[b],
                                 {TermSpec{fl.ct_off[b], h.fam[f][T].o_off[first_at(b, j, T)],
                                           (int32_t)rank_at(f, b, j, T)}},
                                 false, (int)pad_ld(fl.rank[b]));
            }
        }
        WL.push_back(std::move(W));
    }
    // M2L (every level, both families) + near field, one block per unordered pair, both
    // directions in one fused launch
    {
        SymLists SL;
        for (int f = 0; f < 2; ++f) {
            if (!fam_on[f]) continue;
            for (int j = nfam_lo[f]; j <= P.nL; ++j) {
                FamLevel &fl = h.fam[f][j];
                SymGroup G;
                G.y.assign(fl.u_off.begin(), fl.u_off.end());
                G.x.assign(fl.o_off.begin(), fl.o_off.end());
                G.r = fl.rank;
                G.up.assign(fl.nb, {});
                G.self.assign(fl.nb, -1);
                for (auto &m : m2l)
                    if (m.f == f && m.j == j) G.up[m.b].push_back({m.p, m.off});
                sym_lists(G, SL);
            }
        }
        {
            SymGroup G;
            G.y.resize(nleaf);
            G.x.resize(nleaf);
            G.r.resize(nleaf);
            G.up.assign(nleaf, {});
            G.self.assign(nleaf, -1);
            for (int b = 0; b < nleaf; ++b) {
                G.y[b] = h.off_y + P.bstart[P.nL][b];
                G.x[b] = h.off_x + P.bstart[P.nL][b];
                G.r[b] = (int)P.bcount[P.nL][b];
            }
            for (auto &nb : nearb) {
                if (nb.n == nb.b) G.self[nb.b] = nb.off;
                else G.up[nb.b].push_back({nb.n, nb.off});
            }
            sym_lists(G, SL);
        }
        SL.fused.role = 1;
        SL.fused.stage = 1;
        WL.push_back(std::move(SL.fused));
        SL.trans.role = 3;
        SL.trans.stage = 1;
        SL.trans.step = 1;
        SL.otf.role = 1;
        SL.otf.stage = 1;
        std::vector<WorkList> tl, ol;
        tl.push_back(std::move(SL.trans));
        ol.push_back(std::move(SL.otf));
        upload_lists(tl, h.trans, false, s);
        upload_lists(ol, h.otf, false, s);
    }
    // down, levels 1 .. nL-1 (from the levels of a group in one launch)
    for (auto g = groups.rbegin(); g != groups.rend(); ++g) {
        const auto [T, B] = *g;
        WorkList W;
        W.stage = 2;
        W.step = P.nL - (T - 1);
        for (int f = 0; f < 2; ++f) {
            if (!fam_on[f] || T - 1 < nfam_lo[f]) continue;
            const FamLevel &fl = h.fam[f][T - 1], &ft = h.fam[f][T];
            if (B == T - 1) {
                for (int b = 0; b < fl.nb; ++b) {
                    if (fl.e_off[b] < 0) continue;
                    int64_t m = (int64_t)fl.S[b].size();
                    add_item(W, ft.u_off[b * P.nchild], (int)m,
                             {TermSpec{fl.e_off[b], fl.u_off[b], (int32_t)fl.rank[b]}}, false, (int)pad_ld(m));
                }
                continue;
            }
            for (int c = 0; c < ft.nb; ++c) {
                if (ft.c_off[c] < 0) continue;
                const int ld = (int)pad_ld(ft.rank[c]);
                std::vector<TermSpec> t;
                int64_t col = 0;
                for (int j = T - 1; j >= std::max(B, nfam_lo[f]); --j) {
                    const FamLevel &fa = h.fam[f][j];
                    const int a = ancestor(c, T, j);
                    if (fa.rank[a] > 0) t.push_back(TermSpec{ft.c_off[c] + col * ld, fa.u_off[a], (int32_t)fa.rank[a]});
                    col += fa.rank[a];
                }
                add_item(W, ft.u_off[c], ft.rank[c], t, false, ld);
            }
        }
        WL.push_back(std::move(W));
    }
    // down, leaf level: far + vertex into y
    {
        WorkList W;
        W.stage = 2;
        for (int b = 0; b < nleaf; ++b) {
            std::vector<TermSpec> t;
            for (int f = 0; f < 2; ++f) {
                if (!fam_on[f] || P.nL < nfam_lo[f]) continue;
                FamLevel &fl = h.fam[f][P.nL];
                if (fl.e_off[b] >= 0) t.push_back(TermSpec{fl.e_off[b], fl.u_off[b], (int32_t)fl.rank[b]});
            }
            add_item(W, h.off_y + P.bstart[P.nL][b], (int)P.bcount[P.nL][b], t, false,
                     (int)pad_ld(P.bcount[P.nL][b]));
        }
        WL.push_back(std::move(W));
    }
    // semi-nested column factors into y (boxes of all levels overlap: atomic)
    if (!h.pairs.empty()) {
        WorkList W;
        W.role = 2;
        W.stage = 3;
        std::vector<std::vector<std::vector<TermSpec>>> per(P.nL + 1);
        for (int j = 1; j <= P.nL; ++j) per[j].assign(P.nboxes[j], {});
        for (auto &p : h.pairs)
            if (p.rank > 0) per[p.level][p.b].push_back(TermSpec{p.ac_off, p.t_off, (int32_t)p.rank});
        for (int j = 1; j <= P.nL; ++j)
            for (int b = 0; b < P.nboxes[j]; ++b)
                add_item(W, h.off_y + P.bstart[j][b], (int)P.bcount[j][b], per[j][b], true,
                         (int)pad_ld(P.bcount[j][b]));
        WL.push_back(std::move(W));
    }
    std::vector<GItem> items;
    std::vector<GTerm> terms;
    for (auto &W : WL)
        rebalance(W);
    h.launches.clear();
    for (auto &W : WL) {
        if (W.items.empty()) continue;
        Launch Lh;
        Lh.item0 = (int64_t)items.size();
        Lh.nitems = (int64_t)W.items.size();
        Lh.term0 = (int64_t)terms.size();
        Lh.nterms = (int64_t)W.terms.size();
        Lh.role = W.role;
        Lh.stage = W.stage;
        Lh.step = W.step;
        for (auto it : W.items) {
            it.t0 += (int32_t)Lh.term0;
            it.t1 += (int32_t)Lh.term0;
            items.push_back(it);
        }
        terms.insert(terms.end(), W.terms.begin(), W.terms.end());
        Lh.set_wide(items, terms);
        h.launches.push_back(Lh);
    }
    h.d_items.upload(items, s);
    h.d_terms.upload(terms, s);
    h.h_items = items;
    h.h_terms = terms;
    int64_t se = 0;
    h.launch_elems.assign(h.launches.size(), 0);
    for (size_t q = 0; q < h.launches.size(); ++q) {
        const Launch &Lh = h.launches[q];
        for (int64_t i = Lh.item0; i < Lh.item0 + Lh.nitems; ++i)
            for (int t = items[i].t0; t < items[i].t1; ++t) h.launch_elems[q] += (int64_t)items[i].rows * terms[t].cols;
        h.launches[q].avg_item_elems = h.launch_elems[q] / Lh.nitems;
        se += h.launch_elems[q];
    }
    h.stored_elems = se;
    build_inner(h, (double)h.opts.ir_tol_pow);
    H2W_HIP(hipStreamSynchronize(s));
    h.d_lr.release();
    phase("work lists");
    if (verbose)
        std::fprintf(stderr, "[h2w] memory %.0f elements (%.3f GB fp64), pool %.3f GB, %zu launches, %zu items\n",
                     h.memory, h.memory * 8e-9, h.mat_len * 8e-9, h.launches.size(), items.size());
    h.assembled = true;
    h.assembly_seconds = now_s() - t0;
}

// ------------------------------------------------------------------ matvec
// y_tree = A x_tree inside the vector pool (x already at off_x)
}  // namespace

int64_t LrForm::add(const int32_t *Ir, const int32_t *Ic, int k) {
    LrFormJob J;
    J.ir = (int64_t)idx.size();
    idx.insert(idx.end(), Ir, Ir + k);
    J.ic = (int64_t)idx.size();
    idx.insert(idx.end(), Ic, Ic + k);
    J.out = len;
    J.k = k;
    J.pad = 0;
    len += 2LL * k * k;
    jobs.push_back(J);
    return J.out;
}
void LrForm::run(const Handle &h, hipStream_t s) {
    if (jobs.empty()) return;
    d_jobs.upload(jobs, s);
    d_idx.upload(idx, s);
    out.ensure(len);
    launch_lr_form(d_jobs.p, (int)jobs.size(), d_idx.p, out.p, h.kp, s);
    H2W_HIP(hipGetLastError());
}
void LrForm::clear() {
    jobs.clear();
    idx.clear();
    len = 0;
}

// operator phase of the assembly from skeletons already in the handle (loading a saved operator)
void rebuild_operators(Handle &h) {
    drop_graphs(h);
    DevBuf<double> scratch;
    assemble_operators(h, now_s(), scratch);
}

bool is32(int precision) { return precision == H2W_FP32 || precision == H2W_FP32_OTF || precision == H2W_FP32_INNER; }

// Stage 1 is one fused launch (role 1): every stored block K(b, p), p >= b, applied to
// x_p, and its transpose to x_b with the product added to y_p.  The on-the-fly
// precisions evaluate the blocks from the points instead, over the directed lists.
void run_launch(Handle &h, const Launch &Lh, int precision) {
    hipStream_t s = h.stream;
    if (h.cplx) {  // complex operators: FP64 only, every role through the complex GEMV
        launch_cgemv(h.d_items.p + Lh.item0, (int)Lh.nitems, h.d_terms.p, reinterpret_cast<const double2 *>(h.mat64.p),
                     reinterpret_cast<double2 *>(h.vec64.p), Lh.role, per_wave_gemv(Lh), s);
        return;
    }
    const bool otf = (precision == H2W_FP32_OTF || precision == H2W_FP64_OTF) && Lh.role == 1;
    if (otf) {
        for (auto &Lo : h.otf.launches) {
            if (is32(precision))
                launch_otf32(h.otf.d_items.p + Lo.item0, (int)Lo.nitems, h.otf.d_terms.p, h.sp, h.vec32.p, s);
            else
                launch_otf64(h.otf.d_items.p + Lo.item0, (int)Lo.nitems, h.otf.d_terms.p, h.sp, h.vec64.p, s);
        }
        return;
    }
    const bool in = precision == H2W_FP32_INNER;
    const GItem *items = (in ? h.inner.d_items.p : h.d_items.p) + Lh.item0;
    const GTerm *terms = in ? h.inner.d_terms.p : h.d_terms.p;
    const bool pw = per_wave_gemv(Lh);
    if (in) launch_bgemv32(items, (int)Lh.nitems, terms, h.mat32.p, h.mat32in.p, h.vec32.p, Lh.role, Lh.unr, pw, s);
    else if (is32(precision))
        launch_bgemv32(items, (int)Lh.nitems, terms, h.mat32.p, nullptr, h.vec32.p, Lh.role, Lh.unr32, pw, s);
    else launch_bgemv64(items, (int)Lh.nitems, terms, h.mat64.p, nullptr, h.vec64.p, Lh.role, Lh.unr, pw, s);
}

void zero_outputs(Handle &h, int precision) {
    if (h.cplx) launch_cfill(reinterpret_cast<double2 *>(h.vec64.p) + h.off_y, h.vec_len - h.off_y, h.stream);
    else if (is32(precision)) launch_fill32(h.vec32.p + h.off_y, h.vec_len - h.off_y, 0.0f, h.stream);
    else launch_fill(h.vec64.p + h.off_y, h.vec_len - h.off_y, 0.0, h.stream);
}

const std::vector<Launch> &launches_for(Handle &h, int precision) {
    if (precision == H2W_FP32_INNER) {
        if (h.inner.launches.empty()) throw Error{H2W_ESTATE, "the inner operator was not built (opts.ir_tol_pow)"};
        return h.inner.launches;
    }
    return h.launches;
}

void run_launches_eager(Handle &h, int precision) {
    for (auto &Lh : launches_for(h, precision)) run_launch(h, Lh, precision);
    H2W_HIP(hipGetLastError());
}

// The launch sequence of a matvec is fixed per handle and precision (pool pointers and work
// lists do not change after assembly), so it is captured once into a HIP graph and replayed.
// Every node is a kernel.  The outputs are zeroed before it (with the input, in one kernel, or
// by zero_outputs).
// A replay costs the host about 6 us more than its first kernel alone, each plain launch 4.7 us, which pass
// while the GPU works on the launches before it: the graph is for sequences that run faster than the host
// can launch them.  (Plain launches against replays, whole products: 1D N = 2048, 5 launches 37 / 45 us, its
// inner operator's 11 launches 81 / 64 us; 3D N = 20011 220 / 224 us.)
bool replay_pays(Handle &h, int precision) {
    const auto &L = launches_for(h, precision);
    const auto &e = precision == H2W_FP32_INNER ? h.inner.elems : h.launch_elems;
    const double bytes = h.cplx ? 16.0 : is32(precision) ? 4.0 : 8.0;
    double gpu = 6.0;
    for (size_t q = 0; q < L.size(); ++q) gpu += std::max(3.5, (double)e[q] * bytes / 5.0e6);
    return 4.7 * (double)L.size() > gpu;
}
void run_launches(Handle &h, int precision) {
    if (!h.use_graph || !replay_pays(h, precision)) {
        run_launches_eager(h, precision);
        return;
    }
    if (!h.graph[precision]) {
        hipGraph_t g = nullptr;
        H2W_HIP(hipStreamBeginCapture(h.stream, hipStreamCaptureModeThreadLocal));
        try {
            run_launches_eager(h, precision);
        } catch (...) {
            (void)hipStreamEndCapture(h.stream, &g);
            if (g) (void)hipGraphDestroy(g);
            throw;
        }
        H2W_HIP(hipStreamEndCapture(h.stream, &g));
        hipGraphExec_t ex = nullptr;
        hipError_t e = hipGraphInstantiate(&ex, g, nullptr, nullptr, 0);
        (void)hipGraphDestroy(g);
        if (e != hipSuccess) throw Error{H2W_EHIP, std::string("hipGraphInstantiate: ") + hipGetErrorString(e)};
        h.graph[precision] = ex;
    }
    H2W_HIP(hipGraphLaunch(h.graph[precision], h.stream));
}

// graphs of the single-vector and the kNR-wide matvec.  The stream is drained first, so no
// replay of an exec is in flight when it is destroyed, and callers that go on to free or
// reallocate the buffers it read (build_inner) free idle memory.
void drop_graph(Handle &h, int precision) {
    if (!h.graph[precision] && !h.graph_m[precision]) return;
    if (h.stream) (void)hipStreamSynchronize(h.stream);  // (also on error paths: never throws)
    for (hipGraphExec_t *g : {&h.graph[precision], &h.graph_m[precision]})
        if (*g) {
            (void)hipGraphExecDestroy(*g);
            *g = nullptr;
        }
}

void drop_graphs(Handle &h) {
    for (int p = 0; p < 5; ++p) drop_graph(h, p);
}

// pool input (scale x, or x / sqrt(*norm2); tree order, kept at copy too) and zeroed outputs of a product
// (real kernels)
void begin_product(Handle &h, const double *x, double scale, const double *norm2, double *copy, int precision) {
    const int64_t len = h.vec_len - h.off_y;
    if (is32(precision))
        launch_begin32(x, scale, norm2, copy, nullptr, h.vec32.p + h.off_x, h.N, h.vec32.p + h.off_y, len, h.stream);
    else
        launch_begin64(x, scale, norm2, copy, nullptr, h.vec64.p + h.off_x, h.N, h.vec64.p + h.off_y, len, h.stream);
}

// device-pointer matvec on one vector; tree-ordered in/out when tree == true
void matvec_dev(Handle &h, const double *x, double *y, int precision, bool tree) {
    hipStream_t s = h.stream;
    const int64_t N = h.N;
    if (h.cplx) {
        // complex vectors: N (re, im) pairs
        if (precision != H2W_FP64) throw Error{H2W_EINVAL, "complex kernels: precision H2W_FP64 only"};
        double2 *pool = reinterpret_cast<double2 *>(h.vec64.p);
        const double2 *xc = reinterpret_cast<const double2 *>(x);
        double2 *yc = reinterpret_cast<double2 *>(y);
        launch_cbegin(xc, tree ? nullptr : h.d_perm.p, pool + h.off_x, N, pool + h.off_y, h.vec_len - h.off_y, s);
        run_launches(h, precision);
        if (tree) H2W_HIP(hipMemcpyAsync(yc, pool + h.off_y, N * 16, hipMemcpyDeviceToDevice, s));
        else launch_cpermute_out(pool + h.off_y, yc, h.d_perm.p, N, s);
        H2W_HIP(hipGetLastError());
        return;
    }
    if (is32(precision)) {
        if (!h.mat32.p) throw Error{H2W_ESTATE, "FP32 matvec requested but the FP32 shadow was not built"};
        launch_begin32(x, 1.0, nullptr, nullptr, tree ? nullptr : h.d_perm.p, h.vec32.p + h.off_x, N, h.vec32.p + h.off_y, h.vec_len - h.off_y,
                       s);
        run_launches(h, precision);
        if (tree) launch_to_fp64(h.vec32.p + h.off_y, y, N, s);
        else launch_permute_out32(h.vec32.p + h.off_y, N, y, N, h.d_perm.p, N, 1, s);
    } else {
        launch_begin64(x, 1.0, nullptr, nullptr, tree ? nullptr : h.d_perm.p, h.vec64.p + h.off_x, N, h.vec64.p + h.off_y, h.vec_len - h.off_y,
                       s);
        run_launches(h, precision);
        if (tree) H2W_HIP(hipMemcpyAsync(y, h.vec64.p + h.off_y, N * 8, hipMemcpyDeviceToDevice, s));
        else launch_permute_out(h.vec64.p + h.off_y, N, y, N, h.d_perm.p, N, 1, s);
    }
    H2W_HIP(hipGetLastError());
}

}  // namespace h2w

namespace h2w {
namespace {

// ------------------------------------------------------------------ GMRES (tree order, device vectors)
// Unrestarted GMRES as the reference's iterative_solver::GMRES (1D/codes/gmres.hpp:91-200):
// restart = max_iter, Givens rotations (:30-75), resid = |s_{i+1}| / ||b|| (:162),
// back-substitution update (:77-90).  The Arnoldi step orthogonalises with
// classical Gram-Schmidt applied twice (two fused passes over the basis instead
// of the reference's i+1 dependent modified Gram-Schmidt steps); all of it FP64.
struct GmresOut {
    int iters = 0;
    double resid = 0.0;
    bool conv = false;
    int matvecs = 0;
    std::vector<std::vector<double>> H;  // Hessenberg columns (rows 0..j+1) of a plain solve
};

// A space kept from one correction of the refinement for the next ones (same operator):
// C = A U with orthonormal C, k columns; C sits in the first k columns of the GMRES basis
// buffer, so that one fused pass orthogonalises against C and the new Arnoldi vectors.
struct Recycled {
    int k = 0;
    // C spans approximate eigenvectors (a deflation space): C^T A v is small for v orthogonal to C,
    // so the second Gram-Schmidt pass is taken against the new Arnoldi vectors only
    bool invariant = false;
};

void ensure_V(Handle &h, int64_t cols) {
    if (cols <= h.g_Vcols) return;
    int64_t nc = std::max<int64_t>(cols, std::max<int64_t>(16, h.g_Vcols * 2));
    double *np = nullptr;
    if (hipMalloc(&np, (size_t)nc * h.N * 8) != hipSuccess) throw Error{H2W_ENOMEM, "GMRES basis allocation failed"};
    if (h.g_Vcols > 0)
        H2W_HIP(hipMemcpyAsync(np, h.g_V.p, (size_t)h.g_Vcols * h.N * 8, hipMemcpyDeviceToDevice, h.stream));
    H2W_HIP(hipStreamSynchronize(h.stream));
    h.g_V.release();
    h.g_V.p = np;
    h.g_V.n = (size_t)nc * h.N;
    h.g_Vcols = nc;
}

// work arrays of the Arnoldi passes for up to k columns
CgsArgs cgs_args(Handle &h, double *w, int64_t k) {
    if (!h.g_cnt.p) {
        h.g_cnt.alloc(1);
        H2W_HIP(hipMemsetAsync(h.g_cnt.p, 0, 4, h.stream));
    }
    h.g_part.ensure((size_t)cgs_blocks(h.N) * std::max<int64_t>(k, 1));
    CgsArgs a;
    a.V = nullptr;
    a.ldv = a.n = h.N;
    a.w = w;
    a.partial = h.g_part.p;
    a.arrived = h.g_cnt.p;
    a.out = nullptr;
    return a;
}

// A pass whose results go to the host, and the wait for them: a poll of the flag that the pass writes last,
// in page-locked memory, with a look at the stream now and then (an error there, or a stream that ended
// without the flag, ends the wait).
void launch_cgs_host(Handle &h, CgsArgs &a) {
    if (!h.g_flag.p) {
        h.g_flag.ensure(1);
        std::memset(h.g_flag.p, 0, sizeof(uint64_t));
    }
    a.flag = reinterpret_cast<uint64_t *>(h.g_flag.p);
    a.seq = ++h.g_seq;
    launch_cgs(a, h.stream);
    H2W_HIP(hipGetLastError());
}
void wait_cgs_host(Handle &h) {
    const volatile uint64_t *f = reinterpret_cast<const volatile uint64_t *>(h.g_flag.p);
    for (int64_t spin = 1; *f < h.g_seq; ++spin) {
        if (spin % 16384 != 0) continue;
        const hipError_t e = hipStreamQuery(h.stream);
        if (e == hipErrorNotReady) continue;
        H2W_HIP(e);
        if (*f < h.g_seq) throw Error{H2W_EHIP, "an Arnoldi pass ended without its results"};
    }
    std::atomic_thread_fence(std::memory_order_acquire);
}

// a . b (b == nullptr: a . a), read back through page-locked memory; neither is written
double dev_dot(Handle &h, const double *a, const double *b) {
    CgsArgs c = cgs_args(h, const_cast<double *>(a), 1);
    h.g_h.ensure(8);
    c.V = b;
    c.nd = b ? 1 : 0;
    c.norm = !b;
    c.out = h.g_h.p;
    c.host = h.g_pin.ensure(8);
    c.all_h = h.g_h.p;
    c.nhost = 1;  // (out follows at host[1])
    launch_cgs_host(h, c);
    wait_cgs_host(h);
    return h.g_pin.p[1];
}

double dev_norm(Handle &h, const double *v) { return std::sqrt(dev_dot(h, v, nullptr)); }

// Solves A x = b (tree order, device).  x_zero: x0 = 0 and no initial matvec.
// normb_in > 0 overrides ||b|| in the stopping test.
GmresOut gmres_core(Handle &h, const double *b, double *x, int max_iter, double tol, int prec, bool x_zero,
                    double normb_in, const Recycled *rc = nullptr, bool keep_h = false) {
    const int64_t N = h.N;
    hipStream_t s = h.stream;
    GmresOut out;
    h.g_w.ensure(N);
    h.g_b.ensure(N);  // residual of this solve
    double *r = h.g_b.p;
    double normb = normb_in > 0 ? normb_in : dev_norm(h, b);
    // recycled space (x starts at zero): x = U C^T r, r -= C C^T r, and every Arnoldi vector is
    // orthogonalised against C as well (its coefficients B = C^T A v_j enter the update of x)
    const int kc = rc && x_zero ? rc->k : 0;
    const bool once = kc > 0 && rc->invariant;
    if (!once) h.gv_defl = -1;  // (its basis overwrites the first columns of g_V)
    const int m = max_iter;
    CgsArgs A = cgs_args(h, r, kc + std::min<int64_t>(m + 1, 32));  // (grows with the basis)
    h.g_h.ensure((size_t)2 * (kc + m + 2) + 2);
    double *hh = h.g_pin.ensure(2 * (kc + m + 2) + 8);
    if (x_zero) {
        H2W_HIP(hipMemcpyAsync(r, b, N * 8, hipMemcpyDeviceToDevice, s));
    } else {
        matvec_dev(h, x, h.g_w.p, prec, true);
        out.matvecs++;
        H2W_HIP(hipMemcpyAsync(r, b, N * 8, hipMemcpyDeviceToDevice, s));
        launch_axpby(-1.0, h.g_w.p, 1.0, r, N, s);
    }
    double beta;
    if (kc > 0) {
        A.V = h.g_V.p;
        A.nd = kc;
        A.out = h.g_h.p;
        launch_cgs(A, s);  // C^T r
        launch_vec_update(h.g_U.p, N, kc, h.g_h.p, x, N, s);
        CgsArgs B = A;
        B.ns = kc;
        B.sub = h.g_h.p;
        B.norm = 1;
        B.out = h.g_h.p + kc;
        B.all_h = h.g_h.p;
        B.nhost = 1;
        B.host = hh;
        launch_cgs_host(h, B);  // r -= C C^T r, and its norm
        wait_cgs_host(h);
        beta = std::sqrt(hh[1]);
    } else {
        beta = dev_norm(h, r);
    }
    if (normb == 0.0) normb = 1;
    out.resid = beta / normb;
    if (out.resid <= tol) {
        out.conv = true;
        return out;
    }
    std::vector<std::vector<double>> H;  // Hessenberg columns as they are produced (rows 0..j+1)
    std::vector<std::vector<double>> Bc; // (recycled) C^T A v_j
    std::vector<double> sv(m + 1, 0.0), cs(m + 1, 0.0), sn(m + 1, 0.0);
    auto Hh = [&](int i, int j) -> double & { return H[j][i]; };
    ensure_V(h, kc + std::min<int64_t>(m + 1, 32));
    sv[0] = beta;
    const double *next = r;  // v_i = next scale
    double scale = 1.0 / beta;
    // The product of step i + 1 needs the norm of step i's vector only, which the device has: it is queued
    // before the host has read step i's coefficients, unless the residual, shrinking as it did in the step
    // before, would reach the tolerance (a product too many costs more than the idle time it hides).
    bool ahead = false;
    double res1 = out.resid, res2 = 0.0;  // residuals of the last two steps
    for (int i = 0; i < m; ++i) {
        ensure_V(h, kc + i + 3);
        A.partial = cgs_args(h, r, h.g_Vcols).partial;
        double *C = h.g_V.p, *V = h.g_V.p + (int64_t)kc * N;
        // w = A v_i: left in the pool (FP64) or taken from there by the first pass (FP32)
        const bool f32 = is32(prec);
        if (!ahead) {
            begin_product(h, next, scale, nullptr, V + (int64_t)i * N, prec);
            run_launches(h, prec);
        }
        out.matvecs++;
        double *w = f32 ? h.g_w.p : h.vec64.p + h.off_y;
        const int k = kc + i + 1;  // vectors orthogonalised against: C, v_0 .. v_i (contiguous)
        // second pass: against C as well, or (a deflation space) against v_0 .. v_i only
        const int k0 = once ? kc : 0;
        A.V = C;
        A.w = w;
        A.src32 = f32 ? h.vec32.p + h.off_y : nullptr;
        A.nd = k;
        A.out = h.g_h.p;
        launch_cgs(A, s);  // h = V^T w
        CgsArgs B = A;
        B.src32 = nullptr;
        B.ns = k;
        B.sub = h.g_h.p;
        B.d0 = k0;
        B.nd = k - k0;
        B.out = h.g_h.p + k + k0;
        if (f32) B.w = w;
        launch_cgs(B, s);  // w -= V h, second dots
        B.s0 = k0;
        B.ns = k - k0;
        B.sub = h.g_h.p + k + k0;
        B.norm = 1;
        B.out = h.g_h.p + 2 * k;
        B.all_h = h.g_h.p;
        B.nhost = 2 * k;
        B.host = hh;
        launch_cgs_host(h, B);  // w -= V h, norm; all of it to the host
        const double guess = res2 > res1 ? res1 * (res1 / res2) : res1;
        ahead = i + 1 < m && !(guess < tol);
        if (ahead) {
            begin_product(h, w, 1.0, h.g_h.p + 2 * k, V + (int64_t)(i + 1) * N, prec);
            run_launches(h, prec);
        }
        wait_cgs_host(h);
        for (int q = 0; q < k0; ++q) hh[k + q] = 0.0;
        if (kc > 0) {
            Bc.emplace_back(kc);
            for (int q = 0; q < kc; ++q) Bc.back()[q] = hh[q] + hh[k + q];
        }
        H.emplace_back(i + 2, 0.0);
        for (int q = 0; q <= i; ++q) Hh(q, i) = hh[kc + q] + hh[k + kc + q];
        Hh(i + 1, i) = std::sqrt(hh[2 * k]);
        if (keep_h) out.H.push_back(H.back());  // (before the rotations)
        // H(i+1, i) = 0: the Krylov space is invariant and the least-squares solution is exact
        // (the reference's gap, 1D/codes/gmres.hpp:153-154, divides by it); the next basis
        // vector is left zero, the rotation below leaves s_{i+1} = 0 and the solve ends here
        const bool breakdown = !(Hh(i + 1, i) > 0.0);
        next = w;
        scale = breakdown ? 0.0 : 1.0 / Hh(i + 1, i);
        for (int q = 0; q < i; ++q) app_rot(Hh(q, i), Hh(q + 1, i), cs[q], sn[q]);
        gen_rot(Hh(i, i), Hh(i + 1, i), cs[i], sn[i]);
        app_rot(Hh(i, i), Hh(i + 1, i), cs[i], sn[i]);
        app_rot(sv[i], sv[i + 1], cs[i], sn[i]);
        out.resid = std::fabs(sv[i + 1]) / normb;
        out.iters = i + 1;
        res2 = res1;
        res1 = out.resid;
        bool done = out.resid < tol || i == m - 1 || breakdown;
        if (done) {
            // (the next basis vector, for a space kept from this solve)
            if (keep_h && breakdown) launch_fill(V + (int64_t)(i + 1) * N, N, 0.0, s);
            else if (keep_h && !ahead) launch_axpby(scale, w, 0.0, V + (int64_t)(i + 1) * N, N, s);
            std::vector<double> y(sv.begin(), sv.begin() + i + 1);
            for (int q = i; q >= 0; q--) {
                y[q] /= Hh(q, q);
                for (int jj = q - 1; jj >= 0; jj--) y[jj] -= Hh(jj, q) * y[q];
            }
            // x += V y - U (B y)
            std::vector<double> cy(y);
            if (kc > 0) {
                cy.resize(i + 1 + kc, 0.0);
                for (int jj = 0; jj <= i; ++jj)
                    for (int q = 0; q < kc; ++q) cy[i + 1 + q] -= Bc[jj][q] * y[jj];
            }
            H2W_HIP(hipMemcpyAsync(h.g_h.p, cy.data(), cy.size() * 8, hipMemcpyHostToDevice, s));
            launch_vec_update(V, N, i + 1, h.g_h.p, x, N, s);
            if (kc > 0) launch_vec_update(h.g_U.p, N, kc, h.g_h.p + i + 1, x, N, s);
            H2W_HIP(hipStreamSynchronize(s));
            out.conv = out.resid < tol || (breakdown && out.resid == 0.0);
            return out;
        }
    }
    return out;
}

// The space of a finished correction kept for the next ones: with the Arnoldi relation
// A V_j = V_{j+1} Hbar, a selection V_j S of its space (S: j x k, the whole space when S is null,
// S = I) has A V_j S = V_{j+1} Z with Z = Hbar S; with Z = Q R (thin QR, host) U = V_j S R^-1 and
// C = V_{j+1} Q satisfy A U = C with orthonormal C.  C replaces the first k basis columns, U goes
// to g_U.  Returns false (nothing kept) for fewer than two iterations or a near-singular R.
bool keep_space(Handle &h, const GmresOut &o, Recycled &rc, const std::vector<std::vector<double>> *S = nullptr) {
    rc.k = 0;
    h.gv_defl = -1;
    const int j = (int)o.H.size();
    if (j < 2 || o.iters != j) return false;
    const int kk = S ? (int)S->size() : j;
    if (kk < 1) return false;
    const int64_t N = h.N;
    hipStream_t s = h.stream;
    // Z columns (j+1 rows), Gram-Schmidt twice in double
    std::vector<std::vector<double>> Q(kk, std::vector<double>(j + 1, 0.0));
    std::vector<std::vector<double>> R(kk, std::vector<double>(kk, 0.0));  // R[col][row]
    for (int c = 0; c < kk; ++c) {
        std::vector<double> v(j + 1, 0.0);
        if (S) {
            for (int t = 0; t < j; ++t) {
                const double sc = (*S)[c][t];
                for (int q = 0; q < (int)o.H[t].size() && q <= j; ++q) v[q] += o.H[t][q] * sc;
            }
        } else {
            for (int q = 0; q < (int)o.H[c].size() && q <= j; ++q) v[q] = o.H[c][q];
        }
        for (int pass = 0; pass < 2; ++pass)
            for (int p = 0; p < c; ++p) {
                double d = 0.0;
                for (int q = 0; q <= j; ++q) d += Q[p][q] * v[q];
                for (int q = 0; q <= j; ++q) v[q] -= d * Q[p][q];
                R[c][p] += d;
            }
        double nv = 0.0;
        for (int q = 0; q <= j; ++q) nv += v[q] * v[q];
        nv = std::sqrt(nv);
        const double ref = c == 0 ? nv : R[0][0];
        if (!std::isfinite(nv) || !(nv > 1e-12 * ref)) return false;
        R[c][c] = nv;
        for (int q = 0; q <= j; ++q) Q[c][q] = v[q] / nv;
    }
    // Rinv (upper triangular), column by column: R Rinv[:, c] = e_c
    std::vector<std::vector<double>> Ri(kk, std::vector<double>(kk, 0.0));
    for (int c = 0; c < kk; ++c)
        for (int q = c; q >= 0; --q) {
            double v = q == c ? 1.0 : 0.0;
            for (int p = q + 1; p <= c; ++p) v -= R[p][q] * Ri[c][p];
            Ri[c][q] = v / R[q][q];
        }
    // coefficients: C_c = V Q[:, c] (j+1 terms), U_c = V S Ri[:, c] (j terms, padded to j+1)
    std::vector<double> coef((size_t)2 * kk * (j + 1), 0.0);
    for (int c = 0; c < kk; ++c) {
        for (int q = 0; q <= j; ++q) coef[(size_t)c * (j + 1) + q] = Q[c][q];
        double *u = coef.data() + (size_t)(kk + c) * (j + 1);
        for (int p = 0; p <= c; ++p) {
            if (S)
                for (int q = 0; q < j; ++q) u[q] += (*S)[p][q] * Ri[c][p];
            else
                u[p] = Ri[c][p];
        }
    }
    h.g_coef.ensure(coef.size());
    H2W_HIP(hipMemcpyAsync(h.g_coef.p, coef.data(), coef.size() * 8, hipMemcpyHostToDevice, s));
    h.g_U.ensure((size_t)2 * kk * N);  // U, then C before it moves into the basis
    launch_fill(h.g_U.p, 2 * kk * N, 0.0, s);
    for (int c = 0; c < kk; ++c) {
        launch_vec_update(h.g_V.p, N, j + 1, h.g_coef.p + (size_t)c * (j + 1), h.g_U.p + (int64_t)(kk + c) * N, N, s);
        launch_vec_update(h.g_V.p, N, j + 1, h.g_coef.p + (size_t)(kk + c) * (j + 1), h.g_U.p + (int64_t)c * N, N, s);
    }
    H2W_HIP(hipMemcpyAsync(h.g_V.p, h.g_U.p + (int64_t)kk * N, (size_t)kk * N * 8, hipMemcpyDeviceToDevice, s));
    H2W_HIP(hipGetLastError());
    // (the coefficients must outlive the copy: wait before the host vector goes)
    H2W_HIP(hipStreamSynchronize(s));
    rc.k = kk;
    return true;
}

// Eigen-decomposition of the symmetric n x n matrix a (row-major, destroyed): Householder reduction
// to tridiagonal form T = Q^T A Q, then implicit QL iterations with shifts on T, the rotations
// accumulated into Q.  Eigenvalues in w, eigenvectors as the columns of z (row-major).
void sym_eig(std::vector<double> &a, int n, std::vector<double> &w, std::vector<double> &z) {
    auto A = [&](int i, int j) -> double & { return a[(size_t)i * n + j]; };
    z.assign((size_t)n * n, 0.0);
    for (int i = 0; i < n; ++i) z[(size_t)i * n + i] = 1.0;
    std::vector<double> v(n), p(n), e(n, 0.0);
    // Householder: column k below the subdiagonal is zeroed by H = I - 2 v v^T on rows/cols k+1..n-1
    for (int k = 0; k + 2 < n; ++k) {
        double nx = 0.0;
        for (int i = k + 1; i < n; ++i) nx += A(i, k) * A(i, k);
        nx = std::sqrt(nx);
        if (nx == 0.0) continue;
        const double alpha = A(k + 1, k) > 0 ? -nx : nx;
        for (int i = k + 1; i < n; ++i) v[i] = A(i, k);
        v[k + 1] -= alpha;
        double nv = 0.0;
        for (int i = k + 1; i < n; ++i) nv += v[i] * v[i];
        nv = std::sqrt(nv);
        if (nv == 0.0) continue;
        for (int i = k + 1; i < n; ++i) v[i] /= nv;
        // p = A_sub v, K = v^T p, q = p - K v; A_sub -= 2 (v q^T + q v^T)
        double K = 0.0;
        for (int i = k + 1; i < n; ++i) {
            double s = 0.0;
            for (int j = k + 1; j < n; ++j) s += A(i, j) * v[j];
            p[i] = s;
            K += v[i] * s;
        }
        for (int i = k + 1; i < n; ++i) p[i] -= K * v[i];
        for (int i = k + 1; i < n; ++i)
            for (int j = k + 1; j < n; ++j) A(i, j) -= 2.0 * (v[i] * p[j] + p[i] * v[j]);
        A(k + 1, k) = A(k, k + 1) = alpha;
        for (int i = k + 2; i < n; ++i) A(i, k) = A(k, i) = 0.0;
        // Q <- Q H: Q[:, k+1:] -= 2 (Q[:, k+1:] v) v^T
        for (int r = 0; r < n; ++r) {
            double s = 0.0;
            for (int j = k + 1; j < n; ++j) s += z[(size_t)r * n + j] * v[j];
            s *= 2.0;
            for (int j = k + 1; j < n; ++j) z[(size_t)r * n + j] -= s * v[j];
        }
    }
    w.resize(n);
    for (int i = 0; i < n; ++i) w[i] = A(i, i);
    for (int i = 0; i + 1 < n; ++i) e[i] = A(i + 1, i);
    e[n - 1] = 0.0;
    // implicit QL with Wilkinson-type shifts: eigenvalue l converges when e[l] vanishes
    const double eps = 2.220446049250313e-16;
    for (int l = 0; l < n; ++l) {
        for (int iter = 0; iter < 60; ++iter) {
            int m = l;
            for (; m + 1 < n; ++m) {
                const double dd = std::fabs(w[m]) + std::fabs(w[m + 1]);
                if (std::fabs(e[m]) <= eps * dd) break;
            }
            if (m == l) break;
            // shift from the leading 2 x 2 block at l
            double g = (w[l + 1] - w[l]) / (2.0 * e[l]);
            double r = std::hypot(g, 1.0);
            g = w[m] - w[l] + e[l] / (g + (g >= 0 ? r : -r));
            double s = 1.0, c = 1.0, pp = 0.0;
            int i = m - 1;
            bool under = false;
            for (; i >= l; --i) {
                double f = s * e[i], b = c * e[i];
                r = std::hypot(f, g);
                e[i + 1] = r;
                if (r == 0.0) {  // (underflow: split here)
                    w[i + 1] -= pp;
                    e[m] = 0.0;
                    under = true;
                    break;
                }
                s = f / r;
                c = g / r;
                g = w[i + 1] - pp;
                r = (w[i] - g) * s + 2.0 * c * b;
                pp = s * r;
                w[i + 1] = g + pp;
                g = c * r - b;
                for (int k = 0; k < n; ++k) {
                    const double zi1 = z[(size_t)k * n + i + 1], zi = z[(size_t)k * n + i];
                    z[(size_t)k * n + i + 1] = s * zi + c * zi1;
                    z[(size_t)k * n + i] = c * zi - s * zi1;
                }
            }
            if (under) continue;
            w[l] -= pp;
            e[l] = g;
            e[m] = 0.0;
        }
    }
}

// The deflation space of the refinement's inner operator: m Arnoldi steps of that operator from a
// fixed pseudo-random vector (independent of any right-hand side).  A Krylov space of a generic
// vector holds good approximations of the operator's outlying eigenvectors, so a correction that
// starts from it (x = U C^T r, every Arnoldi vector orthogonalised against C) needs fewer steps.
// k = 0 keeps the whole space (U = V_m R^-1, C = V_{m+1} Q, as keep_space keeps a correction's
// space); 0 < k < m keeps the k Ritz vectors (eigenvectors of the symmetric part of H_m) whose
// Ritz values lie farthest from the diagonal value d: the operators here are d I plus a kernel
// matrix, their spectrum clusters at d and GMRES spends its steps on the eigenvalues away from it,
// so those k vectors give nearly the reduction of the whole space at k/m of the orthogonalisation
// cost per step.  m = 0 drops the space.
void build_deflation(Handle &h, int m, int k, int prec) {
    const int64_t N = h.N;
    hipStream_t s = h.stream;
    H2W_HIP(hipStreamSynchronize(s));
    h.defl_k = 0;
    h.defl_prec = -1;
    ++h.defl_serial;
    h.g_defl.release();
    h.g_defl_rm.release();
    if (m <= 0) return;
    std::vector<double> v(N);
    uint64_t st = 0x9e3779b97f4a7c15ull;
    for (int64_t i = 0; i < N; ++i) {  // splitmix64, uniform in [-1, 1)
        uint64_t z = (st += 0x9e3779b97f4a7c15ull);
        z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
        z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
        z ^= z >> 31;
        v[i] = (double)(z >> 11) * (2.0 / 9007199254740992.0) - 1.0;
    }
    h.g_r.ensure(N);
    h.g_d.ensure(N);
    H2W_HIP(hipMemcpyAsync(h.g_r.p, v.data(), N * 8, hipMemcpyHostToDevice, s));
    launch_fill(h.g_d.p, N, 0.0, s);
    // tol 0: exactly m steps unless the space becomes invariant first
    GmresOut o = gmres_core(h, h.g_r.p, h.g_d.p, m, 0.0, prec, true, -1.0, nullptr, true);
    Recycled rc;
    const int j = (int)o.H.size();
    std::vector<std::vector<double>> S;
    if (k > 0 && k < j) {
        // symmetric part of H_j (the operator is symmetric; its FP32 products are so up to rounding)
        std::vector<double> T((size_t)j * j, 0.0), w, Z;
        for (int c = 0; c < j; ++c)
            for (int q = 0; q < (int)o.H[c].size() && q < j; ++q) {
                T[(size_t)q * j + c] += 0.5 * o.H[c][q];
                T[(size_t)c * j + q] += 0.5 * o.H[c][q];
            }
        sym_eig(T, j, w, Z);
        std::vector<int> idx(j);
        for (int i = 0; i < j; ++i) idx[i] = i;
        const double d = h.diag;
        std::stable_sort(idx.begin(), idx.end(),
                         [&](int a, int b) { return std::fabs(w[a] - d) > std::fabs(w[b] - d); });
        S.assign(k, std::vector<double>(j));
        for (int c = 0; c < k; ++c)
            for (int t = 0; t < j; ++t) S[c][t] = Z[(size_t)t * j + idx[c]];
    }
    if (!keep_space(h, o, rc, S.empty() ? nullptr : &S))
        throw Error{H2W_EINVAL, "deflation space: fewer than 2 steps, or a singular Arnoldi relation"};
    h.g_defl.alloc((size_t)2 * rc.k * N);
    H2W_HIP(hipMemcpyAsync(h.g_defl.p, h.g_U.p, (size_t)2 * rc.k * N * 8, hipMemcpyDeviceToDevice, s));
    h.g_defl_rm.alloc((size_t)2 * rc.k * N);
    launch_to_rowmajor(h.g_defl.p, N, rc.k, h.g_defl_rm.p, s);
    launch_to_rowmajor(h.g_defl.p + (int64_t)rc.k * N, N, rc.k, h.g_defl_rm.p + (int64_t)rc.k * N, s);
    H2W_HIP(hipStreamSynchronize(s));
    h.defl_k = rc.k;
    h.defl_prec = prec;
    h.defl_gen = h.inner_gen;
}

}  // namespace

// Complex GMRES (the reference's -DUSE_Complex / USE_Helm / USE_Hankel branch of
// iterative_solver::GMRES, 1D/codes/gmres.hpp:52-67 and :91-200) on the tree-ordered complex
// right-hand side bt (N (re, im) pairs, device), starting from and updating h.g_x.  Unrestarted,
// Arnoldi by classical Gram-Schmidt twice with the Hermitian inner product h_{k,i} = v_k^H w, complex
// Givens rotations G = [c, s; -conj(s), c] with real c = |dx| / n and s = (dx / |dx|) conj(dy) / n,
// resid = |s_{i+1}| / ||b||, back-substitution.  (The reference's branch forms h_{k,i} as
// w.dot(v_k) = w^H v_k, the conjugate, and applies -s instead of -conj(s); for complex data those
// leave the Krylov basis non-orthogonal and the subdiagonal unreduced, so this restatement keeps the
// textbook forms, which coincide with the reference's for real data.)
h2w_gmres_stats solve_tree_c(Handle &h, const double *bt, int max_iter, double tol) {
    using cd = std::complex<double>;
    const int64_t N = h.N;
    hipStream_t s = h.stream;
    const double t0 = now_s();
    h2w_gmres_stats S;
    std::memset(&S, 0, sizeof(S));
    double2 *x = reinterpret_cast<double2 *>(h.g_x.p);
    const double2 *b = reinterpret_cast<const double2 *>(bt);
    h.g_w.ensure(2 * N);
    h.g_r.ensure(2 * N);
    double2 *w = reinterpret_cast<double2 *>(h.g_w.p), *r = reinterpret_cast<double2 *>(h.g_r.p);
    const int nb = cmdot_blocks(N);
    const int m = max_iter;
    h.g_part.ensure((size_t)2 * nb * (m + 2));
    h.g_h.ensure((size_t)2 * (2 * (m + 2) + 2));
    double2 *part = reinterpret_cast<double2 *>(h.g_part.p), *hv = reinterpret_cast<double2 *>(h.g_h.p);
    auto norm2 = [&](const double2 *v) {
        launch_cmdot(v, N, 1, v, N, part, nb, s);
        launch_cmdot_reduce(part, nb, 1, hv, s);
        double2 q;
        H2W_HIP(hipMemcpyAsync(&q, hv, 16, hipMemcpyDeviceToHost, s));
        H2W_HIP(hipStreamSynchronize(s));
        return std::sqrt(std::max(0.0, q.x));
    };
    // basis: (m + 1) complex vectors in g_V
    const int64_t vcols = std::min<int64_t>(m + 1, 1024);
    if ((int64_t)h.g_V.n < vcols * 2 * N) {
        h.g_V.alloc((size_t)vcols * 2 * N);
        h.g_Vcols = 0;  // (the real basis layout is rebuilt on its next use)
        h.gv_defl = -1;
    }
    double2 *V = reinterpret_cast<double2 *>(h.g_V.p);
    double normb = norm2(b);
    if (normb == 0.0) normb = 1.0;
    matvec_dev(h, h.g_x.p, h.g_w.p, H2W_FP64, true);
    S.matvecs_fp64 = 1;
    H2W_HIP(hipMemcpyAsync(r, b, N * 16, hipMemcpyDeviceToDevice, s));
    launch_caxpby(make_double2(-1.0, 0.0), w, make_double2(1.0, 0.0), r, N, s);
    const double beta = norm2(r);
    S.resid = beta / normb;
    if (S.resid <= tol) {
        S.converged = 1;
        S.seconds = now_s() - t0;
        return S;
    }
    const int mm = (int)std::min<int64_t>(m, vcols - 1);
    std::vector<std::vector<cd>> H;
    std::vector<cd> sv(mm + 1, cd(0.0)), cs(mm + 1, cd(0.0)), sn(mm + 1, cd(0.0));
    launch_caxpby(make_double2(1.0 / beta, 0.0), r, make_double2(0.0, 0.0), V, N, s);
    sv[0] = beta;
    std::vector<double2> hh(2 * (mm + 2) + 2);
    auto rot = [](cd &dx, cd &dy, cd c, cd sg) {
        const cd t = c * dx + sg * dy;
        dy = -std::conj(sg) * dx + c * dy;
        dx = t;
    };
    for (int i = 0; i < mm; ++i) {
        matvec_dev(h, reinterpret_cast<double *>(V + (int64_t)i * N), h.g_w.p, H2W_FP64, true);
        S.matvecs_fp64++;
        const int k = i + 1;
        launch_cmdot(V, N, k, w, N, part, nb, s);
        launch_cmdot_reduce(part, nb, k, hv, s);
        launch_cmgemv(V, N, k, hv, w, N, -1.0, s);
        launch_cmdot(V, N, k, w, N, part, nb, s);
        launch_cmdot_reduce(part, nb, k, hv + k, s);
        launch_cmgemv(V, N, k, hv + k, w, N, -1.0, s);
        launch_cmdot(w, N, 1, w, N, part, nb, s);
        launch_cmdot_reduce(part, nb, 1, hv + 2 * k, s);
        H2W_HIP(hipMemcpyAsync(hh.data(), hv, (2 * k + 1) * 16, hipMemcpyDeviceToHost, s));
        H2W_HIP(hipStreamSynchronize(s));
        H.emplace_back(i + 2, cd(0.0));
        std::vector<cd> &Hc = H.back();
        for (int q = 0; q <= i; ++q) Hc[q] = cd(hh[q].x + hh[k + q].x, hh[q].y + hh[k + q].y);
        const double hn = std::sqrt(std::max(0.0, hh[2 * k].x));
        Hc[i + 1] = hn;
        const bool breakdown = !(hn > 0.0);
        if (breakdown) launch_cfill(V + (int64_t)(i + 1) * N, N, s);
        else launch_caxpby(make_double2(1.0 / hn, 0.0), w, make_double2(0.0, 0.0), V + (int64_t)(i + 1) * N, N, s);
        for (int q = 0; q < i; ++q) rot(Hc[q], Hc[q + 1], cs[q], sn[q]);
        {
            const cd dx = Hc[i], dy = Hc[i + 1];
            if (std::abs(dx) == 0.0) {
                cs[i] = 0.0;
                sn[i] = 1.0;
            } else {
                const double sc = std::abs(dx) + std::abs(dy);
                const double nrm = sc * std::sqrt(std::norm(dx / sc) + std::norm(dy / sc));
                const cd alpha = dx / std::abs(dx);
                cs[i] = std::abs(dx) / nrm;
                sn[i] = alpha * std::conj(dy) / nrm;
            }
        }
        rot(Hc[i], Hc[i + 1], cs[i], sn[i]);
        rot(sv[i], sv[i + 1], cs[i], sn[i]);
        S.resid = std::abs(sv[i + 1]) / normb;
        S.iterations = i + 1;
        if (S.resid < tol || i == mm - 1 || breakdown) {
            std::vector<cd> y(sv.begin(), sv.begin() + i + 1);
            for (int q = i; q >= 0; --q) {
                y[q] /= H[q][q];
                for (int jj = q - 1; jj >= 0; --jj) y[jj] -= H[q][jj] * y[q];
            }
            std::vector<double2> yd(i + 1);
            for (int q = 0; q <= i; ++q) yd[q] = make_double2(y[q].real(), y[q].imag());
            H2W_HIP(hipMemcpyAsync(hv, yd.data(), (i + 1) * 16, hipMemcpyHostToDevice, s));
            launch_cmgemv(V, N, i + 1, hv, x, N, 1.0, s);
            S.converged = S.resid < tol || (breakdown && S.resid == 0.0);
            break;
        }
    }
    H2W_HIP(hipStreamSynchronize(s));
    S.seconds = now_s() - t0;
    return S;
}

// GMRES on the tree-ordered right-hand side bt (device), starting from and
// updating h.g_x: plain FP64 GMRES, or FP64 iterative refinement whose
// corrections come from GMRES on an FP32 operator.
h2w_gmres_stats solve_tree(Handle &h, const double *bt, int max_iter, double tol, int mode) {
    hipStream_t s = h.stream;
    const int64_t N = h.N;
    const int inner_prec = mode == H2W_GMRES_FP32_OTF_IR ? H2W_FP32_OTF
                           : mode == H2W_GMRES_FP32_INNER_IR ? H2W_FP32_INNER
                                                              : H2W_FP32;
    double t0 = now_s();
    h2w_gmres_stats S;
    std::memset(&S, 0, sizeof(S));
    if (mode == H2W_GMRES_FP64) {
        auto o = gmres_core(h, bt, h.g_x.p, max_iter, tol, H2W_FP64, false, -1.0);
        S.iterations = o.iters;
        S.resid = o.resid;
        S.matvecs_fp64 = o.matvecs;
        S.converged = o.conv;
    } else {
        // FP64 iterative refinement: r = b - A x in FP64, correction from GMRES on the FP32 operator.
        // The first residual is the FP32 operator's own: the first correction then solves the
        // FP32 system itself (x1 = A32^-1 b to the inner tolerance, as a low-precision first
        // solve), which is as close to the solution as a correction of the FP64 residual of x0
        // would be, one FP64 product earlier.  Convergence is only ever decided on an FP64
        // residual.
        double normb = dev_norm(h, bt);
        if (normb == 0.0) normb = 1.0;
        int total = 0, outer = 0;
        double rn = 0.0;
        bool fp64_resid = max_iter < 1;  // (no correction allowed: report x0's FP64 residual)
        Recycled rc;
        // a deflation space built for this inner operator serves every correction (it goes where
        // keep_space puts a kept space: U in g_U, C in the first basis columns)
        const bool defl = h.defl_k > 0 && h.defl_prec == inner_prec &&
                          (inner_prec != H2W_FP32_INNER || h.defl_gen == h.inner_gen);
        if (defl) {
            const int k = h.defl_k;
            ensure_V(h, k + 2);  // (a larger basis buffer keeps its columns)
            const bool fresh = h.g_U.n < (size_t)k * N;  // (ensure reallocates: nothing kept)
            h.g_U.ensure((size_t)k * N);
            if (fresh || h.gv_defl != h.defl_serial) {  // (still there after an earlier deflated solve)
                H2W_HIP(hipMemcpyAsync(h.g_U.p, h.g_defl.p, (size_t)k * N * 8, hipMemcpyDeviceToDevice, s));
                H2W_HIP(hipMemcpyAsync(h.g_V.p, h.g_defl.p + (int64_t)k * N, (size_t)k * N * 8,
                                       hipMemcpyDeviceToDevice, s));
                h.gv_defl = h.defl_serial;
            }
            rc.k = k;
            rc.invariant = true;
        }
        while (true) {
            if (fp64_resid) {
                matvec_dev(h, h.g_x.p, h.g_d.p, H2W_FP64, true);
                S.matvecs_fp64++;
            } else {
                matvec_dev(h, h.g_x.p, h.g_d.p, inner_prec, true);
                S.matvecs_fp32++;
            }
            if (outer == 0) {
                // start from alpha x0 with alpha minimising |b - alpha A x0| (no extra product):
                // the first correction then starts from a residual no larger than b
                const double dd = dev_dot(h, h.g_d.p, h.g_d.p);
                const double alpha = dd > 0.0 ? dev_dot(h, h.g_d.p, bt) / dd : 1.0;
                if (std::isfinite(alpha) && alpha != 1.0) {
                    launch_scal(alpha, h.g_x.p, N, s);
                    launch_scal(alpha, h.g_d.p, N, s);
                }
            }
            H2W_HIP(hipMemcpyAsync(h.g_r.p, bt, N * 8, hipMemcpyDeviceToDevice, s));
            launch_axpby(-1.0, h.g_d.p, 1.0, h.g_r.p, N, s);
            double nr = dev_norm(h, h.g_r.p);
            rn = nr / normb;
            if (fp64_resid && (rn <= tol || total >= max_iter || outer >= 50)) break;
            // (the first correction, from the FP32 residual, stops at sqrt(tol): the FP64 residual
            // after it is bounded by the FP32 operator's error anyway, and the second correction
            // finishes from there)
            double floor_eta = mode == H2W_GMRES_FP32_INNER_IR ? std::pow(10.0, -h.ir_exp) : 1e-6;
            if (!fp64_resid) floor_eta = std::max(floor_eta, std::sqrt(tol));
            double eta = std::min(1e-2, std::max(floor_eta, 0.1 * tol / rn));
            launch_fill(h.g_d.p, N, 0.0, s);
            // later corrections (same FP32 operator) recycle the first one's Krylov space
            auto o = gmres_core(h, h.g_r.p, h.g_d.p, max_iter - total, eta, inner_prec, true, nr,
                                rc.k > 0 ? &rc : nullptr, outer == 0 && !defl);
            if (outer == 0 && !defl) keep_space(h, o, rc);
            total += o.iters;
            S.matvecs_fp32 += o.matvecs;
            launch_axpby(1.0, h.g_d.p, 1.0, h.g_x.p, N, s);
            ++outer;
            // (no iteration and no recycled projection: the correction was zero)
            if (o.iters == 0 && fp64_resid && rc.k == 0) break;
            fp64_resid = true;
        }
        S.iterations = total;
        S.outer_iterations = outer;
        S.resid = rn;
        S.converged = rn <= tol;
    }
    H2W_HIP(hipStreamSynchronize(s));
    S.seconds = now_s() - t0;
    return S;
}


// ------------------------------------------------------------------ autotuner
namespace {

struct EventPair {
    Event a, b;
    double ms(hipStream_t) { return elapsed_ms(a, b); }
};

double time_launch(Handle &h, const Launch &Lh, int precision, int nrep, EventPair &ev) {
    run_launch(h, Lh, precision);
    H2W_HIP(hipEventRecord(ev.a, h.stream));
    for (int r = 0; r < nrep; ++r) run_launch(h, Lh, precision);
    H2W_HIP(hipEventRecord(ev.b, h.stream));
    H2W_HIP(hipGetLastError());
    return ev.ms(h.stream) / nrep;
}

// unit input in the pool's x segment, zero outputs
void tune_inputs(Handle &h, int precision) {
    if (is32(precision)) launch_fill32(h.vec32.p + h.off_x, h.N, 1.0f, h.stream);
    else launch_fill(h.vec64.p + h.off_x, h.N, 1.0, h.stream);
    zero_outputs(h, precision);
}

}  // namespace

// one whole matvec (graph replay when enabled), ms
double time_matvec(Handle &h, int precision, int nrep) {
    EventPair ev;
    tune_inputs(h, precision);
    run_launches(h, precision);
    H2W_HIP(hipEventRecord(ev.a, h.stream));
    for (int r = 0; r < nrep; ++r) {
        zero_outputs(h, precision);
        run_launches(h, precision);
    }
    H2W_HIP(hipEventRecord(ev.b, h.stream));
    return ev.ms(h.stream) / nrep;
}

// Per launch of one precision's matvec: 2, 4 or 8 column loads in flight per lane,
// whichever runs fastest (4 unless another is at least 2 % faster).
void tune_unroll(Handle &h, int precision) {
    std::vector<Launch> &L = precision == H2W_FP32_INNER ? h.inner.launches : h.launches;
    if (L.empty()) return;
    EventPair ev;
    tune_inputs(h, precision);
    for (auto &Lh : L) {
        int &u = precision == H2W_FP32 ? Lh.unr32 : Lh.unr;
        const int64_t elems = precision == H2W_FP32_INNER ? h.inner.elems[&Lh - &L[0]] : h.launch_elems[&Lh - &L[0]];
        const int nrep = elems > (int64_t)1 << 26 ? 3 : 8;
        u = 4;
        double tb = time_launch(h, Lh, precision, nrep, ev);
        int best = 4;
        for (int c : {2, 8}) {
            u = c;
            double t = time_launch(h, Lh, precision, nrep, ev);
            if (t < 0.98 * tb) {
                tb = t;
                best = c;
            }
        }
        u = best;
    }
    H2W_HIP(hipStreamSynchronize(h.stream));
    drop_graph(h, precision);
}

// Inner tolerance of the refinement: 10^-p for p = 4, 4.5, ..., 8 below tol_pow.  Each
// candidate solves A x = bt from x0 = 0 and from x0 = 1 (the reference's start); its score
// is the slower of the two, raised by a fifth when a final residual sits within 3x of the
// tolerance (a rounding change could then cost another refinement step).  The best score
// is kept.
void tune_inner(Handle &h, const double *bt, double tol, int max_iter, bool unroll, h2w_tune *out) {
    const double p0 = h.ir_exp > 0 ? h.ir_exp : (double)h.opts.ir_tol_pow;
    double best = 0.0, sbest = 1e300;
    out->n_cand = 0;
    for (int q = 8; q <= 16 && 0.5 * q < h.tol_pow && out->n_cand < H2W_TUNE_MAX_CAND; ++q) {
        const double p = 0.5 * q;
        build_inner(h, p);
        if (h.inner.launches.empty()) continue;
        if (unroll) tune_unroll(h, H2W_FP32_INNER);
        time_matvec(h, H2W_FP32_INNER, 1);  // captures the graphs outside the timed solves
        time_matvec(h, H2W_FP64, 1);
        h2w_gmres_stats S{};
        double worst = 0.0, rmax = 0.0;
        bool conv = true;
        for (int start = 0; start < 2; ++start) {
            launch_fill(h.g_x.p, h.N, start == 0 ? 0.0 : 1.0, h.stream);
            h2w_gmres_stats S2 = solve_tree(h, bt, max_iter, tol, H2W_GMRES_FP32_INNER_IR);
            conv = conv && S2.converged;
            rmax = std::max(rmax, S2.resid);
            if (S2.seconds > worst) {
                worst = S2.seconds;
                S = S2;
            }
        }
        const double score = worst * (rmax > tol / 2.0 ? 1.2 : 1.0);
        const int c = out->n_cand++;
        out->cand_ir_tol_exp[c] = p;
        out->cand_seconds[c] = worst;
        out->cand_iterations[c] = S.iterations;
        out->cand_outer[c] = S.outer_iterations;
        out->cand_converged[c] = conv;
        out->cand_inner_bytes[c] = h.inner_elems * 4;
        if (conv && score < sbest) {
            sbest = score;
            best = p;
        }
    }
    if (best == 0.0) best = p0;
    if (best != h.ir_exp || h.inner.launches.empty()) {
        build_inner(h, best);
        if (unroll) tune_unroll(h, H2W_FP32_INNER);
    }
    out->ir_tol_exp = h.ir_exp;
}

// Deflation spaces for the chosen inner operator, scored as tune_inner scores tolerances (the
// slower of the solves from x0 = 0 and x0 = 1, a fifth more when a final residual exceeds tol / 2);
// then, with retune_inner, the inner tolerances half a decade either side under the chosen
// space.  Leaves the best (inner tolerance, space) built.
void tune_deflation(Handle &h, const double *bt, double tol, int max_iter, bool unroll, bool retune_inner,
                    h2w_tune *out) {
    static const int cand[][2] = {{0, 0}, {64, 32}, {128, 48}, {256, 64}, {256, 96}, {384, 128}};
    out->n_defl_cand = 0;
    double sbest = 1e300, pbest = h.ir_exp;
    int bm = 0, bk = 0;
    auto score = [&](int m, int k) {
        build_deflation(h, m, k, H2W_FP32_INNER);
        double worst = 0.0, rmax = 0.0;
        bool conv = true;
        h2w_gmres_stats S{};
        for (int start = 0; start < 2; ++start) {
            launch_fill(h.g_x.p, h.N, start == 0 ? 0.0 : 1.0, h.stream);
            h2w_gmres_stats S2 = solve_tree(h, bt, max_iter, tol, H2W_GMRES_FP32_INNER_IR);
            conv = conv && S2.converged;
            rmax = std::max(rmax, S2.resid);
            if (S2.seconds > worst) {
                worst = S2.seconds;
                S = S2;
            }
        }
        const double sc = worst * (rmax > tol / 2.0 ? 1.2 : 1.0);
        if (out->n_defl_cand < H2W_TUNE_MAX_CAND) {
            const int c = out->n_defl_cand++;
            out->cand_defl_m[c] = m;
            out->cand_defl_k[c] = k;
            out->cand_defl_ir_tol_exp[c] = h.ir_exp;
            out->cand_defl_seconds[c] = worst;
            out->cand_defl_iterations[c] = S.iterations;
            out->cand_defl_outer[c] = S.outer_iterations;
            out->cand_defl_converged[c] = conv;
        }
        if (conv && sc < sbest) {
            sbest = sc;
            bm = m;
            bk = k;
            pbest = h.ir_exp;
        }
    };
    time_matvec(h, H2W_FP32_INNER, 1);  // (graphs captured outside the timed solves)
    time_matvec(h, H2W_FP64, 1);
    for (auto &c : cand)
        if ((int64_t)c[0] < h.N) score(c[0], c[1]);
    if (retune_inner && bm > 0) {
        const double p0 = h.ir_exp;
        const int m = bm, k = bk;
        for (double p : {p0 - 0.5, p0 + 0.5}) {
            if (!(p >= 4.0) || !(p < h.tol_pow)) continue;
            build_inner(h, p);
            if (h.inner.launches.empty()) continue;
            if (unroll) tune_unroll(h, H2W_FP32_INNER);
            time_matvec(h, H2W_FP32_INNER, 1);
            score(m, k);
        }
        if (pbest != h.ir_exp) {
            build_inner(h, pbest);
            if (unroll) tune_unroll(h, H2W_FP32_INNER);
            time_matvec(h, H2W_FP32_INNER, 1);
        }
    }
    const double t0 = now_s();
    build_deflation(h, bm, bk, H2W_FP32_INNER);
    out->defl_build_seconds = now_s() - t0;
    out->defl_m = bm;
    out->defl_k = bk;
    out->ir_tol_exp = h.ir_exp;
}
}  // namespace h2w

namespace h2w {
// The device side of a handle whose plan is built: stream, tree-order points and
// permutation on the device.  Needs a visible HIP device.
void attach_device(Handle &h) {
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0)
        throw Error{H2W_ENOLIB, "no HIP device visible; libh2w has no CPU fallback"};
    if (h.opts.device < 0 || h.opts.device >= ndev) throw Error{H2W_EINVAL, "device ordinal out of range"};
    h.opts.plan_only = 0;
    H2W_HIP(hipSetDevice(h.opts.device));
    H2W_HIP(hipStreamCreateWithFlags(&h.stream, hipStreamNonBlocking));
    h.d_px.upload(h.plan.px, h.stream);
    h.d_py.upload(h.plan.py, h.stream);
    h.d_pz.upload(h.plan.pz, h.stream);
    h.d_perm.upload(h.plan.perm, h.stream);
    std::vector<int32_t> iperm(h.N);
    for (int64_t t = 0; t < h.N; ++t) iperm[h.plan.perm[t]] = (int32_t)t;
    h.d_iperm.upload(iperm, h.stream);
    H2W_HIP(hipStreamSynchronize(h.stream));
    noalloc_setup(h.opts.device);
    h.kp.dim = h.dim;
    h.kp.choice = h.choice;
    h.kp.diag = h.diag;
    h.kp.px = h.d_px.p;
    h.kp.py = h.d_py.p;
    h.kp.pz = h.d_pz.p;
    h.kpc.dim = h.dim;
    h.kpc.choice = h.choice;
    h.kpc.diag = h.diag;
    h.kpc.diag_im = h.diag_im;
    h.kpc.px = h.d_px.p;
    h.kpc.py = h.d_py.p;
    h.kpc.pz = h.d_pz.p;
}
}  // namespace h2w

// ------------------------------------------------------------------ C ABI
using h2w::Error;

#define H2W_TRY try {
#define H2W_CATCH                                         \
    }                                                     \
    catch (const Error &e) {                              \
        h2w::set_error(e.msg);                            \
        return e.code;                                    \
    }                                                     \
    catch (const std::bad_alloc &) {                      \
        h2w::set_error("host allocation failed");         \
        return H2W_ENOMEM;                                \
    }                                                     \
    catch (const std::exception &e) {                     \
        h2w::set_error(e.what());                         \
        return H2W_EINVAL;                                \
    }

extern "C" {

void h2w_default_opts(h2w_opts *o) {
    if (!o) return;
    std::memset(o, 0, sizeof(*o));
    o->compat = 1;
    o->nlevels = 0;
    o->fp32_shadow = 1;
    o->device = 0;
    o->rank_cap = 256;
    o->workspace_bytes = 0;
    o->plan_only = 0;
    o->ir_tol_pow = 6;
}

const char *h2w_last_error(void) { return h2w::g_err.c_str(); }

int h2w_create(int dim, int variant, int64_t N, const double *points, int n_max, double L, int tol_pow, int choice,
               const h2w_opts *opts, h2w_handle **out) {
    H2W_TRY
    if (!out) throw Error{H2W_EINVAL, "out is NULL"};
    *out = nullptr;
    if (dim < 1 || dim > 3) throw Error{H2W_EINVAL, "dim must be 1, 2 or 3"};
    if (variant != H2W_NESTED && variant != H2W_SEMI_NESTED && variant != H2W_NON_NESTED)
        throw Error{H2W_EINVAL, "unknown variant"};
    if (variant == H2W_NON_NESTED && dim == 1) throw Error{H2W_EINVAL, "H* is defined for 2D and 3D"};
    if (choice == H2W_CHOICE_HELMHOLTZ && dim != 3)
        throw Error{H2W_EINVAL, "choice 2 (Helmholtz, e^{iR}/(4 pi)) is the 3D complex kernel"};
    if (choice == H2W_CHOICE_HANKEL && dim != 2)
        throw Error{H2W_EINVAL, "choice 10 (Hankel, (i/4) H0^(1)(R)) is the 2D complex kernel"};
    if (choice != 0 && choice != 1 && choice != H2W_CHOICE_HELMHOLTZ && choice != H2W_CHOICE_HANKEL)
        throw Error{H2W_EINVAL, "Wrong choice! choice must be 0 (IE), 1 (RBF), 2 (3D Helmholtz) or 10 (2D Hankel)"};
    if (N < 2 || N > INT32_MAX) throw Error{H2W_EINVAL, "N out of range"};
    if (n_max < 1) throw Error{H2W_EINVAL, "n_max must be positive"};
    if (!(L > 0.0)) throw Error{H2W_EINVAL, "L must be positive"};
    if (tol_pow < 0 || tol_pow > 20) throw Error{H2W_EINVAL, "tol_pow out of range"};
    h2w_opts o;
    h2w_default_opts(&o);
    if (opts) o = *opts;
    int ndev = 0;
    if (!o.plan_only) {
        if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0)
            throw Error{H2W_ENOLIB, "no HIP device visible; libh2w has no CPU fallback"};
        if (o.device < 0 || o.device >= ndev) throw Error{H2W_EINVAL, "device ordinal out of range"};
    }
    std::vector<double> grid;
    const bool is_grid = points == nullptr;
    if (is_grid) {
        // the reference's uniform grids (1D/codes/HODLR1Dtree.hpp:59-65, 2D/codes/HODLR2Dtree.hpp:75-91,
        // 3D/codes/HODLR3Dtree.hpp:82-102)
        grid.assign((size_t)dim * N, 0.0);
        if (dim == 1) {
            for (int64_t k = 0; k < N; ++k) grid[k] = -1.0 + 2.0 * (k + 1.0) / (N + 1.0);
        } else {
            int64_t n = std::llround(dim == 2 ? std::sqrt((double)N) : std::cbrt((double)N));
            if ((dim == 2 && n * n != N) || (dim == 3 && n * n * n != N))
                throw Error{H2W_EINVAL, "the uniform grid needs N to be a square (2D) or a cube (3D)"};
            std::vector<double> nd(n);
            for (int64_t k = 0; k < n; ++k) nd[k] = -L + 2.0 * L * (k + 1.0) / (n + 1.0);
            if (dim == 2) {
                for (int64_t j = 0; j < n; ++j)
                    for (int64_t k = 0; k < n; ++k) {
                        grid[j * n + k] = nd[k];
                        grid[N + j * n + k] = nd[j];
                    }
            } else {
                for (int64_t j = 0; j < n; ++j)
                    for (int64_t k = 0; k < n; ++k)
                        for (int64_t i = 0; i < n; ++i) {
                            int64_t p = (j * n + k) * n + i;
                            grid[p] = nd[k];
                            grid[N + p] = nd[j];
                            grid[2 * N + p] = nd[i];
                        }
            }
        }
        points = grid.data();
    }
    int nl = o.nlevels > 0 ? o.nlevels : h2w::ref_nlevels(dim, N, n_max, is_grid);
    if (nl < 1) throw Error{H2W_EINVAL, "nLevels < 1: N must exceed n_max"};
    if (nl > (dim == 1 ? 24 : (dim == 2 ? 12 : 8))) throw Error{H2W_EINVAL, "tree too deep"};
    std::unique_ptr<h2w_handle> h(new h2w_handle());
    h->dim = dim;
    h->variant = variant;
    h->choice = choice;
    h->tol_pow = tol_pow;
    h->n_max = n_max;
    h->N = N;
    h->L = L;
    h->opts = o;
    h->use_graph = std::getenv("H2W_NO_GRAPH") == nullptr;
    h->sym16 = std::getenv("H2W_NO_SYM16") == nullptr;
    h->plan.build(dim, N, points, L, nl);
    h->cplx = choice == H2W_CHOICE_HELMHOLTZ || choice == H2W_CHOICE_HANKEL;
    if (h->cplx) {
        // complex kernels: FP64 operators only (no FP32 copies, no refinement operator)
        h->opts.fp32_shadow = 0;
        h->opts.ir_tol_pow = 0;
        h2w::diag_value_c(dim, choice, N, h->diag, h->diag_im);
    } else {
        h->diag = h2w::diag_value(dim, choice, N, o.compat);
    }
    if (!o.plan_only) h2w::attach_device(*h);
    *out = h.release();
    return H2W_OK;
    H2W_CATCH
}

int h2w_assemble(h2w_handle *h) {
    H2W_TRY
    if (!h) throw Error{H2W_EINVAL, "NULL handle"};
    if (h->opts.plan_only) throw Error{H2W_ESTATE, "handle was created with plan_only"};
    H2W_HIP(hipSetDevice(h->opts.device));
    h2w::assemble(*h);
    return H2W_OK;
    H2W_CATCH
}

int h2w_assemble_many(h2w_handle *const *hs, int n, int nthreads) {
    H2W_TRY
    if (!hs || n < 0 || nthreads < 1) throw Error{H2W_EINVAL, "bad arguments"};
    for (int i = 0; i < n; ++i) {
        if (!hs[i]) throw Error{H2W_EINVAL, "NULL handle"};
        if (hs[i]->opts.plan_only) throw Error{H2W_ESTATE, "handle was created with plan_only"};
        for (int j = 0; j < i; ++j)
            if (hs[j] == hs[i]) throw Error{H2W_EINVAL, "a handle appears twice"};
    }
    // host threads take the handles in turn; each assembles on its handle's own stream, so the
    // small systems' level-by-level launches overlap on the device
    std::atomic<int> next{0};
    std::mutex mu;
    int code = H2W_OK;
    std::string msg;
    auto work = [&]() {
        for (int i = next++; i < n; i = next++) {
            const int rc = h2w_assemble(hs[i]);
            if (rc != H2W_OK) {
                std::lock_guard<std::mutex> lk(mu);
                if (code == H2W_OK) {
                    code = rc;
                    msg = std::string("system ") + std::to_string(i) + ": " + h2w_last_error();
                }
            }
        }
    };
    const int nt = std::min(nthreads, n);
    std::vector<std::thread> th;
    for (int t = 1; t < nt; ++t) th.emplace_back(work);
    if (nt >= 1) work();
    for (auto &t : th) t.join();
    if (code != H2W_OK) throw Error{code, msg};
    return H2W_OK;
    H2W_CATCH
}

int h2w_matvec_ex(h2w_handle *h, const double *x, double *y, int nrhs, int64_t ld, int precision, int order,
                  int where) {
    H2W_TRY
    if (!h || !x || !y) throw Error{H2W_EINVAL, "NULL argument"};
    if (!h->assembled) throw Error{H2W_ESTATE, "h2w_matvec before h2w_assemble"};
    if (nrhs < 1 || ld < h->N) throw Error{H2W_EINVAL, "bad nrhs / ld"};
    if (precision < H2W_FP64 || precision > H2W_FP32_INNER) throw Error{H2W_EINVAL, "bad precision"};
    H2W_HIP(hipSetDevice(h->opts.device));
    const int64_t N = h->N;
    if (h->cplx) {
        // complex kernels: x, y hold N (re, im) pairs per right-hand side, ld counts complex entries
        if (precision != H2W_FP64) throw Error{H2W_EINVAL, "complex kernels: precision H2W_FP64 only"};
        for (int r = 0; r < nrhs; ++r) {
            const double *xr = x + 2 * r * ld;
            double *yr = y + 2 * r * ld;
            if (where == H2W_HOST) {
                h->d_stage_in.ensure(2 * N);
                h->d_stage_out.ensure(2 * N);
                H2W_HIP(hipMemcpyAsync(h->d_stage_in.p, xr, N * 16, hipMemcpyHostToDevice, h->stream));
                h2w::matvec_dev(*h, h->d_stage_in.p, h->d_stage_out.p, H2W_FP64, order == H2W_ORDER_TREE);
                H2W_HIP(hipMemcpyAsync(yr, h->d_stage_out.p, N * 16, hipMemcpyDeviceToHost, h->stream));
            } else {
                h2w::matvec_dev(*h, xr, yr, H2W_FP64, order == H2W_ORDER_TREE);
            }
        }
        H2W_HIP(hipStreamSynchronize(h->stream));
        return H2W_OK;
    }
    if (nrhs > 1 && (precision == H2W_FP64 || precision == H2W_FP32 || precision == H2W_FP32_INNER)) {
        // kNR right-hand sides per pass on the matrix cores; host columns go through the handle's staging, one
        // copy each way per pass (a copy per column, and staging allocated and freed by each call: 1175 against 1014 us for
        // 16 products of a 32^3 grid, of which the launches take 610)
        auto copy_columns = [&](double *d, int64_t ldd, const double *v, int64_t ldv, int nc, hipMemcpyKind k) {
            if (ldd == ldv) H2W_HIP(hipMemcpyAsync(d, v, ((nc - 1) * ldv + N) * 8, k, h->stream));
            else H2W_HIP(hipMemcpy2DAsync(d, ldd * 8, v, ldv * 8, N * 8, nc, k, h->stream));
        };
        // (outputs over the inputs of a later pass: those are read from a copy made before the first)
        std::vector<double> own;
        if (where == H2W_HOST && nrhs > h2w::kNR && y > x && y < x + (nrhs - 1) * ld + N) {
            own.assign(x, x + (nrhs - 1) * ld + N);
            x = own.data();
        }
        for (int c0 = 0; c0 < nrhs; c0 += h2w::kNR) {
            const int nc = std::min(h2w::kNR, nrhs - c0);
            const double *xs = x + c0 * ld;
            double *ys = y + c0 * ld;
            int64_t lds = ld;
            if (where == H2W_HOST) {
                lds = N;
                h->d_stage_in.ensure((size_t)N * nc);
                h->d_stage_out.ensure((size_t)N * nc);
                copy_columns(h->d_stage_in.p, N, xs, ld, nc, hipMemcpyHostToDevice);
                xs = h->d_stage_in.p;
                ys = h->d_stage_out.p;
            }
            h2w::matvec_multi_dev(*h, xs, lds, ys, lds, nc, precision, order == H2W_ORDER_TREE);
            if (where == H2W_HOST)
                copy_columns(y + c0 * ld, ld, ys, N, nc, hipMemcpyDeviceToHost);
        }
        H2W_HIP(hipStreamSynchronize(h->stream));
        return H2W_OK;
    }
    for (int r = 0; r < nrhs; ++r) {
        const double *xr = x + r * ld;
        double *yr = y + r * ld;
        if (where == H2W_HOST) {
            h->d_stage_in.ensure(N);
            h->d_stage_out.ensure(N);
            H2W_HIP(hipMemcpyAsync(h->d_stage_in.p, xr, N * 8, hipMemcpyHostToDevice, h->stream));
            h2w::matvec_dev(*h, h->d_stage_in.p, h->d_stage_out.p, precision, order == H2W_ORDER_TREE);
            H2W_HIP(hipMemcpyAsync(yr, h->d_stage_out.p, N * 8, hipMemcpyDeviceToHost, h->stream));
        } else {
            h2w::matvec_dev(*h, xr, yr, precision, order == H2W_ORDER_TREE);
        }
    }
    H2W_HIP(hipStreamSynchronize(h->stream));
    return H2W_OK;
    H2W_CATCH
}

int h2w_matvec(h2w_handle *h, const double *x, double *y, int where) {
    return h2w_matvec_ex(h, x, y, 1, h ? h->N : 0, H2W_FP64, H2W_ORDER_INPUT, where);
}

int h2w_gmres(h2w_handle *h, const double *b, double *x, int max_iter, double tol, int mode, int where,
              h2w_gmres_stats *st) {
    H2W_TRY
    if (!h || !b || !x) throw Error{H2W_EINVAL, "NULL argument"};
    if (!h->assembled) throw Error{H2W_ESTATE, "h2w_gmres before h2w_assemble"};
    if (max_iter < 1) throw Error{H2W_EINVAL, "max_iter must be positive"};
    if (mode < H2W_GMRES_FP64 || mode > H2W_GMRES_FP32_INNER_IR) throw Error{H2W_EINVAL, "bad mode"};
    if (h->cplx) {
        // complex kernels: b, x hold N (re, im) pairs; FP64 GMRES with the complex branch's rotations
        if (mode != H2W_GMRES_FP64) throw Error{H2W_EINVAL, "complex kernels: mode H2W_GMRES_FP64 only"};
        H2W_HIP(hipSetDevice(h->opts.device));
        const int64_t N = h->N;
        hipStream_t s = h->stream;
        h->g_x.ensure(2 * N);
        h->d_stage_in.ensure(2 * N);
        h->d_stage_out.ensure(2 * N);
        const double *bsrc = b, *xsrc = x;
        if (where == H2W_HOST) {
            H2W_HIP(hipMemcpyAsync(h->d_stage_in.p, b, N * 16, hipMemcpyHostToDevice, s));
            H2W_HIP(hipMemcpyAsync(h->d_stage_out.p, x, N * 16, hipMemcpyHostToDevice, s));
            bsrc = h->d_stage_in.p;
            xsrc = h->d_stage_out.p;
        }
        h2w::DevBuf<double> bt;
        bt.alloc(2 * N);
        h2w::launch_cpermute_in(reinterpret_cast<const double2 *>(bsrc), reinterpret_cast<double2 *>(bt.p), h->d_perm.p, N,
                                s);
        h2w::launch_cpermute_in(reinterpret_cast<const double2 *>(xsrc), reinterpret_cast<double2 *>(h->g_x.p),
                                h->d_perm.p, N, s);
        H2W_HIP(hipStreamSynchronize(s));
        h2w_gmres_stats S = h2w::solve_tree_c(*h, bt.p, max_iter, tol);
        double *xdst = where == H2W_HOST ? h->d_stage_out.p : x;
        h2w::launch_cpermute_out(reinterpret_cast<const double2 *>(h->g_x.p), reinterpret_cast<double2 *>(xdst),
                                 h->d_perm.p, N, s);
        if (where == H2W_HOST) H2W_HIP(hipMemcpyAsync(x, h->d_stage_out.p, N * 16, hipMemcpyDeviceToHost, s));
        H2W_HIP(hipStreamSynchronize(s));
        if (st) *st = S;
        return S.converged ? H2W_OK : H2W_ENOCONV;
    }
    if (mode != H2W_GMRES_FP64 && !h->mat32.p) throw Error{H2W_ESTATE, "FP32 shadow not built"};
    if (mode == H2W_GMRES_FP32_INNER_IR && h->inner.launches.empty())
        throw Error{H2W_ESTATE, "the inner operator was not built (opts.ir_tol_pow)"};
    H2W_HIP(hipSetDevice(h->opts.device));
    const int64_t N = h->N;
    hipStream_t s = h->stream;
    h->g_x.ensure(N);
    h->g_r.ensure(N);
    h->g_d.ensure(N);
    h->d_stage_in.ensure(N);
    h->d_stage_out.ensure(N);
    // b and x0 to tree order
    const double *bsrc = b, *xsrc = x;
    if (where == H2W_HOST) {
        H2W_HIP(hipMemcpyAsync(h->d_stage_in.p, b, N * 8, hipMemcpyHostToDevice, s));
        H2W_HIP(hipMemcpyAsync(h->d_stage_out.p, x, N * 8, hipMemcpyHostToDevice, s));
        bsrc = h->d_stage_in.p;
        xsrc = h->d_stage_out.p;
    }
    h2w::DevBuf<double> bt;
    bt.alloc(N);
    h2w::launch_permute_in(bsrc, N, bt.p, N, h->d_perm.p, N, 1, s);
    h2w::launch_permute_in(xsrc, N, h->g_x.p, N, h->d_perm.p, N, 1, s);
    H2W_HIP(hipStreamSynchronize(s));
    h2w_gmres_stats S = h2w::solve_tree(*h, bt.p, max_iter, tol, mode);
    double *xdst = where == H2W_HOST ? h->d_stage_out.p : x;
    h2w::launch_permute_out(h->g_x.p, N, xdst, N, h->d_perm.p, N, 1, s);
    if (where == H2W_HOST) H2W_HIP(hipMemcpyAsync(x, h->d_stage_out.p, N * 8, hipMemcpyDeviceToHost, s));
    H2W_HIP(hipStreamSynchronize(s));
    if (st) *st = S;
    return S.converged ? H2W_OK : H2W_ENOCONV;
    H2W_CATCH
}

int h2w_gmres_multi(h2w_handle *h, const double *B, int64_t ldb, double *X, int64_t ldx, int nrhs, int max_iter,
                    double tol, int mode, int where, h2w_gmres_stats *st) {
    H2W_TRY
    if (!h || !B || !X || !st) throw Error{H2W_EINVAL, "NULL argument"};
    if (!h->assembled) throw Error{H2W_ESTATE, "h2w_gmres_multi before h2w_assemble"};
    if (h->cplx) throw Error{H2W_EINVAL, "complex kernels: several right-hand sides go through h2w_gmres"};
    if (max_iter < 1 || nrhs < 1 || ldb < h->N || ldx < h->N) throw Error{H2W_EINVAL, "bad max_iter / nrhs / ld"};
    if (mode != H2W_GMRES_FP64 && mode != H2W_GMRES_FP32_IR && mode != H2W_GMRES_FP32_INNER_IR)
        throw Error{H2W_EINVAL, "several right-hand sides: modes FP64, FP32_IR and FP32_INNER_IR"};
    if (mode != H2W_GMRES_FP64 && !h->mat32.p) throw Error{H2W_ESTATE, "FP32 shadow not built"};
    if (mode == H2W_GMRES_FP32_INNER_IR && h->inner.launches.empty())
        throw Error{H2W_ESTATE, "the inner operator was not built (opts.ir_tol_pow)"};
    H2W_HIP(hipSetDevice(h->opts.device));
    const int64_t N = h->N;
    hipStream_t s = h->stream;
    const int64_t len = N * h2w::kNR;
    h2w::DevBuf<double> hb, hx, bt, xt;
    const double *bs = B;
    double *xs = X;
    if (where == H2W_HOST) {
        hb.alloc((size_t)ldb * nrhs);
        hx.alloc((size_t)ldx * nrhs);
        H2W_HIP(hipMemcpyAsync(hb.p, B, (size_t)ldb * nrhs * 8, hipMemcpyHostToDevice, s));
        H2W_HIP(hipMemcpyAsync(hx.p, X, (size_t)ldx * nrhs * 8, hipMemcpyHostToDevice, s));
        bs = hb.p;
        xs = hx.p;
    }
    bt.alloc(len);
    xt.alloc(len);
    for (int c0 = 0; c0 < nrhs; c0 += h2w::kNR) {
        const int nc = std::min(h2w::kNR, nrhs - c0);
        h2w::launch_gather_m64(bs + c0 * ldb, ldb, nc, h->d_perm.p, N, bt.p, s);
        h2w::launch_gather_m64(xs + c0 * ldx, ldx, nc, h->d_perm.p, N, xt.p, s);
        h2w::solve_tree_m(*h, bt.p, xt.p, nc, max_iter, tol, mode, st + c0);
        h2w::launch_scatter_m64(xt.p, N, xs + c0 * ldx, ldx, nc, h->d_perm.p, s);
    }
    if (where == H2W_HOST)
        for (int c = 0; c < nrhs; ++c)
            H2W_HIP(hipMemcpyAsync(X + c * ldx, hx.p + c * ldx, N * 8, hipMemcpyDeviceToHost, s));
    H2W_HIP(hipStreamSynchronize(s));
    for (int c = 0; c < nrhs; ++c)
        if (!st[c].converged) return H2W_ENOCONV;
    return H2W_OK;
    H2W_CATCH
}

int h2w_dense_matvec(h2w_handle *h, const double *x, double *y, const int64_t *rows, int64_t nrows, int where) {
    H2W_TRY
    if (!h || !x || !y) throw Error{H2W_EINVAL, "NULL argument"};
    if (h->opts.plan_only) throw Error{H2W_ESTATE, "handle was created with plan_only"};
    H2W_HIP(hipSetDevice(h->opts.device));
    const int64_t N = h->N;
    hipStream_t s = h->stream;
    if (!rows) nrows = N;
    if (nrows < 0) throw Error{H2W_EINVAL, "nrows < 0"};
    // inverse permutation: input index -> tree index
    std::vector<int32_t> tr(nrows);
    {
        std::vector<int32_t> inv(N);
        for (int64_t t = 0; t < N; ++t) inv[h->plan.perm[t]] = (int32_t)t;
        for (int64_t q = 0; q < nrows; ++q) {
            int64_t i = rows ? rows[q] : q;
            if (i < 0 || i >= N) throw Error{H2W_EINVAL, "row index out of range"};
            tr[q] = inv[i];
        }
    }
    h2w::DevBuf<int32_t> drows;
    drows.upload(tr, s);
    h2w::DevBuf<double> xin, xt, yo;
    if (h->cplx) {
        // complex kernels: x (N) and y (nrows) hold (re, im) pairs
        xt.alloc(2 * N);
        yo.alloc(2 * std::max<int64_t>(nrows, 1));
        const double *xs = x;
        if (where == H2W_HOST) {
            xin.alloc(2 * N);
            H2W_HIP(hipMemcpyAsync(xin.p, x, N * 16, hipMemcpyHostToDevice, s));
            xs = xin.p;
        }
        h2w::launch_cpermute_in(reinterpret_cast<const double2 *>(xs), reinterpret_cast<double2 *>(xt.p), h->d_perm.p, N,
                                s);
        h2w::launch_cdense_rows(drows.p, nrows, reinterpret_cast<const double2 *>(xt.p), reinterpret_cast<double2 *>(yo.p),
                                N, h->kpc, s);
        H2W_HIP(hipGetLastError());
        H2W_HIP(hipMemcpyAsync(y, yo.p, nrows * 16, where == H2W_HOST ? hipMemcpyDeviceToHost : hipMemcpyDeviceToDevice,
                               s));
        H2W_HIP(hipStreamSynchronize(s));
        return H2W_OK;
    }
    xt.alloc(N);
    yo.alloc(std::max<int64_t>(nrows, 1));
    const double *xs = x;
    if (where == H2W_HOST) {
        xin.alloc(N);
        H2W_HIP(hipMemcpyAsync(xin.p, x, N * 8, hipMemcpyHostToDevice, s));
        xs = xin.p;
    }
    h2w::launch_permute_in(xs, N, xt.p, N, h->d_perm.p, N, 1, s);
    h2w::launch_dense_rows(drows.p, nrows, xt.p, yo.p, N, h->kp, s);
    H2W_HIP(hipGetLastError());
    H2W_HIP(hipMemcpyAsync(y, yo.p, nrows * 8, where == H2W_HOST ? hipMemcpyDeviceToHost : hipMemcpyDeviceToDevice, s));
    H2W_HIP(hipStreamSynchronize(s));
    return H2W_OK;
    H2W_CATCH
}

int h2w_get_stats(const h2w_handle *h, h2w_stats *st) {
    if (!h || !st) {
        h2w::set_error("NULL argument");
        return H2W_EINVAL;
    }
    std::memset(st, 0, sizeof(*st));
    st->dim = h->dim;
    st->variant = h->variant;
    st->choice = h->choice;
    st->nlevels = h->plan.nL;
    st->N = h->N;
    st->memory = h->memory;
    st->diag = h->diag;
    st->assembly_seconds = h->assembly_seconds;
    st->aca_reruns = h->aca_reruns;
    st->aca_batches = h->aca_batches;
    st->inner_tol_exp = h->inner.launches.empty() ? 0.0 : h->ir_exp;
    st->aca_pool_bytes = h->aca_pool_bytes;
    st->rank_pred_blocks = h->rank_pred_blocks;
    st->rank_pred_under = h->rank_pred_under;
    st->rank_pred_mae_log2 = h->rank_pred_blocks ? h->rank_pred_abs_log2 / h->rank_pred_blocks : 0.0;
    st->rank_fixed_blocks = h->rank_fix_blocks;
    st->rank_fixed_resumed = h->rank_fix_resumed;
    st->rank_fixed_extra_steps = h->rank_fix_extra_steps;
    st->rank_fixed_sampled_err = h->rank_fix_sampled_err;
    for (int f = 0; f < 2; ++f) {
        int mx = 0;
        double sum = 0.0;
        int64_t cnt = 0;
        for (auto &fl : h->fam[f])
            for (int r : fl.rank) {
                mx = std::max(mx, r);
                sum += r;
                ++cnt;
            }
        if (f == 1)
            for (auto &p : h->pairs) {
                mx = std::max(mx, p.rank);
                sum += p.rank;
                ++cnt;
            }
        if (f == 0) {
            st->max_rank_far = mx;
            st->mean_rank_far = cnt ? sum / cnt : 0.0;
        } else {
            st->max_rank_vertex = mx;
            st->mean_rank_vertex = cnt ? sum / cnt : 0.0;
        }
    }
    st->stored_bytes_fp64 = h->stored_elems * (h->cplx ? 16 : 8);
    st->diag_im = h->diag_im;
    st->stored_bytes_fp32 = h->mat32.p ? h->stored_elems * 4 : 0;
    st->n_launches_matvec = (int)h->launches.size() + 3;
    st->stored_bytes_inner_fp32 = h->inner_elems * 4;
    return H2W_OK;
}

int h2w_tree_order(const h2w_handle *h, int32_t *perm) {
    if (!h || !perm) {
        h2w::set_error("NULL argument");
        return H2W_EINVAL;
    }
    std::copy(h->plan.perm.begin(), h->plan.perm.end(), perm);
    return H2W_OK;
}

int h2w_box_skeleton(const h2w_handle *h, int family, int level, int box, int32_t *ir, int32_t *ic, int cap) {
    if (!h || family < 0 || family > 1 || level < 1 || level > h->plan.nL || box < 0 ||
        box >= h->plan.nboxes[level]) {
        h2w::set_error("bad skeleton query");
        return -H2W_EINVAL;
    }
    if (!h->assembled) {
        h2w::set_error("not assembled");
        return -H2W_ESTATE;
    }
    const auto &F = h->fam[family];
    if ((int)F.size() <= level || F[level].rank.empty()) return 0;
    const auto &fl = F[level];
    int r = fl.rank[box];
    for (int q = 0; q < r && q < cap; ++q) {
        if (ir) ir[q] = h->plan.perm[fl.Ir[box][q]];
        if (ic) ic[q] = h->plan.perm[fl.Ic[box][q]];
    }
    return r;
}

int h2w_interaction_list(const h2w_handle *h, int level, int box, int32_t *il, int32_t *isv, int cap) {
    if (!h || level < 1 || level > h->plan.nL || box < 0 || box >= h->plan.nboxes[level]) {
        h2w::set_error("bad list query");
        return -H2W_EINVAL;
    }
    const auto &l = h->plan.il[level][box];
    const auto &v = h->plan.ilv[level][box];
    for (size_t q = 0; q < l.size() && (int)q < cap; ++q) {
        if (il) il[q] = l[q];
        if (isv) isv[q] = v[q];
    }
    return (int)l.size();
}

int h2w_near_list(const h2w_handle *h, int level, int box, int32_t *nb, int cap) {
    if (!h || level != h->plan.nL || box < 0 || box >= h->plan.nboxes[level]) {
        h2w::set_error("near lists exist at the leaf level only");
        return -H2W_EINVAL;
    }
    const auto &l = h->plan.near[box];
    for (size_t q = 0; q < l.size() && (int)q < cap; ++q)
        if (nb) nb[q] = l[q];
    return (int)l.size();
}

int h2w_bench_stream_read(int device, int64_t bytes, int nrep, double *gbps) {
    H2W_TRY
    if (!gbps || nrep < 1 || bytes < (1 << 20)) throw Error{H2W_EINVAL, "bad argument"};
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0)
        throw Error{H2W_ENOLIB, "no HIP device visible; libh2w has no CPU fallback"};
    if (device < 0 || device >= ndev) throw Error{H2W_EINVAL, "device ordinal out of range"};
    H2W_HIP(hipSetDevice(device));
    bytes -= bytes % h2w::stream_chunk_bytes();
    int cus = 0;
    H2W_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device));
    const int grid = 16 * std::max(cus, 1);
    h2w::DevBuf<uint8_t> buf;
    h2w::DevBuf<uint32_t> sink;
    buf.alloc(bytes);
    sink.alloc(grid);
    // (on the null stream, which waits for the device's other work before it starts)
    h2w::Event e0, e1;
    H2W_HIP(hipMemset(buf.p, 0x5A, bytes));
    h2w::launch_stream_read(buf.p, bytes, sink.p, grid, nullptr);  // warm-up
    H2W_HIP(hipEventRecord(e0, nullptr));
    for (int r = 0; r < nrep; ++r) h2w::launch_stream_read(buf.p, bytes, sink.p, grid, nullptr);
    H2W_HIP(hipEventRecord(e1, nullptr));
    H2W_HIP(hipGetLastError());
    const double ms_total = h2w::elapsed_ms(e0, e1);
    H2W_HIP(hipDeviceSynchronize());
    *gbps = (double)bytes * nrep / (ms_total * 1e-3) * 1e-9;
    return H2W_OK;
    H2W_CATCH
}

int h2w_bench_matvec(h2w_handle *h, int nrep, int precision, h2w_bench *out) {
    H2W_TRY
    if (!h || !out || nrep < 1) throw Error{H2W_EINVAL, "bad argument"};
    if (!h->assembled) throw Error{H2W_ESTATE, "not assembled"};
    if (precision < H2W_FP64 || precision > H2W_FP32_INNER) throw Error{H2W_EINVAL, "bad precision"};
    if (h2w::is32(precision) && !h->mat32.p) throw Error{H2W_ESTATE, "FP32 shadow not built"};
    if (h->cplx && precision != H2W_FP64) throw Error{H2W_EINVAL, "complex kernels: precision H2W_FP64 only"};
    const auto &LL = h2w::launches_for(*h, precision);
    H2W_HIP(hipSetDevice(h->opts.device));
    std::memset(out, 0, sizeof(*out));
    hipStream_t s = h->stream;
    const int64_t N = h->N;
    // deterministic input in the pool's x segment
    if (h->cplx) h2w::launch_fill(h->vec64.p + 2 * h->off_x, 2 * N, 1.0, s);
    else {
        h2w::launch_fill(h->vec64.p + h->off_x, N, 1.0, s);
        h2w::launch_fill32(h->vec32.p + h->off_x, N, 1.0f, s);
    }
    const int nl = std::min<int>((int)h2w::launches_for(*h, precision).size(), H2W_MAX_LAUNCHES - 1);
    std::vector<h2w::Event> ev(nl + 2);
    std::vector<double> acc(nl + 1, 0.0);
    // warm-up
    h2w::zero_outputs(*h, precision);
    h2w::run_launches(*h, precision);
    H2W_HIP(hipStreamSynchronize(s));
    h2w::Event t0, t1;
    H2W_HIP(hipEventRecord(t0, s));
    for (int r = 0; r < nrep; ++r) {
        h2w::zero_outputs(*h, precision);
        h2w::run_launches(*h, precision);
    }
    H2W_HIP(hipEventRecord(t1, s));
    out->ms_per_matvec = h2w::elapsed_ms(t0, t1) / nrep;
    // per-launch durations: fill + each bgemv launch
    for (int r = 0; r < nrep; ++r) {
        H2W_HIP(hipEventRecord(ev[0], s));
        h2w::zero_outputs(*h, precision);
        H2W_HIP(hipEventRecord(ev[1], s));
        for (int q = 0; q < nl; ++q) {
            h2w::run_launch(*h, LL[q], precision);
            H2W_HIP(hipEventRecord(ev[q + 2], s));
        }
        for (int q = 0; q <= nl; ++q) acc[q] += h2w::elapsed_ms(ev[q], ev[q + 1]);
    }
    out->n_launch = nl + 1;
    const int es = h->cplx ? 16 : h2w::is32(precision) ? 4 : 8;
    out->launch_ms[0] = acc[0] / nrep;
    out->launch_bytes[0] = (h->vec_len - h->off_y) * (int64_t)es;
    out->launch_role[0] = -1;
    for (int q = 0; q < nl; ++q) {
        out->launch_ms[q + 1] = acc[q + 1] / nrep;
        auto &Lh = LL[q];
        out->launch_role[q + 1] = Lh.role;
        out->launch_bytes[q + 1] =
            (precision == H2W_FP32_INNER ? h->inner.elems[q] : h->launch_elems[q]) * es;
        if ((precision == H2W_FP32_OTF || precision == H2W_FP64_OTF) && Lh.role == 1) {
            // the on-the-fly launches evaluate every entry of the directed lists (both
            // directions of each pair), element size times that count
            int64_t e = 0;
            for (auto v : h->otf.elems) e += v;
            out->launch_bytes[q + 1] = e * es;
        }
    }
    return H2W_OK;
    H2W_CATCH
}

int h2w_set_inner_tolerance(h2w_handle *h, double ir_tol_pow) {
    H2W_TRY
    if (!h) throw Error{H2W_EINVAL, "NULL handle"};
    if (!h->assembled) throw Error{H2W_ESTATE, "not assembled"};
    if (h->cplx) throw Error{H2W_EINVAL, "complex kernels: FP64 operators only (no inner operator)"};
    if (!h->mat32.p) throw Error{H2W_ESTATE, "the inner operator needs the FP32 shadow (opts.fp32_shadow)"};
    if (!(ir_tol_pow >= 0.0) || (ir_tol_pow > 0.0 && ir_tol_pow >= h->tol_pow))
        throw Error{H2W_EINVAL, "ir_tol_pow must be 0 or in (0, tol_pow)"};
    H2W_HIP(hipSetDevice(h->opts.device));
    h2w::build_inner(*h, ir_tol_pow);
    return H2W_OK;
    H2W_CATCH
}

int h2w_set_deflation(h2w_handle *h, int m, int k, int precision) {
    H2W_TRY
    if (!h) throw Error{H2W_EINVAL, "NULL handle"};
    if (!h->assembled) throw Error{H2W_ESTATE, "not assembled"};
    if (h->cplx) throw Error{H2W_EINVAL, "complex kernels: no refinement, no deflation space"};
    if (m < 0 || m > 512 || m == 1) throw Error{H2W_EINVAL, "m must be 0 or in [2, 512]"};
    if (k < 0 || k > m) throw Error{H2W_EINVAL, "k must be in [0, m]"};
    if (precision != H2W_FP32 && precision != H2W_FP32_INNER && precision != H2W_FP32_OTF)
        throw Error{H2W_EINVAL, "precision must be an inner precision (H2W_FP32, H2W_FP32_INNER, H2W_FP32_OTF)"};
    if ((precision == H2W_FP32 || precision == H2W_FP32_INNER) && !h->mat32.p)
        throw Error{H2W_ESTATE, "the FP32 operators need the FP32 shadow (opts.fp32_shadow)"};
    if (precision == H2W_FP32_INNER && !(h->ir_exp > 0.0)) throw Error{H2W_ESTATE, "no inner operator built"};
    if ((int64_t)m >= h->N) throw Error{H2W_EINVAL, "m must be below N"};
    H2W_HIP(hipSetDevice(h->opts.device));
    h2w::build_deflation(*h, m, k, precision);
    return H2W_OK;
    H2W_CATCH
}

int h2w_autotune(h2w_handle *h, const double *b, int where, double tol, int max_iter, int flags, h2w_tune *out) {
    H2W_TRY
    if (!h || !out) throw Error{H2W_EINVAL, "NULL argument"};
    if (!h->assembled) throw Error{H2W_ESTATE, "not assembled"};
    if (flags & ~(H2W_TUNE_UNROLL | H2W_TUNE_INNER | H2W_TUNE_DEFLATION)) throw Error{H2W_EINVAL, "unknown flags"};
    if (h->cplx) throw Error{H2W_EINVAL, "complex kernels: no autotuner (one complex GEMV kernel)"};
    const bool solves = (flags & (H2W_TUNE_INNER | H2W_TUNE_DEFLATION)) != 0;
    if (solves && (!b || max_iter < 1 || !(tol > 0.0)))
        throw Error{H2W_EINVAL, "inner and deflation tuning need b, tol > 0 and max_iter >= 1"};
    if (solves && !h->mat32.p) throw Error{H2W_ESTATE, "FP32 shadow not built"};
    if ((flags & H2W_TUNE_DEFLATION) && !(flags & H2W_TUNE_INNER) && h->inner.launches.empty())
        throw Error{H2W_ESTATE, "deflation tuning needs an inner operator"};
    H2W_HIP(hipSetDevice(h->opts.device));
    std::memset(out, 0, sizeof(*out));
    const int64_t N = h->N;
    hipStream_t s = h->stream;
    const int precs[3] = {H2W_FP64, H2W_FP32, H2W_FP32_INNER};
    auto have = [&](int p) {
        return p == H2W_FP64 || (h->mat32.p && (p != H2W_FP32_INNER || !h->inner.launches.empty()));
    };
    for (int q = 0; q < 3; ++q) out->matvec_ms_before[q] = have(precs[q]) ? h2w::time_matvec(*h, precs[q], 5) : 0.0;
    if (flags & H2W_TUNE_UNROLL)
        for (int q = 0; q < 2; ++q)
            if (have(precs[q])) h2w::tune_unroll(*h, precs[q]);
    h2w::DevBuf<double> bin, bt;
    if (solves) {
        h->g_x.ensure(N);
        h->g_r.ensure(N);
        h->g_d.ensure(N);
        bt.alloc(N);
        const double *bsrc = b;
        if (where == H2W_HOST) {
            bin.alloc(N);
            H2W_HIP(hipMemcpyAsync(bin.p, b, N * 8, hipMemcpyHostToDevice, s));
            bsrc = bin.p;
        }
        h2w::launch_permute_in(bsrc, N, bt.p, N, h->d_perm.p, N, 1, s);
        H2W_HIP(hipStreamSynchronize(s));
    }
    if (flags & H2W_TUNE_INNER) {
        h2w::tune_inner(*h, bt.p, tol, max_iter, (flags & H2W_TUNE_UNROLL) != 0, out);
    } else {
        if ((flags & H2W_TUNE_UNROLL) && have(H2W_FP32_INNER)) h2w::tune_unroll(*h, H2W_FP32_INNER);
        out->ir_tol_exp = h->inner.launches.empty() ? 0.0 : h->ir_exp;
    }
    if ((flags & H2W_TUNE_DEFLATION) && !h->inner.launches.empty())
        h2w::tune_deflation(*h, bt.p, tol, max_iter, (flags & H2W_TUNE_UNROLL) != 0, (flags & H2W_TUNE_INNER) != 0,
                            out);
    for (int q = 0; q < 3; ++q) out->matvec_ms_after[q] = have(precs[q]) ? h2w::time_matvec(*h, precs[q], 5) : 0.0;
    H2W_HIP(hipStreamSynchronize(s));
    return H2W_OK;
    H2W_CATCH
}

int h2w_set_rank_model(h2w_handle *h, const uint16_t *params, int64_t count) {
    H2W_TRY
    if (!h) throw Error{H2W_EINVAL, "NULL handle"};
    if (params && count != h2w::kRankParams)
        throw Error{H2W_EINVAL, "rank model: expected " + std::to_string(h2w::kRankParams) + " BF16 parameters"};
    if (h->opts.plan_only) throw Error{H2W_ESTATE, "handle was created with plan_only"};
    H2W_HIP(hipSetDevice(h->opts.device));
    if (!params) {
        h->rank_model.release();
        return H2W_OK;
    }
    std::vector<uint16_t> v(params, params + count);
    h->rank_model.upload(v, h->stream);
    H2W_HIP(hipStreamSynchronize(h->stream));
    return H2W_OK;
    H2W_CATCH
}

int64_t h2w_rank_samples(const h2w_handle *h, float *feat, int32_t *rank, int64_t cap) {
    if (!h) {
        h2w::set_error("NULL handle");
        return -H2W_EINVAL;
    }
    const int64_t n = (int64_t)h->sample_rank.size();
    for (int64_t q = 0; q < std::min(n, cap); ++q) {
        if (feat) std::copy(h->sample_feat[q].begin(), h->sample_feat[q].end(), feat + q * h2w::kRankFeatures);
        if (rank) rank[q] = h->sample_rank[q];
    }
    return n;
}

int h2w_rank_predict(h2w_handle *h, const float *feat, int64_t n, float *out) {
    H2W_TRY
    if (!h || (!feat && n > 0) || (!out && n > 0) || n < 0) throw Error{H2W_EINVAL, "bad arguments"};
    if (!h->rank_model.p) throw Error{H2W_ESTATE, "no rank model (h2w_set_rank_model)"};
    H2W_HIP(hipSetDevice(h->opts.device));
    if (n == 0) return H2W_OK;
    std::vector<float> F(feat, feat + n * h2w::kRankFeatures);
    h2w::DevBuf<float> dF, dO;
    dF.upload(F, h->stream);
    dO.alloc(n);
    h2w::launch_rank_mlp(dF.p, (int)n, h->rank_model.p, dO.p, h->stream);
    H2W_HIP(hipGetLastError());
    H2W_HIP(hipMemcpyAsync(out, dO.p, n * 4, hipMemcpyDeviceToHost, h->stream));
    H2W_HIP(hipStreamSynchronize(h->stream));
    return H2W_OK;
    H2W_CATCH
}

void h2w_destroy(h2w_handle *h) {
    if (!h) return;
    if (!h->opts.plan_only) (void)hipSetDevice(h->opts.device);
    if (h->stream) (void)hipStreamSynchronize(h->stream);
    h2w::drop_graphs(*h);
    if (h->stream) (void)hipStreamDestroy(h->stream);
    delete h;
}

}  // extern "C"
