// sgs_resident.hip -- the multicolour SGS-preconditioned BiCGSTAB (sgs.hip) of systems that fit
// the registers of the device, many iterations in one launch.
//
// An iteration of sgs.hip is 4 nc + 1 dependent launches, 43 us on two colours at 48^3 (110,592
// rows) whatever the data; here it takes 16 us, bound by nine hops of 0.3-0.5 us between blocks
// and three reductions of 1.7 us.  Each thread keeps one position: its off-diagonal entries,
// 1 / d and its elements of all vectors stay in registers, and blocks exchange, through words
// that carry their own flag (exchange.h), only what a sweep hands to a neighbour:
//   F: the forward result y (z) of a position, read by the forward sweeps of later colours and,
//      for the last colour, by the backward sweeps;
//   B: the final value of a colour that is neither the first nor the last, read by the backward
//      sweeps of earlier colours;
//   E: the backward correction, read by the products.
// A sweep waits for its neighbours' words only; a wave takes its positions colour by colour, so
// that no lane waits for a later step of its own wave.  The three reductions, (r0, v), (t, t)
// with (t, s), and (r0, r) with (r, r), gather at one block that has no rows (resident.hip) and
// order everything else: the words of the y half are marked again after the first, those of the
// z half after the second, each block's sums after their own totals, and every mark is in
// memory (the s_waitcnt before the first two reductions) before its owner takes part in the
// reduction after which the word is polled next; the totals are marked one reduction later,
// when every block has read them, and are in memory before the next totals are posted.
// Sums run per thread, wave, 256 positions and then over those in index order, as in sgs.hip, and
// the sweeps and updates use its expressions: the iterates are the same bits.
// Every wait is bounded, as in resident.hip.
#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>

#include <algorithm>

#include "exchange.h"
#include "resident.h"
#include "sgs.h"

namespace prism_hip {

namespace {

constexpr int BS = RES_BS;
constexpr int NW = BS / 64;
constexpr int SUB = BS / SGS_BS;     // groups of SGS_BS positions in a block
constexpr int SUBW = SGS_BS / 64;    // waves of such a group
constexpr double EPS = 2.220446049250313e-16;

// words of a block's line: (r0, v); (t, t), (t, s); (r0, r), (r, r); SUB of each
enum { LINE_V = 0, LINE_T = SUB, LINE_X = 3 * SUB, LINE_USED = 5 * SUB };
static_assert(LINE_USED <= RES_LINE && SUB == 2);

struct Sums {
    unsigned long long* line;  // of block 0, this launch
    int G, lb;
    unsigned limit;
    int* stuck;
    int* fail;
    double* sh;  // 2 NW wave sums, then 2 totals
};

// Totals of K values per thread over all positions (words at `at` of each line).  own: this
// block's sums (of thread k SUB + u: value k, group u).  False when the launch is to end.
template <int K>
__device__ inline bool totals(const Sums& S, int at, const double (&v)[K], double (&out)[K], double& own) {
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    {
        const double two[2] = {v[0], v[K - 1]};
        const double s = waveSums<2>(two);
#pragma unroll
        for (int k = 0; k < K; ++k)
            if (lane == sumLane<2>(k)) S.sh[k * NW + w] = s;
    }
    __syncthreads();
    if (tid < K * SUB) {
        double s = 0.0;
#pragma unroll
        for (int i = 0; i < SUBW; ++i) s += S.sh[(tid / SUB) * NW + (tid % SUB) * SUBW + i];
        own = s;
        if (S.lb < S.G) post(&S.line[RES_LINE * S.lb + at + tid], asWord(s));
    }
    unsigned polls = 0;
    if (S.lb == S.G) {
        // wave w: value w / SUBW, groups (w % SUBW) 64 + lane and 256 further (reduceParts in sgs.hip)
        const int k = w / SUBW, i = (w % SUBW) * 64 + lane;
        __syncthreads();  // sh is written again
        if (k < K) {
            unsigned long long u[2];
            const unsigned long long* p[2];
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const int g = i + q * SGS_BS;
                p[q] = g < SUB * S.G ? &S.line[RES_LINE * (g / SUB) + at + k * SUB + g % SUB] : nullptr;
                u[q] = p[q] ? peek(p[q]) : 0;
            }
            bool miss;
            do {
                miss = false;
#pragma unroll
                for (int q = 0; q < 2; ++q)
                    if (u[q] == Word<double>::MARK) {
                        u[q] = peek(p[q]);
                        miss |= u[q] == Word<double>::MARK;
                    }
            } while (miss && keepWaiting(polls, S.limit, S.stuck, S.fail));
            const double t = (0.0 + asValue<double>(u[0])) + asValue<double>(u[1]);
            const double two[2] = {t, t};
            const double s = waveSums<2>(two);
            if (lane == 0) S.sh[k * NW + w % SUBW] = s;
        }
        // the marks of earlier totals are in memory before these are posted
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (tid < K * RES_COPIES) {
            double s = 0.0;
#pragma unroll
            for (int q = 0; q < SUBW; ++q) s += S.sh[(tid / RES_COPIES) * NW + q];
            post(&S.line[RES_LINE * (S.G + tid % RES_COPIES) + at + (tid / RES_COPIES) * SUB], asWord(s));
            if (tid % RES_COPIES == 0) S.sh[2 * NW + tid / RES_COPIES] = s;
        }
    } else if (tid < K) {
        const unsigned long long* p =
            &S.line[RES_LINE * (S.G + (int)(blockIdx.x & (RES_COPIES - 1))) + at + tid * SUB];
        unsigned long long u = peek(p);
        while (u == Word<double>::MARK && keepWaiting(polls, S.limit, S.stuck, S.fail)) u = peek(p);
        S.sh[2 * NW + tid] = asValue<double>(u);
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; ++k) out[k] = S.sh[2 * NW + k];
    return *S.fail == 0;
}

template <int W>
__global__ void __launch_bounds__(BS) k_sgs_resident(SgsView V, SgsResidentView R, long long k0, int fresh) {
    constexpr unsigned long long MARK = Word<double>::MARK;
    __shared__ double sh[2 * NW + 2], sh0[3 * SUBW];
    __shared__ int fail, gone;
    SgsState* st = V.st;
    const int tid = threadIdx.x, lane = tid & 63, G = R.blocks, n = V.n, nc = V.nc;
    const int lb = (int)blockIdx.x < G ? (int)blockIdx.x : G;
    // One thread's reading of the event words decides for its block: a launch whose first test finds an
    // event ends without any exchange, so block 0 may write it while other blocks begin.  Those
    // that see it leave whole, their stale words marked; the others find the same event themselves.
    const int event = st->done | st->flag | st->stuck;
    if (tid < RES_LINE * (lb < G ? 1 : RES_COPIES)) post(&R.stale[RES_LINE * lb + tid], MARK);
    if (tid == 0) {
        fail = 0;
        gone = event;
    }
    // totals of the last X (or the seed), as the first kernel of an iteration forms them
    double red[3];
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        double s = 0.0;
        if (tid < SGS_BS)
            for (int i = tid; i < V.G; i += SGS_BS) s += V.part_x[q * V.G + i];
        const double two[2] = {s, s};
        s = waveSums<2>(two);
        if (tid < SGS_BS && lane == 0) sh0[q * SUBW + (tid >> 6)] = s;
    }
    __syncthreads();
    if (gone) return;
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        double s = 0.0;
#pragma unroll
        for (int i = 0; i < SUBW; ++i) s += sh0[q * SUBW + i];
        red[q] = s;
    }
    const Sums S{R.line, G, lb, R.spin, &st->stuck, &fail, sh};

    // this thread's position
    const int i = lb * BS + tid;
    const bool ok = lb < G && i < n;
    int c = 0, lo = 0, hi = 0;
    for (int q = 0; q < nc; ++q)
        if (ok && i >= V.cptr[q]) {
            c = q;
            lo = V.cptr[q];
            hi = V.cptr[q + 1];
        }
    double a[W];
    unsigned at[W];
    unsigned before = 0, after = 0, final = 0;  // entries of earlier and later colours; of the last colour
    {
        const int o = ok ? V.soff[i >> 6] : 0, w = ok ? (V.soff[(i >> 6) + 1] - o) >> 6 : 0;
#pragma unroll
        for (int k = 0; k < W; ++k) {
            int j = i;
            a[k] = 0.0;
            if (k < w) {
                j = V.scol[o + 64 * k + (i & 63)];
                a[k] = V.sval[o + 64 * k + (i & 63)];
            }
            at[k] = (unsigned)j * 8u;
            if (k < w && j < lo) before |= 1u << k;
            if (k < w && j >= hi) after |= 1u << k;
            if (k < w && j >= V.cptr[nc - 1]) final |= 1u << k;
        }
    }
    const unsigned me = ok ? (unsigned)i * 8u : FAR;
    auto load = [&](const double* p) { return ok ? p[i] : 0.0; };
    const double dinv = load(V.dinv), r0 = load(V.r0);
    double x = load(V.x), r = load(V.r), p = load(V.p), v = load(V.v), y = 0.0, s = 0.0, z = 0.0, t = 0.0;
    // colours of this wave's positions
    int cmin = 0, cmax = -1;
    for (int q = nc - 1; q >= 0; --q)
        if (__ballot(ok && c == q)) {
            cmin = q;
            if (cmax < 0) cmax = q;
        }

    const __amdgpu_buffer_rsrc_t pub = __builtin_amdgcn_make_buffer_rsrc(R.pub, 0, 6 * n * 8, 0x00020000);
    const unsigned bytes = (unsigned)n * 8u;
    // sum over the entries in `use` of a_ij w_j: w published at byte `base`, or at `other` where
    // the bit of `elsewhere` is set.  A word not there yet makes the sum a NaN (resident.hip).
    auto gather = [&](unsigned use, unsigned base, unsigned elsewhere, unsigned other) {
        unsigned long long u[W];
        auto from = [&](int k) {
            return bufPeek<unsigned long long>(
                pub, use >> k & 1 ? at[k] + (elsewhere >> k & 1 ? other : base) : FAR, 0);
        };
#pragma unroll
        for (int k = 0; k < W; ++k) u[k] = from(k);
        unsigned polls = 0;
        for (;;) {
            double sum = 0.0;
#pragma unroll
            for (int k = 0; k < W; ++k)
                if (use >> k & 1) sum += a[k] * asValue<double>(u[k]);
            if (sum == sum) return sum;
            bool miss = false;
            asm volatile("" ::: "memory");
#pragma unroll
            for (int k = 0; k < W; ++k)
                if (u[k] == MARK) {
                    miss = true;
                    u[k] = from(k);
                }
            if (!miss || !keepWaiting(polls, R.spin, &st->stuck, &fail)) return sum;
        }
    };
    // w = M^-1 u and A w (sgs.hip: forward, backward, product), words F, B, E at byte `half`
    auto sweep = [&](double u, double& w, unsigned half) {
        const unsigned F = half, B = half + bytes, E = half + 2 * bytes;
        for (int q = cmin; q <= cmax; ++q)
            if (ok && c == q) {
                const double lw = q > 0 ? gather(before, F, 0u, 0u) : 0.0;
                w = (u - lw) * dinv;
                bufPost(pub, me, F, asWord(w));
            }
        for (int q = std::min(cmax, nc - 2); q >= cmin; --q)
            if (ok && c == q) {
                const double e = -gather(after, B, final, F) * dinv;
                w += e;
                bufPost(pub, me, E, asWord(e));
                if (q > 0) bufPost(pub, me, B, asWord(w));
            }
        return ok ? u + (c > 0 ? gather(before, E, 0u, 0u) : 0.0) : 0.0;
    };
    auto markHalf = [&](unsigned half) {
        bufPost(pub, me, half, MARK);
        bufPost(pub, me, half + bytes, MARK);
        bufPost(pub, me, half + 2 * bytes, MARK);
    };
    auto markSums = [&](int word, int words) {  // a block's own
        if (lb < G && tid < words) post(&R.line[RES_LINE * lb + word + tid], MARK);
    };
    auto markTotals = [&](int word, int words) {  // the summing block's
        if (lb == G && tid < words * RES_COPIES) post(&R.line[RES_LINE * (G + tid / words) + word + tid % words], MARK);
    };

    const SgsSlot prev = st->s[(int)(k0 & 1) ^ 1];
    double rho = 0.0, alpha = prev.alpha, omega = prev.omega, beta = 0.0, rho_old = prev.rho;
    double tol2 = st->tol2, r0sq = prev.r0sq, own = 0.0, ownX = 0.0, rr = 0.0;
    if (fresh == 1) tol2 = st->tol * st->tol * red[2];
    if (fresh) r0sq = red[1];
    int done = 0, flag = 0, m = 0;
    double xt[2] = {red[0], red[1]};
    for (;;) {
        if (m >= R.quota) break;
        rho = xt[0];
        rr = xt[1];
        beta = (rho / rho_old) * (alpha / omega);
        const bool first = m == 0 && fresh;
        if (fresh == 1 && m == 0 && red[2] == 0.0) done = 4;  // Eigen: b == 0 -> x = 0
        else if (!(rr == rr)) done = 3;
        else if (rr <= tol2) done = 1;
        else if (!first && fabs(rho) < EPS * EPS * r0sq) flag = 2;
        if (done || flag) break;
        p = r + beta * (p - omega * v);
        v = sweep(p, y, 0u);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        const double dv[1] = {0.0 + r0 * v};
        double tv[1];
        if (!totals<1>(S, LINE_V, dv, tv, own)) return;
        if (m > 0) markTotals(LINE_X, 2 * SUB);
        markSums(LINE_V, SUB);
        markHalf(0u);
        alpha = rho / tv[0];
        s = r - alpha * v;
        t = sweep(s, z, 3 * bytes);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        const double dt[2] = {0.0 + t * t, 0.0 + t * s};
        double tt[2];
        if (!totals<2>(S, LINE_T, dt, tt, own)) return;
        markTotals(LINE_V, SUB);
        markSums(LINE_T, 2 * SUB);
        markHalf(3 * bytes);
        omega = tt[0] > 0.0 ? tt[1] / tt[0] : 0.0;
        x += alpha * y + omega * z;
        r = s - omega * t;
        const double dx[2] = {0.0 + r0 * r, 0.0 + r * r};
        if (!totals<2>(S, LINE_X, dx, xt, ownX)) return;
        markTotals(LINE_T, 2 * SUB);
        markSums(LINE_X, 2 * SUB);
        rho_old = rho;
        ++m;
    }
    if (m > 0 && ok) {
        V.x[i] = x;
        V.r[i] = r;
        V.p[i] = p;
        V.v[i] = v;
    }
    if (m > 0 && lb < G && tid < 2 * SUB && SUB * lb + tid % SUB < V.G)
        V.part_x[(tid / SUB) * V.G + SUB * lb + tid % SUB] = ownX;
    if (lb == 0 && tid == 0) {
        st->rr = rr;
        if (fresh == 1) {
            st->bb = red[2];
            st->tol2 = tol2;
        }
        if (m > 0) st->s[(int)((k0 + m) & 1) ^ 1] = SgsSlot{rho_old, alpha, omega, beta, r0sq};
        if (done || flag) {
            st->done = done;
            st->flag = flag;
            st->k_event = k0 + m;
        }
    }
}

}  // namespace

bool sgs_resident_fits(int n, int wmax, int n_cu, int* blocks) {
    *blocks = (n + BS - 1) / BS;
    return n > 0 && wmax <= 8 && *blocks <= std::min(n_cu - 1, RES_MAX_BLOCKS);
}

void launch_sgs_resident(const Launch& L, const SgsView& V, const SgsResidentView& R, int wmax, long long k, int fresh) {
    if (wmax <= 4) PRISM_LAUNCH("sgs_resident", k_sgs_resident<4>, R.blocks + 1, BS, V, R, k, fresh);
    else if (wmax <= 6) PRISM_LAUNCH("sgs_resident", k_sgs_resident<6>, R.blocks + 1, BS, V, R, k, fresh);
    else PRISM_LAUNCH("sgs_resident", k_sgs_resident<8>, R.blocks + 1, BS, V, R, k, fresh);
}

}  // namespace prism_hip
