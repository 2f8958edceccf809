// resident.hip -- BiCGSTAB iterations of small and medium systems in one resident kernel.
//
// The three-kernel iteration (krylov.hip) of a system that fits the caches is bound by its
// launches: a dependent launch costs 2.4 us and its prologue 2-3 us more, 14-20 us per
// iteration, where the data would take 1-4 us (64^3 cells, 20 MB).  Here one launch runs up
// to `quota` iterations of the same recurrences.  Each thread keeps R rows: their matrix entries
// (values and element addresses) and their elements of x, r, r0, rhat, p, v, s and t stay in
// registers from the first iteration to the last (but see keptRows), so an iteration moves only
// p and s between blocks, and the partial sums of its two reductions.  Per iteration, three kernels -> this
// one: 200 rows FP64 14 -> 2.6 us, 16,384 rows FP64 15 -> 5.8 us, 82,944 rows of tetrahedra
// FP32 17.5 -> 7.0 us, 110,592 rows FP64 17 -> 7.8 us, 262,144 rows FP64 19.3 -> 10.0 us,
// 512,000 rows FP64 29.8 -> 18.7 us.  What bounds it now is latency: four to five hops of
// 0.3-0.5 us between blocks per iteration, and at two and three rows per thread (262,144 rows
// are 1,088 a block: three in one wave of eight) the products' wait for their neighbours' words
// (0.7 us per row and product).
//
// Exchange without barriers.  A word that another block waits for carries its own flag: it
// holds the mark, a signalling NaN that no arithmetic produces (results are quiet NaNs), until
// its owner stores the value; a reader polls until the word is not the mark.  Loads and
// stores are relaxed atomics of agent scope, which all XCDs see without cache writebacks or
// invalidations.  Per iteration k:
//   sums (rhat, p_k), (r, r) -> the block's line; publish p_k
//   V: A p_k (waits for the neighbours' p only); wait for the two totals; alpha;
//      s = r - alpha v; publish s_k
//   T: t = A s (waits for the neighbours' s only); sums (t,t), (t,s), (r0,s), (r0,t); wait for
//      the four totals
//   X: omega, beta, x, r, p_{k+1}
// A block that has T's totals knows that every block has read s_k, the first two totals and
// p_k: at the start of iteration k + 1 it marks its words of p_{k-1} and s_k and those sums
// again (p_k stays: an event in iteration k + 1 hands it back to the host's state; the launch's
// last p is marked after one more round, when every block has read it); T's sums
// are marked after the next first totals.  Every word marked again is next polled after a
// reduction that its owner took part in only when the marks were in memory (the s_waitcnt
// before T's sums), so no reader sees an old value: p has three buffers, s, the sums and the
// totals two.  Elements of the block's own rows are read from LDS instead.
//
// The reductions sum per thread, wave, block and then over the blocks in index order, with one
// row per thread in exactly the order of the three-kernel iteration (of its kernels with a row per
// thread; those with packed rows have another).  One block more than
// the rows need does nothing else: a block that also has rows delays every reduction by its
// own products (64^3: 12.2 us per iteration instead of 11.0).
//
// All blocks must run at the same time: at most one per compute unit.  Every wait is bounded
// (rv.spin polls): if it runs out, ks->stuck tells the other blocks and the host, and the
// launch ends; the host continues with the three-kernel iteration from the current x.
#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>

#include <algorithm>

#include "../../include/prism_hip.h"
#include "exchange.h"
#include "internal.h"
#include "krylov.h"
#include "resident.h"

namespace prism_hip {

namespace {

constexpr int BS = RES_BS;
constexpr int NW = BS / 64;

__device__ inline double inOrder(const double* s) {  // the NW waves' sums
    double t = 0.0;
#pragma unroll
    for (int i = 0; i < NW; ++i) t += s[i];
    return t;
}

// blockIdx -> logical block: the blocks of one XCD own one contiguous range of rows.
__device__ inline int logicalBlock(int nblk) {
    const int b = blockIdx.x, q = nblk >> 3, r = nblk & 7, xcd = b & 7, idx = b >> 3;
    return (xcd < r) ? xcd * (q + 1) + idx : r * (q + 1) + (xcd - r) * q + idx;
}

// Totals over all blocks of K values per thread, in two halves: postSums hands in this block's
// sums (words slot[RES_LINE b + k] for block b, a cache line to each block), awaitTotals returns
// the totals (block G's words); what is done between them hides the round trip.  The block without
// rows (lb == G) gathers the sums and posts the totals that the others poll: every block
// polling every sum took 3.1 us a round on 256 blocks, all of them reading the same lines
// at once; one gather and one broadcast take 1.7 us.  The totals have a line for each XCD: 216
// blocks polling one line lengthened an iteration of 48^3 rows from 8.2 to 9.5 us.  A
// single block keeps both in LDS.
// sh: K NW sums of waves, then the K totals.
template <int K>
__device__ inline void postSums(const double (&v)[K], unsigned long long* slot, int G, int lb, double* sh) {
    const int tid = threadIdx.x, lane = tid & 63;
    const double s = waveSums<K>(v);
#pragma unroll
    for (int k = 0; k < K; ++k)
        if (lane == sumLane<K>(k)) sh[k * NW + (tid >> 6)] = s;
    __syncthreads();
    if (G > 1 && lb < G && tid < K) post(&slot[RES_LINE * lb + tid], asWord(inOrder(sh + tid * NW)));
}
template <int K>
__device__ inline bool awaitTotals(unsigned long long* slot, int G, int lb, unsigned limit, KrylovScalars* ks,
                                   double* sh, int* fail, double (&out)[K]) {
    const int tid = threadIdx.x, lane = tid & 63;
    if (G == 1) {
#pragma unroll
        for (int k = 0; k < K; ++k) out[k] = inOrder(sh + k * NW);
        return true;
    }
    unsigned polls = 0;
    if (lb == G) {  // wave k gathers the sums k of up to RES_MAX_BLOCKS blocks
        const int k = tid >> 6;
        if (k < K) {
            unsigned long long u[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) u[i] = lane + 64 * i < G ? peek(&slot[RES_LINE * (lane + 64 * i) + k]) : 0;
            bool miss;
            do {
                miss = false;
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (u[i] == Word<double>::MARK) {
                        u[i] = peek(&slot[RES_LINE * (lane + 64 * i) + k]);
                        miss |= u[i] == Word<double>::MARK;
                    }
            } while (miss && keepWaiting(polls, limit, &ks->stuck, fail));
            const double part[4] = {asValue<double>(u[0]), asValue<double>(u[1]), asValue<double>(u[2]),
                                    asValue<double>(u[3])};
            const double s = waveSums<4>(part);
            double t = 0.0;
#pragma unroll
            for (int i = 0; i < 4; ++i) t += laneValue(s, sumLane<4>(i));
            if (lane < RES_COPIES) post(&slot[RES_LINE * (G + lane) + k], asWord(t));
            if (lane == 0) sh[K * NW + k] = t;
        }
    } else if (tid < K) {
        const unsigned long long* total = &slot[RES_LINE * (G + (int)(blockIdx.x & (RES_COPIES - 1))) + tid];
        unsigned long long u = peek(total);
        while (u == Word<double>::MARK && keepWaiting(polls, limit, &ks->stuck, fail)) u = peek(total);
        sh[K * NW + tid] = asValue<double>(u);
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; ++k) out[k] = sh[K * NW + k];
    return *fail == 0;
}

// Orders the reads of a row's elements before their first use: one wait for all of them.  (Left
// alone, the compiler reads each into the same register and waits for it, W LDS latencies in a
// row.)  Up to two rows per thread in FP64, four in FP32: per iteration, without / with, seven
// diagonals, FP64 110,592 rows (one) 8.6 / 8.4 us, 180,000 rows (two) 8.9 / 8.6 us, FP32 262,144
// rows (three) 10.2 / 9.3 us, 512,000 rows (four) 12.4 / 10.4 us; 82,944 rows of tetrahedra in FP32
// 360 / 337 us per launch.  With more rows it spills up to 24 more registers, and 512,000 rows
// FP64 went from 18.7 to 19.1 us per iteration.
template <typename U, int W>
__device__ inline void together(U (&l)[W]) {
    if constexpr (W == 5) {
        asm volatile("" : "+v"(l[0]), "+v"(l[1]), "+v"(l[2]), "+v"(l[3]), "+v"(l[4]));
    } else if constexpr (W == 7) {
        asm volatile("" : "+v"(l[0]), "+v"(l[1]), "+v"(l[2]), "+v"(l[3]), "+v"(l[4]), "+v"(l[5]), "+v"(l[6]));
    } else {
        static_assert(W % 8 == 0);
#pragma unroll
        for (int k = 0; k < W; k += 8)
            asm volatile(""
                         : "+v"(l[k]), "+v"(l[k + 1]), "+v"(l[k + 2]), "+v"(l[k + 3]), "+v"(l[k + 4]), "+v"(l[k + 5]),
                           "+v"(l[k + 6]), "+v"(l[k + 7]));
    }
}

// Rows per thread up to which the coefficients stay in registers with everything else, and up
// to which the element addresses do.  Above the first, DIA coefficients (7 per row at most) are
// read again for each product: a thread's 256 registers hold 9 vectors, addresses and the elements
// on their way, and the coefficients of the whole system come from the L2s (4 MB each) and the
// Infinity Cache.  Above the second, the product goes row by row, the next row's elements and
// coefficients on their way, and forms the addresses each time (the compiler spills 51
// registers otherwise).  Per iteration, all rows at once / row by row: FP64 4 rows 18.7 / 21.3 us,
// 5 rows 30.1 / 26.7 us; FP32 5 rows 16.9 / 17.6 us, 6 rows 18.6 / 22.2 us, 7 rows 27.4 / 25.8 us.
template <typename T>
constexpr int keptRows() { return sizeof(T) == 8 ? 3 : 4; }
template <typename T>
constexpr int heldRows() { return sizeof(T) == 8 ? 4 : 6; }
// Rows per thread at most (see resident_plan).
template <typename T>
constexpr int mostRows(bool dia, int W) {
    return W == 16 ? 1 : dia && W <= 7 ? (sizeof(T) == 4 ? 6 : 5) : keptRows<T>();
}

// FP64: plain row products; FP32: the difference form (matRow in krylov.hip; the diagonal
// coefficient holds the row sum, or zero where the matrix has zero row sums).
template <typename T, bool DIA, int W, int R>
__global__ void __launch_bounds__(BS) k_resident(KView<T> kv, ResidentView<T> rv) {
    using U = typename Word<T>::U;
    constexpr U MARK = Word<T>::MARK;
    constexpr bool STREAM = R > keptRows<T>(), BYROW = R > heldRows<T>(),
                   AHEAD = R * sizeof(T) <= 16;  // see together
    constexpr bool DIFF = sizeof(T) == 4;
    __shared__ T own[2][R * BS + 1];  // this block's p and s, and a zero
    __shared__ double shA[2 * NW + 2], shC[4 * NW + 4];
    __shared__ int fail;
    KrylovScalars* ks = kv.ks;
    const int tid = threadIdx.x, G = rv.blocks, n = kv.n;
    // the last block has no rows: it gathers the sums of the others (a single block: none does)
    const int lb = (int)blockIdx.x < G ? logicalBlock(G) : G;
    const int r0 = lb < G ? lb * rv.rows : n, r1 = min(r0 + rv.rows, n);
    // rows of this wave: j < live holds one in some lane
    const int live = __builtin_amdgcn_readfirstlane(max(0, (r1 - r0 - (tid & ~63) + BS - 1) / BS));
    // done and flag: the same values in every thread of the grid, as a launch writes them only after
    // a last round of all blocks, so none leaves here with its stale words unmarked unless all
    // do.  stuck can be new: then this launch's results count for nothing.  (Marking first: 1.1 %
    // more per launch of 39,330 rows of tetrahedra FP32, by the compiler's schedule.)
    if (ks->done | ks->flag | ks->stuck) return;
    if (tid == 0) {
        fail = 0;
        own[0][R * BS] = own[1][R * BS] = T(0);
    }
    if (tid < RES_LINE * (lb < G ? 1 : RES_COPIES)) post(&rv.stale[RES_LINE * lb + tid], Word<double>::MARK);

    // this thread's rows r0 + tid + j BS; at[j][k]: where entry k's element is, as a byte offset
    // into own[] (this block's), or FAR + its byte offset in the published vector
    T a[STREAM ? 1 : R][W], x[R], r[R], z[R], h[R], p[R], v[R], s[R], t[R];
    unsigned at[BYROW ? 1 : R][W];
    auto rowOf = [&](int j) { return r0 + tid + j * BS; };
    auto mine = [&](int j) { return (unsigned)(tid + j * BS) * (unsigned)sizeof(T); };
    auto rowAt = [&](int j) { return rowOf(j) < r1 ? (unsigned)rowOf(j) * (unsigned)sizeof(T) : FAR; };
#pragma unroll
    for (int j = 0; j < R; ++j) {
        const int row = rowOf(j);
        const bool ok = row < r1;
        x[j] = ok ? kv.x[row] : T(0);
        r[j] = ok ? kv.r[row] : T(0);
        z[j] = ok ? kv.r0[row] : T(0);
        h[j] = ok ? kv.rhat[row] : T(0);
        p[j] = ok ? kv.p_new[row] : T(0);
        v[j] = s[j] = t[j] = T(0);
        int o = 0, w = 0;
        if (!DIA && ok) {
            o = kv.soff[row >> 6];
            w = (kv.soff[(row >> 6) + 1] - o) >> 6;
        }
#pragma unroll
        for (int k = 0; k < W; ++k) {
            int c = row;  // a missing entry: coefficient zero, the row's own element
            T e = T(0);
            if constexpr (DIA) {
                if (ok && k < kv.ndia && (unsigned)(row + kv.doff[k]) < (unsigned)n) {
                    c = row + kv.doff[k];
                    if constexpr (!STREAM) e = kv.sval[(int64_t)k * n + row];
                }
            } else if (k < w) {
                const int q = (int)sellPos(o, w, k, row & 63);
                c = kv.srel ? row + kv.sbase[(o >> 6) + k] + (int)kv.srel[q] : kv.scol[q];
                e = kv.sval[q];
            }
            if (DIFF && kv.diff == 2 && c == row) e = T(0);
            if constexpr (BYROW) continue;
            if constexpr (!STREAM) a[j][k] = e;
            const int l = ok ? c - r0 : 0;
            at[j][k] = (unsigned)l < (unsigned)rv.rows ? (unsigned)l * (unsigned)sizeof(T)
                                                        : FAR + (unsigned)c * (unsigned)sizeof(T);
        }
    }
    auto place = [&](int j, int k) {
        if constexpr (BYROW) {  // formed each time
            const int l = tid + j * BS + kv.doff[k], c = r0 + l;
            const bool in = k < kv.ndia && rowOf(j) < r1 && (unsigned)c < (unsigned)n;
            return !in ? mine(j) : (unsigned)l < (unsigned)rv.rows ? (unsigned)l * (unsigned)sizeof(T)
                                                                   : FAR + (unsigned)c * (unsigned)sizeof(T);
        } else {
            return at[j][k];
        }
    };
    unsigned long long wants = 0;  // bit j W + k: some lane of the wave reads entry k of row j from another block
#pragma unroll
    for (int j = 0; j < R; ++j)
#pragma unroll
        for (int k = 0; k < W; ++k)
            if (__ballot(place(j, k) >= FAR)) wants |= 1ull << (j * W + k);
    const __amdgpu_buffer_rsrc_t pub =
        __builtin_amdgcn_make_buffer_rsrc(rv.pub, 0, 5 * n * (int)sizeof(T), 0x00020000);
    const unsigned bytes = (unsigned)n * (unsigned)sizeof(T);  // of one published vector
    const __amdgpu_buffer_rsrc_t vals = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<T*>(kv.sval), 0, STREAM ? kv.ndia * n * (int)sizeof(T) : 0, 0x00020000);
    auto coef = [&](int j, int k) {
        if constexpr (STREAM) {  // of a row there is none of: reads as zero
            if (k >= kv.ndia || (DIFF && kv.diff == 2 && kv.doff[k] == 0)) return T(0);
            return asValue<T>(bufPeek<U, 0>(vals, rowAt(j), (unsigned)k * bytes));
        } else {
            return a[j][k];
        }
    };
    const bool mixed = kv.mixed != 0, pc = kv.precond != 0;
    const double tol2 = ks->tol2, ref2 = ks->delta2 * ks->rr_ref, tiny = ks->breakdown * ks->r0n;
    double rho = ks->rho[kv.par], alpha = ks->alpha, omega = ks->omega;
    double rho_old = 0.0, beta = 0.0, tt = 0.0, ts = 0.0, rp = 0.0, rr = 0.0;
    const long long iter0 = ks->iter, maxit = ks->maxit;
    int done = 0, flag = 0, m = 0;
    __syncthreads();  // fail

    // y = A w for the vector published at byte `base` (this block's elements in own[q]).  An
    // element that is not there yet reads as the mark and makes the row's sum a NaN: only then
    // are the elements looked at one by one.
    auto product = [&](unsigned base, int q, const T (&w)[R], T (&y)[R]) {
        const char* mem = reinterpret_cast<const char*>(own[q]);
        auto local = [&](unsigned at) {
            return asWord(*reinterpret_cast<const T*>(mem + min(at, (unsigned)(R * BS * sizeof(T)))));
        };
        if constexpr (BYROW) {
            // row by row, with the next row's values, addresses and far elements on their way
            T cf[2][W];
            U u[2][W];
            unsigned pl[2][W];
            auto issue = [&](int j) {
                if (j >= live) return;
#pragma unroll
                for (int k = 0; k < W; ++k) {
                    pl[j & 1][k] = place(j, k);
                    cf[j & 1][k] = coef(j, k);
                    u[j & 1][k] = U(0);
                    if (wants >> (j * W + k) & 1) u[j & 1][k] = bufPeek<U>(pub, pl[j & 1][k] ^ FAR, base);
                }
            };
            issue(0);
#pragma unroll
            for (int j = 0; j < R; ++j) {
                if (j + 1 < R) issue(j + 1);
                if (j >= live) continue;
                unsigned polls = 0;
                for (;;) {
                    T sum = T(0);
#pragma unroll
                    for (int k = 0; k < W; ++k) {
                        const T e = asValue<T>(local(pl[j & 1][k]) | u[j & 1][k]);
                        if (DIFF) sum += cf[j & 1][k] * (pl[j & 1][k] == mine(j) ? w[j] : e - w[j]);
                        else sum += cf[j & 1][k] * e;
                    }
                    y[j] = sum;
                    if (sum == sum) break;
                    bool miss = false;
                    asm volatile("" ::: "memory");
#pragma unroll
                    for (int k = 0; k < W; ++k)
                        if (u[j & 1][k] == MARK) {
                            miss = true;
                            u[j & 1][k] = bufPeek<U>(pub, pl[j & 1][k] ^ FAR, base);
                        }
                    if (!miss || !keepWaiting(polls, rv.spin, &ks->stuck, &fail)) break;
                }
            }
        } else {
            U u[R][W];
#pragma unroll
            for (int j = 0; j < R; ++j)
#pragma unroll
                for (int k = 0; k < W; ++k) {
                    asm volatile("" : "+v"(at[j][k]));  // no copies of what follows kept per iteration
                    u[j][k] = U(0);
                    if (wants >> (j * W + k) & 1) u[j][k] = bufPeek<U>(pub, at[j][k] ^ FAR, base);
                }
            unsigned polls = 0;
            for (;;) {
                bool nan = false;
#pragma unroll
                for (int j = 0; j < R; ++j) {
                    if (j >= live) continue;
                    T sum = T(0);
                    U l[W];
                    if constexpr (AHEAD) {
#pragma unroll
                        for (int k = 0; k < W; ++k) l[k] = local(at[j][k]);
                        together(l);
                    }
#pragma unroll
                    for (int k = 0; k < W; ++k) {
                        if constexpr (!AHEAD) l[k] = local(at[j][k]);
                        // one of the two is zero: own[q] ends with one, the buffer read was out of range
                        const T e = asValue<T>(l[k] | u[j][k]), c = coef(j, k);
                        if (DIFF) sum += c * (at[j][k] == mine(j) ? w[j] : e - w[j]);
                        else sum += c * e;
                    }
                    y[j] = sum;
                    nan |= sum != sum;
                }
                if (!nan) break;
                bool miss = false;
                asm volatile("" ::: "memory");
#pragma unroll
                for (int j = 0; j < R; ++j)
#pragma unroll
                    for (int k = 0; k < W; ++k)
                        if (u[j][k] == MARK) {
                            miss = true;
                            u[j][k] = bufPeek<U>(pub, at[j][k] ^ FAR, base);
                        }
                if (!miss || !keepWaiting(polls, rv.spin, &ks->stuck, &fail)) break;
            }
        }
    };
    auto keep = [&](int q, const T (&w)[R]) {
#pragma unroll
        for (int j = 0; j < R; ++j)
            if (j < live) own[q][tid + j * BS] = w[j];
    };
    auto publish = [&](unsigned base, const T (&w)[R]) {
#pragma unroll
        for (int j = 0; j < R; ++j)
            if (j < live) bufPost(pub, rowAt(j), base, asWord(w[j]));
    };
    auto mark = [&](unsigned base) {
#pragma unroll
        for (int j = 0; j < R; ++j)
            if (j < live) bufPost(pub, rowAt(j), base, MARK);
    };
    auto sBase = [&](int k) { return (unsigned)(3 + (k & 1)) * bytes; };
    // words of a block's line: the two sums of each parity, then the four of each parity; the
    // summing block's line (the last one) holds the totals
    auto slotA = [&](int k) { return rv.slots + (k & 1) * 2; };
    auto slotC = [&](int k) { return rv.slots + 4 + (k & 1) * 4; };
    auto markSums = [&](unsigned long long* sl, int words) {
        if (G > 1 && tid < (lb < G ? words : words * RES_COPIES))
            post(&sl[RES_LINE * (lb + tid / words) + tid % words], Word<double>::MARK);
    };

    double acc[2] = {0.0, 0.0};
#pragma unroll
    for (int j = 0; j < R; ++j) {
        acc[0] += (double)h[j] * (double)p[j];
        acc[1] += (double)r[j] * (double)r[j];
    }
    unsigned pm = 0, pm_old = 2;  // m modulo 3, and of the previous iteration
    for (;;) {
        keep(0, p);
        postSums<2>(acc, slotA(m), G, lb, shA);
        publish(pm * bytes, p);  // a single block's, too: p_{k-1} is read back at the end
        if (m > 0) {  // every block has read these
            if (m > 1 && G > 1) mark((pm_old == 0 ? 2 : pm_old - 1) * bytes);
            if (G > 1) mark(sBase(m - 1));
            markSums(slotA(m - 1), 2);
        }
        if (live) product(pm * bytes, 0, p, s);  // v_k; v keeps v_{k-1} until the event test
        double red[2];
        if (!awaitTotals<2>(slotA(m), G, lb, rv.spin, ks, shA, &fail, red)) return;
        rp = red[0];
        rr = red[1];
        if (m > 0) markSums(slotC(m - 1), 4);
        // convergence and events, in the order of the three-kernel iteration
        if (!(rr == rr)) done = 3;
        else if (mixed) {
            if (rr <= tol2 || rr <= ref2 || iter0 + m >= maxit) flag = 1;
        } else if (rr <= tol2) done = 1;
        else if (iter0 + m >= maxit) done = 2;
        if (!done && !flag) {
            if (!(rp == rp) || !(rho == rho)) done = 3;
            else if (fabs(rho) < tiny) flag = 2;
        }
        if (done || flag || m >= rv.quota) break;
        alpha = rho / rp;
        const T al = (T)alpha;
#pragma unroll
        for (int j = 0; j < R; ++j) {
            if (j >= live) continue;
            v[j] = s[j];
            s[j] = r[j] - al * v[j];
        }
        if (G > 1) publish(sBase(m), s);
        keep(1, s);
        __syncthreads();
        if (live) product(sBase(m), 1, s, t);
        double d[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int j = 0; j < R; ++j) {
            if (j >= live) continue;
            const double td = (double)t[j], sd = (double)s[j], zd = (double)z[j];
            d[0] += td * td;
            d[1] += td * sd;
            d[2] += zd * sd;
            d[3] += zd * td;
        }
        // the marks stored since the last of these sums are in memory before this block's are
        if (G > 1) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        postSums<4>(d, slotC(m), G, lb, shC);
        double tot[4];
        if (!awaitTotals<4>(slotC(m), G, lb, rv.spin, ks, shC, &fail, tot)) return;
        tt = tot[0];
        ts = tot[1];
        omega = tt > 0.0 ? ts / tt : 0.0;
        const double rho1 = tot[2] - omega * tot[3];
        beta = (rho1 / rho) * (alpha / omega);
        const T w = (T)omega, b = (T)beta;
        acc[0] = acc[1] = 0.0;
#pragma unroll
        for (int j = 0; j < R; ++j) {
            if (j >= live) continue;
            const T di = pc && rowOf(j) < r1 ? kv.dinv[rowOf(j)] : T(1);
            const T yi = pc ? di * p[j] : p[j], zi = pc ? di * s[j] : s[j];
            x[j] = x[j] + (al * yi + w * zi);
            r[j] = s[j] - w * t[j];
            p[j] = r[j] + b * (p[j] - w * v[j]);
            const double rd = (double)r[j];
            acc[0] += (double)h[j] * (double)p[j];
            acc[1] += rd * rd;
        }
        rho_old = rho;
        rho = rho1;
        ++m;
        pm_old = pm;
        pm = pm == 2 ? 0 : pm + 1;
    }

    // The totals say that every block has posted its sums, not that it has read its neighbours' p_k
    // yet: one more round (the next four sums' words are free), after which p_k can be marked.  A
    // block whose wait for this round's totals runs out leaves its old x beside the others' new
    // one: a valid guess, as the host starts anew from x and looks at nothing else (stuck).
    if (G > 1) {
        const double none[2] = {0.0, 0.0};
        double all[2];
        postSums<2>(none, slotC(m), G, lb, shC);
        if (!awaitTotals<2>(slotC(m), G, lb, rv.spin, ks, shC, &fail, all)) return;
    }
    // the state as the three-kernel iteration keeps it: p_k and rho_k in slot k & 1, p_{k-1},
    // v_{k-1} and rho_{k-1} in the other one
    const bool even = (m & 1) == 0;
    T* pk = even ? kv.p_new : kv.p_old;
    T* pl = even ? kv.p_old : kv.p_new;
    T* vl = even ? kv.v_old : kv.v_new;
    const bool flush = mixed && flag;
    if (m > 0 || flush) {
#pragma unroll
        for (int j = 0; j < R; ++j) {
            const int row = rowOf(j);
            if (row >= r1) continue;
            if (flush) rv.x64[row] += (double)x[j];
            kv.x[row] = flush ? T(0) : x[j];
        }
    }
    if (m > 0) {
#pragma unroll
        for (int j = 0; j < R; ++j) {
            const int row = rowOf(j);
            if (row >= r1) continue;
            kv.r[row] = r[j];
            pk[row] = p[j];
            pl[row] = asValue<T>(bufPeek<U>(pub, rowAt(j), pm_old * bytes));
            vl[row] = v[j];
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        mark(pm_old * bytes);
    }
    mark(pm * bytes);
    if (lb == 0)  // the partial sums that the three-kernel iteration's V reduces
        for (int i = tid; i < kv.G; i += BS) {
            kv.part_x[i] = i == 0 ? rp : 0.0;
            kv.part_x[kv.G + i] = i == 0 ? rr : 0.0;
        }
    if (lb == 0 && tid == 0) {
        ks->rr = rr;
        if (m > 0) {
            const int q = kv.par ^ (m & 1);
            ks->rho[q] = rho;
            ks->rho[q ^ 1] = rho_old;
            ks->alpha = alpha;
            ks->omega = omega;
            ks->beta = beta;
            ks->tt = tt;
            ks->ts = ts;
            ks->iter = iter0 + m;
            ks->nit += m;
        }
        ks->r0v = rp;
        if (done) ks->done = done;
        else if (flag) ks->flag = flag;
    }
}

template <typename T>
__global__ void k_mark(T* p, size_t count, unsigned long long* q, size_t more) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) reinterpret_cast<typename Word<T>::U*>(p)[i] = Word<T>::MARK;
    if (i < more) q[i] = Word<double>::MARK;
}

template <typename T, bool DIA, int W, int R>
void launchOne(const Launch& L, const KView<T>& kv, const ResidentView<T>& rv) {
    PRISM_LAUNCH(sizeof(T) == 8 ? "bicgstab_resident_f64" : "bicgstab_resident_f32", (k_resident<T, DIA, W, R>),
                 rv.blocks + (rv.blocks > 1 ? 1 : 0), BS, kv, rv);
}

// The instance with `rows` rows per thread: there is one for each number that a plan may ask for.
template <typename T, bool DIA, int W, int R = 1>
void launchRows(const Launch& L, const KView<T>& kv, const ResidentView<T>& rv, int rows) {
    if (rows == R) launchOne<T, DIA, W, R>(L, kv, rv);
    else if constexpr (R < mostRows<T>(DIA, W)) launchRows<T, DIA, W, R + 1>(L, kv, rv, rows);
    else throw Error(PRISM_ERR_RUNTIME, "resident BiCGSTAB: no kernel for this many rows per thread");
}

}  // namespace

// R rows per thread at most, as few as the blocks allow (one less than the compute units: one
// block sums).  With one row per thread, the rows per block of the three-kernel iteration: the
// sums are then formed in the same order, and the iterates are the same bits.  With more, as
// many blocks as there can be, so that the rows of a block, and with them an iteration's
// work, are fewest.  Where the line lies: with up to seven diagonals, FP64 5 rows per thread
// (652,800 in all) 27.6 us per iteration against 31.9 us of the three kernels at 643,280 rows
// (its 84 spilled registers leave no room for a sixth); FP32 6 rows (783,360 in all) 18.6 us against 32.8 us (row per thread) at
// 665,280, while 7 take 25.8 us against 24.9 us of the packed kernels at 847,872.  Else as many
// as hold their coefficients in registers (keptRows), one with up to 16 entries per row.
template <typename T>
ResidentPlan resident_plan(int64_t n, bool dia, int wmax, int n_cu) {
    ResidentPlan p;
    const int W = wmax <= 5 ? 5 : wmax <= 8 ? (dia && wmax <= 7 ? 7 : 8) : wmax <= 16 && !dia ? 16 : 0;
    const int most = std::min(n_cu - 1, RES_MAX_BLOCKS);
    if (!W || n < 1 || most < 1) return p;
    int spb = 0;
    krylov_grid(n, &spb);
    int64_t rows = (int64_t)spb * 64;
    if (n > (int64_t)most * RES_BS) rows = ((n + most - 1) / most + 63) / 64 * 64;
    const int64_t R = (rows + RES_BS - 1) / RES_BS;
    if (R > mostRows<T>(dia, W)) return p;
    p.blocks = (int)((n + rows - 1) / rows);
    p.rows = (int)rows;
    p.R = (int)R;
    p.W = W;
    return p;
}

template <typename T>
void launch_resident_mark(const Launch& L, T* p, size_t count, unsigned long long* q, size_t more) {
    const size_t most = std::max(count, more);
    PRISM_LAUNCH("resident_mark", k_mark<T>, (int)((most + 255) / 256), 256, p, count, q, more);
}

template <typename T>
void launch_resident(const Launch& L, const KView<T>& kv, const ResidentView<T>& rv, const ResidentPlan& plan) {
    if (kv.ndia) {
        if (plan.W == 5) launchRows<T, true, 5>(L, kv, rv, plan.R);
        else if (plan.W == 7) launchRows<T, true, 7>(L, kv, rv, plan.R);
        else launchRows<T, true, 8>(L, kv, rv, plan.R);
    } else {
        if (plan.W == 5) launchRows<T, false, 5>(L, kv, rv, plan.R);
        else if (plan.W == 8) launchRows<T, false, 8>(L, kv, rv, plan.R);
        else launchRows<T, false, 16>(L, kv, rv, plan.R);
    }
}

template ResidentPlan resident_plan<double>(int64_t, bool, int, int);
template ResidentPlan resident_plan<float>(int64_t, bool, int, int);
template void launch_resident_mark<double>(const Launch&, double*, size_t, unsigned long long*, size_t);
template void launch_resident_mark<float>(const Launch&, float*, size_t, unsigned long long*, size_t);
template void launch_resident<double>(const Launch&, const KView<double>&, const ResidentView<double>&,
                                      const ResidentPlan&);
template void launch_resident<float>(const Launch&, const KView<float>&, const ResidentView<float>&,
                                     const ResidentPlan&);

}  // namespace prism_hip
