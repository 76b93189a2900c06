// isph_resident.hip -- BiCGSTAB iterations of systems that fit on the chip.
//
// An iteration of the launched kernels (isph_solver.hip) is six dependent
// launches, 29 us at 2.5k rows and 32 us at 87k, whatever the work.  Here one
// cooperative launch runs thousands of iterations.  A block owns R = 256 G
// consecutive rows, one per thread.  The row's matrix entries are copied to
// LDS once; the row's vector entries stay in registers.  The rows outside the
// block that its rows refer to are its halo (the same heights of the two
// adjacent cell columns, so about two rows a row): each thread also carries the
// entries of up to M halo rows in registers, so the vector a product gathers
// is complete in LDS.  Own and halo rows in ascending order are the block's
// window; a bitmap of them gives a row's place in it.
//
//   p = r + beta q, v = A p               own and halo p into LDS, product
//     exchange (v, rhat) -> alpha         v of the halo rows is read after it
//   s = r - alpha v, t = A s              own and halo s into LDS, product
//     exchange (t, s), (t, t) -> omega    t of the halo rows is read after it
//   x += alpha p + omega s, r = s - omega t, q = p - omega v   own and halo
//     exchange (r, rhat), (r, r) -> beta, stop tests
//
// A halo row's r, q, p, s are recomputed from its v and t with the owner's
// expressions, so only v and t go through memory, 8 bytes a row each.  The
// exchanges are the only grid-wide synchronisations (isph_gridsync.h).
//
// What bounds it: the chain of three exchanges (2 us each for the words' way to
// the leader and back, about 1 us for the sums on either side), two products
// from LDS (0.5 us each) and the halo reads (0.8 us).  Measured per iteration,
// launched kernels and here: 30 and 12.8 us at 36.6k rows, 32 and 13 us at 87k.
//
// The arithmetic is the launched kernels', term for term: the same row sums,
// the same reduction tree (wave butterfly, four waves of 256 rows, then
// k_finish's tree over the 256-row partials, of which a block of G partials
// does the first log2(G) butterfly levels itself), and finish_update for the
// scalars.
#include <algorithm>
#include <type_traits>

#include "isph_finish.h"
#include "isph_gridsync.h"
#include "isph_host.h"
#include "isph_kernels.h"
#include "isph_spmv.h"

namespace isph {

constexpr int RESIDENT_M = 3;          // halo rows a thread carries
constexpr int RESIDENT_SPAN = 16384;   // rows from a window's first to its last, at most
constexpr int RESIDENT_WORDS = RESIDENT_SPAN / 32;

// entries of a row loaded together (with 1024 threads a thread has 128 registers)
template <int G>
struct ResidentUnroll {
    static constexpr int value = G == 4 ? 6 : 8;
};

// The block's window: a bit per row of [base, base + RESIDENT_SPAN), and the
// rows before each word.
struct Window {
    unsigned int bits[RESIDENT_WORDS];
    int before[RESIDENT_WORDS];
    __device__ __forceinline__ int place(int d) const {  // of row base + d
        return before[d >> 5] + __popc(bits[d >> 5] & ((1u << (d & 31)) - 1u));
    }
};

// One row times the vector in LDS, as spmv_row (unit diagonal at dp) or, for
// FP32 values with FP64 vectors, as spmv_row_diff (FP64 row sum si).  Entries
// k < kl come from LDS (every STRIDE-th element, places in the window), a
// group that reaches past them from the matrix in memory (columns).  Indices
// are clamped to the row's last entry; the sum takes the row's own entries
// only, in order.
template <int U, bool DIFF, int STRIDE, class TV, class TX>
__device__ __forceinline__ TX resident_row(int i, int c, int dp, double si, int kl, int base,
                                           const Window& W, const TV* lv,
                                           const unsigned short* lj, const short* nbr, const TV* val,
                                           size_t ld, TX xi, const TX* win) {
    TX s = (TX)0;
    for (int k = 0; k < c; k += U) {
        TV v[U];
        TX x[U];
        int j[U];
        if (min(k + U, c) <= kl) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int e = min(k + u, c - 1) * STRIDE;
                j[u] = lj[e];
                v[u] = lv[e];
            }
        } else {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const size_t o = (size_t)min(k + u, c - 1) * ld + i;
                j[u] = col_of(nbr[o], i);
                v[u] = val[o];
            }
#pragma unroll
            for (int u = 0; u < U; ++u) j[u] = W.place(j[u] - base);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) x[u] = win[j[u]];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (!DIFF && k + u == dp && k + u < c) s = s + xi;
            const TX t = DIFF ? s + (TX)v[u] * (x[u] - xi) : s + (TX)v[u] * x[u];
            s = k + u < c ? t : s;
        }
    }
    if (DIFF) return (TX)si * xi + s;
    if (dp == c) s = s + xi;
    return s;
}

// A worker's part of an exchange: the block's partials in the launched
// kernels' tree, published by one thread.  STORED: the waves have stored
// vector entries that others read after the exchange; vmcnt counts stores on
// this architecture, so each wave waits for its own before the block's barrier.
template <int G, bool TWO, bool STORED>
__device__ __forceinline__ void publish_sums(const GridSync& gs, double (*wsum)[16], uint32_t e,
                                             int block, double v0, double v1) {
    const int w = threadIdx.x >> 6;
    v0 = wave_sum(v0);
    if (TWO) v1 = wave_sum(v1);
    if (STORED) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if ((threadIdx.x & 63) == 0) {
        wsum[0][w] = v0;
        if (TWO) wsum[1][w] = v1;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double p[2] = {0.0, 0.0};
#pragma unroll
        for (int q = 0; q < (TWO ? 2 : 1); ++q) {
            double b[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int g = 0; g < G; ++g) {
                const double* r = wsum[q] + 4 * g;
                // k_finish adds a thread's partials to 0
                b[g] = 0.0 + ((r[0] + r[1]) + (r[2] + r[3]));
            }
            p[q] = G == 1 ? b[0] : G == 2 ? b[0] + b[1] : (b[0] + b[1]) + (b[2] + b[3]);
        }
        gs_publish(gs, e, block, TWO, p[0], p[1]);
    }
}

// The leader: finishes each exchange's reduction and the solver scalars, and
// broadcasts the scalar that the workers wait for.
template <int G>
__device__ __forceinline__ void resident_leader(const GridSync& gs, double (*red)[16], int* lost,
                                                int nw, SolverScalars* sc, const SolveCtl& ctl,
                                                int maxiter) {
    constexpr int PER = 64 / G;  // workers per wave of k_finish's tree
    if (threadIdx.x >= 256) return;
    const int t = threadIdx.x;
    if (t < 32) red[t >> 4][t & 15] = 0.0;
    if (t == 0) *lost = 0;
    __syncthreads();
    SolverScalars s = *sc;
    auto tree = [](const double* r) {
        double a[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) a[k] = r[2 * k] + r[2 * k + 1];
#pragma unroll
        for (int k = 0; k < 4; ++k) a[k] = a[2 * k] + a[2 * k + 1];
        return (a[0] + a[1]) + (a[2] + a[3]);
    };
    // epoch 1: do all blocks' windows fit?
    uint32_t e = 1;
    {
        double a = 0.0, b = 0.0;
        if (t < nw && !gs_collect<1>(gs, e, t, 0, nw, false, &a, &b)) *lost = 1;
        if (a != 0.0) *lost = 2;
    }
    __syncthreads();
    const int refused = *lost;
    gs_broadcast(gs, e, 0.0, refused);
    if (refused) {
        if (t == 0) refused == 1 ? atomicOr(gs.err, ERR_SYNC) : atomicOr(gs.state, GS_REFUSED);
        return;
    }
    for (int it = 0; it < maxiter; ++it) {
#pragma unroll 1
        for (int kind = FIN_ALPHA; kind <= FIN_BETA; ++kind) {
            ++e;
            const bool two = kind != FIN_ALPHA;
            double a = 0.0, b = 0.0;
            if (t < nw && !gs_collect<1>(gs, e, t, 0, nw, two, &a, &b)) *lost = 1;
            a = lanes_sum<PER>(a);
            b = lanes_sum<PER>(b);
            if (t % PER == 0) {
                red[0][t / PER] = a;
                red[1][t / PER] = b;
            }
            __syncthreads();
            if (*lost) {
                if (t == 0) atomicOr(gs.err, ERR_SYNC);
                return;
            }
            finish_update(kind, tree(red[0]), tree(red[1]), s, ctl);
            gs_broadcast(gs, e, kind == FIN_ALPHA ? s.alpha : kind == FIN_OMEGA ? s.wi : s.betas,
                         s.done);
            __syncthreads();  // red is read before the next exchange writes it
        }
        if (s.done) break;
    }
    if (t == 0) *sc = s;
}

template <class TV, class TX, int G>
__global__ void __launch_bounds__(BLOCK* G) k_bicg_resident(KrylovArgs<TV, TX, short> a, GridSync gs,
                                                             SolverScalars* sc, SolveCtl ctl,
                                                             int first, int maxiter,
                                                             int kl) {
    using P2 = typename Pair2<TX>::type;
    constexpr bool DIFF = std::is_same<TV, float>::value && std::is_same<TX, double>::value;
    constexpr int R = BLOCK * G;
    constexpr int M = RESIDENT_M;
    constexpr int U = ResidentUnroll<G>::value;
    extern __shared__ double dyn[];
    __shared__ double sums[2][16];
    __shared__ Window W;
    __shared__ int jlo, jhi, total;
    const int nw = gridDim.x - 1;
    if ((int)blockIdx.x == nw) {
        resident_leader<G>(gs, sums, &jlo, nw, sc, ctl, maxiter);
        return;
    }
    const int block = xcd_tile(blockIdx.x, nw);
    const int t = threadIdx.x;
    const int i0 = block * R, i1 = min(i0 + R, a.n), i = i0 + t;
    const bool own = i < i1;
    if (t == 0) {
        jlo = i0;
        jhi = i1 - 1;
    }
    for (int w = t; w < RESIDENT_WORDS; w += R) W.bits[w] = 0;
    __syncthreads();
    int c = 0, dp = 0;
    double si = 0.0;
    TX r = (TX)0, q = (TX)0, x = (TX)0, rhat = (TX)0;
    if (own) {
        c = a.cnt[i];
        if (DIFF) si = a.rsum[i];
        else dp = a.dpos[i];
        const P2 u = a.rq[i];
        r = u.x;
        q = u.y;
        x = a.xs[i];
        rhat = a.rhat[i];
        if (c > 0) {  // entries ascend
            atomicMin(&jlo, col_of(a.nbr[i], i));
            atomicMax(&jhi, col_of(a.nbr[(size_t)(c - 1) * a.ld + i], i));
        }
    }
    __syncthreads();
    const int base = jlo;
    const bool spans = jhi - base < RESIDENT_SPAN;
    if (own && spans) {
        atomicOr(&W.bits[(i - base) >> 5], 1u << ((i - base) & 31));
        for (int k = 0; k < c; ++k) {
            const int d = col_of(a.nbr[(size_t)k * a.ld + i], i) - base;
            atomicOr(&W.bits[d >> 5], 1u << (d & 31));
        }
    }
    __syncthreads();
    if (t < 64) {  // one wave scans the words
        constexpr int PER = RESIDENT_WORDS / 64;
        int n = 0;
        for (int w = 0; w < PER; ++w) n += __popc(W.bits[t * PER + w]);
        int s = n;
        for (int o = 1; o < 64; o <<= 1) {
            const int u = __shfl_up(s, o, 64);
            if (t >= o) s += u;
        }
        if (t == 63) total = s;
        s -= n;
        for (int w = 0; w < PER; ++w) {
            W.before[t * PER + w] = s;
            s += __popc(W.bits[t * PER + w]);
        }
    }
    __syncthreads();
    const int nown = i1 - i0;
    const bool fits = spans && total - nown <= M * R;
    uint32_t e = 1;
    double coef = 0.0;
    int done = 0;
    if (t == 0) gs_publish(gs, e, block, false, fits ? 0.0 : 1.0, 0.0);
    if (!gs_receive(gs, e, block, coef, done)) {
        atomicOr(gs.err, ERR_SYNC);
        return;
    }
    if (done) return;  // some block's window does not fit
    const int nh = total - nown, nl = W.place(i0 - base);
    TX* win = reinterpret_cast<TX*>(dyn);
    TV* lv = reinterpret_cast<TV*>(win + (M + 1) * R) + t;
    unsigned short* lj = reinterpret_cast<unsigned short*>(lv - t + (size_t)kl * R) + t;
    if (own)
        for (int k = 0; k < min(c, kl); ++k) {
            lv[k * R] = a.val[(size_t)k * a.ld + i];
            lj[k * R] =
                (unsigned short)W.place(col_of(a.nbr[(size_t)k * a.ld + i], i) - base);
        }
    // halo row h is the window's h-th row that is not the block's own; the
    // list of them passes through the window's memory
    unsigned short* list = reinterpret_cast<unsigned short*>(dyn);
    for (int w = t; w < RESIDENT_WORDS; w += R) {
        int at = W.before[w];
        for (unsigned int b = W.bits[w]; b; b &= b - 1, ++at) {
            const int h = at < nl ? at : at - nown;
            if (at < nl || at >= nl + nown) list[h] = (unsigned short)(w * 32 + __ffs(b) - 1);
        }
    }
    __syncthreads();
    int hj[M], hw[M];  // row and place in the window of this thread's halo rows
#pragma unroll
    for (int m = 0; m < M; ++m) {
        const int h = t + m * R;
        hj[m] = h < nh ? base + list[h] : -1;
        hw[m] = h < nl ? h : h + nown;
    }
    __syncthreads();
    TX hr[M], hq[M], hp[M], hv[M], hs[M];
#pragma unroll
    for (int m = 0; m < M; ++m) {
        hr[m] = hq[m] = hp[m] = hv[m] = hs[m] = (TX)0;
        if (hj[m] >= 0) {
            const P2 u = a.rq[hj[m]];
            hr[m] = u.x;
            hq[m] = u.y;
        }
    }
    TX* vout = a.si;   // the launched kernels' s and t vectors carry v and t
    TX* tout = a.mm2;
    coef = sc->betas;
    bool ok = true;
    for (int it = 0; it < maxiter; ++it) {
        const bool fst = first && it == 0;
        // p = r + beta q, v = A p
        const TX beta = (TX)coef;
        const TX p = fst ? r : r + beta * q;
        if (own) win[nl + t] = p;
#pragma unroll
        for (int m = 0; m < M; ++m)
            if (hj[m] >= 0) {
                hp[m] = fst ? hr[m] : hr[m] + beta * hq[m];
                win[hw[m]] = hp[m];
            }
        __syncthreads();
        TX v = (TX)0;
        if (own) {
            v = resident_row<U, DIFF, R>(i, c, dp, si, kl, base, W, lv, lj, a.nbr, a.val, a.ld, p, win);
            gs_store(vout + i, v);
        }
        publish_sums<G, false, true>(gs, sums, ++e, block, own ? (double)v * (double)rhat : 0.0,
                                     0.0);
        if (!(ok = gs_receive(gs, e, block, coef, done))) break;
        // s = r - alpha v, t = A s
        const TX alpha = (TX)coef;
        const TX sv = r - alpha * v;
        if (own) win[nl + t] = sv;
#pragma unroll
        for (int m = 0; m < M; ++m)
            if (hj[m] >= 0) hv[m] = gs_load(vout + hj[m]);
#pragma unroll
        for (int m = 0; m < M; ++m)
            if (hj[m] >= 0) {
                hs[m] = hr[m] - alpha * hv[m];
                win[hw[m]] = hs[m];
            }
        __syncthreads();
        TX tv = (TX)0;
        if (own) {
            tv = resident_row<U, DIFF, R>(i, c, dp, si, kl, base, W, lv, lj, a.nbr, a.val, a.ld, sv, win);
            gs_store(tout + i, tv);
        }
        publish_sums<G, true, true>(gs, sums, ++e, block, own ? (double)tv * (double)sv : 0.0,
                                    own ? (double)tv * (double)tv : 0.0);
        if (!(ok = gs_receive(gs, e, block, coef, done))) break;
        // x, r, q
        const TX w = (TX)coef;
        TX ht[M];
#pragma unroll
        for (int m = 0; m < M; ++m)
            ht[m] = hj[m] >= 0 ? gs_load(tout + hj[m]) : (TX)0;
        x = (x + alpha * p) + w * sv;
        r = sv - w * tv;
        q = p - w * v;
        publish_sums<G, true, false>(gs, sums, ++e, block, own ? (double)r * (double)rhat : 0.0,
                                     own ? (double)r * (double)r : 0.0);
        if (!(ok = gs_receive(gs, e, block, coef, done))) break;
        if (done) break;
        // the halo rows' t arrived while the block waited
#pragma unroll
        for (int m = 0; m < M; ++m) {
            hr[m] = hs[m] - w * ht[m];
            hq[m] = hp[m] - w * hv[m];
        }
    }
    if (!ok) {  // the solve's state in memory is still the one the launch began with
        atomicOr(gs.err, ERR_SYNC);
        return;
    }
    if (t == 0) atomicOr(gs.state, GS_WRITTEN);
    if (own) {
        a.xs[i] = x;
        P2 u;
        u.x = r;
        u.y = q;
        a.rq[i] = u;
    }
}

namespace host {

template <class TV, class TX, int G>
static int launch(isph_ctx* c, const KrylovArgs<TV, TX, short>& ka, const SolveCtl& ctl, bool& first,
                  int maxiter, bool& ran) {
    auto kern = k_bicg_resident<TV, TX, G>;
    constexpr int R = BLOCK * G;
    const int blocks = (nblk(c->n) + G - 1) / G + 1;
    if (blocks > c->cus) return ISPH_OK;
    // the gathered window, then as many entries of each row as fit
    constexpr size_t win = sizeof(TX) * (RESIDENT_M + 1) * R;
    constexpr size_t per = (sizeof(TV) + sizeof(unsigned short)) * R;
    const int kl = (int)std::min<size_t>((size_t)c->prm.max_nbr, (RESIDENT_LDS - win) / per);
    const size_t lds = win + per * kl;
    KrylovArgs<TV, TX, short> a = ka;
    GridSync gs{c->gs_words, c->err, c->err + 1, GS_MAXB};
    SolverScalars* sc = c->sc;
    SolveCtl t = ctl;
    int f = first, m = maxiter, l = kl;
    void* args[] = {&a, &gs, &sc, &t, &f, &m, &l};
    if (int rc = grid_launch(c, (const void*)kern, blocks, R, args, lds, GS_MAXB, ran)) return rc;
    if (ran) first = false;
    return ISPH_OK;
}

// Rows per block, 256 G: as few as let the grid hold the system with one
// worker per CU and a CU for the leader: G = 1 up to 65,280 rows, 2 up to
// 130,560, 4 up to 261,120.
template <class TV, class TX>
int resident_iterate(isph_ctx* c, const KrylovArgs<TV, TX, short>& a, const SolveCtl& ctl,
                     bool& first, int maxiter, bool& ran) {
    ran = false;
    if (!c->cooperative || c->n == 0) return ISPH_OK;
    const int nb = nblk(c->n), most = GS_MAXB - 1;
    if (nb <= most) return launch<TV, TX, 1>(c, a, ctl, first, maxiter, ran);
    if (nb <= 2 * most) return launch<TV, TX, 2>(c, a, ctl, first, maxiter, ran);
    if (nb <= 4 * most) return launch<TV, TX, 4>(c, a, ctl, first, maxiter, ran);
    return streamed_iterate<TV, TX>(c, a, ctl, first, maxiter, ran);
}

#define ISPH_RESIDENT(TV, TX)                                                                  \
    template int resident_iterate<TV, TX>(isph_ctx*, const KrylovArgs<TV, TX, short>&,         \
                                          const SolveCtl&, bool&, int, bool&);
ISPH_RESIDENT(double, double)
ISPH_RESIDENT(float, double)
ISPH_RESIDENT(float, float)

}  // namespace host
}  // namespace isph
