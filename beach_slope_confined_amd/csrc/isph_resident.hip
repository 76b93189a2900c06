// isph_resident.hip -- BiCGSTAB iterations of systems that fit on the chip.
//
// An iteration of the launched kernels (isph_solver.hip) is six dependent
// launches, 24 us at 2.5k rows and 27 us at 87k, whatever the work.  Here one
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
//     exchange (v, rhat) -> alpha         v of the halo rows is read with it
//   s = r - alpha v, t = A s              own and halo s into LDS, product
//     exchange (t, s), (t, t) -> omega    t of the halo rows is read after it
//   x += alpha p + omega s, r = s - omega t, q = p - omega v   own and halo
//     exchange (r, rhat), (r, r) -> beta, stop tests
//
// A halo row's r, q, p, s are recomputed from its v and t with the owner's
// expressions, so only v and t go through memory, 8 bytes a row each.  The
// exchanges are the only grid-wide synchronisations (isph_gridsync.h).
//
// The first entries of a row's matrix are in registers, the next in LDS, and
// only where a thread has 128 registers (blocks of 1024 rows) a few stay in
// memory.
//
// What bounds it: the chain of three exchanges (1.3 us each without a leader,
// 2.3 with one: the words' way, the sums on either side), then two products
// (0.5 us), and with a leader the halo reads (0.4 us) and the wait for the
// stores.  Measured per iteration of the solve, launched kernels and here: 24.6
// and 6.1 us at 2.5k rows, 23.4 and 7.7 us at 36.6k, 27 and 9.7 us at 87k, 40
// and 19 us at 255k.  Values and places in LDS instead of registers, with the diagonal
// tested at every entry, made a product 1.3 us.
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

// entries of a row kept in registers (a thread has 512, 256 or 128 of them with
// blocks of 256, 512 or 1024)
template <int G>
struct ResidentRegs {
    static constexpr int value = G == 4 ? 8 : 24;
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

// A row's entries in column order, as spmv_row takes them: the unit diagonal
// is an entry of its own, 1 at position dp (1 x is x, so the sum is the same),
// and for FP32 values with FP64 vectors (spmv_row_diff) there is none.  The
// first NREG are in registers, the next kl in LDS (every STRIDE-th element),
// the rest in memory.  Rows are padded with 0 times their own x: a sum that
// starts from +0 is never -0, so adding 0 changes nothing.
template <bool DIFF, int NREG, int STRIDE, class TV, class TX>
struct ResidentRow {
    int i, c, dp, len, own;    // row, list entries, diagonal, entries, own byte offset in the window
    int wlen;                  // longest row of the wave
    double si;
    TV v[NREG];
    unsigned int off[NREG / 2];  // byte offsets in the window, two a word
    const TV* lv;
    const unsigned short* lo;

    // entry e of the list with the diagonal: its place in the matrix, or -1
    __device__ __forceinline__ int source(int e) const {
        return DIFF ? e : e < dp ? e : e == dp ? -1 : e - 1;
    }
    __device__ __forceinline__ void load(const KrylovArgs<TV, TX, short>& a, const Window& W,
                                         int base, int kl, TV* lvw, unsigned short* low) {
        auto entry = [&](int e, TV& val, unsigned int& o) {
            val = (TV)0;
            o = own;
            if (e < len) {
                const int k = source(e);
                if (k < 0) {
                    val = (TV)1;
                } else {
                    val = a.val[(size_t)k * a.ld + i];
                    o = W.place(i + (int)a.nbr[(size_t)k * a.ld + i] - base) * (int)sizeof(TX);
                }
            }
        };
#pragma unroll
        for (int e = 0; e < NREG; e += 2) {
            unsigned int o0, o1;
            entry(e, v[e], o0);
            entry(e + 1, v[e + 1], o1);
            off[e / 2] = o0 | o1 << 16;
        }
        for (int e = 0; e < kl && NREG + e < ((len + 3) & ~3); ++e) {
            TV val;
            unsigned int o;
            entry(NREG + e, val, o);
            lvw[e * STRIDE] = val;
            low[e * STRIDE] = (unsigned short)o;
        }
        lv = lvw;
        lo = low;
        int m = len;
        for (int s = 1; s < 64; s <<= 1) m = max(m, __shfl_xor(m, s, 64));
        wlen = __builtin_amdgcn_readfirstlane(m);
    }
    __device__ __forceinline__ TX times(const KrylovArgs<TV, TX, short>& a, const Window& W,
                                        int base, int kl, const TX* win, TX xi) const {
        const char* w = reinterpret_cast<const char*>(win);
        auto at = [&](unsigned int o) { return *reinterpret_cast<const TX*>(w + o); };
        auto add = [&](TX s, TV val, TX x) {
            return DIFF ? s + (TX)val * (x - xi) : s + (TX)val * x;
        };
        TX s = (TX)0;
#pragma unroll
        for (int e = 0; e < NREG; e += 8) {
            if (e >= wlen) break;  // the same in the whole wave
            TX x[8];
#pragma unroll
            for (int u = 0; u < 8; u += 2) {
                x[u] = at(off[(e + u) / 2] & 0xffff);
                x[u + 1] = at(off[(e + u) / 2] >> 16);
            }
#pragma unroll
            for (int u = 0; u < 8; ++u) s = add(s, v[e + u], x[u]);
        }
        if (wlen > NREG) {
            const int in_lds = min(len - NREG, kl);
            for (int e = 0; e < in_lds; e += 4) {
                TV val[4];
                TX x[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    val[u] = lv[(e + u) * STRIDE];
                    x[u] = at(lo[(e + u) * STRIDE]);
                }
#pragma unroll
                for (int u = 0; u < 4; ++u) s = add(s, val[u], x[u]);
            }
            for (int e = NREG + kl; e < len; e += 4) {
                TV val[4];
                TX x[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int k = source(min(e + u, len - 1));
                    const size_t o = (size_t)max(k, 0) * a.ld + i;
                    val[u] = k < 0 ? (TV)1 : a.val[o];
                    x[u] = k < 0 ? xi : win[W.place(i + (int)a.nbr[o] - base)];
                }
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const TX t = add(s, val[u], x[u]);
                    s = e + u < len ? t : s;
                }
            }
        }
        return DIFF ? (TX)si * xi + s : s;
    }
};

// Without a leader, vector entries that other blocks read are 64-bit words of
// 32 bits of data under the epoch, like the exchanges' (an FP64 value takes
// two), so that neither the writer waits for its stores before it publishes its
// part of the sum, nor the reader for the sum before it asks for them.  A word
// is written again three epochs later, when its writer has seen every block's
// part of an epoch that the block published after it had read the word.
// Cleared before each launch.  8.2 against 9.2 us an iteration at 17.7k rows in
// blocks of 256; with a leader (the workers' polls of its words and of these
// then compete) it is no faster at 59k and 86k rows, and blocks of 1024 rows
// lack the registers (24.6 against 19.4 us at 255k), so there they are plain.
struct HaloWords {
    gs_word *vh, *vl, *th, *tl;  // high and low words of v and t
};
// 32-bit byte offsets: one register an address
__device__ __forceinline__ gs_word* word_at(gs_word* w, int j) {
    return reinterpret_cast<gs_word*>(reinterpret_cast<char*>(w) + (unsigned int)j * 8u);
}
__device__ __forceinline__ void store_words(gs_word* h, gs_word* l, int i, uint32_t e, double v) {
    gs_store(word_at(h, i), gs_hi(e, v));
    gs_store(word_at(l, i), gs_lo(e, v));
}
__device__ __forceinline__ void store_words(gs_word* h, gs_word*, int i, uint32_t e, float v) {
    gs_store(word_at(h, i), (gs_word)e << 32 | __float_as_uint(v));
}
template <class TX>
struct HaloRead {
    static constexpr bool WIDE = sizeof(TX) == 8;
    gs_word *h, *l;
    const int* row;  // M of them, -1 for none
    uint32_t e;
    gs_word x[RESIDENT_M], y[RESIDENT_M];
    __device__ __forceinline__ void request() {
#pragma unroll
        for (int m = 0; m < RESIDENT_M; ++m) {
            x[m] = y[m] = (gs_word)e << 32;
            if (row[m] >= 0) {
                x[m] = gs_load(word_at(h, row[m]));
                if (WIDE) y[m] = gs_load(word_at(l, row[m]));
            }
        }
    }
    __device__ __forceinline__ bool valid() const {
        bool ok = true;
#pragma unroll
        for (int m = 0; m < RESIDENT_M; ++m)
            ok = ok && (uint32_t)(x[m] >> 32) == e && (!WIDE || (uint32_t)(y[m] >> 32) == e);
        return ok;
    }
    __device__ __forceinline__ TX value(int m) const {
        if constexpr (WIDE) return gs_value(x[m], y[m]);
        else return __uint_as_float((unsigned int)x[m]);
    }
    // a wave that waits for nothing else
    __device__ __forceinline__ bool wait() {
        for (int spin = 0; spin < GS_SPIN; ++spin) {
            request();
            if (__all(valid())) return true;
        }
        return false;
    }
};

__global__ void k_halo_clear(int n, HaloWords w, bool wide) {
    const int i = blockIdx.x * BLOCK + threadIdx.x;
    if (i >= n) return;
    w.vh[i] = 0ull;
    w.th[i] = 0ull;
    if (wide) {
        w.vl[i] = 0ull;
        w.tl[i] = 0ull;
    }
}

// A worker's part of an exchange: the block's partials in the launched
// kernels' tree, published by one thread.  STORED: the waves have stored plain
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

// k_finish's sum of the parts of an exchange in one wave.  Lane l takes the
// parts l + 64 m.  64 / G parts are a wave of k_finish's tree, so the sum over
// the lanes of one m covers G of its waves, in its order: the butterfly's last
// log2(G) steps are the first levels of the tree over the waves.
template <int NP>
struct PartSums {
    double a[NP], b[NP];
    template <class More>
    __device__ __forceinline__ bool collect(const GridSync& gs, uint32_t e, int nw, bool two,
                                            More& more) {
        const int lane = threadIdx.x & 63;
        return __all(gs_collect<NP>(gs, e, lane, 64, nw, two, a, b, more));
    }
    static __device__ __forceinline__ double total(const double* p) {
        double q[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int m = 0; m < NP; ++m) q[m] = lanes_sum<64>(p[m]);
        return ((q[0] + q[1]) + (q[2] + q[3])) + 0.0;  // k_finish's remaining waves are 0
    }
};

// The leader, one wave: finishes each exchange's reduction and the solver
// scalars, and broadcasts the scalar that the workers wait for.
__device__ __forceinline__ void resident_leader(const GridSync& gs, int nw, SolverScalars* sc,
                                                const SolveCtl& ctl, int maxiter) {
    const int t = threadIdx.x;
    if (t >= 64) return;
    SolverScalars s = *sc;
    PartSums<GS_MAXB / 64> sum;
    auto collect = [&](uint32_t e, bool two) {
        GsNone none;
        const bool ok = sum.collect(gs, e, nw, two, none);
        if (!ok && t == 0) atomicOr(gs.err, ERR_SYNC);
        return ok;
    };
    // epoch 1: do all blocks' windows fit?
    uint32_t e = 1;
    if (!collect(e, false)) return;
    const int refused = sum.total(sum.a) != 0.0;
    gs_broadcast(gs, e, 0.0, refused);
    if (refused) {
        if (t == 0) atomicOr(gs.state, GS_REFUSED);
        return;
    }
    for (int it = 0; it < maxiter; ++it) {
        if (!collect(++e, false)) return;
        finish_update(FIN_ALPHA, sum.total(sum.a), 0.0, s, ctl);
        gs_broadcast(gs, e, s.alpha, 0);
        if (!collect(++e, true)) return;
        finish_update(FIN_OMEGA, sum.total(sum.a), sum.total(sum.b), s, ctl);
        gs_broadcast(gs, e, s.wi, 0);
        if (!collect(++e, true)) return;
        finish_update(FIN_BETA, sum.total(sum.a), sum.total(sum.b), s, ctl);
        gs_broadcast(gs, e, s.betas, s.done);
        if (s.done) break;
    }
    if (t == 0) {
        // ahead of the vectors, should the workers lose the last broadcast
        atomicOr(gs.state, GS_WRITTEN);
        *sc = s;
    }
}

// NP > 0: no leader; one wave of every block sums all parts, up to 64 NP, and
// forms the scalars.  The words travel once instead of to the leader and back;
// what grows with the grid is the reading of all parts by all blocks.  (Four
// waves a block that read a quarter each, or all, are slower at any size.)
template <class TV, class TX, int G, int NP>
__global__ void __launch_bounds__(BLOCK* G) k_bicg_resident(KrylovArgs<TV, TX, short> a, GridSync gs,
                                                             SolverScalars* sc, SolveCtl ctl,
                                                             HaloWords words, int first,
                                                             int maxiter, int kl) {
    using P2 = typename Pair2<TX>::type;
    constexpr bool DIFF = std::is_same<TV, float>::value && std::is_same<TX, double>::value;
    constexpr int R = BLOCK * G;
    constexpr int M = RESIDENT_M;
    constexpr int NREG = ResidentRegs<G>::value;
    extern __shared__ double dyn[];
    __shared__ double sums[2][16];
    __shared__ Window W;
    __shared__ int jlo, jhi, total;
    const int nw = NP ? gridDim.x : gridDim.x - 1;
    if (!NP && (int)blockIdx.x == nw) {
        resident_leader(gs, nw, sc, ctl, maxiter);
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
    __shared__ double answer[2];  // NP: the awaited scalar; the stop flag, or -1
    SolverScalars s;
    if (NP) s = *sc;
    auto exchanged = [&](int kind, auto& more) {
        if (!NP) return gs_receive(gs, e, block, coef, done);
        bool ok;
        if (t < 64) {
            PartSums<NP ? NP : 1> sum;
            const bool two = kind == FIN_OMEGA || kind == FIN_BETA;
            ok = sum.collect(gs, e, nw, two, more);
            const double t0 = sum.total(sum.a);
            if (kind < 0) {
                done = t0 != 0.0;
            } else {
                finish_update(kind, t0, two ? sum.total(sum.b) : 0.0, s, ctl);
                coef = kind == FIN_ALPHA ? s.alpha : kind == FIN_OMEGA ? s.wi : s.betas;
                done = kind == FIN_BETA ? s.done : 0;
            }
            if (t == 0) {
                answer[0] = coef;
                answer[1] = ok ? (double)done : -1.0;
            }
        } else {
            ok = more.wait();
        }
        __syncthreads();  // the next exchange's, in publish_sums, orders the reads
        coef = answer[0];
        done = (int)answer[1];
        return ok && done >= 0;
    };
    GsNone none;
    if (t == 0) gs_publish(gs, e, block, false, fits ? 0.0 : 1.0, 0.0);
    if (!exchanged(-1, none)) {
        atomicOr(gs.err, ERR_SYNC);
        return;
    }
    if (done) {  // some block's window does not fit
        if (NP && block == 0 && t == 0) atomicOr(gs.state, GS_REFUSED);
        return;
    }
    const int nh = total - nown, nl = W.place(i0 - base);
    TX* win = reinterpret_cast<TX*>(dyn);
    TV* lv = reinterpret_cast<TV*>(win + (M + 1) * R) + t;
    unsigned short* lj = reinterpret_cast<unsigned short*>(lv - t + (size_t)kl * R) + t;
    ResidentRow<DIFF, NREG, R, TV, TX> row;
    row.i = i;
    row.c = c;
    row.dp = dp;
    row.len = own ? c + (DIFF ? 0 : 1) : 0;
    row.own = (nl + t) * (int)sizeof(TX);
    row.si = si;
    row.load(a, W, base, kl, lv, lj);
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
    // 32-bit byte offsets: one register an address
    auto at = [](TX* v, int j) {
        return reinterpret_cast<TX*>(reinterpret_cast<char*>(v) + (unsigned int)j * (unsigned int)sizeof(TX));
    };
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
            v = row.times(a, W, base, kl, win, p);
            if (NP) store_words(words.vh, words.vl, i, e + 1, v);
            else gs_store(at(vout, i), v);
        }
        publish_sums<G, false, !NP>(gs, sums, ++e, block, own ? (double)v * (double)rhat : 0.0, 0.0);
        HaloRead<TX> rv{words.vh, words.vl, hj, e};
        if (!(ok = exchanged(FIN_ALPHA, rv))) break;
        // s = r - alpha v, t = A s
        const TX alpha = (TX)coef;
        const TX sv = r - alpha * v;
        if (own) win[nl + t] = sv;
#pragma unroll
        for (int m = 0; m < M; ++m)
            if (hj[m] >= 0) hv[m] = NP ? rv.value(m) : gs_load(at(vout, hj[m]));
#pragma unroll
        for (int m = 0; m < M; ++m)
            if (hj[m] >= 0) {
                hs[m] = hr[m] - alpha * hv[m];
                win[hw[m]] = hs[m];
            }
        __syncthreads();
        TX tv = (TX)0;
        if (own) {
            tv = row.times(a, W, base, kl, win, sv);
            if (NP) store_words(words.th, words.tl, i, e + 1, tv);
            else gs_store(at(tout, i), tv);
        }
        publish_sums<G, true, !NP>(gs, sums, ++e, block, own ? (double)tv * (double)sv : 0.0,
                                   own ? (double)tv * (double)tv : 0.0);
        HaloRead<TX> rt{words.th, words.tl, hj, e};
        if (!(ok = exchanged(FIN_OMEGA, none))) break;
        // x, r, q
        const TX w = (TX)coef;
        TX ht[M];
#pragma unroll
        for (int m = 0; m < M; ++m)
            ht[m] = !NP && hj[m] >= 0 ? gs_load(at(tout, hj[m])) : (TX)0;
        x = (x + alpha * p) + w * sv;
        r = sv - w * tv;
        q = p - w * v;
        publish_sums<G, true, false>(gs, sums, ++e, block, own ? (double)r * (double)rhat : 0.0,
                                     own ? (double)r * (double)r : 0.0);
        if (!(ok = exchanged(FIN_BETA, rt))) break;
        if (done) break;
        // the halo rows' t arrived while the block waited
#pragma unroll
        for (int m = 0; m < M; ++m) {
            hr[m] = hs[m] - w * (NP ? rt.value(m) : ht[m]);
            hq[m] = hp[m] - w * hv[m];
        }
    }
    if (!ok) {  // the solve's state in memory is still the one the launch began with
        atomicOr(gs.err, ERR_SYNC);
        return;
    }
    if (t == 0) atomicOr(gs.state, GS_WRITTEN);
    if (NP && block == 0 && t == 0) *sc = s;
    if (own) {
        a.xs[i] = x;
        P2 u;
        u.x = r;
        u.y = q;
        a.rq[i] = u;
    }
}

namespace host {

template <class TV, class TX, int G, int NP>
static int launch(isph_ctx* c, const KrylovArgs<TV, TX, short>& ka, const SolveCtl& ctl, bool& first,
                  int maxiter, bool& ran) {
    auto kern = k_bicg_resident<TV, TX, G, NP>;
    constexpr int R = BLOCK * G;
    const int blocks = (nblk(c->n) + G - 1) / G + (NP ? 0 : 1);
    if (blocks > c->cus) return ISPH_OK;
    // the gathered window, then as many of each row's further entries as fit
    constexpr size_t win = sizeof(TX) * (RESIDENT_M + 1) * R;
    constexpr size_t per = (sizeof(TV) + sizeof(unsigned short)) * R;
    const size_t most = (size_t)std::max(c->prm.max_nbr + 4 - ResidentRegs<G>::value, 0);
    const int kl = (int)std::min(most, (RESIDENT_LDS - win) / per) & ~3;  // taken in fours
    const size_t lds = win + per * kl;
    KrylovArgs<TV, TX, short> a = ka;
    GridSync gs{c->gs_words, c->err, c->err + 1, GS_MAXB};
    SolverScalars* sc = c->sc;
    SolveCtl t = ctl;
    // vectors that the launched kernels write before they read
    auto words = [](void* p) { return static_cast<gs_word*>(p); };
    HaloWords h{words(c->rv64), words(c->rv64) + c->cap, words(c->v64[2]), words(c->v64[3])};
    if (NP) k_halo_clear<<<nblk(c->n), BLOCK, 0, c->stream>>>(c->n, h, sizeof(TX) == 8);
    int f = first, m = maxiter, l = kl;
    void* args[] = {&a, &gs, &sc, &t, &h, &f, &m, &l};
    if (int rc = grid_launch(c, (const void*)kern, blocks, R, args, lds, GS_MAXB, ran)) return rc;
    if (ran) {
        first = false;
        c->forms[ISPH_FORM_RESIDENT] += 1;
    }
    return ISPH_OK;
}

// Rows per block, 256 G, and whether a leader serves the exchanges.  Up to 192
// blocks do without (NP parts a lane): the words' round trip saved is more than
// every block's reading of every part, and so fewer, larger blocks are better
// from 64 on.  A whole step over its iterations (0 to 0.8 us above the solve
// alone) with blocks of 256 and of 512 rows: 6.9 and 6.95 us an iteration at
// 11k rows, 7.8 / 7.0 at 17.7k, 9.1 / 7.9 at 36.6k, 9.7 / 8.1 at 47k; with and
// without a leader 11.6 / 8.2 at 59k, 10.8 / 9.4 at 72.5k, 10.9 / 9.7 at 86k,
// but 11.5 / 13.4 at 103k.  Beyond 98k rows a leader, and beyond 130,560 blocks
// of 1024 rows, as few as let the grid hold the system with one worker per CU
// and a CU for the leader, up to 261,120.
template <class TV, class TX>
int resident_iterate(isph_ctx* c, const KrylovArgs<TV, TX, short>& a, const SolveCtl& ctl,
                     bool& first, int maxiter, bool& ran) {
    ran = false;
    if (!c->cooperative || c->n == 0) return ISPH_OK;
    if (c->hold > 0) {
        c->hold -= 1;
        return ISPH_OK;
    }
    const int nb = nblk(c->n), most = GS_MAXB - 1;
    if (nb <= 64) return launch<TV, TX, 1, 1>(c, a, ctl, first, maxiter, ran);
    if (nb <= 128) return launch<TV, TX, 2, 1>(c, a, ctl, first, maxiter, ran);
    if (nb <= 256) return launch<TV, TX, 2, 2>(c, a, ctl, first, maxiter, ran);
    if (nb <= 384) return launch<TV, TX, 2, 3>(c, a, ctl, first, maxiter, ran);
    if (nb <= 2 * most) return launch<TV, TX, 2, 0>(c, a, ctl, first, maxiter, ran);
    if (nb <= 4 * most) return launch<TV, TX, 4, 0>(c, a, ctl, first, maxiter, ran);
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
