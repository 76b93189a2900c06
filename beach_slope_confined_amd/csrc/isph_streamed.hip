// isph_streamed.hip -- BiCGSTAB iterations in one cooperative launch with the
// matrix read from memory: the systems that isph_resident.hip cannot hold.
//
// A block owns consecutive 256-row blocks, n / 256 rows in all, up to 7 a
// thread of 768.  Its window, the rows from the first to the last that its
// rows refer to (they lie in the adjacent cell columns), is complete in LDS
// for each product.  The window's rows outside the block, its halo, are kept
// up to date from their v and t with the owner's expressions, so v and t are
// all that goes through memory, 8 bytes a row each, stored while the product
// that makes them runs:
//
//   p = r + beta q, v = A p         exchange (v, rhat) -> alpha
//   s = r - alpha v, t = A s        exchange (t, s), (t, t) -> omega
//   x += alpha p + omega s, r = s - omega t, q = p - omega v
//                                   exchange (r, rhat), (r, r) -> beta, stop
//
// The gathers of the launched kernels (20 pairs of 16 bytes a row through L1
// and L2) become LDS reads, their six launches three exchanges, and their 150
// bytes of vectors a row and iteration about 50.  What is left is the matrix,
// twice: the second product walks the rows backwards, so each product starts
// on the rows that the other read last, which the L2s and the Infinity Cache
// still hold.  A persistent grid that only reads the 210 MB of a 1M-row matrix
// back and forth does so at 8.2 TB/s, 26 us a pass (6.9 TB/s always forwards).
//
// Measured per iteration of the solve, launched kernels and here, FP64: 50 and
// 37 us at 365k rows, 75 and 54 us at 647k, 116 and 83 us at 1.06M; FP32 values
// with FP64 vectors: 46 and 29, 64 and 40, 87 and 59 us.  Of the 83 us the two
// products take 58 (7.9 TB/s counting the ragged ends of the rows), the
// exchanges 15.  Below 261k rows the resident form is faster (9.8 against 19.8
// us at 93k, 19 against 28 us at 255k).
//
// Exchange in two hops: each block publishes its 256-row partials; sixteen
// waves (one in each of the first sixteen blocks) sum 64 of k_finish's threads
// each and publish that; every block reads the sixteen and finishes the sum
// and the scalars itself.  One block collecting all 4,133 parts of a 1M-row
// sum took 6 to 10 us.
//
// The arithmetic is the launched kernels', term for term.
#include <algorithm>
#include <type_traits>

#include "isph_finish.h"
#include "isph_gridsync.h"
#include "isph_host.h"
#include "isph_kernels.h"
#include "isph_spmv.h"

namespace isph {

constexpr int ST_THREADS = 768;  // 168 registers a thread
constexpr int ST_WAVES = ST_THREADS / 64;
constexpr int ST_GROUPS = FIN_BLOCK / 64;  // waves of k_finish
constexpr int ST_COPIES = 16;              // of the sixteen sums: lanes of a wave over 4 words
constexpr int ST_U = 8;                    // entries of a row loaded together
constexpr int ST_H = 8;                    // halo rows a thread loads together
constexpr int ST_MAXJ = 7;                 // rows of a thread, at most
constexpr int ST_MAXP = 5;                 // parts of a k_finish thread, at most
static_assert(ST_MAXP * FIN_BLOCK + ST_COPIES * ST_GROUPS <= GS_PARTS, "words of the parts");
static_assert(ST_GROUPS == 16 && ST_MAXP < ST_WAVES, "groups are a row of lanes; collecting waves");

// One row times the window, as spmv_row or spmv_row_diff; `li` is the row's
// own place, so an entry's is li + its offset.  Entry k of row i lies at byte
// offset ov + k * ldv of the values and ov / sizeof(TV) * 2 of the offsets
// (32 bits, checked on the host): one register an address.
template <bool DIFF, class TV, class TX>
__device__ __forceinline__ TX streamed_row(unsigned int i, unsigned int ld, int li, int c, int dp,
                                           double si, const short* nbr, const TV* val,
                                           const TX* win) {
    constexpr int U = ST_U;
    const TX xi = win[li];
    TX s = (TX)0;
    for (int k = 0; k < c; k += U) {
        TV v[U];
        int j[U];
        TX x[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const unsigned int o = (unsigned int)min(k + u, c - 1) * ld + i;
            j[u] = *reinterpret_cast<const short*>(reinterpret_cast<const char*>(nbr) + 2u * o);
            v[u] = *reinterpret_cast<const TV*>(reinterpret_cast<const char*>(val) +
                                                (unsigned int)sizeof(TV) * o);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) x[u] = win[li + j[u]];
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

struct StreamedShared {
    double part[2][ST_MAXP][64];         // a group's parts
    int arrived;                         // waves that have stored theirs, over all epochs
    double wsum[2][ST_MAXJ * ST_WAVES];  // sums of 64 rows
    SolverScalars s;
    double coef;
    int done, lost, jlo, jhi;
};

// the sixteen wave sums of epoch e: copy, then word of a sum, then group
__device__ __forceinline__ gs_word* st_sums(const GridSync& g, uint32_t e, int copy) {
    return g.words + 2 * GS_LINES * GS_LINE + 2 * 4 * (size_t)g.parts +
           ((size_t)(e & 1) * ST_COPIES + copy) * 4 * ST_GROUPS;
}

// One exchange, by all threads of the block.  wsum holds the block's sums of
// 64 rows; kind is the scalar to finish (0: epoch 1, the go-ahead).  False
// when a wait was in vain.  `between` runs while the parts travel.
template <class F>
__device__ __forceinline__ bool st_exchange(const GridSync& gs, StreamedShared& sh, uint32_t e,
                                            int kind, int block, int b0, int b1, int np,
                                            const SolveCtl& ctl, double& coef, int& done,
                                            F&& between) {
    const int t = threadIdx.x, lane = t & 63;
    const bool two = kind == FIN_OMEGA || kind == FIN_BETA;
    const int np_t = (np + FIN_BLOCK - 1) / FIN_BLOCK;  // parts of a k_finish thread
    __syncthreads();
    if (t < b1 - b0) {
        const double* w0 = sh.wsum[0] + 4 * t;
        const double* w1 = sh.wsum[1] + 4 * t;
        gs_publish(gs, e, b0 + t, two, (w0[0] + w0[1]) + (w0[2] + w0[3]),
                   two ? (w1[0] + w1[1]) + (w1[2] + w1[3]) : 0.0);
    }
    // the first blocks collect group `block`: wave 1 + m the m-th parts of
    // k_finish's threads, then wave 1 their sums
    if (block < ST_GROUPS && t >= 64 && t < 64 * (1 + np_t)) {
        const int m = (t >> 6) - 1, part = block * 64 + lane + m * FIN_BLOCK;
        double x = 0.0, y = 0.0;
        if (part < np && !gs_collect<1>(gs, e, part, 0, np, two, &x, &y)) sh.lost = 1;
        if (m > 0) {
            sh.part[0][m][lane] = x;
            sh.part[1][m][lane] = y;
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
            if (lane == 0) atomicAdd(&sh.arrived, 1);
        } else {
            bool ok = false;
            for (int spin = 0; spin < GS_SPIN && !ok; ++spin)
                ok = __hip_atomic_load(&sh.arrived, __ATOMIC_ACQUIRE,
                                       __HIP_MEMORY_SCOPE_WORKGROUP) >= (int)e * (np_t - 1);
            if (!ok) sh.lost = 1;
            double s0 = 0.0, s1 = 0.0;
            if (part < np) {
                s0 = s0 + x;
                s1 = s1 + y;
            }
            for (int k = 1; k < np_t; ++k)
                if (part + k * FIN_BLOCK < np) {
                    s0 = s0 + sh.part[0][k][lane];
                    s1 = s1 + sh.part[1][k][lane];
                }
            s0 = lanes_sum<64>(s0);
            s1 = lanes_sum<64>(s1);
            const int q = lane & 3;
            const gs_word w = q == 0   ? gs_hi(e, s0)
                              : q == 1 ? gs_lo(e, s0)
                              : q == 2 ? gs_hi(e, s1)
                                       : gs_lo(e, s1);
            gs_store(st_sums(gs, e, lane >> 2) + q * ST_GROUPS + block, w);
        }
    }
    between();
    // wave 0 finishes the sum: lane = word * 16 + group
    if (t < 64) {
        const gs_word* w = st_sums(gs, e, block & (ST_COPIES - 1)) + lane;
        gs_word x = 0;
        bool ok = false;
        for (int spin = 0; spin < GS_SPIN && !ok; ++spin) {
            x = gs_load(w);
            ok = __all((uint32_t)(x >> 32) == e);
        }
        // pairwise tree over the groups: lanes that differ in bits 0 to 3
        const gs_word lo = __shfl(x, (lane & 32) + 16 + (lane & 15), 64);
        const gs_word hi = __shfl(x, (lane & 32) + (lane & 15), 64);
        const double sum = lanes_sum<16>(gs_value(hi, lo));
        const double t0 = __shfl(sum, 0, 64), t1 = __shfl(sum, 32, 64);
        if (!ok) {
            sh.lost = 1;
        } else if (kind == 0) {
            if (t == 0) sh.done = t0 != 0.0;
        } else {
            SolverScalars s = sh.s;
            finish_update(kind, t0, two ? t1 : 0.0, s, ctl);
            if (t == 0) {
                sh.s = s;
                sh.coef = kind == FIN_ALPHA ? s.alpha : kind == FIN_OMEGA ? s.wi : s.betas;
                sh.done = s.done;
            }
        }
    }
    __syncthreads();
    coef = sh.coef;
    done = sh.done;
    return sh.lost == 0;
}

template <class TV, class TX, int J>
__global__ void __launch_bounds__(ST_THREADS) k_bicg_streamed(KrylovArgs<TV, TX, short> a,
                                                               GridSync gs, SolverScalars* sc,
                                                               SolveCtl ctl, int first,
                                                               int maxiter, int lds) {
    using P2 = typename Pair2<TX>::type;
    constexpr bool DIFF = std::is_same<TV, float>::value && std::is_same<TX, double>::value;
    extern __shared__ double dyn[];
    __shared__ StreamedShared sh;
    const int np = (a.n + BLOCK - 1) / BLOCK;
    const int block = xcd_tile(blockIdx.x, gridDim.x);
    const int t = threadIdx.x, wave = t >> 6;
    // 256-row blocks [b0, b1) and rows [i0, i1) of this block
    const int per = np / (int)gridDim.x, more = np % (int)gridDim.x;
    const int b0 = block * per + min(block, more), b1 = b0 + per + (block < more ? 1 : 0);
    const int i0 = b0 * BLOCK, i1 = min(b1 * BLOCK, a.n), nown = i1 - i0;
    const unsigned int ld = (unsigned int)a.ld;
    if (t == 0) {
        sh.s = *sc;
        sh.lost = 0;
        sh.arrived = 0;
        sh.jlo = i0;
        sh.jhi = i1 - 1;
    }
    for (int w = t; w < ST_MAXJ * ST_WAVES; w += ST_THREADS) sh.wsum[0][w] = sh.wsum[1][w] = 0.0;
    __syncthreads();
    // row u of this thread is i0 + u ST_THREADS + t: its entry count and
    // diagonal position (0 entries past the last row), and r, q, v; t takes
    // r's place after s has gone to the window, p takes q's
    int cd[J];
    TX r[J], q[J], v[J];
    {
        int lo = i0, hi = i1 - 1;
#pragma unroll
        for (int u = 0; u < J; ++u) {
            const int i = i0 + u * ST_THREADS + t;
            cd[u] = 0;
            r[u] = q[u] = v[u] = (TX)0;
            if (i < i1) {
                const int c = a.cnt[i];
                cd[u] = c | (DIFF ? 0 : a.dpos[i] << 16);
                const P2 w = a.rq[i];
                r[u] = w.x;
                q[u] = w.y;
                if (c > 0) {  // entries ascend
                    lo = min(lo, i + (int)a.nbr[i]);
                    hi = max(hi, i + (int)a.nbr[(size_t)(c - 1) * a.ld + i]);
                }
            }
        }
        atomicMin(&sh.jlo, lo);
        atomicMax(&sh.jhi, hi);
    }
    __syncthreads();
    // LDS: the window, the halo's second value, x if it fits
    const int base = sh.jlo, wlen = sh.jhi + 1 - base, nl = i0 - base, nh = wlen - nown;
    const size_t fixed = sizeof(TX) * ((size_t)wlen + nh), xbytes = sizeof(TX) * (size_t)nown;
    const bool fits = fixed <= (size_t)lds, xin = fixed + xbytes <= (size_t)lds;
    TX* win = reinterpret_cast<TX*>(dyn);
    TX* halo = win + wlen;
    TX* xl = halo + nh;
    if (!fits)
        for (int w = t; w < 4 * (b1 - b0); w += ST_THREADS) sh.wsum[0][w] = 1.0;
    uint32_t e = 1;
    double coef = 0.0;
    int done = 0;
    auto idle = [] {};
    if (!st_exchange(gs, sh, e, 0, block, b0, b1, np, ctl, coef, done, idle)) {
        if (t == 0) atomicOr(gs.err, ERR_SYNC);
        return;
    }
    if (done) {  // some block's window does not fit
        if (t == 0 && block == 0) atomicOr(gs.state, GS_REFUSED);
        return;
    }
    if (xin)
        for (int o = t; o < nown; o += ST_THREADS) xl[o] = a.xs[i0 + o];
    // halo row h: place in the window
    auto place = [&](int h) { return h < nl ? h : h + nown; };
    // r in halo[], q in the window
    for (int h = t; h < nh; h += ST_THREADS) {
        const P2 w = a.rq[base + place(h)];
        halo[h] = w.x;
        win[place(h)] = w.y;
    }
    // The launched kernels' s, p and t vectors carry v and t.  Blocks read each
    // other's t for the last time before they publish their part of the next
    // iteration's first sum, which its owner collects before it stores t again.
    // v is read up to the end of the BETA exchange, after the reader's part of
    // that sum has gone out, so its owner may be at the next v by then: v
    // alternates between two arrays, and is stored to one of them again after
    // the next iteration's BETA sum, to which every reader has added since.
    TX* tout = a.mm2;
    coef = sc->betas;
    bool ok = true;
    TX alpha = (TX)0, om = (TX)0;
    for (int it = 0; it < maxiter; ++it) {
        const bool fst = first && it == 0;
        TX* vout = it & 1 ? a.p : a.si;
        // opaque, so that the rows' addresses are formed where they are used:
        // kept across the iteration they do not fit the registers
        int t = threadIdx.x;
        asm volatile("" : "+v"(t));
        // p, v = A p
        const TX beta = (TX)coef;
        for (int h = t; h < nh; h += ST_THREADS) {
            const TX hr = halo[h];
            win[place(h)] = fst ? hr : hr + beta * win[place(h)];
        }
#pragma unroll
        for (int u = 0; u < J; ++u) {
            const int o = u * ST_THREADS + t;
            q[u] = fst ? r[u] : r[u] + beta * q[u];
            if (o < nown) win[nl + o] = q[u];
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < J; ++u) {
            const int o = u * ST_THREADS + t, i = i0 + o;
            double z = 0.0;
            if (o < nown) {
                const TX rh = a.rhat[i];
                v[u] = streamed_row<DIFF>(i, ld, nl + o, cd[u] & 0xffff, cd[u] >> 16,
                                          DIFF ? a.rsum[i] : 0.0, a.nbr, a.val, win);
                gs_store(vout + i, v[u]);
                z = (double)v[u] * (double)rh;
            }
            z = wave_sum(z);
            if ((t & 63) == 0) sh.wsum[0][u * ST_WAVES + wave] = z;
        }
        // the wave's stores have reached memory (vmcnt counts them) before
        // the block's barrier and its parts
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if (!(ok = st_exchange(gs, sh, ++e, FIN_ALPHA, block, b0, b1, np, ctl, coef, done, idle)))
            break;
        // s, t = A s, the rows backwards; the halo's p to halo[]
        alpha = (TX)coef;
        for (int h0 = t; h0 < nh; h0 += ST_H * ST_THREADS) {
            TX hv[ST_H];
#pragma unroll
            for (int m = 0; m < ST_H; ++m)
                hv[m] = gs_load(vout + base + place(min(h0 + m * ST_THREADS, nh - 1)));
#pragma unroll
            for (int m = 0; m < ST_H; ++m) {
                const int h = h0 + m * ST_THREADS, w = place(h);
                if (h < nh) {
                    const TX s = halo[h] - alpha * hv[m];
                    halo[h] = win[w];
                    win[w] = s;
                }
            }
        }
#pragma unroll
        for (int u = 0; u < J; ++u) {
            const int o = u * ST_THREADS + t;
            if (o < nown) win[nl + o] = r[u] - alpha * v[u];
        }
        __syncthreads();
#pragma unroll
        for (int u = J - 1; u >= 0; --u) {
            const int o = u * ST_THREADS + t, i = i0 + o;
            double z0 = 0.0, z1 = 0.0;
            if (o < nown) {
                r[u] = streamed_row<DIFF>(i, ld, nl + o, cd[u] & 0xffff, cd[u] >> 16,
                                          DIFF ? a.rsum[i] : 0.0, a.nbr, a.val, win);
                gs_store(tout + i, r[u]);
                z0 = (double)r[u] * (double)win[nl + o];
                z1 = (double)r[u] * (double)r[u];
            }
            z0 = wave_sum(z0);
            z1 = wave_sum(z1);
            if ((t & 63) == 0) {
                sh.wsum[0][u * ST_WAVES + wave] = z0;
                sh.wsum[1][u * ST_WAVES + wave] = z1;
            }
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        TX rh[J];  // read while the sums travel
#pragma unroll
        for (int u = 0; u < J; ++u) {
            const int o = u * ST_THREADS + t;
            rh[u] = o < nown ? a.rhat[i0 + o] : (TX)0;
        }
        if (!(ok = st_exchange(gs, sh, ++e, FIN_OMEGA, block, b0, b1, np, ctl, coef, done, idle)))
            break;
        // x, r, q
        om = (TX)coef;
#pragma unroll
        for (int u = 0; u < J; ++u) {
            const int o = u * ST_THREADS + t, i = i0 + o;
            double z0 = 0.0, z1 = 0.0;
            if (o < nown) {
                const TX s = win[nl + o];
                TX* x = xin ? xl + o : a.xs + i;
                *x = (*x + alpha * q[u]) + om * s;
                r[u] = s - om * r[u];
                q[u] = q[u] - om * v[u];
                z0 = (double)r[u] * (double)rh[u];
                z1 = (double)r[u] * (double)r[u];
            }
            z0 = wave_sum(z0);
            z1 = wave_sum(z1);
            if ((t & 63) == 0) {
                sh.wsum[0][u * ST_WAVES + wave] = z0;
                sh.wsum[1][u * ST_WAVES + wave] = z1;
            }
        }
        // while the sums travel: the halo's r to halo[], its q to the window
        auto halo_update = [&] {
            for (int h0 = t; h0 < nh; h0 += ST_H * ST_THREADS) {
                TX hv[ST_H], ht[ST_H];
#pragma unroll
                for (int m = 0; m < ST_H; ++m) {
                    const int j = base + place(min(h0 + m * ST_THREADS, nh - 1));
                    hv[m] = gs_load(vout + j);
                    ht[m] = gs_load(tout + j);
                }
#pragma unroll
                for (int m = 0; m < ST_H; ++m) {
                    const int h = h0 + m * ST_THREADS, w = place(h);
                    if (h < nh) {
                        const TX s = win[w], p = halo[h];
                        halo[h] = s - om * ht[m];
                        win[w] = p - om * hv[m];
                    }
                }
            }
        };
        if (!(ok = st_exchange(gs, sh, ++e, FIN_BETA, block, b0, b1, np, ctl, coef, done,
                                  halo_update)))
            break;
        if (done) break;
    }
    if (!ok) {  // unless x is in memory, the state there is the one the launch began with
        if (t == 0) {
            atomicOr(gs.err, ERR_SYNC);
            if (!xin) atomicOr(gs.state, GS_WRITTEN);
        }
        return;
    }
    if (t == 0) {
        atomicOr(gs.state, GS_WRITTEN);
        if (block == 0) *sc = sh.s;
    }
#pragma unroll
    for (int u = 0; u < J; ++u) {
        const int o = u * ST_THREADS + t, i = i0 + o;
        if (o < nown) {
            if (xin) a.xs[i] = xl[o];
            P2 w;
            w.x = r[u];
            w.y = q[u];
            a.rq[i] = w;
        }
    }
}

namespace host {

template <class TV, class TX, int J>
static int launch(isph_ctx* c, const KrylovArgs<TV, TX, short>& ka, const SolveCtl& ctl,
                  bool& first, int maxiter, bool& ran) {
    KrylovArgs<TV, TX, short> a = ka;
    const int parts = ST_MAXP * FIN_BLOCK;
    GridSync gs{c->gs_words, c->err, c->err + 1, parts};
    SolverScalars* sc = c->sc;
    SolveCtl t = ctl;
    int f = first, m = maxiter, l = (int)RESIDENT_LDS;
    void* args[] = {&a, &gs, &sc, &t, &f, &m, &l};
    if (int rc = grid_launch(c, (const void*)k_bicg_streamed<TV, TX, J>, GS_MAXB, ST_THREADS, args,
                             RESIDENT_LDS, parts + ST_COPIES * ST_GROUPS, ran))
        return rc;
    if (ran) {
        first = false;
        c->forms[ISPH_FORM_STREAMED] += 1;
    }
    return ISPH_OK;
}

// Rows a thread, from the most 256-row blocks that one of 256 blocks gets: 2
// up to 393k rows, 7 up to 1.31M.  Called above 261,120 rows, so every block has
// rows.
template <class TV, class TX>
int streamed_iterate(isph_ctx* c, const KrylovArgs<TV, TX, short>& a, const SolveCtl& ctl,
                     bool& first, int maxiter, bool& ran) {
    ran = false;
    const int np = nblk(c->n);
    // a block per CU; entry counts share a register with the diagonal's
    // position; 32-bit byte offsets into the values
    if (c->cus < GS_MAXB || np > ST_MAXP * FIN_BLOCK || c->prm.max_nbr > 0x7fff ||
        (uint64_t)c->prm.max_nbr * a.ld * sizeof(TV) > 0xffffffffull)
        return ISPH_OK;
    const int most = (np + GS_MAXB - 1) / GS_MAXB * BLOCK;  // rows of a block
    switch ((most + ST_THREADS - 1) / ST_THREADS) {
        case 2: return launch<TV, TX, 2>(c, a, ctl, first, maxiter, ran);
        case 3: return launch<TV, TX, 3>(c, a, ctl, first, maxiter, ran);
        case 4: return launch<TV, TX, 4>(c, a, ctl, first, maxiter, ran);
        case 5: return launch<TV, TX, 5>(c, a, ctl, first, maxiter, ran);
        case 6: return launch<TV, TX, 6>(c, a, ctl, first, maxiter, ran);
        case 7: return launch<TV, TX, 7>(c, a, ctl, first, maxiter, ran);
        default: return ISPH_OK;
    }
}

#define ISPH_STREAMED(TV, TX)                                                                  \
    template int streamed_iterate<TV, TX>(isph_ctx*, const KrylovArgs<TV, TX, short>&,         \
                                          const SolveCtl&, bool&, int, bool&);
ISPH_STREAMED(double, double)
ISPH_STREAMED(float, double)
ISPH_STREAMED(float, float)

}  // namespace host
}  // namespace isph
