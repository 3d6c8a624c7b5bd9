/*
 * hb_resident.hip -- the resident form of the default-order solve: one launch
 * runs many iterations of the seed process with the seed's vectors held by
 * the workgroups that own their rows, and one more advances the shifts.
 *
 * A launch per phase (hb_kernels.hip) moves r^, p, r, s, q and y through
 * memory seven times an iteration and pays, per launch, the chain of
 * dependent reads every workgroup starts with.  Here a workgroup of 1024
 * threads owns up to 8192 rows (one workgroup per compute unit): r, p, q, y
 * stay in its registers, r^ and s in its LDS, and only what others gather (p
 * and q) and what the window flush reads later (q and r) is stored.  An
 * iteration is then bound by its five waits for other workgroups: three
 * reductions (alpha~, omega~, beta~) and two waits for neighbours' rows.
 *
 * Arithmetic and its order are those of the launch-per-phase kernels: row
 * sums in CSR order, the dots from the same 256-row partial sums combined in
 * the same order, so every result is bitwise the same.
 *
 *   k_resident     iterations k .. until the seed converges, the window is
 *                  full, the cap is reached or res_C iterations are done
 *   k_res_stage    the scalar recurrences of every shift over those
 *                  iterations, the stopping rule, the seed switch and the
 *                  window decision (one thread per shift; the seed process
 *                  does not depend on the shifts between switches)
 *   k_res_coef, k_res_flush (hb_kernels.hip)  the window flush
 */
#include <hip/hip_runtime.h>
#include <limits.h>
#include <math.h>
#include "hb_shared.h"
#include "hb_launch.h"
#include "hb_device.h"

#define RB 1024   /* threads of a resident workgroup: four groups of one tile's 256 rows */

/* A launch's workgroups wait for each other, so all of them must be resident.
 * Before they touch anything they count themselves in; the last one to
 * arrive opens the launch, and one that has waited about 15 ms closes it (a
 * compare-and-swap decides), e.g. when another program's kernel holds
 * compute units: every workgroup then returns, and the host goes on with
 * the launch-per-phase kernels.  After the opening no wait can be endless;
 * each is bounded all the same, by about a second. */

#define RES_SPINS      (1 << 20)

typedef unsigned long long u64;

/* lane `from`'s value, known to be the same for the whole wave */
DEV double uniform(double v, int from = 0)
{
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), from),
                            __builtin_amdgcn_readlane(__double2loint(v), from));
}

DEV double shift_p(double p, double r, double s, double pb, double pbw)
{
    double pe = pb * p;   /* src/solver_dynamic.c:208-210 */
    pe = pe + r;
    return pe + pbw * s;
}

/* The matrix by its K diagonals (column - row, res_off), ascending: a row's
 * presence bits say which it has an entry on; FULL: values per row (rdia),
 * else one per diagonal (res_val).  KT 5 and 7: exactly that many, the middle
 * one the main diagonal (the 2-D and 3-D stencils), whose x is the row's own
 * and is not gathered; 8 and 16: at most so many, in any places. */
template <int S, bool SOLO>
struct res_lds {
    double rh[S][RB], s[S][RB];
    double ws[2][4 * S][4], ts[2][4 * S];
    double x[SOLO ? S * RB + 1 : 1];   /* one workgroup: the gathered vector, and a zero */
    double ex[HB_BLOCK / 2], ep[2][HB_BLOCK / 2];
    double red[8];
    unsigned need[8];
    int go;
};

/* Workgroup w of G.  WIDE: a workgroup may own more columns than it has
 * groups of threads (lcw up to 4; batches).  D: the record by value in the
 * kernel's arguments, or in constant memory. */
template <int SB, int E, int KT, bool FULL, bool SOLO, bool WIDE, class D>
DEV void resident_body(const D &d, res_lds<SB * E, SOLO> &L, int w, int G)
{
    constexpr int DP = KT & 1 ? KT / 2 : -1;
    constexpr int S = SB * E;         /* tiles of 256 rows per group of 256 threads */
    constexpr int NT = 4 * S;         /* tiles of the workgroup */
    /* One workgroup is bound by its instructions, 16 waves on four SIMDs, so
     * with few diagonals it keeps r^, s and the LDS address of every row's
     * neighbour in registers: a missing entry's address is that of a zero,
     * whose product leaves the sum as it is (the sum is never -0 and the
     * diagonals' values are finite), and a diagonal takes a read, a product
     * and a sum where clamping and selecting took eight more: 64 x 64, 108
     * iterations, 967 -> 757 us. */
    constexpr bool KEEP = SOLO && KT <= 8 && !(FULL && S * KT > 20);   /* there it spills */
    constexpr bool PACK = S * KT > 20;   /* two 16-bit byte offsets a register */
    /* the rows' values stay in registers where there is room: read from L2
     * in each SpMV they were a trip of their own ahead of the sums (251 x 173,
     * 394 iterations: 4.9 ms a solve with them kept, 5.3 without) */
    constexpr bool VALS = FULL && KT <= 8 && (SOLO ? S * KT <= 16 : S == 1);
    auto &l_rh = L.rh;
    auto &l_s = L.s;
    auto &l_ws = L.ws;
    auto &l_ts = L.ts;
    auto &l_x = L.x;
    auto &l_ex = L.ex;
    auto &l_ep = L.ep;
    auto &l_red = L.red;
    auto &l_need = L.need;
    int &l_go = L.go;

    hb_state *st = d.st;
    const int kf = st->ks;
    /* finished, the shifts have not caught up, or left to the launches */
    if (st->done | (st->k != kf) | st->res_fail) return;
    const int tid = threadIdx.x, lane = tid & 63;
    int lt = tid & 255;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int grp = wave >> 2;
    const int n = d.n, nblk = d.nblk, W = d.W, P = d.res_P;
    const int seed = st->seed, win_k0 = st->win_k0, fresh = st->res_fresh;
    int switched = st->switched;
    const double zscale = st->zscale, dot_zero = st->dot_zero;
    double rTr = st->rTr;
    const double sig = d.sigma[seed];
    const int one_only = d.stop[seed];      /* a stale switch target: switches again at once */
    const double thr = (d.tol * d.tol) * dot_zero;
    const int Rlast = n - HB_BLOCK * (nblk - 1);
    /* the last tile's rows are summed by T lanes each when it is short (the
     * CSR kernels' rule); every other tile has one lane per row */
    int T = 1;
    while ((T << 1) <= HB_BLOCK / Rlast && (T << 1) <= 64) T <<= 1;

    u64 *const mail = d.mail;               /* [3][256][8]: a reduction's column sums */
    int *flags = (int *)(mail + 3 * 2048);  /* [G] 64 bytes apart */

    /* reduce_partials sums the tiles' partial pairs in 256 columns: tiles c,
     * c + 256, c + 512, ... in that order.  A workgroup owns whole columns (w
     * CW ... + CW - 1), so each column's sum is formed inside one workgroup
     * and a reduction hands over 256 pairs whatever the size: with
     * contiguous rows per workgroup it took a second hand-over to combine
     * the columns, 10 us against 5 at 128^3.
     * Slot (u, e) of group g: column w CW + g % CW, row g / CW + 4 u / CW of
     * it, and E > 1: 8 e rows further (CW = 1, SB = 2), the tiles 2048 apart
     * that the seed update's partial sums chain.  CW > 4 (wh = log2(CW / 4)):
     * the columns first, four slot by slot, then the next row.  One workgroup:
     * tile g + 4 u. */
    const int lcw = SOLO ? 0 : d.res_lcw, CW = 1 << lcw;
    const int wh = WIDE ? max(lcw - 2, 0) : 0, wl = lcw - wh;
    const int ncol = min(nblk, 256);
    const int tile_g = SOLO ? grp : (w << lcw) + (grp & (CW - 1)) + 256 * (grp >> lcw);
    const int tile_u = SOLO ? 4 : 256 * (4 >> wl);
    /* its place among the workgroup's wave sums: column by column */
    const int ws_g = SOLO ? grp : (grp & (CW - 1)) * (NT >> lcw) + (grp >> lcw);
    const int ws_u = SOLO ? 4 : 4 >> wl;
    int t0 = tile_g;
    auto tile_of = [&](int sl) {
        const int u = sl / E;
        if (WIDE && !SOLO) return t0 + 4 * (u & ((1 << wh) - 1)) + tile_u * (u >> wh);
        return t0 + tile_u * u + 2048 * (sl % E);
    };
    auto ws_of = [&](int sl) {
        const int u = sl / E;
        if (WIDE && !SOLO) return ws_g + 4 * (u & ((1 << wh) - 1)) * (NT >> lcw) + ws_u * (u >> wh);
        return ws_g + ws_u * u + 8 * (sl % E);
    };
    /* how many rows it has (<= 0: none), uniform across the wave; own rows
     * are base + lt, a uniform address and one constant lane offset */
    auto rows_of = [&](int sl) { return n - tile_of(sl) * HB_BLOCK; };
    auto tile_ok = [&](int sl) { return rows_of(sl) > 0; };
    auto has_row = [&](int sl) { return lt < rows_of(sl); };
    /* called ahead of each phase: lane and tile are unknown to the compiler
     * from here, so what follows from them (addresses, bounds, masks of every
     * slot and diagonal) is formed anew in each phase.  Kept across the
     * iterations it takes hundreds of registers. */
    auto anew = [&]() {
        int a = tid & 255, b = tile_g;
        asm volatile("" : "+v"(a), "+s"(b));
        lt = a;
        t0 = b;
    };
#define ult ((unsigned)lt)
    auto own = [&](int sl, auto *base) { return base + (size_t)tile_of(sl) * HB_BLOCK; };
    int omin = 0, omax = 0;
#pragma unroll
    for (int j = 0; j < KT; ++j) {
        omin = min(omin, d.res_off[j]);
        omax = max(omax, d.res_off[j]);
    }

    /* the word this thread publishes: sum tid & 1 of the workgroup's column
     * tid >> 1.  A column's two sums have 64 bytes to themselves: with eight
     * workgroups' sums in a line each store had the line fetched anew by
     * every poller, and a reduction took 4 us instead of 2.5. */
    constexpr unsigned NOWORD = ~0u;
    unsigned word = NOWORD;
    if (!SOLO) {
        if (tid < 2 * CW && (w << lcw) + (tid >> 1) < ncol) {
            word = (unsigned)(8 * ((w << lcw) + (tid >> 1)) + (tid & 1));
            for (int q = 0; q < 3; ++q) mail_put(mail + 2048 * q + word, HB_MAIL_EMPTY);
        }
        if (tid == 0) __hip_atomic_store(&flags[16 * w], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (tid < 8) l_need[tid] = 0;
        __syncthreads();
        /* whose rows this workgroup gathers: the tiles one diagonal away
         * from one of its own */
        for (int e = tid; e < NT * HB_DIAG_K; e += RB) {
            const int ts = e / HB_DIAG_K, j = e % HB_DIAG_K;
            const int t = (w << lcw) + (ts & (CW - 1)) + 256 * (ts >> lcw);
            if (t < nblk && j < d.res_K) {
                const int o = d.res_off[j], r0 = HB_BLOCK * t;
                const int q0 = min(max(r0 + o, 0), n - 1) / HB_BLOCK;
                const int q1 = min(max(r0 + HB_BLOCK - 1 + o, 0), n - 1) / HB_BLOCK;
                for (int q = q0; q <= q1; ++q) {
                    const int g = (q & 255) >> lcw;
                    atomicOr(&l_need[g >> 5], 1u << (g & 31));
                }
            }
        }
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        if (tid == 0) {
            l_need[w >> 5] &= ~(1u << (w & 31));
            int g = 0;
            if (__hip_atomic_fetch_add(&d.rend[0], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1 == G) {
                int was = 0;
                __hip_atomic_compare_exchange_strong(&d.rend[1], &was, 1, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                     __HIP_MEMORY_SCOPE_AGENT);
                g = was == 0 ? 1 : was;
            } else {
                for (int spins = 0;; ++spins) {
                    g = __hip_atomic_load(&d.rend[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    if (g) break;
                    if (spins >= d.res_join) {
                        int was = 0;
                        __hip_atomic_compare_exchange_strong(&d.rend[1], &was, 2, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                             __HIP_MEMORY_SCOPE_AGENT);
                        g = was == 0 ? 2 : was;
                        break;
                    }
                    __builtin_amdgcn_s_sleep(2);
                }
            }
            l_go = g;
        }
        __syncthreads();
        if (l_go != 1) return;
    }

    /* a column's two published sums */
    auto poll2 = [&](const u64 *base, unsigned i, double &a, double &b) {
        u64 x, y;
        for (int spins = 0;; ++spins) {
            x = __hip_atomic_load(base + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            y = __hip_atomic_load(base + i + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (x != HB_MAIL_EMPTY && y != HB_MAIL_EMPTY) break;
            if (spins == RES_SPINS || ((spins & 255) == 255 && sync_timed_out(st))) {
                atomicOr(&st->status, HB_ST_SYNC_TIMEOUT);
                break;
            }
        }
        a = __longlong_as_double((long long)x);
        b = __longlong_as_double((long long)y);
    };
    /* this workgroup's rows of version `epoch` are stored: tell the others,
     * and wait until the ones it gathers from are as far.  The gathers are
     * agent-scope loads (sc1), which read past stale lines: an acquire fence
     * and plain loads took 4.3 + 3.6 us where this takes 1.2 + 1.0 (64^3: the
     * fence empties the XCD's L2 for every workgroup on it). */
    auto exchange = [&](int epoch) {
        if (SOLO) {
            __syncthreads();
            return;
        }
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        if (tid == 0)
            __hip_atomic_store(&flags[16 * w], epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (tid < 256) {
            if ((l_need[tid >> 5] >> (tid & 31)) & 1u) {
                for (int spins = 0;; ++spins) {
                    if (__hip_atomic_load(&flags[16 * tid], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= epoch) break;
                    if (spins == RES_SPINS || ((spins & 255) == 255 && sync_timed_out(st))) {
                        atomicOr(&st->status, HB_ST_SYNC_TIMEOUT);
                        break;
                    }
                }
            }
        }
        __syncthreads();
    };
    /* Reduction `kind`: the wave sums in l_ws become the tiles' sums (the
     * four waves in order), those of a column's `nr` tiles its sum, and the
     * columns' sums of all workgroups are then combined as reduce_partials
     * does: wave sums over the columns, then the four waves.  A mailbox is
     * emptied one reduction later: everyone has read it by then, having
     * published the next one's words after that. */
    auto reduce = [&](int kind, int nr, double &a0, double &a1) {
        __syncthreads();
        if (wave == 0 && (lane & 31) < NT) {
            const double *x = l_ws[lane >> 5][lane & 31];
            l_ts[lane >> 5][lane & 31] = ((x[0] + x[1]) + x[2]) + x[3];
        }
        if (SOLO) {
            __syncthreads();
            /* at most 16 tiles: one column each, the other waves' sums are 0 */
            const double va = lane < ncol ? 0.0 + l_ts[0][lane] : 0.0;
            const double vb = lane < ncol ? 0.0 + l_ts[1][lane] : 0.0;
            const double v = wave_sum2(va, vb);
            a0 = uniform(v) + 0.0;
            a1 = uniform(v, 32) + 0.0;
            return;
        }
        u64 *const m = mail + 2048 * kind;
        if (word != NOWORD) {
            const double *x = &l_ts[tid & 1][(tid >> 1) * (NT >> lcw)];
            double sum = 0.0;
            if (nr < 4) {
                for (int r = 0; r < nr; ++r) sum += x[r];
            } else {
#pragma unroll 1
                for (int r = 0; r < nr; r += 4) {
                    const double x0 = x[r], x1 = x[r + 1], x2 = x[r + 2], x3 = x[r + 3];
                    sum += x0;
                    sum += x1;
                    sum += x2;
                    sum += x3;
                }
            }
            /* the words emptied last have landed before this one can
             * complete a reduction anywhere */
            __builtin_amdgcn_s_waitcnt(0);
            mail_put_d(m + word, sum);
        }
        if (wave < 4) {
            double va = 0.0, vb = 0.0;
            if (lt < ncol) poll2(m, 8 * ult, va, vb);
            const double v = wave_sum2(va, vb);
            if ((lane & 31) == 0) l_red[wave + 4 * (lane >> 5)] = v;
        }
        __syncthreads();
        a0 = uniform(((l_red[0] + l_red[1]) + l_red[2]) + l_red[3]);
        a1 = uniform(((l_red[4] + l_red[5]) + l_red[6]) + l_red[7]);
        if (word != NOWORD) mail_put(mail + 2048 * ((kind + 2) % 3) + word, HB_MAIL_EMPTY);
    };

    /* ---- this workgroup's rows ---- */
    double r[S], p[S], q[S];
    double k_rh[KEEP ? S : 1], k_s[KEEP ? S : 1], k_av[VALS ? S : 1][VALS ? KT : 1];
    unsigned k_at[KEEP ? S : 1][KEEP ? PACK ? (KT + 1) / 2 : KT : 1];
    unsigned pres[S];
    auto rh_of = [&](int sl) -> double & { return KEEP ? k_rh[KEEP ? sl : 0] : l_rh[sl][tid]; };
    auto s_of = [&](int sl) -> double & { return KEEP ? k_s[KEEP ? sl : 0] : l_s[sl][tid]; };
    {
        const double *rs = d.rring + off((kf - 1) % (W + 1), n);
        const double *ps = fresh ? d.p_set + off(seed, n) : d.pring + off(kf % P, n);
        double *pn = d.pring + off(kf % P, n);
#pragma unroll
        for (int sl = 0; sl < S; ++sl) {
            r[sl] = 0.0; p[sl] = 0.0; q[sl] = 0.0; pres[sl] = 0;
            rh_of(sl) = 0.0;
            if (has_row(sl)) {
                r[sl] = own(sl, rs)[ult];
                p[sl] = own(sl, ps)[ult];
                rh_of(sl) = own(sl, (const double *)d.rhat)[ult];
                pres[sl] = own(sl, (const unsigned short *)d.rpres)[ult];
                if (fresh)
                    __hip_atomic_store(own(sl, pn) + ult, p[sl], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            if (VALS)
#pragma unroll
                for (int j = 0; j < KT; ++j)
                    k_av[VALS ? sl : 0][VALS ? j : 0] =
                        tile_ok(sl) ? ((const double *)d.rdia + ((size_t)tile_of(sl) * KT + j) * HB_BLOCK)[ult] : 0.0;
            if (KEEP)
#pragma unroll
                for (int j = 0; j < KT; ++j) {
                    const unsigned at = 8u * (unsigned)((pres[sl] >> j) & 1u ? tile_of(sl) * HB_BLOCK + lt + d.res_off[j]
                                                                            : S * RB);
                    unsigned &k = k_at[KEEP ? sl : 0][KEEP ? PACK ? j / 2 : j : 0];
                    k = PACK && j % 2 ? k | at << 16 : at;
                }
        }
        if (KEEP && tid == 0) l_x[S * RB] = 0.0;
    }
    /* the short last tile, T lanes per row: its group's threads take row
     * lt / T, lane lt % T */
    const bool tail_wg = T > 1 && (SOLO || ((nblk - 1) & 255) >> lcw == w);
    unsigned pres_t = 0;
    if (tail_wg) pres_t = d.rpres[(nblk - 1) * HB_BLOCK + min(lt / T, Rlast - 1)];

    /* x[base + i], base uniform */
    auto gather = [&](const double *x, int base, unsigned i) -> double {
        if (SOLO) return l_x[base + (int)i];
        x += base;
        return __hip_atomic_load(x + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    /* the row's sum over its diagonals, ascending (CSR order); own: its x */
    auto row_sum_of = [&](int sl, const double *__restrict__ x, double own_x) -> double {
        const int r0 = tile_of(sl) * HB_BLOCK;
        unsigned m = pres[sl];
        asm volatile("" : "+v"(m));   /* its masks: anew, too */
        const double *fv = FULL ? (const double *)d.rdia + (size_t)r0 * KT : nullptr;
        double acc = 0.0;
        if (KEEP && (T == 1 || tile_of(sl) != nblk - 1)) {
            double xv[KT], av[FULL && !VALS ? KT : 1];
#pragma unroll
            for (int j = 0; j < KT; ++j) {
                if (FULL && !VALS) av[FULL && !VALS ? j : 0] = (fv + j * HB_BLOCK)[ult];
                unsigned k = k_at[KEEP ? sl : 0][KEEP ? PACK ? j / 2 : j : 0];
                if (PACK) asm volatile("" : "+v"(k));   /* unpacked here, not ahead of the loop */
                const unsigned at = !PACK ? k : j % 2 ? k >> 16 : k & 0xffffu;
                xv[j] = *(const double *)((const char *)l_x + at);
            }
#pragma unroll
            for (int j = 0; j < KT; ++j)
                acc += (VALS ? k_av[VALS ? sl : 0][VALS ? j : 0] : FULL ? av[FULL && !VALS ? j : 0] : d.res_val[j]) * xv[j];
            return acc;
        }
        if (T == 1 || tile_of(sl) != nblk - 1) {
            constexpr int H = KT > 8 ? 8 : KT;
#pragma unroll
            for (int h = 0; h < KT; h += H) {
                double xv[H], av[FULL ? H : 1];
#pragma unroll
                for (int j = 0; j < H; ++j)
                    if (FULL)
                        av[FULL ? j : 0] = VALS ? k_av[VALS ? sl : 0][VALS ? j : 0] : (fv + (h + j) * HB_BLOCK)[ult];
                if (r0 + omin >= 0 && r0 + HB_BLOCK - 1 + omax < n) {
                    /* every row and diagonal of the tile lies inside x */
#pragma unroll
                    for (int j = 0; j < H; ++j)
                        xv[j] = h + j == DP ? own_x : gather(x, r0 + d.res_off[h + j], ult);
                } else {
#pragma unroll
                    for (int j = 0; j < H; ++j)
                        xv[j] = h + j == DP ? own_x
                                            : gather(x, 0, (unsigned)min(max(r0 + lt + d.res_off[h + j], 0), n - 1));
                }
#pragma unroll
                for (int j = 0; j < H; ++j) {
                    const double s = acc + (FULL ? av[FULL ? j : 0] : d.res_val[h + j]) * xv[j];
                    acc = (m >> (h + j)) & 1u ? s : acc;
                }
            }
            return acc;
        }
        /* the short last tile: row lt / T, whose entry number e belongs to
         * lane e % T */
        const int rl = min(lt / T, Rlast - 1), ln = lt & (T - 1);
        int e = 0;
        for (int j = 0; j < KT; ++j) {
            const double xv = gather(x, 0, (unsigned)min(max(r0 + rl + d.res_off[j], 0), n - 1));
            const double a = FULL ? (fv + j * HB_BLOCK)[(unsigned)rl] : d.res_val[j];
            const bool on = (pres_t >> j) & 1u;
            const double s = acc + a * xv;
            if (on && (e & (T - 1)) == ln) acc = s;
            e += on;
        }
        for (int h = T >> 1; h > 0; h >>= 1) acc += __shfl_xor(acc, h, 64);
        if (ln == 0 && lt / T < Rlast) l_ex[lt / T] = acc;
        return 0.0;
    };
    /* stores the wave sums of one or two slots' pairs */
    auto put_ws = [&](int s0, int s1, double a0, double b0, double a1, double b1) {
        if (s1 != s0) {
            const double v = wave_sum4(a0, b0, a1, b1);   /* rows: a0, a1, b0, b1 */
            const int row = lane >> 4;
            if ((lane & 15) == 0) l_ws[row >> 1][row & 1 ? ws_of(s1) : ws_of(s0)][wave & 3] = v;
        } else {
            const double v = wave_sum2(a0, b0);
            if ((lane & 31) == 0) l_ws[lane >> 5][ws_of(s0)][wave & 3] = v;
        }
    };

    /* x through the matrix: every slot's row sum into end(slot, sum, its two
     * partial sums), two slots' wave sums at a time */
    auto rows = [&](const double *__restrict__ x, const double *own_x, auto &&end) {
#pragma unroll
        for (int sl = 0; sl < S; sl += 2) {
            anew();
            constexpr bool two = S > 1;
            const int s1 = two ? sl + 1 : sl;
            double a0 = 0.0, b0 = 0.0, a1 = 0.0, b1 = 0.0;
            if (tile_ok(sl)) {
                const double t = row_sum_of(sl, x, own_x[sl]);
                if (T == 1 || tile_of(sl) != nblk - 1) end(sl, t, a0, b0);
            }
            if (two && tile_ok(s1)) {
                const double t = row_sum_of(s1, x, own_x[s1]);
                if (T == 1 || tile_of(s1) != nblk - 1) end(s1, t, a1, b1);
            }
            put_ws(sl, s1, a0, b0, a1, b1);
        }
        if (tail_wg) {
            anew();
            /* the short last tile: a row's sum came from T lanes, its first
             * lane's thread, T row, carries the row's share of the dots */
            __syncthreads();
#pragma unroll
            for (int sl = 0; sl < S; ++sl)
                if (tile_ok(sl) && tile_of(sl) == nblk - 1) {
                    double a0, b0;
                    end(sl, l_ex[min(lt, Rlast - 1)], a0, b0);
                    if (lt < Rlast) {
                        l_ep[0][lt] = a0;
                        l_ep[1][lt] = b0;
                    }
                }
            __syncthreads();
#pragma unroll
            for (int sl = 0; sl < S; ++sl)
                if (tile_ok(sl) && tile_of(sl) == nblk - 1) {
                    const bool first = (lt & (T - 1)) == 0 && lt / T < Rlast;
                    put_ws(sl, sl, first ? l_ep[0][lt / T] : 0.0, first ? l_ep[1][lt / T] : 0.0, 0.0, 0.0);
                }
        }
    };

    int status = 0;
    int k = kf;
    double omega = 0.0, qTq = 0.0, qTy = 0.0, rTs = 0.0, dot_r = 0.0, rTr_old = rTr;
    for (;; ++k) {
        anew();
        /* ---- s = (A + sigma) p ---- */
        if (SOLO)
#pragma unroll
            for (int sl = 0; sl < S; ++sl) l_x[tile_of(sl) * HB_BLOCK + lt] = p[sl];
        exchange(2 * k);
        const double *pk = d.pring + off(k % P, n);
        double *rprev = d.rring + off((k - 1) % (W + 1), n);
        const bool snap = k == win_k0;
        auto end1 = [&](int sl, double t, double &pa, double &pb) {
            pa = 0.0;
            pb = 0.0;
            const double si = t + sig * p[sl];
            s_of(sl) = si;
            if (has_row(sl)) {
                const double rh = rh_of(sl);
                if (snap) own(sl, (double *)d.p_snap)[ult] = p[sl];
                pa += rh * si;
                if (switched) {
                    const double rr = r[sl] * zscale;
                    own(sl, rprev)[ult] = rr;
                    r[sl] = rr;
                    pb += rh * rr;
                }
            }
        };
        rows(pk, p, end1);
        double a0, a1;
        anew();
        reduce(0, NT >> lcw, a0, a1);
        const double rtr = switched ? a1 : rTr;
        const double alpha = rtr / a0;
        if (switched) rTr = a1;
        switched = 0;
        rTs = a0;
        if (a0 == 0.0 || !isfinite(alpha)) status |= HB_ST_BREAKDOWN_RTS;

        /* ---- q = r - alpha~ s; y = (A + sigma) q ---- */
        const double nalpha = -alpha;
        anew();
        double *qk = d.qring + off(k % W, n);
#pragma unroll
        for (int sl = 0; sl < S; ++sl) {
            if (tile_ok(sl)) {
                q[sl] = r[sl] + nalpha * s_of(sl);
                if (SOLO) l_x[tile_of(sl) * HB_BLOCK + lt] = q[sl];
                if (has_row(sl))
                    __hip_atomic_store(own(sl, qk) + ult, q[sl], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
        exchange(2 * k + 1);
        double y[S];
        auto end2 = [&](int sl, double t, double &pa, double &pb) {
            pa = 0.0;
            pb = 0.0;
            y[sl] = t + sig * q[sl];
            if (has_row(sl)) {
                pa += q[sl] * q[sl];
                pb += q[sl] * y[sl];
            }
        };
        rows(qk, q, end2);
        anew();
        reduce(1, NT >> lcw, a0, a1);
        omega = a0 / a1;
        qTq = a0;
        qTy = a1;
        rTr_old = rTr;
        if (a1 == 0.0 || !isfinite(omega)) status |= HB_ST_BREAKDOWN_QTY;

        /* ---- r = q - omega~ y ---- */
        const double nw = -omega;
        anew();
        double *rk = d.rring + off(k % (W + 1), n);
#pragma unroll
        for (int u = 0; u < SB; ++u) {
            double ca = 0.0, cb = 0.0;
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const int sl = u * E + e;
                if (tile_ok(sl)) {
                    const double ri = q[sl] + nw * y[sl];
                    r[sl] = ri;
                    if (has_row(sl)) {
                        own(sl, rk)[ult] = ri;
                        ca += ri * ri;
                        cb += rh_of(sl) * ri;
                    }
                }
            }
            put_ws(u * E, u * E, ca, cb, 0.0, 0.0);
        }
        reduce(2, 4 * SB >> lcw, a0, a1);
        dot_r = a0;
        rTr = a1;
        const double beta = (alpha / omega) * (rTr / rTr_old);
        if (w == 0 && tid == 0) {
            d.aa[k] = alpha;
            d.wa[k] = omega;
            d.ba[k] = beta;
            d.drlog[k] = dot_r;
            d.qqlog[k] = qTq;
        }
        /* ---- p = beta~ p + r - beta~ omega~ s ---- */
        const double pbw = -beta * omega;
        anew();
        double *pn = d.pring + off((k + 1) % P, n);
#pragma unroll
        for (int sl = 0; sl < S; ++sl) {
            if (tile_ok(sl)) {
                p[sl] = shift_p(p[sl], r[sl], s_of(sl), beta, pbw);
                if (has_row(sl))
                    __hip_atomic_store(own(sl, pn) + ult, p[sl], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
        /* the seed converged (a switch or the end follows), the cap, a full
         * window, this launch's share */
        if (dot_r <= thr || k + 1 >= d.cap || k - win_k0 + 1 >= W || k - kf + 1 >= d.res_C || one_only) break;
    }
    if (w == 0 && tid == 0) {
        st->ks = k + 1;
        st->rTr = rTr;
        st->rTr_old = rTr_old;
        st->qTq = qTq;
        st->qTy = qTy;
        st->rTs = rTs;
        st->res_fresh = 0;
        st->switched = 0;
        if (status) atomicOr(&st->status, status);
    }
}

template <int SB, int E, int KT, bool FULL, bool SOLO>
__global__ __launch_bounds__(RB) void k_resident(hb_dev d)
{
    __shared__ res_lds<SB * E, SOLO> L;
    resident_body<SB, E, KT, FULL, SOLO, false>(d, L, SOLO ? 0 : (int)xcd_tile(blockIdx.x, gridDim.x),
                                                SOLO ? 1 : (int)gridDim.x);
}

/* ---- the shifts over the iterations a resident launch ran ---------------------
 * src/solver_dynamic.c:243-253 (per-shift recurrences), :278-303 (convergence
 * check), :312-341 (seed switch), as scalar_stage (hb_kernels.hip) does them an
 * iteration at a time.  Between switches no shift depends on another; what
 * an iteration hands to the next is pi, eta and zeta (three dependent
 * operations) and the growth bound (two), while the coefficients, with
 * their six divisions, are most of the work.  So of T = 1024 / M iterations
 * at a time a shift's owner thread runs the recurrences, every thread then
 * forms one (shift, iteration)'s coefficients, and the owner goes through
 * them for the bound and the stopping rule.  A thread taking its shift
 * through everything, and the switch's replay from memory, took 445 us of a
 * 251 x 173 solve (23 shifts, 394 iterations) and 107 of a 64 x 64 one (16,
 * 108); so 284 and 63.
 * The growth guard can close the window inside the range: all of it then
 * runs again up to that iteration (the recurrences do not depend on the
 * window), and the next launch takes the rest. */
struct res_shift {
    double eta, zeta, grow, own, zp;
    int stop_k, last_k, len, bad, spike;
};

/* bits of one (shift, iteration) */
#define RES_F_BAD   1   /* a divisor is 0 or not finite   */
#define RES_F_STOP  2   /* the shift has converged         */
#define RES_F_ABOVE 4   /* its estimate is above the seed's */

template <class D>
DEV void res_stage_body(const D &d)
{
    __shared__ double l_a[HB_RES_CMAX], l_w[HB_RES_CMAX], l_b[HB_RES_CMAX], l_ra[HB_RES_CMAX];
    __shared__ double l_nq[HB_RES_CMAX], l_nr[HB_RES_CMAX + 1], l_dr[HB_RES_CMAX];
    __shared__ double sh_zp[RB];
    __shared__ int sh_j[RB], sh_k[RB], sh_n[RB];
    __shared__ int sh_spike, sh_bad;
    /* T iterations of up to 1024 shifts: pi and the zeta before, the bound's
     * terms, the pi ahead of the first; sh_zp, sh_n: estimates and bits;
     * sh_j, sh_k: a shift's place in the flush list (-1: it has stopped) */
    __shared__ double sh_pi[RB], sh_z[RB], sh_b[RB], sh_o[RB], sh_p0[RB], sh_dj[RB];
    hb_state *st = d.st;
    const int tid = threadIdx.x, M = d.M;
    if (tid == 0) {
        if (d.rend[1] == 2) st->res_fail = 1;
        d.rend[0] = 0;
        d.rend[1] = 0;
        sh_spike = INT_MAX;
        sh_bad = 0;
    }
    const int k0 = st->k, ks = st->ks, s = st->seed;
    if (st->done || ks <= k0) {
        if (tid == 0) st->res_flush = 0;
        return;
    }
    const int win_k0 = st->win_k0, max_sigma0 = st->max_sigma, status0 = st->status, nsw = st->n_switch;
    const double dot_zero = st->dot_zero, dot_r_prev = st->dot_r;
    const double thr = (d.tol * d.tol) * dot_zero, sig_s = d.sigma[s];
    const int stop_s = d.stop[s], stop_count0 = st->stop_count, len0 = k0 - win_k0;
    const int nk = ks - k0;   /* at most HB_RES_CMAX */
    for (int i = tid; i < nk; i += RB) {
        const int k = k0 + i;
        const double dr = d.drlog[k];
        l_a[i] = d.aa[k];
        l_w[i] = d.wa[k];
        l_b[i] = d.ba[k];
        l_ra[i] = d.ba[k - 1] / d.aa[k - 1] * d.aa[k];
        l_nq[i] = sqrt(d.qqlog[k]);
        l_nr[i + 1] = sqrt(dr);
        l_dr[i] = dr;
        if (i == 0) l_nr[0] = sqrt(dot_r_prev);
    }
    if (len0 == 0) {
        /* a window opens: the seed first, then every running shift, ascending */
        int base = 1;
        for (int c0 = 0; c0 < M; c0 += RB) {
            const int j = c0 + tid;
            const int f = (j < M && !d.stop[j] && j != s) ? 1 : 0;
            sh_n[tid] = f;
            __syncthreads();
            for (int o = 1; o < RB; o <<= 1) {
                const int v = tid >= o ? sh_n[tid - o] : 0;
                __syncthreads();
                sh_n[tid] += v;
                __syncthreads();
            }
            if (f) {
                d.flist[base + sh_n[tid] - 1] = j;
                d.fpos[j] = base + sh_n[tid] - 1;
            }
            base += sh_n[RB - 1];
            __syncthreads();
        }
        if (tid == 0) {
            d.flist[0] = s;
            d.fpos[s] = 0;
            st->win_seedpos = 0;
            st->flush_cnt = base;
        }
    }
    __syncthreads();

    /* shifts c0 .. of at most 1024, each its thread's in z, up to kend */
    auto walk = [&](int c0, int kend, res_shift &z) {
        const int Mc = min(M - c0, RB), T = RB / Mc, bt = tid / Mc, bj = tid - bt * Mc;
        const int j = c0 + tid;
        bool live = tid < Mc && j != s && !d.stop[j];
        double pim1 = 1.0;
        z.zp = 0.0;
        z.stop_k = 0; z.last_k = 0; z.len = 0; z.bad = 0; z.spike = INT_MAX;
        if (tid < Mc) {
            sh_j[tid] = live ? d.fpos[j] : -1;
            sh_dj[tid] = sig_s - d.sigma[j];
        }
        if (live) {
            z.eta = d.eta[j];
            z.zeta = d.zeta[j];
            z.grow = d.growth_limit > 0.0 ? d.grow[j] : 0.0;
            z.own = d.growth_limit > 0.0 ? d.grow[M + j] : 0.0;
            pim1 = PI(d, j, k0 - 1);
        }
        for (int kc = k0; kc <= kend; kc += T) {
            const int nt = min(T, kend - kc + 1);
            if (live) {
                const double dj = sh_dj[tid];
                sh_p0[tid] = pim1;
#pragma unroll 4
                for (int t = 0; t < nt; ++t) {
                    const int i = kc - k0 + t;
                    z.eta = l_ra[i] * z.eta - dj * l_a[i] * pim1;
                    pim1 = z.eta + pim1;
                    sh_pi[t * Mc + tid] = pim1;
                    sh_z[t * Mc + tid] = z.zeta;
                    z.zeta = (1.0 - l_w[i] * dj) * z.zeta;
                    PI(d, j, kc + t) = pim1;
                }
            }
            __syncthreads();
            if (bt < nt && sh_j[bj] >= 0) {
                const int k = kc + bt, i = k - k0;
                const double dj = sh_dj[bj], ak = l_a[i], wk = l_w[i], beta = l_b[i];
                const double pik = sh_pi[tid], pm1 = bt ? sh_pi[tid - Mc] : sh_p0[bj];
                const double aj = (pm1 / pik) * ak;
                const double den = 1.0 - wk * dj;
                int f = !(den != 0.0 && isfinite(den) && pik != 0.0 && isfinite(pik)) ? RES_F_BAD : 0;
                const double wj = wk / den;
                const double zj = sh_z[tid];
                const double az = aj * zj;
                const double c1 = wj / (pik * zj);
                const double c2 = wj / (az * pik);
                const double c3 = -wj / (az * pm1);
                const double znew = den * zj;
                const double t = pm1 / pik;
                const double bb = t * t * beta;
                const double c4 = 1.0 / (pik * znew);
                double *c = d.coef + ((size_t)(k - win_k0) * M + sh_j[bj]) * 6;
                c[0] = c1; c[1] = aj; c[2] = c2; c[3] = c3; c[4] = bb; c[5] = c4;
                sh_b[tid] = fabs(bb);
                sh_o[tid] = fabs(bb) * (fabs(c2) * l_nq[i] + fabs(c3) * l_nr[i]) + fabs(c4) * l_nr[i + 1];
                const double zp = fabs(1.0 / (znew * pik));
                sh_zp[tid] = zp;
                if (zp * zp * l_dr[i] <= thr) f |= RES_F_STOP;
                else if (zp > 1.0) f |= RES_F_ABOVE;
                sh_n[tid] = f;
            }
            __syncthreads();
            if (live) {
                for (int t = 0; t < nt; ++t) {
                    const int k = kc + t, e = t * Mc + tid, f = sh_n[e];
                    if (f & RES_F_BAD) z.bad = 1;
                    if (d.growth_limit > 0.0) {
                        const double own = sh_o[e];
                        const double prev = k == 1 ? sqrt(dot_zero) : z.grow;
                        const double bound = sh_b[e] * prev + own;
                        if (!(bound <= d.growth_limit * own) && z.spike == INT_MAX) z.spike = k;
                        z.grow = bound;
                        z.own = own;
                    }
                    z.len = k - win_k0 + 1;
                    if (d.trace) d.trace[(size_t)k * M + j] = sh_zp[e] * sqrt(l_dr[k - k0] / dot_zero);
                    if (f & RES_F_STOP) {
                        z.stop_k = k;
                        live = false;
                        sh_j[tid] = -1;
                        break;
                    } else if (f & RES_F_ABOVE) {
                        z.last_k = k;
                        z.zp = sh_zp[e];
                    }
                }
            }
        }
        __syncthreads();
    };

    int kend = ks - 1;
    res_shift z;
    for (int pass = 0; pass < 2; ++pass) {
        for (int c0 = 0; c0 < M; c0 += RB) {
            walk(c0, kend, z);
            if (z.spike <= kend) atomicMin(&sh_spike, z.spike);
        }
        __syncthreads();
        const int sp = sh_spike;
        if (sp >= kend) break;
        kend = sp;   /* the window ends here: again, up to this iteration */
        __syncthreads();
    }
    const int spike = sh_spike == kend ? 1 : 0;
    const int len = kend - win_k0 + 1;

    /* what the iterations up to kend did to the shifts */
    int nconv = 0, bk = 0, bj = -1;
    double bz = 1.0;
    for (int c0 = 0; c0 < M; c0 += RB) {
        const int j = c0 + tid;
        if (M > RB) walk(c0, kend, z);
        if (j >= M) continue;
        if (j == s) {
            /* the seed in its own list: the recurrence at sigma_j = sigma_s */
            if (stop_s) continue;
            for (int k = k0; k <= kend; ++k) {
                const int i = k - k0;
                double *c = d.coef + (size_t)(k - win_k0) * M * 6;
                const double wa = l_w[i] / l_a[i];
                c[0] = l_w[i]; c[1] = l_a[i]; c[2] = wa; c[3] = -wa; c[4] = l_b[i]; c[5] = 1.0;
                if (d.trace) d.trace[(size_t)k * M + j] = sqrt(l_dr[i] / dot_zero);
            }
            d.act_len[0] = len;
            if (l_dr[kend - k0] <= thr) {
                d.stop[j] = 1;
                d.stop_iter[j] = kend;
                ++nconv;
            }
            continue;
        }
        if (d.stop[j]) continue;
        if (z.stop_k) {
            d.stop[j] = 1;
            d.stop_iter[j] = z.stop_k;
            ++nconv;
        }
        d.eta[j] = z.eta;
        d.zeta[j] = z.zeta;
        d.act_len[d.fpos[j]] = z.len;
        if (d.growth_limit > 0.0) {
            d.grow[j] = z.grow;
            d.grow[M + j] = z.own;
        }
        if (z.bad) sh_bad = 1;
        /* the arg-max rule's last candidates: the latest iteration at which
         * any running shift's estimate was above the seed's, the largest
         * there, the first of equals */
        if (z.last_k > bk || (z.last_k == bk && bj >= 0 && z.zp > bz)) {
            bk = z.last_k;
            bz = z.zp;
            bj = j;
        }
    }
    sh_zp[tid] = bz;
    sh_j[tid] = bj;
    sh_k[tid] = bk;
    sh_n[tid] = nconv;
    __syncthreads();
    for (int h = RB / 2; h > 0; h >>= 1) {
        if (tid < h) {
            const double z2 = sh_zp[tid + h];
            const int j2 = sh_j[tid + h], k2 = sh_k[tid + h];
            if (j2 >= 0 && (sh_j[tid] < 0 || k2 > sh_k[tid] ||
                            (k2 == sh_k[tid] && (z2 > sh_zp[tid] || (z2 == sh_zp[tid] && j2 < sh_j[tid]))))) {
                sh_zp[tid] = z2;
                sh_j[tid] = j2;
                sh_k[tid] = k2;
            }
            sh_n[tid] += sh_n[tid + h];
        }
        __syncthreads();
    }
    const int sc = stop_count0 + sh_n[0];
    const int ms = sh_j[0] >= 0 ? sh_j[0] : max_sigma0;
    const double dot_r = l_dr[kend - k0];
    /* the seed's own test can only hold at the range's last iteration */
    const bool seed_out = (stop_s || dot_r <= thr) && sc < M;
    const int do_switch = seed_out && ms >= 0;
    const int nst = (seed_out && ms < 0) || (status0 & HB_ST_NO_SWITCH_TARGET) != 0;
    __syncthreads();
    if (do_switch) {
        const int m = ms, k = kend;
        const double ds = sig_s - d.sigma[m];
        if (tid == 0) st->zscale = 1.0 / (d.zeta[m] * PI(d, m, k));
        for (int i = 1 + tid; i <= k; i += RB) {
            const double t0 = PI(d, m, i - 1), t1 = PI(d, m, i);
            d.aa[i] = (t0 / t1) * d.aa[i];
            d.ba[i] = (t0 / t1) * (t0 / t1) * d.ba[i];
            d.wa[i] = d.wa[i] / (1.0 - d.wa[i] * ds);
        }
        __syncthreads();
        const double sig_m = d.sigma[m];
        for (int c0 = 0; c0 < M; c0 += RB) {
            const int j = c0 + tid;
            const bool run = j < M && !d.stop[j] && j != m;
            const double dm = j < M ? sig_m - d.sigma[j] : 0.0;
            double e = 0.0, z1 = 1.0, pim1 = run ? PI(d, j, 0) : 1.0;
            /* the archives through LDS: read where they lie, an iteration
             * was two dependent trips to memory and a division, 0.6 us */
            for (int i0 = 1; i0 <= k; i0 += HB_RES_CMAX) {
                const int ni = min(HB_RES_CMAX, k + 1 - i0);
                __syncthreads();
                for (int i = tid; i < ni; i += RB) {
                    const double a = d.aa[i0 + i];
                    l_a[i] = a;
                    l_w[i] = d.wa[i0 + i];
                    l_ra[i] = d.ba[i0 + i - 1] / d.aa[i0 + i - 1] * a;
                }
                __syncthreads();
                if (!run) continue;
#pragma unroll 4
                for (int i = 0; i < ni; ++i) {
                    e = l_ra[i] * e - dm * l_a[i] * pim1;
                    pim1 = e + pim1;
                    PI(d, j, i0 + i) = pim1;
                    z1 = (1.0 - l_w[i] * dm) * z1;
                }
            }
            if (j < M) {
                d.eta[j] = e;
                d.zeta[j] = z1;
            }
        }
    }
    /* a wait that ran out voids the solve: it ends here */
    const int done = sc >= M || kend + 1 >= d.cap || nst || (status0 & HB_ST_SYNC_TIMEOUT);
    const int fl = do_switch || done || len >= d.W || spike;
    const int xonly = fl && done && !do_switch && !spike;
    if (d.growth_limit > 0.0 && fl) {
        __syncthreads();
        for (int j = tid; j < M; j += RB) d.grow[j] = d.grow[M + j];
    }
    if (tid == 0) {
        int bits = 0;
        if (sh_bad) bits |= HB_ST_BREAKDOWN_SHIFT;
        if (seed_out && ms < 0) bits |= HB_ST_NO_SWITCH_TARGET;
        if (bits) atomicOr(&st->status, bits);
        st->stop_count = sc;
        st->max_sigma = ms;
        st->dot_r = dot_r;
        st->kprev = kend;
        st->prev_seed = s;
        if (do_switch) {
            d.switch_k[nsw] = kend;
            d.switch_to[nsw] = ms;
            st->n_switch = nsw + 1;
            st->seed = ms;
            st->switched = 1;
            st->res_fresh = 1;
        }
        st->flush = fl;
        st->flush_xonly = xonly;
        st->res_flush = fl ? (xonly ? 2 : 1) : 0;
        if (fl) {
            st->flush_k0 = win_k0;
            st->flush_len = len;
            st->flush_tail = spike;
            st->win_k0 = kend + 1;
        }
        /* a window that closed inside the range: its successor's first p is
         * still in the ring of p, and the flush keeps it */
        st->res_snap = fl && kend + 1 < ks ? kend + 1 : 0;
        st->k = kend + 1;
        st->done = done;
    }
}

__global__ __launch_bounds__(RB) void k_res_stage(hb_dev d)
{
    res_stage_body(d);
}

/* The launch-per-phase kernels take over (a resident launch could not
 * start): the seed's p moves to where they keep it. */
template <class D>
DEV void res_leave_body(const D &d)
{
    hb_state *st = d.st;
    if (st->done) return;
    if (!st->res_fresh) {
        const double *p = d.pring + off(st->k % d.res_P, d.n);
        double *ps = d.p_set + off(st->seed, d.n);
        const int n = d.n;
        for (int i = blockIdx.x * HB_BLOCK + threadIdx.x; i < n; i += gridDim.x * HB_BLOCK) ps[i] = p[i];
    }
}

__global__ __launch_bounds__(HB_BLOCK) void k_res_leave(hb_dev d) { res_leave_body(d); }

/* ---- layout ------------------------------------------------------------------
 * The diagonals (column - row) of tile t (rows 256 t ...) in ascending order,
 * toff[16 t ...], and their number tK[t]; bad is set when a tile has more
 * than HB_DIAG_K or a row's columns do not ascend. */
__global__ __launch_bounds__(HB_BLOCK) void k_res_scan(int n, const unsigned *__restrict__ ptr,
                                                       const unsigned *__restrict__ col, int *__restrict__ tK,
                                                       int *__restrict__ toff, int *bad)
{
    __shared__ int sh_min[2];
    const int t = blockIdx.x, i = t * HB_BLOCK + threadIdx.x, tid = threadIdx.x;
    unsigned e = i < n ? ptr[i] : 0;
    const unsigned e1 = i < n ? ptr[i + 1] : 0;
    int s = 0;
    bool asc = true;
    if (tid == 0) sh_min[0] = INT_MAX;
    __syncthreads();
    for (;; ++s) {
        /* the smallest diagonal any row has not passed yet */
        const int b = s & 1;
        const int o = e < e1 ? (int)col[e] - i : INT_MAX;
        if (e < e1) atomicMin(&sh_min[b], o);
        __syncthreads();
        const int m = sh_min[b];
        if (tid == 0) sh_min[b ^ 1] = INT_MAX;
        if (m == INT_MAX || s == HB_DIAG_K) break;
        if (o == m && e < e1) {
            if (e + 1 < e1 && col[e + 1] <= col[e]) asc = false;
            ++e;
        }
        __syncthreads();
        if (tid == 0) toff[HB_DIAG_K * t + s] = m;
    }
    if (!asc || e < e1) atomicOr(bad, 1);
    if (tid == 0) tK[t] = s;
}

/* Presence bits of every row on the matrix's diagonals d.res_off; lo and hi
 * get the smallest and largest bit pattern of each diagonal's values. */
__global__ __launch_bounds__(HB_BLOCK) void k_res_bits(hb_dev d, unsigned short *__restrict__ pres,
                                                       u64 *__restrict__ lo, u64 *__restrict__ hi)
{
    __shared__ u64 sh_lo[HB_DIAG_K], sh_hi[HB_DIAG_K];
    const int i = blockIdx.x * HB_BLOCK + threadIdx.x, K = d.res_K;
    if (threadIdx.x < HB_DIAG_K) {
        sh_lo[threadIdx.x] = ~0ull;
        sh_hi[threadIdx.x] = 0;
    }
    __syncthreads();
    if (i < d.n) {
        unsigned bits = 0;
        int j = 0;
        for (unsigned e = d.ptr[i]; e < d.ptr[i + 1]; ++e) {
            const int o = (int)d.col[e] - i;
            while (j < K - 1 && d.res_off[j] != o) ++j;
            const u64 v = (u64)__double_as_longlong(d.val[e]);
            if (v < sh_lo[j]) atomicMin(&sh_lo[j], v);
            if (v > sh_hi[j]) atomicMax(&sh_hi[j], v);
            bits |= 1u << j;
        }
        pres[i] = (unsigned short)bits;
    }
    __syncthreads();
    if (threadIdx.x < (unsigned)K) {
        atomicMin(&lo[threadIdx.x], sh_lo[threadIdx.x]);
        atomicMax(&hi[threadIdx.x], sh_hi[threadIdx.x]);
    }
}

/* The rows' values by diagonal, [tile][KT][256], read in CSR order from val
 * at every solve (a caller may change them in place). */
template <class D>
DEV void res_fill_body(const D &d, int t)
{
    const int i = t * HB_BLOCK + threadIdx.x, KT = d.res_KT;
    const unsigned m = i < d.n ? d.rpres[i] : 0;
    unsigned e = i < d.n ? d.ptr[i] : 0;
    double *out = d.rdia + (size_t)t * KT * HB_BLOCK + threadIdx.x;
    const double *val = d.val;
    for (int j = 0; j < KT; ++j) out[(size_t)j * HB_BLOCK] = (m >> j) & 1u ? val[e++] : 0.0;
}

__global__ __launch_bounds__(HB_BLOCK) void k_res_fill(hb_dev d) { res_fill_body(d, blockIdx.x); }

/* ---- batches -----------------------------------------------------------------
 * One launch runs every problem's iterations, each problem in a cluster of
 * workgroups of its own that rendezvous and wait among themselves only;
 * tab[2 b], tab[2 b + 1]: the problem of workgroup b and its place in the
 * cluster, a cluster's workgroups side by side.  The dispatcher deals
 * workgroups to the XCDs in order, so the clusters that do not fit the
 * compute units at once follow as earlier ones end, and a waiting cluster is
 * never ahead of one it keeps out.
 *
 * A batch took 8 launches an iteration whose workgroups each began with the
 * dependent reads problem, record, vectors; here an iteration costs a problem
 * its waits, about 18 us in a cluster of 16 tiles a workgroup.  48 problems
 * of 1000 to 200000 rows: 60.9 ms a solve before, 30.4 ms so; bound by the
 * first rounds, whose 440 workgroups take the 256 compute units twice. */
template <int SB, int KT, bool FULL>
DEV void resident_of(const HB_K hb_dev &d, unsigned char *lds, int w)
{
    if (d.res_G == 1)
        resident_body<4, 1, KT, FULL, true, true>(d, *(res_lds<4, true> *)lds, 0, 1);
    else
        resident_body<SB, 1, KT, FULL, false, true>(d, *(res_lds<SB, false> *)lds, w, d.res_G);
}

template <int SB>
__global__ __launch_bounds__(RB) void kb_resident(const hb_dev *__restrict__ devs, const int *__restrict__ tab)
{
    __shared__ __attribute__((aligned(16))) unsigned char
        lds[sizeof(res_lds<4, true>) > sizeof(res_lds<SB, false>) ? sizeof(res_lds<4, true>)
                                                                  : sizeof(res_lds<SB, false>)];
    const HB_K int *t = read_only(tab) + 2 * blockIdx.x;
    const HB_K hb_dev &d = read_only(devs)[t[0]];
    const int w = t[1];
    switch (d.res_KT + (d.res_full ? 100 : 0)) {
    case 5: return resident_of<SB, 5, false>(d, lds, w);
    case 7: return resident_of<SB, 7, false>(d, lds, w);
    case 16: return resident_of<SB, 16, false>(d, lds, w);
    case 105: return resident_of<SB, 5, true>(d, lds, w);
    case 107: return resident_of<SB, 7, true>(d, lds, w);
    case 116: return resident_of<SB, 16, true>(d, lds, w);
    }
}

__global__ __launch_bounds__(RB) void kb_res_stage(const hb_dev *__restrict__ devs)
{
    res_stage_body(read_only(devs)[blockIdx.x]);
}

__global__ __launch_bounds__(HB_BLOCK) void kb_res_fill(const hb_dev *__restrict__ devs, const int *__restrict__ tab)
{
    const HB_K int *t = read_only(tab) + 2 * blockIdx.x;
    const HB_K hb_dev &d = read_only(devs)[t[0]];
    if (d.res_full) res_fill_body(d, t[1]);
}

__global__ __launch_bounds__(HB_BLOCK) void kb_res_leave(const hb_dev *__restrict__ devs)
{
    res_leave_body(read_only(devs)[blockIdx.y]);
}

/* ---- launch layer --------------------------------------------------------- */
template <int SB, int E, int KT, bool FULL>
static int launch_res(const hb_dev *d, hipStream_t s)
{
    if (d->res_G > 1) {
        if constexpr (SB < 4) {
            hipLaunchKernelGGL((k_resident<SB, E, KT, FULL, false>), dim3(d->res_G), dim3(RB), 0, s, *d);
            return (int)hipGetLastError();
        }
    } else if constexpr (E == 1) {
        hipLaunchKernelGGL((k_resident<SB, E, KT, FULL, true>), dim3(1), dim3(RB), 0, s, *d);
        return (int)hipGetLastError();
    }
    return -1;
}

template <int SB, int E>
static int launch_res_k(const hb_dev *d, hipStream_t s)
{
    switch (d->res_KT + (d->res_full ? 100 : 0)) {
    case 5: return launch_res<SB, E, 5, false>(d, s);
    case 7: return launch_res<SB, E, 7, false>(d, s);
    case 8: return launch_res<SB, E, 8, false>(d, s);
    case 16: return launch_res<SB, E, 16, false>(d, s);
    case 105: return launch_res<SB, E, 5, true>(d, s);
    case 107: return launch_res<SB, E, 7, true>(d, s);
    case 108: return launch_res<SB, E, 8, true>(d, s);
    case 116: return launch_res<SB, E, 16, true>(d, s);
    }
    return -1;
}

extern "C" {

/* Shape for nblk tiles: workgroups (returned, 0 where the rows do not fit),
 * SB and E (tiles per group of 256 threads), lcw (log2 of the columns per
 * workgroup). */
int hb_k_res_shape(int nblk, int cus, int *SB, int *E, int *lcw)
{
    *SB = *E = 1;
    *lcw = 0;
    if (nblk <= 16) {
        /* one workgroup: every wait is a barrier of its own */
        *SB = nblk <= 4 ? 1 : nblk <= 8 ? 2 : 4;
        return 1;
    }
    if (nblk <= 256) *lcw = 2;
    else if (nblk <= 512) *lcw = 1;
    else if (nblk > 1024) *SB = 2;
    if (nblk > 2048) *E = nblk <= 4096 ? 2 : 4;
    const int G = ((nblk < 256 ? nblk : 256) + (1 << *lcw) - 1) >> *lcw;
    return nblk <= 8192 && G <= cus ? G : 0;
}

/* A problem of a batch whose workgroups take 4 SB tiles: its workgroups (one
 * up to 16 tiles), 0 where the rows do not fit; lcw up to 4. */
int hb_k_res_shape_b(int nblk, int SB, int *lcw)
{
    *lcw = 0;
    if (nblk <= 16) return 1;
    const int rows = (nblk + 255) / 256;   /* tiles of a column */
    if (rows > 4 * SB || nblk > 2048) return 0;
    while ((rows << (*lcw + 1)) <= 4 * SB) ++*lcw;
    return ((nblk < 256 ? nblk : 256) + (1 << *lcw) - 1) >> *lcw;
}

int hb_kb_res_iterations(const hb_batch *B, hipStream_t s)
{
    const dim3 g(B->n_res), bl(RB);
    if (B->res_SB == 1) hipLaunchKernelGGL(kb_resident<1>, g, bl, 0, s, B->devs, B->t_res);
    else if (B->res_SB == 2) hipLaunchKernelGGL(kb_resident<2>, g, bl, 0, s, B->devs, B->t_res);
    else hipLaunchKernelGGL(kb_resident<4>, g, bl, 0, s, B->devs, B->t_res);
    hipLaunchKernelGGL(kb_res_stage, dim3(B->nprob), bl, 0, s, B->devs);
    return (int)hipGetLastError();
}

int hb_kb_res_fill(const hb_batch *B, hipStream_t s)
{
    hipLaunchKernelGGL(kb_res_fill, dim3(B->n_spmv_tiles), dim3(HB_BLOCK), 0, s, B->devs, B->t_spmv);
    return (int)hipGetLastError();
}

int hb_kb_res_leave(const hb_batch *B, hipStream_t s)
{
    hipLaunchKernelGGL(kb_res_leave, dim3(64, B->nprob), dim3(HB_BLOCK), 0, s, B->devs);
    return (int)hipGetLastError();
}

int hb_k_res_scan(const hb_dev *d, int *tK, int *toff, int *bad, hipStream_t s)
{
    hipLaunchKernelGGL(k_res_scan, dim3(d->nblk), dim3(HB_BLOCK), 0, s, d->n, d->ptr, d->col, tK, toff, bad);
    return (int)hipGetLastError();
}

int hb_k_res_bits(const hb_dev *d, unsigned short *pres, unsigned long long *lo, unsigned long long *hi,
                  hipStream_t s)
{
    hipLaunchKernelGGL(k_res_bits, dim3(d->nblk), dim3(HB_BLOCK), 0, s, *d, pres, lo, hi);
    return (int)hipGetLastError();
}

int hb_k_res_fill(const hb_dev *d, hipStream_t s)
{
    hipLaunchKernelGGL(k_res_fill, dim3(d->nblk), dim3(HB_BLOCK), 0, s, *d);
    return (int)hipGetLastError();
}

int hb_k_res_stage(const hb_dev *d, hipStream_t s)
{
    hipLaunchKernelGGL(k_res_stage, dim3(1), dim3(RB), 0, s, *d);
    return (int)hipGetLastError();
}

int hb_k_res_iterations(const hb_dev *d, hipStream_t s)
{
    int e = -1;
    if (d->res_E == 1) {
        if (d->res_SB == 1) e = launch_res_k<1, 1>(d, s);
        else if (d->res_SB == 2) e = launch_res_k<2, 1>(d, s);
        else if (d->res_SB == 4) e = launch_res_k<4, 1>(d, s);   /* one workgroup */
    } else if (d->res_SB == 2) {
        if (d->res_E == 2) e = launch_res_k<2, 2>(d, s);
        else if (d->res_E == 4) e = launch_res_k<2, 4>(d, s);
    }
    if (e) return e;
    return hb_k_res_stage(d, s);
}

int hb_k_res_leave(const hb_dev *d, hipStream_t s)
{
    hipLaunchKernelGGL(k_res_leave, dim3(d->vec_grid), dim3(HB_BLOCK), 0, s, *d);
    return (int)hipGetLastError();
}

} /* extern "C" */
