/*
 * hb_device.h -- device helpers shared by the kernel files: constant-memory
 * reads, wave sums, words handed between the workgroups of one launch.
 */
#ifndef HB_DEVICE_H
#define HB_DEVICE_H

#include <hip/hip_runtime.h>
#include "hb_shared.h"

#define DEV __device__ __forceinline__

typedef double dbl2 __attribute__((ext_vector_type(2)));

/* Constant address space: the compiler takes what is read through it as
 * unchanged for the rest of the launch, and a wave-uniform address there
 * becomes a scalar load. */
#define HB_K __attribute__((address_space(4)))

/* p, from here to the end of the launch read-only, as constant memory.  The
 * empty asm makes the returned pointer unknown to the compiler until this
 * point, so no read through it moves above what comes before (a wait for
 * the data in the same launch).  Without it a kernel with a barrier or an
 * atomic anywhere before the reads loses their scalar loads: the compiler
 * cannot show that nothing in between stored to them, and makes every
 * uniform read a vector load. */
template <typename T>
DEV const HB_K T *read_only(const T *p)
{
    asm volatile("" : "+s"(p));
    return (const HB_K T *)p;
}

/* ---- reductions ----------------------------------------------------------- */
DEV double wave_sum(double v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

/* ---- values handed between the workgroups of one launch ---------------------
 * A workgroup dispatched first computes a value the launch's other
 * workgroups need.  It stores it with an agent-scope relaxed atomic store (a
 * write-through store, sc1, on gfx950) into a mailbox that holds
 * HB_MAIL_EMPTY until then; the others poll it with agent-scope relaxed
 * atomic loads (sc1), which read past any stale cache line.  Every word
 * that crosses workgroups inside a launch moves this way, so no L2
 * write-back or invalidate (what an agent-scope release or acquire costs)
 * is needed.  The first workgroups of a grid are dispatched before the
 * later ones (in order on each XCD), so the publisher is always running
 * when a waiter spins; the spin is bounded all the same (about 0.5 s), and
 * a waiter that gives up sets HB_ST_SYNC_TIMEOUT and goes on instead of
 * hanging; every later waiter sees the bit and does not wait at all. */
#define HB_SPIN_LIMIT (1 << 17)

/* a waiter polls the status word too: once one has timed out, none waits */
DEV bool sync_timed_out(hb_state *st)
{
    return (__hip_atomic_load(&st->status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & HB_ST_SYNC_TIMEOUT) != 0;
}

DEV void mail_put(unsigned long long *slot, unsigned long long v)
{
    __hip_atomic_store(slot, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

DEV void mail_put_d(unsigned long long *slot, double v)
{
    mail_put(slot, (unsigned long long)__double_as_longlong(v));
}

/* the published word, polled by the calling thread alone (HB_MAIL_EMPTY
 * after a time-out) */
DEV unsigned long long mail_poll_bits(unsigned long long *slot, hb_state *st)
{
    unsigned long long v;
    for (int spins = 0;; ++spins) {
        v = __hip_atomic_load(slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (v != HB_MAIL_EMPTY) break;
        if (spins == HB_SPIN_LIMIT || ((spins & 255) == 255 && sync_timed_out(st))) {
            atomicOr(&st->status, HB_ST_SYNC_TIMEOUT);
            break;
        }
        /* a few hundred cycles between polls: thousands of resident
         * workgroups poll one word, and the publisher needs the memory
         * system more than they do */
        __builtin_amdgcn_s_sleep(8);
    }
    return v;
}

DEV double mail_poll(unsigned long long *slot, hb_state *st)
{
    return __longlong_as_double((long long)mail_poll_bits(slot, st));
}

/* the published double; thread 0 of the workgroup waits, every thread gets it */
DEV double mail_wait(unsigned long long *slot, hb_state *st)
{
    __shared__ double sh_v;
    if (threadIdx.x == 0) sh_v = mail_poll(slot, st);
    __syncthreads();
    return sh_v;
}

/* the published word, to every thread of the workgroup */
DEV unsigned long long mail_wait_bits(unsigned long long *slot, hb_state *st)
{
    __shared__ unsigned long long sh_u;
    if (threadIdx.x == 0) sh_u = mail_poll_bits(slot, st);
    __syncthreads();
    return sh_u;
}

/* a value the kernel's other workgroups read before the launch ends */
template <bool PUB>
DEV void store_pub(double *p, double v)
{
    if (PUB) __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else *p = v;
}

template <bool PUB>
DEV void store_pub(int *p, int v)
{
    if (PUB) __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else *p = v;
}

/* a word another workgroup of the launch stored with store_pub<true> */
DEV int load_pub(const int *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

DEV size_t off(int j, int n) { return (size_t)j * (size_t)n; }
#define PI(d, j, i) ((d).pi[(size_t)(j) * (size_t)(d).cap + (size_t)(i)])

/* Workgroup b runs on XCD b % 8 (the dispatcher deals workgroups round
 * robin over the eight XCDs, each with its own L2).  Tile order: XCD x gets
 * the contiguous tiles [start(x), start(x+1)), so a tile's column halo (the
 * rows around it, and the rows a plane away for stencils) was mostly
 * fetched into the same L2 by its neighbours.  A bijection on 0 .. nb-1. */
DEV unsigned xcd_tile(unsigned b, unsigned nb)
{
    const unsigned q = nb / 8, r = nb % 8, x = b % 8;
    return x * q + min(x, r) + b / 8;
}


/* ---- sums over a wavefront without LDS ---------------------------------------
 * wave_sum adds, for o = 32, 16, 8, 4, 2, 1, lane i ^ o to lane i.  Addition
 * commutes, so any exchange that pairs the same lanes gives the same bits:
 * the gfx950 half and row swaps for 32 and 16 (which also let two values
 * share a step), DPP for the rest.  A wave_sum through __shfl_xor is twelve
 * LDS permutes; eight tiles' sums of a 1024-thread workgroup took longer
 * than the SpMV that fed them. */
template <int CTRL>
DEV double dpp(double v)
{
    int lo = __double2loint(v), hi = __double2hiint(v);
    lo = __builtin_amdgcn_update_dpp(0, lo, CTRL, 0xf, 0xf, true);
    hi = __builtin_amdgcn_update_dpp(0, hi, CTRL, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}

/* sum over each row of 16 lanes: o = 8, 4, 2, 1 */
DEV double row_sum(double v)
{
    v += dpp<0x128>(v);                /* row_ror:8  = i ^ 8 */
    v += dpp<0x1b>(dpp<0x141>(v));     /* half mirror (i ^ 7), quad 3,2,1,0 (i ^ 3): i ^ 4 */
    v += dpp<0x4e>(v);                 /* quad 2,3,0,1: i ^ 2 */
    v += dpp<0xb1>(v);                 /* quad 1,0,3,2: i ^ 1 */
    return v;
}

/* lanes below 32: a's halves added; the others: b's */
DEV double swap32_add(double a, double b)
{
    const auto l = __builtin_amdgcn_permlane32_swap(__double2loint(a), __double2loint(b), false, false);
    const auto h = __builtin_amdgcn_permlane32_swap(__double2hiint(a), __double2hiint(b), false, false);
    return __hiloint2double(h[0], l[0]) + __hiloint2double(h[1], l[1]);
}

/* even rows of 16 lanes: a's row pairs added; odd rows: b's */
DEV double swap16_add(double a, double b)
{
    const auto l = __builtin_amdgcn_permlane16_swap(__double2loint(a), __double2loint(b), false, false);
    const auto h = __builtin_amdgcn_permlane16_swap(__double2hiint(a), __double2hiint(b), false, false);
    return __hiloint2double(h[0], l[0]) + __hiloint2double(h[1], l[1]);
}

/* wave sums of two values: every lane below 32 gets a's, the others b's */
DEV double wave_sum2(double a, double b)
{
    const double v = swap32_add(a, b);
    return row_sum(swap16_add(v, v));
}

/* wave sums of four values: rows 0..3 of 16 lanes get a's, c's, b's, d's */
DEV double wave_sum4(double a, double b, double c, double d)
{
    return row_sum(swap16_add(swap32_add(a, b), swap32_add(c, d)));
}

#endif
