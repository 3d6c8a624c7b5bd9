/*
 * hb_pool.h -- device memory kept between plans.  A plan's workspace is tens
 * of buffers, gigabytes for the window's rings; a program that makes plans
 * in turn (a drop-in call, a gradient step on other data) allocated and
 * freed them each time.  Freed device memory has to be cleared before the
 * driver hands it out again, so past the first gigabytes an allocation
 * waits: two 2.4 GB plans a pass took 100 ms.
 *
 * Blocks that are given back wait here for the next request of about their
 * size: at most 1/32 of the device's memory and 4096 blocks in all, the
 * longest unused freed first; everything is freed when an allocation fails,
 * and by hbicg_trim().  The caller has waited for all work on a block before
 * it gives it back.  Safe from several threads.
 */
#ifndef HB_POOL_H
#define HB_POOL_H

#include <stddef.h>

#ifdef __cplusplus
extern "C" {
#endif

/* A block of at least `bytes` on the current device, NULL when there is none. */
void *hb_pool_get(size_t bytes);
/* Gives a block back (NULL: nothing). */
void hb_pool_put(void *p);
/* Bytes of the current device that wait here. */
size_t hb_pool_held(void);

#ifdef __cplusplus
}
#endif
#endif
