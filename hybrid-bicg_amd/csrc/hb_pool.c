/* hb_pool.c -- device memory kept between plans (hb_pool.h). */
#include <hip/hip_runtime_api.h>
#include <pthread.h>
#include <stdint.h>
#include <stdlib.h>

#include "hb_pool.h"
#include "../../include/hbicg.h"

#define POOL_BLOCKS 4096          /* most waiting blocks                  */
#define POOL_HASH   1024

/* Every block, in use or waiting, is in the table by its address; the
 * waiting ones also in a list, the longest waiting first, and in one of
 * their size, the last given back first. */
struct block {
    void *p;
    size_t bytes;
    int device;
    struct block *next_hash, *prev, *next, *prev_size, *next_size;
};

static pthread_mutex_t lock = PTHREAD_MUTEX_INITIALIZER;
static struct block *table[POOL_HASH], *by_size[POOL_HASH], *oldest, *newest;
static size_t held;
static int count;

static unsigned size_slot(size_t bytes) { return (unsigned)(((bytes >> 8) * 0x9E3779B97F4A7C15ull) >> 54) % POOL_HASH; }
static unsigned slot_of(const void *p) { return (unsigned)(((uintptr_t)p >> 8) * 0x9E3779B1u >> 22) % POOL_HASH; }

/* Sizes in steps of an eighth of their power of two (at least 256 bytes): a
 * block serves requests up to an eighth smaller, so at most that is unused. */
static size_t rounded(size_t bytes)
{
    size_t step = 256;
    while (step * 16 <= bytes) step *= 2;
    return (bytes + step - 1) / step * step;
}

static void unlink_waiting(struct block *b)
{
    if (b->prev) b->prev->next = b->next;
    else oldest = b->next;
    if (b->next) b->next->prev = b->prev;
    else newest = b->prev;
    if (b->prev_size) b->prev_size->next_size = b->next_size;
    else by_size[size_slot(b->bytes)] = b->next_size;
    if (b->next_size) b->next_size->prev_size = b->prev_size;
    b->prev = b->next = b->prev_size = b->next_size = NULL;
    held -= b->bytes;
    --count;
}

/* frees a waiting block (its device's context is that of the address) */
static void drop(struct block *b)
{
    struct block **at = &table[slot_of(b->p)];
    while (*at != b) at = &(*at)->next_hash;
    *at = b->next_hash;
    unlink_waiting(b);
    (void)hipFree(b->p);
    free(b);
}

void *hb_pool_get(size_t bytes)
{
    int dev = 0;
    void *p = NULL;
    const size_t want = rounded(bytes ? bytes : 1);
    if (hipGetDevice(&dev) != hipSuccess) return NULL;
    pthread_mutex_lock(&lock);
    for (struct block *b = by_size[size_slot(want)]; b; b = b->next_size)
        if (b->bytes == want && b->device == dev) {
            unlink_waiting(b);
            p = b->p;
            break;
        }
    if (!p) {
        struct block *b = (struct block *)calloc(1, sizeof *b);
        hipError_t e = b ? hipMalloc(&p, want) : hipErrorOutOfMemory;
        if (b && e != hipSuccess && oldest) {
            (void)hipGetLastError();
            while (oldest) drop(oldest);
            e = hipMalloc(&p, want);
        }
        if (e == hipSuccess) {
            b->p = p;
            b->bytes = want;
            b->device = dev;
            b->next_hash = table[slot_of(p)];
            table[slot_of(p)] = b;
        } else {
            p = NULL;
            free(b);
        }
    }
    pthread_mutex_unlock(&lock);
    return p;
}

void hb_pool_put(void *p)
{
    if (!p) return;
    pthread_mutex_lock(&lock);
    struct block *b = table[slot_of(p)];
    while (b && b->p != p) b = b->next_hash;
    if (b) {
        static size_t total;   /* the device's memory, asked for once */
        size_t free_b = 0;
        if (!total && hipMemGetInfo(&free_b, &total) != hipSuccess) total = 0;
        struct block **const size = &by_size[size_slot(b->bytes)];
        b->next_size = *size;
        if (*size) (*size)->prev_size = b;
        *size = b;
        b->prev = newest;
        if (newest) newest->next = b;
        else oldest = b;
        newest = b;
        held += b->bytes;
        ++count;
        while (oldest && (held > total / 32 || count > POOL_BLOCKS)) drop(oldest);
    }
    pthread_mutex_unlock(&lock);
}

size_t hb_pool_held(void)
{
    int dev = 0;
    size_t sum = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 0;
    pthread_mutex_lock(&lock);
    for (const struct block *b = oldest; b; b = b->next)
        if (b->device == dev) sum += b->bytes;
    pthread_mutex_unlock(&lock);
    return sum;
}

void hbicg_trim(void)
{
    pthread_mutex_lock(&lock);
    while (oldest) drop(oldest);
    pthread_mutex_unlock(&lock);
}
