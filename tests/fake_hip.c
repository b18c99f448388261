/* Host-side stand-in for the HIP calls that the engine's buffer pools make, for
 * tests without a GPU: loaded before libdgq_engine.so, its symbols come first.
 * Host memory is real, nothing runs on a device.  Launches of the copying kernel
 * of descriptor uploads (one workgroup of 1024 threads) are queued and run when
 * the test says so, as those of a busy stream would be; other launches are
 * dropped.  hipDeviceSynchronize returns when the queue is empty, as the real
 * one does when the device is idle. */
#include <pthread.h>
#include <stdint.h>
#include <stdlib.h>
#include <string.h>
#include <unistd.h>

typedef struct { uint32_t x, y, z; } dim3;
typedef struct { const void *src; void *dst; uint32_t n16, *read, ticket; } copy;

static pthread_mutex_t mu = PTHREAD_MUTEX_INITIALIZER;
static copy queue[1024];
static int head, tail, syncs, stream_syncs, pending, capturing;
static uint32_t flags[1024];
static int allocs;
static __thread dim3 cfg_grid, cfg_block;
static __thread size_t cfg_lds;
static __thread void *cfg_stream;

int fake_queued(void) {
    pthread_mutex_lock(&mu);
    const int n = tail - head;
    pthread_mutex_unlock(&mu);
    return n;
}
int fake_syncs(void) { return syncs; }
int fake_allocs(void) { return allocs; }
uint32_t fake_flags(int i) { return flags[i]; }
int fake_stream_syncs(void) { return stream_syncs; }
/* An error that an earlier call of the program left, reported by every hipGetLastError. */
void fake_pending(int e) { pending = e; }
/* Every stream is being captured (1) or none. */
void fake_capture(int on) { capturing = on; }
const void *fake_source(int i) { return queue[i].src; }

/* Runs up to n queued copies, oldest first. */
void fake_run(int n) {
    pthread_mutex_lock(&mu);
    for (; n > 0 && head < tail; n--, head++) {
        const copy *c = &queue[head];
        memcpy(c->dst, c->src, 16 * (size_t)c->n16);
        __atomic_store_n(c->read, c->ticket, __ATOMIC_RELEASE);
    }
    pthread_mutex_unlock(&mu);
}

int __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, void *stream) {
    cfg_grid = grid;
    cfg_block = block;
    cfg_lds = lds;
    cfg_stream = stream;
    return 0;
}
int __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *lds, void **stream) {
    *grid = cfg_grid;
    *block = cfg_block;
    *lds = cfg_lds;
    *stream = cfg_stream;
    return 0;
}
int hipLaunchKernel(const void *f, dim3 grid, dim3 block, void **args, size_t lds, void *stream) {
    (void)f, (void)lds, (void)stream;
    if (grid.x != 1 || block.x != 1024) return 0;
    pthread_mutex_lock(&mu);
    queue[tail].src = *(const void **)args[0];
    queue[tail].dst = *(void **)args[1];
    queue[tail].n16 = *(uint32_t *)args[2];
    queue[tail].read = *(uint32_t **)args[3];
    queue[tail].ticket = *(uint32_t *)args[4];
    tail++;
    pthread_mutex_unlock(&mu);
    return 0;
}

int hipHostMalloc(void **p, size_t bytes, uint32_t f) {
    *p = calloc(1, bytes);
    flags[allocs++] = f;
    return *p ? 0 : 2;
}
int hipHostFree(void *p) {
    free(p);
    return 0;
}
int hipEventCreateWithFlags(void **ev, uint32_t f) {
    (void)f;
    *ev = &queue;
    return 0;
}
int hipEventQuery(void *ev) { (void)ev; return 0; }
int hipEventRecord(void *ev, void *stream) { (void)ev, (void)stream; return 0; }
int hipEventSynchronize(void *ev) { (void)ev; return 0; }
int hipStreamSynchronize(void *stream) {
    (void)stream;
    stream_syncs++;
    return 0;
}
int hipStreamIsCapturing(void *stream, int *status) {
    (void)stream;
    *status = capturing;
    return 0;
}
int hipGetLastError(void) { return pending; }
int hipMemcpyAsync(void *dst, const void *src, size_t bytes, int kind, void *stream) {
    (void)kind, (void)stream;
    memcpy(dst, src, bytes);
    return 0;
}
int hipDeviceSynchronize(void) {
    __atomic_add_fetch(&syncs, 1, __ATOMIC_SEQ_CST);
    while (fake_queued()) usleep(1000);
    return 0;
}
