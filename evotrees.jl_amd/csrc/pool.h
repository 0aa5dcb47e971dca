// Memory and streams that outlive the handle or call that used them.  A fit takes some forty device buffers, a pinned one and a stream: taken
// from here they cost a lock each instead of 5 to 100 us each.  Bounded (POOL_DEVICE_KEPT / POOL_PINNED_KEPT bytes of a kind stay behind at most,
// none in blocks above POOL_BLOCK_KEPT), given back by evt_trim and when an allocation fails; any thread.  A buffer is given
// only when nothing on the device uses it any more (the giver has waited for its stream).
#pragma once
#include "evt_internal.h"

static const size_t POOL_DEVICE_KEPT = (size_t)1 << 30; // of 288 GB, per device
static const size_t POOL_PINNED_KEPT = (size_t)64 << 20;
static const size_t POOL_BLOCK_KEPT = (size_t)256 << 20;

void *dev_take(size_t bytes); // on the current device; nullptr: the error is set
void dev_give(void *p);
void *pinned_take(size_t bytes); // portable, at the same address on host and device; nullptr: the error is set
void pinned_give(void *p);
// pinned memory that the host reads while the kernel that writes it still runs: asked for as coherent, which the runtime otherwise leaves to HIP_HOST_COHERENT
void *coherent_take(size_t bytes);
void coherent_give(void *p);
hipError_t stream_take(hipStream_t *s, bool non_blocking); // on the current device
void stream_give(hipStream_t s, bool non_blocking, int device); // idle; a stream of that device

void models_trim(); // what models keep between their calls, but for those in one (model.hip)
