// Copies between the caller's (pageable) arrays and the device (transfer.hip).
#pragma once
#include "vpmx_internal.h"

namespace vpmx {

struct Copy {
    void *dst;
    const void *src;
    size_t bytes;
};
// Host to device: the sources may change when it returns; ordered before later work on the
// context's stream.  Device to host: after earlier work on the stream, complete at return.
int copy_in(Ctx *c, const Copy *q, int n);
int copy_out(Ctx *c, const Copy *q, int n);
void free_transfer(Ctx *c);

}  // namespace vpmx
