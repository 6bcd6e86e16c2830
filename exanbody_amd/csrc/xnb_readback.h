// xnb_readback.h -- the caller's host memory to and from device arrays (xnb_readback.hip).
#pragma once

#include "xnb_ctx.h"

namespace xnb_impl {

// every context, from xnb_create to xnb_destroy: the pinned blocks live as long as any
void readback_context_created();
void readback_context_destroyed();

// Particles in cell order (ghost cells too), any pointer may be null.  Returns when the
// caller's arrays hold them.
int read_particles(xnb_ctx* c, bool ghosts, uint32_t* cell, double* r, double* v, double* f, double* ep, uint64_t* id, uint8_t* type);

// bytes of device memory into host memory, after the work queued on the context's stream
int read_bytes(xnb_ctx* c, const void* src, size_t bytes, void* dst);

// n particles into slots 0 .. n - 1 of buffer A: slot t takes the caller's particle order[t]
// (cells cell[order[t]]), its position wrapped into the periodic domain; v, id, type may be
// null (0, the particle's index, 0).  Returns when the caller's arrays have been read.
int write_particles(xnb_ctx* c, size_t n, const uint32_t* order, const uint32_t* cell, const double* r, const double* v,
                    const uint64_t* id, const uint8_t* type);

}  // namespace xnb_impl
