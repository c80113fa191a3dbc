// State transfer between the pitched device fields and the caller's arrays
// (fribo_xfer.hip).
#pragma once
#include "fribo_internal.h"

#define XFER_MAXSEG 11

// One array of a transfer: `rows` rows of `n` doubles, pitch `pitch` on the
// device, contiguous on the host.  pressure: rows are pressure planes from
// plane k0 on, and a read-back subtracts the pending means (S->pend from the
// interior, S->goff from row n2 and the ghost planes).
struct XferSeg {
    double* dev;
    double* host;
    int n, pitch, rows, k0, pressure;
};

// Staging ring of one handle: pinned chunks and the events of their kernels.
struct XferRing {
    static constexpr int SLOTS = 3;
    double* stage = nullptr;     // SLOTS chunks of `chunk` doubles
    size_t chunk = 0;
    hipEvent_t ev[SLOTS] = {nullptr, nullptr, nullptr};
};

// Moves every segment (put: host to device, else device to host) on stream
// st and returns when the host side is complete; a put may leave its last
// kernels running (they read the ring, which the next transfer waits for).
hipError_t xfer_run(XferRing& R, const FluidDev& F, XferSeg* segs, int nseg, bool put, hipStream_t st);
void xfer_free(XferRing& R);
