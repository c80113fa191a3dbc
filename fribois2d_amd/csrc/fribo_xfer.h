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

// Events of one handle's transfers, one per chunk in flight.
struct XferEvents {
    static constexpr int SLOTS = 3;
    hipEvent_t ev[SLOTS] = {nullptr, nullptr, nullptr};
};

// Moves every segment (put: host to device, else device to host) on stream
// st of device dev and returns when it is complete on both sides.
hipError_t xfer_run(XferEvents& R, int dev, const FluidDev& F, XferSeg* segs, int nseg, bool put, hipStream_t st);
void xfer_free(XferEvents& R);

// The pinned staging memory belongs to the library: a transfer takes a block
// for as long as it runs.  Handles attach while they live; the last one to
// detach gives the memory back.
void xfer_attach();
void xfer_detach();
