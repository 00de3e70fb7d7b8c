// rf_gnlds.h -- the gate-net engine's LDS kernel (rf_gnlds.hip), which runs
// the wavefront programs of rf_gnplan.h.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define RF_GNL_THREADS 1024u
// LDS of a workgroup (gfx950: 160 KB per CU)
#define RF_GNL_LDS (160u * 1024u - 64u)

struct rf_gnl_params {
    const uint32_t* words;    // the plan's tables
    const uint2* rows;        // its rows, by lines
    uint32_t batch;           // wavefront rows of its batches
    uint32_t off_po, off_ram, ram_words;
    uint32_t n_pi, n_po, n_ram, n_rams, depth, width, abits;
    uint32_t a0, b0;          // LDS byte addresses of input sets A and B
    uint32_t state_bytes;     // the planes kept between launches, a multiple of 4
    uint32_t lds_bytes;
    uint32_t nlanes;          // lanes, sorted by budget (longest first)
    uint32_t k0, k1;          // iterations of this launch: iteration k hashes cycle k - 1
    uint64_t seed;
    uint64_t* M;              // RAM rows [lane][RAM][element]
    uint64_t* hash;           // per lane
    const uint32_t* budget;   // per lane
    const uint32_t* sid;      // stimulus of each lane
    uint32_t* image;          // state planes of every workgroup between launches (k0 > 0 or more to come)
};

// Launches iterations [k0, k1) for ``groups`` workgroups of 8 * pb lanes each
// (plane width pb bytes: 1, 2 or 4).
hipError_t rf_gnl_launch(const rf_gnl_params& p, uint32_t pb, uint32_t groups, hipStream_t stream);
