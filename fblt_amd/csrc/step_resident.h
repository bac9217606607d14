/* Launch interface of the resident decoder step (step_resident.hip). */
#ifndef FBLT_AMD_STEP_RESIDENT_H
#define FBLT_AMD_STEP_RESIDENT_H

#include "blt_hip.h"

struct StepResident {
    const blt_kv_cache *cache;
    size_t batch, n;         /* sequences, new rows of each */
    const size_t *base;      /* [batch] cached lengths */
    const size_t *latent;    /* [batch * n] latent patch of every row */
    const float *d0_rows;    /* input rows, [batch * n, E], or the table row_index points into */
    const uint32_t *row_index; /* one sequence: input row of every new row; NULL: row r itself */
    const size_t *positions; /* one sequence: rotary positions; NULL: base + r */
    const bool *crosses;     /* [num_layers] */
    float *logits;
    size_t window;
    bool block_kind;
};

/* Issues the whole step as one launch; false: not a shape it takes, nothing was issued. */
bool kv_step_resident(const StepResident &st);
/* Ends the process with a message if a resident launch ever gave up waiting. */
void kv_step_resident_check();

#endif
