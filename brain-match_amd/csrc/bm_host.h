/*
 * Host-side graph layout shared by the C ABI implementation, the CSV/synthetic
 * front ends and the search drivers.  Not part of the public ABI.
 *
 * Layout (identical on host and device):
 *   - male out-lists (CSR) and in-lists (CSC): ptr[n+2] int64 row offsets for
 *     rows 0..n (row 0 is always empty) and adj[m] of {neighbour, weight}
 *     int32 pairs, neighbours ascending within a row;
 *   - female out-rows and in-rows: the same CSR/CSC.
 * The hash table of every row that replaces the reference's dense (n+1)^2
 * int16 female matrix (src/graph-re-alignment-gpu-swap.cu:396-418) is built on
 * the device from these lists (bm_rowtab.h).
 */
#ifndef BM_HOST_H
#define BM_HOST_H

#include <stdint.h>
#include <stddef.h>
#include "../../include/brainmatch.h"

#ifdef __cplusplus
extern "C" {
#endif

typedef struct bm_pair32 { int32_t x; int32_t y; } bm_pair32;  /* {neighbour|key, weight} */

typedef struct bm_csr_host {
    int32_t n;
    int64_t m;
    int64_t* ptr;      /* n+2 */
    bm_pair32* adj;    /* m */
} bm_csr_host;

typedef struct bm_graph_host {
    int32_t n;
    int64_t m;
    bm_csr_host out;   /* CSR by source */
    bm_csr_host in;    /* CSC by destination (neighbour = source) */
} bm_graph_host;

/* Sets *err to a static message on failure and returns a BM_ERR_* code. */
int bm_graph_build(int32_t n, const bm_edges* e, bm_graph_host* g, const char** err);
void bm_graph_free(bm_graph_host* g);

/* Thread-local error string for calls without a context. */
void bm_set_global_error(const char* fmt, ...);

/* Host copy of the context's male graph (read-only). */
const bm_graph_host* bm_ctx_male(const bm_ctx* ctx);
/* Sets the context error message (for host drivers). */
int bm_ctx_fail(bm_ctx* ctx, int code, const char* msg);

#ifdef __cplusplus
}
#endif

#endif
