/**
 * host_copy.h - Results from the device into a caller's ordinary memory,
 * through page-locked chunks that a model keeps.
 */
#ifndef VITNA_HOST_COPY_H
#define VITNA_HOST_COPY_H

#include <hip/hip_runtime.h>
#include <stddef.h>

struct host_copy;

/* null when there is no page-locked memory or event for it: host_copy_rows then copies a row at a time */
host_copy* host_copy_create();
void host_copy_destroy(host_copy* c);

/* n rows of `bytes` each, one after another at dev, to dst[0..n), a null dst's row left out; when the stream's earlier
   work is done, and returns with every byte in place (and so the stream's earlier work done, if any row is asked).
   Rows in memory that HIP allocated are copied there by the device. One call at a time. */
hipError_t host_copy_rows(host_copy* c, hipStream_t s, const void* dev, size_t bytes, size_t n, void* const* dst);

#endif
