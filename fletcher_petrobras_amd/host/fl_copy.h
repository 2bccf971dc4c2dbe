/* Host memory copy over all OpenMP threads, for the staging of host transfers. */
#ifndef FLETCHER_FL_COPY_H
#define FLETCHER_FL_COPY_H

#include <stddef.h>

#ifdef __cplusplus
extern "C" {
#endif

void fl_copy_parallel(void *dst, const void *src, size_t bytes);

#ifdef __cplusplus
}
#endif
#endif
