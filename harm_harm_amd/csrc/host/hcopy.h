/* hcopy.h -- large host copies by several threads. */
#ifndef HCOPY_H
#define HCOPY_H

#include <stddef.h>

#ifdef __cplusplus
extern "C" {
#endif

/* memcpy of n bytes (dst and src do not overlap). */
void hc_copy(void* dst, const void* src, size_t n);

#ifdef __cplusplus
}
#endif
#endif
