/*
 * Test-only entry points of libnt_rocm.so. Not part of the ABI in
 * include/nablatensor_rocm.h: no caller of the engine needs them, and they
 * change nothing unless called.
 */
#ifndef NT_TESTING_H
#define NT_TESTING_H

#include <stdint.h>

struct nt_exec;

#ifdef __cplusplus
extern "C" {
#endif

/* Appends `text` to every program the calling thread compiles with hipRTC
 * from now on (null or "" stops it). A test appends source that cannot
 * compile to check that nt_exec_create and nt_compile_check return
 * NT_E_COMPILE with hipRTC's log in nt_last_error, as the reference reports a
 * hipRTC failure with its log (HipRuntime.java:351-354). The appended text is
 * part of the code-object cache key, so such a compile never hits the cache. */
void nt_testing_append_source(const char *text);

/* Dispatches of `exec` since its stream was last waited for: nt_exec_replay
 * returns from a small dispatch once the blocks' sums are in. */
int32_t nt_testing_undrained(const struct nt_exec *exec);

#ifdef __cplusplus
}
#endif
#endif
