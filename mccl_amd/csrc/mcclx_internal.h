// mcclx_internal.h -- shared by the translation units of libmcclx.so only.
#pragma once

#include <exception>
#include <new>

#include "mcclx.h"

// Records the calling thread's error message (what mcclx_last_error() returns)
// and hands back `code`.
extern "C" __attribute__((visibility("hidden"))) int mcclx_fail(int code, const char* fmt, ...)
    __attribute__((format(printf, 2, 3)));

// The body of a C entry that allocates: no exception leaves it.
template <class F>
int mcclx_entry(F&& body) {
    try {
        return body();
    } catch (const std::bad_alloc&) {
        return mcclx_fail(MCCLX_ERR_NOMEM, "out of host memory");
    } catch (const std::exception& e) {  // (a vector asked for more than it can ever hold)
        return mcclx_fail(MCCLX_ERR_STATE, "%s", e.what());
    }
}

// Is `p` pinned host memory?  (Link traffic, where everything else is the device's own.)
extern "C" __attribute__((visibility("hidden"))) bool mcclx_in_host_memory(mcclx_ctx* ctx, const void* p);

// Can the context launch mcclx_fold_encode with this plan and that many segments?
extern "C" __attribute__((visibility("hidden"))) bool mcclx_fold_encode_ok(mcclx_ctx* ctx, const mcclx_plan* plan, uint32_t nseg);

// One launch: the folds of `plan` (a fan-out sum over the wire codec) and the encodes (`enc`), each as
// mcclx_fold_batched takes them, in no order among each other.  Either may be none.
extern "C" __attribute__((visibility("hidden"))) int mcclx_fold_encode(
    mcclx_ctx* ctx, const mcclx_plan* plan, const mcclx_seg* folds, uint32_t nfold,
    const mcclx_plan* enc, const mcclx_seg* encodes, uint32_t nenc);
