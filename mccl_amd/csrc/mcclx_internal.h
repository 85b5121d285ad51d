// mcclx_internal.h -- shared by the translation units of libmcclx.so only.
#pragma once

#include "mcclx.h"

// Records the calling thread's error message (what mcclx_last_error() returns)
// and hands back `code`.
extern "C" __attribute__((visibility("hidden"))) int mcclx_fail(int code, const char* fmt, ...)
    __attribute__((format(printf, 2, 3)));

// Is `p` pinned host memory?  (Link traffic, where everything else is the device's own.)
extern "C" __attribute__((visibility("hidden"))) bool mcclx_in_host_memory(mcclx_ctx* ctx, const void* p);

// Can the context launch mcclx_fold_encode with this plan and that many segments?
extern "C" __attribute__((visibility("hidden"))) bool mcclx_fold_encode_ok(mcclx_ctx* ctx, const mcclx_plan* plan, uint32_t nseg);

// One launch: the folds of `plan` (a fan-out sum over the wire codec) and the encodes (`enc`), each as
// mcclx_fold_batched takes them, in no order among each other.  Either may be none.
extern "C" __attribute__((visibility("hidden"))) int mcclx_fold_encode(
    mcclx_ctx* ctx, const mcclx_plan* plan, const mcclx_seg* folds, uint32_t nfold,
    const mcclx_plan* enc, const mcclx_seg* encodes, uint32_t nenc);
