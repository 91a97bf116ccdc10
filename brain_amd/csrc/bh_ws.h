// The library-held workspaces of a stream (bh_api.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <mutex>

#include "bh_ws_grow.h"

namespace bh {

// What a workspace holds.
// split-K slabs, padded operands, packed MoE rows, int4 weights as int8
enum WsSlot { WS_SPLIT = 0, WS_PAD = 1, WS_MOE = 2, WS_EXPAND = 3, WS_SLOTS = 4 };

constexpr size_t SPLITK_MAX_BYTES = size_t(64) << 20;  // slabs of one call
constexpr size_t PAD_MAX_BYTES = size_t(512) << 20;    // padded operands of one call

// At least `ints` i32 of the stream's workspace `slot`, or null with *err
// (grown outside graph capture only; hipErrorStreamCaptureUnsupported
// otherwise).
int* splitk_workspace(hipStream_t s, size_t ints, hipError_t* err, int slot = WS_SPLIT);

// Holds a stream's workspaces for the launches of one call, from the one that
// writes to the last that reads. The same thread may nest it.
class WsLock {
public:
    hipError_t take(hipStream_t s);

private:
    std::unique_lock<std::recursive_mutex> lock_;
};

}  // namespace bh
