// Internal interface of bh_flash.hip (causal prefill attention).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace bh {

// Where position `pos` of sequence `seq` lives in a layer's cache: the token
// slot whose K (V) row is [slot][hkv] and whose KV8 scales are [slot][nkv].
// Contiguous slabs (bs == 0): slot = seq * max_seq + pos. Paged pool
// (crates/qwen3/src/serve.rs:349-356, the layout of
// paged_kv_append_i8_clipped_batched.wgsl:46-77): slot = block * bs + pos % bs
// with block = bt[seq * max_bt + pos / bs]; bs is a multiple of the attention
// chunk, so a chunk of keys lies inside one block. A table entry outside the
// pool (an unallocated block) maps to block 0: only chunks past a row's
// position read it (their reads are issued before the position is known and
// never used), and the host refuses to run a row whose used blocks are not
// allocated.
struct KvMap {
    const uint32_t* bt;  // [max_batch][max_bt] physical blocks (paged)
    int max_bt, bs, nblk, max_seq;
    __device__ __forceinline__ size_t slot(size_t seq, int pos) const {
        if (bs == 0) return seq * max_seq + pos;
        const uint32_t blk = bt[seq * max_bt + pos / bs];
        return (size_t)(blk < (uint32_t)nblk ? blk : 0u) * bs + pos % bs;
    }
};

struct FlashArgs {
    float* q;          // [rows, hq] rotated queries; the context rows replace them
    const void* kc;    // this layer's caches [slot][hkv] (f32, or int8 codes with kv8)
    const void* vc;
    const float* ks;   // kv8: scales [slot][nkv]
    const float* vs;
    const uint32_t* pos;  // per row; consecutive within a sequence's run of rows
    const uint32_t* seq;  // per row
    int nh, nkv, hq, hkv;
    int rows_per_seq, nseq;
    float scale;
    KvMap map;
};

constexpr int FLASH_MAX_GROUP = 8;       // query heads per kv head
constexpr int FLASH_MAX_SEQ = 65536;     // positions of one sequence

// Whether launch_flash_prefill is built for this geometry.
inline bool flash_ok(int hd, int nh, int nkv, int max_seq) {
    return (hd == 64 || hd == 128) && nh / nkv <= FLASH_MAX_GROUP && max_seq <= FLASH_MAX_SEQ;
}
hipError_t launch_flash_prefill(hipStream_t s, const FlashArgs& a, int hd, bool kv8);

}  // namespace bh
