// The int8 paged KV cache kernels of brain's int8 serving path, as Backend
// step names and typed calls:
//   paged_kv_append_i8_clipped_batched  crates/kernels/wgsl/paged_kv_append_i8_clipped_batched.wgsl:46-77
//   paged_decode_scores_i8_batched      crates/kernels/wgsl/paged_decode_scores_i8_batched.wgsl:28-54
//   paged_decode_apply_i8_batched       crates/kernels/wgsl/paged_decode_apply_i8_batched.wgsl:28-53
// The pool holds int8 codes (4 per u32 word, little-endian) at slot
// physical*block_size + offset, kv_stride bytes per slot; one f32 scale per
// (slot, kv head).
//
// Each output keeps the reference's own summation order (a score sums its
// head_dim products in order, a context element its positions in order), so
// the f32 results are the reference's bit for bit; the parallelism is across
// outputs. Block tables, offsets and sequence lengths are read on the device,
// so the slots they name are checked there against the pool and scale
// lengths the caller passes: an entry outside them is skipped (nothing
// stored, nothing added) instead of the reference's out-of-bounds access.
#include "bh_common.h"
#include "bh_kv8.h"

namespace bh {

// One wave per (sequence, kv head); lane l owns word l of the head (head_dim
// <= 256). The head's absmax is exact in any order.
__global__ __launch_bounds__(64) void paged_kv_append_i8_kernel(const float* src, const uint32_t* blocks,
                                                                const uint32_t* offsets, const float* clip,
                                                                uint32_t* pool, uint64_t pool_words, float* scales,
                                                                uint64_t n_scales, uint32_t kv_stride, uint32_t bs,
                                                                uint32_t hd) {
    const uint32_t n_kv = kv_stride / hd;
    const uint32_t b = blockIdx.x / n_kv, head = blockIdx.x % n_kv;
    const uint32_t lane = threadIdx.x;
    const bool live = 4 * lane < hd;
    const float* x = src + (uint64_t)b * kv_stride + (uint64_t)head * hd + 4 * lane;
    float v[4] = {0.f, 0.f, 0.f, 0.f};
    float mx = 0.0f;
    if (live) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            v[j] = x[j];
            mx = fmaxf(mx, fabsf(v[j]));
        }
    }
    mx = xor_max<32>(mx);
    float scale = fminf(mx, clip[head]) / 127.0f;
    if (scale == 0.0f) scale = 1.0f;
    const uint64_t slot = (uint64_t)blocks[b] * bs + offsets[b];
    const uint64_t base = slot * kv_stride + (uint64_t)head * hd;  // a multiple of 4
    if (slot * n_kv + head >= n_scales || (base + hd) / 4 > pool_words) return;
    if (lane == 0) scales[slot * n_kv + head] = scale;
    if (live) {
        uint32_t w = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) w |= (uint32_t)kv8_code(v[j], scale) << (8 * j);
        pool[base / 4 + lane] = w;
    }
}

__device__ __forceinline__ float code_f(uint32_t w, int e) { return (float)(int8_t)(uint8_t)(w >> (8 * e)); }


// Slot of position j of sequence b, or false when the tables name one
// outside the pool.
__device__ __forceinline__ bool slot_of(const PagedReadArgs& a, uint32_t b, uint32_t j, uint32_t kvh, uint64_t& slot) {
    const uint32_t blk = j / a.bs;
    if (blk >= a.max_bt) return false;
    slot = (uint64_t)a.bt[(uint64_t)b * a.max_bt + blk] * a.bs + j % a.bs;
    const uint32_t n_kv = a.kv_stride / a.hd;
    return slot * n_kv + kvh < a.n_scales && (slot * a.kv_stride + (uint64_t)kvh * a.hd + a.hd + 3) / 4 <= a.pool_words;
}

// Scores, any geometry: one thread per (b, h, j), q . f32(codes) in head_dim
// order, then (acc * kscale) * scale. A workgroup takes 64 consecutive
// positions of one (b, h). Positions at or past the sequence length are not
// written.
template <bool VEC>
__global__ __launch_bounds__(64) void paged_decode_scores_i8_kernel(PagedReadArgs a) {
    const uint32_t nchunk = (a.cap + 63) / 64;
    const uint32_t bh = blockIdx.x / nchunk;
    const uint32_t j = (blockIdx.x % nchunk) * 64 + threadIdx.x;
    const uint32_t b = bh / a.n_heads, h = bh % a.n_heads;
    if (j >= a.cap || j >= a.seq_lens[b]) return;
    const uint32_t kvh = h / a.group;
    uint64_t slot;
    if (!slot_of(a, b, j, kvh, slot)) return;
    const float qscale = a.scales[slot * (a.kv_stride / a.hd) + kvh];
    const uint64_t base = slot * a.kv_stride + (uint64_t)kvh * a.hd;
    const float* q = a.in + (uint64_t)bh * a.hd;
    float acc = 0.0f;
    if constexpr (VEC) {  // base and hd multiples of 16 bytes, pool 16-byte aligned
        const uint4* p = reinterpret_cast<const uint4*>(a.pool) + base / 16;
        for (uint32_t d = 0; d < a.hd; d += 16) {
            const uint4 w = p[d / 16];
            const uint32_t ws[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) acc = acc + q[d + 4 * i + e] * code_f(ws[i], e);
        }
    } else {
        for (uint32_t d = 0; d < a.hd; d += 4) {
            const uint32_t w = a.pool[(base + d) / 4];
#pragma unroll
            for (int e = 0; e < 4; ++e) acc = acc + q[d + e] * code_f(w, e);
        }
    }
    a.out[(uint64_t)bh * a.cap + j] = acc * qscale * a.scale;
}

// Scores for head_dim 64 and 128 with 16-byte key rows: one thread per
// (b, set of a kv head's query heads, j). The latency of the slot lookup and of
// the key row bounds it, so the row's HD / 16 loads all go out together and the
// set's heads share them. Two heads run at once so that two of the ordered
// chains are in flight. q is uniform over the workgroup and comes through scalar
// loads. How many heads a set holds: score_sets.
template <int HD>
__global__ __launch_bounds__(64) void paged_decode_scores_i8_group_kernel(PagedReadArgs a, uint32_t nkvu, uint32_t sets,
                                                                          uint32_t heads,
                                                                          const float* __restrict__ qall,
                                                                          float* __restrict__ out) {
    const uint32_t nchunk = (a.cap + 63) / 64;
    const uint32_t bs = blockIdx.x / nchunk, set = bs % sets, bk = bs / sets;
    const uint32_t b = bk / nkvu, kvh = bk % nkvu;
    const uint32_t j = (blockIdx.x % nchunk) * 64 + threadIdx.x;
    const uint32_t h0 = kvh * a.group;  // below n_heads
    const uint32_t h1 = h0 + min(min(a.group, a.n_heads - h0), (set + 1) * heads);
    if (h0 + set * heads >= h1 || j >= a.cap || j >= a.seq_lens[b]) return;
    uint64_t slot;
    if (!slot_of(a, b, j, kvh, slot)) return;
    const uint4* p = reinterpret_cast<const uint4*>(a.pool) + (slot * a.kv_stride + (uint64_t)kvh * HD) / 16;
    uint4 w[HD / 16];
#pragma unroll
    for (int i = 0; i < HD / 16; ++i) w[i] = p[i];
    const float qscale = a.scales[slot * (a.kv_stride / HD) + kvh];
    for (uint32_t h = h0 + set * heads; h < h1; h += 2) {
        const bool two = h + 1 < h1;
        const float* q0 = qall + ((uint64_t)b * a.n_heads + h) * HD;
        const float* q1 = two ? q0 + HD : q0;
        float acc0 = 0.0f, acc1 = 0.0f;
#pragma unroll
        for (int i = 0; i < HD / 16; ++i) {
            const uint32_t ws[4] = {w[i].x, w[i].y, w[i].z, w[i].w};
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const float c = code_f(ws[e >> 2], e & 3);
                acc0 = acc0 + q0[16 * i + e] * c;
                acc1 = acc1 + q1[16 * i + e] * c;
            }
        }
        float* o = out + ((uint64_t)b * a.n_heads + h) * a.cap + j;
        o[0] = acc0 * qscale * a.scale;
        if (two) o[a.cap] = acc1 * qscale * a.scale;
    }
}

// How many sets the query heads of a kv head are split into. A set of the whole
// group reads each key row once, but its heads run one pair after another: worth
// it while the workgroups fill the chip, 2048 of one wave (8 per CU). Scores of 8
// sequences of 1024-2048 tokens, heads of 128, us (whole group / pairs of heads /
// one thread per head): 16 heads over 8 kv heads 6.6 / 6.8 / 10.5; 32 over 8 (2048
// workgroups) 8.4 / 9.7 / 18.0; 64 over 8 12.3 / 15.4 / 32.5; 32 over 2 (512)
// 17.3 / 9.6 / 15.0; 32 over 1 (256) 28.8 / 9.8 / 11.0, one sequence 28.5 / 4.7 / 4.3.
uint32_t score_sets(uint64_t blocks, uint32_t group) {
    const uint64_t pairs = (group - 1) / 2 + 1;
    return (uint32_t)std::min<uint64_t>(pairs, std::max<uint64_t>(1, 2048 / blocks));
}

template <int HD>
void go_scores_group(hipStream_t s, const PagedReadArgs& a, uint32_t batch) {
    const uint32_t nchunk = (a.cap + 63) / 64, nkvu = (a.n_heads - 1) / a.group + 1;  // kv heads that have queries
    const uint32_t group = std::min(a.group, a.n_heads);
    const uint64_t blocks = (uint64_t)batch * nkvu * nchunk;
    const uint32_t want = score_sets(blocks, group);
    const uint32_t heads = ((group + want - 1) / want + 1) / 2 * 2, sets = (group + heads - 1) / heads;
    paged_decode_scores_i8_group_kernel<HD><<<(unsigned)(blocks * sets), 64, 0, s>>>(a, nkvu, sets, heads, a.in, a.out);
}

// Context: per (b, h, d) the sum over positions j, in order, of
// (p_j * f32(code)) * vscale. The order makes one chain of additions per
// output; everything else is kept off that chain. A workgroup takes 64 consecutive d of one (b, h): eight waves load
// codes, probabilities and scales APF chunks of 128 positions ahead and write
// a chunk's products to LDS while a ninth wave, one lane per d, adds up the
// chunk before it, four positions per LDS read. The block table of the
// sequence is staged in LDS first, so that no load waits for another.
// 8 sequences of 1024-2048 tokens, 16 heads of 128: 19.6 us (before: one
// thread per (b, h, d) with the loads of 8 positions ahead of their adds,
// 884 us, bound by three dependent memory round trips per 8 positions). What
// bounds it now is the instruction issue of the product waves, about 1 us per
// chunk; four waves of twice the width measured 22.1 us, 4 to 6 chunks in
// flight 24-25 us.
//
// Positions whose table entry lies outside the pool add +0, which leaves the
// sum as it is (it starts at +0 and so is never -0).
constexpr int APC = 128;                 // positions per chunk
constexpr int APW = 8;                   // product waves
constexpr int APT = (APW + 1) * 64;      // threads
constexpr int APF = 3;                   // chunks of loads in flight
constexpr uint32_t AP_TBL = 2048;        // table entries staged at a time

struct ApplyIn {
    uint32_t code[4];
    float p[4], s[4];
    uint32_t ok;  // bit u: position u is one to add
};

// B4 (block_size % 4 == 0): the four positions of a product lane share one
// table lookup. T: the type of pool and scale offsets; 32 bits where the pool
// and the scales are smaller than 4 GiB, which halves the address arithmetic
// that the product waves spend most of their time on (23.4 -> 19.6 us).
struct ApplyGeom {
    // The slots that kv head h may read are those below min(pool_slots +
    // (pool_rest >= (h + 1) * hd), scale_slots + (h < scale_rest)).
    uint64_t pool_slots, scale_slots;
    uint32_t pool_rest, scale_rest;
    int bs_shift;  // log2(block_size), or -1
};

template <bool B4, typename T>
__global__ __launch_bounds__(APT) void paged_decode_apply_i8_kernel(PagedReadArgs a, ApplyGeom geo) {
    __shared__ __attribute__((aligned(16))) float prod[2][APC * 64];
    __shared__ uint32_t tbl[AP_TBL];
    const uint32_t nchunk = (a.hd + 63) / 64;
    const uint32_t bh = blockIdx.x / nchunk;
    const uint32_t d0 = (blockIdx.x % nchunk) * 64;
    const uint32_t b = bh / a.n_heads, h = bh % a.n_heads;
    const uint32_t kvh = h / a.group, n_kv = a.kv_stride / a.hd;
    const float* pr = a.in + (uint64_t)bh * a.cap;
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    // Product lane: 4 positions (group jg of the chunk) x 4 consecutive d.
    const uint32_t jg = wave * 4 + (lane >> 4), dl = 4 * (lane & 15);
    const uint32_t dofs = kvh * a.hd + (d0 + dl < a.hd ? d0 + dl : 0);  // hd % 4 == 0
    const uint64_t lim64 = min(geo.pool_slots + (geo.pool_rest >= (kvh + 1) * a.hd ? 1 : 0),
                               geo.scale_slots + (kvh < geo.scale_rest ? 1 : 0));
    const T lim = (T)lim64;
    // Without a slot to read there is none for the masked loads either.
    const uint32_t t = lim64 ? min(a.seq_lens[b], a.cap) : 0u;
    const uint32_t none = (uint32_t)min((lim64 + a.bs - 1) / a.bs, (uint64_t)0xffffffffu);  // the first block with no slot to read
    // LDS slot of (position group g, d): 16 bytes at (g * 64 + (d % 4) * 16 +
    // d / 4) * 16, so the 16 lanes that store one d offset write 16
    // consecutive slots, and so do the lanes that read one group.
    float acc = 0.0f;
    const uint32_t per_seg = AP_TBL <= 0xffffffffu / a.bs ? AP_TBL * a.bs : 0xffffffffu;  // positions per staged table
    for (uint32_t j_seg = 0; j_seg < t;) {
        const uint32_t j_end = t - j_seg > per_seg ? j_seg + per_seg : t;
        const uint32_t blk0 = j_seg / a.bs;
        const uint32_t nblk = (j_end - j_seg - 1) / a.bs + 1;  // (a block size near 2^32 added to the length would wrap)
        __syncthreads();
        for (uint32_t i = threadIdx.x; i < nblk; i += APT)
            tbl[i] = blk0 + i < a.max_bt ? min(a.bt[(uint64_t)b * a.max_bt + blk0 + i], none) : none;
        __syncthreads();
        const uint32_t nch = (j_end - j_seg - 1) / APC + 1;
        // Every load is unconditional, at an address inside the buffers (a
        // load under a branch would be waited for at the join). B4: the four
        // positions lie in one block, so one lookup serves them.
        auto load = [&](uint32_t c, ApplyIn& in) {
            const uint32_t j0 = j_seg + min(c, nch - 1) * APC + 4 * jg;
            const uint32_t live = c < nch ? j_end : 0u;
            uint32_t ok = 0u;
            T slot = 0;
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const uint32_t j = min(j0 + u, j_end - 1);
                if (!B4 || u == 0) {
                    const uint32_t blk = geo.bs_shift >= 0 ? j >> geo.bs_shift : j / a.bs;
                    slot = (T)tbl[blk - blk0] * a.bs + (j - blk * a.bs);
                }
                // (The positions of a B4 lane past the sequence's end may leave
                // the block: they are not added.)
                const T su = B4 ? slot + u : slot;
                const bool in_pool = su < lim;
                ok |= ((uint32_t)in_pool & (uint32_t)(j0 + u < live)) << u;
                const T sl = in_pool ? su : 0;
                in.p[u] = pr[j];
                in.s[u] = a.scales[sl * n_kv + kvh];
                in.code[u] = a.pool[(sl * a.kv_stride + dofs) / 4];
            }
            in.ok = ok;
        };
        auto put = [&](uint32_t c, const ApplyIn& in) {
            float* dst = prod[c & 1] + jg * 256 + (lane & 15) * 4;
            float p[4], s[4];
            uint32_t w[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const bool ok = (in.ok >> u) & 1u;
                p[u] = ok ? in.p[u] : 0.0f;
                s[u] = ok ? in.s[u] : 0.0f;
                w[u] = ok ? in.code[u] : 0u;
            }
#pragma unroll
            for (int e = 0; e < 4; ++e)
                *reinterpret_cast<float4*>(dst + e * 64) =
                    make_float4(p[0] * code_f(w[0], e) * s[0], p[1] * code_f(w[1], e) * s[1],
                                p[2] * code_f(w[2], e) * s[2], p[3] * code_f(w[3], e) * s[3]);
        };
        // Chunk c's products are written in step c and added in step c + 1;
        // the barrier that ends a step orders both (LDS only: the loads in
        // flight are not waited for).
        auto barrier = [&]() {
            __builtin_amdgcn_sched_barrier(0);  // no use of a later chunk's loads moves up
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
        };
        auto add = [&](uint32_t c) {
            const float4* src = reinterpret_cast<const float4*>(prod[c & 1]) + lane;
            const int ng = (int)(min((uint32_t)APC, j_end - j_seg - c * APC) + 3) / 4;
            if (ng == APC / 4) {
#pragma unroll 8
                for (int g = 0; g < APC / 4; ++g) {
                    const float4 v = src[g * 64];
                    acc = acc + v.x;
                    acc = acc + v.y;
                    acc = acc + v.z;
                    acc = acc + v.w;
                }
            } else {
                for (int g = 0; g < ng; ++g) {
                    const float4 v = src[g * 64];
                    acc = acc + v.x;
                    acc = acc + v.y;
                    acc = acc + v.z;
                    acc = acc + v.w;
                }
            }
        };
        const uint32_t steps = (nch + APF) / APF * APF;  // nch + 1, rounded up: the same count in every wave
        if (wave < APW) {
            ApplyIn in[APF];
#pragma unroll
            for (int f = 0; f < APF; ++f) {
                load(f, in[f]);
                __builtin_amdgcn_sched_barrier(0);  // in chunk order, as vmcnt counts
            }
            for (uint32_t c = 0; c < steps; c += APF) {
#pragma unroll
                for (int f = 0; f < APF; ++f) {
                    put(c + f, in[f]);
                    load(c + f + APF, in[f]);
                    barrier();
                }
            }
        } else {
            for (uint32_t c = 0; c < steps; ++c) {
                if (c >= 1 && c <= nch) add(c - 1);
                barrier();
            }
        }
        j_seg = j_end;
    }
    if (wave == APW) {
        const uint32_t d = d0 + (lane & 15) * 4 + (lane >> 4);  // the lane's LDS slot back to its d
        if (d < a.hd) a.out[(uint64_t)b * a.n_heads * a.hd + (uint64_t)h * a.hd + d] = acc;
    }
}

hipError_t launch_paged_kv_append_i8(hipStream_t s, const float* src, const uint32_t* blocks, const uint32_t* offsets,
                                     const float* clip, uint32_t* pool, uint64_t pool_words, float* scales,
                                     uint64_t n_scales, uint32_t batch, uint32_t kv_stride, uint32_t bs, uint32_t hd) {
    const uint64_t grid = (uint64_t)batch * (kv_stride / hd);
    if (grid == 0) return hipSuccess;
    paged_kv_append_i8_kernel<<<(unsigned)grid, 64, 0, s>>>(src, blocks, offsets, clip, pool, pool_words, scales,
                                                            n_scales, kv_stride, bs, hd);
    return hipGetLastError();
}

hipError_t launch_paged_decode_i8(hipStream_t s, bool apply, const PagedReadArgs& a, uint32_t batch) {
    if (!apply) {
        const uint32_t nchunk = (a.cap + 63) / 64;
        const uint64_t grid = (uint64_t)batch * a.n_heads * nchunk;
        if (grid == 0) return hipSuccess;
        const bool vec = a.hd % 16 == 0 && a.kv_stride % 16 == 0 && (reinterpret_cast<uintptr_t>(a.pool) & 15) == 0;
        if (vec && a.hd == 128) go_scores_group<128>(s, a, batch);
        else if (vec && a.hd == 64) go_scores_group<64>(s, a, batch);
        else if (vec) paged_decode_scores_i8_kernel<true><<<(unsigned)grid, 64, 0, s>>>(a);
        else paged_decode_scores_i8_kernel<false><<<(unsigned)grid, 64, 0, s>>>(a);
    } else {
        const uint64_t grid = (uint64_t)batch * a.n_heads * ((a.hd + 63) / 64);
        if (grid == 0) return hipSuccess;
        const uint32_t n_kv = a.kv_stride / a.hd;
        const ApplyGeom g{a.pool_words * 4 / a.kv_stride, a.n_scales / n_kv, (uint32_t)(a.pool_words * 4 % a.kv_stride),
                    (uint32_t)(a.n_scales % n_kv), (a.bs & (a.bs - 1)) == 0 ? __builtin_ctz(a.bs) : -1};
        const bool small = a.pool_words < (1ull << 30) && a.n_scales < (1ull << 30) && a.bs < (1u << 24);
        if (a.bs % 4 == 0 && small) paged_decode_apply_i8_kernel<true, uint32_t><<<(unsigned)grid, APT, 0, s>>>(a, g);
        else if (a.bs % 4 == 0) paged_decode_apply_i8_kernel<true, uint64_t><<<(unsigned)grid, APT, 0, s>>>(a, g);
        else if (small) paged_decode_apply_i8_kernel<false, uint32_t><<<(unsigned)grid, APT, 0, s>>>(a, g);
        else paged_decode_apply_i8_kernel<false, uint64_t><<<(unsigned)grid, APT, 0, s>>>(a, g);
    }
    return hipGetLastError();
}

}  // namespace bh
