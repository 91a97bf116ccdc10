// Causal GQA attention of prompt rows over the KV cache on the bf16 matrix
// cores, at the precision of f32.
//
// The reference computes scores, softmax and the weighted values of a prompt
// row in f32 (paged_decode_scores_batched / decode_softmax_batched /
// paged_decode_apply_batched, and the i8 pair of them over an int8 cache:
// score = (q . code) * kscale * scale, context += (p * code) * vscale). Here
// an f32 operand x is the exact sum of three bf16 numbers, x = x1 + x2 + x3
// (8 significant bits each, each the rounding to nearest of what the ones
// before it leave: |x2| <= 2^-8 |x|, |x3| <= 2^-17 |x|), and a product of two
// such operands is the six partial products x1y1, x1y2, x2y1, x2y2, x1y3,
// x3y1, accumulated in f32 by v_mfma_f32_32x32x16_bf16. The three left out,
// x2y3 + x3y2 + x3y3, are at most 2^-24 of the product, the error of one f32
// multiplication, with either sign; for normal operands 0.06 x 2^-24 on
// average, where the f32 multiplication's is 0.36 x 2^-24. (Truncated parts
// leave out up to 8 x 2^-24, always towards zero.) Codes of the int8 cache are
// exact in one bf16, so a product with them is three partial products.
// f32 MFMA would take 64 cycles per 2048 multiply-adds, against 6 x 32 cycles
// per 16384 here (3 x 32 with an int8 cache).
//
// One workgroup: QG x KS (x DS) waves; wave (qg, ks) holds 32 query vectors (rows x
// heads of one kv head's group) and walks the key tiles of 32 keys whose
// index is ks mod KS, with its own running maximum, sum and context (online
// softmax); at the end the KS parts are merged through LDS in a fixed order.
// The tiles start at multiples of 32 positions and a masked tile leaves a
// vector's state as it is, so a row's numbers do not depend on the rows it
// shares a launch with: any chunking of a prompt gives the same bits. (Where
// an infinity, a NaN or an overflow makes a vector's result not finite, the
// vector is computed once more by plain_row; which vectors of a shared tile a
// NaN value reaches does depend on the chunking, and those agree to rounding.)
//
// Scores are computed transposed (keys x queries): a lane then holds 16 keys
// of one query, the softmax statistics need one exchange with lane ^ 32, and
// the probabilities are already the B operand of (V^T x P^T) once V^T is
// stored with its keys in the order the lanes hold them.
//
// K and V tiles go global -> registers -> (split) -> LDS; the loads of one go
// out while the other is being multiplied (int8 cache), or those of a step
// before the step before it is through (f32 cache, whose workgroup has its CU to
// itself: 2000 tokens 153 -> 143 us, and 139 with the third parts of the queries
// in registers).
//
// Measured, 16 query heads over 8 kv heads of 128, one 2000-token prompt /
// eight of 250, K and V in cache: int8 cache 70 / 28 us, f32 cache 139 / 32 us.
// (The kernel before it, f32 products on the vector units with 32-key partial
// sums through memory, and its merge: 964 + 138 us for the 2000 tokens, int8.)
// What bounds it: without the conversion to bf16 parts the f32 cache's kernel
// takes 16% less, without five of six products 16% less, without either 34%; LDS
// reads, the softmax and the latency of barriers are the rest.
// Waves: 2 x 4 for the int8 cache; for the f32 cache, whose split tiles take
// three times the LDS, 2 x 2 (one workgroup per CU by its registers; limited to
// the registers of two it spills, 191 us), and for few workgroups 1 x 2 x 2 (see
// SPLIT_D_GRID). KS is part of the result's summation order, so it is one per
// cache type and not chosen by length. Against 64-bit attention, one 2000-token
// prompt of normal q, k, v: 1.4e-7 (f32 cache) and 3.0e-7 (int8) in the 2-norm;
// the f32 kernel 2.2e-7 and 3.3e-7.
#include <type_traits>

#include "bh_common.h"
#include "bh_flash.h"

namespace bh {
namespace {

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));

__device__ __forceinline__ uint32_t fbits(float f) { return __builtin_bit_cast(uint32_t, f); }
__device__ __forceinline__ float bitsf(uint32_t u) { return __builtin_bit_cast(float, u); }
// The upper halves of two floats that are exact in bf16, packed.
__device__ __forceinline__ uint32_t hi16x2(float lo, float hi) {
    return __builtin_amdgcn_perm(fbits(hi), fbits(lo), 0x07060302u);
}

// Eight floats as three bf16 fragments. (A non-finite operand leaves NaN in
// the second part and in every result it enters: plain_row takes those.)
__device__ __forceinline__ void split8(const float (&x)[8], v4i& a, v4i& b, v4i& c) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float x0 = x[2 * i], x1 = x[2 * i + 1];
        const uint32_t p = pack_bf16x2(x0, x1);
        const float r0 = x0 - bitsf(p << 16), r1 = x1 - bitsf(p & 0xffff0000u);
        const uint32_t q = pack_bf16x2(r0, r1);
        a[i] = (int)p;
        b[i] = (int)q;
        c[i] = (int)hi16x2(r0 - bitsf(q << 16), r1 - bitsf(q & 0xffff0000u));  // exact: at most 8 bits are left
    }
}
// Softmax in base 2: a weight is exp2(fma(score, c, -m)) with
// c = scale * log2(e) and m the reference of the same base, one rounding at
// the size of the difference (the scaled score itself is never rounded).
// The reference is not the running maximum but within SLACK of it: it moves
// only when a key's score is more than SLACK above it, which spares most
// tiles the rescaling of the context; weights are then up to 2^SLACK, with the
// same relative precision. Each row decides for itself.
constexpr float SLACK = 8.0f;
// The score of a masked key, and a row's reference before its first key:
// finite, so that their differences are, and far enough apart that a masked
// key (times c >= 1/16) weighs 0 against either.
constexpr float MASKED = -1.0e38f, NO_REF = -1.0e34f;

__device__ __forceinline__ float code_f(uint32_t w, int e) { return (float)(int8_t)(uint8_t)(w >> (8 * e)); }

__device__ __forceinline__ v16f mfma(v4i a, v4i b, v16f c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, b), c, 0, 0, 0);
}

template <bool KV8, int HD, int QG, int KS, int DS>
struct FlashCfg {
    static constexpr int NT = QG * KS * DS * 64;
    static constexpr bool DEEP = !KV8;  // the next tiles of K and V both in flight
    static constexpr int KEYS = 32 * KS;               // keys per step
    static constexpr int PARTS = KV8 ? 1 : 3;          // bf16 parts of a cache element
    static constexpr int TILE = 32 * HD * 2;           // bytes of one part of 32 keys
    static constexpr int REGION = KS * PARTS * TILE;   // K, or V, of one step
    static constexpr bool SEP = DEEP || 2 * REGION <= 64 * 1024;  // K and V in LDS side by side
    static constexpr int VOFF = SEP ? REGION : 0;
    static constexpr int LDS = SEP ? 2 * REGION : REGION;
    static constexpr int OREGS = HD / 2 / DS;          // context registers per lane
    static constexpr int MERGE = (KS / 2) * QG * DS * 64 * OREGS * 4;
    static constexpr int NKC = KEYS * HD / 8 / NT;     // 8-element pieces of K per thread
    static constexpr int VB = KEYS * HD / 32;          // 8-key x 4-d blocks of V
    static constexpr int NVB = VB > NT ? VB / NT : 1;  // ... per thread (below VB, the first VB threads)
    static_assert(NKC * NT * 8 == KEYS * HD && (VB <= NT || NVB * NT == VB), "whole pieces per thread");
    static_assert(MERGE <= LDS, "the merge fits the tiles' LDS");
};

// One query vector by one wave in plain f32 over its visible keys alone, for
// the vectors whose result above is not finite: an infinity times a zero part
// or a zero weight is NaN there, a NaN value reaches the rows before it in a
// shared tile, a value that rounds to an infinity in bf16 is lost, and scores
// below NO_REF leave no weight at all. Here each of them is what the formula
// gives. Loads are uncoalesced (a lane reads its key's row): this runs for
// such vectors only. A NaN in the query or a score is NaN in every element and
// ends it early: once a model has gone to NaN every vector comes here.
template <bool KV8, int HD>
__device__ void plain_row(const FlashArgs& p, const uint32_t* tslot, int r, int kh, int h, int lane) {
    float* q = p.q + (size_t)r * p.hq + (size_t)h * HD;
    const int pos = (int)p.pos[r];
    using Elem = std::conditional_t<KV8, int8_t, float>;
    auto row_of = [&](int j) -> size_t { return (size_t)tslot[j >> 5] + (j & 31); };
    auto score = [&](int j) -> float {
        const size_t slot = row_of(j);
        const Elem* k = static_cast<const Elem*>(p.kc) + slot * p.hkv + (size_t)kh * HD;
        float acc = 0.0f;
#pragma unroll 4
        for (int d = 0; d < HD; ++d) acc = acc + q[d] * (float)k[d];
        if constexpr (KV8) acc = acc * p.ks[slot * p.nkv + kh];
        return acc * p.scale;
    };
    bool nan = false;
#pragma unroll
    for (int u = 0; u < HD / 64; ++u) nan |= q[lane + 64 * u] != q[lane + 64 * u];
    float mx = -INFINITY;
    if (!__any(nan)) {
        for (int j = lane; j <= pos; j += 64) {
            const float s = score(j);
            nan |= s != s;
            mx = fmaxf(mx, s);
        }
    }
    if (__any(nan)) {
#pragma unroll
        for (int u = 0; u < HD / 64; ++u) q[lane + 64 * u] = __builtin_nanf("");
        return;
    }
    mx = xor_max<32>(mx);
    float l = 0.0f, ctx[HD / 64];
#pragma unroll
    for (int u = 0; u < HD / 64; ++u) ctx[u] = 0.0f;
    for (int j0 = 0; j0 <= pos; j0 += 64) {
        float w = 0.0f;
        if (j0 + lane <= pos) {
            const float s = score(j0 + lane);
            w = s == -INFINITY ? 0.0f : expf(s - mx);
        }
        l = l + w;
        const int n = min(64, pos + 1 - j0);
        for (int k = 0; k < n; ++k) {
            const float wk = __shfl(w, k, 64);
            const size_t slot = row_of(j0 + k);
            const Elem* v = static_cast<const Elem*>(p.vc) + slot * p.hkv + (size_t)kh * HD;
#pragma unroll
            for (int u = 0; u < HD / 64; ++u) {
                float t = wk * (float)v[lane + 64 * u];
                if constexpr (KV8) t = t * p.vs[slot * p.nkv + kh];
                ctx[u] = ctx[u] + t;
            }
        }
    }
    l = xor_sum<32>(l);
#pragma unroll
    for (int u = 0; u < HD / 64; ++u) q[lane + 64 * u] = ctx[u] / l;
}

template <bool KV8, int HD, int QG, int KS, int DS>
__global__ __launch_bounds__(QG* KS * DS * 64, HD == 64 ? 2 : 1) void flash_prefill_kernel(FlashArgs p) {
    using C = FlashCfg<KV8, HD, QG, KS, DS>;
    __shared__ __attribute__((aligned(1024))) uint8_t lds[C::LDS];
    // int8 cache: the third parts of the queries (one use per key tile) live in
    // LDS: 32 registers fewer at head_dim 128, which is what keeps the kernel from
    // spilling at two waves per SIMD.
    __shared__ __attribute__((aligned(1024))) uint8_t q3[KV8 ? QG * C::TILE : 16];
    __shared__ float sml[QG * KS * DS][2][64];
    __shared__ uint32_t redo_ds[DS == 1 ? 1 : QG * DS];
    __shared__ __attribute__((aligned(16))) float ksc[KV8 ? C::KEYS : 4], vsc[KV8 ? C::KEYS : 4];
    __shared__ uint32_t tslot[FLASH_MAX_SEQ / 32];
    const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5, col = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), qg = wave % QG, ks = wave / QG % KS;
    const int ds = wave / (QG * KS), wd = ds * QG + qg;  // this wave's HD / DS columns of the context
    const int G = p.nh / p.nkv, RW = 32 / G;  // rows per wave
    const int nqb = (p.rows_per_seq + RW * QG - 1) / (RW * QG);
    // The blocks of the latest rows attend the most keys: they start first.
    const int kh = blockIdx.x % p.nkv, bq = blockIdx.x / p.nkv;
    const int b = bq % p.nseq, qb = nqb - 1 - bq / p.nseq;
    const int i0 = qb * RW * QG, nrow = min(RW * QG, p.rows_per_seq - i0);
    const int r0 = b * p.rows_per_seq + i0;
    const size_t seq = p.seq[r0];
    const int maxpos = (int)p.pos[r0 + nrow - 1];
    const int niter = maxpos / C::KEYS + 1;
    // First slot of every 32-key tile (a tile lies inside one block).
    for (int i = tid; i <= maxpos >> 5; i += C::NT) tslot[i] = (uint32_t)p.map.slot(seq, 32 * i);

    // This lane's query vector: row i of the block, head g of the group.
    const int iw = qg * RW + (col < RW * G ? col / G : 0), g = col < RW * G ? col % G : 0;
    const bool qlive = col < RW * G && iw < nrow;
    float* qrow = p.q + (size_t)(r0 + min(iw, nrow - 1)) * p.hq + (size_t)(kh * G + g) * HD;
    const int mypos = qlive ? (int)p.pos[r0 + iw] : -1;
    const bool wlive = qg * RW < nrow;  // a wave without rows only helps to stage
    const int wminpos = wlive ? (int)p.pos[r0 + qg * RW] : 0;
    const int wmaxpos = wlive ? (int)p.pos[r0 + min(qg * RW + RW, nrow) - 1] : -1;
    // LDS image of 32 rows of HD bf16 (a tile of K, or a wave's q3): 16-byte
    // chunk c of row r at c ^ (r & 15) (HD 64: c ^ (r >> 1 & 7)), so the 16
    // lanes of a fragment read on 16 rows hit 16 slots of a bank line.
    auto kchunk = [&](int r, int c) -> int {
        return r * (HD * 2) + ((HD == 128 ? c ^ (r & 15) : c ^ ((r >> 1) & 7)) << 4);
    };
    const uint8_t* q3w = q3 + qg * C::TILE;
    float4 qraw[HD / 8];
#pragma unroll
    for (int s = 0; s < HD / 16; ++s) {
        qraw[2 * s] = *reinterpret_cast<const float4*>(qrow + 16 * s + 8 * half);
        qraw[2 * s + 1] = *reinterpret_cast<const float4*>(qrow + 16 * s + 8 * half + 4);
    }
    // Orders LDS only; the global loads in flight go on.
    auto barrier = [&]() {
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    barrier();  // tslot

    // ---- staging
    constexpr int CPK = HD / 8;  // 16-byte bf16 chunks per key
    float4 kf[KV8 ? 1 : C::NKC * 2], vf[KV8 ? 1 : C::NVB * 8];  // K pieces, V blocks in flight
    uint32_t k8[KV8 ? C::NKC * 2 : 1], v8[KV8 ? C::NVB * 8 : 1];
    float kscale = 0.0f, vscale = 0.0f;
    // A tile's first cache row of this kv head, as a uniform element offset,
    // and its last visible key. Keys past that repeat it: their weights are
    // zero, and what they multiply is a value that is visible.
    struct TileAt {
        size_t base;
        int last;
    };
    auto tile_at = [&](int it, int w) -> TileAt {  // w: uniform
        const int t0 = min(it * KS + w, maxpos >> 5);
        const uint32_t slot = (uint32_t)__builtin_amdgcn_readfirstlane((int)tslot[t0]);
        return {(size_t)slot * (uint32_t)p.hkv + (uint32_t)(kh * HD), min(maxpos - 32 * t0, 31)};
    };
    using Elem = std::conditional_t<KV8, uint8_t, float>;
    auto load_scale = [&](int it, const float* sc, float& to) {
        if constexpr (KV8) {
            if (tid < C::KEYS) {
                const int t0 = min(it * KS + (tid >> 5), maxpos >> 5);
                to = sc[((size_t)tslot[t0] + min(tid & 31, maxpos - 32 * t0)) * p.nkv + kh];
            }
        }
    };
    // K: thread t takes chunk t % CPK of keys t / CPK + u * KPT. A wave's keys
    // of one u lie in one tile.
    constexpr int KPT = C::NT / CPK;
    static_assert(64 / CPK <= 32 && KPT * CPK == C::NT, "a wave's keys lie in one tile");
    const int kkey = tid / CPK;
    const uint32_t kcol = 8 * (tid % CPK);
    auto load_k = [&](int it) {
#pragma unroll
        for (int u = 0; u < C::NKC; ++u) {
            const TileAt t = tile_at(it, __builtin_amdgcn_readfirstlane((kkey + u * KPT) >> 5));
            const Elem* src = static_cast<const Elem*>(p.kc) + t.base;
            const uint32_t o = __umul24((uint32_t)min((kkey + u * KPT) & 31, t.last), (uint32_t)p.hkv) + kcol;
            if constexpr (KV8) {
                const uint2 v = *reinterpret_cast<const uint2*>(src + o);
                k8[2 * u] = v.x;
                k8[2 * u + 1] = v.y;
            } else {
                kf[2 * u] = *reinterpret_cast<const float4*>(src + o);
                kf[2 * u + 1] = *reinterpret_cast<const float4*>(src + o + 4);
            }
        }
        load_scale(it, p.ks, kscale);
    };
    auto store_k = [&]() {
#pragma unroll
        for (int u = 0; u < C::NKC; ++u) {
            const int q = tid + u * C::NT, key = q / CPK, c = q % CPK;
            uint8_t* dst = lds + (key >> 5) * C::PARTS * C::TILE + kchunk(key & 31, c);
            if constexpr (KV8) {
                v4i w;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint32_t cw = k8[2 * u + (i >> 1)];
                    w[i] = (int)hi16x2(code_f(cw, 2 * (i & 1)), code_f(cw, 2 * (i & 1) + 1));
                }
                *reinterpret_cast<v4i*>(dst) = w;
            } else {
                const float4 lo = kf[2 * u], hi = kf[2 * u + 1];
                const float x[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
                v4i w0, w1, w2;
                split8(x, w0, w1, w2);
                *reinterpret_cast<v4i*>(dst) = w0;
                *reinterpret_cast<v4i*>(dst + C::TILE) = w1;
                *reinterpret_cast<v4i*>(dst + 2 * C::TILE) = w2;
            }
        }
        if constexpr (KV8)
            if (tid < C::KEYS) ksc[tid] = kscale;
    };
    // A V block: 8 keys of one k-half of a 16-key step (the keys that half of
    // the lanes holds of the scores: 4h..4h+3 and 8+4h..8+4h+3) x 4 d.
    constexpr int DG = HD / 4;
    static_assert(4 * DG >= 64, "a wave's octets lie in one tile");
    auto load_v = [&](int it) {
#pragma unroll
        for (int u = 0; u < C::NVB; ++u) {
            const int q = tid + u * C::NT, oct = q / DG, dg = q % DG;
            if (C::VB < C::NT && tid >= C::VB) break;
            const TileAt t = tile_at(it, __builtin_amdgcn_readfirstlane(oct >> 2));
            const Elem* src = static_cast<const Elem*>(p.vc) + t.base;
            const int k0 = 16 * ((oct >> 1) & 1) + 4 * (oct & 1);
            auto at = [&](int j, const Elem* v) {
                if constexpr (KV8) v8[8 * u + j] = *reinterpret_cast<const uint32_t*>(v);
                else vf[8 * u + j] = *reinterpret_cast<const float4*>(v);
            };
            if (t.last == 31) {  // a uniform row stride: one lane offset for the eight loads
                const uint32_t o = __umul24((uint32_t)k0, (uint32_t)p.hkv) + 4 * dg;
#pragma unroll
                for (int j = 0; j < 8; ++j) at(j, src + (size_t)((j < 4 ? j : 4 + j) * p.hkv) + o);
            } else {
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    at(j, src + (__umul24((uint32_t)min(k0 + (j < 4 ? j : 4 + j), t.last), (uint32_t)p.hkv) + 4 * dg));
            }
        }
        load_scale(it, p.vs, vscale);
    };
    // LDS: V^T part t of tile w: lines of 256 bytes hold 4 d x 32 keys; the
    // chunk of 8 keys (octet o) of d at slot (4 (d % 4) + o) ^ (line & 15) of
    // line d / 4: neither the stores (16 lines, one d % 4 and o) nor the
    // fragment reads (16 consecutive d, one o) meet in a bank.
    auto vchunk = [&](int line, int d4, int o) -> int { return line * 256 + (((4 * d4 + o) ^ (line & 15)) << 4); };
    auto store_v = [&]() {
#pragma unroll
        for (int u = 0; u < C::NVB; ++u) {
            const int q = tid + u * C::NT, oct = q / DG, dg = q % DG;
            if (C::VB < C::NT && tid >= C::VB) break;
            uint8_t* base = lds + C::VOFF + (oct >> 2) * C::PARTS * C::TILE;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                uint8_t* dst = base + vchunk(dg, e, oct & 3);
                float x[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    if constexpr (KV8) x[j] = code_f(v8[8 * u + j], e);
                    else {
                        const float4 v = vf[8 * u + j];
                        x[j] = e == 0 ? v.x : e == 1 ? v.y : e == 2 ? v.z : v.w;
                    }
                }
                if constexpr (KV8) {
                    *reinterpret_cast<v4i*>(dst) = v4i{(int)hi16x2(x[0], x[1]), (int)hi16x2(x[2], x[3]),
                                                       (int)hi16x2(x[4], x[5]), (int)hi16x2(x[6], x[7])};
                } else {
                    v4i w0, w1, w2;
                    split8(x, w0, w1, w2);
                    *reinterpret_cast<v4i*>(dst) = w0;
                    *reinterpret_cast<v4i*>(dst + C::TILE) = w1;
                    *reinterpret_cast<v4i*>(dst + 2 * C::TILE) = w2;
                }
            }
        }
        if constexpr (KV8)
            if (tid < C::KEYS) vsc[tid] = vscale;
    };
    constexpr int OJ = HD / 32 / DS;
    v16f o[OJ];
#pragma unroll
    for (int j = 0; j < OJ; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[j][e] = 0.0f;
    const float c2 = p.scale * 1.44269504088896341f;
    float m = NO_REF, l = 0.0f;  // l: this half's keys only

    load_k(0);
    if constexpr (C::DEEP) load_v(0);
    v4i qf[HD / 16][2], qf3[KV8 ? 1 : HD / 16];
#pragma unroll
    for (int s = 0; s < HD / 16; ++s) {
        const float4 lo = qraw[2 * s], hi = qraw[2 * s + 1];
        const float x[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
        v4i third;
        split8(x, qf[s][0], qf[s][1], third);
        if constexpr (!KV8) qf3[s] = third;
        else if (ks == 0) *reinterpret_cast<v4i*>(q3 + qg * C::TILE + kchunk(col, 2 * s + half)) = third;
    }
    for (int it = 0; it < niter; ++it) {
        if constexpr (!C::SEP) barrier();  // the last step's V has been read
        store_k();
        if constexpr (!C::DEEP) load_v(it);
        else if (it + 1 < niter) load_k(it + 1);
        barrier();
        const int j0 = it * C::KEYS + 32 * ks;
        const bool live = j0 <= wmaxpos;  // wave-uniform
        v16f s;
        if (live) {
#pragma unroll
            for (int e = 0; e < 16; ++e) s[e] = 0.0f;
            const uint8_t* kb = lds + ks * C::PARTS * C::TILE;
            // The small partial products first: only the HD / 16 sums of
            // k1q1 then round at the size of the score.
#pragma unroll
            for (int t = 0; t < HD / 16; ++t) {
                const uint8_t* src = kb + kchunk(col, 2 * t + half);
                const v4i k1 = *reinterpret_cast<const v4i*>(src);
                if constexpr (KV8) {
                    const v4i qt = *reinterpret_cast<const v4i*>(q3w + kchunk(col, 2 * t + half));
                    s = mfma(k1, qt, s);
                    s = mfma(k1, qf[t][1], s);
                    s = mfma(k1, qf[t][0], s);
                } else {
                    const v4i k2 = *reinterpret_cast<const v4i*>(src + C::TILE);
                    const v4i k3 = *reinterpret_cast<const v4i*>(src + 2 * C::TILE);
                    s = mfma(k3, qf[t][0], s);
                    s = mfma(k1, qf3[t], s);
                    s = mfma(k2, qf[t][1], s);
                    s = mfma(k2, qf[t][0], s);
                    s = mfma(k1, qf[t][1], s);
                }
            }
            if constexpr (!KV8) {
#pragma unroll
                for (int t = 0; t < HD / 16; ++t)
                    s = mfma(*reinterpret_cast<const v4i*>(kb + kchunk(col, 2 * t + half)), qf[t][0], s);
            }
            // Register e: key 8 (e / 4) + 4 half + e % 4 of the tile.
            if constexpr (KV8) {
#pragma unroll
                for (int e4 = 0; e4 < 4; ++e4) {
                    const float4 k = *reinterpret_cast<const float4*>(ksc + 32 * ks + 8 * e4 + 4 * half);
                    s[4 * e4] = s[4 * e4] * k.x;
                    s[4 * e4 + 1] = s[4 * e4 + 1] * k.y;
                    s[4 * e4 + 2] = s[4 * e4 + 2] * k.z;
                    s[4 * e4 + 3] = s[4 * e4 + 3] * k.w;
                }
            }
            if (j0 + 31 > wminpos) {
                const int lim = mypos - j0 - 4 * half;  // keys of this half up to here are visible
#pragma unroll
                for (int e = 0; e < 16; ++e)
                    if (8 * (e >> 2) + (e & 3) > lim) s[e] = MASKED;
            }
            float mx = s[0];
#pragma unroll
            for (int e = 1; e < 16; ++e) mx = fmaxf(mx, s[e]);
            mx = fmaxf(mx, xor_lane<32>(mx)) * c2;  // c2 > 0: the largest scaled score
            const bool up = mx > m + SLACK;
            if (__any(up)) {
                const float mn = up ? mx : m;
                const float alpha = __builtin_amdgcn_exp2f(m - mn);  // 1 where the reference stays
                l = l * alpha;
#pragma unroll
                for (int j = 0; j < OJ; ++j)
#pragma unroll
                    for (int e = 0; e < 16; ++e) o[j][e] = o[j][e] * alpha;
                m = mn;
            }
            float sum = 0.0f;
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                s[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[e], c2, -m));
                sum = sum + s[e];
            }
            l = l + sum;
        }
        if constexpr (!C::SEP) barrier();  // every wave has read this step's K
        store_v();
        if (it + 1 < niter) {
            if constexpr (C::DEEP) load_v(it + 1);
            else load_k(it + 1);
        }
        barrier();
        if (live) {
            if constexpr (KV8) {
#pragma unroll
                for (int e4 = 0; e4 < 4; ++e4) {
                    const float4 v = *reinterpret_cast<const float4*>(vsc + 32 * ks + 8 * e4 + 4 * half);
                    s[4 * e4] = s[4 * e4] * v.x;
                    s[4 * e4 + 1] = s[4 * e4 + 1] * v.y;
                    s[4 * e4 + 2] = s[4 * e4 + 2] * v.z;
                    s[4 * e4 + 3] = s[4 * e4 + 3] * v.w;
                }
            }
            const uint8_t* vb = lds + C::VOFF + ks * C::PARTS * C::TILE;
            v4i pf[2][3];
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                float x[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) x[i] = s[8 * t + i];
                split8(x, pf[t][0], pf[t][1], pf[t][2]);
            }
#pragma unroll
            for (int j = 0; j < OJ; ++j) {
                const int d = 32 * (ds * OJ + j) + col;
                const uint8_t* src[2] = {vb + vchunk(d >> 2, d & 3, half), vb + vchunk(d >> 2, d & 3, 2 + half)};
                if constexpr (KV8) {
#pragma unroll
                    for (int t = 0; t < 2; ++t) {
                        const v4i v1 = *reinterpret_cast<const v4i*>(src[t]);
                        o[j] = mfma(v1, pf[t][2], o[j]);
                        o[j] = mfma(v1, pf[t][1], o[j]);
                        o[j] = mfma(v1, pf[t][0], o[j]);
                    }
                } else {
                    // The tile's sum on its own, small products first, then
                    // one addition to the context.
                    v16f a;
#pragma unroll
                    for (int e = 0; e < 16; ++e) a[e] = 0.0f;
                    v4i v1[2];
#pragma unroll
                    for (int t = 0; t < 2; ++t) {
                        v1[t] = *reinterpret_cast<const v4i*>(src[t]);
                        const v4i v2 = *reinterpret_cast<const v4i*>(src[t] + C::TILE);
                        const v4i v3 = *reinterpret_cast<const v4i*>(src[t] + 2 * C::TILE);
                        a = mfma(v3, pf[t][0], a);
                        a = mfma(v1[t], pf[t][2], a);
                        a = mfma(v2, pf[t][1], a);
                        a = mfma(v2, pf[t][0], a);
                        a = mfma(v1[t], pf[t][1], a);
                    }
#pragma unroll
                    for (int t = 0; t < 2; ++t) a = mfma(v1[t], pf[t][0], a);
#pragma unroll
                    for (int e = 0; e < 16; ++e) o[j][e] = o[j][e] + a[e];
                }
            }
        }
    }

    // Merge the KS parts: the upper half of the waves hands its state to the
    // lower half, until one wave per query group is left.
#pragma unroll
    for (int w = KS / 2; w >= 1; w /= 2) {
        barrier();
        float4* om = reinterpret_cast<float4*>(lds) + (size_t)((ks % w) * QG * DS + wd) * 64 * (C::OREGS / 4) + lane;
        if (ks >= w && ks < 2 * w) {
#pragma unroll
            for (int j = 0; j < OJ; ++j)
#pragma unroll
                for (int e4 = 0; e4 < 4; ++e4)
                    om[(4 * j + e4) * 64] = make_float4(o[j][4 * e4], o[j][4 * e4 + 1], o[j][4 * e4 + 2], o[j][4 * e4 + 3]);
            sml[(ks % w) * QG * DS + wd][0][lane] = m;
            sml[(ks % w) * QG * DS + wd][1][lane] = l;
        }
        barrier();
        if (ks < w) {
            const float m2 = sml[(ks % w) * QG * DS + wd][0][lane], l2 = sml[(ks % w) * QG * DS + wd][1][lane];
            const float mn = fmaxf(m, m2);
            const float a1 = __builtin_amdgcn_exp2f(m - mn), a2 = __builtin_amdgcn_exp2f(m2 - mn);
            m = mn;
            l = l * a1 + l2 * a2;
#pragma unroll
            for (int j = 0; j < OJ; ++j)
#pragma unroll
                for (int e4 = 0; e4 < 4; ++e4) {
                    const float4 v = om[(4 * j + e4) * 64];
                    o[j][4 * e4] = o[j][4 * e4] * a1 + v.x * a2;
                    o[j][4 * e4 + 1] = o[j][4 * e4 + 1] * a1 + v.y * a2;
                    o[j][4 * e4 + 2] = o[j][4 * e4 + 2] * a1 + v.z * a2;
                    o[j][4 * e4 + 3] = o[j][4 * e4 + 3] * a1 + v.w * a2;
                }
        }
    }
    uint32_t redo = 0;
    if (ks == 0) {
        const float inv = 1.0f / (l + xor_lane<32>(l));
        float z = 0.0f;  // NaN once a context element is not finite
#pragma unroll
        for (int j = 0; j < OJ; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                o[j][e] = o[j][e] * inv;
                z = __builtin_fmaf(o[j][e], 0.0f, z);
            }
        const unsigned long long bad = __ballot(qlive && z != 0.0f);
        redo = (uint32_t)bad | (uint32_t)(bad >> 32);  // by col: a vector's two halves
    }
    if constexpr (DS > 1) {  // ... and its DS parts
        if (ks == 0 && lane == 0) redo_ds[wd] = redo;
        barrier();
        redo = 0;
#pragma unroll
        for (int i = 0; i < DS; ++i) redo |= (uint32_t)__builtin_amdgcn_readfirstlane((int)redo_ds[i * QG + qg]);
    }
    if (ks == 0) {
        if (qlive && !((redo >> col) & 1u)) {
#pragma unroll
            for (int j = 0; j < OJ; ++j)
#pragma unroll
                for (int e4 = 0; e4 < 4; ++e4)
                    *reinterpret_cast<float4*>(qrow + 32 * (ds * OJ + j) + 8 * e4 + 4 * half) =
                        make_float4(o[j][4 * e4], o[j][4 * e4 + 1], o[j][4 * e4 + 2], o[j][4 * e4 + 3]);
        }
        // Live columns only (bad is 0 elsewhere); their queries are not yet
        // overwritten.
        for (; ds == 0 && redo; redo &= redo - 1u) {
            const int c = __ffs(redo) - 1, i = qg * RW + c / G;
            plain_row<KV8, HD>(p, tslot, r0 + i, kh, kh * G + c % G, lane);
        }
    }
}

// Up to this many workgroups of 2 x 2 waves, half the chip, the f32 cache's
// kernel is a serial chain in each: half the rows per workgroup then, and two
// waves that each make the whole scores and half of the context's columns (the
// same bits). 16 heads over 8 of 128, us, 2 x 2 / 1 x 2 x 2: 64 tokens 10.2 / 9.0,
// 128 14.0 / 12.5, 200 19.4 / 18.7, 512 (128 workgroups) 36.9 / 33.6; 1000
// (256) 67 / 70, eight sequences of 128 (256) 14.9 / 21.3: more than 256
// workgroups of the second kind take turns on the CUs.
constexpr unsigned SPLIT_D_GRID = 128;

template <bool KV8, int HD, int QG, int KS, int DS>
hipError_t launch(hipStream_t s, const FlashArgs& a, unsigned grid) {
    flash_prefill_kernel<KV8, HD, QG, KS, DS><<<grid, QG * KS * DS * 64, 0, s>>>(a);
    return hipGetLastError();
}

template <bool KV8, int HD>
hipError_t go(hipStream_t s, const FlashArgs& a) {
    auto grid = [&](int qg) -> unsigned {
        const int rb = 32 / (a.nh / a.nkv) * qg;
        return (unsigned)((a.rows_per_seq + rb - 1) / rb * a.nseq * a.nkv);
    };
    if constexpr (KV8) return launch<true, HD, 2, 4, 1>(s, a, grid(2));
    else if (grid(2) <= SPLIT_D_GRID) return launch<false, HD, 1, 2, 2>(s, a, grid(1));
    else return launch<false, HD, 2, 2, 1>(s, a, grid(2));
}

}  // namespace

hipError_t launch_flash_prefill(hipStream_t s, const FlashArgs& a, int hd, bool kv8) {
    if (a.rows_per_seq <= 0 || a.nseq <= 0) return hipSuccess;
    if (hd == 128) return kv8 ? go<true, 128>(s, a) : go<false, 128>(s, a);
    return kv8 ? go<true, 64>(s, a) : go<false, 64>(s, a);
}

}  // namespace bh

// The kernel alone, with its arguments spelled out (not in the public header:
// the engine launches it; the tests call this).
extern "C" int bh_flash_prefill_rows(void* stream, float* q, const void* kc, const void* vc, const float* ks,
                                     const float* vs, const uint32_t* pos, const uint32_t* seq, const uint32_t* bt,
                                     uint32_t nh, uint32_t nkv, uint32_t hd, uint32_t rows_per_seq, uint32_t nseq,
                                     uint32_t max_seq, uint32_t max_bt, uint32_t bs, uint32_t nblk, float scale,
                                     uint32_t kv8) {
    if (!nkv || nh % nkv || !bh::flash_ok((int)hd, (int)nh, (int)nkv, (int)max_seq)) return (int)hipErrorInvalidValue;
    const bh::FlashArgs a{q, kc, vc, ks, vs, pos, seq, (int)nh, (int)nkv, (int)(nh * hd), (int)(nkv * hd),
                          (int)rows_per_seq, (int)nseq, scale,
                          bh::KvMap{bt, (int)max_bt, (int)bs, (int)nblk, (int)max_seq}};
    return (int)bh::launch_flash_prefill((hipStream_t)stream, a, (int)hd, kv8 != 0);
}
