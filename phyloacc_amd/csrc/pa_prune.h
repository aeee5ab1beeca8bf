// pa_prune.h -- the pruning pass over a list of steps, shared by the chain
// kernel (pa_chain.hip) and the likelihood kernel (pa_engine.hip): a thread
// takes one pattern through the steps with the partials it needs next in
// registers.  One copy, so the two kernels apply the same operations in the
// same order and their FP32 results agree bit for bit.
#pragma once
#include <utility>
#include "pa_device.h"

namespace pa {

// A region of memory as a raw buffer: loads and stores take a lane's byte
// offset and a scalar one, and an access outside the region is dropped (a
// load gives 0).
typedef __amdgpu_buffer_rsrc_t Buf;
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

template <typename T>
__device__ __forceinline__ Buf make_buf(T *base, int bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc((void *)(T *)base, 0, bytes, 0x00027000);
}

// An element's leaf codes, S rows of Ppad.  A row's word is what a step keeps
// of it: its byte offset, which a load takes as it is, or (WIDE) the row's
// number, for codes of 4 GiB or more, beyond a 32-bit offset.  The kernels
// that score are built for both (host: wide_codes); the wide ones spend the
// scalar instructions of a 64-bit address on every load.
template <bool WIDE>
struct CodeRows;
template <>
struct CodeRows<false> {
    Buf buf;
    uint32_t Ppad;
    __device__ __forceinline__ CodeRows(const GBL uint8_t *base, int S, int P) : buf(make_buf((GBL uint8_t *)base, (int)((uint32_t)S * (uint32_t)P))), Ppad((uint32_t)P) {}
    __device__ __forceinline__ uint32_t row(int x) const { return (uint32_t)x * Ppad; }
    __device__ __forceinline__ int at(uint32_t row, uint32_t p) const { return __builtin_amdgcn_raw_buffer_load_b8(buf, p, row, 0); }
    // four codes of a row, a lane a row
    __device__ __forceinline__ uint32_t four(int x, uint32_t p) const { return __builtin_amdgcn_raw_buffer_load_b32(buf, (uint32_t)x * Ppad + p, 0, 0); }
};
template <>
struct CodeRows<true> {
    const GBL uint8_t *base;
    uint32_t Ppad;
    __device__ __forceinline__ CodeRows(const GBL uint8_t *b, int S, int P) : base(b), Ppad((uint32_t)P) {}
    __device__ __forceinline__ uint32_t row(int x) const { return (uint32_t)x; }
    __device__ __forceinline__ int at(uint32_t row, uint32_t p) const { return base[(uint64_t)row * Ppad + p]; }
    __device__ __forceinline__ uint32_t four(int x, uint32_t p) const { return *(const GBL uint32_t *)(base + ((uint64_t)(uint32_t)x * Ppad + p)); }
};

template <int... J, typename F>
__device__ __forceinline__ void each_of(std::integer_sequence<int, J...>, F &&f) { (f(std::integral_constant<int, J>()), ...); }
template <int... J, typename F>
__device__ __forceinline__ bool each_while_of(std::integer_sequence<int, J...>, F &&f) { return (f(std::integral_constant<int, J>()) && ...); }
// f(0) ... f(n - 1) with constant arguments until one returns false; whether none did
template <int n, typename F>
__device__ __forceinline__ bool each_while(F &&f) { return each_while_of(std::make_integer_sequence<int, n>(), f); }
// f(0) ... f(n - 1) with constant arguments: what it indexes stays in registers
template <int n, typename F>
__device__ __forceinline__ void each(F &&f) { each_of(std::make_integer_sequence<int, n>(), f); }

template <typename R>
__device__ __forceinline__ V4<R> buf_ld4(Buf b, uint32_t lane_off, uint32_t off)
{
    if constexpr (sizeof(R) == 4) {
        return __builtin_bit_cast(V4<R>, __builtin_amdgcn_raw_buffer_load_b128(b, lane_off, off, 0));
    } else {
        struct { u32x4 lo, hi; } v = {__builtin_amdgcn_raw_buffer_load_b128(b, lane_off, off, 0),
                                      __builtin_amdgcn_raw_buffer_load_b128(b, lane_off + 16, off, 0)};
        return __builtin_bit_cast(V4<R>, v);
    }
}
template <typename R>
__device__ __forceinline__ void buf_st4(Buf b, const V4<R> &v, uint32_t lane_off, uint32_t off)
{
    if constexpr (sizeof(R) == 4) {
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), b, lane_off, off, 0);
    } else {
        struct P { u32x4 lo, hi; };
        const P p = __builtin_bit_cast(P, v);
        __builtin_amdgcn_raw_buffer_store_b128(p.lo, b, lane_off, off, 0);
        __builtin_amdgcn_raw_buffer_store_b128(p.hi, b, lane_off + 16, off, 0);
    }
}

// One step of a pass, an internal node.  Four words:
//   w0: type | SB_* bits | child A's slot << 14 | the slot the node is stored to << 23
//   w1, w2: the code rows' words (CodeRows) of children A and B (row 0's, which is 0, for a child that is no leaf)
//   w3: the children's matrices A | B << 10 (the node's id, + N for a proposal matrix) | child B's slot << 20
// A child comes from its leaf code (L), its stored partial (S), or the result
// of the step just before (P) or the one before that (P2), which the thread
// still holds in registers.  The types are the combinations that occur when
// nothing is missing, so each is straight code; ST_GEN takes any sources and
// missing nodes.  The two children's order does not matter: their messages
// are multiplied.
enum { SK_LEAF = 0, SK_STORED = 1, SK_PREV = 2, SK_PREV2 = 3 };
enum { ST_LL = 0, ST_PL = 1, ST_PP2 = 2, ST_SL = 3, ST_SP = 4, ST_SS = 5, ST_GEN = 6 };
enum { SB_TYPE = 7, SB_STORED_A = 1 << 3, SB_STORED_B = 1 << 4, SB_NOSTORE = 1 << 5, SB_MISS_A = 1 << 7,
       SB_MISS_B = 1 << 8, SB_KIND_A_SHIFT = 9, SB_KIND_B_SHIFT = 11, SB_LATE = 1 << 13, SB_SLOT_A_SHIFT = 14, SB_SLOT_SHIFT = 23,
       SB_MAT_MASK = 0x3ff, SB_MAT_B_SHIFT = 10, SB_SLOT_B_SHIFT = 20 };
static_assert(MAXN <= 512, "slots (below 2 I <= N) in nine bits, matrices (below 2 N) in ten");

// What a step's words say, the children in any order.
struct StepDef {
    int kind[2], miss_kid[2], mat[2], slot[2];   // SK_* source, missing, matrix, stored slot
    uint32_t row[2];                             // code row's word
    int slot_to;                                         // where the node is stored
    bool nostore;
    bool late = false;                                   // a stored child is the step three before (F = 4 below)
};

__device__ __forceinline__ void encode_step(LDS uint32_t *w, const StepDef &d)
{
    // child A: a stored node before the previous result, that before the one before it, a leaf last
    const int rank = 0x2103;      // a nibble per kind
    const int a = ((rank >> (4 * d.kind[1])) & 15) < ((rank >> (4 * d.kind[0])) & 15) ? 1 : 0;
    const int ka = a ? d.kind[1] : d.kind[0], kb = a ? d.kind[0] : d.kind[1];
    const int ma = a ? d.miss_kid[1] : d.miss_kid[0], mb = a ? d.miss_kid[0] : d.miss_kid[1];
    int type = ST_GEN;
    if (!ma && !mb) {
        if (ka == SK_LEAF) type = ST_LL;
        else if (ka == SK_PREV) type = kb == SK_LEAF ? ST_PL : (kb == SK_PREV2 ? ST_PP2 : ST_GEN);
        else if (ka == SK_STORED) type = kb == SK_LEAF ? ST_SL : (kb == SK_PREV ? ST_SP : (kb == SK_STORED ? ST_SS : ST_GEN));
    }
    w[0] = (uint32_t)type | (ka == SK_STORED ? SB_STORED_A : 0) | (kb == SK_STORED ? SB_STORED_B : 0) |
           (d.nostore ? SB_NOSTORE : 0) | (d.late ? SB_LATE : 0) | (ma ? SB_MISS_A : 0) | (mb ? SB_MISS_B : 0) |
           ((uint32_t)ka << SB_KIND_A_SHIFT) | ((uint32_t)kb << SB_KIND_B_SHIFT) |
           ((uint32_t)(a ? d.slot[1] : d.slot[0]) << SB_SLOT_A_SHIFT) | ((uint32_t)d.slot_to << SB_SLOT_SHIFT);
    w[1] = a ? d.row[1] : d.row[0];
    w[2] = a ? d.row[0] : d.row[1];
    w[3] = (uint32_t)(a ? d.mat[1] : d.mat[0]) | ((uint32_t)(a ? d.mat[0] : d.mat[1]) << SB_MAT_B_SHIFT) |
           ((uint32_t)(a ? d.slot[0] : d.slot[1]) << SB_SLOT_B_SHIFT);
}

// The scalar arguments of a pass's pattern loop.
template <typename R, bool WIDE = false>
struct PassArgs {
    const LDS u32x4 *steps;
    const LDS R *PT;             // [2N][16]: the current matrices, then the proposal's
    CodeRows<WIDE> codes;
    int n, slots;                // steps; slots of a pattern block
};

// One child's message at one pattern, or ones where it holds no base; adds
// its exponent and reports the gap.
template <typename R, int K, bool AMB>
__device__ __forceinline__ void message(const LDS R *PT, int code, const ChildIn<R> &in, V4<R> &o, int &e, bool &gap)
{
    if constexpr (K == SK_LEAF) {
        gap = code == PA_GAP_CODE || code == PA_OTHER_CODE;
        o = ld4<R>((const LDS V4<R> *)(PT + 4 * (code & 3)));
        if (AMB && code > PA_OTHER_CODE) {
            o.x = o.y = o.z = o.w = (R)1;
            leaf_mul<R>(PT, code, o.x, o.y, o.z, o.w);
        }
        o.x = gap ? (R)1 : o.x; o.y = gap ? (R)1 : o.y; o.z = gap ? (R)1 : o.z; o.w = gap ? (R)1 : o.w;
    } else {
        gap = in.x == GAPT;
        int x = in.x;
        const V4<R> v = in.v;
        const V4<R> m0 = ld4<R>((const LDS V4<R> *)(PT + 0)), m1 = ld4<R>((const LDS V4<R> *)(PT + 4));
        const V4<R> m2 = ld4<R>((const LDS V4<R> *)(PT + 8)), m3 = ld4<R>((const LDS V4<R> *)(PT + 12));
        o.x = m0.x * v.x + m1.x * v.y + m2.x * v.z + m3.x * v.w;
        o.y = m0.y * v.x + m1.y * v.y + m2.y * v.z + m3.y * v.w;
        o.z = m0.z * v.x + m1.z * v.y + m2.z * v.z + m3.z * v.w;
        o.w = m0.w * v.x + m1.w * v.y + m2.w * v.z + m3.w * v.w;
        if (__ballot(gap)) {
            // rare: some lane's subtree holds only gaps
            o.x = gap ? (R)1 : o.x; o.y = gap ? (R)1 : o.y; o.z = gap ? (R)1 : o.z; o.w = gap ? (R)1 : o.w;
            x = gap ? 0 : x;
        }
        e += x;
    }
}

// A node from its children's messages: their product, rescaled by a power of two.
template <typename R>
__device__ __forceinline__ ChildIn<R> combine(const V4<R> &a, const V4<R> &b, int e, bool gap)
{
    const R x = a.x * b.x, y = a.y * b.y, z = a.z * b.z, w = a.w * b.w;
    const R mx = fmax(fmax(x, y), fmax(z, w));
    int kx = 0;
    frexp(mx, &kx);
    ChildIn<R> r;
    r.v.x = ldexp(x, -kx); r.v.y = ldexp(y, -kx); r.v.z = ldexp(z, -kx); r.v.w = ldexp(w, -kx);
    r.x = gap ? GAPT : e + kx;
    return r;
}

// A block of 64 patterns: `slots` slots of 64 4-vectors of R, then as many of
// 64 exponents.
__host__ __device__ inline int block_bytes(int slots, int rs) { return slots * 64 * (4 * rs + 4); }

// Byte offsets of a slot's partials and exponents within a pattern block.
template <typename R>
__device__ __forceinline__ uint32_t part_off(uint32_t slot) { return slot * (64 * (uint32_t)sizeof(V4<R>)); }
template <typename R>
__device__ __forceinline__ uint32_t exp_off(uint32_t slot, int slots) { return (uint32_t)slots * (64 * (uint32_t)sizeof(V4<R>)) + slot * 256; }

// Slot's partial and exponent of this lane's pattern, from the block's buffer.
template <typename R>
__device__ __forceinline__ ChildIn<R> slot_load(Buf blk, uint32_t slot, uint32_t lane, int slots)
{
    ChildIn<R> in;
    in.v = buf_ld4<R>(blk, lane * (uint32_t)sizeof(V4<R>), part_off<R>(slot));
    in.x = (int)__builtin_amdgcn_raw_buffer_load_b32(blk, lane * 4, exp_off<R>(slot, slots), 0);
    return in;
}

// Takes one pattern a lane (pattern p, of the block at base) through every
// step and returns the last step's partial and exponent.  All lanes run
// (patterns are padded to whole waves).  Step words are read a step before
// the loads they describe; leaf codes are loaded D steps before their use and
// stored partials two steps before (a stored child is at least three steps
// back: nearer ones are in registers), so neither a memory nor an LDS round
// trip stands between two steps.  Every step issues the same code loads,
// whether it needs them or not, since a step's wait for its loads counts the
// memory operations issued after them: a child that is no leaf loads row 0's
// code, and the steps past the last are an empty one.  ALL: every step also
// stores; a step marked SB_NOSTORE through a buffer of no bytes (the hardware
// drops accesses outside a buffer).  Otherwise only the steps not so marked
// store.  F = 4 (with D = 4): stored partials are loaded four steps before
// their use, for lists whose stored partials lie in HBM; a step marked
// SB_LATE, whose child was stored after that, loads them again.
template <typename R, bool AMB, int D, bool ALL, int F = 2, bool WIDE>
__device__ __forceinline__ ChildIn<R> prune_pattern(const PassArgs<R, WIDE> &A, GBL char *base, int blk_bytes, uint32_t p)
{
    const int n = A.n;
    const uint32_t lane = threadIdx.x & 63;
    const Buf blk = make_buf(base, blk_bytes);
    static_assert(F == 2 || F == D, "stored partials are loaded two steps ahead, or with the codes");
    ChildIn<R> inA[F], inB[F], res[2];
    int cdA[D], cdB[D];
    uint32_t w[D][4];
#pragma unroll
    for (int j = 0; j < 2; j++) {
        res[j].x = GAPT;
        res[j].v.x = res[j].v.y = res[j].v.z = res[j].v.w = (R)0;
    }
#pragma unroll
    for (int j = 0; j < F; j++) inA[j] = inB[j] = res[0];
    u32x4 nw = A.steps[0];
    // the words of step k into set j, its codes on their way
    auto fetch_codes = [&](auto J, int k) __attribute__((always_inline)) {
        constexpr int j = decltype(J)::value;
#pragma unroll
        for (int i = 0; i < 4; i++) w[j][i] = (uint32_t)uni((int)nw[i]);
        nw = A.steps[k + 1 < n ? k + 1 : n];
        cdA[j] = A.codes.at(w[j][1], p);
        cdB[j] = A.codes.at(w[j][2], p);
    };
    // the stored partials of the step whose words are set j
    auto fetch_stored = [&](auto J) __attribute__((always_inline)) {
        constexpr int j = decltype(J)::value;
        if (w[j][0] & SB_STORED_A) inA[j % F] = slot_load<R>(blk, (w[j][0] >> SB_SLOT_A_SHIFT) & 511, lane, A.slots);
        if (w[j][0] & SB_STORED_B) inB[j % F] = slot_load<R>(blk, w[j][3] >> SB_SLOT_B_SHIFT, lane, A.slots);
    };
    auto step = [&](auto J, int k) __attribute__((always_inline)) {
        constexpr int d = decltype(J)::value, j = d & 1, f = d % F;
        const uint32_t w0 = w[d][0];
        if constexpr (F > 2)
            if (w0 & SB_LATE) {
                fetch_stored(J);
                __builtin_amdgcn_s_waitcnt(0x0f70);      // vmcnt(0): what is in flight afterwards is as on the other path
            }
        const int type = w0 & SB_TYPE;
        const LDS R *PA = A.PT + 16 * (w[d][3] & SB_MAT_MASK), *PB = A.PT + 16 * ((w[d][3] >> SB_MAT_B_SHIFT) & SB_MAT_MASK);
        int e = 0;
        bool ga, gb;
        V4<R> a, b;
        ChildIn<R> out;
        if (type == ST_PL) {
            message<R, SK_PREV, AMB>(PA, 0, res[j ^ 1], a, e, ga);
            message<R, SK_LEAF, AMB>(PB, cdB[d], inB[f], b, e, gb);
            out = combine<R>(a, b, e, ga && gb);
        } else if (type == ST_LL) {
            message<R, SK_LEAF, AMB>(PA, cdA[d], inA[f], a, e, ga);
            message<R, SK_LEAF, AMB>(PB, cdB[d], inB[f], b, e, gb);
            out = combine<R>(a, b, e, ga && gb);
        } else if (type == ST_PP2) {
            message<R, SK_PREV, AMB>(PA, 0, res[j ^ 1], a, e, ga);
            message<R, SK_PREV2, AMB>(PB, 0, res[j], b, e, gb);
            out = combine<R>(a, b, e, ga && gb);
        } else if (type == ST_SP) {
            message<R, SK_STORED, AMB>(PA, 0, inA[f], a, e, ga);
            message<R, SK_PREV, AMB>(PB, 0, res[j ^ 1], b, e, gb);
            out = combine<R>(a, b, e, ga && gb);
        } else if (type == ST_SL) {
            message<R, SK_STORED, AMB>(PA, 0, inA[f], a, e, ga);
            message<R, SK_LEAF, AMB>(PB, cdB[d], inB[f], b, e, gb);
            out = combine<R>(a, b, e, ga && gb);
        } else if (type == ST_SS) {
            message<R, SK_STORED, AMB>(PA, 0, inA[f], a, e, ga);
            message<R, SK_STORED, AMB>(PB, 0, inB[f], b, e, gb);
            out = combine<R>(a, b, e, ga && gb);
        } else {
            // any sources, missing nodes: a missing child contributes nothing, but its gap state still
            // decides whether the parent is all-gap at this pattern.  A missing node (both children missing)
            // so comes out as ones, its exponent that of their rescaled form like any node's: at a missing
            // root the pattern's term is log sum_j pi_j = 0.
            const int ka = (w0 >> SB_KIND_A_SHIFT) & 3, kb = (w0 >> SB_KIND_B_SHIFT) & 3;
            auto source = [&](int kind, const ChildIn<R> &ld, int code) __attribute__((always_inline)) {
                const ChildIn<R> r1 = res[j ^ 1], r2 = res[j];
                ChildIn<R> ci;
                ci.x = kind == SK_PREV ? r1.x : (kind == SK_PREV2 ? r2.x : (kind == SK_LEAF ? code : ld.x));
                ci.v.x = kind == SK_PREV ? r1.v.x : (kind == SK_PREV2 ? r2.v.x : ld.v.x);
                ci.v.y = kind == SK_PREV ? r1.v.y : (kind == SK_PREV2 ? r2.v.y : ld.v.y);
                ci.v.z = kind == SK_PREV ? r1.v.z : (kind == SK_PREV2 ? r2.v.z : ld.v.z);
                ci.v.w = kind == SK_PREV ? r1.v.w : (kind == SK_PREV2 ? r2.v.w : ld.v.w);
                return ci;
            };
            a.x = a.y = a.z = a.w = b.x = b.y = b.z = b.w = (R)1;
            child_apply<R>(ka == SK_LEAF, w0 & SB_MISS_A, PA, source(ka, inA[f], cdA[d]), a.x, a.y, a.z, a.w, e, ga);
            child_apply<R>(kb == SK_LEAF, w0 & SB_MISS_B, PB, source(kb, inB[f], cdB[d]), b.x, b.y, b.z, b.w, e, gb);
            out = combine<R>(a, b, e, ga && gb);
        }
        if constexpr (D == 2) {
            fetch_codes(J, k + 2);
            fetch_stored(J);
        } else {
            if constexpr (F == 2) fetch_stored(std::integral_constant<int, (d + 2) % D>());
            fetch_codes(J, k + D);
        }
        res[j] = out;
        const uint32_t to = w0 >> SB_SLOT_SHIFT;
        if (ALL || !(w0 & SB_NOSTORE)) {
            const Buf b = ALL ? make_buf(base, (w0 & SB_NOSTORE) ? 0 : blk_bytes) : blk;
            buf_st4<R>(b, out.v, lane * (uint32_t)sizeof(V4<R>), part_off<R>(to));
            __builtin_amdgcn_raw_buffer_store_b32((uint32_t)out.x, b, lane * 4, exp_off<R>(to, A.slots), 0);
        }
        if constexpr (F > 2) fetch_stored(J);
    };
    each<D>([&](auto J) __attribute__((always_inline)) { fetch_codes(J, decltype(J)::value); });
    // no step before the third has a stored child of this pass, but it may have one of an earlier pass
    each<F>([&](auto J) __attribute__((always_inline)) { fetch_stored(J); });
    for (int k = 0; k < n; k += D)
        if (!each_while<D>([&](auto J) __attribute__((always_inline)) {
                step(J, k + decltype(J)::value);
                return k + decltype(J)::value + 1 < n;
            }))
            break;
    const bool odd = (n - 1) & 1;
    ChildIn<R> r;
    r.x = odd ? res[1].x : res[0].x;
    r.v.x = odd ? res[1].v.x : res[0].v.x;
    r.v.y = odd ? res[1].v.y : res[0].v.y;
    r.v.z = odd ? res[1].v.z : res[0].v.z;
    r.v.w = odd ? res[1].v.w : res[0].v.w;
    return r;
}

}  // namespace pa
