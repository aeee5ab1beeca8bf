// pa_chain.hip -- CDNA4 (gfx950) chain kernel for PhyloAcc-ST's per-element MCMC.
//
// The fixed-(Z, r) log-likelihood kernel is in pa_engine.hip.
//
// One workgroup owns one element at a time and runs its three model chains
// (M0, M1, M2 = resZ 0, 2, 1; src/PhyloAcc-ST/main.cpp:466-494) start to
// finish; workgroups pull elements from a device work queue (persistent
// kernel).  Within a workgroup:
//   * threads stride over site patterns (pruning) or sites (ancestral
//     sampling); a pass is a list of steps in post-order (pa_prune.h), and a
//     thread takes its patterns through the whole list, so no barrier is
//     needed between tree nodes;
//   * conditional likelihoods are in HBM scratch by blocks of 64 patterns, two
//     slots per internal node (current / proposal) so an accepted Metropolis
//     move flips a per-node bit instead of copying partials;
//   * partials are linear-space with a power-of-two rescale per node; the
//     cumulative exponent rides along as an int; GAPT marks all-gap subtrees
//     (the reference's Tg >= num_base, src/PhyloAcc-ST/bpp_c.hpp:417-428);
//   * a cherry (a non-root internal node whose children are both leaves) is
//     never stored: a pass that visits its parent computes it as the step just
//     before, and the ancestral sampler from its two leaf codes, with the same
//     operations, so results are unchanged and its store, its reload and one
//     dependent memory round trip are saved;
//   * per-branch 4x4 transition matrices of the current rate class live in
//     LDS (read as broadcasts); FP64 is used for P(t) builds, log tables,
//     emissions, the Z forward-backward, likelihood sums and MH ratios.
// The chain context and the model constants live in LDS behind
// address-space-3 pointers, and every sweep phase is a separate non-inlined
// function, so each phase gets its own register allocation instead of one
// allocation spanning the whole persistent loop.
// The kernel is bound by latency and issue: a wave issues an instruction about
// every five cycles and four share a SIMD.  Matrix instructions for the FP32
// messages (4x4x1, bit for bit the same) took 40 % of the vector instructions
// away and no time.
#include <hip/hip_runtime.h>
#include <type_traits>
#include <algorithm>
#include <stdint.h>
#include "pa_common.h"
#include "pa_rng.h"
#include "pa_chain.h"
#include "pa_device.h"
#include "pa_prune.h"

namespace pa {
namespace chain {

template <typename R>
struct Ctx {
    // element
    int S, N, I, GG, P, Ppad, root, n_nodes, n_int, n_up, has_amb;
    const GBL uint8_t *codes;
    const GBL int32_t *wts, *site;
    // workgroup scratch in HBM
    GBL char *parts;       // partials and exponents by block of 64 patterns (block_bytes)
    GBL double *plin;      // [3][N][16]  P_{j->i} at [j*4+i]
    GBL double *logt;      // [3][N][16]  log P_{j->i} at [i*4+j]
    GBL uint32_t *amb;     // [S][24]
    const GBL double *dist2;   // [N] branch lengths (element node table)
    // LDS arrays
    LDS int16_t *par, *nodes, *inodes, *porder, *upoff;
    LDS uint32_t *urec;    // [I] internal nodes by level: node | child 0 << 10 | child 1 << 20
    LDS uint32_t *desc;    // [I] static pruning descriptor of each internal node (node_desc)
    LDS uint32_t *steps;   // [I + 1][4] the steps of a pass (build_steps)
    LDS uint32_t *srec;    // [I + 1][2] the steps of the sampler (sample_steps)
    LDS uint8_t *flags, *fixZ, *dirty, *cur, *changed;
    LDS int8_t *Z, *maxZ;
    LDS double *E, *msg;   // [N][3] emissions, then Z messages at a node; messages to its parent
    LDS R *PTc, *PTp;      // [N][16], PT[i*4+j] = P_{j->i}
    LDS uint32_t *hist, *cnt9;
    LDS uint8_t *tgs;
    // chain scalars
    double loglik, nrate, crate, g, l, l2, prop_n, prop_c, proposal, old_rate, r, max_loglik;
    double TMf[9], TMn[9];  // log_TM_Int for fixZ / free nodes, [i*3+j] = log P(child i | parent j)
    double red[4], gam[8], mh[5];   // block sums; a sweep's gamma variates; Metropolis terms
    int has_cls[2];                 // any branch in class 1 (conserved), 2 (accelerated)
    unsigned long long bytes;   // algorithmic HBM bytes of this element's passes (see prune / sample_sites)
    int accept_n, accept_c, max_m, skip, accept, fail, work, nch, n_steps, last_step, n_stored, n_cherry, n_leaf;   // fail: PA_F_* bits
};

template <typename R>
using CP = LDS Ctx<R> *;
using MP = LDS const ModelDev *;

__host__ __device__ inline size_t al(size_t x, size_t a) { return (x + a - 1) & ~(a - 1); }

// Dynamic-LDS layout: returns the byte size; BIND also points the context's
// array fields into the block.  The context may sit at LDS address 0, which
// compares equal to a null pointer, so binding is selected at compile time and
// never by testing the context pointer.
template <typename R, bool BIND>
__host__ __device__ size_t smem_arrays(int N, int S, int BS, LDS char *base, CP<R> c)
{
    const int I = N - S;
    size_t o = 0;
#define PA_TAKE(field, T, count)                                                   \
    do {                                                                           \
        o = al(o, sizeof(T) < 4 ? 4 : sizeof(T));                                  \
        if constexpr (BIND) c->field = (LDS T *)(base + o);                        \
        o += sizeof(T) * (size_t)(count);                                          \
    } while (0)
    // matrices first: rows of PT are read as 4-vectors (32-byte aligned base)
    PA_TAKE(PTc, R, 16 * N);
    // Phases that never overlap share storage:
    //   A: per-thread ancestral states (sample_sites) | emissions and Z
    //      messages (emissions, update_Z) | the steps of a pass (prune) |
    //      Z-transition counts (sample_transition);
    //   B: per-branch transition counters (sample_sites, emissions) |
    //      proposal matrices (rate updates).  sample_sites clears the
    //      counters before it counts.
    {
        const size_t szA = std::max({(size_t)(I > 0 ? I : 1) * BS, (size_t)6 * N * sizeof(double), (size_t)20 * 4, (size_t)16 * (I + 1)});
        const size_t szB = std::max((size_t)16 * N * sizeof(uint32_t), (size_t)16 * N * sizeof(R));
        o = al(o, 32);
        if constexpr (BIND) {
            c->PTp = (LDS R *)(base + o);
            c->hist = (LDS uint32_t *)(base + o);
        }
        o += al(szB, 32);
        if constexpr (BIND) {
            c->E = (LDS double *)(base + o);
            c->msg = (LDS double *)(base + o) + 3 * N;
            c->tgs = (LDS uint8_t *)(base + o);
            c->cnt9 = (LDS uint32_t *)(base + o);
            c->steps = (LDS uint32_t *)(base + o);
        }
        o += szA;
    }
    PA_TAKE(desc, uint32_t, I > 0 ? I : 1);
    o = al(o, 8);       // sampler steps as 8-byte vectors
    PA_TAKE(srec, uint32_t, 2 * (I + 1));
    PA_TAKE(urec, uint32_t, I > 0 ? I : 1);
    PA_TAKE(par, int16_t, N);
    PA_TAKE(nodes, int16_t, N);
    PA_TAKE(inodes, int16_t, N);
    PA_TAKE(porder, int16_t, I > 0 ? I : 1);
    PA_TAKE(upoff, int16_t, I + 1);
    PA_TAKE(flags, uint8_t, N);
    PA_TAKE(fixZ, uint8_t, N);
    PA_TAKE(dirty, uint8_t, N);
    PA_TAKE(cur, uint8_t, N);
    PA_TAKE(changed, uint8_t, N);
    PA_TAKE(Z, int8_t, N);
    PA_TAKE(maxZ, int8_t, N);
#undef PA_TAKE
    return al(o, 16);
}

size_t chain_smem_bytes(int N, int S, int BS, int fp64)
{
    return (fp64 ? smem_arrays<double, false>(N, S, BS, nullptr, nullptr)
                 : smem_arrays<float, false>(N, S, BS, nullptr, nullptr)) +
           (fp64 ? sizeof(Ctx<double>) : sizeof(Ctx<float>)) + sizeof(ModelDev);
}

// Partials of an element, by block of 64 patterns: two buffers of I node
// slots (slot = buffer * I + node - S).  A wave's block is one contiguous
// region, so every address in a pass is a scalar base and a small offset.
size_t chain_part_bytes(int N, int S, int Ppad, int fp64)
{
    return al((size_t)(Ppad / 64) * (size_t)block_bytes(2 * (N - S), fp64 ? 8 : 4), 256);
}

// Per-workgroup HBM scratch layout (bytes), shared with the host: the rate
// class tables and ambiguity counters, then the partial region.
size_t slot_scratch_bytes(int N, int S, int Pcap, int fp64, size_t *off)
{
    size_t o = 0;
    off[0] = o; o = al(o + (size_t)3 * N * 16 * 8, 256);          // plin
    off[1] = o; o = al(o + (size_t)3 * N * 16 * 8, 256);          // logt
    off[2] = o; o = al(o + (size_t)S * 24 * 4, 256);              // amb
    off[3] = o; o += chain_part_bytes(N, S, Pcap, fp64);          // parts, exps
    return o;
}

// ------------------------------------------------------------------ helpers

__device__ __forceinline__ void lds_add(LDS uint32_t *p, uint32_t v)
{
    __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Class tables of every branch for class k (0 null, 1 conserved, 2 accelerated)
// at rate r, a lane per matrix row.
// mode 0: model start (dist2 > 1e-10 -> P(dist2*r), else identity; bpp_c.cpp:187-228)
// mode 1: refresh after a rate change (dist2 < 1e-10 keeps the old table;
//         bpp_c.cpp:1115-1131), with the current matrices of the class's branches
template <typename R, int BS>
__device__ __noinline__ void class_tables(MP M, CP<R> c, int k, double r, int mode)
{
    const int N = uni(c->N), n_item = 4 * (uni(c->n_nodes) - 1);
    const LDS int16_t *nodes = uni_ptr(c->nodes);
    const GBL double *dist2 = uni_ptr(c->dist2);
    for (int it = threadIdx.x; it < n_item; it += BS) {
        const int s = nodes[it >> 2], j = it & 3;
        const double d = dist2[s];
        GBL double *P = c->plin + ((size_t)k * N + s) * 16;
        GBL double *L = c->logt + ((size_t)k * N + s) * 16;
        if (mode == 1 && d < 1e-10) continue;       // a whole quad
        double row[4];
        ptrans_row(&M->lam[0], d * r, j, row);
        if (mode == 0 && !(d > 1e-10)) {
#pragma unroll
            for (int i = 0; i < 4; i++) row[i] = i == j ? 1.0 : 0.0;
        }
#pragma unroll
        for (int i = 0; i < 4; i++) {
            P[j * 4 + i] = row[i];
            L[i * 4 + j] = log(row[i]);
        }
        if (mode == 1) {
            const int z = c->Z[s];
            if (z == k) {
                LDS R *dst = c->PTc + 16 * s;
#pragma unroll
                for (int i = 0; i < 4; i++) dst[i * 4 + j] = (R)row[i];
            }
        }
    }
}

// PT of the current class of every branch, or (changed_only) of those whose Z
// the last Z update changed
template <typename R, int BS, int SH>
__device__ __noinline__ void refresh_PTc(CP<R> c, bool changed_only)
{
    for (int q = threadIdx.x; q < c->n_nodes - 1; q += BS) {
        const int s = c->nodes[q];
        const int z = c->Z[s];
        if (changed_only && !c->changed[s]) continue;
        const int k = z == 2 ? 2 : (z == 0 ? 0 : 1);
        const GBL double *P = c->plin + ((size_t)k * c->N + s) * 16;
        LDS R *dst = c->PTc + 16 * s;
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int j = 0; j < 4; j++) dst[i * 4 + j] = (R)P[j * 4 + i];
    }
}

// ----------------------------------------------------------------- pruning

enum { PR_FULL = 0, PR_DIRTY = 1, PR_PROP = 2 };

// Kind of a node's child (node_desc): a leaf, a stored internal node, a cherry.
enum { KD_LEAF = 0, KD_STORED = 1, KD_CHERRY = 2 };

// Static pruning descriptor of an internal node, built when the element is
// bound (node_desc): its children x0 | x1 << 10 and DB_* bits: each child's
// kind (KD_LEAF / KD_STORED / KD_CHERRY) and whether it is missing.
enum { DB_KID = 0x3ff, DB_KID1_SHIFT = 10, DB_KIND0_SHIFT = 20, DB_KIND1_SHIFT = 22, DB_MISS0 = 1 << 24, DB_MISS1 = 1 << 25 };

// Shapes of the sampler's loop.  K: internal nodes whose partials and codes
// are in flight at a time.  FP64 has half FP32's, its partials taking twice
// the registers.  Shape 2 doubles K and was slower where it was measured: 373
// against 355 ms for 50,000 elements of 43 species in FP32.  Shape 1 is shape
// 0: they differed in how many nodes a pass pruned together, and a pass now
// takes one node at a time.
template <typename R, int SH>
struct Shape;
template <> struct Shape<float, 0> { static constexpr int K = 4; };
template <> struct Shape<float, 2> { static constexpr int K = 8; };
template <> struct Shape<double, 0> { static constexpr int K = 2; };
template <> struct Shape<double, 2> { static constexpr int K = 4; };

// The steps of a pass, written by one wave: a ballot per 64 internal nodes
// (in pruning order) places them, and each lane encodes its own node.  A
// child that is the list's previous (or second previous) entry is taken from
// registers.
template <typename R>
__device__ __forceinline__ void build_steps(CP<R> c, int mode, int cls)
{
    const int lane = threadIdx.x;
    const bool prop = mode == PR_PROP;
    const int S = uni(c->S), N = uni(c->N), I = uni(c->I), n_int = uni(c->n_int), Ppad = uni(c->Ppad);
    const LDS int16_t *porder = uni_ptr(c->porder), *par = uni_ptr(c->par);
    const LDS uint8_t *flags = uni_ptr(c->flags), *dirty = uni_ptr(c->dirty), *cur = uni_ptr(c->cur);
    const LDS int8_t *Z = uni_ptr(c->Z);
    const LDS uint32_t *desc = uni_ptr(c->desc);
    LDS uint32_t *steps = uni_ptr(c->steps);
    int base = 0, last1 = -1, last2 = -1, n_node = 0, n_leaf = 0, n_cherry = 0;
    for (int q0 = 0; q0 < n_int; q0 += 64) {
        const int q = q0 + lane;
        bool v = false;
        int s = 0, f = 0, leaves = 0, cherries = 0;
        if (q < n_int) {
            s = porder[q];
            f = flags[s];
            // a cherry is a step of its parent's visit
            const int t = (f & NF_CHERRY) ? par[s] : s;
            v = mode == PR_FULL || (dirty[t] && !(flags[t] & NF_MISSING));
        }
        const unsigned long long bal = __ballot(v);
        const unsigned long long below = bal & ((1ull << lane) - 1);
        const int l1 = below ? 63 - __clzll(below) : -1;
        const unsigned long long below2 = l1 >= 0 ? below ^ (1ull << l1) : 0;
        const int l2 = below2 ? 63 - __clzll(below2) : -1;
        const int s1 = __shfl(s, l1 < 0 ? 0 : l1, 64), s2 = __shfl(s, l2 < 0 ? 0 : l2, 64);
        const int n1 = l1 >= 0 ? s1 : last1, n2 = l2 >= 0 ? s2 : (l1 >= 0 ? last1 : last2);
        if (v) {
            const uint32_t dd = desc[s - S];
            int kind[2], miss[2], m[2], slot[2] = {0, 0};
            uint32_t row[2] = {0, 0};
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const int x = (dd >> (j ? DB_KID1_SHIFT : 0)) & DB_KID;
                const int k = (dd >> (j ? DB_KIND1_SHIFT : DB_KIND0_SHIFT)) & 3;
                m[j] = x + ((prop && Z[x] == cls) ? N : 0);
                miss[j] = (dd & (j ? DB_MISS1 : DB_MISS0)) ? 1 : 0;
                if (k == KD_LEAF) {
                    kind[j] = SK_LEAF;
                    row[j] = (uint32_t)x * (uint32_t)Ppad;
                } else {
                    const int cx = cur[x];
                    kind[j] = x == n1 ? SK_PREV : (x == n2 ? SK_PREV2 : SK_STORED);
                    slot[j] = ((prop && dirty[x]) ? 1 - cx : cx) * I + x - S;
                }
                leaves |= (k == KD_LEAF) << j;
                cherries |= (k == KD_CHERRY) << j;
            }
            const int cs = cur[s];
            StepDef d;
            d.nostore = (f & NF_CHERRY) != 0;
            d.slot_to = (prop ? 1 - cs : cs) * I + s - S;
#pragma unroll
            for (int j = 0; j < 2; j++) { d.kind[j] = kind[j]; d.miss_kid[j] = miss[j]; d.mat[j] = m[j]; d.row[j] = row[j]; d.slot[j] = slot[j]; }
            encode_step(steps + 4 * (base + __popcll(below)), d);
        }
        const int cnt = __popcll(bal);
        if (cnt) {
            const int h1 = 63 - __clzll(bal);
            const unsigned long long rest = bal ^ (1ull << h1);
            const int t1 = __shfl(s, h1, 64);
            const int t2 = __shfl(s, rest ? 63 - __clzll(rest) : 0, 64);
            last2 = cnt > 1 ? t2 : last1;
            last1 = t1;
        }
        base += cnt;
        const unsigned long long nodes = __ballot(v && !(f & NF_CHERRY));
        n_node += __popcll(nodes);
        n_leaf += __popcll(nodes & __ballot(leaves & 1)) + __popcll(nodes & __ballot(leaves & 2));
        n_cherry += __popcll(nodes & __ballot(cherries & 1)) + __popcll(nodes & __ballot(cherries & 2));
    }
    if (lane < 4) steps[4 * base + lane] = 0;       // the step read ahead of the end
    if (lane == 0) {
        c->n_steps = base;
        c->last_step = last1;
        // counted bytes, node by node: write partial + exponent; read each child's partial + exponent, its leaf
        // code, or a cherry's two codes; then the root's partial, exponent and weight
        const unsigned long long W = 4 * sizeof(R) + 4;
        c->bytes += (unsigned long long)c->P * (n_node * W + n_leaf + 2 * n_cherry + (2 * n_node - n_leaf - n_cherry) * W + W + 4);
    }
}

// The pattern loop of a pass: this thread's part of the root's log sum.
template <typename R, int BS, bool AMB>
__device__ __forceinline__ double prune_patterns(MP M, CP<R> c, int mode)
{
    const int tid = threadIdx.x;
    const int P = uni(c->P);
    const PassArgs<R> A = {(const LDS u32x4 *)uni_ptr(c->steps), uni_ptr(c->PTc), {uni_ptr(c->codes), uni(c->S), uni(c->Ppad)}, uni(c->n_steps),
                           2 * uni(c->I)};
    GBL char *parts = uni_ptr(c->parts);
    const int I = uni(c->I), blkB = block_bytes(2 * I, sizeof(R));
    const int r = uni(c->root);
    const GBL int32_t *wts = uni_ptr(c->wts);
    const double p0 = M->pi[0], p1 = M->pi[1], p2 = M->pi[2], p3 = M->pi[3];
    // the root is the last step of every pass that visits it
    const bool in_regs = A.n > 0 && uni(c->last_step) == r;
    const int rc = uni(c->cur[r]), rb = (mode == PR_PROP && uni(c->dirty[r])) ? 1 - rc : rc;
    double acc = 0;
    // whole waves of 64 patterns; wave w takes blocks w, w + BS / 64, ...
    for (int pb = uni(tid & ~63); pb < P; pb += BS) {
        const uint32_t lane = tid & 63, p = (uint32_t)pb + lane;
        GBL char *blk = parts + (int64_t)(pb >> 6) * blkB;
        ChildIn<R> o;
        if (A.n > 0) o = prune_pattern<R, AMB, 2, true>(A, blk, blkB, p);
        if (!in_regs) o = slot_load<R>(make_buf(blk, blkB), rb * I + r - uni(c->S), lane, 2 * I);
        // log sum_j pi_j L_j + exponent * ln 2; all-gap columns contribute 0
        if (o.x != GAPT && (int)p < P) {
            const double L = p0 * (double)o.v.x + p1 * (double)o.v.y + p2 * (double)o.v.z + p3 * (double)o.v.w;
            acc += (double)wts[p] * (log(L) + (double)o.x * 0.69314718055994530942);
        }
    }
    return acc;
}

// One pruning pass (BPP_C::Update_Tg(tosample=false), src/PhyloAcc-ST/bpp_c.cpp:644-671,
// and log_f_Xz, bpp_c.cpp:860-928).  FULL: every internal node of the tree
// (missing nodes only record their GAPT flag) into the current buffer.
// DIRTY: nodes with dirty[] set, in place.  PROP: dirty nodes into the other
// buffer, with PTp for branches whose Z is cls.  A cherry is a step of its
// parent's visit, dirty or not, and is not stored.  Returns the element's log-likelihood (FP64), identical on every
// thread.
//
// A pass is a chain of nodes, and what bounds it is the time of one link.
// The steps are therefore in post-order with the larger subtree of every fork
// first (pruning order), so that a node mostly follows its child: the
// child's partial is still in registers, a cherry's always is, and only the
// larger side of a fork of stored nodes is read back.  Each step's nodes,
// sources and matrices come as four words (build_steps) that are read ahead of
// their use, and the inputs of the step after next are in flight.  (By tree
// level, with each node's descriptor read when its turn came, a step waited
// for three dependent LDS round trips and the loads of both children.)
// A thread owns the patterns p = tid (mod BS) of every node, so the pass
// needs no barrier between steps.  The root's FP64 log sum is a deterministic
// block reduction.
template <typename R, int BS, int SH>
__device__ __noinline__ double prune(MP M, CP<R> c, int mode, int cls)
{
    if (threadIdx.x < 64) build_steps<R>(c, mode, cls);
    __syncthreads();
    const double acc = uni(c->has_amb) ? prune_patterns<R, BS, true>(M, c, mode) : prune_patterns<R, BS, false>(M, c, mode);
    return block_sum(acc, c->red);
}

// ------------------------------------------------------ ancestral sampling

// One step of the sampler: an internal node, in reverse post-order (step 0
// the root).  Two words, built when the element is bound (sample_steps):
//   r0: node | parent << 10 | SR_* bits
//   r1: the node's leaf children A | B << 10 (0: none) | the slot of its partial << 22 (follows cur; a cherry has
//       none stored, and its load goes where the root's does)
enum { SR_ID = 0x3ff, SR_PAR_SHIFT = 10, SR_MISS = 1 << 20, SR_CHERRY = 1 << 21,
       SR_PREV = 1 << 22,                          // the parent is the step before
       SR_LEAF_A = 1 << 23, SR_LEAF_B = 1 << 24,   // leaf children that are counted
       SR_MISS_A = 1 << 25, SR_MISS_B = 1 << 26,   // a cherry's missing leaves
       SR_SLOT_SHIFT = 22 };

// BPP_C::Update_Tg(tosample=true) (src/PhyloAcc-ST/bpp_c.cpp:672-733) for every
// site, plus the per-branch transition counts that getEmission
// (bpp_c2.cpp:355-390) sums over.  Uniform for site g, sampling position t
// (0 = root, then internal nodes in reverse post-order): ANC stream, c1 = g.
//
// One thread per site, whole waves.  As in a pass, what bounds it is the time
// of one step: the steps' words are read ahead, the loads of the next K steps
// are in flight (the same four loads every step, so that their waits are
// counted), the parent's base is in a register when the parent was the step
// before and otherwise read a step early, and a node counts its own leaf
// children, whose parent's base it has just drawn.
template <typename R, int BS, int SH, bool AMB>
__device__ __forceinline__ void draw_sites(MP M, CP<R> c, uint32_t c2, uint32_t c3)
{
    constexpr int K = Shape<R, SH>::K, UN = K < 4 ? 4 : K;     // steps unrolled: whole blocks of four draws
    const int tid = threadIdx.x, S = uni(c->S), I = uni(c->I), n_int = uni(c->n_int), GG = uni(c->GG), Ppad = uni(c->Ppad);
    const int blkB = block_bytes(2 * I, sizeof(R));
    const uint32_t k0 = (uint32_t)uni((int)M->key0), k1 = (uint32_t)uni((int)M->key1);
    const double p0 = M->pi[0], p1 = M->pi[1], p2 = M->pi[2], p3 = M->pi[3];
    const GBL char *parts = uni_ptr(c->parts);
    const CodeRows<false> codes(uni_ptr(c->codes), S, Ppad);
    const GBL int32_t *site = uni_ptr(c->site);
    GBL uint32_t *amb = uni_ptr(c->amb);
    LDS uint8_t *tgs = uni_ptr(c->tgs) + tid - S * BS;      // node s: [s * BS]
    LDS uint32_t *hist = uni_ptr(c->hist);
    const LDS u32x2 *srec = (const LDS u32x2 *)uni_ptr(c->srec);
    const LDS R *PTc = uni_ptr(c->PTc);
    for (int gb = uni(tid & ~63); gb < GG; gb += BS) {
        const int g = gb + (tid & 63);
        const bool on = g < GG;
        const int p = site[on ? g : GG - 1];
        // this pattern's entries of slot 0
        const GBL char *pp = parts + (int64_t)(p >> 6) * blkB + (p & 63) * sizeof(V4<R>);
        const GBL char *pe = parts + (int64_t)(p >> 6) * blkB + exp_off<R>(0, 2 * I) + (p & 63) * 4;
        uint32_t r0[K], r1[K];
        u32x2 nr = srec[0];
        ChildIn<R> in[K];
        int cdA[K], cdB[K];
        auto fetch = [&](auto J, int t) __attribute__((always_inline)) {
            constexpr int j = decltype(J)::value;
            r0[j] = (uint32_t)uni((int)nr.x);
            r1[j] = (uint32_t)uni((int)nr.y);
            nr = srec[t + 1 < n_int ? t + 1 : n_int];
            const uint32_t slot = r1[j] >> SR_SLOT_SHIFT;
            in[j].v = ld4<R>((const GBL V4<R> *)(pp + (uint64_t)part_off<R>(slot)));
            in[j].x = *(const GBL int32_t *)(pe + (uint64_t)(slot * 256));
            cdA[j] = codes.at(codes.row(r1[j] & SR_ID), p);
            cdB[j] = codes.at(codes.row((r1[j] >> 10) & SR_ID), p);
        };
        U4 rnd{0, 0, 0, 0};
        int ts = 0, tp = 0;
        auto count_leaf = [&](int y, int code) __attribute__((always_inline)) {
            if (on && code < 4) lds_add(&hist[y * 16 + ts * 4 + code], 1u);
            if (AMB && on && code > PA_OTHER_CODE)
                __hip_atomic_fetch_add(&amb[y * 24 + ts * 6 + (code - 6)], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        };
        auto step = [&](auto JJ, int t) __attribute__((always_inline)) {
            constexpr int jj = decltype(JJ)::value, j = jj % K;
            if ((jj & 3) == 0) rnd = philox((uint32_t)(t >> 2), (uint32_t)g, c2, c3, k0, k1);
            const double u = u01(pick(rnd, jj & 3));
            const uint32_t w0 = r0[j], w1 = r1[j];
            const int s = w0 & SR_ID;
            const int tp_read = tp & 3;
            // the next step's parent, unless it is this node
            tp = tgs[((r0[(j + 1) % K] >> SR_PAR_SHIFT) & SR_ID) * BS];
            if (!(w0 & SR_MISS)) {
                ChildIn<R> a;
                if (w0 & SR_CHERRY) {
                    // the partial a pass would have stored: the leaves' messages combined
                    V4<R> ma, mb;
                    int e = 0;
                    bool ga, gb2;
                    message<R, SK_LEAF, AMB>(PTc + 16 * (w1 & SR_ID), cdA[j], in[j], ma, e, ga);
                    message<R, SK_LEAF, AMB>(PTc + 16 * ((w1 >> 10) & SR_ID), cdB[j], in[j], mb, e, gb2);
                    if (w0 & SR_MISS_A) ma.x = ma.y = ma.z = ma.w = (R)1;
                    if (w0 & SR_MISS_B) mb.x = mb.y = mb.z = mb.w = (R)1;
                    a = combine<R>(ma, mb, 0, ga && gb2);
                } else {
                    a.v = in[j].v;
                    a.x = in[j].x;
                }
                const bool has = a.x != GAPT;       // else no base below it at this site: not drawn
                double pr[4];
                int from = 0;
                if (t == 0) {
                    pr[0] = has ? p0 * (double)a.v.x : p0; pr[1] = has ? p1 * (double)a.v.y : p1;
                    pr[2] = has ? p2 * (double)a.v.z : p2; pr[3] = has ? p3 * (double)a.v.w : p3;
                } else {
                    from = (w0 & SR_PREV) ? ts : tp_read;
                    const LDS R *PT = PTc + 16 * s + from;
                    pr[0] = (double)PT[0] * (double)a.v.x; pr[1] = (double)PT[4] * (double)a.v.y;
                    pr[2] = (double)PT[8] * (double)a.v.z; pr[3] = (double)PT[12] * (double)a.v.w;
                }
                ts = categorical<4>(pr, u);
                tgs[s * BS] = (uint8_t)ts;
                if (t != 0 && on && has) lds_add(&hist[s * 16 + from * 4 + ts], 1u);
                if (w0 & SR_LEAF_A) count_leaf(w1 & SR_ID, cdA[j]);
                if (w0 & SR_LEAF_B) count_leaf((w1 >> 10) & SR_ID, cdB[j]);
            }
            fetch(std::integral_constant<int, j>(), t + K);
        };
        each<K>([&](auto J) __attribute__((always_inline)) { fetch(J, decltype(J)::value); });
        // whole groups of UN steps: those past the last node are missing nodes
        for (int t0 = 0; t0 < n_int; t0 += UN)
            each<UN>([&](auto J) __attribute__((always_inline)) { step(J, t0 + decltype(J)::value); });
    }
}

template <typename R, int BS, int SH>
__device__ __noinline__ void sample_sites(MP M, CP<R> c, uint32_t c2, uint32_t c3)
{
    const int tid = threadIdx.x, amb_on = uni(c->has_amb), n_hist = 16 * uni(c->N), n_amb = 24 * uni(c->S);
    for (int i = tid; i < n_hist; i += BS) c->hist[i] = 0;   // shares storage with the proposal matrices
    if (amb_on)
        for (int i = tid; i < n_amb; i += BS) c->amb[i] = 0;
    if (tid == 0) {
        // per site: pattern index, root partial, each non-missing internal node's partial
        // (a cherry's two leaf codes), each leaf code
        c->bytes += (unsigned long long)c->GG * (4 + (4 * sizeof(R) + 4) * c->n_stored + 2 * c->n_cherry + c->n_leaf);
    }
    __syncthreads();
    if (amb_on) draw_sites<R, BS, SH, true>(M, c, c2, c3);
    else draw_sites<R, BS, SH, false>(M, c, c2, c3);
}

// The sampler's step words (layout at SR_*) and the node counts its bytes
// are counted from.
template <typename R, int BS>
__device__ __noinline__ void sample_steps(CP<R> c)
{
    const int S = c->S, n_int = c->n_int;
    for (int t = threadIdx.x; t < n_int; t += BS) {
        const int s = c->inodes[n_int - 1 - t];
        const uint32_t dd = c->desc[s - S];
        const int x0 = dd & DB_KID, x1 = (dd >> DB_KID1_SHIFT) & DB_KID;
        const int f = c->flags[s], f0 = c->flags[x0], f1 = c->flags[x1];
        uint32_t w0 = (uint32_t)s | ((f & NF_MISSING) ? SR_MISS : 0) | ((f & NF_CHERRY) ? SR_CHERRY : 0), w1 = 0;
        if (t > 0) {
            const int par = c->par[s];
            w0 |= (uint32_t)par << SR_PAR_SHIFT;
            if (par == c->inodes[n_int - t]) w0 |= SR_PREV;
        } else {
            w0 |= (uint32_t)s << SR_PAR_SHIFT;      // not read
        }
        if (x0 < S) {
            w1 |= (uint32_t)x0;
            if (f0 & NF_MISSING) w0 |= SR_MISS_A;
            else if (f0 & NF_IN_TREE) w0 |= SR_LEAF_A;
        }
        if (x1 < S) {
            w1 |= (uint32_t)x1 << 10;
            if (f1 & NF_MISSING) w0 |= SR_MISS_B;
            else if (f1 & NF_IN_TREE) w0 |= SR_LEAF_B;
        }
        const int v = (f & (NF_MISSING | NF_CHERRY)) ? c->root : s;
        c->srec[2 * t] = w0;
        c->srec[2 * t + 1] = w1 | (uint32_t)(v - S) << SR_SLOT_SHIFT;      // buffer 0
    }
    if (threadIdx.x == 0) {
        // the steps past the last
        c->srec[2 * n_int] = (uint32_t)c->root | (uint32_t)c->root << SR_PAR_SHIFT | SR_MISS;
        c->srec[2 * n_int + 1] = (uint32_t)(c->root - S) << SR_SLOT_SHIFT;
        int nint = 0, nch = 0, nleaf = 0;
        for (int k = 0; k < n_int; k++) {
            const uint8_t f = c->flags[c->inodes[k]];
            if (f & NF_MISSING) continue;
            if (f & NF_CHERRY) nch++; else nint++;
        }
        for (int q = 0; q < S; q++) nleaf += (c->flags[q] & NF_IN_TREE) && !(c->flags[q] & NF_MISSING);
        c->n_stored = nint;
        c->n_cherry = nch;
        c->n_leaf = nleaf;
    }
}

// getEmission (src/PhyloAcc-ST/bpp_c2.cpp:355-390): E[s][k] from the counts,
// one thread per (branch, class), its sixteen log entries loaded together.
template <typename R, int BS, int SH>
__device__ __noinline__ void emissions(CP<R> c)
{
    const int N = uni(c->N), n_item = 3 * (uni(c->n_nodes) - 1);
    const LDS int16_t *nodes = uni_ptr(c->nodes);
    const LDS uint8_t *flags = uni_ptr(c->flags);
    for (int it = threadIdx.x; it < n_item; it += BS) {
        const int q = it / 3, k = it - 3 * q, s = nodes[q];
        if (flags[s] & NF_MISSING) continue;
        const GBL double *L = c->logt + ((size_t)k * N + s) * 16;
        const LDS uint32_t *h = c->hist + s * 16;
        double l[16];
        uint32_t n[16];
#pragma unroll
        for (int i = 0; i < 16; i++) l[i] = L[i];
#pragma unroll
        for (int i = 0; i < 16; i++) n[i] = h[i];
        double e = 0;
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const double t = e + (double)n[j * 4 + i] * l[i * 4 + j];
                e = n[j * 4 + i] ? t : e;
            }
        if (c->has_amb && s < c->S) {
            const GBL uint32_t *a = c->amb + s * 24;
            const GBL double *P = c->plin + ((size_t)k * N + s) * 16;
            double ea = 0;
            for (int j = 0; j < 4; j++)
                for (int x = 0; x < 6; x++) {
                    const uint32_t cnt = a[j * 6 + x];
                    if (!cnt) continue;
                    const int code = 6 + x;
                    const int b1 = (code == 6 || code == 9 || code == 11) ? 0 : (code == 7 || code == 10) ? 1 : 2;
                    const int b2 = (code == 6 || code == 10) ? 2 : (code == 9) ? 1 : 3;
                    ea += (double)cnt * log(P[j * 4 + b1] + P[j * 4 + b2]);
                }
            e += ea;
        }
        c->E[s * 3 + k] = e;
    }
}

// ----------------------------------------------------------------- Z update

// exp(a - m), exp(b - m), exp(d - m) for m the largest of the three: the
// largest one's is 1 (NaN when m is infinite), so two exponentials do.
__device__ __forceinline__ void exp3(double a, double b, double d, double m, double &ea, double &eb, double &ed)
{
    const double one = 1.0 + (m - m);
    const bool am = a == m, bm = !am && b == m;
    const double x = exp((am ? b : a) - m), y = exp((am || bm ? d : b) - m);
    ea = am ? one : x;
    eb = am ? x : (bm ? one : y);
    ed = am || bm ? y : one;
}

// log sum_i exp(T[i*3+j] + y[i]) for parent class j, with the column's own
// maximum taken out first (log_multi2, src/PhyloAcc-ST/bpp.hpp:447-460);
// -inf when every term is -inf.
__device__ __forceinline__ double log_col(const LDS double *T, int j, double y0, double y1, double y2)
{
    const double a = T[j] + y0, b = T[3 + j] + y1, d = T[6 + j] + y2;
    const double mx = fmax(a, fmax(b, d));
    if (mx == -INFINITY) return -INFINITY;
    double ea, eb, ed;
    exp3(a, b, d, mx, ea, eb, ed);
    return mx + log(ea + eb + ed);
}

// BPP_C::Update_Z_subtree (src/PhyloAcc-ST/bpp_c.cpp:1182-1293) in log space:
// messages up the tree, then draws down it; the draw for node s uses Z-stream
// slot tz[s], its place in the reverse post-order.  Log space matters: over
// thousands of sites the classes' emissions differ by thousands of nats, and
// products of linear messages would underflow to zero.
//
// The phase is a chain of dependent logarithms and exponentials, so only what
// depends on the level below is left in the chain: the leaves' messages are
// computed by all threads at once; one wave then takes the internal levels, a
// lane per (node, parent class), without barriers; and the draws are tabled
// for every node and every class its parent could take, all at once, so that
// going down the tree is following each node's ancestors through those
// tables.
template <typename R, int BS, int SH>
__device__ __noinline__ void update_Z(MP M, CP<R> c, uint32_t c2, uint32_t c3)
{
    const int tid = threadIdx.x;
    const Key key{M->key0, M->key1};
    const int n_nodes = uni(c->n_nodes), S = uni(c->S), N = uni(c->N), root = uni(c->root), n_up = uni(c->n_up);
    const LDS int16_t *nodes = uni_ptr(c->nodes), *par = uni_ptr(c->par), *upoff = uni_ptr(c->upoff);
    const LDS uint32_t *urec = uni_ptr(c->urec);
    const LDS uint8_t *flags = uni_ptr(c->flags), *fixZ = uni_ptr(c->fixZ);
    const LDS double *TMf = uni_ptr(c->TMf), *TMn = uni_ptr(c->TMn);
    LDS double *beta = uni_ptr(c->E), *msg = uni_ptr(c->msg);      // beta starts as the emissions
    for (int q = tid; q < n_nodes; q += BS) {
        const int s = nodes[q];
        if (s == root) {
            beta[s * 3] = beta[s * 3 + 1] = beta[s * 3 + 2] = 0;
        } else if (flags[s] & NF_MISSING) {
            beta[s * 3] = beta[s * 3 + 2] = log(M->nconstomis);
            beta[s * 3 + 1] = log(M->constomis);
        }
        if (fixZ[s]) beta[s * 3 + 2] = -INFINITY;
        c->changed[s] = 0;
        c->dirty[s] = 0;
    }
    if (tid == 0) c->nch = 0;
    __syncthreads();
    for (int i = tid; i < 3 * S; i += BS) {
        const int s = i / 3, j = i - 3 * s;
        if (!(flags[s] & NF_IN_TREE)) continue;
        msg[i] = log_col(fixZ[s] ? TMf : TMn, j, beta[s * 3], beta[s * 3 + 1], beta[s * 3 + 2]);
    }
    __syncthreads();
    if (tid < 64) {
        // 21 nodes at a time, three lanes each: a node's lanes read its beta
        // together before they write it
        const int r = tid / 3, j = tid - 3 * r;
        int a = 0, b = uni(upoff[0]);
        uint32_t rec = r < b ? urec[r] : 0;
        for (int h = 0; h < n_up; h++) {
            const int b2 = h + 1 < n_up ? uni(upoff[h + 1]) : b;
            for (int q0 = a; q0 < b; q0 += 21) {
                const bool on = tid < 63 && q0 + r < b;
                const uint32_t w = rec;
                // the next group's record
                const int qn = (q0 + 21 < b ? q0 + 21 : b) + r;
                rec = qn < b2 ? urec[qn] : 0;
                if (on) {
                    const int p = w & 0x3ff, x0 = (w >> 10) & 0x3ff, x1 = w >> 20;
                    const LDS double *T = fixZ[p] ? TMf : TMn;
                    const double b0 = beta[p * 3] + msg[x0 * 3] + msg[x1 * 3], b1 = beta[p * 3 + 1] + msg[x0 * 3 + 1] + msg[x1 * 3 + 1],
                                 bb = beta[p * 3 + 2] + msg[x0 * 3 + 2] + msg[x1 * 3 + 2];
                    __builtin_amdgcn_wave_barrier();
                    beta[p * 3 + j] = j == 0 ? b0 : (j == 1 ? b1 : bb);
                    msg[p * 3 + j] = log_col(T, j, b0, b1, bb);
                }
                // the lanes of a wave see each other's LDS writes in program order
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                __builtin_amdgcn_wave_barrier();
            }
            a = b;
            b = b2;
        }
    }
    __syncthreads();
    // every node's draw for each class of its parent; the root's has the prior (1/2, 1/2, 0) and no parent
    LDS uint8_t *zn = (LDS uint8_t *)msg;
    const int n_item = 3 * (n_nodes - 1) + 1;
    for (int i = tid; i < n_item; i += BS) {
        const int q = i / 3, zp = i - 3 * q, s = nodes[q];
        const LDS double *T = fixZ[s] ? TMf : TMn;
        const bool rt = q == n_nodes - 1;
        const double y0 = (rt ? log(0.5) : T[0 * 3 + zp]) + beta[s * 3], y1 = (rt ? log(0.5) : T[1 * 3 + zp]) + beta[s * 3 + 1],
                     y2 = (rt ? -INFINITY : T[2 * 3 + zp]) + beta[s * 3 + 2];
        const double mx = fmax(y0, fmax(y1, y2));
        double pr[3];
        exp3(y0, y1, y2, mx, pr[0], pr[1], pr[2]);
        zn[s * 4 + zp] = (uint8_t)categorical<3>(pr, slot_uniform(key, 0, c2, c3, (uint32_t)(n_nodes - 1 - q)));
    }
    __syncthreads();
    const LDS uint32_t *znw = (const LDS uint32_t *)msg;
    const int z_root = uni((int)zn[root * 4]);
    for (int q = tid; q < n_nodes; q += BS) {
        const int s = nodes[q];
        int z = z_root;
        if (s != root) {
            // w: the node's class for each class of the ancestor reached so far
            uint32_t w = znw[s];
            int a = par[s];
            while (a != root) {
                const uint32_t f = znw[a];
                const int up = par[a];
                w = ((w >> (8 * (f & 3))) & 3) | ((w >> (8 * ((f >> 8) & 3)) & 3) << 8) | ((w >> (8 * ((f >> 16) & 3)) & 3) << 16);
                a = up;
            }
            z = (w >> (8 * z_root)) & 3;
        }
        if (c->Z[s] == z) continue;
        c->Z[s] = (int8_t)z;
        c->changed[s] = 1;
        c->nch = 1;     // every writer stores the same value
        // dirty = strict ancestors of changed nodes (getUpdateNode, bpp_c.cpp:620-642)
        for (int a = par[s]; a != N; a = par[a]) c->dirty[a] = 1;
    }
    __syncthreads();
}

// ------------------------------------------------------------- rate update

// log_TM_Int, [i*3+j] = log P(child i | parent j), the six logarithms a lane
// each (lane < 64 of one wave).  fixZ nodes (bpp_c.cpp:305-316, 577-585):
// column 2 is never set there and keeps its initial log 1 (a fixZ node's
// parent is never accelerated, so it is unused).
__device__ __forceinline__ void set_TM(LDS double *F, LDS double *T, double g, double l, double l2, int lane)
{
    const double y = 1 - l;   // the reference forms P(1 -> 2) as 1 - (1 - l)
    const double x = lane == 0 ? 1 - g : lane == 1 ? g : lane == 2 ? y : lane == 3 ? 1 - y : lane == 4 ? l2 : 1 - l2;
    const double v = log(x);
    if (lane == 0) { F[0] = v; T[0] = v; F[6] = F[1] = F[7] = T[6] = T[1] = T[2] = -INFINITY; }
    else if (lane == 1) { F[3] = v; T[3] = v; F[4] = F[2] = F[5] = F[8] = 0; }
    else if (lane == 2) T[4] = v;
    else if (lane == 3) T[7] = v;
    else if (lane == 4) T[5] = v;
    else if (lane == 5) T[8] = v;
}

// The gamma variates of one sweep, drawn together by one wave (a draw is a
// long chain of FP64 functions, so its time is the same for one lane or
// eight): lanes 0-5 those of the three transition Beta draws
// (BPP_C::sample_transition, src/PhyloAcc-ST/bpp_c.cpp:522-613;
// Beta(a, b) = X / (X + Y), X ~ Gamma(a) on sub-stream 2k, Y ~ Gamma(b) on
// sub-stream 2k + 1, the l2 pair not drawn when its prior is off), lane 6 the
// accelerated rate's proposal (bpp_c.cpp:1000-1010) or, when no branch
// carries the class, its prior draw, lane 7 the conserved rate's prior draw.
// Each variate has its own stream, so drawing early changes none.  The counts
// cnt9 and has_cls are those of the Z the rates are drawn under.
enum { GV_R2 = 6, GV_R1 = 7, GV_N = 8 };

template <typename R>
__device__ __noinline__ void draw_gammas(MP M, CP<R> c, int ms, int m, int resZ)
{
    const int j = threadIdx.x;
    const Key key{M->key0, M->key1};
    double n[9], nf[9];
    for (int i = 0; i < 9; i++) { n[i] = c->cnt9[i]; nf[i] = n[i] - c->cnt9[9 + i]; }
    double shape, scale = 1.0;
    uint32_t sub = (uint32_t)j, c3 = tagword(ms, TAG_TRANS);
    bool on = true;
    switch (j) {
    case 0: shape = M->ha_g + n[1 * 3 + 0] + n[2 * 3 + 0]; break;
    case 1: shape = M->hb_g + n[0]; break;
    case 2: shape = M->ha_l + nf[2 * 3 + 1]; break;
    case 3: shape = M->hb_l + nf[1 * 3 + 1]; break;
    case 4: shape = M->ha_l2 + nf[1 * 3 + 2]; on = M->ha_l2 != 0; break;
    case 5: shape = M->hb_l2 + nf[2 * 3 + 2]; on = M->ha_l2 != 0; break;
    case GV_R2:
        c3 = tagword(ms, TAG_R2);
        if (c->has_cls[1]) {
            shape = c->nrate / c->prop_n;
            scale = c->prop_n;
            sub = 1;
        } else {
            shape = M->nprior_a;
            scale = M->nprior_b;
            sub = 2;
            on = resZ != 0;
        }
        break;
    default:
        c3 = tagword(ms, TAG_R1);
        shape = M->cprior_a;
        scale = M->cprior_b;
        sub = 2;
        on = !c->has_cls[0] && resZ != 0;
        break;
    }
    double x = 0.0;
    int capped = 0;
    if (on) {
        Stream st{key, sub, (uint32_t)m, c3, 0};
        x = gamma_draw(st, shape, scale, &capped);
    }
    if (capped) __hip_atomic_fetch_or(&c->fail, PA_F_SAMPLER, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    c->gam[j] = x;
}

// Scalar head of BPP_C::sample_rate (src/PhyloAcc-ST/bpp_c.cpp:930-1041), one
// lane: the prior draw when no branch carries the class, else the proposal
// and its range checks.
template <typename R>
__device__ __forceinline__ void rate_propose(MP M, CP<R> c, int ms, int m, int resZ, bool neut)
{
    const double old = neut ? c->nrate : c->crate;
    c->old_rate = old;
    const Key key{M->key0, M->key1};
    const uint32_t c3 = tagword(ms, neut ? TAG_R2 : TAG_R1), c2 = (uint32_t)m;
    double cur = old;
    c->skip = 1;
    c->accept = 0;
    if (!c->has_cls[neut ? 1 : 0]) {
        if (resZ != 0) {
            cur = c->gam[neut ? GV_R2 : GV_R1];
            if (neut) {
                if (M->ropt == 1 && cur < M->nlb) cur = old;
                else if (M->ropt == 2 && cur < c->crate) cur = old;
            } else {
                if (M->ropt == 1 && cur > M->cub) cur = old;
                else if (M->ropt == 2 && cur > c->nrate) cur = old;
            }
        }
    } else {
        const double r = slot_uniform(key, 0, c2, c3, 0);
        double prop;
        int skip = 0;
        if (neut) {
            prop = c->gam[GV_R2];
            if (M->ropt == 1 && prop < M->nlb) skip = 1;
            else if (M->ropt == 2 && prop < c->crate) skip = 1;
        } else {
            const double ru = M->r1_shared ? r : slot_uniform(key, 1, c2, c3, 0);
            const double u = ru * (c->prop_c - 1 / c->prop_c) + 1 / c->prop_c;
            prop = cur * u;
            if (M->ropt == 1 && prop > M->cub) skip = 1;
            else if (M->ropt == 2 && prop > c->nrate) skip = 1;
        }
        if (!skip && (prop < 1e-12 || prop > 1e8)) {
            skip = 1;
            c->fail |= PA_F_PROPOSAL_RANGE;   // the reference's out-of-range warning (bpp_c.cpp:1024-1041)
        }
        c->skip = skip;
        c->proposal = prop;
        c->r = r;
    }
    if (neut) c->nrate = cur; else c->crate = cur;
}

// The terms of the Metropolis ratio (bpp_c.cpp:1046-1094) that do not need
// the proposal's likelihood, a lane each, FP64: the prior densities of the
// proposal and the old rate, the proposal densities (r2) or the logarithms
// (r1) of the two, and the log of the acceptance uniform.
template <typename R>
__device__ __noinline__ void rate_terms(MP M, CP<R> c, bool neut, double old, int lane)
{
    if (lane >= 5) return;
    const double prop = c->proposal, x = (lane == 1 || lane == 2) ? old : prop;
    double a = neut ? M->nprior_a : M->cprior_a, b = neut ? M->nprior_b : M->cprior_b;
    if (lane == 2) { a = prop / c->prop_n; b = c->prop_n; }
    else if (lane == 3) { a = old / c->prop_n; b = c->prop_n; }
    double t;
    if (lane == 4) t = log(c->r);
    else if (!neut && lane >= 2) t = log(x);
    else t = log_gamma_pdf(x, a, b);
    c->mh[lane] = t;
}

// Metropolis decision (bpp_c.cpp:1046-1094), FP64.
template <typename R>
__device__ __forceinline__ void rate_decide(CP<R> c, bool neut, double lnew)
{
    const double MH = lnew - c->loglik + c->mh[0] - c->mh[1] + c->mh[2] - c->mh[3];
    if (c->mh[4] < MH) {
        c->accept = 1;
        c->loglik = lnew;
        if (neut) c->nrate = c->proposal; else c->crate = c->proposal;
    }
}

// Adaptive proposal scale (bpp_c.cpp:1144-1171).
template <typename R>
__device__ __noinline__ void rate_adapt(MP M, CP<R> c, int m, bool neut)
{
    if ((m + 1) % M->adapt_freq != 0) return;
    double fac = 1 / sqrt((double)((m + 1) / M->adapt_freq));
    if (fac > 0.5) fac = 0.5;
    if (neut) {
        const double ar = (double)c->accept_n / M->adapt_freq;
        const double adj = ar > 0.44 ? exp(fac) : (ar < 0.23 ? exp(-fac) : 1);
        c->prop_n = c->prop_n * adj;
        if (c->prop_n > 1) c->prop_n = 1;
        c->accept_n = 0;
    } else {
        const double ar = (double)c->accept_c / M->adapt_freq;
        const double adj = ar > 0.44 ? exp(fac) : (ar < 0.23 ? exp(-fac) : 1);
        c->prop_c = pow(c->prop_c, adj);
        if (c->prop_c < 1.0001) c->prop_c = 1.0001;
        c->accept_c = 0;
    }
}

template <typename R, int BS, int SH>
__device__ __noinline__ void build_prop_tables(MP M, CP<R> c, int cls, double prop)
{
    const int n_item = 4 * (uni(c->n_nodes) - 1);
    const LDS int16_t *nodes = uni_ptr(c->nodes);
    const GBL double *dist2 = uni_ptr(c->dist2);
    for (int it = threadIdx.x; it < n_item; it += BS) {
        const int s = nodes[it >> 2], j = it & 3;
        if (c->Z[s] != cls || (c->flags[s] & NF_MISSING)) continue;     // a whole quad
        double row[4];
        ptrans_row(&M->lam[0], dist2[s] * prop, j, row);
        LDS R *dst = c->PTp + 16 * s;
#pragma unroll
        for (int i = 0; i < 4; i++) dst[i * 4 + j] = (R)row[i];
    }
}

// dirty (cleared before) = ancestors of the branches of a class
template <typename R, int BS, int SH>
__device__ __noinline__ void mark_class(CP<R> c, int cls)
{
    const int N = uni(c->N), n_nodes = uni(c->n_nodes);
    const LDS int16_t *nodes = uni_ptr(c->nodes), *par = uni_ptr(c->par);
    LDS uint8_t *dirty = uni_ptr(c->dirty);
    for (int q = threadIdx.x; q < n_nodes; q += BS) {
        const int s = nodes[q];
        if ((c->flags[s] & NF_MISSING) || c->Z[s] != cls) continue;
        for (int j = par[s]; j != N; j = par[j]) dirty[j] = 1;
    }
}

// BPP_C::getUpdateNode(neut) + BPP_C::sample_rate (src/PhyloAcc-ST/bpp_c.cpp:836-858, 930-1176)
template <typename R, int BS, int SH>
__device__ __forceinline__ void sample_rate(MP M, CP<R> c, int ms, int m, int resZ, bool neut)
{
    const int tid = threadIdx.x;
    const int cls = neut ? 2 : 1;
    if (c->has_cls[neut ? 1 : 0])
        for (int q = tid; q < c->n_nodes; q += BS) c->dirty[c->nodes[q]] = 0;
    if (tid == 0) rate_propose<R>(M, c, ms, m, resZ, neut);
    __syncthreads();
    const double old = c->old_rate;
    if (!c->skip) {
        mark_class<R, BS, SH>(c, cls);
        build_prop_tables<R, BS, SH>(M, c, cls, c->proposal);
        if (tid >= BS - 64) rate_terms<R>(M, c, neut, old, tid - (BS - 64));
        __syncthreads();
        const double lnew = prune<R, BS, SH>(M, c, PR_PROP, cls);
        if (tid == 0) rate_decide<R>(c, neut, lnew);
        __syncthreads();
        if (c->accept) {
            for (int q = tid; q < c->n_int; q += BS) {
                const int s = c->inodes[q];
                if (c->dirty[s] && !(c->flags[s] & NF_MISSING)) {
                    const int cu = c->cur[s] ^ 1;
                    c->cur[s] = (uint8_t)cu;
                    LDS uint32_t *r1 = c->srec + 2 * (c->n_int - 1 - q) + 1;
                    if (!(c->flags[s] & NF_CHERRY)) *r1 = (*r1 & ((1u << SR_SLOT_SHIFT) - 1)) | (uint32_t)(cu * c->I + s - c->S) << SR_SLOT_SHIFT;
                }
            }
        }
    }
    const double now = neut ? c->nrate : c->crate;
    if (now != old) class_tables<R, BS>(M, c, cls, now, 1);
    if (tid == 0) {
        if (now != old) { if (neut) c->accept_n += 1; else c->accept_c += 1; }
        rate_adapt<R>(M, c, m, neut);
    }
    __syncthreads();
}

// The Z-transition counts and which rate classes any branch carries, then the
// sweep's gamma variates and the transition probabilities they give
// (BPP_C::sample_transition, src/PhyloAcc-ST/bpp_c.cpp:522-613).  Both depend
// on Z alone, so they follow the Z update.
template <typename R, int BS, int SH>
__device__ __forceinline__ void sample_transition(MP M, CP<R> c, int ms, int m, int resZ)
{
    const int tid = threadIdx.x;
    if (tid < 18) c->cnt9[tid] = 0;
    if (tid < 2) c->has_cls[tid] = 0;
    __syncthreads();
    for (int q = tid; q < c->n_nodes - 1; q += BS) {
        const int s = c->nodes[q];
        const int zi = c->Z[s], zp = c->Z[c->par[s]];
        lds_add(&c->cnt9[zi * 3 + zp], 1u);
        if (c->fixZ[s]) lds_add(&c->cnt9[9 + zi * 3 + zp], 1u);
        if (zi > 0 && !(c->flags[s] & NF_MISSING)) c->has_cls[zi - 1] = 1;     // every writer stores the same value
    }
    __syncthreads();
    if (tid < GV_N) draw_gammas<R>(M, c, ms, m, resZ);
    __syncthreads();
    if (tid < 64) {
        const double g = c->gam[0] / (c->gam[0] + c->gam[1]);
        const double l = c->gam[2] / (c->gam[2] + c->gam[3]);
        const double l2 = M->ha_l2 == 0 ? 0.0 : c->gam[4] / (c->gam[4] + c->gam[5]);
        if (tid == 0) { c->g = g; c->l = l; c->l2 = l2; }
        set_TM(c->TMf, c->TMn, g, l, l2, tid);
    }
    __syncthreads();
}

// ---------------------------------------------------------- element setup

// A cherry: a non-root internal node whose children are both leaves (tab: the
// element's node table in global memory).
__device__ __forceinline__ bool is_cherry(const int32_t *tab, int N, int S, int root, int x)
{
    return x >= S && x != root && tab[tab_ch0(N) + x] < S && tab[tab_ch1(N) + x] < S;
}

// The static pruning descriptor of internal node s (layout at DB_*).
__device__ __forceinline__ uint32_t node_desc(const int32_t *tab, int N, int S, int root, int s)
{
    const int x[2] = {tab[tab_ch0(N) + s], tab[tab_ch1(N) + s]};
    uint32_t d = 0;
    for (int j = 0; j < 2; j++) {
        if (x[j] < 0) continue;
        const int kind = x[j] < S ? KD_LEAF : (is_cherry(tab, N, S, root, x[j]) ? KD_CHERRY : KD_STORED);
        d |= (uint32_t)x[j] << (j ? DB_KID1_SHIFT : 0) | (uint32_t)kind << (j ? DB_KIND1_SHIFT : DB_KIND0_SHIFT);
        if (tab[tab_flags(N) + x[j]] & NF_MISSING) d |= j ? DB_MISS1 : DB_MISS0;
    }
    return d;
}

template <typename R, int BS, int SH>
__device__ __noinline__ void bind_element(MP M, CP<R> c, const ChainArgs *A, int work)
{
    const int tid = threadIdx.x, N = M->N;
    const ElemDev E = A->elems[A->work[work]];
    if (tid == 0) {
        c->S = M->S; c->N = N; c->I = M->I;
        c->GG = E.GG; c->P = E.P; c->Ppad = E.Ppad; c->root = E.root;
        c->n_nodes = E.n_nodes; c->n_int = E.n_int; c->n_up = E.n_up; c->has_amb = E.has_amb;
        c->codes = (const GBL uint8_t *)(A->codes + E.off_codes);
        c->wts = (const GBL int32_t *)(A->wts + E.off_w);
        c->site = (const GBL int32_t *)(A->site + E.off_site);
        char *base = A->scratch + (size_t)blockIdx.x * A->slot_bytes;
        const int64_t bo = A->big_off ? A->big_off[work] : -1;
        char *pbase = bo >= 0 ? A->big + bo : base + A->off_parts;
        c->parts = (GBL char *)pbase;
        c->plin = (GBL double *)(base + A->off_plin);
        c->logt = (GBL double *)(base + A->off_logt);
        c->amb = (GBL uint32_t *)(base + A->off_amb);
        c->dist2 = (const GBL double *)(A->tab + E.off_tab + tab_dist(N));
        c->accept_n = 0;
        c->accept_c = 0;
        c->bytes = 0;
    }
    const int32_t *tab = A->tab + E.off_tab;
    for (int i = tid; i < N; i += BS) {
        c->par[i] = (int16_t)tab[tab_par(N) + i];
        // the cherry bit with the rest: the step lists of other waves' threads read it behind the next barrier
        const int f = tab[tab_flags(N) + i];
        c->flags[i] = (uint8_t)(f | ((f & NF_IN_TREE) && is_cherry(tab, N, M->S, E.root, i) ? NF_CHERRY : 0));
        c->nodes[i] = (int16_t)tab[tab_nodes(N) + i];
        c->inodes[i] = (int16_t)tab[tab_int(N) + i];
        c->cur[i] = 0;
        c->dirty[i] = 0;
    }
    for (int i = tid; i < E.n_int; i += BS) c->porder[i] = (int16_t)((uint32_t)tab[tab_porder(N) + i] & PO_NODE);
    for (int i = tid; i < E.n_up; i += BS) c->upoff[i] = (int16_t)tab[tab_upoff(N) + i];
    for (int q = tid; q < E.n_int; q += BS) {
        const int v = tab[tab_up(N) + q];
        c->urec[q] = (uint32_t)v | ((uint32_t)tab[tab_ch0(N) + v] << 10) | ((uint32_t)tab[tab_ch1(N) + v] << 20);
    }
    for (int s = M->S + tid; s < N; s += BS) c->desc[s - M->S] = node_desc(tab, N, M->S, E.root, s);
    __syncthreads();
    sample_steps<R, BS>(c);
    // null-rate tables (rate 1), fixed for the element
    class_tables<R, BS>(M, c, 0, 1.0, 0);
    __syncthreads();
}

// ------------------------------------------------------------- the chain

template <typename R, int BS, int SH>
__device__ __noinline__ void init_model(MP M, CP<R> c, int resZ)
{
    // BPP_C::initMCMC (src/PhyloAcc-ST/bpp_c.cpp:131-343), iter = 0
    const int tid = threadIdx.x, N = M->N;
    for (int i = tid; i < N; i += BS) {
        c->Z[i] = -1;
        c->maxZ[i] = 0;
    }
    __syncthreads();
    const int root = c->root;
    for (int q = tid; q < c->n_nodes; q += BS) {
        const int s = c->nodes[q];
        const uint8_t f = c->flags[s];
        c->Z[s] = (s == root) ? 0 : 1;
        int fz = (f & NF_UPPER) || s == root;
        if (resZ == 2 && (f & NF_UPPER_CONS)) fz = 1;
        if (resZ == 0 && s != root) fz = 1;
        c->fixZ[s] = (uint8_t)fz;
        c->cur[s] = 0;
    }
    for (int t = tid; t < c->n_int; t += BS) {
        // every node's partial in buffer 0
        const int s = c->inodes[c->n_int - 1 - t], v = (c->flags[s] & (NF_MISSING | NF_CHERRY)) ? root : s;
        LDS uint32_t *r1 = c->srec + 2 * t + 1;
        *r1 = (*r1 & ((1u << SR_SLOT_SHIFT) - 1)) | (uint32_t)(v - c->S) << SR_SLOT_SHIFT;
    }
    if (tid == 0) {
        c->prop_c = 1.2;
        c->prop_n = (double)1 / c->GG * 10;
        c->max_loglik = -INFINITY;
        c->max_m = 0;
        c->nrate = M->init_nrate;
        c->crate = M->init_crate;
        c->g = M->init_grate; c->l = M->init_lrate; c->l2 = M->ha_l2 == 0 ? 0.0 : M->init_lrate2;
        c->fail = 0;
    }
    if (tid < 64) set_TM(c->TMf, c->TMn, M->init_grate, M->init_lrate, M->ha_l2 == 0 ? 0.0 : M->init_lrate2, tid);
    __syncthreads();
    const double cr = c->crate, nr = c->nrate;
    class_tables<R, BS>(M, c, 1, cr, 0);
    class_tables<R, BS>(M, c, 2, nr, 0);
    __syncthreads();
    refresh_PTc<R, BS, SH>(c, false);
    __syncthreads();
}

// BPP_C::MonitorChain (src/PhyloAcc-ST/bpp_c.cpp:741-834), one wave: the two
// prior densities a lane each
template <typename R>
__device__ __noinline__ void monitor(MP M, CP<R> c, int m, int resZ, double *trd, int T, int lane)
{
    const double loglik = c->loglik, nrate = c->nrate, crate = c->crate;
    const bool neut = lane & 1;
    const double d = log_gamma_pdf(neut ? nrate : crate, neut ? M->nprior_a : M->cprior_a, neut ? M->nprior_b : M->cprior_b);
    double full = loglik + __shfl(d, 0, 64);
    const double dn = __shfl(d, 1, 64);
    if (resZ != 0) full += dn;
    if (trd && lane == 0) {
        trd[0 * T + m] = loglik; trd[1 * T + m] = full; trd[2 * T + m] = nrate;
        trd[3 * T + m] = crate; trd[4 * T + m] = c->g; trd[5 * T + m] = c->l; trd[6 * T + m] = c->l2;
    }
    if (m >= M->burnin && full > c->max_loglik) {
        for (int i = lane; i < M->N; i += 64) c->maxZ[i] = c->Z[i];
        if (lane == 0) {
            c->max_loglik = full;
            c->max_m = m;
        }
    }
    if (lane == 0) {
        if (isnan(loglik)) c->fail |= PA_F_NAN;
        else if (isinf(loglik)) c->fail |= loglik > 0 ? PA_F_POS_INF : PA_F_NEG_INF;
    }
}

template <typename R, int BS, int SH>
__device__ __noinline__ void write_results(MP M, CP<R> c, const ChainArgs *A, int ms, int work)
{
    const int tid = threadIdx.x, N = M->N;
    if (tid == 0) {
        double *rd = A->res_d + ((size_t)work * 3 + ms) * RES_D;
        int32_t *ri = A->res_i + ((size_t)work * 3 + ms) * RES_I;
        rd[0] = c->max_loglik; rd[1] = c->nrate; rd[2] = c->crate; rd[3] = c->g; rd[4] = c->l; rd[5] = c->l2;
        const bool failed = (c->fail & (PA_F_NAN | PA_F_POS_INF | PA_F_SAMPLER)) || !isfinite(c->max_loglik);
        ri[0] = c->max_m; ri[1] = failed ? PA_STATUS_NUMERIC_FAIL : 0; ri[2] = c->accept_n; ri[3] = c->accept_c;
        ri[4] = c->fail;
    }
    int8_t *mz = A->maxZ + ((size_t)work * 3 + ms) * N;
    for (int i = tid; i < N; i += BS) mz[i] = c->maxZ[i];
}

template <typename R, int BS, int SH>
__device__ __forceinline__ void run_model(MP M, CP<R> c, const ChainArgs *A, int ms, int work)
{
    const int tid = threadIdx.x;
    const int resZ = ms == 0 ? 0 : (ms == 1 ? 2 : 1);
    const int T = M->T, N = M->N;
    init_model<R, BS, SH>(M, c, resZ);
    {
        const double l0 = prune<R, BS, SH>(M, c, PR_FULL, 0);
        if (tid == 0) c->loglik = l0;
        __syncthreads();
    }
    double *trd = A->tr_d ? A->tr_d + ((size_t)work * 3 + ms) * 7 * T : nullptr;
    int8_t *trz = A->tr_Z ? A->tr_Z + ((size_t)work * 3 + ms) * (size_t)T * N : nullptr;
    for (int m = 0; m < T; m++) {
        if (trz)
            for (int i = tid; i < N; i += BS) trz[(size_t)m * N + i] = c->Z[i];
        // the last wave, which has the fewest sites to draw
        if (tid >= BS - 64) monitor<R>(M, c, m, resZ, trd, T, tid - (BS - 64));
        if (m == T - 1) break;
        sample_sites<R, BS, SH>(M, c, (uint32_t)m, tagword(ms, TAG_ANC));
        __syncthreads();
        emissions<R, BS, SH>(c);
        __syncthreads();
        update_Z<R, BS, SH>(M, c, (uint32_t)m, tagword(ms, TAG_Z));
        refresh_PTc<R, BS, SH>(c, true);
        __syncthreads();
        if (c->nch) {
            const double l = prune<R, BS, SH>(M, c, PR_DIRTY, 0);
            if (tid == 0) c->loglik = l;
            __syncthreads();
        }
        sample_transition<R, BS, SH>(M, c, ms, m, resZ);
        sample_rate<R, BS, SH>(M, c, ms, m, resZ, true);
        sample_rate<R, BS, SH>(M, c, ms, m, resZ, false);
    }
    __syncthreads();
    write_results<R, BS, SH>(M, c, A, ms, work);
    __syncthreads();
}

__device__ __forceinline__ MP model_to_lds(const ModelDev &Mk, LDS ModelDev *Ms)
{
    const uint32_t *src = (const uint32_t *)&Mk;
    LDS uint32_t *dst = (LDS uint32_t *)Ms;
    for (int i = threadIdx.x; i < (int)(sizeof(ModelDev) / 4); i += blockDim.x) dst[i] = src[i];
    return (MP)Ms;
}

template <typename R, int BS, int SH>
__global__ void __launch_bounds__(BS, 4) chain_kernel(ModelDev Mk, ChainArgs A)
{
    extern __shared__ __align__(16) char smem_raw[];
    __shared__ ModelDev Ms;
    __shared__ Ctx<R> Cs;
    MP M = model_to_lds(Mk, (LDS ModelDev *)&Ms);
    CP<R> c = (CP<R>)&Cs;
    __syncthreads();
    if (threadIdx.x == 0) smem_arrays<R, true>(M->N, M->S, BS, (LDS char *)smem_raw, c);
    __syncthreads();
    for (;;) {
        if (threadIdx.x == 0) c->work = atomicAdd(A.queue, 1);
        __syncthreads();
        const int w = c->work;
        __syncthreads();
        if (w >= A.n_work) break;
        bind_element<R, BS, SH>(M, c, &A, w);
        for (int ms = 0; ms < 3; ms++) run_model<R, BS, SH>(M, c, &A, ms, w);
        if (threadIdx.x == 0 && A.counters) atomicAdd(A.counters, c->bytes);
        if (threadIdx.x == 0 && A.done) {
            // thread 0 wrote the result rows: make them visible to the host
            // before the flag that announces them
            __threadfence_system();
            __hip_atomic_store(A.done + w, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    }
}

__global__ void reset_queue(int *q) { *q = 0; }

template <typename R, int BS, int SH>
static hipError_t launch_t(const ModelDev &M, const ChainArgs &A, int grid, hipStream_t st)
{
    const size_t sm = smem_arrays<R, false>(M.N, M.S, BS, nullptr, nullptr);
    const hipError_t err = hipFuncSetAttribute((const void *)chain_kernel<R, BS, SH>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)sm);
    if (err != hipSuccess) return err;
    hipLaunchKernelGGL((chain_kernel<R, BS, SH>), dim3(grid), dim3(BS), sm, st, M, A);
    return hipGetLastError();
}

hipError_t launch_reset(int *q, hipStream_t st)
{
    hipLaunchKernelGGL(reset_queue, dim3(1), dim3(1), 0, st, q);
    return hipGetLastError();
}

// Zeroes n 32-bit words: a kernel, so that it can be captured in a HIP graph
// where a memset node would not be used.
__global__ void clear_words(uint32_t *p, int n)
{
    for (int i = threadIdx.x; i < n; i += blockDim.x) p[i] = 0;
}

hipError_t launch_clear(void *p, int words, hipStream_t st)
{
    hipLaunchKernelGGL(clear_words, dim3(1), dim3(64), 0, st, (uint32_t *)p, words);
    return hipGetLastError();
}

template <typename R, int BS, int SH>
static int blocks_t(int N, int S)
{
    const size_t sm = smem_arrays<R, false>(N, S, BS, nullptr, nullptr);
    if (hipFuncSetAttribute((const void *)chain_kernel<R, BS, SH>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)sm) != hipSuccess)
        return 0;
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, chain_kernel<R, BS, SH>, BS, sm) != hipSuccess) return 0;
    return nb;
}

// Runtime (precision, block size, shape) -> template instance.
template <typename R, int SH, typename F>
static auto by_block(int BS, F &&f) -> decltype(f(std::integral_constant<int, 64>()))
{
    if (BS == 64) return f(std::integral_constant<int, 64>());
    if (BS == 128) return f(std::integral_constant<int, 128>());
    return f(std::integral_constant<int, 256>());
}

template <typename R, typename F>
static auto by_shape(int shape, F &&f) -> decltype(f(std::integral_constant<int, 0>()))
{
    if (shape == 2) return f(std::integral_constant<int, 2>());
    return f(std::integral_constant<int, 0>());
}

template <typename R>
static int blocks_r(int BS, int shape, int N, int S)
{
    return by_shape<R>(shape, [&](auto sh) {
        return by_block<R, decltype(sh)::value>(BS, [&](auto bs) { return blocks_t<R, decltype(bs)::value, decltype(sh)::value>(N, S); });
    });
}

template <typename R>
static hipError_t launch_r(const ModelDev &M, const ChainArgs &A, int BS, int shape, int grid, hipStream_t st)
{
    return by_shape<R>(shape, [&](auto sh) {
        return by_block<R, decltype(sh)::value>(BS, [&](auto bs) {
            return launch_t<R, decltype(bs)::value, decltype(sh)::value>(M, A, grid, st);
        });
    });
}

int chain_blocks_per_cu(int fp64, int BS, int N, int S, int shape)
{
    if ((BS != 64 && BS != 128 && BS != 256) || shape < 0 || shape >= N_SHAPES) return 0;
    return fp64 ? blocks_r<double>(BS, shape, N, S) : blocks_r<float>(BS, shape, N, S);
}

hipError_t launch_chain(const ModelDev &M, const ChainArgs &A, int fp64, int BS, int grid, hipStream_t st, int shape)
{
    if ((BS != 64 && BS != 128 && BS != 256) || shape < 0 || shape >= N_SHAPES) return hipErrorInvalidValue;
    return fp64 ? launch_r<double>(M, A, BS, shape, grid, st) : launch_r<float>(M, A, BS, shape, grid, st);
}

}  // namespace chain
}  // namespace pa
