// pa_engine.hip -- CDNA4 (gfx950) log-likelihood kernels: the element's
// log-likelihood at fixed ancestral states Z and rates (r1, r2), or at
// per-call branch lengths for an element with its own tree
// (BPP_C::log_f_Xz, src/PhyloAcc-ST/bpp_c2.cpp:392-425).  The MCMC chains
// are in pa_chain.hip.
//
// One workgroup owns one element (or part of a long one) at a time;
// workgroups pull work from a device counter (persistent kernel).  Within a
// workgroup:
//   * each branch's 4x4 transition matrix P(t * rate of its class) is built
//     in FP64 by a quad of lanes, a row a lane, and stored in LDS in the
//     partials' precision;
//   * the pass is a list of steps (pa_prune.h), a pattern a lane; a thread
//     keeps its patterns through the whole pass, so no barrier is needed
//     between tree nodes;
//   * conditional likelihoods are linear-space with a power-of-two rescale
//     per node; the cumulative exponent rides along as an int; GAPT marks
//     all-gap subtrees (the reference's Tg >= num_base,
//     src/PhyloAcc-ST/bpp_c.hpp:417-428);
//   * the root sum over patterns is FP64 with a fixed reduction order.
// score_kernel keeps no partials; keep_kernel stores every node's (but the
// cherries', which are recomputed where they are read) for the gene-tree
// moves that read them.
// No matrix instructions: 4x4x1 ones gave the FP32 messages bit for bit and
// took vector instructions from 437 M to 269 M in 8,000 elements of 120
// leaves, but 817 -> 835 us: a step waits on latency, not on the vector units.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "pa_common.h"
#include "pa_kernels.h"
#include "pa_device.h"
#include "pa_prune.h"
#include "pa_eig.h"
#include "pa_rng.h"

#include <mutex>

namespace pa {

// Scratch of the allocation-free likelihood entry point: the work counter in
// its first 256 bytes, then one slot per workgroup.  Every GPU the library
// runs on holds its own copy until the process ends.  Host code must never
// use the array's name as an address (on the host it is a stand-in symbol);
// it uses the device address from noalloc_scratch().
static __device__ __align__(256) char scratch[NOALLOC_SCRATCH_BYTES];

hipError_t noalloc_scratch(int device, char **ptr)
{
    static std::mutex mu;
    static char *addr[64] = {nullptr};
    if (device < 0 || device >= 64) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(mu);
    if (!addr[device]) {
        // the caller has made `device` current
        void *p = nullptr;
        const hipError_t err = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (err != hipSuccess) return err;
        addr[device] = (char *)p;
    }
    *ptr = addr[device];
    return hipSuccess;
}

using MP = LDS const ModelDev *;
using AP = LDS const LoglikArgs *;

__host__ __device__ inline size_t al(size_t x, size_t a) { return (x + a - 1) & ~(a - 1); }

// A slot of a launch that keeps partials: blocks of 64 patterns with a slot
// per internal node.
size_t loglik_slot_bytes(int N, int S, int Pcap, int fp64)
{
    return al((size_t)(Pcap / 64) * block_bytes(N - S, fp64 ? 8 : 4), 256);
}

// Resident partials: the blocks, then the patterns' root terms.
size_t loglik_resident_bytes(int N, int S, int Ppad, int fp64)
{
    return loglik_slot_bytes(N, S, Ppad, fp64) + al((size_t)Ppad * 8, 256);
}

// ------------------------------------------------------------------ helpers

// An element's record in scalar registers.  What is read through a pointer
// held in LDS is not known to be the same in every lane, and a buffer made
// from it would be used lane group by lane group, in a loop around every load.
__device__ __forceinline__ ElemDev uni_elem(const ElemDev *e)
{
    ElemDev E;
    const uint32_t *src = (const uint32_t *)e;
    uint32_t w[sizeof(ElemDev) / 4];
#pragma unroll
    for (int i = 0; i < (int)(sizeof(ElemDev) / 4); i++) w[i] = (uint32_t)uni((int)src[i]);
    __builtin_memcpy(&E, w, sizeof E);
    return E;
}


// A work position's own eigensystems (the gBGC classes of its row, or its
// element's base frequencies) are kept in LDS behind the rest.
size_t loglik_eig_bytes(const LoglikArgs &A) { return A.gb_eig ? GB_CLASSES * GB_EIG_WORDS * 8 : A.el_eig ? GB_EIG_WORDS * 8 : 0; }

__device__ __forceinline__ void fetch_eig(AP A, LDS double *eig, int w, int row)
{
    const double *src = A->gb_eig ? A->gb_eig + (size_t)row * GB_CLASSES * GB_EIG_WORDS : A->el_eig ? A->el_eig + (size_t)w * GB_EIG_WORDS : nullptr;
    const int words = A->gb_eig ? GB_CLASSES * GB_EIG_WORDS : A->el_eig ? GB_EIG_WORDS : 0;
    for (int i = threadIdx.x; i < words; i += blockDim.x) eig[i] = src[i];
}

// Row j of the matrix of branch s, of length d, into PT (PT[16 s + 4 i + j] =
// P_{j->i}), by lane j of a quad (ptrans_row): P(d * rate) in FP64 for length d > 1e-10,
// else the identity (BPP_C::initMats, src/PhyloAcc-ST/bpp_c.cpp:187-228).  A
// thread a matrix took its 16 entries and four exponentials in turn (about
// 1,200 instructions, and registers for an eigensystem), with most of a
// workgroup idle.  A branch takes the rate of its class: Z = 0 (neutral) rate
// 1, Z = 2 (accelerated) r2, any other Z (1, conserved) r1; an own-tree
// element takes its lengths from len_in.
template <typename R>
__device__ __forceinline__ void work_matrix_row(MP M, AP A, const LDS double *eig, LDS R *PT, double d, int cls, int s, int j, int row)
{
    const LDS double *E = &M->lam[0];
    double rate = 1.0;
    if (A->len_in) {
        if (A->el_eig) E = eig;
    } else {
        const int z = cls & 3;
        if (A->gb_eig) E = eig + (z + (cls & 4 ? 3 : 0)) * GB_EIG_WORDS;
        else rate = z == 2 ? A->rates_in[2 * row + 1] : (z == 0 ? 1.0 : A->rates_in[2 * row]);
    }
    double r[4];
    ptrans_row(E, d * rate, j, r);
    LDS R *dst = PT + 16 * s + j;
#pragma unroll
    for (int i = 0; i < 4; i++) dst[4 * i] = (R)(d <= 1e-10 ? (i == j ? 1.0 : 0.0) : r[i]);      // a NaN length gives a NaN matrix
}

// What a pass needs of node i, where its matrix will be: the length (double)
// and the class (0 neutral, 2 accelerated, 1 any other Z; + 4 with gBGC) of its
// branch.  Staged with every load in flight: a matrix read them one behind the
// other from memory, through the node list, in each of its workgroup's rounds
// (45 us of 270 an element of 120 leaves).
template <typename R>
__device__ __forceinline__ LDS double *node_len(LDS R *PT, int i) { return (LDS double *)(PT + 16 * i); }
template <typename R>
__device__ __forceinline__ LDS int32_t *node_int(LDS R *PT, int i) { return (LDS int32_t *)(PT + 16 * i) + 2; }

__device__ __forceinline__ int branch_class(AP A, int z, int b) { return A->len_in ? 0 : (z == 2 ? 2 : (z == 0 ? 0 : 1)) + (A->gb_eig && b != 0 ? 4 : 0); }

// gBGC classes (BPP_C::init_cache_TM, src/PhyloAcc-ST-GBGC/SRC/bpp_c.cpp:
// 1563-1621, with the rate matrices of Gibbs, bpp_c.cpp:191-197): one thread
// per (work position, class).
struct GbgcEigArgs {
    double Q0[16];
    const double *sel;
    int n;
    double *eig;
};

__global__ void gbgc_eig_kernel(GbgcEigArgs a)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= a.n * GB_CLASSES) return;
    const int w = t / GB_CLASSES, k = t % GB_CLASSES;
    const double *sel = a.sel + (size_t)w * 3;
    const double s = k % 3 == 0 ? 0.0 : (k % 3 == 1 ? sel[0] : sel[1]);
    const double b = k >= 3 ? sel[2] : 0.0;
    double Q[16], lam[4], V[16], Vi[16];
    gbgc_rate(a.Q0, s, b, Q);
    const int st = reversible_eig4(Q, lam, V, Vi);
    double *out = a.eig + (size_t)t * GB_EIG_WORDS;
    for (int i = 0; i < 4; i++) out[i] = st == EIG_OK ? lam[i] : NAN;
    for (int i = 0; i < 16; i++) {
        out[4 + i] = V[i];
        out[20 + i] = Vi[i];
    }
}

// Per-element strand-symmetric base frequencies (BPP_C::sample_pi and
// getQmat, src/PhyloAcc-GT/bpp_c.cpp:1545-1548,160-185): one thread per work
// position.
struct GtEigArgs {
    double inst[6];
    const double *piA;
    int n;
    double *eig, *pi;
};

__global__ void gt_eig_kernel(GtEigArgs a)
{
    const int w = blockIdx.x * blockDim.x + threadIdx.x;
    if (w >= a.n) return;
    double Q[16], pi[4], lam[4], V[16], Vi[16];
    gt_strand_q(a.inst, a.piA[w], Q, pi);
    const int st = reversible_eig4(Q, lam, V, Vi);
    double *out = a.eig + (size_t)w * GB_EIG_WORDS;
    for (int i = 0; i < 4; i++) out[i] = st == EIG_OK ? lam[i] : NAN;
    for (int i = 0; i < 16; i++) {
        out[4 + i] = V[i];
        out[20 + i] = Vi[i];
    }
    for (int i = 0; i < 4; i++) a.pi[(size_t)w * 4 + i] = pi[i];
}

hipError_t launch_gt_eig(const double *inst, const double *piA, int n, double *eig, double *pi, hipStream_t st)
{
    GtEigArgs a;
    for (int i = 0; i < 6; i++) a.inst[i] = inst[i];
    a.piA = piA;
    a.n = n;
    a.eig = eig;
    a.pi = pi;
    hipLaunchKernelGGL(gt_eig_kernel, dim3((n + 127) / 128), dim3(128), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_gbgc_eig(const double *Q0, const double *sel, int n, double *eig, hipStream_t st)
{
    GbgcEigArgs a;
    for (int i = 0; i < 16; i++) a.Q0[i] = Q0[i];
    a.sel = sel;
    a.n = n;
    a.eig = eig;
    const int threads = n * GB_CLASSES;
    hipLaunchKernelGGL(gbgc_eig_kernel, dim3((threads + 127) / 128), dim3(128), 0, st, a);
    return hipGetLastError();
}

// The log-likelihoods of work position w, by position and by caller row.
__device__ __forceinline__ void write_scores(AP A, int w, int row, double s0, double s1)
{
    A->ll_out[w] = s0;
    if (A->pre_len) A->ll_out2[w] = s1;
    if (A->row_out0) {
        A->row_out0[row] = s0;
        if (A->pre_len) A->row_out1[row] = s1;
    }
}

// Kernel arguments are copied to LDS once per workgroup: the device
// functions take LDS pointers to them, which keeps the argument blocks out of
// the private (scratch) segment.
template <typename T>
__device__ __forceinline__ LDS const T *to_lds(const T &k, LDS T *dst)
{
    static_assert(sizeof(T) % 4 == 0, "word copy");
    const uint32_t *src = (const uint32_t *)&k;
    LDS uint32_t *d = (LDS uint32_t *)dst;
    for (int i = threadIdx.x; i < (int)(sizeof(T) / 4); i += blockDim.x) d[i] = src[i];
    return (LDS const T *)dst;
}

// ------------------------------------------------------------- scores only
//
// A launch that wants nothing but log-likelihoods (no histories, candidate
// scores or resident partials) keeps no partials: a pass over the element's
// nodes in pruning order holds the one or two it needs next in registers,
// and a node whose parent comes later waits in a stack of a few slots per
// wave.  What is left is the latency of a step (about 1,500 cycles at the four
// waves a SIMD that 128 registers allow, half of them waiting), no longer
// storing and reloading every node: 8,000 elements of 120 leaves, FP32 3.40 ms
// before and 0.77 now, 5,000 of 43 leaves, FP64 0.94 and 0.29.  Three waves a
// SIMD took 0.39 ms where four took 0.36 (FP64), five 0.95 where four took 0.85
// (FP32, spills).

constexpr int SCORE_DEPTH = 4;      // steps a leaf code is loaded ahead

// Stack slots of a wave for trees of I internal nodes (the depth of a waiting
// partial is below log2 of the nodes, see PO_WAITS).
__host__ __device__ inline int score_slots(int I)
{
    int d = 1;
    while ((1 << d) <= I) d++;
    return d;
}

template <typename R>
__host__ __device__ inline size_t score_smem(int N)
{
    // matrices, then one step per internal node and the empty one behind them
    return (size_t)16 * N * sizeof(R) + (size_t)16 * (N / 2 + 2);
}

size_t score_slot_bytes(int N, int S, int BS, int Pcap, int fp64)
{
    return al((size_t)Pcap * 8, 256) + (size_t)(BS / 64) * block_bytes(score_slots(N - S), fp64 ? 8 : 4);
}

// The nodes' words of a scoring pass, where their matrices will be (node_len).
// Then its steps, every internal node, one node a thread, and the
// bytes a pass that stores every node but the cherries would move per
// pattern (the counted bytes of a call).
template <typename R, int BS>
__device__ __forceinline__ void score_stage(MP M, AP A, LDS R *PT, const int32_t *tab, int n_int, int row)
{
    const int N = uni(M->N);
    const int32_t *po = tab + tab_porder(N), *ch0 = tab + tab_ch0(N), *ch1 = tab + tab_ch1(N), *fl = tab + tab_flags(N);
    const double *len = A->len_in ? A->len_in + (size_t)row * N : (const double *)(tab + tab_dist(N));
    const int32_t *zin = A->len_in ? tab : A->Zin + (size_t)row * N;      // (unused with lengths of its own)
    const int32_t *bin = A->gb_eig ? A->Bin + (size_t)row * N : tab;      // (unused without gBGC)
    // two nodes a thread, past the end the last one again
    for (int i0 = threadIdx.x; i0 < N; i0 += 2 * BS) {
        const int i1 = i0 + BS < N ? i0 + BS : i0;
        const double l0 = len[i0], l1 = len[i1];
        const int z0 = zin[i0], z1 = zin[i1], g0 = bin[i0], g1 = bin[i1];
        const int a0 = ch0[i0], a1 = ch0[i1], b0 = ch1[i0], b1 = ch1[i1], f0 = fl[i0], f1 = fl[i1];
        const int o0 = po[i0 < n_int ? i0 : 0], o1 = po[i1 < n_int ? i1 : 0];
        auto put = [&](int i, double l, int z, int g, int a, int b, int f, int o) __attribute__((always_inline)) {
            LDS int32_t *w = node_int(PT, i);
            *node_len(PT, i) = l;
            w[0] = branch_class(A, z, g);
            w[1] = (a & 0x3ff) | (b & 0x3ff) << 10 | ((f & NF_MISSING) ? 1 << 20 : 0);
            w[2] = o;        // the i-th node of the pruning order
        };
        put(i0, l0, z0, g0, a0, b0, f0, o0);
        put(i1, l1, z1, g1, a1, b1, f1, o1);
    }
}

template <typename R, int BS, bool WIDE>
__device__ __forceinline__ void score_steps(MP M, LDS R *PT, LDS uint32_t *steps, LDS uint32_t *per, int n_int, int root, const CodeRows<WIDE> &codes)
{
    const int S = uni(M->S);
    constexpr uint32_t W = 4 * sizeof(R) + 4;
    for (int t = threadIdx.x; t <= n_int; t += BS) {
        LDS uint32_t *o = steps + 4 * t;
        if (t == n_int) {
            o[0] = o[1] = o[2] = o[3] = 0;
            continue;
        }
        const uint32_t word = (uint32_t)node_int(PT, t)[2];
        const int s = word & PO_NODE, mine = node_int(PT, s)[1];
        const int p1 = t > 0 ? (int)((uint32_t)node_int(PT, t - 1)[2] & PO_NODE) : -1, p2 = t > 1 ? (int)((uint32_t)node_int(PT, t - 2)[2] & PO_NODE) : -1;
        const int x[2] = {mine & 0x3ff, (mine >> 10) & 0x3ff};
        StepDef d;
        d.nostore = !(word & PO_WAITS);
        d.slot_to = (word >> PO_SLOT_SHIFT) & 31;
        uint32_t b = W;
        for (int j = 0; j < 2; j++) {
            const bool leaf = x[j] < S;
            const int kid = node_int(PT, x[j])[1];
            d.kind[j] = leaf ? SK_LEAF : (x[j] == p1 ? SK_PREV : (x[j] == p2 ? SK_PREV2 : SK_STORED));
            d.miss_kid[j] = kid >> 20 & 1;
            d.mat[j] = x[j];
            d.row[j] = leaf ? codes.row(x[j]) : 0;
            d.slot[j] = d.kind[j] == SK_STORED ? (int)((word >> PO_DEPTH_SHIFT) & PO_DEPTH) : 0;
            b += leaf ? 1 : ((kid & 0x3ff) < S && (kid >> 10 & 0x3ff) < S ? 2 : W);
        }
        encode_step(o, d);
        const bool cherry = s != root && x[0] < S && x[1] < S;
        if (!cherry) __hip_atomic_fetch_add(per, b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
}

// Brings the codes of one block of 64 patterns (a cache line of every leaf's
// row) near, a row a lane; the value only keeps the loads.  The rows are read
// once a call, mostly from HBM, whose latency is longer than the steps a code
// is loaded ahead.
template <bool WIDE>
__device__ __forceinline__ uint32_t touch_codes(const CodeRows<WIDE> &codes, int S, int pb)
{
    uint32_t x = 0;
    for (int r = threadIdx.x & 63; r < S; r += 64) x |= codes.four(r, pb);
    return x;
}

// The sums of a pass (log_f_Xz, src/PhyloAcc-ST/bpp_c2.cpp:392-425): log
// sum_j pi_j L_j + exponent * ln 2 over the patterns, or over the sites of
// the two prefixes by way of a table of the patterns' terms.  FP64; all-gap
// columns contribute 0.
template <typename R, int BS, bool AMB, bool WIDE>
__device__ __forceinline__ void score_patterns(MP M, AP A, const PassArgs<R, WIDE> &a, const ElemDev &E, const double (&pi)[4], char *scratch,
                                               int row, int first, int P, LDS double *red, double &s0, double &s1)
{
    const int tid = threadIdx.x;
    const GBL int32_t *wts = (const GBL int32_t *)(A->wts + E.off_w);
    GBL double *term = (GBL double *)scratch;
    const size_t term_bytes = A->pre_len ? al((size_t)E.Ppad * 8, 256) : 0;
    const int blkB = block_bytes(a.slots, sizeof(R));
    GBL char *stack = (GBL char *)scratch + term_bytes + (size_t)uni(tid >> 6) * blkB;
    const bool pre = A->pre_len != nullptr;
    double acc = 0, acc1 = 0;
    for (int pb = first + uni(tid & ~63); pb < P; pb += BS) {
        const int p = pb + (tid & 63);
        const uint32_t ahead = pb + BS < P ? touch_codes(a.codes, uni(M->S), pb + BS) : 0;
        const ChildIn<R> o = prune_pattern<R, AMB, SCORE_DEPTH, false>(a, stack, blkB, (uint32_t)p);
        asm volatile("" ::"v"(ahead));
        double t = 0;
        if (o.x != GAPT) {
            const double L = pi[0] * (double)o.v.x + pi[1] * (double)o.v.y + pi[2] * (double)o.v.z + pi[3] * (double)o.v.w;
            t = log(L) + (double)o.x * 0.69314718055994530942;
        }
        if (pre) term[p] = t;
        else if (p < P && o.x != GAPT) acc += (double)wts[p] * t;
    }
    if (pre) {
        __syncthreads();
        const GBL int32_t *site = (const GBL int32_t *)(A->site + E.off_site);
        const int n0 = A->pre_len[2 * row], n1 = A->pre_len[2 * row + 1];
        for (int g = tid; g < n0; g += BS) {
            const double t = term[site[g]];
            acc += t;
            if (g < n1) acc1 += t;
        }
        s1 = block_sum(acc1, red);
    }
    s0 = block_sum(acc, red);
}

template <typename R, int BS, bool WIDE = false>
__global__ void __launch_bounds__(BS, 4) score_kernel(ModelDev Mk, LoglikArgs Ak)
{
    extern __shared__ __align__(32) char smem_raw[];
    __shared__ ModelDev Ms;
    __shared__ LoglikArgs As;
    __shared__ double red[4];
    __shared__ int work_sh;
    __shared__ uint32_t per_sh;
    MP M = to_lds(Mk, (LDS ModelDev *)&Ms);
    AP A = to_lds(Ak, (LDS LoglikArgs *)&As);
    __syncthreads();
    const int N = uni(M->N), S = uni(M->S), tid = threadIdx.x;
    LDS R *PT = (LDS R *)(LDS char *)smem_raw;
    LDS uint32_t *steps = (LDS uint32_t *)(PT + 16 * N);
    LDS double *eig = (LDS double *)((LDS char *)smem_raw + score_smem<R>(N));
    for (bool first_work = true;; first_work = false) {
        if (tid == 0) {
            // the first position without the counter (2,048 increments at once: gene trees 819 -> 787 us);
            // later ones when they are needed, since one taken ahead waits for this one to end
            work_sh = first_work ? (int)blockIdx.x : (int)gridDim.x + atomicAdd(A->queue, 1);
            per_sh = 0;
        }
        __syncthreads();
        const int it = uni(work_sh);
        if (it >= uni(A->items ? A->n_items : A->n_work)) break;
        ScoreItem item{it, 0, 0, -1};
        if (A->items) item = A->items[it];
        const int w = uni(item.w), part = uni(item.part);
        // an id outside the arenas, or an element without patterns (filtered, or of no sites), scores NaN
        const int id = uni(A->work[w]);
        const int row = A->len_row ? uni(A->len_row[w]) : w;
        if (id < 0 || id >= uni(A->n_elems) || A->elems[id].P <= 0) {
            if (tid == 0) write_scores(A, w, row, __builtin_nan(""), __builtin_nan(""));
            __syncthreads();
            continue;
        }
        const double *pw = A->el_pi ? A->el_pi + (size_t)w * 4 : nullptr;
        double pi[4];
        for (int j = 0; j < 4; j++) pi[j] = pw ? pw[j] : M->pi[j];
        const int64_t bo = A->big_off ? A->big_off[w] : -1;
        const ElemDev E = uni_elem(A->elems + id);
        const int32_t *hdr = A->hdr_call ? A->hdr_call + (size_t)row * 4 : nullptr;
        const int32_t *tab = uni_ptr(A->tab_call ? A->tab_call + (size_t)row * tab_words(N) : A->tab + E.off_tab);
        const int root = uni(hdr ? hdr[0] : E.root), n_int = (uni(hdr ? hdr[1] : E.n_nodes) - 1) / 2;
        const int first = uni(item.p0), P = part < 0 ? E.P : uni(item.p1);
        const CodeRows<WIDE> codes(uni_ptr((GBL uint8_t *)(A->codes + E.off_codes)), S, E.Ppad);
        const uint32_t ahead = first + (tid & ~63) < P ? touch_codes(codes, S, first + (tid & ~63)) : 0;
        score_stage<R, BS>(M, A, PT, tab, n_int, row);
        fetch_eig(A, eig, w, row);
        __syncthreads();
        score_steps<R, BS>(M, PT, steps, (LDS uint32_t *)&per_sh, n_int, root, codes);
        __syncthreads();
        // every node's matrix (the root's and absent nodes' are never read)
        for (int i = tid; i < 4 * N; i += BS) work_matrix_row<R>(M, A, eig, PT, *node_len(PT, i >> 2), *node_int(PT, i >> 2), i >> 2, i & 3, row);
        char *scratch = uni_ptr(bo >= 0 ? A->big + bo : A->scratch + (int64_t)blockIdx.x * A->slot_bytes);
        asm volatile("" ::"v"(ahead));
        __syncthreads();
        const PassArgs<R, WIDE> a = {(const LDS u32x4 *)steps, PT, codes, n_int, score_slots(N - S)};
        double s0 = 0, s1 = 0;
        if (E.has_amb) score_patterns<R, BS, true>(M, A, a, E, pi, scratch, row, first, P, (LDS double *)red, s0, s1);
        else score_patterns<R, BS, false>(M, A, a, E, pi, scratch, row, first, P, (LDS double *)red, s0, s1);
        if (tid == 0) {
            if (part >= 0) {
                A->part_sum[part] = s0;
            } else {
                write_scores(A, w, row, s0, s1);
            }
            // and the root's partial, exponent and pattern weight
            if (A->counters) atomicAdd(A->counters, (unsigned long long)(P - first) * (per_sh + 4 * sizeof(R) + 8));
        }
        __syncthreads();
    }
}

// ------------------------------------------------------ partials that stay
//
// A launch whose partials are read afterwards: resident partials (the height
// moves), histories and candidate scores.  Every node but the cherries is
// stored to its slot (node - S) of the pattern's block.
//
// Resident partials.  A full pass stores every node.  A row with path_node =
// v scores a proposal that changes the branches at v, and stores none of the
// path from v to the root: an accepted move only marks that path stale
// (gt_hdecide_kernel).  Stale nodes form a top part of the tree, and those
// that hang off the next move's path are pruned first, into their slots.  So
// over a sweep a node is stored about once, where storing every proposal's
// path stored it at each move below it: a move's pass over 4,000 elements of
// 120 leaves took 324 us that way and takes 250 now, 0.57 GB moved.  What is
// left is latency: a dozen steps for each of a wave's three blocks (half the
// time) and the set-up of each element (a third).

enum { MK_PATH = 1, MK_STALE = 2, MK_MISS = 4, MK_CHERRY = 8 };

constexpr int CAND_CHUNK = 16;      // candidates whose matrices are built together
constexpr int KEEP_CHUNKS = MAXN / 2 / 64;      // masks of 64 positions of the pruning order

template <typename R>
__host__ __device__ inline size_t keep_smem(int N, int BS, bool history)
{
    // matrices, steps, the internal nodes' children and pruning order, parents, marks; the sampler's steps and the
    // threads' bases
    const size_t I = N / 2 + 1;
    return (size_t)16 * N * sizeof(R) + 16 * (I + 1) + al(3 * (size_t)N + 6 * I, 16) + (history ? 8 * (I + 2) + I * BS : 0);
}

// Dynamic and static LDS (the kernels' __shared__ variables) of a workgroup.
size_t loglik_smem_bytes(int N, int fp64, int BS, LoglikUse use)
{
    const size_t args = sizeof(ModelDev) + sizeof(LoglikArgs) + 8;
    if (use == LoglikUse::Score) return (fp64 ? score_smem<double>(N) : score_smem<float>(N)) + args + 4 * 8;
    const bool history = use == LoglikUse::History;
    return (fp64 ? keep_smem<double>(N, BS, history) : keep_smem<float>(N, BS, history)) + args + 2 * KEEP_CHUNKS * 8 +
           CAND_CHUNK * 4 * 8 + (use == LoglikUse::Candidates ? CAND_CHUNK * 16 * 8 : 0);
}

// Waves per SIMD the kernel is declared for: what holds its registers with few
// or no spills (FP64 240, histories and candidates 168), and for the height
// moves, which wait on memory, the most that LDS lets run.
constexpr int keep_waves(int rs, LoglikUse use) { return rs == 8 ? 2 : (use == LoglikUse::Keep ? 4 : 3); }

template <typename R>
struct KeepLds {
    LDS R *PT;
    LDS uint32_t *steps;         // [I + 1][4]
    LDS int16_t *ch0, *ch1;      // indexed by node, internal nodes only
    LDS int16_t *par, *order;    // [N]; [I] the nodes in pruning order
    LDS uint8_t *mark;
    LDS u32x2 *hrec;             // [I + 2] the history's steps
    LDS uint8_t *tgs;            // [I][BS] the threads' drawn bases
};

template <typename R>
__device__ __forceinline__ KeepLds<R> keep_lds(LDS char *base, int N, int S)
{
    KeepLds<R> k;
    const size_t I = N / 2 + 1;
    k.PT = (LDS R *)base;
    LDS char *o = base + (size_t)16 * N * sizeof(R);
    k.steps = (LDS uint32_t *)o;
    o += 16 * (I + 1);
    k.ch0 = (LDS int16_t *)o - S;
    k.ch1 = k.ch0 + I;
    k.order = k.ch1 + S + I;
    k.par = k.order + I;
    k.mark = (LDS uint8_t *)(k.par + N);
    o += al(3 * (size_t)N + 6 * I, 16);
    k.hrec = (LDS u32x2 *)o;
    k.tgs = (LDS uint8_t *)(o + 8 * (I + 2));
    return k;
}

// The steps of a pass: every node, or (path) first the stale nodes off the
// path, which are stored, then the path.  Which of 64 positions of the pruning
// order a phase visits is a bit mask, a wave a mask (keep_visits); a position's
// place in the list and the steps just before it follow from the masks.
// keep_steps returns the number of steps and adds to per what a pass that
// stores the nodes it scores (all, or the path's) and reads all their children
// would move per pattern.
template <typename R, int BS>
__device__ __forceinline__ void keep_visits(const KeepLds<R> &k, LDS unsigned long long *visit, int n_int, bool path)
{
    const int lane = threadIdx.x & 63;
    for (int c = uni(threadIdx.x >> 6); c < KEEP_CHUNKS; c += BS / 64) {
        const int q = c * 64 + lane;
        bool a = false, b = false;
        if (q < n_int) {
            const int s = k.order[q], mk = k.mark[s];
            // a cherry off the path is a step of its parent's visit
            const int t = (mk & MK_CHERRY) && !(mk & MK_PATH) ? k.mark[k.par[s]] : mk;
            a = path && (t & MK_STALE) && !(t & MK_PATH);
            b = !path || (t & MK_PATH);
        }
        const unsigned long long va = __ballot(a), vb = __ballot(b);
        if (lane == 0) {
            visit[c] = va;
            visit[KEEP_CHUNKS + c] = vb;
        }
    }
}

template <typename R, int BS, bool WIDE>
__device__ __forceinline__ int keep_steps(const KeepLds<R> &k, const LDS unsigned long long *visit, LDS uint32_t *per, int S, int n_int,
                                          const CodeRows<WIDE> &codes, GBL uint8_t *stale)
{
    constexpr int W = 4 * sizeof(R) + 4;
    const int lane = threadIdx.x & 63;
    int total = 0;
    for (int m = 0; m < 2 * KEEP_CHUNKS; m++) total += __popcll(visit[m]);
    for (int c = uni(threadIdx.x >> 6); c * 64 < n_int; c += BS / 64) {
        for (int phase = 0; phase < 2; phase++) {
            const int m = phase * KEEP_CHUNKS + c;
            const unsigned long long mine = visit[m];
            if (!mine) continue;
            if (!((mine >> lane) & 1)) continue;
            int at = __popcll(mine & ((1ull << lane) - 1));
            for (int x = 0; x < m; x++) at += __popcll(visit[x]);
            // the nodes of the three steps before
            int before[3] = {-1, -1, -1};
            unsigned long long bits = mine & ((1ull << lane) - 1);
            int f = m;
#pragma unroll
            for (int i = 0; i < 3; i++) {
                while (!bits && f > 0) bits = visit[--f];
                if (bits) {
                    const int h = 63 - __clzll(bits);
                    before[i] = k.order[(f % KEEP_CHUNKS) * 64 + h];
                    bits ^= 1ull << h;
                }
            }
            const int s = k.order[c * 64 + lane], mk = k.mark[s];
            const int x[2] = {k.ch0[s], k.ch1[s]};
            StepDef d;
            d.nostore = (mk & MK_CHERRY) || (mk & MK_PATH);
            d.slot_to = s - S;
            uint32_t b = W;
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const bool leaf = x[j] < S;
                d.kind[j] = leaf ? SK_LEAF : (x[j] == before[0] ? SK_PREV : (x[j] == before[1] ? SK_PREV2 : SK_STORED));
                d.late = d.late || (!leaf && x[j] == before[2]);
                d.miss_kid[j] = (k.mark[x[j]] & MK_MISS) ? 1 : 0;
                d.mat[j] = x[j];
                d.row[j] = leaf ? codes.row(x[j]) : 0;
                d.slot[j] = leaf ? 0 : x[j] - S;
                b += leaf ? 1 : ((k.mark[x[j]] & MK_CHERRY) ? 2 : W);
            }
            encode_step(k.steps + 4 * at, d);
            if (phase == 1 && !(mk & MK_CHERRY)) __hip_atomic_fetch_add(per, b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            if (phase == 0 && !(mk & MK_CHERRY)) stale[s] = 0;      // stored by this pass
        }
    }
    if (threadIdx.x < 4) k.steps[4 * total + threadIdx.x] = 0;
    return total;
}

// The pass over an element's blocks and its root sums (see score_patterns;
// with site prefixes the patterns' terms lie behind the blocks).
template <typename R, int BS, bool AMB, bool WIDE>
__device__ __forceinline__ void keep_patterns(AP A, const PassArgs<R, WIDE> &a, const ElemDev &E, const double (&pi)[4], GBL char *blocks,
                                              const GBL int32_t *site, int row, LDS double *red, double &s0, double &s1)
{
    const int tid = threadIdx.x, P = E.P, blkB = block_bytes(a.slots, sizeof(R));
    const GBL int32_t *wts = (const GBL int32_t *)(A->wts + E.off_w);
    const bool pre = A->pre_len != nullptr;
    GBL double *term = (GBL double *)(blocks + al((size_t)(E.Ppad / 64) * blkB, 256));
    double acc = 0, acc1 = 0;
    for (int pb = uni(tid & ~63); pb < P; pb += BS) {
        const int p = pb + (tid & 63);
        const ChildIn<R> o = prune_pattern<R, AMB, SCORE_DEPTH, true, SCORE_DEPTH>(a, blocks + (size_t)(pb >> 6) * blkB, blkB, (uint32_t)p);
        double t = 0;
        if (o.x != GAPT) {
            const double L = pi[0] * (double)o.v.x + pi[1] * (double)o.v.y + pi[2] * (double)o.v.z + pi[3] * (double)o.v.w;
            t = log(L) + (double)o.x * 0.69314718055994530942;
        }
        if (pre) term[p] = t;
        else if (p < P && o.x != GAPT) acc += (double)wts[p] * t;
    }
    if (pre) {
        __syncthreads();
        const int n0 = A->pre_len[2 * row], n1 = A->pre_len[2 * row + 1];
        // four sites' loads at a time, added in the sites' order
        for (int g0 = tid; g0 < n0; g0 += 4 * BS) {
            int at[4];
            double t[4];
#pragma unroll
            for (int i = 0; i < 4; i++) at[i] = site[g0 + i * BS < n0 ? g0 + i * BS : g0];
#pragma unroll
            for (int i = 0; i < 4; i++) t[i] = term[at[i]];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                if (g0 + i * BS < n0) acc += t[i];
                if (g0 + i * BS < n1) acc1 += t[i];
            }
        }
        s1 = block_sum(acc1, red);
    }
    s0 = block_sum(acc, red);
}

// A node's partial and exponent at pattern p (each lane its own block); a
// cherry's is recomputed from its leaf codes, as a pass does.
template <typename R, bool WIDE>
__device__ __forceinline__ ChildIn<R> kept_node(const KeepLds<R> &k, const GBL char *blocks, const CodeRows<WIDE> &codes, int S, int I, int v, int p)
{
    ChildIn<R> in;
    if (k.mark[v] & MK_CHERRY) {
        const int yA = uni(k.ch0[v]), yB = uni(k.ch1[v]);
        return cherry_in<R>(k.PT + 16 * yA, k.PT + 16 * yB, k.mark[yA] & MK_MISS, k.mark[yB] & MK_MISS,
                            codes.at(codes.row(yA), p), codes.at(codes.row(yB), p));
    }
    const GBL char *blk = blocks + (size_t)(p >> 6) * block_bytes(I, sizeof(R));
    in.v = ld4<R>((const GBL V4<R> *)(blk + part_off<R>(v - S)) + (p & 63));
    in.x = ((const GBL int32_t *)(blk + exp_off<R>(v - S, I)))[p & 63];
    return in;
}

// ------------------------------------------- gene-tree moves (PhyloAcc-GT)

// A leaf code as a history base: 0-3, -1 for an ambiguity code, 4 for a gap
// or another character (src/PhyloAcc-GT/bpp_c.hpp:340-384).
__device__ inline int leaf_base(int code)
{
    return code < 4 ? code : (code == PA_GAP_CODE || code == PA_OTHER_CODE ? 4 : -1);
}

// The history's steps: the internal nodes in the reverse of the pruning
// order (a parent before its children), two words each.
//   x: node | parent << 10 | HR_* bits
//   y: its leaf children + 1, A | B << 10 (0: none) | the slot its partial is loaded from << 20
enum { HR_MISS = 1 << 20, HR_CHERRY = 1 << 21, HR_PREV = 1 << 22, HR_MISS_A = 1 << 23, HR_MISS_B = 1 << 24 };

template <typename R, int BS>
__device__ __forceinline__ void history_steps(const KeepLds<R> &k, int S, int n_int, int root)
{
    for (int t = threadIdx.x; t <= n_int; t += BS) {
        u32x2 w;
        if (t == n_int) {
            // read ahead of the end
            w.x = (uint32_t)root | (uint32_t)root << 10 | HR_MISS;
            w.y = (uint32_t)(root - S) << 20;
        } else {
            const int s = k.order[n_int - 1 - t], x0 = k.ch0[s], x1 = k.ch1[s], mk = k.mark[s];
            const int pa = t > 0 ? k.par[s] : s;
            w.x = (uint32_t)s | (uint32_t)pa << 10 | ((mk & MK_MISS) ? HR_MISS : 0) | ((mk & MK_CHERRY) ? HR_CHERRY : 0) |
                  (t > 0 && k.order[n_int - t] == pa ? HR_PREV : 0) |
                  (x0 < S && (k.mark[x0] & MK_MISS) ? HR_MISS_A : 0) | (x1 < S && (k.mark[x1] & MK_MISS) ? HR_MISS_B : 0);
            w.y = (x0 < S ? (uint32_t)x0 + 1 : 0) | (x1 < S ? (uint32_t)(x1 + 1) << 10 : 0) |
                  (uint32_t)(((mk & (MK_MISS | MK_CHERRY)) ? root : s) - S) << 20;
        }
        k.hrec[t] = w;
    }
}

// GTree::Update_Tg with tosample = true (src/PhyloAcc-GT/genetree.cpp:
// 1416-1532) after the pass: one thread per site draws the gene root's base
// from pi * L_root, then every internal gene node's from P(parent base -> .)
// * L over its whole branch (the law of the reference's species-by-species
// steps), and writes every node's base.  The steps are the chain sampler's:
// words read ahead, the loads of the next four steps in flight.
template <typename R, int BS, bool AMB, bool WIDE>
__device__ __forceinline__ void draw_history(MP M, AP A, const KeepLds<R> &k, const GBL char *blocks, const CodeRows<WIDE> &codes,
                                             const double (&pi)[4], const GBL int32_t *site, int row, int n_int, int S, int I)
{
    constexpr int K = 4;
    const int tid = threadIdx.x, len = uni(A->hist_len[row]), stride = uni(A->hist_ns[row]);
    GBL int8_t *out = (GBL int8_t *)A->hist + A->hist_off[row];
    const Key key{M->key0, M->key1};
    const uint32_t c2 = (uint32_t)A->hist_sweep, c3 = tagword(0, TAG_GT_HIST);
    LDS uint8_t *tgs = k.tgs + tid - S * BS;
    for (int gb = uni(tid & ~63); gb < len; gb += BS) {
        const int g = gb + (tid & 63);
        const bool on = g < len;
        const int p = site[on ? g : len - 1];
        const GBL char *pp = blocks + (size_t)(p >> 6) * block_bytes(I, sizeof(R)) + (p & 63) * sizeof(V4<R>);
        const GBL char *pe = blocks + (size_t)(p >> 6) * block_bytes(I, sizeof(R)) + exp_off<R>(0, I) + (p & 63) * 4;
        u32x2 w[K], nr = k.hrec[0];
        ChildIn<R> in[K];
        int cdA[K], cdB[K];
        auto fetch = [&](auto J, int t) __attribute__((always_inline)) {
            constexpr int j = decltype(J)::value;
            w[j].x = (uint32_t)uni((int)nr.x);
            w[j].y = (uint32_t)uni((int)nr.y);
            nr = k.hrec[t + 1 < n_int ? t + 1 : n_int];
            const uint32_t slot = w[j].y >> 20, a = w[j].y & 0x3ff, b = (w[j].y >> 10) & 0x3ff;
            in[j].v = ld4<R>((const GBL V4<R> *)(pp + (uint64_t)part_off<R>(slot)));
            in[j].x = *(const GBL int32_t *)(pe + (uint64_t)(slot * 256));
            cdA[j] = codes.at((uint32_t)uni((int)codes.row(a ? a - 1 : 0)), p);
            cdB[j] = codes.at((uint32_t)uni((int)codes.row(b ? b - 1 : 0)), p);
        };
        int res = 4, tp = 4;
        auto step = [&](auto J, int t) __attribute__((always_inline)) {
            constexpr int j = decltype(J)::value;
            const uint32_t w0 = w[j].x;
            const int s = w0 & 0x3ff, yA = (int)(w[j].y & 0x3ff) - 1, yB = (int)((w[j].y >> 10) & 0x3ff) - 1;
            const int from = (w0 & HR_PREV) ? res : tp;
            tp = tgs[((w[(j + 1) % K].x >> 10) & 0x3ff) * BS];
            if (t < n_int) {
                int r = 4;
                if (!(w0 & HR_MISS) || t == 0) {
                    ChildIn<R> a = in[j];
                    if (w0 & HR_CHERRY) {
                        V4<R> ma, mb;
                        int e = 0;
                        bool ga, gb2;
                        message<R, SK_LEAF, AMB>(k.PT + 16 * yA, cdA[j], in[j], ma, e, ga);
                        message<R, SK_LEAF, AMB>(k.PT + 16 * yB, cdB[j], in[j], mb, e, gb2);
                        if (w0 & HR_MISS_A) ma.x = ma.y = ma.z = ma.w = (R)1;
                        if (w0 & HR_MISS_B) mb.x = mb.y = mb.z = mb.w = (R)1;
                        a = combine<R>(ma, mb, 0, ga && gb2);
                    }
                    const double u = slot_uniform(key, (uint32_t)g, c2, c3, (uint32_t)s);
                    const bool has = a.x != GAPT && !(w0 & HR_MISS);
                    double q[4];
                    if (t == 0) {
                        q[0] = has ? pi[0] * (double)a.v.x : pi[0]; q[1] = has ? pi[1] * (double)a.v.y : pi[1];
                        q[2] = has ? pi[2] * (double)a.v.z : pi[2]; q[3] = has ? pi[3] * (double)a.v.w : pi[3];
                        r = categorical<4>(q, u);
                    } else {
                        const LDS R *PT = k.PT + 16 * s + (from & 3);      // PT[i*4+j] = P_{j->i}
                        q[0] = (double)PT[0] * (double)a.v.x; q[1] = (double)PT[4] * (double)a.v.y;
                        q[2] = (double)PT[8] * (double)a.v.z; q[3] = (double)PT[12] * (double)a.v.w;
                        const int d = categorical<4>(q, u);
                        r = has && from < 4 ? d : 4;
                    }
                }
                res = r;
                tgs[s * BS] = (uint8_t)r;
                if (on) {
                    out[(size_t)s * stride + g] = (int8_t)r;
                    if (yA >= 0) out[(size_t)yA * stride + g] = (int8_t)leaf_base(cdA[j]);
                    if (yB >= 0) out[(size_t)yB * stride + g] = (int8_t)leaf_base(cdB[j]);
                }
            }
            fetch(J, t + K);
        };
        each<K>([&](auto J) __attribute__((always_inline)) { fetch(J, decltype(J)::value); });
        for (int t0 = 0; t0 < n_int; t0 += K)
            each<K>([&](auto J) __attribute__((always_inline)) { step(J, t0 + decltype(J)::value); });
    }
}

// P(d) = V e^{lam d} Vi in FP64 into Pc[a*4+b] = P_{a->b}, clamped at 0; the
// identity below 1e-8 (BPP::getlogTM_len, src/PhyloAcc-GT/bpp.cpp:238-252).
template <typename PE>
__device__ inline void full_transition(PE lam, PE V, PE Vi, double d, LDS double *Pc)
{
    double e[4];
    for (int k = 0; k < 4; k++) e[k] = exp(lam[k] * d);
    for (int a = 0; a < 4; a++)
        for (int j = 0; j < 4; j++) {
            double v = 0;
            for (int k = 0; k < 4; k++) v += V[a * 4 + k] * e[k] * Vi[k * 4 + j];
            Pc[a * 4 + j] = d < 1e-8 ? (a == j ? 1.0 : 0.0) : (v < 0 ? 0.0 : v);
        }
}

// Candidate scores of GTree::Sample_tree2 (src/PhyloAcc-GT/genetree.cpp:
// 2190-2380) after the pass over the current tree: for each candidate new
// grandparent of branch b at substitution distance d, the sum over sites
// where b holds a base of: kind 0, log (P(d) L_b)[x_t] at the candidate's
// sampled base x_t (the pi-average of P(d) L_b when it has none); kind 1, the
// pi-average; kind 2, log sum_i pi_i P(d)_{x_b -> i} at b's own base.  The
// matrices of CAND_CHUNK candidates are built at once, a thread each, and
// their sums meet once.
template <typename R, int BS, bool WIDE>
__device__ __noinline__ void gt_candidates(MP M, AP A, const KeepLds<R> k, const GBL char *blocks_, const GBL uint8_t *codes_,
                                           const GBL int32_t *site, LDS double *Pc, LDS double *red, int w, int row_, int S_, int I_,
                                           int Ppad_, double pi0, double pi1, double pi2, double pi3)
{
    // arguments of a call come in vector registers
    const int row = uni(row_), S = uni(S_), I = uni(I_);
    const GBL char *blocks = uni_ptr(blocks_);
    const CodeRows<WIDE> codes(uni_ptr(codes_), S, uni(Ppad_));
    const int tid = threadIdx.x, stride = A->hist_ns[row], cm = A->cand_max;
    const GBL int8_t *tg = (const GBL int8_t *)A->hist + A->hist_off[row];
    const int b = uni(A->cand_branch[row]), nc = uni(A->cand_n[row]), len = uni(A->cand_sites[row]);
    const double *E = A->el_eig ? A->el_eig + (size_t)w * GB_EIG_WORDS : nullptr;
    const double pi[4] = {pi0, pi1, pi2, pi3}, lp[4] = {log(pi0), log(pi1), log(pi2), log(pi3)};
    for (int q0 = 0; q0 < nc; q0 += CAND_CHUNK) {
        const int nq = min(CAND_CHUNK, nc - q0);
        if (tid < nq) {
            const double d = A->cand_len[(size_t)row * cm + q0 + tid];
            if (E) full_transition(E, E + 4, E + 20, d, Pc + 16 * tid);
            else full_transition(M->lam, M->V, M->Vi, d, Pc + 16 * tid);
        }
        __syncthreads();
        for (int q = 0; q < nq; q++) {
            const int t = uni(A->cand_node[(size_t)row * cm + q0 + q]), kind = uni(A->cand_kind[(size_t)row * cm + q0 + q]);
            const LDS double *P = Pc + 16 * q;
            const bool at_node = kind == 0 && !(k.mark[t] & MK_MISS);
            double acc = 0;
            for (int g = tid; g < len; g += BS) {
                const int xb = tg[(size_t)b * stride + g];
                if (xb >= 4) continue;
                if (kind == 2) {
                    if (xb < 0) continue;
                    double sum = 0;
                    for (int i = 0; i < 4; i++) sum += pi[i] * P[xb * 4 + i];
                    acc += log(sum);
                    continue;
                }
                const int p = site[g];
                const int xt = at_node ? tg[(size_t)t * stride + g] : 4;
                double L[4];
                int e = 0;
                if (b < S) {
                    const int code = codes.at(codes.row(b), p);
                    for (int j = 0; j < 4; j++) L[j] = 0;
                    if (code < 4) {
                        for (int j = 0; j < 4; j++) L[j] = j == code ? 1 : 0;
                    } else {
                        const int b1 = (code == 6 || code == 9 || code == 11) ? 0 : (code == 7 || code == 10) ? 1 : 2;
                        const int b2 = (code == 6 || code == 10) ? 2 : (code == 9) ? 1 : 3;
                        for (int j = 0; j < 4; j++) L[j] = j == b1 || j == b2 ? 1 : 0;
                    }
                } else {
                    const ChildIn<R> in = kept_node<R>(k, blocks, codes, S, I, b, p);
                    L[0] = in.v.x; L[1] = in.v.y; L[2] = in.v.z; L[3] = in.v.w;
                    e = in.x;
                }
                auto term = [&](int a) {
                    return log(P[a * 4 + 0] * L[0] + P[a * 4 + 1] * L[1] + P[a * 4 + 2] * L[2] + P[a * 4 + 3] * L[3]) +
                           (double)e * 0.69314718055994530942;
                };
                if (xt >= 0 && xt < 4) {
                    acc += term(xt);
                } else {
                    double Mv[4], mx = -INFINITY;
                    for (int a = 0; a < 4; a++) {
                        Mv[a] = term(a);
                        mx = fmax(mx, Mv[a] + lp[a]);
                    }
                    double sum = 0;
                    for (int a = 0; a < 4; a++) sum += exp(Mv[a] + lp[a] - mx);
                    acc += mx == -INFINITY ? -INFINITY : log(sum) + mx;
                }
            }
            // a fixed tree inside each wave; the waves' sums in order below
#pragma unroll
            for (int off = 32; off >= 1; off >>= 1) acc += __shfl_xor(acc, off, 64);
            if ((tid & 63) == 0) red[4 * q + (tid >> 6)] = acc;
        }
        __syncthreads();
        if (tid < nq) {
            double s = 0;
            for (int i = 0; i < BS / 64; i++) s += red[4 * tid + i];
            A->cand_score[(size_t)row * cm + q0 + tid] = s;
        }
        __syncthreads();
    }
}

template <typename R, int BS, LoglikUse USE, bool WIDE = false>
__global__ void __launch_bounds__(BS, keep_waves(sizeof(R), USE)) keep_kernel(ModelDev Mk, LoglikArgs Ak)
{
    extern __shared__ __align__(32) char smem_raw[];
    __shared__ ModelDev Ms;
    __shared__ LoglikArgs As;
    __shared__ double red[CAND_CHUNK * 4], Pc[CAND_CHUNK * 16];
    __shared__ unsigned long long visit[2 * KEEP_CHUNKS];
    __shared__ int work_sh;
    __shared__ uint32_t per_sh;
    MP M = to_lds(Mk, (LDS ModelDev *)&Ms);
    AP A = to_lds(Ak, (LDS LoglikArgs *)&As);
    __syncthreads();
    const int N = uni(M->N), S = uni(M->S), I = N - S, tid = threadIdx.x;
    const KeepLds<R> k = keep_lds<R>((LDS char *)smem_raw, N, S);
    LDS double *eig = (LDS double *)((LDS char *)smem_raw + keep_smem<R>(N, BS, USE == LoglikUse::History));
    for (bool first_work = true;; first_work = false) {
        if (tid == 0) {
            work_sh = first_work ? (int)blockIdx.x : (int)gridDim.x + atomicAdd(A->queue, 1);
            per_sh = 0;
        }
        __syncthreads();
        const int w = uni(work_sh);
        if (w >= uni(A->n_work)) break;
        const int id = uni(A->work[w]);
        const int row = A->len_row ? uni(A->len_row[w]) : w;
        if (id < 0 || id >= uni(A->n_elems) || A->elems[id].P <= 0) {
            if (tid == 0) write_scores(A, w, row, __builtin_nan(""), __builtin_nan(""));
            __syncthreads();
            continue;
        }
        const double *pw = A->el_pi ? A->el_pi + (size_t)w * 4 : nullptr;
        double pi[4];
        for (int j = 0; j < 4; j++) pi[j] = pw ? pw[j] : M->pi[j];
        const int64_t bo = A->big_off ? A->big_off[w] : -1;
        const ElemDev E = uni_elem(A->elems + id);
        const int32_t *hdr = A->hdr_call ? A->hdr_call + (size_t)row * 4 : nullptr;
        const int32_t *tab = uni_ptr(A->tab_call ? A->tab_call + (size_t)row * tab_words(N) : A->tab + E.off_tab);
        const int root = uni(hdr ? hdr[0] : E.root), n_int = (uni(hdr ? hdr[1] : E.n_nodes) - 1) / 2;
        const int moved = A->path_node ? uni(A->path_node[row]) : -1;
        const bool path = moved >= S && moved < N;
        const CodeRows<WIDE> codes(uni_ptr((GBL uint8_t *)(A->codes + E.off_codes)), S, E.Ppad);
        GBL uint8_t *stale = A->stale ? (GBL uint8_t *)(A->stale + (size_t)row * N) : nullptr;
        const int32_t *po = tab + tab_porder(N);
        const double *len = A->len_in ? A->len_in + (size_t)row * N : (const double *)(tab + tab_dist(N));
        const int32_t *zin = A->len_in ? tab : A->Zin + (size_t)row * N;      // (unused with lengths of its own)
        // every load in flight at once: two nodes a thread, past the end the last one again
        for (int i0 = tid; i0 < N; i0 += 2 * BS) {
            const int i1 = i0 + BS < N ? i0 + BS : i0;
            const int a0 = tab[tab_ch0(N) + i0], b0 = tab[tab_ch1(N) + i0], f0 = tab[tab_flags(N) + i0], p0 = tab[tab_par(N) + i0];
            const int a1 = tab[tab_ch0(N) + i1], b1 = tab[tab_ch1(N) + i1], f1 = tab[tab_flags(N) + i1], p1 = tab[tab_par(N) + i1];
            const int o0 = po[i0 < n_int ? i0 : 0], o1 = po[i1 < n_int ? i1 : 0];
            const uint8_t *st = stale ? (const uint8_t *)stale : (const uint8_t *)tab;
            const int s0 = st[i0], s1 = st[i1];
            const double l0 = len[i0], l1 = len[i1];
            const int z0 = zin[i0], z1 = zin[i1];
            auto put = [&](int i, int a, int b, int f, int pa, int o, int st, double l, int z) __attribute__((always_inline)) {
                if (i >= S) {
                    k.ch0[i] = (int16_t)a;
                    k.ch1[i] = (int16_t)b;
                }
                k.par[i] = (int16_t)pa;
                if (i < n_int) k.order[i] = (int16_t)((uint32_t)o & PO_NODE);
                k.mark[i] = (uint8_t)(((f & NF_MISSING) ? MK_MISS : 0) | (stale && st ? MK_STALE : 0) |
                                      (i >= S && i != root && a >= 0 && a < S && b >= 0 && b < S ? MK_CHERRY : 0));
                *node_len(k.PT, i) = l;
                *node_int(k.PT, i) = branch_class(A, z, 0);
            };
            put(i0, a0, b0, f0, p0, o0, s0, l0, z0);
            put(i1, a1, b1, f1, p1, o1, s1, l1, z1);
        }
        fetch_eig(A, eig, w, row);
        __syncthreads();
        if (path) {
            if (tid == 0)
                for (int x = moved, q = 0; x >= 0 && x < N && q < N; x = k.par[x], q++) {
                    k.mark[x] |= MK_PATH;
                    if (x == root) break;
                }
            __syncthreads();
        }
        keep_visits<R, BS>(k, (LDS unsigned long long *)visit, n_int, path);
        __syncthreads();
        const int n = uni(keep_steps<R, BS>(k, (LDS unsigned long long *)visit, (LDS uint32_t *)&per_sh, S, n_int, codes, stale));
        if constexpr (USE == LoglikUse::History) history_steps<R, BS>(k, S, n_int, root);
        __syncthreads();
        // the matrices of the steps' children
        for (int i = tid; i < 8 * n; i += BS) {
            const uint32_t m = k.steps[4 * (i >> 3) + 3];
            const int s = (i & 4) ? (m >> SB_MAT_B_SHIFT) & SB_MAT_MASK : m & SB_MAT_MASK;
            work_matrix_row<R>(M, A, eig, k.PT, *node_len(k.PT, s), *node_int(k.PT, s), s, i & 3, row);
        }
        GBL char *blocks = uni_ptr((GBL char *)(bo >= 0 ? A->big + bo : A->scratch + (int64_t)blockIdx.x * A->slot_bytes));
        __syncthreads();
        const PassArgs<R, WIDE> a = {(const LDS u32x4 *)k.steps, k.PT, codes, n, I};
        const GBL int32_t *site = (const GBL int32_t *)(A->site + E.off_site);
        double s0 = 0, s1 = 0;
        if (E.has_amb) keep_patterns<R, BS, true>(A, a, E, pi, blocks, site, row, (LDS double *)red, s0, s1);
        else keep_patterns<R, BS, false>(A, a, E, pi, blocks, site, row, (LDS double *)red, s0, s1);
        // every wave's partials, before sites read other waves' patterns
        __syncthreads();
        if constexpr (USE == LoglikUse::History) {
            if (E.has_amb) draw_history<R, BS, true>(M, A, k, blocks, codes, pi, site, row, n_int, S, I);
            else draw_history<R, BS, false>(M, A, k, blocks, codes, pi, site, row, n_int, S, I);
        }
        if constexpr (USE == LoglikUse::Candidates)
            gt_candidates<R, BS, WIDE>(M, A, k, blocks, (const GBL uint8_t *)(A->codes + E.off_codes), site, (LDS double *)Pc, (LDS double *)red, w, row, S, I, E.Ppad, pi[0], pi[1], pi[2], pi[3]);
        if (tid == 0) {
            write_scores(A, w, row, s0, s1);
            // and the root's partial, exponent and pattern weight
            if (A->counters) atomicAdd(A->counters, (unsigned long long)E.P * (per_sh + 4 * sizeof(R) + 8));
        }
        __syncthreads();
    }
}

__global__ void reset_queue(int *q) { *q = 0; }

__global__ void score_sum_kernel(LoglikArgs A, const ScoreSplit *splits, int n)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const ScoreSplit s = splits[i];
    double t = 0;
    for (int k = 0; k < s.n; k++) t += A.part_sum[s.part0 + k];
    A.ll_out[s.w] = t;
    if (A.row_out0) A.row_out0[A.len_row ? A.len_row[s.w] : s.w] = t;
}

hipError_t launch_score_sum(const LoglikArgs &A, const ScoreSplit *splits, int n, hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(score_sum_kernel, dim3((n + 63) / 64), dim3(64), 0, st, A, splits, n);
    return hipGetLastError();
}


template <typename R, int BS, bool WIDE = false>
static hipError_t launch_t(const ModelDev &M, const LoglikArgs &A, int grid, hipStream_t st)
{
    // dynamic LDS above 64 KB needs the per-kernel limit raised (large trees only)
    if (loglik_use(A) == LoglikUse::Score) {
        const size_t sm = score_smem<R>(M.N) + loglik_eig_bytes(A);
        if (sm > 65536) {
            const hipError_t err = hipFuncSetAttribute((const void *)score_kernel<R, BS, WIDE>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)sm);
            if (err != hipSuccess) return err;
        }
        hipLaunchKernelGGL((score_kernel<R, BS, WIDE>), dim3(grid), dim3(BS), sm, st, M, A);
        return hipGetLastError();
    }
    auto keep = [&](auto U) {
        constexpr LoglikUse use = decltype(U)::value;
        const size_t sm = keep_smem<R>(M.N, BS, use == LoglikUse::History) + loglik_eig_bytes(A);
        if (sm > 65536) {
            const hipError_t err = hipFuncSetAttribute((const void *)keep_kernel<R, BS, use, WIDE>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)sm);
            if (err != hipSuccess) return err;
        }
        hipLaunchKernelGGL((keep_kernel<R, BS, use, WIDE>), dim3(grid), dim3(BS), sm, st, M, A);
        return hipGetLastError();
    };
    switch (loglik_use(A)) {
    case LoglikUse::History: return keep(std::integral_constant<LoglikUse, LoglikUse::History>());
    case LoglikUse::Candidates: return keep(std::integral_constant<LoglikUse, LoglikUse::Candidates>());
    default: return keep(std::integral_constant<LoglikUse, LoglikUse::Keep>());
    }
}

hipError_t launch_reset(int *q, hipStream_t st)
{
    hipLaunchKernelGGL(reset_queue, dim3(1), dim3(1), 0, st, q);
    return hipGetLastError();
}

template <typename R, int BS>
static int blocks_t(int N, LoglikUse use)
{
    const bool scores = use == LoglikUse::Score;
    const void *k = scores ? (const void *)score_kernel<R, BS>
                    : use == LoglikUse::History ? (const void *)keep_kernel<R, BS, LoglikUse::History>
                    : use == LoglikUse::Candidates ? (const void *)keep_kernel<R, BS, LoglikUse::Candidates>
                                                   : (const void *)keep_kernel<R, BS, LoglikUse::Keep>;
    const size_t sm = scores ? score_smem<R>(N) : keep_smem<R>(N, BS, use == LoglikUse::History);
    if (sm > 65536 && hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)sm) != hipSuccess) return 0;
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k, BS, sm) != hipSuccess) return 0;
    return nb;
}

int loglik_blocks_per_cu(int fp64, int BS, int N, LoglikUse use)
{
    if (fp64) {
        if (BS == 64) return blocks_t<double, 64>(N, use);
        if (BS == 128) return blocks_t<double, 128>(N, use);
        if (BS == 256) return blocks_t<double, 256>(N, use);
    } else {
        if (BS == 64) return blocks_t<float, 64>(N, use);
        if (BS == 128) return blocks_t<float, 128>(N, use);
        if (BS == 256) return blocks_t<float, 256>(N, use);
    }
    return 0;
}

hipError_t launch_loglik(const ModelDev &M, const LoglikArgs &A, int fp64, int BS, int grid, hipStream_t st)
{
    if (A.wide) return fp64 ? launch_t<double, WIDE_BLOCK, true>(M, A, grid, st) : launch_t<float, WIDE_BLOCK, true>(M, A, grid, st);
    if (fp64) {
        if (BS == 64) return launch_t<double, 64>(M, A, grid, st);
        if (BS == 128) return launch_t<double, 128>(M, A, grid, st);
        if (BS == 256) return launch_t<double, 256>(M, A, grid, st);
    } else {
        if (BS == 64) return launch_t<float, 64>(M, A, grid, st);
        if (BS == 128) return launch_t<float, 128>(M, A, grid, st);
        if (BS == 256) return launch_t<float, 256>(M, A, grid, st);
    }
    return hipErrorInvalidValue;
}

}  // namespace pa
