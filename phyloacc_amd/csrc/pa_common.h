// pa_common.h -- plain structs shared by the host encoder and the device
// kernels: model constants, per-element descriptors and the node-table layout.
#pragma once
#include <stdint.h>

#if defined(__HIPCC__)
#define PA_TAB __host__ __device__ inline
#else
#define PA_TAB inline
#endif

namespace pa {

constexpr int MAXN = 512;          // max nodes per tree (S <= 256)
constexpr int GAPT = -0x40000000;  // scale-exponent sentinel: subtree has only gap/N leaves

// node flags (per element, per node id)
enum : uint32_t {
    NF_MISSING = 1u,       // BPP_C::missing
    NF_IN_TREE = 2u,       // in BPP_C::nodes (the element's, possibly collapsed, tree)
    NF_UPPER = 4u,         // in BPP::upper (outgroup lineage)
    NF_UPPER_CONS = 8u,    // in BPP::upper_conserve
    NF_LEAF = 16u,
};

// Model constants passed by value to every kernel.
struct ModelDev {
    int S, N, I;                 // species, nodes, internal-node slots (N - S)
    int T, burnin, mcmc, adapt_freq, ropt;
    double cub, nlb;
    double cprior_a, cprior_b, nprior_a, nprior_b;
    double init_crate, init_nrate, init_grate, init_lrate, init_lrate2;
    double ha_g, hb_g, ha_l, hb_l, ha_l2, hb_l2;
    double constomis, nconstomis;
    double pi[4];
    double lam[4];               // eigenvalues of Q
    double V[16], Vi[16];        // P(t)[i][j] = sum_k V[i][k] e^{lam_k t} Vi[k][j] = P_{i->j}
    uint32_t key0, key1;         // SEED
    int r1_shared;
};

// Per-element descriptor.  Offsets index the engine's arenas.
struct ElemDev {
    int GG, P, Ppad, root;
    int n_nodes, n_int, n_up;   // n_up: number of height levels
    int has_amb;
    int64_t off_codes;   // uint8 [S][Ppad] leaf codes, pattern index fastest
    int64_t off_w;       // int32 [P] pattern weights
    int64_t off_site;    // int32 [GG] site -> pattern
    int64_t off_tab;     // int32 node table (TAB_WORDS(N) words)
};

// Node table layout (int32 words, per element; N = model N).
//   ch0[N] ch1[N] par[N] flags[N] nodes[N] internal[N]
//   up[N] up_off[N+1] porder[N/2+1] dist2 (double, 2N words)
//   up: internal nodes of the element's tree by height (1, 2, ...);
//       level h occupies up[up_off[h-1] .. up_off[h]).
//   porder: the internal nodes in pruning order (post-order, the child with the
//       larger subtree first, child 0 on ties), PO_* words.
PA_TAB int tab_ch0(int N) { return 0; }
PA_TAB int tab_ch1(int N) { return N; }
PA_TAB int tab_par(int N) { return 2 * N; }
PA_TAB int tab_flags(int N) { return 3 * N; }
PA_TAB int tab_nodes(int N) { return 4 * N; }
PA_TAB int tab_int(int N) { return 5 * N; }
PA_TAB int tab_up(int N) { return 6 * N; }
PA_TAB int tab_upoff(int N) { return 7 * N; }
PA_TAB int tab_porder(int N) { return 8 * N + 1; }
// behind everything the tree's shape decides, so that a new tree's table can
// replace what lies before the lengths
PA_TAB int tab_dist(int N) { return (tab_porder(N) + N / 2 + 2) & ~1; }   // even -> 8-byte aligned doubles
PA_TAB int tab_words(int N) { return tab_dist(N) + 2 * N + 2; }           // even, so every table stays aligned

// A word of porder: the node; how many earlier nodes' partials are waiting
// for their parent when it is reached (its stack depth); and, when its parent
// comes more than two nodes later, that its partial waits in the slot given.
// A waiting partial's subtree is at least as large as the rest of its parent's
// (two internal nodes or more), so the depth stays below log2 of the nodes.
enum : uint32_t { PO_NODE = 0x3ffu, PO_DEPTH_SHIFT = 10, PO_DEPTH = 31u, PO_WAITS = 1u << 15, PO_SLOT_SHIFT = 16 };

}  // namespace pa
