// pa_kernels.h -- launch interface between the engine host code and the
// log-likelihood kernel in pa_engine.hip (the chain kernel: pa_chain.h).
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>
#include "pa_common.h"

#define PA_GAP_CODE 4
#define PA_OTHER_CODE 5
#define PA_STATUS_NUMERIC_FAIL 2
// chain failure and warning bits, as PA_FLAG_* in include/phyloacc_gpu.h
#define PA_F_NAN 1
#define PA_F_POS_INF 2
#define PA_F_NEG_INF 4
#define PA_F_SAMPLER 8
#define PA_F_PROPOSAL_RANGE 16

namespace pa {

// Patterns [p0, p1) of work position w (p0 a multiple of 64); part: see LoglikArgs.
struct ScoreItem { int w, p0, p1, part; };
// A split element's parts: work position w, parts [part0, part0 + n).
struct ScoreSplit { int w, part0, n; };

// Arguments of the log-likelihood launch.  Work position w evaluates element
// work[w] with row r = len_row[w] (or w) of the call's arrays: either at
// ancestral states Zin[r] and rates rates_in[r] over the element's stored
// branch lengths, or, when len_in is set, at the lengths len_in[r] with every
// branch at rate 1 (Zin, rates_in unused).
struct LoglikArgs {
    const ElemDev *elems;
    const int32_t *work;      // element ids in schedule order
    int n_work;
    int *queue;               // work counter, reset before each launch
    const uint8_t *codes;     // arenas
    int wide;                 // some element's codes are beyond a 32-bit offset (wide_codes)
    const int32_t *wts;
    const int32_t *tab;
    int n_elems;              // elements in the arenas: ids outside [0, n_elems) score NaN
    char *scratch;            // one slot per workgroup
    int64_t slot_bytes;
    // Elements too long for a slot: work position w keeps its partials at
    // big + big_off[w] (loglik_resident_bytes of its Ppad); big_off[w] < 0,
    // or big_off null, means the workgroup's slot.
    char *big;
    const int64_t *big_off;
    // Resident partials (gene-tree height moves), or null: every work
    // position's partials stay at big + big_off[w] (loglik_resident_bytes of
    // its Ppad), node x's in slot x - S; stale[r][x] != 0 says that row r's
    // stored partial of x is not its current tree's.  A row with path_node[r]
    // >= 0 scores the path from that node to the root and stores none of it;
    // the stale nodes off the path that it needs are stored first, and marked
    // current.
    uint8_t *stale;
    const int32_t *path_node;
    const int32_t *Zin;       // [rows][N] (when len_in is null)
    const double *rates_in;   // [rows][2] (r1, r2) (when len_in is null)
    const double *len_in;     // [rows][N] per-call branch lengths, or null
    const int32_t *len_row;   // [n_work] the call's row of each work position, or null (row w)
    double *ll_out;           // [n_work]
    // gBGC substitution model, or null: branch s of row r takes P(dist) of
    // class k = c(Z) + 3 * (Bin[r][s] != 0), c(0) = 0 (background), c(2) = 2
    // (accelerated), else 1 (conserved), whose eigensystem is gb_eig[r][k] =
    // {lam[4], V[16], Vi[16]} (gbgc_eig_kernel).
    const double *gb_eig;     // [rows][6][GB_EIG_WORDS]
    const int32_t *Bin;       // [rows][N]
    unsigned long long *counters;   // [0] += algorithmic HBM bytes of the launch, or null
    // Per-element substitution model for the own-tree path, or null: work
    // position w prunes with the eigensystem el_eig[w] = {lam[4], V[16],
    // Vi[16]} and sums its root with the base frequencies el_pi[w][4]
    // (gt_eig_kernel).
    const double *el_eig;     // [n_work][GB_EIG_WORDS]
    const double *el_pi;      // [n_work][4]
    // Work items of a launch that only scores, or null (item i = work position
    // i, all its patterns): n_items ranges of patterns.  An item with part >=
    // 0 covers part of its element and leaves its sum in part_sum[part]; the
    // sums of a split element are then added in order (launch_score_sum).
    const struct ScoreItem *items;
    int n_items;
    double *part_sum;
    // Two site prefixes per caller row, or null: instead of the pattern sum,
    // the root sums run over the element's sites, g < pre_len[r][0] into
    // ll_out and g < pre_len[r][1] into ll_out2 (r = len_row[w], or w; the
    // site -> pattern map is `site`).
    const int32_t *pre_len;   // [rows][2]
    double *ll_out2;          // [n_work]
    // The log-likelihoods by caller row as well, or null (device-resident
    // callers): row_out0[r] = ll_out, row_out1[r] = ll_out2.
    double *row_out0, *row_out1;
    // PhyloAcc-GT gene-tree moves.  Arrays below are per caller row: work
    // position w uses row len_row[w] (or w).
    // Per-call trees, or null: row r prunes the tree of node table
    // tab_call[r] (tab_words(N) words; children, parents, flags, post-order,
    // levels) with root, node count and level count in hdr_call[r][0..2].
    const int32_t *tab_call;
    const int32_t *hdr_call;  // [rows][4]
    const int32_t *site;      // the site -> pattern arena (ElemDev::off_site)
    // Gene-node histories, or null: row r's lives at hist + hist_off[r],
    // node v's sites at v * hist_ns[r] from there (int8: leaves 0-3, -1
    // ambiguous, 4 no base; internal nodes their drawn base, 4 when missing).
    // hist_draw: after pruning, draw sites g < hist_len[r] there (tag
    // GT_HIST, sub-stream g, sweep hist_sweep, slot v); else the history is
    // only read, by the candidate scores.
    int8_t *hist;
    const int64_t *hist_off;
    const int32_t *hist_ns, *hist_len;
    int hist_draw, hist_sweep;
    // Candidate scores, or null: for row r, branch cand_branch[r] and
    // candidates q < cand_n[r] (node cand_node, kind cand_kind, distance
    // cand_len; cand_max per row), sum over sites g < cand_sites[r] the score
    // of kind 0 (node's base, or the pi-average when it has none), 1 (the
    // pi-average) or 2 (the branch's own base's pi-row) into cand_score,
    // reading the history.
    const int32_t *cand_branch, *cand_n, *cand_node, *cand_kind, *cand_sites;
    const double *cand_len;
    int cand_max;
    double *cand_score;
};

constexpr int GB_CLASSES = 6, GB_EIG_WORDS = 36;

// Eigensystems of the six gBGC classes of every work position: class k has
// selection 0, sel[w][0] (conserved) or sel[w][1] (accelerated) for k % 3 =
// 0, 1, 2, and bias sel[w][2] when k >= 3, else 0 (Q from Q0 by gbgc_rate).
// A class whose Q is not time-reversible gets NaN eigenvalues.
hipError_t launch_gbgc_eig(const double *Q0 /*[16], host*/, const double *sel /*[n][3], device*/, int n,
                           double *eig /*[n][6][36], device*/, hipStream_t st);

// Eigensystem and base frequencies of PhyloAcc-GT's strand-symmetric model
// for every work position: pi = (a, 1/2 - a, 1/2 - a, a) with a = piA[w],
// Q from the six exchangeabilities inst (gt_strand_q).  A non-reversible
// result gets NaN eigenvalues.
hipError_t launch_gt_eig(const double *inst /*[6], host*/, const double *piA /*[n], device*/, int n,
                         double *eig /*[n][36], device*/, double *pi /*[n][4], device*/, hipStream_t st);

// What a launch is for: log-likelihoods alone; resident partials; candidate
// scores; a history draw.
enum class LoglikUse { Score, Keep, Candidates, History };
// LDS bytes of one workgroup of BS threads, without the eigensystems of loglik_eig_bytes.
size_t loglik_smem_bytes(int N, int fp64, int BS, LoglikUse use);
// Bytes of one workgroup's HBM slot for elements of up to Pcap (padded)
// patterns: the partials (4 values each) and exponents of every internal node.
size_t loglik_slot_bytes(int N, int S, int Pcap, int fp64);
// Bytes of one element's resident partials at Ppad patterns, and its root terms.
size_t loglik_resident_bytes(int N, int S, int Ppad, int fp64);
// Bytes of one workgroup's HBM slot in a launch that only scores: the stacks
// of its waves, and with site prefixes the terms of Pcap (padded) patterns
// (Pcap 0: none).  Never more than loglik_slot_bytes of the element's own
// padded patterns, so a launch with such slots can score too.
size_t score_slot_bytes(int N, int S, int BS, int Pcap, int fp64);
// LDS of the eigensystems of a launch whose work positions have their own.
size_t loglik_eig_bytes(const LoglikArgs &A);
inline LoglikUse loglik_use(const LoglikArgs &A)
{
    return A.hist_draw ? LoglikUse::History : A.cand_score ? LoglikUse::Candidates : A.stale ? LoglikUse::Keep : LoglikUse::Score;
}
// Workgroups resident on one CU (registers, LDS, launch bound).
int loglik_blocks_per_cu(int fp64, int BS, int N, LoglikUse use);
// A launch over arenas with wide codes takes WIDE_BLOCK threads whatever BS
// says (the one size that such kernels are built for).
constexpr int WIDE_BLOCK = 256;
inline bool wide_codes(int S, int64_t Ppad) { return S * Ppad >= (int64_t)1 << 32; }
hipError_t launch_loglik(const ModelDev &M, const LoglikArgs &A, int fp64, int BS, int grid, hipStream_t st);

// Size of the device scratch array of the allocation-free likelihood entry
// point, and the device address of the current device's copy (looked up once
// per device with that device current).
constexpr size_t NOALLOC_SCRATCH_BYTES = (size_t)256 << 20;
hipError_t noalloc_scratch(int device, char **ptr);
hipError_t launch_reset(int *q, hipStream_t st);
// The split elements' log-likelihoods from their parts' sums.
hipError_t launch_score_sum(const LoglikArgs &A, const ScoreSplit *splits, int n, hipStream_t st);

}  // namespace pa
