// kernels.hpp -- launch-side declarations shared by the host code and kernels.hip.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "device_model.hpp"

namespace edenhip {

// One multi-compartment cell as seen by tree_kernel.
struct TreeCell {
    int64_t comp_begin;   // first global compartment
    int32_t n;            // compartments
    int32_t longest;      // Hines rounds on the schedule's longest path (information)
    int32_t n_junction;   // nodes in the schedule's junction (information)
    int32_t words_off;    // offset of its schedule block (plan_tree_waves)
    int32_t words_len;    // length of that block in 32-bit words
    int32_t n_gate;       // gate variables (one per gate of every channel distribution)
    int64_t gate_off;     // offset of its gate variables
    int32_t n_input;      // compartments with Poisson inputs
    int32_t input_off;    // offset of its input-list entries
    int32_t n_ctask;      // gated channel distributions
    int32_t ctask_off;    // offset of its channel tasks
    int32_t n_cx;         // complex compartments (see TreeComplex)
    int32_t cx_off;       // offset of their records
    int32_t const_tree;   // 1: constant diagonals below the root (see tree_kernel)
    int32_t root_children;   // children of the root (BFS positions 1 .. root_children)
    int32_t lean;         // 1: a constant tree with no complex compartment but a root without
                          // inputs, synapses or channels of another pass (lean_tree_kernel)
    int32_t lean_len;     // its lean block, 32-bit words (a multiple of 4)
    int64_t lean_off;     // where it starts
};

// Per-compartment flag word of tree cells: 0 for a simple compartment (one ungated channel,
// no pulse, no Poisson input, no spike event column, not recorded), else TCX_COMPLEX | index
// of its TreeComplex record within the cell (bits 0-15; the kernel keeps the compartment's
// position in bits 16-26).
constexpr uint32_t TCX_COMPLEX = 1u << 31;

// Compartment word of the tree kernel: channel count (bits 0-2), gated-channel-slot mask
// (bits 3-6), Poisson-input flag (bit 7), chemical-synapse flag (bit 8), first channel task
// (bits 16-31).
constexpr uint32_t TCM_INPUT = 1u << 7;
constexpr uint32_t TCM_SYN = 1u << 8;
constexpr uint32_t TCM_XCH = 1u << 9;    // channels run in ext_channels_kernel (chmeta CHM_EXTERNAL)

constexpr int TREE_SLOTS = 4;        // compartments per thread



// Dynamic LDS of the tree kernel, in 4-byte units: Hines node records [nmax+1] of 16 bytes
// ((diagonal, rhs), (Ui, Uj)) | sIn [nmax] float2
// (only with Poisson inputs) | sV [nbuf][nvmax+1] | sQ [ngmax] | sGT [ngmax] | sF [nbuf][nctmax]
// | sCT [nctmax] | sIL [ninmax] | schedule block [words_max] (16-byte aligned) | sCX [cxmax]
// TreeComplex (only when the records are staged in LDS) | gate table [n_gates] DGate (n_gates 0
// where it is read from global memory) |
// synapse types [n_stypes] DSynType; nbuf = 2 when a separate wave runs the channel phase,
// else 1. nvmax: voltage slots of the bucket's cells (1 for a constant tree, whose only
// voltage read from LDS is the root's, else its compartment count).
struct TreeLds {
    int32_t node, in, v, q, gt, f, ct, il, w, cx, gtab, stab, total;
};

__host__ __device__ inline TreeLds tree_lds(int32_t nmax, int32_t nvmax, int32_t ngmax, int32_t nctmax,
                                            int32_t ninmax, int32_t words_max, int32_t cxmax, int32_t n_gates,
                                            int32_t n_stypes, bool split) {
    // the node records first, at the start of dynamic LDS: their address is then a constant,
    // which the compiler folds into the offsets of the Hines solve's LDS instructions
    TreeLds L;
    const int32_t nbuf = split ? 2 : 1;
    L.node = 0;
    L.in = L.node + 4 * (nmax + 1);
    L.v = L.in + (ninmax > 0 ? 2 * nmax : 0);
    L.q = L.v + nbuf * (nvmax + 1);
    L.gt = L.q + ngmax;
    L.f = L.gt + ngmax;
    L.ct = L.f + 2 * nctmax;                // open fractions, double-buffered
    L.il = L.ct + nctmax;
    L.w = (L.il + ninmax + 3) & ~3;         // task words, read up to 16 bytes at a time
    L.cx = (L.w + words_max + 3) & ~3;      // 16-byte records
    L.gtab = L.cx + 24 * cxmax;             // 64-byte DGate records (multiple of 4 units)
    L.stab = L.gtab + 16 * n_gates;         // 32-byte DSynType records
    L.total = L.stab + 8 * n_stypes;
    return L;
}

// Tables of the windowed network path for networks of one-compartment cells. Lane l of
// wave b advances point cell 64 b + l; its synapses use the block-interleaved slots of
// DevTables (synapse k at syn_base + 64 k). Ring word (step, b, w, l) =
// (step & ring_mask) * ring_stride + (b * nw + w) * 64 + l, bit j: synapse 32 w + j of that
// cell receives its event at that step. State arrays come in two copies: a window reads
// copy `cur` and writes copy `cur ^ 1`, so a window can be run again.
struct NetTables {
    int32_t n_blocks;              // waves of 64 point cells
    int32_t nw;                    // ring words per cell (ceil(max synapses per cell / 32))
    int32_t ring_mask;
    int64_t ring_stride;           // words per ring step = n_blocks * nw * 64
    const uint32_t *runs;          // [NC * 4] per compartment: type run end | type << 16, 0 = none
    float *gA[2], *gB[2];          // expTwo state per slot
    uint32_t *ring;                // [R * ring_stride]
    float *V[2], *q[2];            // compartment voltage and gate state
    float *poi_tsince[2], *poi_isi[2], *poi_A[2], *poi_B[2];
    uint64_t *spike_mask;          // [NC] spikes of the window, bit = step - window start
    int32_t *spk_list;             // compartments that spiked in the window
    uint32_t *spk_count;           // this window's count; the deliver kernel zeroes the next one's
    uint32_t *spk_count_next;
    const uint32_t *tgt_rw;        // per spike target (CSR spk_begin): ring word offset << 5 | bit
    int32_t *conflict;             // set when a window's result differs from step-by-step order
    unsigned long long *n_deliv;   // synaptic events received (spike-triggered), counted
};

// Device copy of the tables for what net_quad_kernel's step loop does seldom (events, Poisson
// intervals, second pulses): read through a pointer there, so that the loop does not keep all
// tables' addresses in registers.
struct NetRare {
    DevTables T;
};

// The synapse types a network uses, ascending, with what net_quad_kernel needs of each.
constexpr int NET_CLASSES = 4;
struct alignas(16) NetClass {
    float gbase, erev, jump;       // jump: weight property * waveform factor
    int32_t type;
    Recip2 rise, decay;            // of the time constants
};
struct NetClasses {
    int32_t n;                     // types in use, at most NET_CLASSES
    NetClass c[NET_CLASSES];
};

// net_quad_kernel holds a wave's synapses in groups of four slots a lane (16 synapses a cell); it
// is built for up to each of these numbers of groups. Registers: 8 a group.
constexpr int NET_QUAD_GROUPS[] = {1, 2, 4, 6, 8, 10, 12, 16};
constexpr int NET_QUAD_MAX = 16;

// form: a workgroup's threads without a channel wave (64, 128, 256, 512), plus 1 where the gate
// table is read from global memory (256 and 512 only), plus 2 in a network where a compartment's
// synapses are read eight at a time, plus 4 where its launches are of one step (64 only). net: the variant for networks (synapses on tree compartments,
// spikes sent to recipients), only without a channel wave. Null where there is none.
const void *tree_kernel_ptr(int form, bool split, bool net);
// Synapses of one compartment from which a bucket's kernel reads eight at a time, each a register
// set of its own: 48 trees of 20 to 150 compartments with 50 on each soma 11.9 -> 11.4 ms, 120 24.2 ->
// 22.1, 600 trees with 50 7.5 -> 6.7 (401 and 201 steps). Below, two at a time: most have one or two,
// and the same trees with 470 synapses in all take 2.3 ms, with eight at a time 2.6.
constexpr int SYN_MANY = 16;
// for buckets whose cells are all TreeCell::lean
const void *lean_tree_kernel_ptr(int tpb, bool split);
// Dynamic LDS of lean_tree_kernel: a few scalars, from LEAN_X on the right-hand sides (two more
// than nodes), then the cell's block, all multiples of 16 bytes.
constexpr uint32_t LEAN_X = 32;
__host__ __device__ inline int64_t lean_nodes(int64_t n) { return (n + 2 + 3) & ~(int64_t)3; }
inline int64_t lean_lds(int64_t lean_len, int64_t n) { return LEAN_X + 4 * (lean_nodes(n) + lean_len); }
const void *net_window_kernel_ptr();
const void *net_quad_kernel_ptr(int groups);
const void *net_deliver_kernel_ptr();
const void *point_kernel_ptr();
const void *ext_channels_kernel_ptr();
const void *point_quad_kernel_ptr();

}  // namespace edenhip
