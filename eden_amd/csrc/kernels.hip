// kernels.hip -- gfx950 kernels of the per-timestep loop.
//
//  point_kernel   one lane per single-compartment cell; time loop inside the launch, state in
//                 registers (a launch may cover one step, as in the network path).
//  point_quad_kernel  four lanes per uncoupled single-compartment cell, each advancing one
//                 of its gate variables beside the voltage update.
//  tree_kernel    one workgroup (TPB threads, one or more wave64s) per multi-compartment
//                 cell, popped from a work queue sorted by compartment count (largest first);
//                 compartment state in registers (4 compartments per thread), the Hines solve
//                 in LDS as rounds of independent per-node gathers. The gather at each tree
//                 node folds its children in ascending index order, which is the order EDEN's
//                 serial depth-first elimination (eden/Eden.cpp:6114-6225) applies them, so
//                 every diagonal and right-hand-side value sees the same operations in the
//                 same order as the serial chain.
#include "device_model.hpp"
#include "kernels.hpp"
#include "tree_schedule.hpp"

namespace edenhip {

__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(1, 2)))
point_kernel(DevTables T, const DGate *__restrict__ gates_g, int n_gates, const DSynType *__restrict__ stypes_g,
             int n_stypes, const int32_t *__restrict__ comps, int32_t n, int64_t s0, int64_t s1, int64_t row0,
             float dt) {
    __shared__ DGate gates[MAX_CHAN_TYPES * GATES_PER_TYPE];
    __shared__ DSynType stypes[64];
    for (int i = threadIdx.x; i < n_gates; i += blockDim.x) gates[i] = gates_g[i];
    for (int i = threadIdx.x; i < n_stypes; i += blockDim.x) stypes[i] = stypes_g[i];
    __syncthreads();
    const int32_t idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= n) return;
    const int64_t g = comps[idx];
    CompConst k;
    load_comp_const(T, g, k);
    float V = T.V[g];
    float q[NQ];
#pragma unroll
    for (int s = 0; s < NQ; s++) q[s] = T.q[g * NQ + s];
    const int32_t syn_base = T.syn_base[g], syn_cnt = T.syn_cnt[g];
    const bool has_syn = syn_cnt > 0;
    const bool has_poi = T.poi_begin[g + 1] > T.poi_begin[g];
    const bool has_spk = T.spk_begin[g + 1] > T.spk_begin[g];

    // time_f64 accumulates `time += dt` in double, as the reference's engine loop does
    double time = (s0 >= 1) ? T.t_row[s0 - 1] : 0.0;
    for (int64_t s = s0; s < s1; s++) {
        const bool init = s <= 0;
        const float t = (float)time;
        const int now = (int)((s + 3) & 1), nxt = now ^ 1;
        if (!init && k.rec >= 0) trace_at(T, k.rec, s - 1 - row0) = V;
        float I_ch, G_ch;
        channels_step(gates, k, V, q, init, dt, I_ch, G_ch);
        if (k.chmeta == CHM_EXTERNAL) {
            const float2 e = T.chx_ext[g];   // channels of this step (ext_channels_kernel)
            I_ch = e.x;
            G_ch = e.y;
        }
        float I_syn = 0.0f, G_syn = 0.0f;
        if (has_syn) {
            if (T.syn_ext) {
                const float2 e = T.syn_ext[g];   // generic synapses of this step (lems_syn_kernel)
                I_syn = e.x;
                G_syn = e.y;
            } else {
                synapses_step<8>(T, stypes, syn_base, syn_cnt, V, init, t, dt, now, s, I_syn, G_syn);
            }
        }
        float I_in = pulses_current(T, k, g, t), G_in = 0.0f;
        if (has_poi) {
            const PoiState ps{T.poi_tsince, T.poi_isi, T.poi_A, T.poi_B};
            poisson_step(T, stypes, g, V, init, s, dt, I_in, G_in, ps, ps);
        }
        if (T.inp_ext && has_syn) {
            const float2 e = T.inp_ext[g];   // LEMS inputs of this step, after the native ones
            I_in += e.x;
            G_in += e.y;
        }
        const float I_int = I_ch + I_in + I_syn;
        const float G_int = G_ch + G_in + G_syn;
        float D = 1 * (G_int / k.C) + k.invrc;
        float Vn;
        if (init) {
            Vn = V;
        } else {
            Vn = V + (dt * (I_int + ((V * G_int))) / k.C);
            D = 1 + D * dt;     // one-compartment tree: no elimination, root divide only
            Vn = Vn / D;
        }
        if (V < k.vthr && k.vthr < Vn) {
            if (has_spk) send_spike(T, g, nxt, (int)(s - s0));
            log_event(T, k.ev, s);
        }
        V = Vn;
        if (!init) time += (double)dt;
    }
    T.V[g] = V;
#pragma unroll
    for (int s = 0; s < NQ; s++) T.q[g * NQ + s] = q[s];
}

// Uncoupled one-compartment cells (no synapses, Poisson inputs or spike recipients), four
// lanes per cell: lane s of the quad forms channel s's current and advances gate variable s
// (QuadChannels); every lane forms the cell's sums and voltage update identically. A step's
// currents use the present gate values, while the gate updates feed only the next step
// (eden/Eden.cpp:5330: each gate's present value enters the open fraction before it is
// updated), so the gates' rate and exp chains run side by side and beside the voltage update
// instead of one after another. Bound by the issue of one wave's instructions: 1,000 cells
// 1.46 us a step with a loop over each gate's powers and fp32 divisions, now 0.81 us.
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(1, 2)))
point_quad_kernel(DevTables T, const DGate *__restrict__ gates_g, const int32_t *__restrict__ comps,
                  int32_t n, int64_t s0, int64_t s1, int64_t row0, float dt) {
    const int32_t gid = blockIdx.x * blockDim.x + threadIdx.x;
    const int32_t at = gid >> 2, qs = gid & 3;
    const bool valid = at < n;
    const int64_t g = comps[valid ? at : n - 1];   // spare quads repeat the last cell and store nothing
    CompConst k;
    load_comp_const(T, g, k);
    const double rC = 1.0 / (double)k.C;
    float V = T.V[g];
    float qv = T.q[g * NQ + qs];   // gate variable qs of the cell
    QuadChannels ch;
    ch.load(gates_g, k, qs);
    // time_f64 accumulates `time += dt` in double, as the reference's engine loop does
    double time = (s0 >= 1) ? T.t_row[s0 - 1] : 0.0;
    for (int64_t s = s0; s < s1; s++) {
        const bool init = s <= 0;
        const float t = (float)time;
        if (!init && k.rec >= 0 && qs == 0 && valid) trace_at(T, k.rec, s - 1 - row0) = V;
        float I_ch, G_ch;
        ch.currents(qv, V, I_ch, G_ch);
        const float nv = ch.next(qv, V, init, dt);
        const float I_in = pulses_current(T, k, g, t), G_in = 0.0f;
        const float I_syn = 0.0f, G_syn = 0.0f;
        const float I_int = I_ch + I_in + I_syn;
        const float G_int = G_ch + G_in + G_syn;
        const float Vn = init ? V : point_update(V, I_int, G_int, k.invrc, rC, dt);
        if (V < k.vthr && k.vthr < Vn && qs == 0 && valid) log_event(T, k.ev, s);
        V = Vn;
        qv = nv;
        if (!init) time += (double)dt;
    }
    if (valid) {
        if (qs == 0) T.V[g] = V;
        T.q[g * NQ + qs] = qv;
    }
}

// LDS-only workgroup barrier: waits for this wave's LDS operations, then (for more than one
// wave) the hardware barrier. Outstanding global loads/stores (the trace write, the next
// step's time prefetch) are not drained, unlike __syncthreads().
// A single wave needs no wait at all: LDS executes one wave's instructions in issue order,
// so a later read sees an earlier write; only the compiler must not reorder across it.
template <int TPB>
__device__ __forceinline__ void lds_barrier() {
    if constexpr (TPB <= 64) {
        __builtin_amdgcn_wave_barrier();
        asm volatile("" ::: "memory");
    } else {
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    }
}

// Open fraction of every channel of a compartment from its gate values (in gate order,
// each multiplied in `instances` times, eden/Eden.cpp:5679-5721), then the channel current
// and conductance sums in distribution order (eden/Eden.cpp:5805-5898).
__device__ __forceinline__ void tree_channels(const CompConst &k, uint32_t tcm, const float *sF, float V, float &I_ch,
                                              float &G_ch) {
    // channel slot c uses the open fraction of its channel task (gated channels, in slot
    // order from the compartment's first task) or 1 (conductance_scaling alone)
    const int nch = tcm & 7;
    const uint32_t mask = (tcm >> 3) & 15;
    int idx = tcm >> 16;
    I_ch = 0.0f; G_ch = 0.0f;
#pragma unroll
    for (int c = 0; c < NCH; c++) {
        const bool gated = (mask >> c) & 1;
        const float f = gated ? sF[idx] : 1.0f;
        idx += gated ? 1 : 0;
        const float Gscaled = k.g[c] * f;
        const float iDensity = Gscaled * (k.e[c] - V) * 1e-5f;
        const float gDensity = (Gscaled) * 1e-5f;
        I_ch = (c < nch) ? I_ch + (iDensity * k.A) : I_ch;
        G_ch = (c < nch) ? G_ch + (gDensity * k.A) : G_ch;
    }
}

// Open fraction of a channel from its gate values, multiplied in gate order, each gate
// `instances` times, starting from conductance_scaling = 1 (eden/Eden.cpp:5679-5721).
__device__ __forceinline__ float channel_fopen(const DGate *gates, int type, const float *q) {
    const int ng = gates[type * GATES_PER_TYPE].forms >> 24;
    float f = 1.0f;
    for (int gi = 0; gi < ng; gi++) {
        const int inst = (gates[type * GATES_PER_TYPE + gi].forms >> 16) & 0xFF;
        const float qv = q[gi];
        for (int i = 0; i < inst; i++) f = f * qv;
    }
    return f;
}

// Channel phase of a cell, on the lanes `lane` + `stride` k of the channel group: every gate
// variable's next value from its compartment's voltage (one lane per gate), then, after
// `sync`, each gated channel's open fraction for the next step (one lane per channel).
template <class Sync>
__device__ __forceinline__ void channel_phase(const DGate *gates, const uint32_t *sCT, const uint32_t *sGT, float *sQ,
                                              float *sF_out, const float *sV_in, int NG, int NCT, int lane,
                                              int stride, bool init, float dt, Sync sync) {
    for (int g = lane; g < NG; g += stride) {
        const uint32_t gt = sGT[g];
        const uint32_t w = sCT[gt & 0xFFFFu];
        const int type = (w >> 11) & 63;
        sQ[g] = gate_next(gates[type * GATES_PER_TYPE + (gt >> 16)], sV_in[w & 0x7FF], sQ[g], init, dt);
    }
    sync();
    for (int i = lane; i < NCT; i += stride) {
        const uint32_t w = sCT[i];
        sF_out[i] = channel_fopen(gates, (w >> 11) & 63, sQ + (w >> 17));
    }
}

// One workgroup per multi-compartment cell, cells popped from a queue in decreasing size.
// The cable group (TPB threads) owns compartments t + TPB j (j < 4) in registers and runs,
// per step:
//   inputs     per-cell list of compartments with Poisson inputs -> sIn (LDS)
//   membrane   currents from the channels' open fractions (sF) and inputs, semi-implicit RHS
//   Hines      in LDS on breadth-first positions (tree_schedule.hpp): a 16-byte record per
//              node, (diagonal, rhs) then (Ui, Uj) of the edge to its parent, one task word per
//              thread per round
//   readback   new voltages, spike detection
// The channel phase (next gate values and open fractions from the present voltages) runs
// either in the cable group after the membrane phase, or, with SPLIT, in one extra wave at
// the same time as the cable group's step; voltages and open fractions are then
// double-buffered and the two meet at one workgroup barrier per step.
// A step is bound by the latency of its rounds, one wave's dependent trips through LDS: a round
// takes its header from a lane, reads everything before its first use and divides by constants
// through double (div_c); the root's update runs its channels on a quad (QuadChannels). 7 trees of up
// to 300 compartments, 1,004 steps and their rows read: 4.1 -> 3.6 ms.
// NET: networks, launched for a window of steps shorter than every delay (see trig_fold_kernel),
// else one step at a time. A compartment with chemical synapses
// (TCM_SYN) runs them in its complex update, with the trigger flags of the step's parity as
// the point kernel does, and a compartment with spike recipients sends its spikes to the
// next step's flags; both are complex compartments, so the per-slot code of the other
// compartments is unchanged and the NET = false kernels carry none of it.
// FORM: the cable group's threads, and
//   1 more where the gate table, up to 16 KiB, is read from global memory. That is for the largest
//     cells, whose other tables leave no room for it: a binary tree with HH channels on every
//     compartment, in a model of 64 channel types, takes up to 1,743 compartments with the table in
//     LDS and 1,937 without.
//   2 more where a compartment's synapses are read eight at a time (a bucket with a long list,
//     SYN_MANY), else two.
//   4 more where such a bucket's launches are of one step: compiled for two waves a SIMD, a launch
//     loads and stores no spilled registers (600 trees of 20 to 300 compartments with 50 synapses on
//     each soma 17.7 -> 17.1 ms, 4,000 of 20 to 100 with 30 23.0 -> 16.5). With windows it leaves too few
//     cells in flight (2,000 of 20 to 150 with 20 2.8 -> 3.4 ms), and so it does beyond 64 threads (500
//     of 100 to 600 with 40 9.6 -> 10.2).
template <int FORM, bool SPLIT, bool NET>
__global__ void __launch_bounds__((FORM & ~7) + (SPLIT ? 64 : 0)) __attribute__((amdgpu_waves_per_eu((FORM & 4) ? 2 : 4)))
tree_kernel(DevTables T, const DGate *__restrict__ gates_g, int n_gates, const DSynType *__restrict__ stypes_g,
            int n_stypes, const TreeCell *__restrict__ cells, const int32_t *__restrict__ task_order, int32_t n_tasks,
            int32_t *__restrict__ queue, const uint32_t *__restrict__ words_g, const int32_t *__restrict__ pos_g,
            const float2 *__restrict__ u_g, const uint32_t *__restrict__ tcm_g, const uint32_t *__restrict__ ctask_g,
            float *__restrict__ gq_g, const uint32_t *__restrict__ gt_g, const uint32_t *__restrict__ inl_g,
            const uint32_t *__restrict__ cflag_g, const TreeComplex *__restrict__ cx_g, int32_t cxmax_lds, int32_t nmax,
            int32_t nvmax, int32_t ngmax, int32_t nctmax, int32_t ninmax, int32_t words_max, int64_t s0, int64_t s1,
            int64_t row0, float dt) {
    constexpr int TPB = FORM & ~7;
    constexpr bool GATES_LDS = (FORM & 1) == 0;
    constexpr int K = TREE_SLOTS;
    constexpr int NT = TPB + (SPLIT ? 64 : 0);
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ int32_t s_task;
    // dynamic LDS, laid out by tree_lds()
    const TreeLds L =
        tree_lds(nmax, nvmax, ngmax, nctmax, ninmax, words_max, cxmax_lds, GATES_LDS ? n_gates : 0, n_stypes, SPLIT);
    float *sm = reinterpret_cast<float *>(smem);
    const DGate *const gates = GATES_LDS ? reinterpret_cast<const DGate *>(sm + L.gtab) : gates_g;
    DSynType *stypes = reinterpret_cast<DSynType *>(sm + L.stab);
    TreeComplex *sCX = reinterpret_cast<TreeComplex *>(sm + L.cx);
    // Hines node records, 16 bytes at position p: sDX(p) = (diagonal, rhs), then sU(p) =
    // (Ui, Uj) of the edge from p to its parent; one record serves a task's reads of both
    char *const nodes = reinterpret_cast<char *>(sm + L.node);
    auto sDX = [nodes](int p) -> float2 & { return *reinterpret_cast<float2 *>(nodes + 16 * p); };
    auto sU = [nodes](int p) -> float2 & { return *reinterpret_cast<float2 *>(nodes + 16 * p + 8); };
    float2 *sIn = reinterpret_cast<float2 *>(sm + L.in);
    float *sVb = sm + L.v;
    float *sQ = sm + L.q;
    uint32_t *sGT = reinterpret_cast<uint32_t *>(sm + L.gt);
    float *sFb = sm + L.f;
    uint32_t *sCT = reinterpret_cast<uint32_t *>(sm + L.ct);
    uint32_t *sIL = reinterpret_cast<uint32_t *>(sm + L.il);
    uint32_t *sW = reinterpret_cast<uint32_t *>(sm + L.w);   // schedule block: round headers, task words
    const int tid = threadIdx.x;
    const bool cable = !SPLIT || tid < TPB;
    if constexpr (GATES_LDS)
        for (int i = tid; i < n_gates; i += NT) reinterpret_cast<DGate *>(sm + L.gtab)[i] = gates_g[i];
    for (int i = tid; i < n_stypes; i += NT) stypes[i] = stypes_g[i];

    for (;;) {
        __syncthreads();
        if (tid == 0) s_task = atomicAdd(&queue[0], 1);
        __syncthreads();
        const int32_t task = s_task;
        if (task >= n_tasks) break;
        const TreeCell cell = cells[task_order[task]];
        const int32_t N = cell.n;
        const int32_t NG = cell.n_gate;
        const int32_t NCT = cell.n_ctask;
        const int32_t NIN = cell.n_input;
        const int64_t c0 = cell.comp_begin;
        const int64_t gq0 = cell.gate_off;
        // const_tree: every non-root compartment has a constant diagonal (ungated channels,
        // no conductance input), so below the root the eliminated diagonals D' and the ratios
        // Uj / D' are the same every step. They are computed once per task below, with the
        // per-step operations, and the forward sweep then reads the ratio in place of Uj.
        const bool const_tree = cell.const_tree != 0;
        {
            const uint32_t *Wg = words_g + cell.words_off;
            for (int i = tid; i < cell.words_len; i += NT) sW[i] = Wg[i];
        }
        // Hines task lists (tree_schedule.hpp, plan_tree_waves): cable wave wv runs the lists
        // of its subtrees, wave 0 also those of the junction. run_list calls body(word) round
        // after round with no barrier (a wave's LDS accesses are performed in order), on the
        // lanes below the round's task count. Task words hold byte offsets of node records, which
        // start at a constant LDS address. Every lane reads a word from the round (the block ends
        // with padding for the lanes beyond a round's count).
        // A list's round headers are kept a lane each (read again every 62 rounds), so a round
        // takes its header from a lane instead of from LDS. The loop is unrolled twice: after a
        // round's body is issued, the words of the round after next are read into the registers
        // that the round had used, complete before their use and with no register moved.
        constexpr int W = TPB / 64;
        const int wv = tid >> 6, lane = tid & 63;
        const uint32_t dummy_off = 16u * (uint32_t)N;
        char *const dxb = nodes;       // task words: byte offsets 16 p of node records
        char *const ub = nodes + 8;
        struct List {
            int first, cnt;     // first round header, rounds
            uint32_t hv;        // lane r: header r
        };
        auto load_list = [&](int dir) {
            List L;
            const uint32_t e = __builtin_amdgcn_readfirstlane(sW[dir]);
            L.first = e & 0xFFFFu;
            L.cnt = e >> 16;
            L.hv = sW[L.first + lane];
            return L;
        };
        auto run_list = [&](const List &L, auto type, auto body) {
            using Word = decltype(type);
            if (L.cnt == 0) return;
            uint32_t hv = L.hv;
            int hbase = 0;
            auto head = [&](int r) -> uint32_t {
                if (__builtin_expect(r - hbase >= 64, 0)) {
                    // (read and used here, so that the usual way waits for no LDS access)
                    hbase = r;
                    hv = sW[L.first + r + lane];
                    return (uint32_t)__builtin_amdgcn_readlane(hv, 0);
                }
                return (uint32_t)__builtin_amdgcn_readlane(hv, r - hbase);
            };
            auto word = [&](uint32_t h) { return reinterpret_cast<const Word *>(sW + (h & 0xFFFFu))[lane]; };
            uint32_t ha = head(0), hb = head(1);
            Word wa = word(ha), wb = word(hb);
            for (int r = 0;;) {
                if ((uint32_t)lane < (ha >> 16)) body(wa);
                if (++r >= L.cnt) break;
                ha = head(r + 1);
                wa = word(ha);
                if ((uint32_t)lane < (hb >> 16)) body(wb);
                if (++r >= L.cnt) break;
                hb = head(r + 1);
                wb = word(hb);
            }
        };
        // constant trees take four-word fold tasks with merged children (plan_tree_waves
        // with merge): c0, c1 and the grandchildren refolded through each, dummy where absent
        const uint4 fold4{};
        const uint2 fold2{}, bwd2{};
        for (int i = tid; i < N; i += NT) sU(i) = u_g[c0 + i];
        for (int i = tid; i < NG; i += NT) {
            sQ[i] = gq_g[gq0 + i];
            sGT[i] = gt_g[gq0 + i];
        }
        for (int i = tid; i < NCT; i += NT) sCT[i] = ctask_g[cell.ctask_off + i];
        for (int i = tid; i < NIN; i += NT) sIL[i] = inl_g[cell.input_off + i];
        // complex-compartment records: staged in LDS when the bucket's largest count fits,
        // else read from global memory
        const TreeComplex *CX = cx_g + cell.cx_off;
        if (cxmax_lds > 0) {
            const uint4 *src = reinterpret_cast<const uint4 *>(cx_g + cell.cx_off);
            uint4 *dst = reinterpret_cast<uint4 *>(sCX);
            for (int i = tid; i < cell.n_cx * (int)(sizeof(TreeComplex) / 16); i += NT) dst[i] = src[i];
            CX = sCX;
        }
        // voltages read from LDS: the root's in a constant tree (no gated channel or input
        // below it), else every compartment's
        const int32_t NV = const_tree ? 1 : N;
        for (int i = tid; i < NV; i += NT) sVb[i] = T.V[c0 + i];
        if (tid == 0) {
            // dummy slot for threads without a task: finite values, never read back
            sU(N) = make_float2(0.0f, 0.0f);
            sDX(N) = make_float2(1.0f, 0.0f);
        }

        // Per slot registers: voltage, BFS position, flag word, trace column, and for a simple
        // compartment its channel's Gbase and Erev, area, capacitance, and the conductance sum
        // and Hines diagonal, which do not change from step to step (computed here with the
        // per-step operation order). A complex compartment's constants come from its record.
        // Slots beyond the cell behave as simple compartments with no channel conductance,
        // C = 1 and the dummy position N, so they compute exactly the dummy slot's (1, 0).
        float V[K], g0[K], e0[K], Ar[K], Gs[K], Ds[K];
        double rC[K];           // 1 / C (div_c)
        // fl: the compartment's flag word (TCX_COMPLEX | record index, or 0) | BFS position << 16
        uint32_t fl[K];
        auto posof = [&](int j) { return (int)((fl[j] >> 16) & 0x7FFu); };
        bool slot_any[K], slot_simple[K], slot_cx[K];   // per wave and slot: any valid lane, no complex
                                                        // lane but the root's, any complex lane
        const int wbase = __builtin_amdgcn_readfirstlane(tid & ~63);
#pragma unroll
        for (int j = 0; j < K; j++) {
            const int c = tid + TPB * j;
            const bool valid = cable && c < N;
            V[j] = 0.0f; g0[j] = 0.0f; e0[j] = 0.0f; Ar[j] = 0.0f; rC[j] = 1.0; Gs[j] = 0.0f; Ds[j] = 1.0f;
            fl[j] = (uint32_t)N << 16;
            if (valid) {
                const int64_t g = c0 + c;
                fl[j] = cflag_g[g] | ((uint32_t)pos_g[g] << 16);
                V[j] = T.V[g];
                if (!(fl[j] & TCX_COMPLEX)) {
                    g0[j] = T.chg[g * NCH];
                    e0[j] = T.che[g * NCH];
                    Ar[j] = T.A[g];
                    rC[j] = 1.0 / (double)T.C[g];
                    const float G_ch = 0.0f + (((g0[j] * 1.0f) * 1e-5f) * Ar[j]);
                    const float G_int = (G_ch + 0.0f) + 0.0f;
                    const float Dd = 1 * (G_int / T.C[g]) + T.invrc[g];
                    Gs[j] = G_int;
                    Ds[j] = 1 + Dd * dt;
                }
            }
            slot_any[j] = __builtin_amdgcn_readfirstlane(wbase + TPB * j) < N && cable;
            // the root (thread 0, slot 0) is updated separately, after wave 0's fold rounds
            slot_simple[j] = __ballot(valid && c != 0 && (fl[j] & TCX_COMPLEX)) == 0ull;
            slot_cx[j] = __ballot(valid && (fl[j] & TCX_COMPLEX)) != 0ull;
        }
        __syncthreads();
        // the Hines lists of this wave (for the channel wave, unused) and of the junction
        const int lw = cable ? wv : 0;
        const List Lf = load_list(2 * lw), Lb = load_list(2 * lw + 1);
        const List Ljf = load_list(2 * W), Ljb = load_list(2 * W + 1);
        if (const_tree) {
            // eliminated diagonals of the constant subtrees: the forward sweep's diagonal part
            // on this step-independent matrix, with the per-step operations
#pragma unroll
            for (int j = 0; j < K; j++) {
                const int c = tid + TPB * j;
                if (cable && c < N) {
                    float Dr = Ds[j];
                    if (fl[j] & TCX_COMPLEX) {
                        const TreeComplex &cx = CX[fl[j] & 0xFFFFu];
                        const CompConst k = cx.k;
                        float I_ch, G_ch;
                        tree_channels(k, cx.tcm, sFb, V[j], I_ch, G_ch);
                        const float G_in = 0.0f, G_syn = 0.0f;
                        const float G_int = G_ch + G_in + G_syn;
                        const float Dd = 1 * (G_int / k.C) + k.invrc;
                        Dr = 1 + Dd * dt;
                    }
                    sDX(posof(j)) = make_float2(Dr, 0.0f);
                }
            }
            __syncthreads();
            // a fold task's diagonal part; a merged child's eliminated diagonal is formed again
            // from its children, as that child's own task forms it in the same round (the
            // dummy slot, D 1 and U 0, gives exactly zero terms for an unmerged child)
            auto diag_task = [&](uint4 w) {
                const uint32_t po = w.x & 0xFFFFu, ao = w.x >> 16, bo = w.y & 0xFFFFu;
                auto dprime = [&](uint32_t c, uint32_t g0, uint32_t g1) {
                    const float dc = reinterpret_cast<const float2 *>(dxb + c)->x;
                    const float d0 = reinterpret_cast<const float2 *>(dxb + g0)->x;
                    const float d1 = reinterpret_cast<const float2 *>(dxb + g1)->x;
                    const float2 u0 = *reinterpret_cast<const float2 *>(ub + g0);
                    const float2 u1 = *reinterpret_cast<const float2 *>(ub + g1);
                    return (dc - (u0.y / d0) * u0.x) - (u1.y / d1) * u1.x;
                };
                const float d = reinterpret_cast<const float2 *>(dxb + po)->x;
                const float da = dprime(ao, w.y >> 16, w.z & 0xFFFFu);
                const float db = dprime(bo, w.z >> 16, w.w);
                const float2 ua = *reinterpret_cast<const float2 *>(ub + ao);
                const float2 ubb = *reinterpret_cast<const float2 *>(ub + bo);
                reinterpret_cast<float2 *>(dxb + po)->x = (d - (ua.y / da) * ua.x) - (ubb.y / db) * ubb.x;
            };
            if (cable) run_list(Lf, fold4, diag_task);
            __syncthreads();
            if (cable && wv == 0) run_list(Ljf, fold4, diag_task);
            __syncthreads();
            // from here on, below the root: sDX[c] = (ratio Uj / D', right-hand side) and
            // sU[c] = (Ui, D'); the per-step diagonal register Ds holds the ratio
#pragma unroll
            for (int j = 0; j < K; j++) {
                const int c = tid + TPB * j;
                if (cable && c < N && posof(j) != 0) {
                    const float Dp = sDX(posof(j)).x;
                    Ds[j] = sU(posof(j)).y / Dp;
                    sU(posof(j)).y = Dp;
                }
            }
            // dummy slot: ratio 1 (times right-hand side 0), D' = 1 for the idle backward task
            if (tid == 0) sU(N) = make_float2(0.0f, 1.0f);
        }
        __syncthreads();
        // open fractions of the gated channels from the present gate values
        for (int i = tid; i < NCT; i += NT) {
            const uint32_t w = sCT[i];
            sFb[i] = channel_fopen(gates, (w >> 11) & 63, sQ + (w >> 17));
        }
        __syncthreads();

        // diagonal and right-hand side of a complex compartment (slot j, cell-local index c)
        auto complex_update = [&](int j, int c, const float *sF, float t, bool init, int64_t s, float &Dn,
                                  float &Vn) {
            const TreeComplex &cx = CX[fl[j] & 0xFFFFu];
            const CompConst k = cx.k;
            float I_ch, G_ch;
            tree_channels(k, cx.tcm, sF, V[j], I_ch, G_ch);
            if (k.chmeta == CHM_EXTERNAL) {
                const float2 e = T.chx_ext[c0 + c];   // channels of this step (ext_channels_kernel)
                I_ch = e.x;
                G_ch = e.y;
            }
            float I_in = pulses_current(T, k, c0 + c, t), G_in = 0.0f;
            if (cx.tcm & TCM_INPUT) {
                const float2 in = sIn[c];
                I_in += in.x;
                G_in += in.y;
            }
            float I_syn = 0.0f, G_syn = 0.0f;
            if constexpr (NET) {
                // synapses of this compartment, with the flags of this step's parity (the
                // trigger buffers alternate as in point_kernel)
                if (cx.tcm & TCM_SYN) {
                    const int64_t g = c0 + c;
                    if (T.syn_ext) {
                        const float2 e = T.syn_ext[g];   // generic synapses of this step (lems_syn_kernel)
                        I_syn = e.x;
                        G_syn = e.y;
                        if (T.inp_ext) {
                            const float2 e2 = T.inp_ext[g];   // LEMS inputs, after the native ones
                            I_in += e2.x;
                            G_in += e2.y;
                        }
                    } else {
                        synapses_step<(FORM & 2) ? 8 : 2>(T, stypes, cx.syn_base, cx.syn_cnt, V[j], init, t, dt,
                                                          (int)((s + 3) & 1), s, I_syn, G_syn);
                    }
                }
            }
            const float I_int = I_ch + I_in + I_syn;
            const float G_int = G_ch + G_in + G_syn;
            const float Dd = 1 * div_c(G_int, cx.rC) + k.invrc;
            Dn = (const_tree && posof(j) != 0) ? Ds[j] : 1 + Dd * dt;
            Vn = init ? V[j] : V[j] + div_c(dt * (I_int + ((V[j] * G_int))), cx.rC);
        };
        // The root's update runs on the first quad of wave 0, a channel a lane (channel c's density
        // and its place in sF on lane c), the currents added in channel order by quad_add2, as on
        // point cells. A root with inputs, synapses or channels from elsewhere keeps the general
        // update on one lane, and so does a simple one (whose terms are constants).
        bool root_quad = false;
        float rk_g = 0.0f, rk_e = 0.0f, rk_A = 0.0f, rk_inv = 0.0f, rk_p0s = 0.0f, rk_p0e = -1.0f, rk_p0a = 0.0f;
        int rk_f = -1;
        double rk_rC = 1.0;
        if (wv == 0 && cable) {
            const uint32_t rf = __builtin_amdgcn_readfirstlane(fl[0]);
            if (rf & TCX_COMPLEX) {
                const TreeComplex &cx = CX[rf & 0xFFFFu];
                root_quad = !(cx.tcm & (TCM_INPUT | TCM_SYN | TCM_XCH)) && !(cx.k.gmeta & GM_MORE_PULSES);
                const int nch = cx.tcm & 7;
                const uint32_t mask = (cx.tcm >> 3) & 15;
                int idx = cx.tcm >> 16;
#pragma unroll
                for (int c = 0; c < NCH; c++) {
                    const bool gated = (mask >> c) & 1;
                    if (lane == c && c < nch) {
                        rk_g = cx.k.g[c];
                        rk_e = cx.k.e[c];
                        rk_f = gated ? idx : -1;
                    }
                    idx += gated ? 1 : 0;
                }
                rk_A = cx.k.A;
                rk_inv = cx.k.invrc;
                rk_rC = cx.rC;
                rk_p0s = cx.k.p0s;
                rk_p0e = cx.k.p0e;
                rk_p0a = cx.k.p0a;
            }
        }
        root_quad = __builtin_amdgcn_readfirstlane(root_quad);
        int cur = 0, fcur = 0;
        if (SPLIT && !cable) {
            // channel wave, in a step loop of its own (so that none of the cable group's
            // per-slot registers are live across its gate updates): next open fractions from
            // this step's voltages, overlapping the cable group's step
            for (int64_t s = s0; s < s1; s++) {
                const bool init = s <= 0;
                const float *sV = sVb + cur * (nvmax + 1);
                float *sFn = sFb + (fcur ^ 1) * nctmax;
                // With several cable waves the channel wave takes part in their barriers
                // (the input and compartment barriers first, then, after its own work, the
                // three of the Hines solve), so that every wave passes the same barriers.
                if constexpr (TPB > 64) {
                    if (NIN > 0) lds_barrier<TPB>();
                    lds_barrier<TPB>();
                }
                channel_phase(gates, sCT, sGT, sQ, sFn, sV, NG, NCT, tid - TPB, 64, init, dt, [] { lds_barrier<64>(); });
                if constexpr (TPB > 64) {
                    if (!init) {
                        lds_barrier<TPB>();
                        lds_barrier<TPB>();
                        lds_barrier<TPB>();
                    }
                }
                // the end-of-step barrier of the cable group's loop
                asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
                cur ^= 1;
                fcur ^= 1;
            }
        } else {
            // time_f64 accumulates `time += dt` in double, as the reference's engine loop does
            double time = (s0 >= 1) ? T.t_row[s0 - 1] : 0.0;
            for (int64_t s = s0; s < s1; s++) {
                const bool init = s <= 0;
                const float t = (float)time;
                if (!init) time += (double)dt;
                const int nxt = SPLIT ? cur ^ 1 : cur;
                const float *sV = sVb + cur * (nvmax + 1);
                float *sVn = sVb + nxt * (nvmax + 1);
                // open fractions double-buffered in every mode: the root compartment's update, which
                // reads them, runs after the gate updates may have written the next ones
                const float *sF = sFb + fcur * nctmax;
                float *sFn = sFb + (fcur ^ 1) * nctmax;
                if (cable) {
                    // Poisson inputs of the compartments that have any
                    if (NIN > 0) {
                        for (int i = tid; i < NIN; i += TPB) {
                            const uint32_t e = sIL[i];
                            const int c = e & 0x7FF;
                            float Ii = 0.0f, Gi = 0.0f;
                            const PoiState ps{T.poi_tsince, T.poi_isi, T.poi_A, T.poi_B};
                            poisson_step(T, stypes, c0 + c, sV[c], init, s, dt, Ii, Gi, ps, ps);
                            sIn[c] = make_float2(Ii, Gi);
                        }
                        lds_barrier<TPB>();
                    }
                    // compartments: currents from the present open fractions, semi-implicit RHS.
                    // Slots without a valid lane in this wave are skipped; a wave whose valid
                    // lanes in a slot are all simple compartments takes the short form of the
                    // same operations (the constant conductance and diagonal computed above).
    #pragma unroll
                    for (int j = 0; j < K; j++) {
                        if (!slot_any[j]) continue;
                        const int c = tid + TPB * j;
                        // simple form: channel slot 0, Gbase * 1 (ungated) * (E - V) * 1e-5f * A,
                        // then the empty input and synapse terms, as in the general form below
                        const float I_ch_s = 0.0f + ((((g0[j] * 1.0f) * (e0[j] - V[j])) * 1e-5f) * Ar[j]);
                        const float I_int_s = (I_ch_s + 0.0f) + 0.0f;
                        float Dn = Ds[j];
                        float Vn = init ? V[j] : V[j] + div_c(dt * (I_int_s + ((V[j] * Gs[j]))), rC[j]);
                        if (!slot_simple[j] && c != 0 && (fl[j] & TCX_COMPLEX)) complex_update(j, c, sF, t, init, s, Dn, Vn);
                        sDX(posof(j)) = make_float2(Dn, Vn);
                    }
                    lds_barrier<TPB>();
                    if constexpr (!SPLIT) {
                        // gates on the last cable wave (lanes of that wave, wave-local sync), before
                        // its Hines rounds; the schedule gives that wave a lighter share of the tree.
                        // The open fractions are read again only after the step's last barrier.
                        if (wv == W - 1)
                            channel_phase(gates, sCT, sGT, sQ, sFn, sV, NG, NCT, lane, 64, init, dt, [] { lds_barrier<64>(); });
                    }
                    if (!init) {
                        // forward elimination: fold tasks of at most two children, applied in
                        // ascending child order (the dummy slot N, with right-hand side and Ui 0,
                        // stands in for a missing second child: its terms are exactly zero)
                        // constant tree: below the root sDX[c] = (constant ratio Uj / D', rhs), so
                        // only right-hand sides change; a merged child's right-hand side is folded
                        // again from its children, with the operations of its own task, which
                        // reads the same values and writes that child in the same round
                        auto fold_const = [&](uint4 w) {
                            const uint32_t po = w.x & 0xFFFFu, ao = w.x >> 16, bo = w.y & 0xFFFFu;
                            auto at = [&](uint32_t o) { return *reinterpret_cast<const float2 *>(dxb + o); };
                            // (every read before the first use)
                            const float2 a = at(ao), a0 = at(w.y >> 16), a1 = at(w.z & 0xFFFFu);
                            const float2 b = at(bo), b0 = at(w.z >> 16), b1 = at(w.w);
                            float *xp = reinterpret_cast<float *>(dxb + po) + 1;
                            const float x = *xp;
                            __builtin_amdgcn_sched_barrier(0);
                            const float xa = (a.y - a0.x * a0.y) - a1.x * a1.y;
                            const float xb = (b.y - b0.x * b0.y) - b1.x * b1.y;
                            *xp = (x - a.x * xa) - b.x * xb;
                        };
                        // general tree: diagonal and right-hand side
                        auto fold_task = [&](uint2 w) {
                            const uint32_t po = w.x & 0xFFFFu, ao = w.x >> 16, bo = w.y;
                            float2 *dp = reinterpret_cast<float2 *>(dxb + po);
                            const float2 dx = *dp;
                            const float2 da = *reinterpret_cast<const float2 *>(dxb + ao);
                            const float2 ua = *reinterpret_cast<const float2 *>(ub + ao);
                            const float2 db = *reinterpret_cast<const float2 *>(dxb + bo);
                            const float2 ubb = *reinterpret_cast<const float2 *>(ub + bo);
                            const float r0 = ua.y / da.x;
                            const float r1 = ubb.y / db.x;
                            float2 o;
                            o.x = (dx.x - r0 * ua.x) - r1 * ubb.x;
                            o.y = (dx.y - r0 * da.y) - r1 * db.y;
                            *dp = o;
                        };
                        // back-substitution of one non-root node from its solved parent, or from its
                        // solved grandparent through the parent (solved again, the same operations,
                        // when the parent's own task shares the round); mid = dummy slot N for the
                        // first form, whose extra solve is discarded
                        auto bwd_task = [&](uint2 w) {
                            const uint32_t po = w.x & 0xFFFFu, so = w.x >> 16, mo = w.y;
                            // node records: x ratio or diagonal, y rhs, z Ui, w D' (constant tree)
                            const float xs = reinterpret_cast<const float2 *>(dxb + so)->y;
                            const float4 m = *reinterpret_cast<const float4 *>(dxb + mo);
                            const float4 p = *reinterpret_cast<const float4 *>(dxb + po);
                            __builtin_amdgcn_sched_barrier(0);
                            float xm = (m.y - m.z * xs) / (const_tree ? m.w : m.x);
                            xm = mo == dummy_off ? xs : xm;
                            reinterpret_cast<float2 *>(dxb + po)->y = (p.y - p.z * xm) / (const_tree ? p.w : p.x);
                        };
                        if (const_tree)
                            run_list(Lf, fold4, fold_const);
                        else
                            run_list(Lf, fold2, fold_task);
                        // the root compartment's update, left out of the compartment phase: only
                        // the root fold reads the root's diagonal and right-hand side
                        if (root_quad) {
                            const float Vr = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(V[0])));
                            const float f = rk_f >= 0 ? sF[rk_f] : 1.0f;
                            const float Gscaled = rk_g * f;
                            const float iDensity = Gscaled * (rk_e - Vr) * 1e-5f;
                            const float gDensity = (Gscaled) * 1e-5f;
                            float I_ch = 0.0f, G_ch = 0.0f;
                            quad_add2(I_ch, G_ch, iDensity * rk_A, gDensity * rk_A);
                            const float I_in = (rk_p0s <= t && t <= rk_p0e) ? rk_p0a : 0.0f, G_in = 0.0f;
                            const float I_syn = 0.0f, G_syn = 0.0f;
                            const float I_int = I_ch + I_in + I_syn;
                            const float G_int = G_ch + G_in + G_syn;
                            const float Dd = 1 * div_c(G_int, rk_rC) + rk_inv;
                            const float Vn = Vr + div_c(dt * (I_int + ((Vr * G_int))), rk_rC);
                            if (tid == 0) sDX(0) = make_float2(1 + Dd * dt, Vn);
                        } else if (tid == 0 && (fl[0] & TCX_COMPLEX)) {
                            float Dn = Ds[0], Vn = V[0];
                            complex_update(0, 0, sF, t, false, s, Dn, Vn);
                            sDX(0) = make_float2(Dn, Vn);
                        }
                        lds_barrier<TPB>();
                        if (wv == 0) {
                            // the junction is the serial part of the step; without a channel
                            // wave, wave 0 takes it at raised issue priority among the waves of
                            // its SIMD (config 4 about 1.5 % faster; with a channel wave, which
                            // it would hold back, config 2 was slower)
                            if constexpr (!SPLIT) __builtin_amdgcn_s_setprio(3);
                            if (const_tree)
                                run_list(Ljf, fold4, fold_const);
                            else
                                run_list(Ljf, fold2, fold_task);
                            if (lane == 0) {
                                // the root: all its children (positions 1 .. nr) in order, loads
                                // issued four at a time, then its solve
                                const int nr = cell.root_children;
                                float2 r0 = sDX(0);
                                for (int c = 1; c <= nr; c += 4) {
                                    // (the dummy slot past the last child: its terms are zero)
                                    float2 a[4], u[4];
    #pragma unroll
                                    for (int k = 0; k < 4; k++) {
                                        const int p = c + k <= nr ? c + k : N;
                                        a[k] = sDX(p);
                                        u[k] = sU(p);
                                    }
    #pragma unroll
                                    for (int k = 0; k < 4; k++) {
                                        const float r = const_tree ? a[k].x : u[k].y / a[k].x;
                                        r0.x = r0.x - r * u[k].x;
                                        r0.y = r0.y - r * a[k].y;
                                    }
                                }
                                r0.y = r0.y / r0.x;
                                sDX(0) = r0;
                            }
                            run_list(Ljb, bwd2, bwd_task);
                            if constexpr (!SPLIT) __builtin_amdgcn_s_setprio(0);
                        }
                        lds_barrier<TPB>();
                        run_list(Lb, bwd2, bwd_task);
                        lds_barrier<TPB>();
                    }
                    // new voltages: every slot's read in flight (slots beyond the cell read the
                    // dummy), then spikes and traces where the wave has complex compartments
                    float Vn[K];
    #pragma unroll
                    for (int j = 0; j < K; j++) Vn[j] = init || !slot_any[j] ? V[j] : sDX(posof(j)).y;
    #pragma unroll
                    for (int j = 0; j < K; j++) {
                        const int c = tid + TPB * j;
                        if (slot_cx[j] && (fl[j] & TCX_COMPLEX)) {
                            const TreeComplex &cx = CX[fl[j] & 0xFFFFu];
                            // a recorded compartment is complex: its trace column is in its
                            // record; the trace row of step s holds the voltage the step
                            // started from
                            if (!init && cx.k.rec >= 0) trace_at(T, cx.k.rec, s - 1 - row0) = V[j];
                            const float vthr = cx.k.vthr;
                            if (V[j] < vthr && vthr < Vn[j]) {
                                log_event(T, cx.k.ev, s);
                                if constexpr (NET) send_spike(T, c0 + c, (int)((s + 3) & 1) ^ 1, (int)(s - s0));
                            }
                        }
                        V[j] = Vn[j];
                        if (slot_any[j] && c < NV) sVn[c] = Vn[j];
                    }
                }
                // the next step reads voltages and open fractions written above by other lanes
                if constexpr (SPLIT) {
                    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
                } else {
                    lds_barrier<TPB>();
                }
                cur = nxt;
                fcur ^= 1;
            }
        }
        if (cable) {
#pragma unroll
            for (int j = 0; j < K; j++) {
                const int c = tid + TPB * j;
                if (c < N) T.V[c0 + c] = V[j];
            }
        }
        for (int i = tid; i < NG; i += NT) gq_g[gq0 + i] = sQ[i];
    }
    // the last workgroup out resets the queue for the next launch
    if (tid == 0) {
        __threadfence();
        if (atomicAdd(&queue[1], 1) == (int)gridDim.x - 1) {
            queue[0] = 0;
            queue[1] = 0;
        }
    }
}

// The value at an LDS address. lean_tree_kernel has no LDS but the dynamic one, which starts at
// address 0, so that its task records hold addresses to be used as they are.
typedef float LdsF2 __attribute__((ext_vector_type(2)));
typedef float LdsF4 __attribute__((ext_vector_type(4)));
typedef uint32_t LdsU2 __attribute__((ext_vector_type(2)));
typedef uint32_t LdsU4 __attribute__((ext_vector_type(4)));
template <class V>
__device__ __forceinline__ __attribute__((address_space(3))) V &lds_at(uint32_t a) {
    return *reinterpret_cast<__attribute__((address_space(3))) V *>(a);
}

// Task records of lean_tree_kernel (lean_block). read() issues a round's reads: the values at the
// task's addresses and the record's constants. next() reads another record's addresses in place
// of the task's, whose own node stays in p; value() is the node's new value.
//
// Fold, 48 bytes: two children into a node's right-hand side; a merged child's is formed again
// from its children (tree_kernel, fold_const). Words: the ratios of c0, c1, g00, g01; addresses
// c0, g00, g01, c1; ratios of g10, g11, addresses g10 and (g11 | node << 16).
struct LeanFold {
    static constexpr uint32_t SIZE = 48;
    uint32_t p;
    LdsU4 a;
    LdsU2 b;
    float x, c0, a0, a1, c1, b0, b1;
    LdsF4 r;
    LdsF2 r2;
    __device__ __forceinline__ void next(uint32_t rec) {
        a = lds_at<LdsU4>(rec + 16);
        b = lds_at<LdsU2>(rec + 40);
    }
    __device__ __forceinline__ void read(uint32_t rec) {
        p = b.y >> 16;
        c0 = lds_at<float>(a.x); a0 = lds_at<float>(a.y); a1 = lds_at<float>(a.z);
        c1 = lds_at<float>(a.w); b0 = lds_at<float>(b.x); b1 = lds_at<float>(b.y & 0xFFFFu);
        x = lds_at<float>(p);
        r = lds_at<LdsF4>(rec);
        r2 = lds_at<LdsF2>(rec + 32);
    }
    __device__ __forceinline__ float value() const {
        const float xa = (c0 - r.z * a0) - r.w * a1;
        const float xb = (c1 - r2.x * b0) - r2.y * b1;
        return (x - r.x * xa) - r.y * xb;
    }
};
// Backward, 32 bytes: a node from its solved parent, or from its solved grandparent through its
// parent mid. Words: 1 / D' of mid, Ui of the node, of mid; 1 / D' of the node, addresses of the
// solved one and (mid | node << 16). Without mid that is the dummy, with 1 / D' = 1 and Ui = -1,
// which hands the solved voltage on.
struct LeanBwd {
    static constexpr uint32_t SIZE = 32;
    uint32_t p;
    LdsU2 a, rp;
    LdsU4 c;
    float x, xs, m;
    __device__ __forceinline__ void next(uint32_t rec) {
        a = lds_at<LdsU2>(rec + 24);
    }
    __device__ __forceinline__ void read(uint32_t rec) {
        p = a.y >> 16;
        xs = lds_at<float>(a.x); m = lds_at<float>(a.y & 0xFFFFu); x = lds_at<float>(p);
        c = lds_at<LdsU4>(rec);
        rp = lds_at<LdsU2>(rec + 16);
    }
    __device__ __forceinline__ float value() const {
        const float xm = div_c(m - __uint_as_float(c.w) * xs, __hiloint2double((int)c.y, (int)c.x));
        return div_c(x - __uint_as_float(c.z) * xm, __hiloint2double((int)rp.y, (int)rp.x));
    }
};

// Cells of passive dendrites on an active soma (TreeCell::lean), as tree_kernel runs them but with
// nothing general in the step loop, which is bound by the latency of the Hines rounds: a round is
// one dependent trip through LDS and a short chain of operations.
//   - Every non-root compartment's diagonal is constant, so what a round needs of it (ratios,
//     reciprocals of eliminated diagonals, Ui) is formed on the host and lies in the round's task
//     records (lean_block); of a node only its right-hand side, 4 bytes, is gathered. The
//     back-substitution multiplies by the double reciprocal (div_c) where it divided.
//   - A round first issues its gathers and the reads of its constants, behind them those of the
//     next round's addresses, and makes the address of the record after that while they are on
//     their way. Lanes beyond its tasks repeat the last one (the same value to the same place),
//     so there is no execution mask to set.
//   - The root's update, its gates, its trace and its spikes belong to the gate wave: the extra
//     wave with SPLIT, else the last cable wave. It updates the root, down to the reciprocal of
//     its eliminated diagonal, beside wave 0's forward rounds (the longest lists), and moves the
//     gates beside the backward ones, both on its first quad (QuadChannels).
// With the reading of their rows, 2,005 steps of 512 trees of up to 400 compartments 11.4 -> 5.6 ms
// (tree_kernel, this one), 1,004 of 7 of up to 300 3.6 -> 2.0 ms; a forward round takes about 270
// cycles, a backward one 210 (430 and 385).
template <int TPB, bool SPLIT>
__global__ void __launch_bounds__(TPB + (SPLIT ? 64 : 0)) __attribute__((amdgpu_waves_per_eu(3)))
lean_tree_kernel(DevTables T, const DGate *__restrict__ gates_g, const TreeCell *__restrict__ cells,
                 int32_t n_tasks, int32_t *__restrict__ queue, const uint32_t *__restrict__ blocks_g,
                 const int32_t *__restrict__ pos_g, float *__restrict__ gq_g, int64_t s0, int64_t s1, int64_t row0,
                 float dt) {
    constexpr int K = TREE_SLOTS, W = TPB / 64, NT = TPB + (SPLIT ? 64 : 0);
    // the cell's number, its root's voltage at the start of the step, right-hand side and the
    // reciprocal of its eliminated diagonal, then (LEAN_X) the right-hand sides by position: the
    // dummy at N is -0, which folds with ratio -1 leave as it is, N + 1 takes what nobody reads
    constexpr uint32_t AT_TASK = 0, AT_V = 4, AT_R = 8, AT_RHS = 16;
    const int tid = threadIdx.x, wv = tid >> 6, lane = tid & 63;
    const bool cable = !SPLIT || tid < TPB;
    const bool gate_wave = SPLIT ? !cable : wv == W - 1;
    auto X = [](uint32_t o) -> auto & { return lds_at<float>(o); };
    for (;;) {
        __syncthreads();
        if (tid == 0) lds_at<int32_t>(AT_TASK) = atomicAdd(&queue[0], 1);
        __syncthreads();
        const int32_t task = lds_at<int32_t>(AT_TASK);
        if (task >= n_tasks) break;
        const TreeCell cell = cells[task];
        const int32_t N = cell.n;
        const int64_t c0 = cell.comp_begin, gq0 = cell.gate_off;
        const uint32_t blk = LEAN_X + 4u * (uint32_t)lean_nodes(N);
        const uint4 *const bg = reinterpret_cast<const uint4 *>(blocks_g + cell.lean_off);
        for (int i = tid; i < cell.lean_len / 4; i += NT) {
            const uint4 w = bg[i];
            lds_at<LdsU4>(blk + 16u * (uint32_t)i) = LdsU4{w.x, w.y, w.z, w.w};
        }
        if (tid == 0) {
            X(LEAN_X + 4 * N) = -0.0f;
            lds_at<float>(AT_V) = T.V[c0];
        }
        // cable slots: voltage, channel, area, conductance sum, 1 / C and position, as in
        // tree_kernel; the root's and those beyond the cell write to N + 1
        float V[K], g0[K], e0[K], Ar[K], Gs[K];
        double rC[K];
        uint32_t po[K];
        const int slots = (N - (tid & ~63) + TPB - 1) / TPB;     // of the wave
#pragma unroll
        for (int j = 0; j < K; j++) {
            const int c = tid + TPB * j;
            V[j] = 0.0f; g0[j] = 0.0f; e0[j] = 0.0f; Ar[j] = 0.0f; Gs[j] = 0.0f; rC[j] = 1.0;
            po[j] = LEAN_X + 4u * (uint32_t)N + 4u;
            if (cable && c < N && c > 0) {
                const int64_t g = c0 + c;
                po[j] = LEAN_X + 4u * (uint32_t)pos_g[g];
                V[j] = T.V[g];
                g0[j] = T.chg[g * NCH];
                e0[j] = T.che[g * NCH];
                Ar[j] = T.A[g];
                rC[j] = 1.0 / (double)T.C[g];
                const float G_ch = 0.0f + (((g0[j] * 1.0f) * 1e-5f) * Ar[j]);
                Gs[j] = (G_ch + 0.0f) + 0.0f;
            }
        }
        // gate wave: the root's constants and gate variable lane & 3
        QuadChannels ch;
        CompConst k;
        float qv = 0.0f;
        double root_rC = 1.0;
        const int qs = lane & 3;
        if (gate_wave) {
            load_comp_const(T, c0, k);
            ch.load(gates_g, k, qs);
            root_rC = 1.0 / (double)k.C;
            if (qs < cell.n_gate) qv = gq_g[gq0 + qs];
        }
        __syncthreads();
        // a list: its rounds' headers (two words: the address of the first record, tasks - 1), a
        // lane each for the first 64, the last one repeated
        struct List {
            int first, cnt;
            LdsU2 h;
        };
        auto dir = [&](int i) { return (uint32_t)__builtin_amdgcn_readfirstlane(lds_at<uint32_t>(blk + 4u * (uint32_t)i)); };
        auto headers = [&](const List &L, int r) {
            const uint32_t at = blk + 8u * (uint32_t)(L.first + min(r + lane, L.cnt - 1));
            return (LdsU2)lds_at<LdsU2>(at);
        };
        auto load_list = [&](int i) {
            List L;
            const uint32_t e = dir(i);
            L.first = e & 0xFFFFu;
            L.cnt = e >> 16;
            L.h = LdsU2{0u, 0u};
            if (L.cnt > 0) L.h = headers(L, 0);
            return L;
        };
        const int lw = cable ? wv : 0;
        const List Lf = load_list(2 * lw), Lb = load_list(2 * lw + 1);
        const List Ljf = load_list(2 * W), Ljb = load_list(2 * W + 1);
        // the root's first 64 children (positions 1 .. nr), a lane each: ratio * Ui and ratio,
        // both 0 beyond them
        const int nr = cell.root_children;
        const uint32_t kids = blk + 4u * dir(2 * W + 2);
        auto kid_at = [&](int i) { return (LdsF2)lds_at<LdsF2>(kids + 8u * (uint32_t)i); };
        LdsF2 kid = {0.0f, 0.0f};
        if (lane < nr) kid = kid_at(lane);
        const uint32_t kid_x = LEAN_X + 4u * (uint32_t)(lane < nr ? 1 + lane : N);
        // a - v[0] - v[1] ... over the lanes' values, in order
        auto minus_lanes = [](float a, float v, int n) {
            for (int i = 0; i < n; i += 4) {
#pragma unroll
                for (int j = 0; j < 4; j++)
                    a = a - __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), i + j));
            }
            return a;
        };
        // the record of a lane's task in the round with header r of h
        auto record = [&](LdsU2 h, int r, uint32_t size) -> uint32_t {
            const uint32_t n = (uint32_t)__builtin_amdgcn_readlane(h.y, r);
            return (uint32_t)__builtin_amdgcn_readlane(h.x, r) + __umul24(min((uint32_t)lane, n), size);
        };
        // a list about to run: its first round's record and addresses
        auto begin = [&](const List &L, auto &t, uint32_t &rec) {
            if (L.cnt == 0) return;
            rec = record(L.h, 0, t.SIZE);
            t.next(rec);
        };
        // Round after round with no barrier, as in tree_kernel
        auto run_list = [&](const List &L, auto t, uint32_t rec) {
            LdsU2 h = L.h;
            for (int r0 = 0; r0 < L.cnt; r0 += 63) {
                if (r0 > 0) h = headers(L, r0);
                const int n = __builtin_amdgcn_readfirstlane(min(63, L.cnt - r0));
                for (int r = 1; r <= n; r++) {
                    t.read(rec);
                    rec = record(h, r, t.SIZE);
                    __builtin_amdgcn_sched_barrier(0);
                    t.next(rec);
                    __builtin_amdgcn_sched_barrier(0);
                    X(t.p) = t.value();
                }
            }
        };
        auto barrier_all = [] {
            if constexpr (NT > 64)
                asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            else
                lds_barrier<64>();
        };
        float Vr = 0.0f;           // the root's voltage (gate wave)
        double time = (s0 >= 1) ? T.t_row[s0 - 1] : 0.0;
        for (int64_t s = s0; s < s1; s++) {
            const bool init = s <= 0;
            const float t = (float)time;
            if (!init) time += (double)dt;
            if (gate_wave) {
                // the spike of the step before, this step's trace row
                const float Vp = Vr;
                Vr = lds_at<float>(AT_V);
                if (s > s0 && Vp < k.vthr && k.vthr < Vr && lane == 0) log_event(T, k.ev, s - 1);
                if (!init && k.rec >= 0 && lane == 0) trace_at(T, k.rec, s - 1 - row0) = Vr;
            }
            if (!init) {
                LeanFold tf{};
                LeanBwd tb{};
                uint32_t rf = 0, rb = 0;     // their records
                if (cable) {
#pragma unroll
                    for (int j = 0; j < K; j++) {
                        if (j >= 2 && j >= slots) continue;
                        const float I_ch = 0.0f + ((((g0[j] * 1.0f) * (e0[j] - V[j])) * 1e-5f) * Ar[j]);
                        const float I_int = (I_ch + 0.0f) + 0.0f;
                        X(po[j]) = V[j] + div_c(dt * (I_int + ((V[j] * Gs[j]))), rC[j]);
                    }
                    begin(Lf, tf, rf);
                }
                if constexpr (TPB > 64) barrier_all();
                else lds_barrier<64>();
                if (gate_wave) {
                    float I_ch, G_ch;
                    ch.currents(qv, Vr, I_ch, G_ch);
                    const float I_in = pulses_current(T, k, c0, t), G_in = 0.0f;
                    const float I_syn = 0.0f, G_syn = 0.0f;
                    const float I_int = I_ch + I_in + I_syn;
                    const float G_int = G_ch + G_in + G_syn;
                    const float Dd = 1 * div_c(G_int, root_rC) + k.invrc;
                    const float x = Vr + div_c(dt * (I_int + ((Vr * G_int))), root_rC);
                    float D = minus_lanes(1 + Dd * dt, kid.x, min(nr, 64));
                    for (int b = 64; b < nr; b += 64)
                        D = minus_lanes(D, b + lane < nr ? kid_at(b + lane).x : 0.0f,
                                        min(nr - b, 64));
                    double r = recip64(D);
                    const float ad = fabsf(D);
                    if (__builtin_expect(!((ad >= 0x1p-60f) & (ad <= 0x1p60f)), 0)) r = 1.0 / (double)D;
                    if (lane == 0) {
                        lds_at<float>(AT_RHS) = x;
                        lds_at<double>(AT_R) = r;
                    }
                }
                if (cable) {
                    run_list(Lf, tf, rf);
                    begin(Lb, tb, rb);
                }
                barrier_all();      // forward lists and the root's update done
                if (wv == 0) {
                    if (Ljf.cnt > 0) {
                        begin(Ljf, tf, rf);
                        run_list(Ljf, tf, rf);
                    }
                    float x = minus_lanes(lds_at<float>(AT_RHS), kid.y * X(kid_x), min(nr, 64));
                    for (int b = 64; b < nr; b += 64)
                        x = minus_lanes(x, b + lane < nr ? kid_at(b + lane).y *
                                                               X(LEAN_X + 4u * (uint32_t)(1 + b + lane))
                                                         : 0.0f,
                                        min(nr - b, 64));
                    x = div_c(x, lds_at<double>(AT_R));
                    if (lane == 0) {
                        X(LEAN_X) = x;
                        lds_at<float>(AT_V) = x;
                    }
                    lds_barrier<64>();
                    if (Ljb.cnt > 0) {
                        LeanBwd tj{};
                        begin(Ljb, tj, rf);
                        run_list(Ljb, tj, rf);
                    }
                }
                if constexpr (TPB > 64) barrier_all();
                if (cable) run_list(Lb, tb, rb);
            }
            if (gate_wave) qv = ch.next(qv, Vr, init, dt);
            if constexpr (TPB > 64)
                if (!init) barrier_all();       // every node solved
            if (cable && !init) {
#pragma unroll
                for (int j = 0; j < K; j++) V[j] = X(po[j]);
            }
            // (the next step starts with a lane's own right-hand sides; the root's voltage was
            // written before the junction's barrier, or, with one cable wave, by this one)
            if constexpr (TPB == 64 && SPLIT) barrier_all();
        }
        if (gate_wave) {
            const float Vn = lds_at<float>(AT_V);
            if (Vr < k.vthr && k.vthr < Vn && lane == 0) log_event(T, k.ev, s1 - 1);
            if (lane == 0) T.V[c0] = Vn;
            if (lane < cell.n_gate) gq_g[gq0 + lane] = qv;
        }
        if (cable) {
#pragma unroll
            for (int j = 0; j < K; j++) {
                const int c = tid + TPB * j;
                if (c < N && c > 0) T.V[c0 + c] = V[j];
            }
        }
    }
    // the last workgroup out resets the queue for the next launch
    if (tid == 0) {
        __threadfence();
        if (atomicAdd(&queue[1], 1) == (int)gridDim.x - 1) {
            queue[0] = 0;
            queue[1] = 0;
        }
    }
}

// (a cell of up to 512 compartments leaves room for the gate table at any channel count)
template <bool SPLIT, bool NET>
static const void *tree_kernel_of(int form) {
    switch (form) {
    case 64: return reinterpret_cast<const void *>(&tree_kernel<64, SPLIT, NET>);
    case 128: return reinterpret_cast<const void *>(&tree_kernel<128, SPLIT, NET>);
    case 256: return reinterpret_cast<const void *>(&tree_kernel<256, SPLIT, NET>);
    case 512: return reinterpret_cast<const void *>(&tree_kernel<512, SPLIT, NET>);
    case 257: return reinterpret_cast<const void *>(&tree_kernel<257, SPLIT, NET>);
    case 513: return reinterpret_cast<const void *>(&tree_kernel<513, SPLIT, NET>);
    }
    if constexpr (NET) {
        switch (form) {
        case 70: return reinterpret_cast<const void *>(&tree_kernel<70, SPLIT, NET>);
        case 66: return reinterpret_cast<const void *>(&tree_kernel<66, SPLIT, NET>);
        case 130: return reinterpret_cast<const void *>(&tree_kernel<130, SPLIT, NET>);
        case 258: return reinterpret_cast<const void *>(&tree_kernel<258, SPLIT, NET>);
        case 514: return reinterpret_cast<const void *>(&tree_kernel<514, SPLIT, NET>);
        case 259: return reinterpret_cast<const void *>(&tree_kernel<259, SPLIT, NET>);
        case 515: return reinterpret_cast<const void *>(&tree_kernel<515, SPLIT, NET>);
        }
    }
    return nullptr;
}

template <bool SPLIT>
static const void *lean_kernel_of(int tpb) {
    switch (tpb) {
    case 64: return reinterpret_cast<const void *>(&lean_tree_kernel<64, SPLIT>);
    case 128: return reinterpret_cast<const void *>(&lean_tree_kernel<128, SPLIT>);
    case 256: return reinterpret_cast<const void *>(&lean_tree_kernel<256, SPLIT>);
    case 512: return reinterpret_cast<const void *>(&lean_tree_kernel<512, SPLIT>);
    default: return nullptr;
    }
}

const void *tree_kernel_ptr(int form, bool split, bool net) {
    if (net) return split ? nullptr : tree_kernel_of<false, true>(form);
    return split ? tree_kernel_of<true, false>(form) : tree_kernel_of<false, false>(form);
}

const void *lean_tree_kernel_ptr(int tpb, bool split) {
    return split ? lean_kernel_of<true>(tpb) : lean_kernel_of<false>(tpb);
}

// Channels of compartments beyond the compartment kernels' slots (more than NCH channel
// distributions or NQ gate variables), one lane per compartment, before the step's
// compartment kernels: each channel in distribution order takes its open fraction from its
// gates' present values (each gate `instances` times, conductance_scaling = 1), the gates move
// to their next values, and the channel's current and conductance join the totals
// (eden/Eden.cpp:5679-5898), as channels_step does for the others.
__global__ void __launch_bounds__(64) ext_channels_kernel(DevTables T, const DGate *__restrict__ gates, ExtChanArgs X,
                                                          int64_t step, float dt) {
    ext_channels(T, gates, X, step, dt);
}

const void *ext_channels_kernel_ptr() { return reinterpret_cast<const void *>(&ext_channels_kernel); }
const void *point_kernel_ptr() { return reinterpret_cast<const void *>(&point_kernel); }
const void *point_quad_kernel_ptr() { return reinterpret_cast<const void *>(&point_quad_kernel); }

}  // namespace edenhip
