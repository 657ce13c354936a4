// lems_kernel.hip -- synapse kernel template for generic LEMS synapse types, compiled at
// context creation with hiprtc together with the generated functions (edenhip_lems_synapses:
// `lems_syn`, emitted by eden_amd.lems), the counterpart of the reference's per-cell-type C
// emission and gcc step (eden/Eden.cpp:2339-2995, 3561-3740, 6992-7216).
//
// Per step, for each synapse instance of each compartment that has chemical synapses: the
// trigger read and clear and the single-slot delay rule (eden/Eden.cpp:3636-3707, the same code
// as synapses_step), then the instance's LEMS step (lems_syn, given the voltage at the start of
// the step of the instance's peer compartment for gap junctions), its exposures times the
// connection weight aggregated per synapse type, the types' aggregates summed in order
// (eden/Eden.cpp:3721-3735). Every compartment's V is the start-of-step value here: this kernel
// runs before the step's compartment kernels. The totals go to syn_ext, where the compartment
// kernels of the same step read them in place of their own synapse code. State is updated in
// place (the generated code reads an instance's whole present state before writing).
//
// An instance is a chain of dependent loads and divisions, so its latency, not its work, is what
// a step costs: the instances of a compartment (where it has several) go to lanes of their own,
// LEMS_SYN_COMPS compartments side by side (their slots are neighbours: 64-byte accesses) times as many
// instances as the workgroup has room for, and leave their currents in LDS; one lane per
// compartment then sums them in list order. 700 cells with 30 synapses each: 49.9 us a step with
// a lane per compartment, now 9.5 us.
//
// lems_cell_kernel runs LEMS point neurons (the reference's artificial cells,
// eden/Eden.cpp:6603-6910): one lane per cell; per step, the external current (the cell's
// synapse currents from syn_ext, then its pulse inputs), the generated `lems_cell` step, the
// compartment's V set to the membrane-voltage state variable, and a spike sent to the
// recipients and logged as a physical cell's is.
//
// The generated source (`lems_syn` and `lems_cell`) is inserted where
// lems_synapse_functions.h is included. It also defines EDENHIP_LEMS, for the kernels that the
// model runs (compiling them is most of what creating a context costs): 0 neither synapses nor
// point neurons, 1 synapses, 2 point neurons too, 3 both by lems_window_kernel.
#define EDENHIP_LEMS_RATES 1
#include "device_model.hpp"

#define EXP edenhip::exp_f
#define LOG edenhip::log_f
#define POW edenhip::pow_f
#define SIN(x) ((float)sin((double)(x)))
#define COS(x) ((float)cos((double)(x)))
#define TAN(x) ((float)tan((double)(x)))
#define SINH(x) ((float)sinh((double)(x)))
#define COSH(x) ((float)cosh((double)(x)))
#define TANH(x) ((float)tanh((double)(x)))
__device__ __forceinline__ float stepf(float x) { return x < 0.0f ? 0.0f : 1.0f; }
// random(x) of a point neuron's generated step: randof stamped with the cell's RNG seed, the
// step, the call's number and, as the instance, the reference's NOT_AN_INSTANCE marker of
// code outside a table loop (~0xFee1600dLL, eden/Eden.cpp:3255-3256)
__device__ __forceinline__ float lems_randof(float x, int seed, long long step, int n) {
    return edenhip::randof(x, seed, (int64_t)~0xFee1600dLL, (int64_t)step, n);
}

#include "lems_synapse_functions.h"

// One synapse instance's step: its current and conductance times the connection weight. flags:
// this step reads trigger flags (a later step of a launch has none, see trig_fold_kernel).
__device__ __forceinline__ float2 lems_instance(const edenhip::DevTables &T, const edenhip::LemsArgs &L, int32_t g,
                                                int32_t s, int32_t ty, float V, int64_t step, float t, float dt,
                                                bool flags) {
    using namespace edenhip;
    const bool init = step <= 0;
    int32_t *const trig_now = T.trig[(int)((step + 3) & 1)];
    const float weight = T.syn_weight[s];
    bool spike_now = false;
    const int32_t tp = L.tpos ? L.tpos[s] : -1;
    if (tp >= 0) {
        // a firing-synapse input: its spike list's times before the end of the step fire it
        // in the same step (eden/Eden.cpp:3780-3788); the list ends with a sentinel
        // (events of the initial steps are ignored by the generated code, so not raised)
        int32_t pos = tp;
        bool fired = false;
        while (L.ttimes[pos] < t + dt) { fired = true; pos++; }
        if (!init) {
            L.tpos[s] = pos;
            spike_now = fired;
        }
    } else if (L.pspk && L.pspk[s] >= 0) {
        // a Poisson firing-synapse input's spiker (poissonFiringSynapse,
        // transientPoissonFiringSynapse): tsince' = 1; when tsince > isi, tsince = 0, a new
        // interval and a spike, the synapse's event of the same step
        const int32_t k = L.pspk[s];
        const float averageIsi = L.pk_isi[k];
        const int32_t seed = (int32_t)T.cell_seed[T.comp_cell[g]], inst = L.pk_inst[k], roff = L.pk_roff[k];
        const bool transient = L.pk_transient[k] != 0;
        const float2 win = L.pk_window[k];
        const float2 st = L.pk_state[k];
        float tn, in;
        if (init) {
            tn = 0.0f;
            const float nextIsi = (-averageIsi) * log_f(1.0f - randof(1.0f, seed, inst, step, roff + 0));
            in = transient ? nextIsi + win.x : nextIsi;
        } else {
            tn = st.x + dt * 1.0f;
            in = st.y;
            if (st.x > st.y) {
                tn = 0.0f;
                const float nextIsi = (-averageIsi) * log_f(1.0f - randof(1.0f, seed, inst, step, roff + 1));
                // after the window, the next interval is pushed 1e9 hours (3.6e18 us) away
                in = transient ? nextIsi + stepf(((t + nextIsi) - (win.x + win.y)) / win.y) * 3.6e18f : nextIsi;
                spike_now = true;
            }
        }
        L.pk_state[k] = make_float2(tn, in);
    } else {
        bool flag = false;
        if (!init && flags) {
            flag = trig_now[s] != 0;
            if (flag) trig_now[s] = 0;
        }
        const float delay = T.syn_delay[s];
        const float next_spike = T.syn_next[s];
        float nn = next_spike;
        if (!init) {
            if (t <= next_spike && next_spike < t + dt) spike_now = true;
            if (flag) {
                const float fresh = t + delay;
                if (t <= fresh && fresh < t + dt) spike_now = true;
                if (nn < t + dt && nn < fresh) nn = fresh;
            }
        }
        if (nn != next_spike) T.syn_next[s] = nn;
    }
    if (spike_now && T.log_syn) {
        const uint32_t slot = atomicAdd(T.n_syn_events, 1u);
        if (slot < T.max_syn_events) T.syn_events[slot] = (step << 32) | (int64_t)T.syn_orig[s];
    }
    float i, gx;
    float *S = L.state + s;
    const int32_t pc = L.peer[s];
    const float vpeer = pc >= 0 ? T.V[pc] : V;
    const float *P = L.params + (L.poff ? L.poff[s] : L.param_begin[ty]);
    lems_syn(ty, P, S, S, (long)L.stride, V, vpeer, t, init ? 1 : 0, spike_now ? 1 : 0, dt, &i, &gx);
    return make_float2(i * weight, gx * weight);
}

// A workgroup: LEMS_SYN_COMPS compartments with as many lanes each as instances run side by side
// (at most LEMS_SYN_LANES), or, where a compartment has one instance (or many compartments two), a
// wave of 64 compartments (L.wave_comps). Its LDS (lems_syn_lds bytes, dynamic): the compartments' voltages,
// then per lane of a compartment two sets of its instances' values, so that one may be summed
// while the next is filled. 12 KiB for the most lanes there can be would leave only 13 workgroups a
// CU in flight, where large populations have more. 100,000 cells with a synapse each 21.1 -> 14.2 us a
// step (17.5 with a lane a compartment and no LDS), 200,000 with two 40.0 -> 24.5, 50,000 point
// neurons with two 7.0 -> 5.1.
struct LemsLane {
    float2 v[2][edenhip::LEMS_SYN_COMPS];
    int32_t type[2][edenhip::LEMS_SYN_COMPS];
};
extern __shared__ __align__(16) float lems_shared[];
__device__ __forceinline__ LemsLane *lems_lanes() { return reinterpret_cast<LemsLane *>(lems_shared + 64); }

// Totals of a compartment's synapses and LEMS inputs.
struct LemsTotals {
    float I_syn, G_syn, I_inp, G_inp;
};

// The synapses of a workgroup's compartments at a step (every lane calls it; c: the lane's
// compartment, lane: its place among the compartment's lanes). The compartments' first lanes get
// their totals.
__device__ __forceinline__ LemsTotals lems_synapses(const edenhip::DevTables &T, const edenhip::LemsArgs &L,
                                                    int c, int lane, int32_t g, int32_t base, int32_t cnt,
                                                    int32_t most, float V, int64_t step, float t, float dt, bool flags) {
    using namespace edenhip;
    constexpr int INPUT = 1 << 30;
    const int lanes = L.wave_comps ? 1 : blockDim.x / LEMS_SYN_COMPS;
    LemsLane *const sh = lems_lanes();
    LemsTotals r{0.0f, 0.0f, 0.0f, 0.0f};   // I_inp: i * weight per instance (eden/Eden.cpp:3929)
    float I_agg = 0.0f, G_agg = 0.0f;
    int32_t cur = -1;
    auto add = [&](float2 v, int32_t ty) {
        if (ty & INPUT) {
            r.I_inp += v.x;
            r.G_inp += v.y;
            return;
        }
        if (ty != cur) {
            if (cur >= 0) { r.I_syn += I_agg; r.G_syn += G_agg; }
            I_agg = 0.0f; G_agg = 0.0f; cur = ty;
        }
        I_agg += v.x;
        G_agg += v.y;
    };
    for (int32_t k0 = 0, set = 0; k0 < most; k0 += lanes, set ^= 1) {
        if (k0 + lane < cnt) {
            const int32_t s = base + 64 * (k0 + lane), ty = T.syn_type[s];
            const float2 v = lems_instance(T, L, g, s, ty, V, step, t, dt, flags);
            const int32_t kind = ty | (L.flags && (L.flags[ty] & 1) ? INPUT : 0);
            if (lanes == 1) {
                add(v, kind);
            } else {
                sh[lane].v[set][c] = v;
                sh[lane].type[set][c] = kind;
            }
        }
        if (lanes == 1) continue;
        __syncthreads();
        if (lane > 0) continue;
        // (lanes is a multiple of 4)
        const int n = min(cnt - k0, lanes);
        for (int j0 = 0; j0 < n; j0 += 4) {
            float2 v[4];
            int32_t ty[4];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                v[j] = sh[j0 + j].v[set][c];
                ty[j] = sh[j0 + j].type[set][c];
            }
#pragma unroll
            for (int j = 0; j < 4; j++)
                if (j0 + j < n) add(v[j], ty[j]);
        }
    }
    r.I_syn += I_agg;
    r.G_syn += G_agg;
    return r;
}

// The largest value of a workgroup's compartments (a wave holds all of them, or several times).
__device__ __forceinline__ int32_t lems_most(int32_t x) {
    for (int m = 1; m < 64; m <<= 1) x = max(x, __shfl_xor(x, m));
    return x;
}

// Compartments of a workgroup, and a lane's compartment and place there.
struct LemsPlace {
    int comps, c, lane;
    __device__ __forceinline__ explicit LemsPlace(const edenhip::LemsArgs &L) {
        comps = L.wave_comps ? 64 : edenhip::LEMS_SYN_COMPS;
        c = threadIdx.x & (comps - 1);
        lane = L.wave_comps ? 0 : threadIdx.x / edenhip::LEMS_SYN_COMPS;
    }
};

#if EDENHIP_LEMS == 1 || EDENHIP_LEMS == 2
extern "C" __global__ void __launch_bounds__(edenhip::LEMS_SYN_COMPS * edenhip::LEMS_SYN_LANES)
lems_syn_kernel(edenhip::DevTables T, edenhip::LemsArgs L, int64_t step, float dt) {
    using namespace edenhip;
    const LemsPlace at(L);
    const int32_t idx = blockIdx.x * at.comps + at.c;
    const bool have = idx < L.n_comps;
    const int32_t g = have ? L.comps[idx] : 0;
    // time_f32 of the step, from the reference's double accumulation
    const float t = (float)(step >= 1 ? T.t_row[step - 1] : 0.0);
    const int32_t cnt = have ? T.syn_cnt[g] : 0;
    const LemsTotals r = lems_synapses(T, L, at.c, at.lane, g, T.syn_base[g], cnt, lems_most(cnt), T.V[g], step, t, dt, true);
    if (at.lane > 0 || !have) return;
    L.syn_ext[g] = make_float2(r.I_syn, r.G_syn);
    if (L.inp_ext) L.inp_ext[g] = make_float2(r.I_inp, r.G_inp);
}
#endif

#if EDENHIP_LEMS >= 2
// A point neuron's step: synapse and input currents, the generated step, V (returned), its spike.
__device__ __forceinline__ float lems_neuron(const edenhip::DevTables &T, const edenhip::LemsCellArgs &A, int32_t idx,
                                             int32_t g, float V, int64_t step, float t, float dt, float I_syn,
                                             bool has_inp, float I_inp, int at) {
    using namespace edenhip;
    const int32_t ty = A.type[idx];
    const bool init = step <= 0;
    const int nxt = (int)((step + 3) & 1) ^ 1;
    // external current: synapses, then inputs (eden/Eden.cpp:6856-6880)
    float I_in = 0.0f;
    const int32_t pb = T.pulse_begin[g], pe = T.pulse_begin[g + 1];
    if (pe > pb) {
        float Ip = 0.0f;
        for (int32_t p = pb; p < pe; p++)
            if (T.pulse_start[p] <= t && t <= T.pulse_end[p]) Ip += T.pulse_amp[p];
        I_in += Ip;
        I_in += 0.0f;
    }
    if (has_inp) I_in += I_inp;   // LEMS inputs, after the native ones
    const float ext = I_syn + I_in;
    float *S = A.state + idx;
    int spike = 0;
    const float *P = A.params + (A.poff ? A.poff[idx] : A.param_begin[ty]);
    lems_cell(ty, P, S, S, (long)A.n, t, dt, init ? 1 : 0, ext, (int)T.cell_seed[T.comp_cell[g]], (long long)step,
              &spike);
    const int32_t vs = A.v_state[ty];
    if (vs >= 0) {
        V = S[(int64_t)vs * A.n];
        T.V[g] = V;
    }
    if (spike) {
        send_spike(T, g, nxt, at);
        log_event(T, T.ev_col[g], step);
    }
    return V;
}
#endif

#if EDENHIP_LEMS == 2
extern "C" __global__ void __launch_bounds__(64)
lems_cell_kernel(edenhip::DevTables T, edenhip::LemsCellArgs A, int64_t step, float dt) {
    const int32_t idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= A.n) return;
    const int32_t g = A.comps[idx];
    const float t = (float)(step >= 1 ? T.t_row[step - 1] : 0.0);
    const bool has_syn = T.syn_cnt[g] > 0;
    const float I_syn = T.syn_ext && has_syn ? T.syn_ext[g].x : 0.0f;
    const bool has_inp = T.inp_ext && has_syn;
    lems_neuron(T, A, idx, g, 0.0f, step, t, dt, I_syn, has_inp, has_inp ? T.inp_ext[g].x : 0.0f, 0);
}
#endif

#if EDENHIP_LEMS == 3
// Steps [s0, s1) of point neurons with their synapses and recorded state variables, in one launch:
// where only they have generic synapses and none looks at another cell's voltage, nothing passes
// between cells but spikes, whose delays span the window (trig_fold_kernel). Launches of the three
// kernels for every step took 17.3 us a step with 700 cells of 30 synapses, this 6.6.
extern "C" __global__ void __launch_bounds__(edenhip::LEMS_SYN_COMPS * edenhip::LEMS_SYN_LANES)
lems_window_kernel(edenhip::DevTables T, edenhip::LemsArgs L, edenhip::LemsCellArgs A, const int32_t *rec_begin,
                   const int32_t *rec_var, const int32_t *rec_col, int64_t s0, int64_t s1, int64_t row0, float dt) {
    using namespace edenhip;
    const LemsPlace at(L);
    const int c = at.c;
    const int32_t idx = blockIdx.x * at.comps + c;
    const bool have = idx < A.n, cell = have && at.lane == 0;
    float *const sV = lems_shared;
    const int32_t g = have ? A.comps[idx] : 0;
    const int32_t base = T.syn_base[g], cnt = have ? T.syn_cnt[g] : 0, most = lems_most(cnt);
    int32_t rb = 0, re = 0;
    if (cell && rec_begin) { rb = rec_begin[idx]; re = rec_begin[idx + 1]; }
    if (at.lane == 0) sV[c] = T.V[g];
    for (int64_t s = s0; s < s1; s++) {
        __syncthreads();
        const float t = (float)(s >= 1 ? T.t_row[s - 1] : 0.0), V = sV[c];
        // state after the step before, before this one changes it
        if (s >= 1)
            for (int32_t r = rb; r < re; r++) trace_at(T, rec_col[r], s - 1 - row0) = A.state[(int64_t)rec_var[r] * A.n + idx];
        const LemsTotals r = lems_synapses(T, L, c, at.lane, g, base, cnt, most, V, s, t, dt, s == s0);
        if (cell)
            sV[c] = lems_neuron(T, A, idx, g, V, s, t, dt, cnt > 0 ? r.I_syn : 0.0f, T.inp_ext && cnt > 0, r.I_inp,
                                  (int)(s - s0));
    }
}
#endif

// Channels of the compartments run outside the compartment kernels, here with the user rate
// ComponentTypes' generated lems_rate (gates of form RATE_LEMS); the statically compiled
// ext_channels_kernel runs the same code for models without them.
extern "C" __global__ void __launch_bounds__(64)
ext_channels_kernel_rtc(edenhip::DevTables T, const edenhip::DGate *__restrict__ gates, edenhip::ExtChanArgs X,
                        int64_t step, float dt) {
    edenhip::ext_channels(T, gates, X, step, dt);
}
