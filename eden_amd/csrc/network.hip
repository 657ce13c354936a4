// network.hip -- windowed time loop for networks of one-compartment cells.
//
// The reference advances every synapse every step and carries spikes to the next step
// through trigger flags (eden/Eden.cpp:3636-3740, 3946-3995): a spike at step n sets the
// target's trigger, read at step n + 1, where the single-slot NextSpike rule either keeps a
// pending arrival or replaces it with t + delay; the synapse receives its event at the step
// whose window [t, t + dt) holds NextSpike. With every delay at least D steps, a spike
// cannot reach any cell within D - 1 steps, so cells can be advanced W < D steps at a time
// without seeing each other:
//
//   net_window_kernel   W steps of every cell (one lane per cell, synapses in the
//                       block-interleaved slots); a synapse's events come from a device
//                       ring buffer of per-step bit masks instead of its trigger flag,
//                       NextSpike and delay; the spikes of the window are kept as a bit mask
//                       per cell and the spiking cells are compacted into a list (wavefront
//                       ballot + prefix count, one atomic per wave)
//   net_deliver_kernel  for every spiking cell and target synapse, in step order: the
//                       trigger read at step n + 1 and the NextSpike rule with the
//                       reference's float comparisons; the steps whose windows hold the
//                       new NextSpike get the synapse's bit in the ring
//
// One case cannot be decided inside a window: a pending arrival that lies in two
// consecutive step windows (their float bounds overlap by an ulp) and is replaced at the
// first of them, so the reference drops the second delivery. The deliver kernel's check
// pass reports it (and any arrival inside the window just run); the host then runs that
// window again one step at a time, from the state copy the window did not write.
#include <hip/hip_runtime.h>

#include "device_model.hpp"
#include "kernels.hpp"

namespace edenhip {

namespace {

__device__ __forceinline__ void log_event_n(const DevTables &T, int32_t col, int64_t step) {
    if (col >= 0 && step < T.total_rows) {
        uint32_t slot = atomicAdd(T.n_events, 1u);
        if (slot < T.max_events) T.events[slot] = ((int64_t)step << 24) | (int64_t)col;
    }
}

// A cell's chemical synapses for one step: events from the ring words, expTwo dynamics,
// per-type aggregation in list order (eden/Eden.cpp:3636-3740): each type run summed from
// 0, the run sums added in order. State is read from (rA, rB) and written to (wA, wB).
constexpr int NET_CH = 8;

__device__ __forceinline__ void net_synapses(const DevTables &T, const DSynType *stypes, const uint32_t (&runs)[4],
                                             int32_t base, int32_t cnt, const uint32_t *wd, float V, bool init,
                                             float dt, int64_t step, const float *rA, const float *rB, float *wA,
                                             float *wB, uint32_t &n_ev, float &I_syn, float &G_syn) {
    I_syn = 0.0f;
    G_syn = 0.0f;
    int32_t k = 0;
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int32_t e = (int32_t)(runs[r] & 0xFFFFu);
        if (e == 0) break;
        const DSynType st = stypes[runs[r] >> 16];
        float I_agg = 0.0f, G_agg = 0.0f;
        for (; k < e; k += NET_CH) {
            float a[NET_CH], b[NET_CH], w[NET_CH];
#pragma unroll
            for (int u = 0; u < NET_CH; u++) {
                const int32_t s = base + 64 * min(k + u, e - 1);
                a[u] = rA[s];
                b[u] = rB[s];
                w[u] = T.syn_weight[s];
            }
#pragma unroll
            for (int u = 0; u < NET_CH; u++) {
                if (k + u >= e) break;
                const int32_t kk = k + u;
                const int32_t s = base + 64 * kk;
                const bool ev = !init && ((wd[kk >> 5] >> (kk & 31)) & 1u);
                if (ev) {
                    n_ev++;
                    if (T.log_syn) {
                        const uint32_t slot = atomicAdd(T.n_syn_events, 1u);
                        if (slot < T.max_syn_events) T.syn_events[slot] = (step << 32) | (int64_t)T.syn_orig[s];
                    }
                }
                float A = a[u], B = b[u], i, g;
                exptwo_step(st, V, A, B, init, ev, dt, i, g);
                wA[s] = A;
                wB[s] = B;
                I_agg += i * w[u];
                G_agg += g * w[u];
            }
        }
        I_syn += I_agg;
        G_syn += G_agg;
        k = e;   // the chunked loop may have stepped past the run's end
    }
    (void)cnt;
}

}  // namespace

__global__ void __launch_bounds__(64)
net_window_kernel(DevTables T, NetTables Nt, const DGate *__restrict__ gates_g, int n_gates,
                  const DSynType *__restrict__ stypes_g, int n_stypes, const int32_t *__restrict__ comps, int32_t n,
                  int64_t s0, int64_t s1, int64_t row0, float dt, int cur) {
    extern __shared__ __align__(16) unsigned char net_smem[];
    DGate *gates = reinterpret_cast<DGate *>(net_smem);   // [n_gates], dynamic LDS
    __shared__ DSynType stypes[64];
    const int lane = threadIdx.x;
    for (int i = lane; i < n_gates; i += 64) gates[i] = gates_g[i];
    for (int i = lane; i < n_stypes; i += 64) stypes[i] = stypes_g[i];
    __syncthreads();
    const int nxt = cur ^ 1;
    const int32_t idx = blockIdx.x * 64 + lane;
    const bool valid = idx < n;
    uint64_t mask = 0;
    int64_t g = 0;
    if (valid) {
        g = comps[idx];
        CompConst k;
        load_comp_const(T, g, k);
        float V = Nt.V[cur][g];
        float q[NQ];
#pragma unroll
        for (int s = 0; s < NQ; s++) q[s] = Nt.q[cur][g * NQ + s];
        const int32_t syn_base = T.syn_base[g], syn_cnt = T.syn_cnt[g];
        uint32_t runs[4];
#pragma unroll
        for (int r = 0; r < 4; r++) runs[r] = Nt.runs[g * 4 + r];
        const int nwc = (syn_cnt + 31) >> 5;
        const int64_t rbase = ((int64_t)blockIdx.x * Nt.nw) * 64 + lane;
        const bool has_poi = T.poi_begin[g + 1] > T.poi_begin[g];
        uint32_t n_ev = 0;
        double time = (s0 >= 1) ? T.t_row[s0 - 1] : 0.0;
        for (int64_t s = s0; s < s1; s++) {
            const bool init = s <= 0;
            const float t = (float)time;
            const int rb = s == s0 ? cur : nxt;
            if (!init && k.rec >= 0) trace_at(T, k.rec, s - 1 - row0) = V;
            float I_ch, G_ch;
            channels_step(gates, k, V, q, init, dt, I_ch, G_ch);
            float I_syn = 0.0f, G_syn = 0.0f;
            if (syn_cnt > 0) {
                uint32_t wd[8] = {0u, 0u, 0u, 0u, 0u, 0u, 0u, 0u};
                if (!init) {
                    const uint32_t *rw = Nt.ring + (s & Nt.ring_mask) * Nt.ring_stride + rbase;
#pragma unroll
                    for (int w = 0; w < 8; w++)
                        if (w < nwc) wd[w] = rw[w * 64];
                }
                net_synapses(T, stypes, runs, syn_base, syn_cnt, wd, V, init, dt, s, Nt.gA[rb], Nt.gB[rb],
                             Nt.gA[nxt], Nt.gB[nxt], n_ev, I_syn, G_syn);
            }
            float I_in = pulses_current(T, k, g, t), G_in = 0.0f;
            if (has_poi) {
                const PoiState rd{Nt.poi_tsince[rb], Nt.poi_isi[rb], Nt.poi_A[rb], Nt.poi_B[rb]};
                const PoiState wr{Nt.poi_tsince[nxt], Nt.poi_isi[nxt], Nt.poi_A[nxt], Nt.poi_B[nxt]};
                poisson_step(T, stypes, g, V, init, s, dt, I_in, G_in, rd, wr);
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
                if (s - s0 < 64) mask |= 1ull << (s - s0);
                log_event_n(T, k.ev, s);
            }
            V = Vn;
            if (!init) time += (double)dt;
        }
        Nt.V[nxt][g] = V;
#pragma unroll
        for (int s = 0; s < NQ; s++) Nt.q[nxt][g * NQ + s] = q[s];
        if (n_ev) atomicAdd(Nt.n_deliv, (unsigned long long)n_ev);
        if (mask) Nt.spike_mask[g] = mask;
    }
    // spiking cells of this wave: ballot, prefix count, one atomic
    const bool spk = valid && mask != 0ull;
    const uint64_t bal = __ballot(spk);
    if (bal) {
        const int first = __ffsll((long long)bal) - 1;
        uint32_t base = 0;
        if (lane == first) base = atomicAdd(Nt.spk_count, (uint32_t)__popcll(bal));
        base = __shfl(base, first);
        const uint32_t below = __builtin_amdgcn_mbcnt_hi((uint32_t)(bal >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)bal, 0u));
        if (spk) Nt.spk_list[base + below] = (int32_t)g;
    }
}

// One wave's LDS accesses are performed in order; only the compiler must not reorder them.
__device__ __forceinline__ void wave_lds_order() {
    __builtin_amdgcn_wave_barrier();
    asm volatile("" ::: "memory");
}

// net_window_kernel with four lanes per cell and the synapses in registers for the whole window:
// lane l of a cell's quad holds every fourth synapse (its weight in LDS) of each type, in slots that
// start at the same place for the wave's 16 cells, so a slot's type is a scalar and absent
// synapses are zeros whose terms leave the sums as they are. Four slots make a group (up to NG
// of them, static register indices; a wave skips the groups beyond its own).
// The sums are in list order: a group's currents and conductances go to LDS by lane and come
// back as the quad's four of a slot, and even lanes add the currents, odd ones the
// conductances, four adds a slot, beside the next group's work. Lane s also forms channel s's
// current and advances gate variable s (QuadChannels), and input s of up to four Poisson
// inputs. A step's events are few: each lane marks its ring words' bits in LDS, in the slot
// mask of the lane that holds the synapse; a group without a mark in the wave takes the
// decay alone.
// Against one lane per cell, which moves 20 bytes a synapse and step through the caches (a
// window of 38 steps, launch to end): 24,000 cells of 100 synapses 1160 -> 225 us, 1,000 cells of 50
// synapses 644 -> 118 us. Bound by instruction issue, about 650 cycles a group and step and
// 3,000 beside the synapses, with one or two waves a SIMD.
template <int NG>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2, 2)))
net_quad_kernel(DevTables T, NetTables Nt, const DGate *__restrict__ gates_g, NetClasses cls, const NetRare *__restrict__ tables, const int32_t *__restrict__ comps, int32_t n, int64_t s0, int64_t s1, int64_t row0,
                float dt, int cur, int clear) {
    __shared__ NetClass sC[NET_CLASSES];
    __shared__ uint32_t sK[16 * NET_CLASSES];        // a cell's synapses of each class: list range, begin | end << 16
    __shared__ uint32_t sE[2 * 64 + 2];              // the step's events: slot masks by lane, of all lanes
    __shared__ __align__(16) float sP[4 * 2 * 64];   // a group's currents and conductances by slot and lane
    __shared__ float4 sW[NG * 64];                   // weights by group and lane
    const int lane = threadIdx.x, qs = lane & 3;
    const int nxt = cur ^ 1;
    const int32_t at = blockIdx.x * 16 + (lane >> 2);
    const bool valid = at < n;
    const int32_t idx = valid ? at : n - 1;   // spare quads repeat the last cell and store nothing
    const int64_t g = comps[idx];
    CompConst k;
    load_comp_const(T, g, k);
    const double rC = 1.0 / (double)k.C;
    float V = Nt.V[cur][g];
    float qv = Nt.q[cur][g * NQ + qs];
    QuadChannels ch;
    ch.load(gates_g, k, qs);
    // synapses: per class the cell's range of list indices, its groups (their ends, a byte each,
    // the same for the wave), and per group its class and whether it is the class's first
    const int32_t base = T.syn_base[g], cnt = valid ? T.syn_cnt[g] : 0;
    int ng = 0;
    uint32_t gend = 0, gclass = 0, gfirst = 0;
    if (lane < NET_CLASSES) sC[lane] = cls.c[lane];
#pragma unroll
    for (int c = 0; c < NET_CLASSES; c++) {
        uint32_t range = 0;
        if (c < cls.n && cnt > 0) {
            uint32_t b = 0;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const uint32_t run = Nt.runs[g * 4 + r];
                const uint32_t e = run & 0xFFFFu;
                if (e > 0 && (int)(run >> 16) == cls.c[c].type) range = b | (e << 16);
                b = e;
            }
        }
        sK[(lane >> 2) * NET_CLASSES + c] = range;
        int w = ((int)(range >> 16) - (int)(range & 0xFFFFu) + 15) >> 4;
#pragma unroll
        for (int m = 4; m < 64; m <<= 1) w = max(w, __shfl_xor(w, m));
        w = __builtin_amdgcn_readfirstlane(w);
        if (w > 0) gfirst |= 1u << ng;
        for (int i = 0; i < w; i++) gclass |= (uint32_t)c << (2 * (ng + i));
        ng += w;
        gend |= (uint32_t)ng << (8 * c);
    }
    wave_lds_order();
    auto first_group = [&](int c) { return c == 0 ? 0 : (int)(gend >> (8 * c - 8)) & 0xFF; };
    // list index of this lane's synapse in slot u of group i, or -1
    auto syn_at = [&](int i, int u) {
        const int c = (gclass >> (2 * i)) & 3;
        const uint32_t range = sK[(lane >> 2) * NET_CLASSES + c];
        const int kk = (int)(range & 0xFFFFu) + 16 * (i - first_group(c)) + 4 * u + qs;
        return kk < (int)(range >> 16) ? kk : -1;
    };
    float A[NG][4], B[NG][4];
#pragma unroll
    for (int i = 0; i < NG; i++) {
        float w[4];
#pragma unroll
        for (int u = 0; u < 4; u++) A[i][u] = B[i][u] = w[u] = 0.0f;
        if (i < ng) {
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const int kk = syn_at(i, u);
                if (kk >= 0) {
                    const int32_t s = base + 64 * kk;
                    A[i][u] = Nt.gA[cur][s];
                    B[i][u] = Nt.gB[cur][s];
                    w[u] = T.syn_weight[s];
                }
            }
        }
        sW[64 * i + lane] = make_float4(w[0], w[1], w[2], w[3]);
    }
    sE[2 * lane] = sE[2 * lane + 1] = 0u;
    if (lane < 2) sE[128 + lane] = 0u;
    float *const sum_w = sP + lane;
    const float4 *const sum_r = reinterpret_cast<const float4 *>(sP + 64 * (lane & 1) + 4 * (lane >> 2));
    // Poisson input qs of the cell: its state, its weight and its class's place in sC
    const int32_t pb = T.poi_begin[g], np = T.poi_begin[g + 1] - pb;
    const bool poi = qs < np;
    float pt = 0.f, pi = 0.f, pA = 0.f, pB = 0.f, pwt = 0.f;
    int pc = 0;
    if (poi) {
        const int32_t p = pb + qs;
        pt = Nt.poi_tsince[cur][p];
        pi = Nt.poi_isi[cur][p];
        pA = Nt.poi_A[cur][p];
        pB = Nt.poi_B[cur][p];
        pwt = T.poi_weight[p];
        const int ty = T.poi_syn_type[p];
#pragma unroll
        for (int c = 1; c < NET_CLASSES; c++)
            if (c < cls.n && cls.c[c].type == ty) pc = c;
    }
    const bool any_poi = __ballot(poi) != 0ull;
    // ring words qs and qs + 4 of the cell, read a step ahead
    const int nwc = (cnt + 31) >> 5;
    const uint32_t rbase = 4u * ((uint32_t)(idx >> 6) * (uint32_t)Nt.nw * 64u + (uint32_t)(idx & 63));
    auto ring_at = [&](int64_t s, int w) -> uint32_t & {
        char *const row = reinterpret_cast<char *>(Nt.ring + (s & Nt.ring_mask) * Nt.ring_stride);
        return *reinterpret_cast<uint32_t *>(row + (rbase + 256u * (uint32_t)w));
    };
    auto ring_word = [&](int64_t s, int w) { return w < nwc && s >= 1 && s < s1 ? ring_at(s, w) : 0u; };
    uint32_t wd0 = ring_word(s0, qs), wd1 = Nt.nw > 4 ? ring_word(s0, qs + 4) : 0u;
    auto rare = [&]() -> const DevTables & {
        const NetRare *r = tables;
        asm volatile("" : "+s"(r));
        return r->T;
    };
    uint64_t smask = 0;
    uint32_t n_ev = 0;
    double time = (s0 >= 1) ? T.t_row[s0 - 1] : 0.0;
    for (int64_t s = s0; s < s1; s++) {
        const bool init = s <= 0;
        const float t = (float)time;
        // this step's events: each lane takes its words' bits one after the other and marks the
        // synapse in the slot mask of the lane that holds it
        uint64_t evm = 0, ev_any = 0;
        if (__ballot((wd0 | wd1) != 0u)) {
            if (clear) {
                if (wd0) ring_at(s, qs) = 0u;
                if (wd1) ring_at(s, qs + 4) = 0u;
            }
            auto mark = [&](uint32_t word, int first) {
                while (word) {
                    const int kk = first + __ffs((int)word) - 1;
                    word &= word - 1u;
                    int rel = 0, slot = 0;
#pragma unroll
                    for (int c = 0; c < NET_CLASSES; c++) {
                        const uint32_t range = sK[(lane >> 2) * NET_CLASSES + c];
                        if (kk >= (int)(range & 0xFFFFu) && kk < (int)(range >> 16)) {
                            rel = kk - (int)(range & 0xFFFFu);
                            slot = 4 * first_group(c) + (rel >> 2);
                        }
                    }
                    const uint32_t bit = 1u << (slot & 31);
                    const int word_at = slot >> 5;
                    atomicOr(&sE[2 * ((lane & ~3) + (rel & 3)) + word_at], bit);
                    atomicOr(&sE[128 + word_at], bit);
                    n_ev++;
                    const DevTables &R = rare();
                    if (R.log_syn) {
                        const uint32_t at_log = atomicAdd(R.n_syn_events, 1u);
                        if (at_log < R.max_syn_events)
                            R.syn_events[at_log] = (s << 32) | (int64_t)R.syn_orig[base + 64 * kk];
                    }
                }
            };
            mark(wd0, 32 * qs);
            mark(wd1, 32 * qs + 128);
            wave_lds_order();
            evm = (uint64_t)sE[2 * lane] | (uint64_t)sE[2 * lane + 1] << 32;
            ev_any = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)sE[128]) |
                     (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)sE[129]) << 32;
            wave_lds_order();
            sE[2 * lane] = sE[2 * lane + 1] = 0u;
            if (lane < 2) sE[128 + lane] = 0u;
            wave_lds_order();
        }
        // (the trace's store here, a step ahead of the next wait for ring words: loads and stores
        // are waited for with one counter)
        if (!init && k.rec >= 0 && qs == 0 && valid) trace_at(T, k.rec, s - 1 - row0) = V;
        wd0 = ring_word(s + 1, qs);
        if (Nt.nw > 4) wd1 = ring_word(s + 1, qs + 4);
        float I_ch, G_ch;
        ch.currents(qv, V, I_ch, G_ch);
        const float nv = ch.next(qv, V, init, dt);
        // synapses: exptwo_step on each, summed per type in list order, the types in order
        float I_syn = 0.0f, G_syn = 0.0f;
        if (init) {
#pragma unroll
            for (int i = 0; i < NG; i++)
#pragma unroll
                for (int u = 0; u < 4; u++) A[i][u] = B[i][u] = 0.0f;
        } else {
            // (compared afresh each step: kept across steps, one mask a group would spill)
            int ng_s = __builtin_amdgcn_readfirstlane(ng);
            uint32_t first_s = __builtin_amdgcn_readfirstlane(gfirst);
            asm volatile("" : "+s"(ng_s), "+s"(first_s));
            float sum = 0.0f, agg = 0.0f, dv = 0.0f;
            float4 p[4];
#pragma unroll
            for (int u = 0; u < 4; u++) p[u] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            auto add = [&]() {
#pragma unroll
                for (int u = 0; u < 4; u++) agg = (((agg + p[u].x) + p[u].y) + p[u].z) + p[u].w;
            };
            NetClass K = sC[gclass & 3];
#pragma unroll
            for (int i = 0; i < NG; i++) {
                if (i < ng_s) {
                    const float4 w4 = sW[64 * i + lane];
                    const float w[4] = {w4.x, w4.y, w4.z, w4.w};
                    add();               // the group before: zeros before the first
                    if ((first_s >> i) & 1) {
                        sum += agg;      // (the first class: 0 + 0)
                        agg = 0.0f;
                        K = sC[(gclass >> (2 * i)) & 3];
                        dv = K.erev - V;
                    }
#pragma unroll
                    for (int u = 0; u < 4; u++) {
                        const float gs = K.gbase * (B[i][u] - A[i][u]);
                        sum_w[128 * u] = (gs * dv) * w[u];
                        sum_w[128 * u + 64] = gs * w[u];
                    }
                    wave_lds_order();
#pragma unroll
                    for (int u = 0; u < 4; u++) p[u] = sum_r[32 * u];
                    wave_lds_order();
                    float An[4], Bn[4];
#pragma unroll
                    for (int u = 0; u < 4; u++) {
                        An[u] = A[i][u] + dt * div_c2(-A[i][u], K.rise);
                        Bn[u] = B[i][u] + dt * div_c2(-B[i][u], K.decay);
                    }
                    if ((ev_any >> (4 * i)) & 15) {
#pragma unroll
                        for (int u = 0; u < 4; u++)
                            if ((evm >> (4 * i + u)) & 1) {
                                An[u] = A[i][u] + K.jump;
                                Bn[u] = B[i][u] + K.jump;
                            }
                    }
#pragma unroll
                    for (int u = 0; u < 4; u++) {
                        A[i][u] = An[u];
                        B[i][u] = Bn[u];
                    }
                }
            }
            add();
            sum += agg;
            I_syn = quad_bcast<0>(sum);
            G_syn = quad_bcast<1>(sum);
        }
        float I_in = pulses_current(rare(), k, g, t), G_in = 0.0f;
        if (any_poi) {
            float i = 0.0f, gp = 0.0f;
            if (poi) {
                const NetClass K = sC[pc];
                gp = K.gbase * (pB - pA);
                i = gp * (K.erev - V);
                const bool fired = init || pt > pi;
                const float a = pA, b = pB;
                pt = pt + dt * 1.0f;
                pA = a + dt * div_c2(-a, K.rise);
                pB = b + dt * div_c2(-b, K.decay);
                if (fired) {
                    // (addresses formed here, not kept for the window)
                    int32_t p = pb + qs, gc = (int32_t)g;
                    asm volatile("" : "+v"(p), "+v"(gc));
                    const DevTables &R = rare();
                    pt = 0.0f;
                    pi = (-R.poi_isi_mean[p]) * log_f(1.0f - randof(1.0f, (int32_t)R.cell_seed[R.comp_cell[gc]],
                                                                    R.poi_inst[p], s, R.poi_roff[p] + (init ? 0 : 1)));
                    pA = init ? 0.0f : a + K.jump;
                    pB = init ? 0.0f : b + K.jump;
                }
                i = i * pwt;
                gp = gp * pwt;
            }
            float I_agg = 0.0f, G_agg = 0.0f;
            quad_add2(I_agg, G_agg, i, gp);
            I_in = np > 0 ? I_in + I_agg : I_in;
            G_in = np > 0 ? G_in + G_agg : G_in;
        }
        const float I_int = I_ch + I_in + I_syn;
        const float G_int = G_ch + G_in + G_syn;
        const float Vn = init ? V : point_update(V, I_int, G_int, k.invrc, rC, dt);
        if (V < k.vthr && k.vthr < Vn && qs == 0 && valid) {
            if (s - s0 < 64) smask |= 1ull << (s - s0);
            log_event_n(rare(), k.ev, s);
        }
        V = Vn;
        qv = nv;
        if (!init) time += (double)dt;
    }
    if (valid) {
        if (qs == 0) Nt.V[nxt][g] = V;
        Nt.q[nxt][g * NQ + qs] = qv;
        if (poi) {
            const int32_t p = pb + qs;
            Nt.poi_tsince[nxt][p] = pt;
            Nt.poi_isi[nxt][p] = pi;
            Nt.poi_A[nxt][p] = pA;
            Nt.poi_B[nxt][p] = pB;
        }
        if (smask) Nt.spike_mask[g] = smask;
    }
#pragma unroll
    for (int i = 0; i < NG; i++) {
        if (i < ng) {
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const int kk = syn_at(i, u);
                if (kk >= 0) {
                    Nt.gA[nxt][base + 64 * kk] = A[i][u];
                    Nt.gB[nxt][base + 64 * kk] = B[i][u];
                }
            }
        }
    }
    for (int m = 1; m < 64; m <<= 1) n_ev += __shfl_xor(n_ev, m);
    if (lane == 0 && n_ev) atomicAdd(Nt.n_deliv, (unsigned long long)n_ev);
    // spiking cells of this wave: ballot, prefix count, one atomic
    const bool spk = smask != 0ull;
    const uint64_t bal = __ballot(spk);
    if (bal) {
        const int first = __ffsll((long long)bal) - 1;
        uint32_t at_list = 0;
        if (lane == first) at_list = atomicAdd(Nt.spk_count, (uint32_t)__popcll(bal));
        at_list = __shfl(at_list, first);
        const uint32_t below = __builtin_amdgcn_mbcnt_hi((uint32_t)(bal >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)bal, 0u));
        if (spk) Nt.spk_list[at_list + below] = (int32_t)g;
    }
}

namespace {

// steps j >= jmin (and <= last) whose window [t_j, t_j + dt) in float holds x
template <class F>
__device__ __forceinline__ void for_deliveries(const DevTables &T, float x, float dt, int64_t m, float tm, int64_t jmin,
                                               int64_t last, F f) {
    if (!(x > -3.0e38f && x < 3.0e38f)) return;
    const int64_t jc = m + (int64_t)floorf((x - tm) / dt);
    for (int64_t j = jc - 2; j <= jc + 2; j++) {
        if (j < jmin || j < 1 || j > last) continue;
        const float tj = (float)T.t_row[j - 1];
        if (tj <= x && x < tj + dt) f(j);
    }
}

}  // namespace

// flags: 1 commit, 2 the window kernel has cleared the ring words it consumed
__global__ void __launch_bounds__(64)
net_deliver_kernel(DevTables T, NetTables Nt, int64_t s0, int64_t s1, int64_t last, float dt, int flags) {
    const bool commit = (flags & 1) != 0;
    if (commit && blockIdx.x == 0 && threadIdx.x == 0) *Nt.spk_count_next = 0u;
    const int lane = threadIdx.x;
    const uint32_t count = *Nt.spk_count;
    const int64_t ring_stride = Nt.ring_stride;
    for (uint32_t i = blockIdx.x; i < count; i += gridDim.x) {
        const int32_t gc = Nt.spk_list[i];
        const uint64_t M = Nt.spike_mask[gc];
        for (int32_t kt = T.spk_begin[gc] + lane; kt < T.spk_begin[gc + 1]; kt += 64) {
            const int32_t slot = T.spk_target[kt];
            const uint32_t rl = Nt.tgt_rw[kt];
            const int64_t rword = (int64_t)(rl >> 5);
            const uint32_t bit = 1u << (rl & 31u);
            float nn = T.syn_next[slot];
            const float delay = T.syn_delay[slot];
            bool bad = false;
            for (uint64_t mm = M; mm; mm &= mm - 1ull) {
                const int b = __ffsll((long long)mm) - 1;
                const int64_t m = s0 + b + 1;     // the trigger is read one step after the spike
                if (m > last) break;
                const float tm = (float)T.t_row[m - 1];
                const float tpd = tm + dt;
                const float fresh = tm + delay;
                if (nn < tpd && nn < fresh) {
                    // the replaced value's delivery after step m (overlapping windows) is dropped
                    for_deliveries(T, nn, dt, m, tm, m + 1, last, [&](int64_t j) {
                        if (j < s1) bad = true;
                        else if (commit) atomicAnd(&Nt.ring[(j & Nt.ring_mask) * ring_stride + rword], ~bit);
                    });
                    nn = fresh;
                    for_deliveries(T, nn, dt, m, tm, m, last, [&](int64_t j) {
                        if (j < s1) bad = true;
                        else if (commit) atomicOr(&Nt.ring[(j & Nt.ring_mask) * ring_stride + rword], bit);
                    });
                }
            }
            if (commit) T.syn_next[slot] = nn;
            if (bad) atomicOr(Nt.conflict, 1);
        }
    }
    if (commit && !(flags & 2)) {
        // the window's ring slots were consumed: clear them for their next use
        const int64_t a = s0 < 1 ? 1 : s0;
        const int64_t n = (s1 > a ? s1 - a : 0) * ring_stride;
        for (int64_t i = (int64_t)blockIdx.x * 64 + lane; i < n; i += (int64_t)gridDim.x * 64) {
            const int64_t j = a + i / ring_stride;
            Nt.ring[(j & Nt.ring_mask) * ring_stride + (i % ring_stride)] = 0u;
        }
    }
}

const void *net_window_kernel_ptr() { return reinterpret_cast<const void *>(&net_window_kernel); }
const void *net_quad_kernel_ptr(int groups) {
    switch (groups) {
    case 1: return reinterpret_cast<const void *>(&net_quad_kernel<1>);
    case 2: return reinterpret_cast<const void *>(&net_quad_kernel<2>);
    case 4: return reinterpret_cast<const void *>(&net_quad_kernel<4>);
    case 6: return reinterpret_cast<const void *>(&net_quad_kernel<6>);
    case 8: return reinterpret_cast<const void *>(&net_quad_kernel<8>);
    case 10: return reinterpret_cast<const void *>(&net_quad_kernel<10>);
    case 12: return reinterpret_cast<const void *>(&net_quad_kernel<12>);
    case 16: return reinterpret_cast<const void *>(&net_quad_kernel<16>);
    default: return nullptr;
    }
}
const void *net_deliver_kernel_ptr() { return reinterpret_cast<const void *>(&net_deliver_kernel); }

}  // namespace edenhip
