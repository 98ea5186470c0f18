// qb_introws.hip -- gfx950 kernels of the integer annealer for graphs whose couplings all
// have one magnitude (max-cut and +-J graphs): adjacency rows as 16-bit words (neighbour,
// sign in the top bit), which fit a CU's LDS where 32-bit neighbours and weights do not.
//
//   int_ref_rows_kernel  the reference's own trajectory (wising::anneal,
//                        src/ising_weighted.hpp:250-267), a wave per replica, several
//                        replicas of a workgroup sharing the rows in LDS;
//   int_wide_kernel      the colour-class trajectory (qb_run_batch), a workgroup per
//                        replica, for few replicas;
//   int_sweep_rows_kernel  the same with a wave per replica, for many.
#include <algorithm>

#include "qb_internal.h"
#include "qb_rng.h"

namespace qb {

namespace {

// f[neighbours] -= 2 w s for the rows of the lanes in m (bounds row0, row1 and spin si of each
// lane); the additions are atomic, so rows may share neighbours. Few or long rows go one at a
// time over the whole wave, the next row's entries read before the current one's additions.
// Several short rows (`quarters`) go four at a time: their bounds and signs are moved to
// consecutive lanes and each quarter of the wave takes one, 64 entries in flight, so four
// rows share the LDS latency that one would pay alone (205 sweeps at degree 8: 5.7 -> 4.7 ms;
// at degree 48, where a row fills the wave, 6.1 -> 6.6 ms, so those stay apart).
__device__ __forceinline__ void rows_add(const uint16_t* rows, uint64_t m, int lane, int row0, int row1, int si, int w2,
                                         int32_t* f, bool quarters) {
    const int count = __popcll(m);
    if (!quarters || count < 4) {
        for (; m; m &= m - 1) {
            const int js = __builtin_ctzll(m);
            const int q0 = __builtin_amdgcn_readlane(row0, js), q1 = __builtin_amdgcn_readlane(row1, js);
            const int d = w2 * __builtin_amdgcn_readlane(si, js);
            for (int q = q0 + lane; q < q1; q += 64) {
                const uint32_t e = rows[q];
                atomicAdd(&f[e & 0x7FFFu], (e & 0x8000u) ? d : -d);
            }
        }
        return;
    }
    // a permutation of the wave: the lanes of m first, in order, then the others
    const int rank = __popcll(m & ((uint64_t(1) << lane) - 1u));
    const int to = 4 * (((m >> lane) & 1u) ? rank : count + lane - rank);
    const int pa = __builtin_amdgcn_ds_permute(to, row0 | (si > 0 ? int(0x80000000u) : 0));
    const int pb = __builtin_amdgcn_ds_permute(to, row1);
    for (int k = 0; k < count; k += 4) {
        const int src = k + (lane >> 4);
        const int a = __builtin_amdgcn_ds_bpermute(src * 4, pa), b = __builtin_amdgcn_ds_bpermute(src * 4, pb);
        const int end = src < count ? b : 0;
        const int d = a < 0 ? w2 : -w2;
        for (int q = (a & 0x7FFFFFFF) + (lane & 15); __ballot(q < end) != 0; q += 64) {
            uint32_t e[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) e[u] = rows[min(q + 16 * u, max(end - 1, 0))];
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (q + 16 * u < end) atomicAdd(&f[e[u] & 0x7FFFu], (e[u] & 0x8000u) ? d : -d);
        }
    }
}

// The rows in position order.
__global__ void __launch_bounds__(256) position_rows_kernel(DevGraph g, uint16_t* prows) {
    for (int q = int(blockIdx.x) * 256 + int(threadIdx.x); q < g.m_dir; q += int(gridDim.x) * 256)
        prows[q] = uint16_t(g.nb[q] | (g.nw[q] < 0 ? 0x8000 : 0));
}

// The rows in original bit order, one wave a bit, and each bit's band.
__global__ void __launch_bounds__(256) bit_rows_kernel(DevGraph g, uint16_t* orows, uint64_t* band) {
    const int i = int(blockIdx.x) * 4 + int(threadIdx.x) / 64, lane = int(threadIdx.x) % 64;
    if (i >= g.n) return;   // the whole wave
    const int p = g.bit_pos[i], q0 = g.nb_ptr[p], len = g.nb_ptr[p + 1] - q0;
    uint16_t* row = orows + g.ostart[i];
    uint64_t m = 0;
    for (int k = lane; k < len; k += 64) {
        const int j = g.pos_bit[g.nb[q0 + k]], back = i - j;
        row[k] = uint16_t(j | (g.nw[q0 + k] < 0 ? 0x8000 : 0));
        if (back >= 1 && back <= 64) m |= uint64_t(1) << (64 - back);
    }
    for (int o = 32; o > 0; o >>= 1) m |= uint64_t(__shfl_xor((unsigned long long)m, o));
    if (lane == 0) band[i] = m;
}

}  // namespace

hipError_t launch_position_rows(const DevGraph& g, uint16_t* prows, hipStream_t st) {
    position_rows_kernel<<<unsigned(std::min(2048, (g.m_dir + 255) / 256)), 256, 0, st>>>(g, prows);
    return hipGetLastError();
}

hipError_t launch_bit_rows(const DevGraph& g, uint16_t* orows, uint64_t* band, hipStream_t st) {
    bit_rows_kernel<<<unsigned((g.n + 3) / 4), 256, 0, st>>>(g, orows, band);
    return hipGetLastError();
}

// ---- the reference's own trajectory --------------------------------------------------------
// int_ref_kernel's windows (the next 64 bits evaluated at once, the k-th uphill one drawing
// state + k gamma) on rows and row starts in LDS, in original bit order, so a window's spins,
// fields and starts are consecutive words. A flip of the window changes the decision of a
// later lane only if that lane is its neighbour: g.band[i] holds which of the 64 bits before
// bit i are (bit 63: i - 1), so one comparison with the accepted lanes finds the first lane
// that an accepted flip before it reaches. Everything before that lane is committed together
// -- the flips' rows go out back to back, with no read between them -- and the next window
// starts there. int_ref_kernel commits flip by flip, reading the later lanes' fields back
// after each to find the one it changed: 205 sweeps of an 800-vertex graph of degree 48 from
// T = 9.8 took 12.3 ms a replica there with the rows in L2, 8.9 with them in LDS, and take
// 6.4 here (2,048 replicas at once 14.2 -> 7.7 ms; degree 8, 13.0 -> 4.7 ms). What is left is
// the chain of a window: fields, draws, decisions, the comparison.
template <bool LDS_ROWS>
__global__ void __launch_bounds__(1024) int_ref_rows_kernel(DevGraph g, int R, uint64_t seed_base, const double* temp,
                                                            int sweep_begin, int sweep_end, int init, int8_t* s_state,
                                                            int32_t* f_state, uint64_t* rng, long long* energy) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int n = g.n, np = g.n_pad;
    const int w = int(threadIdx.x) / 64, lane = int(threadIdx.x) % 64, waves = int(blockDim.x) / 64;
    uint64_t* band = reinterpret_cast<uint64_t*>(smem);
    int32_t* start = reinterpret_cast<int32_t*>(band + np);
    int32_t* fields = start + ((n + 4) & ~3);
    uint16_t* lrows = reinterpret_cast<uint16_t*>(fields + size_t(waves) * np);
    int8_t* spins = reinterpret_cast<int8_t*>(lrows + (LDS_ROWS ? (g.m_dir + 7) & ~7 : 0));
    const uint16_t* rows = LDS_ROWS ? lrows : g.orows;
    for (int i = int(threadIdx.x); i < n; i += int(blockDim.x)) band[i] = g.band[i];
    for (int i = int(threadIdx.x); i <= n; i += int(blockDim.x)) start[i] = g.ostart[i];
    for (int i = int(threadIdx.x); LDS_ROWS && i < g.m_dir / 2; i += int(blockDim.x))   // m_dir is even
        reinterpret_cast<uint32_t*>(lrows)[i] = reinterpret_cast<const uint32_t*>(g.orows)[i];
    __syncthreads();
    const int r = int(blockIdx.x) * waves + w;
    if (r >= R) return;   // the whole wave leaves; the rest never syncs across waves
    int32_t* f = fields + size_t(w) * np;
    int8_t* s = spins + size_t(w) * np;
    int8_t* gs = s_state + size_t(r) * size_t(np);
    int32_t* gf = f_state + size_t(r) * size_t(np);
    uint64_t st;
    long long e = 0;   // this lane's part of the energy change
    for (int i = lane; i < n; i += 64) {
        const int p = g.bit_pos[i];
        s[i] = init ? int8_t(-1) : gs[p];
        f[i] = init ? g.f0[p] : gf[p];
    }
    st = init ? (seed_base + uint64_t(r)) * 0x2545F4914F6CDD1Dull + 1 : rng[r];
    auto sync = [] {
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    sync();
    const uint64_t below = (uint64_t(1) << lane) - 1u;
    const int w2 = 2 * g.w0;
    const bool quarters = g.m_dir <= 32 * n;
    for (int sweep = sweep_begin; sweep < sweep_end; ++sweep) {
        const double T = temp[sweep];
        const double nrT = -1.0 / T;
        int i0 = 0;
        while (i0 < n) {
            const int i = i0 + lane;
            const bool valid = i < n;
            const int at = valid ? i : 0;
            const int si = s[at];
            const int32_t fi = f[at];
            const int row0 = start[at], row1 = start[at + 1];
            // the window's lanes before this one that are neighbours, lane j in bit j
            const uint64_t near = lane > 0 ? band[at] >> (64 - lane) : 0u;
            const int dE = valid ? -si * fi : 0;   // the plan bounds it
            const bool up = valid && dE > 0;
            const uint64_t m_up = __ballot(up);
            bool acc = valid && dE <= 0;
            if (up) acc = ref_accept(mix64(st + uint64_t(__popcll(m_up & below) + 1) * kGamma) >> 11, dE, T, nrT);
            const uint64_t m_acc = __ballot(acc);
            const uint64_t m_stale = __ballot(valid && (near & m_acc) != 0);
            const int lim = m_stale ? __builtin_ctzll(m_stale) : 64;   // lanes < lim stand
            const uint64_t in = lim == 64 ? ~uint64_t(0) : (uint64_t(1) << lim) - 1u;
            st += uint64_t(__popcll(m_up & in)) * kGamma;
            if (acc && lane < lim) {
                s[i] = int8_t(-si);
                e += dE;
            }
            rows_add(rows, m_acc & in, lane, row0, row1, si, w2, f, quarters);
            sync();
            i0 += lim;
        }
    }
    for (int i = lane; i < n; i += 64) {
        const int p = g.bit_pos[i];
        gs[p] = s[i];
        gf[p] = f[i];
    }
    for (int o = 32; o > 0; o >>= 1) e += __shfl_xor(e, o);
    if (lane == 0) {
        rng[r] = st;
        energy[r] = (init ? 0 : energy[r]) + e;
    }
}

static size_t ref_rows_lds(const DevGraph& g, int waves, bool lds_rows) {
    return 8 * size_t(g.n_pad) + 4 * (size_t((g.n + 4) & ~3) + size_t(waves) * g.n_pad) +
           (lds_rows ? 2 * size_t((g.m_dir + 7) & ~7) : 0) + size_t(waves) * g.n_pad;
}

// Replicas per workgroup of int_ref_rows_kernel, 0 where int_ref_kernel is the shorter, by the
// estimated time of R in rounds of what a CU holds at a time, in units of int_ref_kernel's one wave.
// There 32 waves or what its LDS holds run at 1 + 0.04 w; here workgroups of 1 to 16 replicas, as
// many side by side as the LDS holds (32 waves at most), at a base + 0.022 w, the base by the mean row:
// up to 32 entries (four rows at a time) 0.36 with the rows in LDS and 0.40 with them in L2, up to 64 0.51
// and 0.59, longer ones 0.60 and 0.72. Measured at n = 800 to 8,000 (degree 8: 0.30 of int_ref_kernel's
// time at one wave, 30: 0.40 and 0.46, 48: 0.50 and 0.57, 100: 0.67, 375: 0.75). Where rounds decide: 2,000
// vertices of degree 100 at 14 replicas a CU, two rounds of 7 against one of 14, 10.1 against 8.9 ms;
// of degree 48 the two rounds are the shorter (9.7 and 10.1); 1,500 of degree 375 at 18, 9.7 against 8.0.
int int_ref_rows_waves(const DevGraph& g, int R, int cus, bool* lds_rows) {
    if (g.w0 == 0) return 0;
    const int per_cu = (R + cus - 1) / cus;
    auto up = [](int a, int b) { return (a + b - 1) / b; };
    const size_t state = size_t(g.n_pad) * 5;
    if (state > kRefLdsLimit) return 0;
    const int held = 4 * state <= kRefLdsLimit ? int(std::min<size_t>(8, kRefLdsLimit / (4 * state))) * 4
                                               : int(kRefLdsLimit / state);
    const int old_rounds = up(per_cu, held);
    double best = old_rounds * (1.0 + 0.04 * up(per_cu, old_rounds));
    int waves = 0;
    const int64_t entries = g.m_dir, n = g.n;
    for (const bool in_lds : {true, false}) {
        const double base = entries <= 32 * n   ? (in_lds ? 0.36 : 0.40)
                            : entries <= 64 * n ? (in_lds ? 0.51 : 0.59)
                                                : (in_lds ? 0.60 : 0.72);
        for (int w = std::min(16, per_cu); w > 0; --w) {
            const size_t lds = ref_rows_lds(g, w, in_lds);
            if (lds > kRefLdsLimit) continue;
            const int groups = up(up(R, w), cus);   // of the fullest CU
            const int rounds = up(groups, std::max(1, std::min(32 / w, int(kRefLdsLimit / lds))));
            const double c = rounds * (base + 0.022 * (up(groups, rounds) * w));
            if (c < best) {
                best = c;
                waves = w;
                *lds_rows = in_lds;
            }
        }
    }
    return waves;
}

hipError_t launch_int_ref_rows(const DevGraph& g, int R, int waves, bool lds_rows, uint64_t seed_base,
                               const double* temp, int sweep_begin, int sweep_end, int init, int8_t* s_state,
                               int32_t* f_state, uint64_t* rng, long long* energy, hipStream_t st) {
    const size_t lds = ref_rows_lds(g, waves, lds_rows);
    const void* k = lds_rows ? reinterpret_cast<const void*>(&int_ref_rows_kernel<true>)
                             : reinterpret_cast<const void*>(&int_ref_rows_kernel<false>);
    const hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
    if (e != hipSuccess) return e;
    const unsigned blocks = unsigned((R + waves - 1) / waves), threads = unsigned(64 * waves);
    if (lds_rows)
        int_ref_rows_kernel<true><<<blocks, threads, lds, st>>>(g, R, seed_base, temp, sweep_begin, sweep_end, init,
                                                                s_state, f_state, rng, energy);
    else
        int_ref_rows_kernel<false><<<blocks, threads, lds, st>>>(g, R, seed_base, temp, sweep_begin, sweep_end, init,
                                                                 s_state, f_state, rng, energy);
    return hipGetLastError();
}

// ---- the colour-class trajectory, few replicas -----------------------------------------------
// A workgroup anneals one replica with its spins, fields and (where they fit) rows in LDS. A
// class is cut into steps of at most kWideDraws bits; in a step each of kWideStepWaves waves
// decides its share of the bits and sends out its own flips' rows -- LDS atomics, and no bit
// of a class reads a field that the class changes, so one barrier per step suffices --
// while the draw waves make the next step's draws. int_sweep_kernel gives a replica one wave,
// which decides up to 64 bits, draws for them and walks the flips' rows in L2 one after the
// other. At n = 800, degree 48, 18 classes and 16 replicas, 1,000 sweeps take 17.2 ms there and
// 8.4 here (0.95 and 0.47 us a class); what is left is a step's chain of draw, LDS reads and
// barrier. Draws split over two groups of waves took 9.4 ms, 12 step waves 9.4, 4 step waves
// 8.8, the next step's bits read ahead 9.2.
template <bool LDS_ROWS>
__global__ void __launch_bounds__(kWideBlock) int_wide_kernel(DevGraph g, uint64_t seed_base, const double* beta,
                                                              int sweep_begin, int sweep_end, int init,
                                                              int8_t* s_state, int32_t* f_state, long long* energy) {
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ Draw draws[2][kWideDraws];
    __shared__ long long red[kWideBlock / 64];
    const int n = g.n, np = g.n_pad, S = g.n_steps;
    const int tid = int(threadIdx.x), lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int32_t* start = reinterpret_cast<int32_t*>(smem);
    int2* steps = reinterpret_cast<int2*>(start + ((n + 4) & ~3));   // {first position, past the last}
    int32_t* f = reinterpret_cast<int32_t*>(steps + ((S + 1) & ~1));
    uint16_t* bit = reinterpret_cast<uint16_t*>(f + np);
    uint16_t* lrows = bit + np;
    int8_t* s = reinterpret_cast<int8_t*>(lrows + (LDS_ROWS ? (g.m_dir + 7) & ~7 : 0));
    const uint16_t* rows = LDS_ROWS ? lrows : g.prows;
    const int r = int(blockIdx.x);
    int8_t* gs = s_state + size_t(r) * size_t(np);
    int32_t* gf = f_state + size_t(r) * size_t(np);
    for (int i = tid; i <= n; i += kWideBlock) start[i] = g.nb_ptr[i];
    for (int i = tid; i < S; i += kWideBlock) steps[i] = int2{g.steps[i], g.steps[i + 1]};
    for (int i = tid; LDS_ROWS && i < g.m_dir / 2; i += kWideBlock)   // m_dir is even
        reinterpret_cast<uint32_t*>(lrows)[i] = reinterpret_cast<const uint32_t*>(g.prows)[i];
    for (int i = tid; i < n; i += kWideBlock) {
        bit[i] = uint16_t(g.pos_bit[i]);
        f[i] = init ? g.f0[i] : gf[i];
        s[i] = init ? int8_t(-1) : gs[i];
    }
    __syncthreads();
    const uint64_t seed = seed_base + uint64_t(r);
    const bool stepper = wave < kWideStepWaves;
    const int w2 = 2 * g.w0;
    const bool quarters = g.m_dir <= 32 * n;
    const int di = tid - 64 * kWideStepWaves;   // a draw wave's bit in a step
    auto put_draw = [&](int2 step, int sweep, float temperature, int buf) {
        const int p = step.x + di;
        if (p < step.y)
            draws[buf][di] = make_draw(draw_u01(seed, uint32_t(sweep), uint32_t(bit[p])), temperature);
    };
    auto step_at = [&](int k) {
        const int2 v = steps[k];
        return int2{__builtin_amdgcn_readfirstlane(v.x), __builtin_amdgcn_readfirstlane(v.y)};
    };
    int2 cur = step_at(0), nxt = step_at(S > 1 ? 1 : 0);
    double bt_next = beta[sweep_begin];
    float temp_next = float(1.0 / bt_next);
    if (!stepper) put_draw(cur, sweep_begin, temp_next, 0);
    __syncthreads();
    long long dsum = 0;
    int buf = 0, ahead = S > 2 ? 2 : 0;
    for (int sweep = sweep_begin; sweep < sweep_end; ++sweep) {
        const double bt = bt_next;
        const float temp = temp_next;
        bt_next = beta[min(sweep + 1, sweep_end - 1)];
        temp_next = float(1.0 / bt_next);
        for (int k = 0; k < S; ++k) {
            const int2 after = steps[ahead];   // read two steps ahead
            ahead = ahead + 1 < S ? ahead + 1 : 0;
            if (stepper) {
                const int p0 = cur.x, p1 = cur.y;
                const int share = (p1 - p0 + kWideStepWaves - 1) / kWideStepWaves;   // <= 64
                const int off = wave * share + lane, pos = p0 + off;
                const bool mine = lane < share && pos < p1;
                const int at = mine ? pos : p0;
                const int si = s[at], fi = f[at];
                const int row0 = start[at], row1 = start[at + 1];
                Draw dr = draws[buf][mine ? off : 0];
                asm("" : "+v"(dr.lo), "+v"(dr.hi));   // read with the others, not in the branch below
                const int dE = -si * fi;   // State::dE, ising_weighted.hpp:209 (the plan bounds it)
                bool acc = false;
                if (mine) {
                    const float ef = float(dE);
                    const bool below = dE <= 0 || ef < dr.lo, above = ef > dr.hi;
                    acc = below;
                    if (!below && !above) [[unlikely]] acc = uphill_accept(-double(dE) * bt, dr.u);
                }
                const uint64_t m = __ballot(acc);
                if (m) {
                    if (acc) {
                        dsum += dE;
                        s[at] = int8_t(-si);
                    }
                    rows_add(rows, m, lane, row0, row1, si, w2, f, quarters);
                }
            } else {
                const bool wrap = k + 1 == S;
                put_draw(nxt, wrap ? sweep + 1 : sweep, wrap ? temp_next : temp, buf ^ 1);
            }
            buf ^= 1;
            cur = nxt;
            nxt = int2{__builtin_amdgcn_readfirstlane(after.x), __builtin_amdgcn_readfirstlane(after.y)};
            __syncthreads();
        }
    }
    for (int i = tid; i < n; i += kWideBlock) {
        gf[i] = f[i];
        gs[i] = s[i];
    }
    for (int o = 32; o > 0; o >>= 1) dsum += __shfl_xor(dsum, o);
    if (lane == 0) red[wave] = dsum;
    __syncthreads();
    if (tid == 0) {
        long long t = 0;
        for (int w = 0; w < kWideBlock / 64; ++w) t += red[w];
        energy[r] = (init ? 0 : energy[r]) + t;
    }
}

static size_t wide_lds(const DevGraph& g, bool lds_rows) {
    return 4 * (size_t((g.n + 4) & ~3) + 2 * size_t((g.n_steps + 1) & ~1) + size_t(g.n_pad)) + 2 * size_t(g.n_pad) +
           (lds_rows ? 2 * size_t((g.m_dir + 7) & ~7) : 0) + size_t(g.n_pad);
}
constexpr size_t kWideStatic = 2 * kWideDraws * sizeof(Draw) + (kWideBlock / 64) * sizeof(long long);

// ---- the colour-class trajectory, many replicas ----------------------------------------------
// A wave per replica, as in int_sweep_kernel, several of a workgroup sharing the 16-bit rows
// in LDS, and an uphill move decided through the float exponential's band instead of the
// FP64 exponential. Nothing is shared between waves after the rows are in. 8,192 replicas x
// 1,000 sweeps at n = 800, degree 48: 93.7 -> 63.0 ms; the bound is vector issue (an instruction
// in 77% of the SIMDs' cycles; the LDS is active in 24%).
template <bool LDS_ROWS>
__global__ void __launch_bounds__(1024) int_sweep_rows_kernel(DevGraph g, int R, uint64_t seed_base, const double* beta,
                                                              int sweep_begin, int sweep_end, int init,
                                                              int8_t* s_state, int32_t* f_state, long long* energy) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int n = g.n, np = g.n_pad, K = g.n_classes;
    const int tid = int(threadIdx.x), lane = tid & 63, wave = tid >> 6, block = int(blockDim.x), waves = block / 64;
    int32_t* start = reinterpret_cast<int32_t*>(smem);
    int32_t* cls = start + ((n + 4) & ~3);
    int32_t* fields = cls + ((K + 4) & ~3);
    uint16_t* bit = reinterpret_cast<uint16_t*>(fields + size_t(waves) * np);
    uint16_t* lrows = bit + np;
    int8_t* spins = reinterpret_cast<int8_t*>(lrows + (LDS_ROWS ? (g.m_dir + 7) & ~7 : 0));
    const uint16_t* rows = LDS_ROWS ? lrows : g.prows;
    for (int i = tid; i <= n; i += block) start[i] = g.nb_ptr[i];
    for (int i = tid; i <= K; i += block) cls[i] = g.cls_ptr[i];
    for (int i = tid; i < n; i += block) bit[i] = uint16_t(g.pos_bit[i]);
    for (int i = tid; LDS_ROWS && i < g.m_dir / 2; i += block)   // m_dir is even
        reinterpret_cast<uint32_t*>(lrows)[i] = reinterpret_cast<const uint32_t*>(g.prows)[i];
    __syncthreads();
    const int r = int(blockIdx.x) * waves + wave;
    if (r >= R) return;   // the whole wave leaves; the rest never syncs across waves
    int32_t* f = fields + size_t(wave) * np;
    int8_t* s = spins + size_t(wave) * np;
    int8_t* gs = s_state + size_t(r) * size_t(np);
    int32_t* gf = f_state + size_t(r) * size_t(np);
    for (int i = lane; i < n; i += 64) {
        f[i] = init ? g.f0[i] : gf[i];
        s[i] = init ? int8_t(-1) : gs[i];
    }
    auto sync = [] {
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    sync();
    const uint64_t seed = seed_base + uint64_t(r);
    const int w2 = 2 * g.w0;
    const bool quarters = g.m_dir <= 32 * n;
    long long dsum = 0;
    for (int sweep = sweep_begin; sweep < sweep_end; ++sweep) {
        const double bt = beta[sweep];
        for (int c = 0; c < K; ++c) {
            const int c1 = cls[c + 1];
            for (int base = cls[c]; base < c1; base += 64) {
                const int pos = base + lane;
                const bool mine = pos < c1;
                const int at = mine ? pos : base;
                const int si = s[at];
                const int dE = -si * f[at];   // State::dE, ising_weighted.hpp:209 (the plan bounds it)
                const int row0 = start[at], row1 = start[at + 1];
                const uint32_t b = bit[at];
                bool acc = mine && dE <= 0;
                if (mine && dE > 0) acc = uphill_accept(-double(dE) * bt, draw_u01(seed, uint32_t(sweep), b));
                const uint64_t m = __ballot(acc);
                if (m) {
                    if (acc) {
                        dsum += dE;
                        s[at] = int8_t(-si);
                    }
                    rows_add(rows, m, lane, row0, row1, si, w2, f, quarters);
                    sync();
                }
            }
        }
    }
    for (int i = lane; i < n; i += 64) {
        gf[i] = f[i];
        gs[i] = s[i];
    }
    for (int o = 32; o > 0; o >>= 1) dsum += __shfl_xor(dsum, o);
    if (lane == 0) energy[r] = (init ? 0 : energy[r]) + dsum;
}

static size_t sweep_rows_lds(const DevGraph& g, int waves, bool lds_rows) {
    return 4 * (size_t((g.n + 4) & ~3) + size_t((g.n_classes + 4) & ~3)) + 2 * size_t(g.n_pad) +
           (lds_rows ? 2 * size_t((g.m_dir + 7) & ~7) : 0) + size_t(waves) * g.n_pad * 5;
}

// The kernel of a colour-class launch of R replicas: the least of the estimated times of a
// sweep, in us, over the rounds that R takes at what the LDS holds per CU. At one replica a
// sweep takes about 0.35 per class + 0.045 per bit in int_sweep_kernel, 0.33 per 64 bits of a
// class + 0.017 per bit in int_sweep_rows_kernel (1.28 times that with the rows in L2), and
// 0.4 per step + 0.0035 per bit in int_wide_kernel (1.1 times that with the rows in L2: 2,000 vertices
// of degree 48 at 16 replicas a CU take 152 us a sweep there and 129 in int_sweep_kernel); more
// waves per CU lengthen it by 4 to 5.5% each, a second int_wide_kernel workgroup by 30%. Measured at n = 100 to 8,000, degree 8
// to 48 (n = 800, degree 48: 37, 19.5 and 10.3 us at one replica, 42, 21 and 42 at 1,024, 97
// and 65 at 8,192).
IntShape int_shape(const DevGraph& g, int R, int cus) {
    IntShape best{kIntSweep, 0};
    if (g.w0 == 0) return best;
    const int per_cu = (R + cus - 1) / cus;
    auto cost = [&](int capacity, double base, double slope) {
        const int rounds = (per_cu + capacity - 1) / capacity;
        return rounds * base * (1.0 + slope * ((per_cu + rounds - 1) / rounds - 1));
    };
    const int held = int(std::min<size_t>(32, kRefLdsLimit / (size_t(g.n_pad) * 5)));
    if (held < 1) return best;
    double least = 0.95 * cost(held, 0.35 * g.n_classes + 0.045 * g.n, 0.04);
    for (const bool in_lds : {true, false}) {
        const double far = in_lds ? 1.0 : 1.28;
        const size_t wide = wide_lds(g, in_lds) + kWideStatic;
        if (wide <= kRefLdsLimit) {
            const int capacity = 2 * wide <= kRefLdsLimit ? 2 : 1;
            const double c = (in_lds ? 1.0 : 1.1) * cost(capacity, 0.4 * g.n_steps + 0.0035 * g.n, 0.3);
            if (c < least) {
                least = c;
                best = IntShape{in_lds ? kIntWide : kIntWideL2, 0};
            }
        }
        int fit = std::min(16, per_cu);
        while (fit > 0 && sweep_rows_lds(g, fit, in_lds) > kRefLdsLimit) --fit;
        if (fit > 0) {
            const int groups = std::max(1, std::min(32 / fit, int(kRefLdsLimit / sweep_rows_lds(g, fit, in_lds))));
            const double c = cost(fit * groups, far * (0.33 * (g.n / 64.0 + 0.5 * g.n_classes) + 0.017 * g.n),
                                  in_lds ? 0.04 : 0.055);
            if (c < least) {
                least = c;
                const int rounds = (per_cu + fit - 1) / fit;   // of workgroups
                best = IntShape{in_lds ? kIntRows : kIntRowsL2, (per_cu + rounds - 1) / rounds};
            }
        }
        if (wide <= kRefLdsLimit) break;   // with the rows in LDS there is no need to ask for L2
    }
    return best;
}

hipError_t launch_int_rows(const DevGraph& g, int R, const IntShape& sh, uint64_t seed_base, const double* beta,
                           int sweep_begin, int sweep_end, int init, int8_t* s_state, int32_t* f_state,
                           long long* energy, hipStream_t st) {
    const bool lds_rows = sh.kind == kIntRows;
    const size_t lds = sweep_rows_lds(g, sh.waves, lds_rows);
    const void* k = lds_rows ? reinterpret_cast<const void*>(&int_sweep_rows_kernel<true>)
                             : reinterpret_cast<const void*>(&int_sweep_rows_kernel<false>);
    const hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
    if (e != hipSuccess) return e;
    const unsigned blocks = unsigned((R + sh.waves - 1) / sh.waves), threads = unsigned(64 * sh.waves);
    if (lds_rows)
        int_sweep_rows_kernel<true><<<blocks, threads, lds, st>>>(g, R, seed_base, beta, sweep_begin, sweep_end, init,
                                                                  s_state, f_state, energy);
    else
        int_sweep_rows_kernel<false><<<blocks, threads, lds, st>>>(g, R, seed_base, beta, sweep_begin, sweep_end, init,
                                                                   s_state, f_state, energy);
    return hipGetLastError();
}

hipError_t launch_int_wide(const DevGraph& g, int R, const IntShape& sh, uint64_t seed_base, const double* beta, int sweep_begin,
                           int sweep_end, int init, int8_t* s_state, int32_t* f_state, long long* energy,
                           hipStream_t st) {
    const bool lds_rows = sh.kind == kIntWide;
    const size_t lds = wide_lds(g, lds_rows);
    const void* k = lds_rows ? reinterpret_cast<const void*>(&int_wide_kernel<true>)
                             : reinterpret_cast<const void*>(&int_wide_kernel<false>);
    const hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
    if (e != hipSuccess) return e;
    if (lds_rows)
        int_wide_kernel<true><<<unsigned(R), kWideBlock, lds, st>>>(g, seed_base, beta, sweep_begin, sweep_end, init,
                                                                   s_state, f_state, energy);
    else
        int_wide_kernel<false><<<unsigned(R), kWideBlock, lds, st>>>(g, seed_base, beta, sweep_begin, sweep_end, init,
                                                                    s_state, f_state, energy);
    return hipGetLastError();
}

}  // namespace qb
