// qb_introws.hip -- gfx950 kernels of the integer annealer for graphs whose couplings all
// have one magnitude (max-cut and +-J graphs): adjacency rows as 16-bit words (neighbour,
// sign in the top bit), which fit a CU's LDS where 32-bit neighbours and weights do not.
//
//   int_ref_rows_kernel  the reference's own trajectory (wising::anneal,
//                        src/ising_weighted.hpp:250-267), a wave per replica, several
//                        replicas of a workgroup sharing the rows in LDS.
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

}  // namespace

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
            const long long dE = valid ? -(long long)si * (long long)fi : 0;
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

// Replicas per workgroup of int_ref_rows_kernel, 0 where int_ref_kernel is the shorter. Each
// candidate runs R in rounds of what its LDS holds per CU (at most 16 waves here, 32 there), a
// round of w waves taking about 0.51 + 0.022 w with the rows in LDS, 0.57 + 0.02 w with them
// in L2, and 1 + 0.04 w in int_ref_kernel (measured at n = 800 and 2,000, degree 48: 6.4, 8.4
// and 12.3 or 14.5 ms at one wave; at 4,096 replicas of the larger graph int_ref_kernel's one
// round of 16 waves beats two of 13).
int int_ref_rows_waves(const DevGraph& g, int R, int cus, bool* lds_rows) {
    if (!g.orows) return 0;
    const int per_cu = (R + cus - 1) / cus;
    auto cost = [&](int capacity, double base, double slope) {
        const int rounds = (per_cu + capacity - 1) / capacity;
        return rounds * (base + slope * ((per_cu + rounds - 1) / rounds));
    };
    const size_t state = size_t(g.n_pad) * 5;
    if (state > kRefLdsLimit) return 0;
    const int held = 4 * state <= kRefLdsLimit ? int(std::min<size_t>(8, kRefLdsLimit / (4 * state))) * 4
                                               : int(kRefLdsLimit / state);
    double best = cost(held, 1.0, 0.04);
    int waves = 0;
    for (const bool in_lds : {true, false}) {
        int fit = std::min(16, per_cu);
        while (fit > 0 && ref_rows_lds(g, fit, in_lds) > kRefLdsLimit) --fit;
        if (fit == 0) continue;
        const double c = in_lds ? cost(fit, 0.51, 0.022) : cost(fit, 0.57, 0.02);
        if (c < best) {
            best = c;
            const int rounds = (per_cu + fit - 1) / fit;
            waves = (per_cu + rounds - 1) / rounds;
            *lds_rows = in_lds;
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

}  // namespace qb
