// qb_solo.hip -- gfx950 kernel of the ray x voxel anneal for problems whose branch state
// fits one CU's LDS (qb_anneal_branches; branch_fractions, src/ising_recon.hpp:121-166).
//
// One workgroup anneals one branch from its first sweep to its last with the branch's
// residuals and spins in LDS, so a colour class costs LDS gathers, the chain sums, the
// decisions and one workgroup barrier. The XCD-team kernel pays an L2 round trip per
// gather and a barrier through L2 per class, about 4.5 us however few bits the class has.
//
// What bounds a class here is the instructions its longest wave issues, so its work is
// spread over lanes and waves:
//   - kSoloStepWaves waves step tiles, one wave's unit of work each, of three kinds: four
//     lanes per chain of kSeg entries (16 chains, a lane makes 4 terms), two lanes per chain
//     (32 chains; classes whose chains do not fit the waves the other way, and bits of 17 to
//     32 chains), and ray-free bits, a lane each. The terms are added in the chain's order,
//     the running sum passed from lane to lane by DPP. A bit's chains stay inside its tile,
//     so the chain sums meet and the decision spreads with no workgroup sync; a bit with
//     more than kSoloChains chains (wide) is evaluated by the whole workgroup.
//   - the other kSoloDrawWaves waves make the next class's draws (a lane per bit) and turn
//     each into the two energies between which its decision is not settled.
// Each step wave runs down its own list of tiles of every kind; a tile has a fixed layout,
// and the next one's operands are loaded into registers as soon as the current one's are
// read, so the loads stay in flight across the class barrier. Every load of a kind is
// unconditional and lands in registers that are dead when it is issued: a branch around
// them makes the compiler merge copies, which wait for the loads at once.
//
// Every sum is the packed step's, term for term and in its order (chains of kSeg, runs of
// kChainRun, runs in order, then the neighbours in CSR order), so spins and residuals are
// the team kernel's bit for bit.
//
// Measured, team kernel -> here (kernel and call): 1,964 bits x 960 rays, 8 branches, 250
// sweeps, FP32 24.3 -> 5.4 ms (0.95 us a class); 24,633 bits x 8,640 rays, 16 branches, FP64
// 64.7 -> 37.4 ms (3.0 us a class; some instruction in 70% of its CUs' SIMD cycles, a vector
// one in 47%, and the rest waits of two waves a SIMD at once); at 256
// branches the same problems take 10.6 -> 1.0 and 15.6 -> 3.1 us a class.
#include <type_traits>

#include "qb_internal.h"
#include "qb_rng.h"

namespace qb {

namespace {

__device__ __forceinline__ void lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// A workgroup barrier that orders LDS only: the waves' loads for their next tiles stay in
// flight across it (a full fence would wait for them).
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

__device__ __forceinline__ int uniform(uint32_t v) { return __builtin_amdgcn_readfirstlane(int(v)); }

__device__ __forceinline__ double u64_double(uint32_t lo, uint32_t hi) {
    return __longlong_as_double((long long)((uint64_t(hi) << 32) | lo));
}

template <int CTRL>
__device__ __forceinline__ double dpp_double(double v) {
    const uint64_t b = uint64_t(__double_as_longlong(v));
    const uint32_t lo = uint32_t(__builtin_amdgcn_mov_dpp(int(uint32_t(b)), CTRL, 0xF, 0xF, true));
    const uint32_t hi = uint32_t(__builtin_amdgcn_mov_dpp(int(uint32_t(b >> 32)), CTRL, 0xF, 0xF, true));
    return u64_double(lo, hi);
}

// A branch's spins in LDS, in position order: a byte per bit where they fit beside the
// residuals (one instruction fewer per word and shift on each of a bit's seven reads), else
// a bit.
template <bool BITS>
struct Spins {
    unsigned char* x;
    __device__ __forceinline__ uint32_t at(int pos) const {
        if constexpr (BITS) return (reinterpret_cast<const uint32_t*>(x)[pos >> 5] >> (pos & 31)) & 1u;
        else return x[pos];
    }
    __device__ __forceinline__ void flip(int pos, uint32_t was) const {
        if constexpr (BITS) atomicXor(reinterpret_cast<uint32_t*>(x) + (pos >> 5), 1u << (pos & 31));
        else x[pos] = static_cast<unsigned char>(was ^ 1u);
    }
};

// The exact decision, out of line: it is rare, and its constants inlined at every site would
// crowd the scalar registers of the loop.
__device__ __attribute__((noinline)) bool exact_accept(double x, double u) { return uphill_accept(x, u); }

template <typename T, bool BITS>
struct SoloState {
    T* r;             // [n_rays + 1]
    Spins<BITS> x;
    double* part;     // this wave's chain sums
    int lane;
    // lambda * (+-1): |lambda|'s words, and the spin a like neighbour must differ from when
    // lambda is negative
    uint32_t lam_hi, lam_lo, lam_neg;
    double lambda;
};

// A copy the compiler keeps apart from `v`, so that v's register is free for the next load.
template <typename V>
__device__ __forceinline__ V kept(V v) {
    asm("" : "+v"(v));
    return v;
}

// The running sum of a chain over its four lanes, from each lane's four terms (dE: the
// chain's seed); every lane returns the chain's sum.
__device__ __forceinline__ double four_lane_sum(double dE, const double (&tm)[4]) {
#pragma unroll
    for (int u = 0; u < 4; ++u) dE += tm[u];
    dE = dpp_double<0x00>(dE);
#pragma unroll
    for (int u = 0; u < 4; ++u) dE += tm[u];
    dE = dpp_double<0x55>(dE);
#pragma unroll
    for (int u = 0; u < 4; ++u) dE += tm[u];
    dE = dpp_double<0xAA>(dE);
#pragma unroll
    for (int u = 0; u < 4; ++u) dE += tm[u];
    return dpp_double<0xFF>(dE);
}

// A wave's list of tiles of one kind, with the operands of its next tile loaded (or in
// flight). LPC lanes per chain; LPC = 1: ray-free bits, no entries and a fourth granule of
// head (the draw's key).
template <int LPC>
struct Pipe {
    static constexpr int kHeads = LPC == 1 ? 4 : 3;
    static constexpr int kRows = LPC == 1 ? 0 : kSeg / LPC;
    static constexpr int kChains = 64 / LPC;
    static constexpr int kBytes = solo_tile_bytes(LPC);
    uint4 h[kHeads];
    uint4 e[kRows > 0 ? kRows : 1];
    const char* list;    // uniform
    int n, at;           // tiles, and the loaded one's index
    int cls, sweep;      // the loaded tile's class and sweep

    __device__ __forceinline__ void issue(int lane) {
        const char* b = list + int64_t(at) * kBytes;
        const uint32_t hv = uint32_t(lane / LPC) * 16u, ev = uint32_t(lane) * 16u;
#pragma unroll
        for (int v = 0; v < kHeads; ++v) h[v] = *reinterpret_cast<const uint4*>(b + hv + v * kChains * 16);
#pragma unroll
        for (int u = 0; u < kRows; ++u) e[u] = *reinterpret_cast<const uint4*>(b + ev + kHeads * kChains * 16 + u * 1024);
    }
    __device__ __forceinline__ void start(const char* tiles, int64_t offset, int count, int first_cls, int sweep0, int lane) {
        list = tiles + offset;
        n = count;
        at = 0;
        cls = count > 0 ? first_cls : -1;
        sweep = sweep0;
        if (count > 0) issue(lane);
    }
    // On to the next tile: its class is in the current one's head.
    __device__ __forceinline__ void advance(int next_cls, int lane) {
        if (++at == n) {
            at = 0;
            ++sweep;
        }
        cls = next_cls;
        issue(lane);
    }
};

// The step of the pipe's tile; issues the next tile's loads once the operands are read.
template <typename T, bool BITS, int LPC>
__device__ __forceinline__ void tile_step(const DevProblem& p, const SoloState<T, BITS>& s, Pipe<LPC>& t,
                                          const Draw* draws, uint64_t branch_key, int sweep, double beta,
                                          float temperature) {
    constexpr int kRows = Pipe<LPC>::kRows;
    const int lane = s.lane;
    const int pos = kept(int(t.h[0].x));
    const uint32_t info = kept(t.h[0].y);
    const int next_cls = uniform(t.h[0].z);
    const uint32_t flags = uint32_t(uniform(info));   // the tile's, the same in every lane
    T rv[kRows > 0 ? kRows : 1];
    uint32_t ray[kRows > 0 ? kRows : 1];
    float ea[kRows > 0 ? kRows : 1];
#pragma unroll
    for (int u = 0; u < kRows; ++u) {
        ray[u] = kept(t.e[u].x);
        rv[u] = s.r[ray[u]];
    }
    const uint32_t xb = s.x.at(pos);
    const uint32_t nq[kNb] = {t.h[1].x, t.h[1].y, t.h[1].z, t.h[1].w, t.h[2].x, t.h[2].y};
    uint32_t xn[kNb];
#pragma unroll
    for (int v = 0; v < kNb; ++v) xn[v] = s.x.at(int(nq[v]));
    Draw dr{};
    uint64_t key = 0;
    uint32_t dbit = 0;
    if constexpr (LPC == 1) {
        key = kept((uint64_t(t.h[3].y) << 32) | t.h[3].x);
        dbit = kept(t.h[3].z);
    } else {
        dr = draws[t.h[0].w];
    }
    const int j = int((info >> 5) & 255u), nn = int((info >> 21) & 1023u);
    const bool lead = (lane & (LPC - 1)) == 0;   // the chain's first lane
    const bool first = lead && j == 0;           // the bit's (padding chains have j = 255)
    const double delta = xb ? -1.0 : 1.0;
    double dE = j == 0 ? u64_double(t.h[2].z, t.h[2].w) * delta : 0.0;
    // terms w (r a + a^2 / 2), a = a_k delta: a^2 is exact in FP64 (24-bit shares), so the
    // fused form rounds as r a + 0.5 a a does
    double tm[kRows > 0 ? kRows : 1];
#pragma unroll
    for (int u = 0; u < kRows; ++u) {
        ea[u] = kept(__uint_as_float(t.e[u].y));
        const double ad = double(ea[u]) * delta;
        tm[u] = u64_double(t.e[u].z, t.e[u].w) * fma(0.5 * ad, ad, double(rv[u]) * ad);
    }
    t.advance(next_cls, lane);
    if constexpr (LPC > 1) {
        // added in the chain's order: each lane of a chain continues the sum of the lane before
if constexpr (LPC == 4) {
            dE = four_lane_sum(dE, tm);
        } else {
#pragma unroll
            for (int u = 0; u < kRows; ++u) dE += tm[u];
            dE = dpp_double<0xA0>(dE);
#pragma unroll
            for (int u = 0; u < kRows; ++u) dE += tm[u];
            dE = dpp_double<0xF5>(dE);
        }
        if (flags & kSoloMulti) {
            // runs of kChainRun chain sums by their first lanes, then the runs by the bit's first
            const int nch = int((info >> 13) & 255u), slot = lane / LPC;
            if (lead) s.part[slot] = dE;
            lds_fence();
            if (lead && j % kChainRun == 0) {
                double v[kChainRun];
#pragma unroll
                for (int w = 1; w < 4; ++w) v[w] = s.part[slot + w];
#pragma unroll
                for (int w = 1; w < 4; ++w) dE = j + w < nch ? dE + v[w] : dE;
                if (flags & kSoloHalf) {   // some run is longer than four
#pragma unroll
                    for (int w = 4; w < kChainRun; ++w) v[w] = s.part[slot + w];
#pragma unroll
                    for (int w = 4; w < kChainRun; ++w) dE = j + w < nch ? dE + v[w] : dE;
                }
            }
            if (flags & kSoloRuns) {
                lds_fence();
                if (lead && j % kChainRun == 0) s.part[slot] = dE;
                lds_fence();
                if (first) {
                    constexpr int kRuns = kSoloChains / kChainRun;
                    double v[kRuns];
#pragma unroll
                    for (int w = 1; w < kRuns; ++w) v[w] = s.part[slot + w * kChainRun];
#pragma unroll
                    for (int w = 1; w < kRuns; ++w) dE = w * kChainRun < nch ? dE + v[w] : dE;
                }
            }
            lds_fence();
        }
    }
    bool acc = false;
    if (first) {
        // lambda * (+-1) per neighbour in CSR order (an exact 0 past the bit's count)
        const uint32_t xs = xb ^ s.lam_neg;
#pragma unroll
        for (int v = 0; v < kNb; ++v) {
            const uint32_t hi = ((xn[v] ^ xs) << 31) | s.lam_hi;
            dE += u64_double(v < nn ? s.lam_lo : 0u, v < nn ? hi : 0u);
        }
        if (nn > kNb) [[unlikely]] {
            const int nb0 = p.nb_ptr[pos];
            for (int k = nb0 + kNb; k < nb0 + nn; ++k) dE += s.lambda * (s.x.at(p.nb[k]) != xb ? -1.0 : 1.0);
        }
        if constexpr (LPC == 1) {
            dr = make_draw(draw_u01(branch_key + key, uint32_t(sweep), dbit), temperature);
        } else if (flags & kSoloOwn) [[unlikely]] {
            // a bit past the class's draws made ahead
            dr = make_draw(draw_u01(branch_key + p.draw_key[pos], uint32_t(sweep), uint32_t(p.draw_bit[pos])),
                           temperature);
        }
        const float ef = float(dE);
        const bool below = dE <= 0.0 || ef < dr.lo, above = ef > dr.hi;
        acc = below;
        if (!below && !above) [[unlikely]] acc = exact_accept(-dE * beta, dr.u);
    }
    const uint64_t flips = __ballot(acc);
    if (flips == 0) return;
    if (acc) s.x.flip(pos, xb);
    if constexpr (LPC > 1) {
        const int head = (lane & ~(LPC - 1)) - j * LPC;   // the bit's first lane
        bool mine = j < kSoloChains && ((flips >> (head & 63)) & 1u);
        if (flags & kSoloSeq) [[unlikely]] {
            // some column of the tile repeats a ray: those bits' first lanes scatter in CSR order
            if (mine && (info >> 31)) {
                if (first)
                    for (int k = p.col_ptr[pos]; k < p.col_ptr[pos + 1]; ++k) {
                        const RayEnt ek = p.ent[k];
                        s.r[ek.ray] = residual_add<T>(s.r[ek.ray], ek.a, delta);
                    }
                mine = false;
            }
        }
        if (mine) {
#pragma unroll
            for (int u = 0; u < kRows; ++u) s.r[ray[u]] = residual_add<T>(rv[u], ea[u], delta);
        }
    }
}

// A bit with more than kSoloChains chains, by the whole workgroup, four lanes per chain: the
// chain sums meet in `sums`, the runs are added there, and the first lane of the last wave,
// which read the neighbours and made the draw meanwhile, adds the runs and decides. A bit's
// operands come from memory in one round: its record's head and its entries together.
template <typename T, bool BITS>
__device__ __forceinline__ void wide_step(const DevProblem& p, const SoloState<T, BITS>& s, const SoloWide* rec,
                                          double* sums, int* flag, uint64_t branch_key, int sweep, double beta) {
    constexpr int kPass = kSoloBlock / 4;   // chains per pass
    const int tid = int(threadIdx.x), k = tid & 3;
    const int pos = rec->pos, k0 = rec->k0, n_ent = rec->k1 - k0;
    const int n_chain = (n_ent + kSeg - 1) / kSeg, n_run = (n_chain + kChainRun - 1) / kChainRun;
    const bool decider = tid == kSoloBlock - 64;
    RayEnt e[4];
    auto load = [&](int chain) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int i = chain * kSeg + 4 * k + u;
            e[u] = i < n_ent ? p.ent[k0 + i] : RayEnt{p.n_rays, 0.0f, 0.0};   // padding adds exact zeros
        }
    };
    load(tid >> 2);
    const uint32_t xb = s.x.at(pos);
    const double delta = xb ? -1.0 : 1.0;
    const double lin = rec->lin;
    uint32_t unlike = 0;
    double u01 = 0.0;
    if (decider) {
#pragma unroll
        for (int v = 0; v < kNb; ++v) unlike |= (s.x.at(rec->q[v]) ^ xb) << v;
        u01 = draw_u01(branch_key + rec->key, uint32_t(sweep), uint32_t(rec->bit));
    }
    for (int c0 = 0; c0 < n_chain; c0 += kPass) {
        const int chain = c0 + (tid >> 2);
        if (c0 > 0) load(chain);
        double tm[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const double ad = double(e[u].a) * delta;
            tm[u] = e[u].w * fma(0.5 * ad, ad, double(s.r[e[u].ray]) * ad);
        }
        const double sum = four_lane_sum(chain == 0 ? lin * delta : 0.0, tm);
        if (k == 0 && chain < n_chain) sums[chain] = sum;
    }
    lds_barrier();
    if (tid < n_run) {   // n_run <= kSoloBlock: the host keeps longer bits off this path
        const int m = min(kChainRun, n_chain - tid * kChainRun);
        double g = sums[tid * kChainRun];
#pragma unroll
        for (int u = 1; u < kChainRun; ++u) {
            const double v = sums[min(tid * kChainRun + u, n_chain - 1)];
            g = u < m ? g + v : g;
        }
        sums[tid * kChainRun] = g;
    }
    lds_barrier();
    if (decider) {
        double dE = sums[0];
        for (int q = 1; q < n_run; ++q) dE += sums[q * kChainRun];
        const int nn = rec->nn;
        for (int v = 0; v < min(nn, kNb); ++v) dE += p.lambda * (((unlike >> v) & 1u) ? -1.0 : 1.0);
        if (nn > kNb) [[unlikely]] {
            const int nb0 = p.nb_ptr[pos];
            for (int v = nb0 + kNb; v < nb0 + nn; ++v) dE += p.lambda * (s.x.at(p.nb[v]) != xb ? -1.0 : 1.0);
        }
        const bool acc = dE <= 0.0 || exact_accept(-dE * beta, u01);
        *flag = acc ? 1 : 0;
        if (acc) s.x.flip(pos, xb);
    }
    lds_barrier();
    if (*flag) {
        if (rec->seq) {
            if (tid == 0)
                for (int i = k0; i < k0 + n_ent; ++i)
                    s.r[p.ent[i].ray] = residual_add<T>(s.r[p.ent[i].ray], p.ent[i].a, delta);
        } else {
            for (int c0 = 0; c0 < n_chain; c0 += kPass) {
                if (n_chain > kPass) load(c0 + (tid >> 2));
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int i = (c0 + (tid >> 2)) * kSeg + 4 * k + u;
                    if (i < n_ent) s.r[e[u].ray] = residual_add<T>(s.r[e[u].ray], e[u].a, delta);
                }
            }
        }
    }
    lds_barrier();   // sums and flag are written again by the next wide bit
}

}  // namespace

template <typename T, bool BITS>
__global__ void __launch_bounds__(kSoloBlock) ray_solo_kernel(DevProblem p, DevSolo d, uint32_t* xs, T* rs,
                                                              uint64_t seed_offset, const double* beta,
                                                              int sweep_begin, int sweep_end, int recompute_every) {
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ int s_flag;
    __shared__ Draw s_draw[2][kSoloDraws];
    __shared__ double s_part[kSoloStepWaves][kSoloPart];
    double* sums = reinterpret_cast<double*>(smem);
    T* r = reinterpret_cast<T*>(sums + d.wide_chains);
    const Spins<BITS> x{reinterpret_cast<unsigned char*>(r + p.n_rays + 1)};
    const int tid = int(threadIdx.x), lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int branch = int(blockIdx.x);
    const int words = (p.n + 31) / 32;   // a branch's spins in memory, a bit each
    uint32_t* xg = xs + size_t(branch) * size_t(words);
    T* rg = rs + size_t(branch) * size_t(p.n_rays);
    // the branch's state into LDS: x = 0, r = -d, or what the last launch left
    for (int k = tid; k < p.n_rays; k += kSoloBlock) r[k] = sweep_begin == 0 ? T(-p.d[k]) : rg[k];
    if (tid == 0) r[p.n_rays] = T(0);
    if constexpr (BITS) {
        for (int w = tid; w < words; w += kSoloBlock) reinterpret_cast<uint32_t*>(x.x)[w] = sweep_begin > 0 ? xg[w] : 0u;
    } else {
        for (int i = tid; i < p.n; i += kSoloBlock) x.x[i] = 0;
        if (sweep_begin > 0)
            for (int i = tid; i < p.n; i += kSoloBlock)
                x.x[i] = static_cast<unsigned char>((xg[i >> 5] >> (i & 31)) & 1u);
    }
    const uint64_t branch_key = seed_offset + uint64_t(branch) + 1u;
    const bool stepper = wave < kSoloStepWaves;
    const uint64_t lam = uint64_t(__double_as_longlong(p.lambda));
    const SoloState<T, BITS> s{r, x, s_part[stepper ? wave : 0], lane, uint32_t(lam >> 32) & 0x7FFFFFFFu,
                               uint32_t(lam), uint32_t(lam >> 63), p.lambda};
    const int K = p.n_classes;
    // The wave's lists of tiles of four lanes per chain, two (step waves), and ray-free bits.
    Pipe<4> t4;
    Pipe<2> t2;
    Pipe<1> t1;
    {
        const SoloLists* l = d.lists + wave;
        const char* base = reinterpret_cast<const char*>(d.blk);
        t4.start(base, l->at[0], l->n[0], l->cls[0], sweep_begin, lane);
        t2.start(base, l->at[1], l->n[1], l->cls[1], sweep_begin, lane);
        t1.start(base, l->at[2], l->n[2], l->cls[2], sweep_begin, lane);
    }
    // Draw waves: lane `di` makes the draw of the class's di-th bit with entries. A class's
    // record {first position, bits} is read three classes ahead, its keys two, and its draws
    // are made one ahead.
    const int di = (wave - kSoloStepWaves) * 64 + lane;
    int2 crec{}, krec{};   // the record read last, and the one whose keys are loaded
    uint64_t dkey = 0;
    uint32_t dbit = 0;
    bool dlive = false;
    auto load_class = [&](int c) {
        uint32_t zero = 0;
        asm("" : "+v"(zero));
        crec = *reinterpret_cast<const int2*>(reinterpret_cast<const char*>(d.cls_draw + c) + zero);
    };
    auto load_keys = [&] {
        krec = crec;
        dlive = di < crec.y;
        if (dlive) {
            dkey = p.draw_key[crec.x + di];
            dbit = uint32_t(p.draw_bit[crec.x + di]);
        }
    };
    // the class's first chunk of bits from the loaded keys, further chunks from memory
    auto put_draw = [&](int2 rec, int sweep, float temperature, int buf) {
        if (dlive) s_draw[buf][di] = make_draw(draw_u01(branch_key + dkey, uint32_t(sweep), dbit), temperature);
        for (int i = di + 64 * kSoloDrawWaves; i < rec.y; i += 64 * kSoloDrawWaves)
            s_draw[buf][i] = make_draw(draw_u01(branch_key + p.draw_key[rec.x + i], uint32_t(sweep),
                                                uint32_t(p.draw_bit[rec.x + i])), temperature);
    };
    double bt_next = beta[sweep_begin];
    float temp_next = float(1.0 / bt_next);
    if (!stepper) {
        load_class(0);
        load_keys();
        put_draw(krec, sweep_begin, temp_next, 0);
        load_class(1 % K);
        load_keys();
        load_class(2 % K);
    }
    int buf = 0;
    int wi = 0;   // the next wide bit of the sweep
    int wcls = d.n_wide > 0 ? d.wide[0].cls : -1;
    __syncthreads();
    for (int sweep = sweep_begin; sweep < sweep_end; ++sweep) {
        const double bt = bt_next;
        const float temp = temp_next;
        bt_next = beta[min(sweep + 1, sweep_end - 1)];
        temp_next = float(1.0 / bt_next);
        for (int c = 0; c < K; ++c) {
            while (wcls == c) [[unlikely]] {
                wide_step<T, BITS>(p, s, d.wide + wi, sums, &s_flag, branch_key, sweep, bt);
                ++wi;
                wcls = wi < d.n_wide ? d.wide[wi].cls : -1;
            }
            if (stepper) {
                while (t4.cls == c && t4.sweep == sweep)
                    tile_step<T, BITS, 4>(p, s, t4, s_draw[buf], branch_key, sweep, bt, temp);
                while (t2.cls == c && t2.sweep == sweep)
                    tile_step<T, BITS, 2>(p, s, t2, s_draw[buf], branch_key, sweep, bt, temp);
            } else {
                const bool wrap = c + 1 == K;
                put_draw(krec, wrap ? sweep + 1 : sweep, wrap ? temp_next : temp, buf ^ 1);
                load_keys();
                load_class((c + 3) % K);
            }
            while (t1.cls == c && t1.sweep == sweep)
                tile_step<T, BITS, 1>(p, s, t1, s_draw[buf], branch_key, sweep, bt, temp);
            buf ^= 1;
            lds_barrier();
        }
        wi = 0;
        wcls = d.n_wide > 0 ? d.wide[0].cls : -1;
        if (recompute_every > 0 && (sweep + 1) % recompute_every == 0) [[unlikely]] {
            // residuals from scratch: -d + sum of a over the ray's set bits, in original bit order
            for (int ray = tid; ray < p.n_rays; ray += kSoloBlock) {
                double v = -p.d[ray];
                const int q0 = p.rt_ptr[ray], q1 = p.rt_ptr[ray + 1];
                for (int qa = q0; qa < q1; qa += 8) {
                    BitEnt e[8];
#pragma unroll
                    for (int u = 0; u < 8; ++u) e[u] = p.rt[min(qa + u, q1 - 1)];
#pragma unroll
                    for (int u = 0; u < 8; ++u) {
                        const double nxt = v + double(e[u].a);
                        v = qa + u < q1 && x.at(e[u].pos) ? nxt : v;
                    }
                }
                r[ray] = T(v);
            }
            lds_barrier();
        }
    }
    __syncthreads();
    int words_out = (p.n + 31) / 32, branch_out = int(blockIdx.x);
    asm("" : "+s"(words_out), "+s"(branch_out));   // nothing of this is kept through the sweeps
    uint32_t* x_out = xs + size_t(branch_out) * size_t(words_out);
    for (int k = tid; k < p.n_rays; k += kSoloBlock) rg[k] = r[k];
    if constexpr (BITS) {
        for (int w = tid; w < words_out; w += kSoloBlock) x_out[w] = reinterpret_cast<const uint32_t*>(x.x)[w];
    } else {
        for (int i0 = wave * 64; i0 < p.n; i0 += kSoloBlock) {   // 64 spins a wave
            const int i = i0 + lane;
            const uint64_t m = __ballot(i < p.n && x.x[min(i, p.n - 1)] != 0);
            const int w = i0 / 32 + lane;
            if (lane < 2 && w < words_out) x_out[w] = uint32_t(lane == 0 ? m : m >> 32);
        }
    }
}

// The spins of R branches as the solo kernel leaves them into masks of kGroup branches.
__global__ void __launch_bounds__(256) solo_masks_kernel(const uint32_t* xs, int n, int R, uint16_t* x16) {
    const int pos = int(blockIdx.x * blockDim.x + threadIdx.x);
    if (pos >= n) return;
    const size_t words = size_t(n + 31) / 32;
    const int b0 = int(blockIdx.y) * kGroup;
    unsigned m = 0;
#pragma unroll
    for (int q = 0; q < kGroup; ++q) {
        const int b = min(b0 + q, R - 1);
        const unsigned v = (xs[size_t(b) * words + size_t(pos >> 5)] >> (pos & 31)) & 1u;
        m |= (b0 + q < R ? v : 0u) << q;
    }
    x16[size_t(blockIdx.y) * size_t(n) + size_t(pos)] = uint16_t(m);
}

// One workgroup per tile: writes its chains' heads (planes of one granule per chain; a fourth
// for ray-free tiles) and its entries (planes of 64 lanes), padding the chains the tile does
// not use (j = 255, position 0, padding entries).
__global__ void __launch_bounds__(64) solo_blocks_kernel(DevProblem p, const SoloTile* tiles, const SlotDesc* desc,
                                                         char* blk) {
    const SoloTile m = tiles[blockIdx.x];
    const int lane = int(threadIdx.x);
    const int lpc = m.lpc, ci = lane / lpc, k = lane % lpc, chains = 64 / lpc;
    const bool used = ci < m.chains;
    const SlotDesc s = used ? desc[m.chain0 + ci] : SlotDesc{0, 0, 0, 255u << 5};
    uint4* h = reinterpret_cast<uint4*>(blk + m.at);
    if (k == 0) {
        const int nn = int((s.info >> 21) & 1023u);
        const int nb0 = p.nb_ptr[s.pos];
        int q[kNb];
        for (int u = 0; u < kNb; ++u) q[u] = nn > 0 ? p.nb[nb0 + min(u, nn - 1)] : s.pos;
        const uint64_t lin = uint64_t(__double_as_longlong(p.lin[s.pos])), key = p.draw_key[s.pos];
        h[ci] = uint4{uint32_t(s.pos), (s.info & ~31u) | uint32_t(m.flags), uint32_t(m.next_cls), uint32_t(s.nb0)};
        h[chains + ci] = uint4{uint32_t(q[0]), uint32_t(q[1]), uint32_t(q[2]), uint32_t(q[3])};
        h[2 * chains + ci] = uint4{uint32_t(q[4]), uint32_t(q[5]), uint32_t(lin), uint32_t(lin >> 32)};
        if (lpc == 1) h[3 * chains + ci] = uint4{uint32_t(key), uint32_t(key >> 32), uint32_t(p.draw_bit[s.pos]), 0u};
    }
    static_assert(kNb == 6, "six neighbours in the head");
    if (lpc == 1) return;
    const int len = int(s.info & 31u), rows = kSeg / lpc;
    uint4* e = h + 3 * chains + lane;
    for (int u = 0; u < rows; ++u) {
        uint4 v{uint32_t(p.n_rays), 0u, 0u, 0u};
        if (k * rows + u < len) {
            const RayEnt g = p.ent[s.ka + k * rows + u];
            const uint64_t w = uint64_t(__double_as_longlong(g.w));
            v = uint4{uint32_t(g.ray), __float_as_uint(g.a), uint32_t(w), uint32_t(w >> 32)};
        }
        e[u * 64] = v;
    }
}

__global__ void __launch_bounds__(64) solo_wide_kernel(DevProblem p, SoloWide* wide, int n_wide) {
    const int i = int(blockIdx.x * blockDim.x + threadIdx.x);
    if (i >= n_wide) return;
    SoloWide w = wide[i];
    const int nb0 = p.nb_ptr[w.pos];
    for (int u = 0; u < kNb; ++u) w.q[u] = w.nn > 0 ? p.nb[nb0 + min(u, w.nn - 1)] : w.pos;
    w.bit = p.draw_bit[w.pos];
    w.lin = p.lin[w.pos];
    w.key = p.draw_key[w.pos];
    wide[i] = w;
}

hipError_t launch_solo_blocks(const DevProblem& p, const SoloTile* tiles, const SlotDesc* desc, int n_tiles, void* blk,
                              SoloWide* wide, int n_wide, hipStream_t st) {
    if (n_tiles > 0) solo_blocks_kernel<<<unsigned(n_tiles), 64, 0, st>>>(p, tiles, desc, static_cast<char*>(blk));
    if (n_wide > 0) solo_wide_kernel<<<unsigned((n_wide + 63) / 64), 64, 0, st>>>(p, wide, n_wide);
    return hipGetLastError();
}

// The sums of the longest wide bit, the residuals with their padding slot, the spins.
size_t solo_dynamic_lds(int n, int n_rays, int wide_chains, int precision, bool bits) {
    const size_t tsz = precision == 1 ? sizeof(float) : sizeof(double);
    return sizeof(double) * size_t(wide_chains) + tsz * (size_t(n_rays) + 1) +
           (bits ? sizeof(uint32_t) * ((size_t(n) + 31) / 32) : size_t(n));
}

// A CU's LDS less the kernel's static arrays (draws, chain sums, flag).
size_t solo_lds_limit() {
    return size_t(160) * 1024 - 2 * kSoloDraws * sizeof(Draw) - size_t(kSoloStepWaves) * kSoloPart * sizeof(double) - 64;
}

bool solo_spins_in_bits(int n, int n_rays, int wide_chains, int precision) {
    return solo_dynamic_lds(n, n_rays, wide_chains, precision, false) > solo_lds_limit();
}

hipError_t launch_solo_masks(const void* x, int n, int R, uint16_t* x16, hipStream_t st) {
    const dim3 grid{unsigned((n + 255) / 256), unsigned((R + kGroup - 1) / kGroup)};
    if (n > 0) solo_masks_kernel<<<grid, 256, 0, st>>>(static_cast<const uint32_t*>(x), n, R, x16);
    return hipGetLastError();
}

hipError_t launch_ray_solo(const DevProblem& p, const DevSolo& d, int precision, void* x, void* r, int R,
                           uint64_t seed_offset, const double* beta, int sb, int se, int recompute_every,
                           hipStream_t st) {
    const bool bits = solo_spins_in_bits(p.n, p.n_rays, d.wide_chains, precision);
    const size_t lds = solo_dynamic_lds(p.n, p.n_rays, d.wide_chains, precision, bits);
    if (lds > solo_lds_limit()) return hipErrorInvalidValue;
    auto go = [&](auto zero, auto packed) -> hipError_t {
        using T = decltype(zero);
        constexpr bool BITS = decltype(packed)::value;
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&ray_solo_kernel<T, BITS>),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
        if (e != hipSuccess) return e;
        ray_solo_kernel<T, BITS><<<unsigned(R), kSoloBlock, lds, st>>>(
            p, d, static_cast<uint32_t*>(x), static_cast<T*>(r), seed_offset, beta, sb, se, recompute_every);
        return hipGetLastError();
    };
    if (bits) return precision == 1 ? go(0.0f, std::true_type{}) : go(0.0, std::true_type{});
    return precision == 1 ? go(0.0f, std::false_type{}) : go(0.0, std::false_type{});
}

}  // namespace qb
